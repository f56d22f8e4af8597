"""Single-pass FFTs of many adjacent rows (whole rows fill a tile) against the oracle bit for
bit: every length up to one pass, row counts around whole tiles and their remainders."""
import numpy as np
import pytest

import oracle as O
from helpers import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2n", range(1, 12))
@pytest.mark.parametrize("count", [2, 1023, 1024, 1537, 5000])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_fft_rows(log2n, count, dtype):
    import torch
    import sfft_amd as S
    n = 1 << log2n
    rng = np.random.default_rng(log2n * 100003 + count)
    x = (rng.standard_normal((count, n)) + 1j * rng.standard_normal((count, n))).astype(dtype)
    t = torch.from_numpy(x).cuda()
    fft = O.fft32 if dtype == np.complex64 else O.fft64
    rows = sorted({0, 1, count // 2, count - 1, *rng.integers(0, count, 40).tolist()})
    for inverse in (False, True):
        got = S.fft(t, inverse=inverse).cpu().numpy()
        # every row against numpy, some against the oracle's bits
        ref = np.fft.ifft(x.astype(np.complex128)) * n if inverse else \
            np.fft.fft(x.astype(np.complex128))
        eps = 1e-6 if dtype == np.complex64 else 1e-14
        err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
        assert err.max() <= eps * (log2n + 1)
        for c in rows:
            assert np.array_equal(bits(got[c]), bits(fft(x[c], inverse))), f"row {c}"
