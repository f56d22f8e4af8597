"""The dense FFT's special first loads and last stores (truth spectra, filter design), in-place
transforms and scratch kept between calls, against the canonical FFT of the oracle bit for
bit."""
import numpy as np
import pytest

import oracle as O
from helpers import bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import sfft_amd
    return sfft_amd


def _x(n, dtype, seed=0):
    rng = np.random.default_rng(n + seed)
    return (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(dtype)


# one, two and three passes, the edges between them
@pytest.mark.parametrize("log2n", [1, 2, 5, 11, 12, 16, 22, 23])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_truth_spectrum_bits(S, log2n, dtype):
    import torch
    n = 1 << log2n
    x = _x(n, dtype)
    got = S.truth_spectrum(torch.from_numpy(x).cuda()).cpu().numpy()
    want = O.fft64(x.astype(np.complex128)) / n
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("log2n", [3, 12, 23])
def test_truth_spectrum_in_place(S, log2n):
    """d_X on top of the signal (complex128), and on top of a complex64 signal inside it"""
    import ctypes as C
    import torch
    n = 1 << log2n
    for fp32 in (0, 1):
        x = _x(n, np.complex64 if fp32 else np.complex128, 5)
        buf = torch.zeros(n, dtype=torch.complex128, device="cuda")
        flat = torch.view_as_real(buf).view(-1)
        src = torch.view_as_real(torch.from_numpy(x).cuda()).view(-1)
        if fp32:
            flat.view(torch.float32)[2 * n:] = src      # the upper half of the spectrum
            px = buf.data_ptr() + 8 * n
        else:
            flat[:] = src
            px = buf.data_ptr()
        torch.cuda.synchronize()
        assert S.lib.sfft_truth_spectrum(C.c_void_p(px), n, fp32, C.c_void_p(buf.data_ptr()),
                                         None) == 0
        want = O.fft64(x.astype(np.complex128)) / n
        assert np.array_equal(bits(buf.cpu().numpy()), bits(want))


@pytest.mark.parametrize("log2n,count", [(4, 3), (11, 2), (12, 3), (17, 2), (23, 1)])
@pytest.mark.parametrize("inverse", [False, True])
def test_fft_in_place(S, log2n, count, inverse):
    import torch
    for dtype in (np.complex64, np.complex128):
        x = np.stack([_x(1 << log2n, dtype, i) for i in range(count)])
        t = torch.from_numpy(x).cuda()
        want = S.fft(t, inverse=inverse).cpu().numpy()
        assert S.fft(t, inverse=inverse, out=t) is t
        assert np.array_equal(bits(t.cpu().numpy()), bits(want))


def test_scratch_between_streams_and_threads(S):
    """transforms that share the scratch pool from several threads and streams keep apart"""
    import threading
    import torch
    xs = [torch.from_numpy(_x(1 << 18, np.complex128, i)).cuda() for i in range(4)]
    want = [S.fft(x).cpu().numpy() for x in xs]
    torch.cuda.synchronize()
    got = [None] * 4

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            outs = [S.fft(xs[i]) for _ in range(6)]
        s.synchronize()
        got[i] = [o.cpu().numpy() for o in outs]

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for i in range(4):
        for o in got[i]:
            assert np.array_equal(bits(o), bits(want[i]))


@pytest.mark.parametrize("n,w", [(1 << 12, 1849), (1 << 14, 3), (1 << 14, 1 << 14), (1 << 23, 631)])
def test_design_modes_share_their_ffts(S, n, w):
    """the taps' load and the head's store in both designs: the faithful taps and response are
    the oracle's bits; a response asked for on the device does not change the taps"""
    ft, ff = S.make_filter(0.01, 1e-8, n, 40, w=w, mode="faithful", freq="host")
    fo, fr = O.make_multiple_t(0.01, 1e-8, n, 40, w)
    assert np.array_equal(bits(ft.cpu().numpy()), bits(fo))
    assert np.array_equal(bits(ff), bits(fr))
    a, ra = S.make_filter(0.01, 1e-8, n, 40, w=w, mode="parallel", freq="device")
    b, _ = S.make_filter(0.01, 1e-8, n, 40, w=w, mode="parallel", freq=None)
    assert np.array_equal(bits(a.cpu().numpy()), bits(b.cpu().numpy()))
