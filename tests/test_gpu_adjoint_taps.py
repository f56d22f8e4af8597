"""The taps step of the adjoint (each signal index looks its taps up) against the oracle, bit for
bit, where its lookup can go wrong: one and many taps per bucket, no residue, one tail tap, more
loops than are loaded together, both fold modes."""
import numpy as np
import pytest

import oracle as O
from helpers import bits, draws, params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fold_mode", [O.FOLD_REFERENCE, O.FOLD_ALL_TAPS])
@pytest.mark.parametrize("B,w", [(1024, 1024), (1024, 1025), (1024, 2047), (512, 1536),
                                 (128, 1849), (64, 4097), (8, 16383), (128, 16384)])
@pytest.mark.parametrize("loops", [2, 8, 9, 17])
def test_adjoint_taps_edges(B, w, loops, fold_mode):
    import torch
    import sfft_amd as S
    prm = dict(params((14, 20, 1.0, 2, 2, 5, 4, 2)), B=B, w=w, loops=loops, loops_est=loops - 2,
               B_thresh=min(40, B // 2), W_RLFC=max(512, (1 << 14) // B))
    n = prm["n"]
    rng = np.random.default_rng(B + w + loops)
    ft = rng.standard_normal(w) + 1j * rng.standard_normal(w)
    win = 1.0 + rng.random(n // B) + 1j * rng.random(n // B)
    a, ai, offs = draws(n, loops, prm["RLFC_loops"], prm["W_RLFC"], 9)
    nh = 300
    hits = rng.integers(0, n, nh).astype(np.int32)
    sel = rng.integers(0, loops, (nh, 2)).astype(np.uint8)
    g = rng.standard_normal(nh) + 1j * rng.standard_normal(nh)
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to("cuda")  # noqa: E731
    plan = S.Plan(prm, "fp64", fold_mode=fold_mode, front_end="gather")
    plan.set_filter(dev(ft), win)
    got = plan.value_adjoint(dev(g), a, ai, offs, dev(hits), dev(sel)).cpu().numpy()
    want = O.value_adjoint64(prm, ft, win, ai, hits, sel, g, fold_mode)
    assert np.array_equal(bits(got), bits(want))
