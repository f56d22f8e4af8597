"""The taps step of the adjoint on both sides of the rule that sends few taps in a long signal in
their own order, against the oracle, bit for bit: a fraction of the border, the last width below and
the first above it, with and without tail taps, up to and beyond one chunk of loops."""
import numpy as np
import pytest

import oracle as O
from helpers import bits, draws, params

pytestmark = pytest.mark.gpu

N = 1 << 23


def _border(loops):
    """the widest w whose taps go in their own order"""
    places = (loops + 3) // 4 * 4
    return N // 80 if loops <= 8 else N * places // (72 * loops)


@pytest.mark.parametrize("fold_mode", [O.FOLD_REFERENCE, O.FOLD_ALL_TAPS])
@pytest.mark.parametrize("loops", [2, 8, 9])
@pytest.mark.parametrize("width", ["few", "no tail", "below", "above"])
def test_adjoint_taps_rule(width, loops, fold_mode):
    import torch
    import sfft_amd as S
    B = 8192
    w = {"few": B + 5, "no tail": 8 * B, "below": _border(loops),
         "above": _border(loops) + 1}[width]
    prm = dict(params((23, 300, 0.99, 2, 2, 3, 256, 2)), B=B, w=w, loops=loops,
               loops_est=loops - 2, B_thresh=600)
    rng = np.random.default_rng(w + loops)
    ft = rng.standard_normal(w) + 1j * rng.standard_normal(w)
    win = 1.0 + rng.random(N // B) + 1j * rng.random(N // B)
    a, ai, offs = draws(N, loops, prm["RLFC_loops"], prm["W_RLFC"], 9)
    nh = 300
    hits = rng.integers(0, N, nh).astype(np.int32)
    sel = rng.integers(0, loops, (nh, 2)).astype(np.uint8)
    g = rng.standard_normal(nh) + 1j * rng.standard_normal(nh)
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to("cuda")  # noqa: E731
    plan = S.Plan(prm, "fp64", fold_mode=fold_mode, front_end="gather", hit_capacity=4096)
    plan.set_filter(dev(ft), win)
    got = plan.value_adjoint(dev(g), a, ai, offs, dev(hits), dev(sel)).cpu().numpy()
    want = O.value_adjoint64(prm, ft, win, ai, hits, sel, g, fold_mode)
    assert np.array_equal(bits(got), bits(want))
