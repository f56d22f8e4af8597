"""The walk's hits and their values in one launch, where a block lists more hits than it takes at a
time, where the capacity cuts the list inside a block, and where blocks have none."""
import numpy as np
import pytest

import oracle as O
from helpers import draws, params

pytestmark = pytest.mark.gpu


def _case(n, B, K, W, loops_loc, thresh, loops, seed):
    prm = dict(params((14, 20, 1.0, 2, 2, 5, 4, 2)), n=n, B=B, w=max(B, 1849), B_thresh=K, W_RLFC=W,
               loops_loc=loops_loc, loops_thresh=thresh, loops=loops, loops_est=loops - loops_loc)
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    ft = rng.standard_normal(prm["w"]) + 1j * rng.standard_normal(prm["w"])
    win = 1.0 + rng.random(n // B) + 1j * rng.random(n // B)
    a, ai, offs = draws(n, loops, prm["RLFC_loops"], W, seed)
    return prm, x, ft, win, a, ai, offs


# dense: nearly every position of long windows approved (thousands of hits per block); sparse
@pytest.mark.parametrize("K,thresh,loops", [(60, 1, 3), (63, 2, 18), (1, 1, 2)])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("capacity", [0, 1, 700, 3000])
def test_nodes_lists(K, thresh, loops, fp32, capacity):
    import ctypes as C
    import torch
    import sfft_amd as S
    n, B, W = 1 << 14, 64, 1 << 8
    prm, x, ft, win, a, ai, offs = _case(n, B, K, W, 2, thresh, loops, 11 + K)
    if fp32:
        x, ft = x.astype(np.complex64), ft.astype(np.complex64)
    ref = (O.outer_loop32 if fp32 else O.outer_loop64)(prm, x, ft, win, a, ai, offs)
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to("cuda")  # noqa: E731
    plan = S.Plan(prm, "fp32" if fp32 else "fp64", hit_capacity=capacity)
    ftd, xd = dev(ft), dev(x)
    plan.set_filter(ftd, win)
    cap = capacity or 524288
    got = torch.zeros(cap * 24 + 48, dtype=torch.uint8, device="cuda")
    cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
    plan.execute_async(xd, a, ai, offs, d_nodes=got, d_count=cnt)
    torch.cuda.synchronize()
    assert int(cnt.item()) == ref["I_F"]
    k = min(cap, ref["I_F"])
    buf = got.cpu().numpy()
    assert buf[:24 * k].tobytes() == ref["nodes"][:k].tobytes()
    assert not buf[24 * k:].any()           # nothing past the hits or the capacity
    assert np.array_equal(plan.debug_array(3, k, np.int32), ref["hits"][:k])
