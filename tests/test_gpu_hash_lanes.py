"""The reverse hash's lanes per bucket window (they depend on the window length and on how many
windows there are) against the oracle's ordered hit list, from windows of 2 positions to long
ones, few and many of them."""
import numpy as np
import pytest

import oracle as O
from helpers import draws, params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,K", [(8192, 3000), (4096, 2000), (2048, 37), (1024, 900), (256, 3),
                                 (256, 200), (64, 60), (16, 1), (16, 12), (4, 3)])
@pytest.mark.parametrize("loops_loc,thresh", [(1, 1), (2, 2), (3, 2)])
def test_hit_list(B, K, loops_loc, thresh):
    import torch
    import sfft_amd as S
    n, W = 1 << 14, 1 << 13
    K = min(K, B - 1)
    prm = dict(params((14, 20, 1.0, 2, 2, 5, 4, 2)), B=B, w=max(B, 1849), B_thresh=K, W_RLFC=W,
               loops_loc=loops_loc, loops_thresh=thresh, loops=loops_loc + 2, loops_est=2)
    rng = np.random.default_rng(B + K)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    ft = rng.standard_normal(prm["w"]) + 1j * rng.standard_normal(prm["w"])
    win = 1.0 + rng.random(n // B) + 1j * rng.random(n // B)
    a, ai, offs = draws(n, prm["loops"], prm["RLFC_loops"], W, 5)
    ref = O.outer_loop64(prm, x, ft, win, a, ai, offs)
    plan = S.Plan(prm, "fp64")
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to("cuda")  # noqa: E731
    ftd = dev(ft)
    plan.set_filter(ftd, win)
    nodes, cnt = plan.execute(dev(x), a, ai, offs)
    assert cnt == ref["I_F"]
    assert np.array_equal(plan.debug_array(3, cnt, np.int32), ref["hits"])
    assert nodes.tobytes() == ref["nodes"].tobytes()
