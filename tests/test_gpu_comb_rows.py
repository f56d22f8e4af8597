"""Comb FFTs of copied comb rows whose sibling sub-FFTs fill a tile or are more than its columns
(long windows n/B), against the front end that gathers the comb, bit for bit."""
import numpy as np
import pytest

from helpers import draws, params

pytestmark = pytest.mark.gpu


# (log2 n, B, log2 W): quarter and full tiles, siblings a fraction of the columns to 2^4 times them
@pytest.mark.parametrize("q,B,lw", [(14, 64, 12), (15, 32, 12), (17, 32, 12), (17, 32, 13),
                                    (17, 64, 17), (18, 32, 18), (20, 32, 15), (20, 32, 19),
                                    (20, 64, 20), (21, 32, 21), (22, 32, 17)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_sibling_tiles(precision, q, B, lw):
    import torch
    import sfft_amd as S
    n = 1 << q
    prm = dict(params((14, 20, 1.0, 2, 2, 5, 4, 2)), n=n, B=B, w=5 * B + 3, B_thresh=9,
               W_RLFC=1 << lw, RLFC_loops=2, loops_loc=2, loops_thresh=2, loops=4, loops_est=2)
    rng = np.random.default_rng(q + lw)
    cdt = np.complex64 if precision == "fp32" else np.complex128
    x = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(cdt)
    ft = (rng.standard_normal(prm["w"]) + 1j * rng.standard_normal(prm["w"])).astype(cdt)
    win = 1.0 + rng.random(n // B) + 0j
    d = draws(n, prm["loops"], 2, 1 << lw, 7)
    dx, dft = torch.from_numpy(x).cuda(), torch.from_numpy(ft).cuda()
    keys, out = [], []
    for fe in ("columns", "gather"):
        plan = S.Plan(prm, precision, front_end=fe)
        plan.set_filter(dft, win)
        nodes, cnt = plan.execute(dx, *d)
        out.append((nodes.tobytes(), cnt))
        keys.append(plan.debug_array(8, 2 << lw, np.uint32 if precision == "fp32" else np.uint64))
    assert out[0] == out[1]
    assert np.array_equal(keys[0], keys[1])   # every comb key
