"""Short transforms, whose comb and bucket stages share their launches, against the same plan with
profiling on (a launch per stage) and against the gathering front end, bit for bit: one- and
two-pass FFTs of either, each length of the one-workgroup cutoffs and the first above it, many
loops, and signals whose keys all tie or overflow."""
import numpy as np
import pytest

import oracle as O
from helpers import N20_K1000, SMALL_CONFIGS, draws, oracle_filter, params, sparse_signal

pytestmark = pytest.mark.gpu

CONFIGS = SMALL_CONFIGS + [
    (14, 20, 1.0, 4, 3, 15, 8, 3), (15, 30, 1.0, 2, 2, 5, 4, 2), (17, 100, 1.0, 2, 2, 5, 64, 2),
    (18, 200, 1.0, 2, 2, 5, 128, 8), (18, 300, 1.40, 2, 2, 5, 32, 2), N20_K1000,
    (20, 600, 1.0, 2, 2, 3, 256, 2), (21, 1000, 1.40, 2, 2, 5, 128, 2)]


@pytest.mark.parametrize("kind", ["noise", "zero", "huge"])
@pytest.mark.parametrize("cfg", CONFIGS, ids=lambda c: "q%d_k%d_l%d" % (c[0], c[1], c[3] + c[5]))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_shared_launches_keep_the_bits(precision, cfg, kind):
    import torch
    import sfft_amd as S
    prm = params(cfg)
    n = prm["n"]
    cdt = np.complex64 if precision == "fp32" else np.complex128
    x, _, _ = sparse_signal(n, prm["k"], 5, snr_db=30.0)
    if kind == "zero":
        x = np.zeros_like(x)
    elif kind == "huge":   # its square overflows: nearly every key is infinite
        x[n // 3] = 1e25 if precision == "fp32" else 1e200
    ft, ff = oracle_filter(prm)
    dx = torch.from_numpy(x.astype(cdt)).cuda()
    dft = torch.from_numpy(ft.astype(cdt)).cuda()
    win = O.filter_window_slice(ff, n, prm["B"])
    d = draws(n, prm["loops"], prm["RLFC_loops"], prm["W_RLFC"], 17)
    out = {}
    for how in ("shared", "profiled", "gather"):
        plan = S.Plan(prm, precision, front_end="gather" if how == "gather" else "auto")
        plan.set_filter(dft, win)
        plan.set_profiling(how == "profiled")
        try:
            out[how] = plan.execute(dx, *d)
        except S.SfftError as e:
            out[how] = (np.zeros(0, np.uint8), str(e))
        for graph in ((True,) if how == "shared" else ()):
            plan.set_graph(graph)
            for _ in range(3):
                try:
                    nodes, cnt = plan.execute(dx, *d)
                except S.SfftError as e:
                    nodes, cnt = np.zeros(0, np.uint8), str(e)
                assert cnt == out["shared"][1]
                assert nodes.tobytes() == out["shared"][0].tobytes()
    for how in ("profiled", "gather"):
        assert out[how][1] == out["shared"][1], how
        assert out[how][0].tobytes() == out["shared"][0].tobytes(), how
