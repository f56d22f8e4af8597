"""The column front end on shapes that the slab fold does not take (too many taps per bucket, fewer
buckets than a slab has columns, too many loops): the per-thread column fold against the gathering
front end, bit for bit, launched, profiled, replayed and enqueued."""
import numpy as np
import pytest

import oracle as O
from helpers import draws, params, sparse_signal

pytestmark = pytest.mark.gpu

# over the q = 14, k = 20 configuration: (B, w, B_thresh, W_RLFC, loops)
SHAPES = [(64, 64 * 40 + 7, 20, 512, 7),     # 41 taps per bucket
          (8, 8 * 20 + 3, 4, 2048, 7),       # 8 buckets: half a slab's columns and less
          (512, 512 * 9, 40, 512, 32)]       # 32 loops, no tail tap


@pytest.mark.parametrize("fold_mode", [O.FOLD_REFERENCE, O.FOLD_ALL_TAPS])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%d_w%d_l%d" % (s[0], s[1], s[4]))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_columns_without_the_slab(precision, shape, fold_mode):
    import torch
    import sfft_amd as S
    B, w, K, W, loops = shape
    prm = dict(params((14, 20, 1.0, 2, 2, 5, 4, 2)), B=B, w=w, B_thresh=K, W_RLFC=W, loops=loops,
               loops_est=loops - 2)
    n = prm["n"]
    cdt = np.complex64 if precision == "fp32" else np.complex128
    rng = np.random.default_rng(B + w)
    x, _, _ = sparse_signal(n, prm["k"], 5, snr_db=30.0)
    dx = torch.from_numpy(x.astype(cdt)).cuda()
    taps = torch.from_numpy((rng.standard_normal(w) + 1j * rng.standard_normal(w))
                            .astype(cdt)).cuda()
    win = 1.0 + rng.random(n // B) + 0j
    sets = [draws(n, loops, prm["RLFC_loops"], W, 60 + i) for i in range(3)]
    ref = S.Plan(prm, precision, fold_mode=fold_mode, front_end="gather")
    ref.set_filter(taps, win)
    want = [ref.execute(dx, *d) for d in sets]
    assert want[0][1] > 0
    auto = S.Plan(prm, precision, fold_mode=fold_mode)
    assert auto.front_end == "gather"            # a shape that the slab does not take
    plan = S.Plan(prm, precision, fold_mode=fold_mode, front_end="columns")
    assert plan.front_end == "columns"
    plan.set_filter(taps, win)
    for mode in ("eager", "profiled", "graph"):
        plan.set_profiling(mode == "profiled")
        plan.set_graph(mode == "graph")
        for d, (nodes, cnt) in list(zip(sets, want)) * 2:
            got, c = plan.execute(dx, *d)
            assert c == cnt and got.tobytes() == nodes.tobytes(), mode
        buf = torch.zeros(plan.capacity * 24, dtype=torch.uint8, device="cuda")
        num = torch.zeros(1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        for d in sets:                           # queued: the last one's result
            plan.execute_async(dx, *d, d_nodes=buf, d_count=num)
        torch.cuda.synchronize()
        nodes, cnt = want[-1]
        assert int(num.item()) == cnt, mode
        assert buf.cpu().numpy()[:24 * cnt].tobytes() == nodes.tobytes(), mode
