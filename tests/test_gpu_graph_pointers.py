"""Transforms whose signal and result buffers change from call to call, in graph mode: queued ones
give the waited-for ones' results, and a call on new buffers does not wait for the transforms queued
before it."""
import numpy as np
import pytest

import oracle as O
from helpers import SMALL_CONFIGS, draws, oracle_filter, params, sparse_signal

pytestmark = pytest.mark.gpu

# transforms whose comb and bucket stages run on two streams
CONFIGS = [(SMALL_CONFIGS[1], "gather", "fp64"), ((22, 300, 0.99, 2, 2, 3, 256, 2), "columns", "fp32")]
IDS = ["q14_gather_fp64", "q22_columns_fp32"]


def _setup(cfg, front_end, precision, sets):
    import torch
    import sfft_amd as S
    prm = params(cfg)
    n = prm["n"]
    cdt = np.complex64 if precision == "fp32" else np.complex128
    ft, ff = oracle_filter(prm)
    dft = torch.from_numpy(ft.astype(cdt)).cuda()
    win = O.filter_window_slice(ff, n, prm["B"])
    stream = torch.cuda.Stream()
    plan = S.Plan(prm, precision, stream=stream, front_end=front_end, hit_capacity=65536)
    plan.set_filter(dft, win)
    xs = [torch.from_numpy(sparse_signal(n, prm["k"], 20 + i)[0].astype(cdt)).cuda()
          for i in range(sets)]
    ds = [tuple(np.ascontiguousarray(v, np.int32) for v in
                draws(n, prm["loops"], prm["RLFC_loops"], prm["W_RLFC"], 30 + i))
          for i in range(3)]
    want = [[plan.execute(x, *d) for d in ds] for x in xs]
    bufs = [(torch.zeros(plan.capacity * 24, dtype=torch.uint8, device="cuda"),
             torch.zeros(1, dtype=torch.int32, device="cuda")) for _ in xs]
    plan.set_graph(True)
    torch.cuda.synchronize()
    return plan, stream, xs, ds, want, bufs


@pytest.mark.parametrize("cfg,front_end,precision", CONFIGS, ids=IDS)
def test_queued_on_changing_buffers(cfg, front_end, precision):
    import torch
    plan, stream, xs, ds, want, bufs = _setup(cfg, front_end, precision, 3)
    order = [0, 1, 2, 0, 0, 1, 1, 1, 2, 0, 2, 2, 1, 0, 1, 2] * 3   # changed and kept buffers
    for wait in (False, True):
        last = {}
        for j, s in enumerate(order):
            d = (j * 7 + s) % len(ds)
            buf, cnt = bufs[s]
            plan.execute_async(xs[s], *ds[d], d_nodes=buf, d_count=cnt)
            last[s] = d
            if wait:
                torch.cuda.synchronize()
        torch.cuda.synchronize()
        for s, d in last.items():
            nodes, k = want[s][d]
            assert int(bufs[s][1].item()) == k
            assert bufs[s][0].cpu().numpy()[:24 * k].tobytes() == nodes.tobytes()
            bufs[s][0].zero_()
        # and waited-for transforms between them
        for s in (0, 1, 1, 1):
            nodes, k = plan.execute(xs[s], *ds[1])
            assert k == want[s][1][1] and nodes.tobytes() == want[s][1][0].tobytes()
    plan.close()


@pytest.mark.parametrize("cfg,front_end,precision", CONFIGS, ids=IDS)
def test_new_buffers_do_not_wait(cfg, front_end, precision):
    import torch
    plan, stream, xs, ds, want, bufs = _setup(cfg, front_end, precision, 3)
    busy = torch.cuda.Event()
    with torch.cuda.stream(stream):
        a = torch.randn(8192, 8192, device="cuda")
        out = torch.mm(a, a)
        torch.cuda.synchronize()
        for _ in range(60):                      # some hundred milliseconds of work in front
            torch.mm(a, a, out=out)
        busy.record(stream)
    waited = []
    for s in (0, 1, 2, 2, 2, 0):
        plan.execute_async(xs[s], *ds[s], d_nodes=bufs[s][0], d_count=bufs[s][1])
        waited.append(busy.query())
    torch.cuda.synchronize()
    for s in range(3):
        nodes, k = want[s][s]
        assert int(bufs[s][1].item()) == k
        assert bufs[s][0].cpu().numpy()[:24 * k].tobytes() == nodes.tobytes()
    plan.close()
    assert not any(waited), waited
