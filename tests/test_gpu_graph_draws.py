"""The draws travel as the first kernel's argument: graph replays and eager launches with a new
draw set each, enqueued one behind the other without waiting, equal the waited-for transform of
each draw set, for every front end and on both sides of the size that replays a graph."""
import numpy as np
import pytest

import oracle as O
from helpers import N20_K1000, SMALL_CONFIGS, draws, oracle_filter, params, sparse_signal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("front_end", ["columns", "gather", "stream"])
@pytest.mark.parametrize("cfg", [SMALL_CONFIGS[1], N20_K1000, (22, 300, 0.99, 2, 2, 3, 256, 2)],
                         ids=["q14", "q20", "q22"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_queued_transforms_keep_their_draws(front_end, cfg, precision):
    import torch
    import sfft_amd as S
    prm = params(cfg)
    n = prm["n"]
    cdt = np.complex64 if precision == "fp32" else np.complex128
    x, _, _ = sparse_signal(n, prm["k"], 3)
    ft, ff = oracle_filter(prm)
    dx = torch.from_numpy(x.astype(cdt)).cuda()
    dft = torch.from_numpy(ft.astype(cdt)).cuda()
    win = O.filter_window_slice(ff, n, prm["B"])
    sets = [draws(n, prm["loops"], prm["RLFC_loops"], prm["W_RLFC"], 40 + i) for i in range(5)]
    plan = S.Plan(prm, precision, front_end=front_end)
    plan.set_filter(dft, win)
    want = [plan.execute(dx, *d) for d in sets]
    assert len({w[0].tobytes() for w in want}) == len(sets)   # the draw sets tell apart
    cap = 16384
    for graph in (False, True):
        plan.set_graph(graph)
        for rep in range(2):
            # one result buffer (the graph's), copied out behind each transform
            buf = torch.zeros(plan.capacity * 24, dtype=torch.uint8, device="cuda")
            cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
            got = []
            torch.cuda.synchronize()
            for d in sets + sets[::-1]:
                plan.execute_async(dx, *d, d_nodes=buf, d_count=cnt)
                if graph:
                    torch.cuda.synchronize()   # (a plan's own stream: copies cannot follow it)
                got.append((buf[:24 * cap].clone(), cnt.clone()))
            torch.cuda.synchronize()
            for (b, c), (nodes, k) in zip(got, want + want[::-1]):
                assert int(c.item()) == k
                m = min(k, cap)
                assert b.cpu().numpy()[:24 * m].tobytes() == nodes[:m].tobytes()
        # queued without waiting in between: the last one's result
        for first in range(len(sets)):
            for d in sets[first:] + sets[:first]:
                plan.execute_async(dx, *d, d_nodes=buf, d_count=cnt)
            torch.cuda.synchronize()
            nodes, k = want[first - 1]
            assert int(cnt.item()) == k
            assert buf.cpu().numpy()[:24 * k].tobytes() == nodes.tobytes()
        for d, (nodes, k) in zip(sets, want):
            got_nodes, kk = plan.execute(dx, *d)
            assert kk == k and got_nodes.tobytes() == nodes.tobytes()
