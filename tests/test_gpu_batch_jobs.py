"""A batch whose signals fall on different sides of every stage's variants (one- and two-pass
FFTs, one-workgroup and chained cutoffs, loop counts with kernels of their own), against the
single transforms bit for bit, with the nodes in pinned, pageable or no host memory."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from helpers import draws, oracle_filter, params, sparse_signal

pytestmark = pytest.mark.gpu

# comb lengths 512 .. 65536, buckets 32 .. 8192, 3 .. 19 loops, thresholds 1 .. 3
CONFIGS = [(14, 20, 1.0, 2, 2, 5, 4, 2), (12, 8, 1.0, 2, 2, 3, 8, 2), (17, 100, 0.8, 2, 1, 1, 32, 1),
           (20, 600, 1.0, 2, 2, 3, 256, 2), (16, 50, 1.0, 3, 2, 4, 16, 2),
           (14, 20, 1.0, 4, 3, 15, 8, 3), (20, 1000, 1.40, 2, 2, 5, 128, 2)]
NODE = np.dtype([("key", np.uint32), ("pad", np.uint32), ("re", np.float64), ("im", np.float64)])


@pytest.fixture(scope="module")
def S():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import sfft_amd
    return sfft_amd


# every signal gathered; every signal the plan's own choice (columns where the slab applies); an
# oversized window beside them, which the slab does not take
@pytest.mark.parametrize("front_end", ["gather", "auto"])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_batch_mixed_variants_and_node_memory(S, precision, front_end):
    import torch
    cdt = np.complex64 if precision == "fp32" else np.complex128
    prms = [params(c) for c in CONFIGS]
    prms.append(dict(prms[0], B=64, w=64 * 40 + 7, B_thresh=20))   # 41 taps per bucket
    xs, fts, wins, dr, want = [], [], [], [], []
    for i, p in enumerate(prms):
        x, _, _ = sparse_signal(p["n"], p["k"], 50 + i, snr_db=30.0)
        if i < len(CONFIGS):
            ft, ff = oracle_filter(p)
            win = O.filter_window_slice(ff, p["n"], p["B"])
        else:
            rng = np.random.default_rng(8)
            ft = rng.standard_normal(p["w"]) + 1j * rng.standard_normal(p["w"])
            win = 1.0 + rng.random(p["n"] // p["B"]) + 0j
        xs.append(torch.from_numpy(x.astype(cdt)).cuda())
        fts.append(torch.from_numpy(ft.astype(cdt)).cuda())
        wins.append(win)
        dr.append(draws(p["n"], p["loops"], p["RLFC_loops"], p["W_RLFC"], 70 + i))
        plan = S.Plan(p, precision)
        plan.set_filter(fts[i], wins[i])
        want.append(plan.execute(xs[i], *dr[i]))
    b = S.Batch(prms, precision, front_end=front_end)
    fronts = {S.lib.sfft_plan_front_end(S.lib.sfft_batch_plan(b._h, i)) for i in range(len(prms))}
    assert fronts == ({1} if front_end == "gather" else {1, 3})
    for i in range(len(prms)):
        b.set_filter(i, fts[i], wins[i])
    cap = 524288
    ptrs, cdr, keep = b._args(xs, dr)
    for graph in (False, True):
        b.set_graph(graph)
        for rep in range(2):
            pinned = torch.zeros(len(prms) * cap * 24, dtype=torch.uint8, pin_memory=True)
            pageable = [np.zeros(cap, NODE) for _ in prms]
            # signal i: 0 pinned, 1 pageable, 2 none, in turn and differently in each repetition
            how = [(i + rep) % 3 for i in range(len(prms))]
            addr = [pinned.data_ptr() + i * cap * 24 if h == 0 else
                    pageable[i].ctypes.data if h == 1 else None for i, h in enumerate(how)]
            counts = np.zeros(len(prms), np.int32)
            torch.cuda.synchronize()
            assert S.lib.sfft_batch_execute(b._h, ptrs, cdr, (C.c_void_p * len(prms))(*addr),
                                            counts.ctypes.data_as(C.c_void_p)) == 0
            host = pinned.numpy().view(NODE).reshape(len(prms), cap)
            for i, (nodes, cnt) in enumerate(want):
                assert counts[i] == cnt, f"signal {i}"
                if how[i] < 2:
                    got = host[i] if how[i] == 0 else pageable[i]
                    assert got[:cnt].tobytes() == nodes.tobytes(), f"signal {i}"
                    assert not got[cnt:].view(np.uint8).any()   # nothing past the count
        # and through the binding, which reads the nodes from the plans' device buffers
        for (nodes, cnt), (wn, wc) in zip(b.execute(xs, dr), want):
            assert cnt == wc and nodes.tobytes() == wn.tobytes()
    b.close()


def test_batch_device_nodes_beside_pinned_ones(S):
    """the plans' node buffers hold the batch's last transform also when the nodes went to pinned
    memory"""
    import torch
    p = params(CONFIGS[0])
    x, _, _ = sparse_signal(p["n"], p["k"], 3)
    ft, ff = oracle_filter(p)
    d = draws(p["n"], p["loops"], p["RLFC_loops"], p["W_RLFC"], 4)
    b = S.Batch([p, p], "fp64")
    xt, ftt = torch.from_numpy(x).cuda(), torch.from_numpy(ft).cuda()
    for i in range(2):
        b.set_filter(i, ftt, O.filter_window_slice(ff, p["n"], p["B"]))
    ptrs, cdr, keep = b._args([xt, xt], [d, d])
    pinned = torch.zeros(2 * 524288 * 24, dtype=torch.uint8, pin_memory=True)
    counts = np.zeros(2, np.int32)
    torch.cuda.synchronize()
    addr = (C.c_void_p * 2)(pinned.data_ptr(), pinned.data_ptr() + 524288 * 24)
    assert S.lib.sfft_batch_execute(b._h, ptrs, cdr, addr, counts.ctypes.data_as(C.c_void_p)) == 0
    for i in range(2):
        dev = np.empty(counts[i], NODE)
        src = S.lib.sfft_plan_debug_buffer(S.lib.sfft_batch_plan(b._h, i), 5)
        hip = C.CDLL("libamdhip64.so")
        assert hip.hipMemcpy(dev.ctypes.data_as(C.c_void_p), C.c_void_p(src),
                             C.c_size_t(dev.nbytes), 2) == 0
        host = pinned.numpy().view(NODE)[i * 524288:i * 524288 + counts[i]]
        assert dev.tobytes() == host.tobytes()
    b.close()


def test_tune_of_a_batch_that_gathers_and_folds(S):
    """the tuner times the gathering signals' launch, whose table holds only them"""
    import torch
    prms = [params(CONFIGS[0]), dict(params(CONFIGS[0]), B=64, w=64 * 40 + 7, B_thresh=20),
            params(CONFIGS[3])]
    rng = np.random.default_rng(9)
    xs, taps, dr, b = [], [], [], S.Batch(prms, "fp32", front_end="auto")
    fronts = [S.lib.sfft_plan_front_end(S.lib.sfft_batch_plan(b._h, i)) for i in range(3)]
    assert fronts.count(1) == 1 and fronts.count(3) == 2
    want = []
    for i, p in enumerate(prms):
        x, _, _ = sparse_signal(p["n"], p["k"], 80 + i, snr_db=30.0)
        ft = rng.standard_normal(p["w"]) + 1j * rng.standard_normal(p["w"])
        win = 1.0 + rng.random(p["n"] // p["B"]) + 0j
        xs.append(torch.from_numpy(x.astype(np.complex64)).cuda())
        taps.append(torch.from_numpy(ft.astype(np.complex64)).cuda())
        dr.append(draws(p["n"], p["loops"], p["RLFC_loops"], p["W_RLFC"], 90 + i))
        b.set_filter(i, taps[i], win)
        plan = S.Plan(p, "fp32")
        plan.set_filter(taps[i], win)
        want.append(plan.execute(xs[i], *dr[i]))
    b.tune(xs, dr, reps=1)
    for (nodes, cnt), (wn, wc) in zip(b.execute(xs, dr), want):
        assert cnt == wc and nodes.tobytes() == wn.tobytes()
    b.close()
