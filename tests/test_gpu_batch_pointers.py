"""A batch whose signal and node pointers change from call to call: the results are the single
transforms' bit for bit, launched and replayed, with calls queued one behind the other, and a call
on new pointers does not wait for the device work in front of it."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from helpers import draws, oracle_filter, params, sparse_signal

pytestmark = pytest.mark.gpu

# column and gathering signals, one-workgroup and chained cutoffs
CONFIGS = [(14, 20, 1.0, 2, 2, 5, 4, 2), (17, 100, 0.8, 2, 1, 1, 32, 1), (20, 600, 1.0, 2, 2, 3, 256, 2)]
NODE = np.dtype([("key", np.uint32), ("pad", np.uint32), ("re", np.float64), ("im", np.float64)])
CAP = 524288


class _Setup:
    """two sets of signals and draws of one batch on a stream of the caller's, and their results"""

    def __init__(self, precision, graph):
        import torch
        import sfft_amd as S
        self.S, self.torch = S, torch
        cdt = np.complex64 if precision == "fp32" else np.complex128
        prms = [params(c) for c in CONFIGS]
        prms.append(dict(prms[0], B=64, w=64 * 40 + 7, B_thresh=20))   # the slab does not take it
        self.count = len(prms)
        arr = (S._lib.Params * self.count)(*[S.core._cparams(p, 0, 0, "auto") for p in prms])
        handle = C.c_void_p()
        assert C.CDLL("libamdhip64.so").hipStreamCreateWithFlags(C.byref(handle), 1) == 0
        self.stream = torch.cuda.ExternalStream(handle.value)
        self.b = C.c_void_p()
        assert S.lib.sfft_batch_create(arr, self.count, 1 if precision == "fp32" else 0,
                                       C.c_void_p(self.stream.cuda_stream), C.byref(self.b)) == 0
        self.xs, self.dr, self.want, self.keep = [[], []], [[], []], [[], []], []
        rng = np.random.default_rng(12)
        for i, p in enumerate(prms):
            if i < len(CONFIGS):
                ft, ff = oracle_filter(p)
                win = np.ascontiguousarray(O.filter_window_slice(ff, p["n"], p["B"]))
            else:
                ft = rng.standard_normal(p["w"]) + 1j * rng.standard_normal(p["w"])
                win = 1.0 + rng.random(p["n"] // p["B"]) + 0j
            ft = torch.from_numpy(ft.astype(cdt)).cuda()
            assert S.lib.sfft_batch_set_filter(self.b, i, C.c_void_p(ft.data_ptr()),
                                               win.ctypes.data_as(C.c_void_p)) == 0
            plan = S.Plan(p, precision)
            plan.set_filter(ft, win)
            self.keep += [ft, win]
            for s in range(2):
                x, _, _ = sparse_signal(p["n"], p["k"], 200 + 10 * s + i, snr_db=30.0)
                x = torch.from_numpy(x.astype(cdt)).cuda()
                d = draws(p["n"], p["loops"], p["RLFC_loops"], p["W_RLFC"], 300 + 10 * s + i)
                d = tuple(np.ascontiguousarray(v, dtype=np.int32) for v in d)
                self.xs[s].append(x)
                self.dr[s].append(d)
                self.want[s].append(plan.execute(x, *d))
        assert S.lib.sfft_batch_set_graph(self.b, int(graph)) == 0
        torch.cuda.synchronize()

    def args(self, s):
        ptrs = (C.c_void_p * self.count)(*[x.data_ptr() for x in self.xs[s]])
        dr = (self.S._lib.Draws * self.count)(
            *[self.S._lib.Draws(*[v.ctypes.data for v in d]) for d in self.dr[s]])
        return ptrs, dr

    def enqueue(self, s):
        ptrs, dr = self.args(s)
        assert self.S.lib.sfft_batch_execute_async(self.b, ptrs, dr) == 0

    def execute(self, s, addr):
        ptrs, dr = self.args(s)
        counts = np.zeros(self.count, np.int32)
        assert self.S.lib.sfft_batch_execute(self.b, ptrs, dr, addr,
                                             counts.ctypes.data_as(C.c_void_p)) == 0
        return counts

    def check_device(self, s):
        """the plans' node buffers hold set s"""
        self.torch.cuda.synchronize()
        hip = C.CDLL("libamdhip64.so")
        counts = np.empty(self.count, np.int32)
        dev = self.S.lib.sfft_batch_counts_device(self.b)
        assert hip.hipMemcpy(counts.ctypes.data_as(C.c_void_p), C.cast(dev, C.c_void_p),
                             C.c_size_t(counts.nbytes), 2) == 0
        for i, (nodes, cnt) in enumerate(self.want[s]):
            assert counts[i] == cnt
            got = np.empty(cnt, NODE)
            src = self.S.lib.sfft_plan_debug_buffer(self.S.lib.sfft_batch_plan(self.b, i), 5)
            assert hip.hipMemcpy(got.ctypes.data_as(C.c_void_p), C.c_void_p(src),
                                 C.c_size_t(got.nbytes), 2) == 0
            assert got.tobytes() == nodes.tobytes(), f"set {s} signal {i}"

    def close(self):
        self.S.lib.sfft_batch_destroy(self.b)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_batch_alternating_pointers(precision, graph):
    import torch
    t = _Setup(precision, graph)
    pinned = torch.zeros(t.count * CAP * 24, dtype=torch.uint8, pin_memory=True)
    addr = (C.c_void_p * t.count)(*[pinned.data_ptr() + i * CAP * 24 for i in range(t.count)])
    host = pinned.numpy().view(NODE).reshape(t.count, CAP)
    for last in (0, 1):
        for s in [0, 1, 1, 0, 1 - last, last]:   # queued: the last one's results
            t.enqueue(s)
        t.check_device(last)
        # pinned nodes in between, on the other set
        pinned.zero_()
        counts = t.execute(1 - last, addr)
        for i, (nodes, cnt) in enumerate(t.want[1 - last]):
            assert counts[i] == cnt and host[i][:cnt].tobytes() == nodes.tobytes()
            assert not host[i][cnt:cnt + 8].view(np.uint8).any()
        t.enqueue(last)
        t.check_device(last)
        # other launch shapes: other tables
        assert t.S.lib.sfft_batch_set_shape(t.b, 2, 128, 1024, 4, 8) == 0
        t.enqueue(1 - last)
        t.check_device(1 - last)
        assert t.S.lib.sfft_batch_set_shape(t.b, 3, 256, 2048, 0, 0) == 0
    t.close()


@pytest.mark.parametrize("graph", [False, True])
def test_batch_new_pointers_do_not_wait(graph):
    import torch
    t = _Setup("fp32", graph)
    t.enqueue(0)
    torch.cuda.synchronize()
    with torch.cuda.stream(t.stream):
        a = torch.randn(8192, 8192, device="cuda")
        out = torch.mm(a, a)
        torch.cuda.synchronize()
        for _ in range(40):                      # some hundred milliseconds of work in front
            torch.mm(a, a, out=out)
    t.enqueue(1)
    waited = t.stream.query()
    t.check_device(1)
    t.close()
    assert not waited
