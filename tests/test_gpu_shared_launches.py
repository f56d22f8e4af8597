"""Short transforms take the column front end and share the launches of their comb and bucket stages
(counted in a capture of one transform), and give the bits of a launch per stage and of the gathering
front end; where the hits exceed the capacity, every path reports the same count and stores the same
first nodes.  No other status is accepted."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from helpers import N20_K1000, SMALL_CONFIGS, draws, oracle_filter, params, sparse_signal

pytestmark = pytest.mark.gpu

OVERFLOW = 4
# combs and buckets of up to 32768 points whose FFTs take quarter tiles
SHORT = [SMALL_CONFIGS[1], (15, 30, 1.0, 2, 2, 5, 4, 2),
         (17, 100, 1.0, 2, 2, 5, 64, 2), N20_K1000]
B2048 = (18, 300, 1.40, 2, 2, 5, 32, 2)      # FP64: a bucket FFT is a full tile
LONG = (21, 1000, 1.0, 2, 2, 5, 256, 2)      # a comb above that
MANY_LOOPS = (14, 20, 1.0, 4, 3, 15, 8, 3)   # the slab does not take it: gathers


class _Run:
    def __init__(self, cfg, precision, kind):
        import torch
        import sfft_amd as S
        self.S, self.torch, self.precision = S, torch, precision
        self.prm = prm = params(cfg)
        n = prm["n"]
        cdt = np.complex64 if precision == "fp32" else np.complex128
        x, _, _ = sparse_signal(n, prm["k"], 5, snr_db=30.0)
        if kind == "zero":
            x = np.zeros_like(x)
        ft, ff = oracle_filter(prm)
        self.dx = torch.from_numpy(x.astype(cdt)).cuda()
        self.dft = torch.from_numpy(ft.astype(cdt)).cuda()
        self.win = O.filter_window_slice(ff, n, prm["B"])
        self.draws = tuple(np.ascontiguousarray(v, np.int32) for v in draws(
            n, prm["loops"], prm["RLFC_loops"], prm["W_RLFC"], 17))

    def plan(self, front_end="auto", capacity=0, stream=None):
        p = self.S.Plan(self.prm, self.precision, front_end=front_end, hit_capacity=capacity,
                        stream=stream)
        p.set_filter(self.dft, self.win)
        return p

    def execute(self, plan):
        """status, count, nodes (at most the capacity)"""
        self.torch.cuda.synchronize()
        nodes = np.zeros(plan.capacity, self.S.NODE_DTYPE)
        cnt = C.c_int(-1)
        dr = plan._draws(*self.draws)
        st = self.S.lib.sfft_execute(plan._h, C.c_void_p(self.dx.data_ptr()), C.byref(dr),
                                     nodes.ctypes.data_as(C.c_void_p), C.byref(cnt))
        assert st == (OVERFLOW if cnt.value > plan.capacity else 0), st
        if st:   # the nodes the plan stored (the call copies none)
            nodes = plan.debug_array(5, plan.capacity, self.S.NODE_DTYPE)
        return st, cnt.value, nodes[:min(cnt.value, plan.capacity)].tobytes()

    def launches(self):
        """kernel launches and events of one captured transform"""
        hip = C.CDLL("libamdhip64.so")
        st = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        plan = self.plan(stream=self.torch.cuda.ExternalStream(st.value))
        self.torch.cuda.synchronize()
        g, num = C.c_void_p(), C.c_size_t()
        assert hip.hipStreamBeginCapture(st, 1) == 0
        plan.execute_async(self.dx, *self.draws)
        assert hip.hipStreamEndCapture(st, C.byref(g)) == 0
        assert hip.hipGraphGetNodes(g, None, C.byref(num)) == 0
        hip.hipGraphDestroy(g)
        plan.close()
        hip.hipStreamDestroy(st)
        return num.value


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_short_transforms_share_launches(precision):
    got = {}
    for cfg in SHORT + [B2048, LONG, MANY_LOOPS]:
        r = _Run(cfg, precision, "noise")
        # fold, two FFT passes, cutoffs, nodes (and the walk, where it is long)
        got[cfg] = (r.plan().front_end, r.launches() <= 6)
    want = {cfg: ("columns", True) for cfg in SHORT}
    want.update({B2048: ("columns", precision == "fp32"), LONG: ("columns", False),
                 MANY_LOOPS: ("gather", False)})
    assert got == want


@pytest.mark.parametrize("kind", ["noise", "zero"])
@pytest.mark.parametrize("cfg", SHORT + [B2048, LONG, MANY_LOOPS], ids=lambda c: "q%d_k%d_l%d" % (c[0], c[1], c[3] + c[5]))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_paths_agree_with_and_without_overflow(precision, cfg, kind):
    r = _Run(cfg, precision, kind)
    want = r.execute(r.plan("gather"))
    assert want[1] > 0 or kind == "zero"
    caps = [0] + ([max(1, want[1] // 2)] if want[1] > 1 else [])
    for cap in caps:
        ref = r.execute(r.plan("gather", cap))
        assert ref[0] == (OVERFLOW if cap else want[0])
        assert ref[1] == want[1]
        if cap and want[0] == 0:
            assert ref[2] == want[2][:cap * r.S.NODE_DTYPE.itemsize]
        for profiled in (False, True):
            plan = r.plan("auto", cap)
            plan.set_profiling(profiled)
            for _ in range(2):
                assert r.execute(plan) == ref, (cap, profiled)
