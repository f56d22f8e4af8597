"""The comb FFT's keys in their storage order, and the cutoff's list behind the histogram that the
last pass counts, against the dense FFT of the same points and a sorted selection: combs of the
whole signal whose last pass has each tile shape (quarter, half-filled and full tiles)."""
import numpy as np
import pytest

from helpers import params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("front_end", ["columns", "gather"])
@pytest.mark.parametrize("log2W", [16, 17, 21, 23, 24])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_comb_keys_and_cutoff(precision, log2W, front_end):
    import torch
    import sfft_amd as S
    n = 1 << log2W
    cdt, kdt = (np.complex64, np.uint32) if precision == "fp32" else (np.complex128, np.uint64)
    B, K = 4096, 700
    prm = dict(params((18, 50, 1.0, 2, 2, 5, 32, 2)), n=n, q=log2W, B=B, w=B * 10 + 3, B_thresh=K,
               W_RLFC=n, RLFC_loops=1)
    rng = np.random.default_rng(log2W)
    x = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(cdt)
    x[1::2] = x[::2]                              # a spectrum with many ties
    dx = torch.from_numpy(x).cuda()
    taps = torch.from_numpy((rng.standard_normal(prm["w"]) + 0j).astype(cdt)).cuda()
    plan = S.Plan(prm, precision, front_end=front_end, hit_capacity=1 << 20)
    assert plan.front_end == front_end
    plan.set_filter(taps, np.ones(n // B, np.complex128))
    a = np.array([2 * int(v) + 1 for v in rng.integers(0, n // 2, prm["loops"])], np.int32)
    ai = np.array([pow(int(v), -1, n) for v in a], np.int32)
    buf = torch.zeros((1 << 20) * 24, dtype=torch.uint8, device="cuda")
    num = torch.zeros(1, dtype=torch.int32, device="cuda")
    plan.execute_async(dx, a, ai, np.zeros(1, np.int32), d_nodes=buf, d_count=num)
    torch.cuda.synchronize()
    X = S.fft(dx).cpu().numpy()
    want = (X.real * X.real + X.imag * X.imag).view(kdt)
    lo, mid = plan.comb_key_order()
    s = np.arange(n, dtype=np.int64)
    bins = s if mid == 0 else ((s & ((1 << lo) - 1)) | (((s >> lo) & ((1 << mid) - 1)) <<
                               (log2W - mid)) | ((s >> (lo + mid)) << lo))
    got = plan.debug_array(8, n, kdt)
    assert np.array_equal(got, want[bins])
    order = np.lexsort((np.arange(n), ~want))     # by key, larger first, then by index
    J2 = plan.debug_array(2, K, np.int32)
    assert np.array_equal(np.sort(J2), np.sort(order[:K]))
    plan.close()
