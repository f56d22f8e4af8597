"""The one-workgroup cutoff of short segments (sel_block_kernel) against the oracle: the edges of
its elements per thread, its LDS candidate list and its narrowing on tied and flat keys, in
FP64 through samples_indices and in FP32 and for the comb through whole transforms."""
import numpy as np
import pytest

import oracle as O
from helpers import SMALL_CONFIGS, bits, draws, oracle_filter, params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import sfft_amd
    return sfft_amd


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _keys(kind, N, rng):
    if kind == "random":
        v = rng.standard_normal(N)
    elif kind == "flat":
        v = np.full(N, 0.75)
    elif kind == "close":      # one first and second digit, distinct keys below them
        v = 1.5 + rng.integers(0, 1 << 20, N) * 2.0 ** -50
    elif kind == "binade":     # one first digit, more candidates than the LDS list holds
        v = 1.0 + rng.random(N) * 2.0 ** -6
    else:                      # infinities, zeros and the smallest numbers among them
        v = rng.choice([0.0, np.inf, 1e-170, 3e-162, 1.0, 2.0 ** 100, 1e155], N)
    return v.astype(np.complex128)


@pytest.mark.parametrize("kind", ["random", "flat", "close", "binade", "extremes"])
@pytest.mark.parametrize("N,K", [(2, 1), (63, 62), (8192, 2000), (8193, 8192), (16385, 37),
                                 (32767, 32766), (32768, 9000), (32769, 9000)])
def test_samples_indices_one_workgroup(S, kind, N, K):
    import ctypes as C
    import torch
    X = _keys(kind, N, np.random.default_rng(N + K))
    out = torch.zeros(K, dtype=torch.int32, device="cuda")
    t = C.c_double(0.0)
    dX = _dev(X)
    assert S.lib.samples_indices(C.c_void_p(dX.data_ptr()), K, N, C.c_void_p(out.data_ptr()),
                                 C.byref(t)) == 0
    assert np.array_equal(out.cpu().numpy(), O.cutoff64(O.samples64(X), K))


# comb lengths of one and of two FFT passes (natural and tiled key order), buckets and combs on
# both sides of the one-workgroup limit of 32768
CONFIGS = [SMALL_CONFIGS[0], SMALL_CONFIGS[3], (20, 600, 1.0, 2, 2, 3, 256, 2),
           (21, 5000, 2.4, 2, 2, 2, 512, 1)]


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("kind", ["noise", "zero", "constant", "integer"])
@pytest.mark.parametrize("cfg", CONFIGS, ids=lambda c: f"q{c[0]}k{c[1]}")
def test_transform_cutoffs(S, cfg, kind, fp32):
    prm = params(cfg)
    n, B, K, Rl, Ll = (prm[k] for k in ("n", "B", "B_thresh", "RLFC_loops", "loops_loc"))
    rng = np.random.default_rng(n + K)
    if kind == "zero":
        x = np.zeros(n, dtype=np.complex128)
    elif kind == "constant":
        x = np.ones(n, dtype=np.complex128)
    elif kind == "integer":
        x = (rng.integers(-2, 3, n) + 1j * rng.integers(-2, 3, n)).astype(np.complex128)
    else:
        x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    ft, ff = oracle_filter(prm)
    win = O.filter_window_slice(ff, n, B)
    a, ai, offs = draws(n, prm["loops"], Rl, prm["W_RLFC"], 21)
    if fp32:
        x, ft = x.astype(np.complex64), ft.astype(np.complex64)
    loop = O.outer_loop32 if fp32 else O.outer_loop64
    ref = loop(prm, x, ft, win, a, ai, offs, want_bins=True, want_J=True)
    plan = S.Plan(prm, "fp32" if fp32 else "fp64")
    plan.set_filter(_dev(ft), win)
    nodes, cnt = plan.execute(_dev(x), a, ai, offs)
    assert np.array_equal(np.unique(plan.debug_array(2, Rl * K, np.int32)), ref["J2"])
    assert np.array_equal(plan.debug_array(1, Ll * K, np.int32).reshape(Ll, K), ref["J"])
    assert cnt == ref["I_F"]
    assert np.array_equal(nodes["key"], ref["nodes"]["key"])
    for f in ("re", "im"):
        assert np.array_equal(bits(nodes[f]), bits(ref["nodes"][f]))
