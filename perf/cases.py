"""The work this library does for its users, as cases that can be timed and compared.

Six kinds, each through the library's public entry points:

* transform  one sparse FFT of a device-resident signal: every size from the smallest
             configurations of the test suite to n = 2^27, both precisions, noiseless and noisy.
             Three ways to call it: "host" is a serving program on the C interface
             (sfft_execute, the nodes in its own pinned memory, the transform replayed from a
             hipGraph or enqueued eagerly), "device" a pipeline whose results stay on the GPU
             (Plan.execute_async), "spectrum" an analysis script (Plan.execute with its
             defaults, the nodes put into a dense spectrum)
* batch      many signals of uneven n and k transformed together (sfft_batch_execute)
* gradient   one training step of the differentiable transform: forward and backward of
             sparse_fft
* design     the filter of a new (n, k), on the device (make_filter, mode "parallel")
* truth      the dense reference spectrum that accuracy checks compare with (truth_spectrum)
* fft        the canonical dense FFT the library exports (fft)

A transform's located indices include false positives that depend on rounding at the noise
floor of the comb spectrum, so transforms, batches and gradients have no value that 64-bit
arithmetic alone determines; the filter design and the dense FFTs have one (exact).
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "gpu-sfft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import sfft_amd as S  # noqa: E402

LINE = 128              # bytes of memory a random 8- or 16-byte read moves on this card
NODE = 24               # bytes of a Node: the index, 4 bytes of padding, two doubles
MAX_HITS = 400000       # expected located indices of a drawn case (a plan's capacity: 524288)


def _transform(name, cfg, precision, snr=0.0, call="host", graph=True):
    q, k, Bcst, ll, lt, le, rc, rl = cfg
    return dict(name=name, kind="transform", q=q, k=k, Bcst=Bcst, loops_loc=ll, loops_thresh=lt,
                loops_est=le, RLFC_cst=rc, RLFC_loops=rl, precision=precision, snr_db=snr,
                call=call, graph=graph)


def listed():
    return [
        # a short record analysed once: the test suite's small configuration, eager, where
        # launches and latency are the whole cost
        _transform("n14_k20_fp64", (14, 20, 1.0, 2, 2, 5, 4, 2), "fp64", call="spectrum",
                   graph=False),
        # the mid-size configuration of the benchmark: served, and in a device pipeline
        _transform("n20_k1000_fp64", (20, 1000, 1.40, 2, 2, 5, 128, 2), "fp64"),
        _transform("n20_k1000_fp32", (20, 1000, 1.40, 2, 2, 5, 128, 2), "fp32", call="device",
                   graph=False),
        # an ordinary recording of 16 M samples with noise and an odd k
        _transform("n24_k2503_40db_fp32", (24, 2503, 1.0, 2, 2, 5, 256, 2), "fp32", snr=40.0),
        # the reference README's run, the benchmark's default workload
        _transform("n27_k16000_fp64", (27, 16000, 0.65, 2, 2, 7, 4096, 2), "fp64"),
        _transform("n27_k16000_fp32", (27, 16000, 0.65, 2, 2, 7, 4096, 2), "fp32"),
        # the benchmark's dense and noisy workload: three location loops, a 2^24-point comb
        _transform("n27_k40000_30db_fp32", (27, 40000, 0.7, 3, 2, 8, 32768, 2), "fp32",
                   snr=30.0),
        # the benchmark's batch of 64 uneven complex64 signals
        dict(name="batch64_fp32", kind="batch", count=64, q_lo=18, q_hi=24, k_lo=50, k_hi=4000,
             workload=0x5FF70002, precision="fp32", snr_db=40.0, graph=True),
        # a training step at the differentiable-path workload
        dict(name="grad_n22_k1000", kind="gradient", q=22, k=1000, Bcst=0.99, loops_loc=2,
             loops_thresh=2, loops_est=5, RLFC_cst=256, RLFC_loops=2),
        # a program that meets a new signal length designs its filter first
        dict(name="design_n22", kind="design", q=22, k=1000, Bcst=0.99),
        # the check of a transform's accuracy: the dense spectrum of its complex64 signal
        dict(name="truth_n22_fp32", kind="truth", q=22, k=1000, precision="fp32"),
        # dense spectra of many complex64 records
        dict(name="fft_2p20_x12_fp32", kind="fft", log2n=20, count=12, precision="fp32",
             inverse=False),
    ]


# the parameter sets a drawn transform takes for its size: (smallest q, largest q, Bcst,
# loops_loc, loops_thresh, loops_est, RLFC_cst, RLFC_loops), from the repository's configurations
_SETS = [
    (12, 15, 1.0, 2, 2, 5, 4, 2),
    (14, 17, 1.0, 3, 2, 4, 16, 2),
    (16, 18, 0.8, 2, 1, 3, 32, 1),
    (17, 22, 1.40, 2, 2, 5, 128, 2),
    (18, 25, 1.0, 2, 2, 5, 256, 2),
    (25, 27, 0.65, 2, 2, 7, 4096, 2),
]


def _expected_hits(p):
    """Located indices to expect: true ones, and false ones that pass the voting."""
    K = p["B_thresh"]
    t = p["loops_thresh"]
    ways = math.comb(p["loops_loc"], t)
    return p["k"] + ways * p["n"] * (K / p["B"]) ** t * min(1.0, p["RLFC_loops"] * K / p["W_RLFC"])


def _draw_k(rng, q, lo, hi, tail, rest):
    """A k, log-uniform and usually odd, whose parameters are valid; None if none was found."""
    for _ in range(60):
        k = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        p = S.derive_params(q, max(k, 2), *tail, *rest)
        if p["assert_ok"] and S.validate(p) == 0 and _expected_hits(p) < MAX_HITS:
            return p["k"]
    return None


def draw(rng):
    kind = rng.choice(["transform"] * 5 + ["batch", "gradient", "design", "truth", "fft", "fft"])
    if kind == "transform":
        while True:
            q = rng.randint(12, 27)
            sets = [s for s in _SETS if s[0] <= q <= s[1]]
            _, _, Bcst, ll, lt, le, rc, rl = rng.choice(sets)
            hi = max(9, min(16000, (1 << q) // 400))
            k = _draw_k(rng, q, 8, hi, (Bcst,), (ll, lt, le, rc, rl))
            if k is not None:
                call = rng.choice(["host", "host", "device", "spectrum" if q < 16 else "device"])
                c = _transform("", (q, k, Bcst, ll, lt, le, rc, rl),
                               rng.choice(["fp64", "fp32"]),
                               snr=rng.choice([0.0, 0.0, 30.0, 40.0]), call=call,
                               graph=rng.random() < 0.6)
                del c["name"]
                return c
    if kind == "batch":
        lo = rng.randint(18, 21)
        return dict(kind="batch", count=rng.randint(3, 48), q_lo=lo,
                    q_hi=rng.randint(lo, 23), k_lo=50, k_hi=rng.choice([400, 1000, 4000]),
                    workload=rng.randint(1, 1 << 30), precision=rng.choice(["fp32", "fp64"]),
                    snr_db=rng.choice([0.0, 40.0]), graph=rng.random() < 0.6)
    if kind == "gradient":
        while True:
            q = rng.randint(14, 23)
            k = _draw_k(rng, q, 8, max(9, min(2000, (1 << q) // 1000)), (0.99,),
                        (2, 2, 5, 256 if q >= 18 else 16, 2))
            if k is not None:
                return dict(kind="gradient", q=q, k=k, Bcst=0.99, loops_loc=2, loops_thresh=2,
                            loops_est=5, RLFC_cst=256 if q >= 18 else 16, RLFC_loops=2)
    if kind == "design":
        while True:
            q = rng.randint(12, 24)
            k = _draw_k(rng, q, 8, max(9, (1 << q) // 1000), (1.0,), (2, 2, 5, 16, 2))
            if k is not None:
                return dict(kind="design", q=q, k=k, Bcst=1.0)
    if kind == "truth":
        q = rng.randint(12, 24)
        return dict(kind="truth", q=q, k=rng.randint(8, max(9, (1 << q) // 1000)),
                    precision=rng.choice(["fp32", "fp64"]))
    precision = rng.choice(["fp32", "fp64"])
    log2n = rng.randint(4, 24)
    total = 1 << rng.randint(max(10, log2n), 24)
    return dict(kind="fft", log2n=log2n,
                count=max(1, (total >> log2n) - rng.randint(0, max(0, (total >> log2n) // 3))),
                precision=precision, inverse=rng.random() < 0.5)


# ---- parameters, inputs -----------------------------------------------------------------------
def _params(c):
    if c["kind"] == "design":
        return S.derive_params(c["q"], c["k"], c["Bcst"], 2, 2, 5, 16, 2)
    return S.derive_params(c["q"], c["k"], c["Bcst"], c["loops_loc"], c["loops_thresh"],
                           c["loops_est"], c["RLFC_cst"], c["RLFC_loops"])


def _batch_params(c):
    return S.batch_workload(c["count"], c["workload"], (c["q_lo"], c["q_hi"]),
                            (c["k_lo"], c["k_hi"]))


def _filter(p, fp32):
    ft, ff = S.make_filter(p["lobefrac"], p["tolerance"], p["n"], p["b_f"], p["w"],
                           mode="parallel", freq="device")
    win = S.filter_window(ff, p["n"], p["B"])
    return (S.to_complex64(ft) if fp32 else ft), win


def _signal(n, k, seed, snr_db, fp32):
    locs, vals = S.signal_spectrum(n, k, seed)
    return S.synthesize(n, k, locs, vals, snr_db=snr_db, noise_seed=seed + 1, fp32=fp32)


def _draws(p, seed):
    return S.draw_permutations(p["n"], p["loops"], p["RLFC_loops"], p["W_RLFC"], seed + 2)


# the C interface (include/sfft.h) as a program that links libsfft.so uses it
class _Params(C.Structure):
    _fields_ = [(f, C.c_int) for f in
                ("n", "B", "B_thresh", "W_RLFC", "RLFC_loops", "loops_thresh", "loops_loc",
                 "loops", "w", "fold_mode", "hit_capacity", "front_end")]

    @classmethod
    def of(cls, p, capacity):
        return cls(p["n"], p["B"], p["B_thresh"], p["W_RLFC"], p["RLFC_loops"],
                   p["loops_thresh"], p["loops_loc"], p["loops"], p["w"], 0, capacity, 0)


class _Draws(C.Structure):
    _fields_ = [("a", C.c_void_p), ("ai", C.c_void_p), ("offsets", C.c_void_p)]


_lib = C.CDLL(S.LIB_PATH)
_VP = C.c_void_p
_lib.sfft_plan_create.argtypes = [C.POINTER(_Params), C.c_int, _VP, C.POINTER(_VP)]
_lib.sfft_plan_set_filter.argtypes = [_VP, _VP, _VP]
_lib.sfft_plan_set_graph.argtypes = [_VP, C.c_int]
_lib.sfft_plan_destroy.argtypes = [_VP]
_lib.sfft_execute.argtypes = [_VP, _VP, C.POINTER(_Draws), _VP, C.POINTER(C.c_int)]
_lib.sfft_batch_create.argtypes = [C.POINTER(_Params), C.c_int, C.c_int, _VP, C.POINTER(_VP)]
_lib.sfft_batch_set_filter.argtypes = [_VP, C.c_int, _VP, _VP]
_lib.sfft_batch_set_graph.argtypes = [_VP, C.c_int]
_lib.sfft_batch_destroy.argtypes = [_VP]
_lib.sfft_batch_execute.argtypes = [_VP, _VP, C.POINTER(_Draws), _VP, _VP]


def _ok(status):
    if status:
        raise RuntimeError("libsfft: status %d" % status)


class _Handle:
    """A plan or batch of the C interface, destroyed with its owner."""

    def __init__(self, destroy):
        self.h, self.destroy = _VP(), destroy

    def __del__(self):
        if self.h:
            self.destroy(self.h)


def _capacity(p):
    """Room for the located indices: twice what is expected, as a program that serves one
    workload would reserve."""
    return min(524288, 4096 + 2 * int(_expected_hits(p)))


def _node_views(buf, count):
    """The fields of Node[] in a byte buffer, as views; entries past the count stay zero."""
    words = buf.view(torch.float64).view(-1, 3)
    return {"key": buf.view(torch.int32).view(-1, 6)[:, 0], "re": words[:, 1], "im": words[:, 2],
            "count": count}


def _prepare_transform(case, seed):
    p, fp32 = _params(case), case["precision"] == "fp32"
    x = _signal(p["n"], p["k"], seed, case["snr_db"], fp32)
    ft, win = _filter(p, fp32)
    draws = _draws(p, seed)
    s = dict(kind="transform", call=case["call"], x=x, ft=ft, draws=draws)
    cap = _capacity(p)
    if case["call"] == "host":
        plan = s["plan"] = _Handle(_lib.sfft_plan_destroy)
        _ok(_lib.sfft_plan_create(C.byref(_Params.of(p, cap)), int(fp32),
                                  torch.cuda.current_stream().cuda_stream, C.byref(plan.h)))
        _ok(_lib.sfft_plan_set_filter(plan.h, ft.data_ptr(), win.ctypes.data))
        _ok(_lib.sfft_plan_set_graph(plan.h, int(case["graph"])))
        s["cdraws"] = _Draws(*(d.ctypes.data for d in draws))
        s["nodes"] = torch.zeros(cap * NODE, dtype=torch.uint8, pin_memory=True)
        s["count"] = np.zeros(1, dtype=np.int32)
        s["out"] = _node_views(s["nodes"], s["count"])
        return s
    s["plan"] = plan = S.Plan(p, case["precision"], hit_capacity=cap)
    plan.set_filter(ft, win)
    plan.set_graph(case["graph"])
    if case["call"] == "device":
        s["nodes"] = torch.zeros(cap * NODE, dtype=torch.uint8, device="cuda")
        s["count"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["out"] = _node_views(s["nodes"], s["count"])
    else:
        s["spectrum"] = np.zeros(p["n"], dtype=np.complex128)
    return s


def _prepare_batch(case, seed):
    ps, fp32 = _batch_params(case), case["precision"] == "fp32"
    n = len(ps)
    caps = [_capacity(p) for p in ps]
    batch = _Handle(_lib.sfft_batch_destroy)
    _ok(_lib.sfft_batch_create((_Params * n)(*[_Params.of(p, c) for p, c in zip(ps, caps)]), n,
                               int(fp32), None, C.byref(batch.h)))
    xs, draws, filters = [], [], []
    for i, p in enumerate(ps):
        xs.append(_signal(p["n"], p["k"], seed + 97 * i, case["snr_db"], fp32))
        draws.append(_draws(p, seed + 97 * i))
        ft, win = _filter(p, fp32)
        _ok(_lib.sfft_batch_set_filter(batch.h, i, ft.data_ptr(), win.ctypes.data))
        filters.append(ft)
    _ok(_lib.sfft_batch_set_graph(batch.h, int(case["graph"])))
    nodes = torch.zeros(sum(caps) * NODE, dtype=torch.uint8, pin_memory=True)
    at = np.concatenate([[0], np.cumsum(caps)[:-1]]) * NODE + nodes.data_ptr()
    count = np.zeros(n, dtype=np.int32)
    return dict(kind="batch", batch=batch, xs=xs, filters=filters, draws=draws, nodes=nodes,
                cxs=(_VP * n)(*[x.data_ptr() for x in xs]),
                cdraws=(_Draws * n)(*[_Draws(*(d.ctypes.data for d in dr)) for dr in draws]),
                cnodes=(_VP * n)(*[int(v) for v in at]), count=count,
                out=_node_views(nodes, count))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "transform":
        return _prepare_transform(case, seed)
    if kind == "batch":
        return _prepare_batch(case, seed)
    if kind == "gradient":
        p = _params(case)
        plan = S.Plan(p, "fp64")
        plan.set_filter(*_filter(p, False))
        x = _signal(p["n"], p["k"], seed, 0.0, False)
        g = torch.Generator(device="cuda").manual_seed(seed)
        weight = torch.rand(p["n"], dtype=torch.float64, device="cuda", generator=g)
        return dict(kind=kind, plan=plan, x=x, draws=_draws(p, seed), weight=weight)
    if kind == "design":   # a passband to try: the boxcar's width, a little wider each time
        p = _params(case)
        return dict(kind=kind, p=p, b_f=p["b_f"] + seed % 64)
    if kind == "truth":
        return dict(kind=kind, x=_signal(1 << case["q"], case["k"], seed, 40.0,
                                         case["precision"] == "fp32"))
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["count"], 1 << case["log2n"])
    re, im = (torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
              for _ in range(2))
    x = torch.complex(re, im)
    if case["precision"] == "fp32":
        x = x.to(torch.complex64)
    return dict(kind=kind, x=x, inverse=case["inverse"])


def run(s):
    kind = s["kind"]
    if kind == "transform":
        if s["call"] == "host":
            _ok(_lib.sfft_execute(s["plan"].h, s["x"].data_ptr(), C.byref(s["cdraws"]),
                                  s["nodes"].data_ptr(),
                                  s["count"].ctypes.data_as(C.POINTER(C.c_int))))
            return s["out"]
        if s["call"] == "device":
            s["plan"].execute_async(s["x"], *s["draws"], d_nodes=s["nodes"], d_count=s["count"])
            return s["out"]
        nodes, _ = s["plan"].execute(s["x"], *s["draws"])
        s["spectrum"][nodes["key"]] = nodes["re"] + 1j * nodes["im"]
        return s["spectrum"]
    if kind == "batch":
        _ok(_lib.sfft_batch_execute(s["batch"].h, s["cxs"], s["cdraws"], s["cnodes"],
                                    s["count"].ctypes.data))
        return s["out"]
    if kind == "gradient":
        x = s["x"].detach().requires_grad_(True)
        vals, keys = S.sparse_fft(x, s["plan"], *s["draws"])
        loss = (s["weight"][keys] * (vals.real ** 2 + vals.imag ** 2)).sum()
        loss.backward()
        return {"loss": loss.detach(), "grad": x.grad}
    if kind == "design":
        p = s["p"]
        taps, resp = S.make_filter(p["lobefrac"], p["tolerance"], p["n"], s["b_f"], p["w"],
                                   mode="parallel", freq="device")
        return {"taps": taps, "response": resp}
    if kind == "truth":
        return S.truth_spectrum(s["x"])
    return S.fft(s["x"], inverse=s["inverse"])


# ---- what a pass cannot do without ------------------------------------------------------------
def _fft_flops(n):
    return 5.0 * n * math.log2(max(n, 2))


def _transform_work(p, fp32):
    """The signal's used samples (a random sample moves its whole line, at most the whole signal
    is read), the filter once, about k nodes; the fold and the FFTs of the buckets and combs."""
    e = 8 if fp32 else 16
    L, w, Rl, W, n = p["loops"], p["w"], p["RLFC_loops"], p["W_RLFC"], p["n"]
    samples = L * w + Rl * W
    return (min(n * e, samples * LINE) + w * e + 24.0 * p["k"],
            8.0 * L * w + L * _fft_flops(p["B"]) + Rl * _fft_flops(W))


def work(case):
    kind = case["kind"]
    if kind == "transform":
        b, f = _transform_work(_params(case), case["precision"] == "fp32")
    elif kind == "batch":
        parts = [_transform_work(p, case["precision"] == "fp32") for p in _batch_params(case)]
        b, f = sum(v[0] for v in parts), sum(v[1] for v in parts)
    elif kind == "gradient":   # the forward transform; the whole gradient written
        p = _params(case)
        b, f = _transform_work(p, False)
        b += 16.0 * p["n"] + 16.0 * p["w"]
        f += 8.0 * p["loops"] * p["w"] + p["loops"] * _fft_flops(p["B"])
    elif kind == "design":     # the response and the taps written; an FFT of w and two of n
        p = _params(case)
        b = 16.0 * (p["n"] + p["w"])
        f = 2 * _fft_flops(p["n"]) + _fft_flops(p["w"])
    elif kind == "truth":
        n = 1 << case["q"]
        b, f = n * (16.0 + (8 if case["precision"] == "fp32" else 16)), _fft_flops(n)
    else:
        n, cnt = 1 << case["log2n"], case["count"]
        b = 2.0 * n * cnt * (8 if case["precision"] == "fp32" else 16)
        f = cnt * _fft_flops(n)
    return {"bytes": b, "flops": f}


# ---- values in 64 bits, where a case has them ---------------------------------------------------
def _design_exact(p, b_f, tol=1e-8):
    """The Dolph-Chebyshev boxcar filter: Chebyshev samples without the direct form's
    cancellation, their DFT, the fold, the boxcar from an extended-precision prefix sum, the
    phase ramp with its angle reduced in integers, and the taps from the inverse transform."""
    n, w = p["n"], p["w"]
    m = w - 1
    a = np.arccosh(1 / tol) / m
    t0, t0m1 = np.cosh(a), 2 * np.sinh(a / 2) ** 2
    half = np.pi * np.arange(w) / (2 * w)
    d = t0m1 - 2 * t0 * np.sin(half) ** 2
    xp1 = 2 * t0 * np.cos(half) ** 2 - t0m1
    s = np.zeros(w)
    up, mid, low = d > 0, (d <= 0) & (d >= -1), (d < -1) & (xp1 >= 0)
    s[up] = np.cosh(m * np.log1p(d[up] + np.sqrt(d[up] * (2 + d[up]))))
    s[mid] = np.cos(2 * m * np.arcsin(np.sqrt(-d[mid] / 2)))
    s[low] = np.cos(m * (np.pi - 2 * np.arcsin(np.sqrt(xp1[low] / 2))))
    shifted = np.roll(np.fft.fft((s * tol).astype(np.complex128)).real, w // 2)
    h = w // 2
    g = np.zeros(n, dtype=np.complex128)
    g[:h] = shifted[h:2 * h]
    g[n - h:] = shifted[:h]
    G = np.fft.fft(g)
    cs = np.concatenate([np.zeros(1, np.clongdouble),
                         np.cumsum(np.concatenate([G, G[:b_f]]).astype(np.clongdouble))])
    idx = np.arange(n)
    box = np.empty(n, dtype=np.clongdouble)
    box[(idx + b_f // 2) % n] = cs[idx + b_f] - cs[idx]
    box /= np.max(np.abs(box))
    ang = (-2 * np.pi) * (((np.int64(h) * idx.astype(np.int64)) % n).astype(np.longdouble) / n)
    ff = (box * (np.cos(ang) + 1j * np.sin(ang))).astype(np.complex128)
    return {"taps": np.fft.ifft(ff)[:w], "response": ff}


def exact(case, seed):
    kind = case["kind"]
    if kind == "design":
        s = prepare(case, seed)
        return _design_exact(s["p"], s["b_f"])
    if kind in ("truth", "fft"):
        s = prepare(case, seed)
        x = s["x"].to(torch.complex128).cpu()
        n = x.shape[-1]
        if kind == "truth":
            return torch.fft.fft(x) / n
        return torch.fft.ifft(x) * n if s["inverse"] else torch.fft.fft(x)
    return None
