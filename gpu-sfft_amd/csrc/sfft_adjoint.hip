// sfft_adjoint.hip -- the estimated values as a function of the signal, and its adjoint.
//
// With the located indices and the median-selected loops of a transform held fixed, each
// estimated value is a real-linear function of the signal (the permute+filter fold, the
// bucket FFT, the filter division of innerLoop.cu:396-466 / :725-773):
//   yhat_h = Re v_{sel[2h]}(I_h) + i Im v_{sel[2h+1]}(I_h)
// value_pick evaluates it from bucket spectra; the adjoint maps g_h = dL/dRe yhat_h +
// i dL/dIm yhat_h back to dL/dRe x + i dL/dIm x in three steps:
//   1. seeds: every (hit, part) entry adds (gr F.x/d, gr F.y/d) (real part) or
//      (-gi F.y/d, gi F.x/d) (imaginary part) to its bucket; entries of one bucket are summed
//      in entry order, so the result does not depend on thread timing;
//   2. the unnormalised inverse FFT of each loop's seed row (the transpose of FFT_B), run by
//      the caller with the canonical FFT kernels;
//   3. taps: gx[(i ai_l) mod n] += conj(f[i]) gb[l][bucket(i)], one loop after the other, the
//      tiled taps (or all taps) of a loop first, then the reference fold's tail taps.  A thread
//      owns a signal index and looks its taps up (i = m a_l mod n), or, where they are few, a
//      launch owns the taps of one loop, which have different indices: no atomics are needed.
// The library is built with -ffp-contract=off: the arithmetic below is exactly the oracle's.
#include <type_traits>

#include "sfft_internal.h"

namespace sfft {

// bucket and filter response of location I in loop l (innerLoop.cu:837-848)
__device__ __forceinline__ void est_term(uint32_t I, int l, uint32_t n, const int* ai_dev,
                                         int B, const double2* win, long long* hashed_out,
                                         double2* F_out) {
  const long long m = (long long)(n / (uint32_t)B);
  const long long nn = n;
  const long long p = (long long)(((uint64_t)(uint32_t)ai_dev[l] * I) & (uint64_t)(n - 1));
  long long hashed = p / m;
  long long dist = p & (m - 1);
  if (dist > m / 2) {
    hashed = (hashed + 1) & (B - 1);
    dist -= m;
  }
  dist = (nn - dist) & (nn - 1);
  *hashed_out = hashed;
  *F_out = win[(dist + m / 2) & (nn - 1)];
}

__global__ __launch_bounds__(256) void value_pick_kernel(
    const int* __restrict__ hits, int nh, const uint8_t* __restrict__ sel,
    const double2* __restrict__ bins_f, uint32_t n, const int* __restrict__ ai_dev, int B,
    const double2* __restrict__ win, double2* __restrict__ values) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= nh) return;
  const uint32_t I = (uint32_t)hits[h];
  const int lr = sel[2 * h], li = sel[2 * h + 1];
  long long hr, hi;
  double2 Fr, Fi;
  est_term(I, lr, n, ai_dev, B, win, &hr, &Fr);
  est_term(I, li, n, ai_dev, B, win, &hi, &Fi);
  const double2 br = bins_f[(long long)lr * B + hr];
  const double2 bi = bins_f[(long long)li * B + hi];
  double2 v;
  v.x = (br.x * Fr.x + br.y * Fr.y) / (Fr.x * Fr.x + Fr.y * Fr.y);
  v.y = (bi.y * Fi.x - bi.x * Fi.y) / (Fi.x * Fi.x + Fi.y * Fi.y);
  values[h] = v;
}

hipError_t value_pick_launch(const int* hits, int nh, const uint8_t* sel,
                             const double2* bins_f, int n, const int* ai_dev, int B,
                             const double2* win, double2* values, hipStream_t st) {
  if (nh <= 0) return hipSuccess;
  hipLaunchKernelGGL(value_pick_kernel, dim3((nh + 255) / 256), dim3(256), 0, st, hits, nh, sel,
                     bins_f, (uint32_t)n, ai_dev, B, win, values);
  return hipGetLastError();
}

// entry e = 2h + part -> bucket key l*B + hashed; per-key singly linked lists (any order)
__global__ __launch_bounds__(256) void adj_link_kernel(
    const int* __restrict__ hits, int nh, const uint8_t* __restrict__ sel, uint32_t n,
    const int* __restrict__ ai_dev, int B, const double2* __restrict__ win, int* head,
    int* __restrict__ next) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 2 * nh) return;
  const int l = sel[e];
  long long hb;
  double2 F;
  est_term((uint32_t)hits[e >> 1], l, n, ai_dev, B, win, &hb, &F);
  next[e] = atomicExch(&head[(long long)l * B + hb], e);
}

// one thread per bucket key: sum its entries in ascending entry order (repeated minimum
// search over the short list)
__global__ __launch_bounds__(256) void adj_sum_kernel(
    const int* __restrict__ hits, const uint8_t* __restrict__ sel,
    const double2* __restrict__ g, uint32_t n, const int* __restrict__ ai_dev, int B,
    int loops, const double2* __restrict__ win, const int* __restrict__ head,
    const int* __restrict__ next, double2* __restrict__ u) {
  const long long key = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (key >= (long long)loops * B) return;
  const int l = (int)(key / B);
  const int first = head[key];
  double2 acc = make_double2(0.0, 0.0);
  int cur = -1;
  while (first >= 0) {
    int best = 0x7fffffff;
    for (int e = first; e >= 0; e = next[e])
      if (e > cur && e < best) best = e;
    if (best == 0x7fffffff) break;
    long long hb;
    double2 F;
    est_term((uint32_t)hits[best >> 1], l, n, ai_dev, B, win, &hb, &F);
    const double d = F.x * F.x + F.y * F.y;
    const double2 gv = g[best >> 1];
    if ((best & 1) == 0) {
      const double q = gv.x / d;
      acc.x = acc.x + q * F.x;
      acc.y = acc.y + q * F.y;
    } else {
      const double q = gv.y / d;
      acc.x = acc.x - q * F.y;
      acc.y = acc.y + q * F.x;
    }
    cur = best;
  }
  u[key] = acc;
}

hipError_t adjoint_seed_launch(const int* hits, int nh, const uint8_t* sel, const double2* g,
                               int n, const int* ai_dev, int B, int loops, const double2* win,
                               int* head, int* next, double2* u, hipStream_t st) {
  const long long keys = (long long)loops * B;
  hipError_t e = fill_u32(head, 0xffffffffu, (size_t)keys, st);
  if (e != hipSuccess) return e;
  if (nh > 0) {
    hipLaunchKernelGGL(adj_link_kernel, dim3((2 * nh + 255) / 256), dim3(256), 0, st, hits, nh,
                       sel, (uint32_t)n, ai_dev, B, win, head, next);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  hipLaunchKernelGGL(adj_sum_kernel, dim3((unsigned)((keys + 255) / 256)), dim3(256), 0, st, hits,
                     sel, g, (uint32_t)n, ai_dev, B, loops, win, head, next, u);
  return hipGetLastError();
}

// gx[m] = sum of conj(f[id]) gb[l][bucket] over the taps id that read x[m]: loop l reads it at
// id = m * a_l mod n (a tap for id < head, bucket id mod B), and in the reference's tiled fold
// also as the tail tap id = i * tiles + B of bucket i < residue.  A thread owns signal index m
// and adds the loops' taps in order, so the gradient is written once, whole lines, in one
// launch: the taps' own order (adj_taps_kernel) reads and writes 16 bytes of a random line per tap
// and loop, after a clear of all n, in one launch per loop and phase (n = 2^22, 7 loops, w/n =
// 3.4 %: 79 us in 15 launches, 43 us in one).  Bound by the lookups' loads (64 lanes of 16 bytes each, tap or not);
// loading under a branch per loop waits for each load in turn and is slower.
// The loads of a chunk of loops go out together, a loop without a tap (or past the last loop)
// reading entry 0: chunks of AT_CHUNK, the last one of half as many where that is enough (HALF:
// a kernel of its own: as a run-time choice it cost 7 loops 590 us for 574; n = 2^26, 9 loops,
// w/n = 1.7 %: 878 -> 790 us).
constexpr int AT_CHUNK = 8;
typedef double d2v __attribute__((ext_vector_type(2)));
template <bool HALF>
__global__ __launch_bounds__(256) void adj_lookup_kernel(
    const double2* __restrict__ f, const double2* __restrict__ gb, const int* __restrict__ a_dev,
    int loops, uint32_t n, int B, uint32_t head, uint32_t residue, uint32_t tiles,
    uint32_t magic, double2* __restrict__ gx) {
  const d2v* __restrict__ fv = (const d2v*)f;
  const d2v* __restrict__ gv = (const d2v*)gb;
  const uint32_t mask = n - 1u, bmask = (uint32_t)B - 1u;
  const uint32_t m = blockIdx.x * 256u + threadIdx.x;
  if (m >= n) return;
  double ax = 0.0, ay = 0.0;
  auto add = [&](d2v t, d2v g) __attribute__((always_inline)) {
    ax = ax + fma(t.x, g.x, t.y * g.y);
    ay = ay + fma(t.x, g.y, -(t.y * g.x));
  };
  auto chunk = [&](int l0, auto size) __attribute__((always_inline)) {
    constexpr int CHUNK = decltype(size)::value;
    uint32_t id[CHUNK];
    d2v t[CHUNK], g[CHUNK];
#pragma unroll
    for (int j = 0; j < CHUNK; ++j) {
      const int l = min(l0 + j, loops - 1);
      id[j] = (m * (uint32_t)a_dev[l]) & mask;
      const uint32_t k = (l0 + j < loops && id[j] < head) ? id[j] : 0u;
      t[j] = fv[k];
      g[j] = gv[(size_t)l * (size_t)B + (k & bmask)];
    }
#pragma unroll
    for (int j = 0; j < CHUNK; ++j) {
      if (l0 + j < loops) {
        if (id[j] < head) add(t[j], g[j]);
        const uint32_t d = id[j] - (uint32_t)B;   // (wraps for id < B: past every tail tap)
        if (d < residue * tiles) {
          // i = d / tiles where tiles divides d (exact for those d: see the launch)
          const uint32_t i = tiles > 1u ? __umulhi(d, magic) : d;
          if (i * tiles == d) add(fv[id[j]], gv[(size_t)(l0 + j) * (size_t)B + i]);
        }
      }
    }
  };
  const int full = HALF ? loops / AT_CHUNK * AT_CHUNK : loops;
  for (int l0 = 0; l0 < full; l0 += AT_CHUNK) chunk(l0, std::integral_constant<int, AT_CHUNK>());
  if (HALF) chunk(full, std::integral_constant<int, AT_CHUNK / 2>());
  ((d2v*)gx)[m] = d2v{ax, ay};
}

// The taps of one loop, one phase, each adding to its signal index (a cleared gx): tap i of
// [0, count) is id = i (head phase, bucket i mod B) or id = i*tiles + B (tail phase, bucket i).
// Within a launch every tap has an index of its own.
__global__ __launch_bounds__(256) void adj_taps_kernel(
    const double2* __restrict__ f, const double2* __restrict__ gb, const int* __restrict__ ai_dev,
    int l, uint32_t mask, int B, uint32_t count, int tail, uint32_t tiles,
    double2* __restrict__ gx) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= count) return;
  const uint32_t id = tail ? i * tiles + (uint32_t)B : i;
  const d2v fv = ((const d2v*)f)[id];
  const d2v gv = ((const d2v*)gb)[(size_t)l * (size_t)B + (tail ? i : i & ((uint32_t)B - 1u))];
  d2v* dst = (d2v*)gx + ((id * (uint32_t)ai_dev[l]) & mask);
  d2v acc = *dst;
  acc.x = acc.x + fma(fv.x, gv.x, fv.y * gv.y);
  acc.y = acc.y + fma(fv.x, gv.y, -(fv.y * gv.x));
  *dst = acc;
}

// Whether the taps go in their own order: few taps in a long signal, where the lookups of all
// n * loops pairs cost more than the clear and the scattered additions of the w * loops taps.
// Taps against lookups, us: n = 2^23, 7 loops, w/n = 0.2 % 56 / 73, 0.85 % 69 / 74, 1.7 % 85 / 77;
// n = 2^24 0.4 % 91 / 139, 1.2 % 138 / 142, 1.7 % 162 / 144; n = 2^26 0.4 % 357 / 532, 1.2 %
// 517 / 561, 1.7 % 610 / 574, 3 loops 0.4 % 274 / 333, 1.2 % 347 / 347; n = 2^27, 9 loops 0.2 %
// 569 / 1456, 1.2 % 1203 / 1490, 1.7 % 1523 / 1481.  Below 2^23 the launches cost more (n = 2^22,
// 0.2 % 45 / 41).  Beyond a chunk of loops the lookups pay for the last chunk's empty places.
static bool taps_in_order(int n, int w, int loops) {
  if (n < (1 << 23)) return false;
  if (loops <= AT_CHUNK) return 80LL * w <= n;
  const int half = AT_CHUNK / 2, places = (loops + half - 1) / half * half;
  return 72LL * w * loops <= (long long)n * places;
}

hipError_t adjoint_taps_launch(const double2* f, const double2* gb, const int* a_dev,
                               const int* ai_dev, int n, int B, int w, int loops, int tiled,
                               double2* gx, hipStream_t st) {
  const uint32_t tiles = (uint32_t)(w / B);
  const uint32_t head = tiled ? tiles * (uint32_t)B : (uint32_t)w;
  const uint32_t residue = tiled ? (uint32_t)(w % B) : 0u;
  if (!taps_in_order(n, w, loops)) {
    // floor(d * magic / 2^32) = d / tiles for the multiples d = i * tiles of a tail tap: magic =
    // (2^32 + e) / tiles with e < tiles, and i * e < B * tiles <= w < 2^32
    const uint32_t magic = tiles > 1 ? 0xFFFFFFFFu / tiles + 1u : 0u;
    const int rest = loops % AT_CHUNK;
    const auto kernel =
        rest > 0 && rest <= AT_CHUNK / 2 ? adj_lookup_kernel<true> : adj_lookup_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(((unsigned)n + 255u) / 256u), dim3(256), 0, st, f, gb, a_dev,
                       loops, (uint32_t)n, B, head, residue, tiles, magic, gx);
    return hipGetLastError();
  }
  hipError_t e = fill_u32(gx, 0u, (size_t)n * 4, st);
  for (int l = 0; l < loops; ++l)
    for (int tail = 0; tail < (residue > 0 ? 2 : 1); ++tail) {
      if (e != hipSuccess) return e;
      const uint32_t count = tail ? residue : head;
      hipLaunchKernelGGL(adj_taps_kernel, dim3((count + 255u) / 256u), dim3(256), 0, st, f, gb,
                         ai_dev, l, (uint32_t)n - 1u, B, count, tail, tiles, gx);
      e = hipGetLastError();
    }
  return e;
}

}  // namespace sfft
