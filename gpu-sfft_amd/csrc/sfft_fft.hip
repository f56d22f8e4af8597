// sfft_fft.hip -- hand-written CDNA4 (gfx950) kernels of the sparse-FFT hot path, part 1.
//
//  * fft_pass_kernel      canonical multi-pass big-radix Stockham FFT (LDS sub-FFT, radix-4/2
//                         stages), optional fused comb gather (RLFC) and |X|^2 key epilogue
//  * perm_filter_kernel   permutation + filtering: bucket-owner gather fold, all loops of a
//                         transform in one launch, fixed (deterministic) tap order
//
// Every floating-point operation that must match the CPU oracle bit for bit is written out
// explicitly (fma where fused, plain ops elsewhere); the library is built with
// -ffp-contract=off so the compiler adds no fusion of its own.
#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "sfft_jobs.h"

namespace sfft {

template <typename R>
struct CT;
template <>
struct CT<double> {
  using T2 = double2;
  using K = unsigned long long;
};
template <>
struct CT<float> {
  using T2 = float2;
  using K = unsigned int;
};

// complex element as a native vector (arrays of HIP's double2/float2 wrappers end up in scratch)
template <typename Real>
struct NV {
  typedef Real type __attribute__((ext_vector_type(2)));
};

__device__ __forceinline__ double2 cmul(double2 a, double2 w) {
  return make_double2(fma(a.x, w.x, -(a.y * w.y)), fma(a.x, w.y, a.y * w.x));
}
__device__ __forceinline__ float2 cmul(float2 a, float2 w) {
  return make_float2(fmaf(a.x, w.x, -(a.y * w.y)), fmaf(a.x, w.y, a.y * w.x));
}
// |X|^2 as the reference's pow(re,2) + pow(im,2) (innerLoop.cu:715): each square rounded,
// then added
__device__ __forceinline__ unsigned long long sample_key(double2 v) {
  return (unsigned long long)__double_as_longlong(v.x * v.x + v.y * v.y);
}
__device__ __forceinline__ unsigned int sample_key(float2 v) {
  return __float_as_uint(v.x * v.x + v.y * v.y);
}

template <typename T2>
__device__ __forceinline__ T2 cadd(T2 a, T2 b) {
  T2 r;
  r.x = a.x + b.x;
  r.y = a.y + b.y;
  return r;
}
template <typename T2>
__device__ __forceinline__ T2 csub(T2 a, T2 b) {
  T2 r;
  r.x = a.x - b.x;
  r.y = a.y - b.y;
  return r;
}

// radix-4 butterfly: t0=a0+a2, t1=a0-a2, t2=a1+a3, t3=(a1-a3)*(-+i); y=(t0+t2, t1+t3, t0-t2, t1-t3)
template <typename T2>
__device__ __forceinline__ void bfly4(T2& a0, T2& a1, T2& a2, T2& a3, int inverse) {
  const T2 t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), d = csub(a1, a3);
  T2 t3;
  if (inverse) {
    t3.x = -d.y;
    t3.y = d.x;
  } else {
    t3.x = d.y;
    t3.y = -d.x;
  }
  a0 = cadd(t0, t2);
  a1 = cadd(t1, t3);
  a2 = csub(t0, t2);
  a3 = csub(t1, t3);
}

// ============================================================================================
// FFT pass
// ============================================================================================
// columns per tile: 32, so that the sub-FFTs of 256 points (FP32) or 128 (FP64) and fewer
// also fill a tile
constexpr int FFT_QMAX = 32;
// complex elements per tile (LDS): 8192 complex64 (66 KB) or 4096 complex128 (66 KB) with
// 1024 threads, so that two workgroups (32 waves) fill a CU and one loads while the other
// computes (1024 threads rather than 512: the n = 2^27 comb and bucket FFT passes run 3-10%
// faster).
// The pass that gathers the comb samples from the signal (random lines) uses one 2048-point
// column per tile (32 KB FP64 / 16 KB FP32) with 512 threads (FP64: four workgroups per CU)
// or 256 (FP32: eight), so more gathers are in flight while other workgroups compute
// (measured at n = 2^27: 256 threads cost FP64 10 us, 1024 cost it 65 us; FP32 gains 6 us).
// LOADX: an FftLoad, plus kSmallTile for a quarter of the elements and threads.  A thread's
// loops cover its share of a full tile whatever the tile holds, so a pass whose columns cannot
// fill one (few columns, short sub-FFTs) takes the quarter instead of idling three of four
// threads (pass_shape).
constexpr int kSmallTile = 16;
template <typename Real, int LOADX = 0>
struct Tile {   // kLoadComb (gathers from x), or any other load (plain)
  static constexpr bool comb = LOADX == kLoadComb, small = (LOADX & kSmallTile) != 0;
  static constexpr int cap = comb ? 2048 : (sizeof(Real) == 8 ? 4096 : 8192) / (small ? 4 : 1);
  // threads per workgroup; FP32 plain tiles: 512, so that a radix-16 step's 16 complex64
  // values and their twiddles fit the 128 registers of two 512-thread workgroups per CU
  // (FP64 keeps 1024 threads and single radix-4 stages: measured faster at 2^22)
  static constexpr int nt = comb ? (sizeof(Real) == 8 ? 512 : 256)
                                 : (sizeof(Real) == 8 ? 1024 : 512) / (small ? 4 : 1);
  static constexpr int ept = cap / nt;                 // elements per thread
  // 8 (FP64) or 4 (FP32) waves per SIMD: two full plain tiles per CU
  static constexpr int waves = comb ? 1 : sizeof(Real) == 8 ? 8 : 4;
};
static int tile_cap(int is_fp32, int load) {
  if (load == kLoadComb) return Tile<float, kLoadComb>::cap;
  return is_fp32 ? Tile<float>::cap : Tile<double>::cap;
}

// Workgroups are dealt to the 8 XCDs round-robin by launch order.  Tiles t, t+1, ... read
// neighbouring columns of the same 128-byte lines, so give the workgroups of one XCD (ids
// x, x+8, x+16, ...) consecutive tiles: the lines are then shared in that XCD's L2 instead
// of being fetched once per XCD.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  return (nb & 7) ? b : (b & 7) * (nb >> 3) + (b >> 3);
}

// LDS layout of a tile: column c at lds[c * RP + LPAD(v)] with one padding slot after every 16
// elements and a one-slot skew between columns, so the radix-4 stage's stride-4 and stride-16
// stores and the column-interleaved loads spread over the LDS banks.
#define LPAD(x) ((x) + ((x) >> 4))

// The twiddles of a stage's butterflies for this thread: radix-4 stage with ns = 4^k > 1 (its
// quads {W^jm, W^2jm, W^3jm}), loaded one stage ahead so that their latency hides behind the
// stage before.  A butterfly's j (and so its slot here) does not depend on the stage.
template <typename T2, int EPT, int NT>
__device__ __forceinline__ void stage4_twiddles(T2 (&w)[EPT / 4][3], int r, int log2ncol,
                                                int log2ns, const T2* __restrict__ tw4) {
  const int Rq = 1 << (r - 2);
  const int nbf = (1 << log2ncol) * Rq;
  const int ns = 1 << log2ns;
  const T2* __restrict__ q4 = tw4 + 4 * ((ns - 4) / 3);   // this stage's quads
#pragma unroll
  for (int kk = 0; kk < EPT / 4; ++kk) {
    const int bi = min((int)threadIdx.x + kk * NT, nbf - 1);
    const T2* q = q4 + 4 * ((bi & (Rq - 1)) & (ns - 1));
    w[kk][0] = q[0];
    w[kk][1] = q[1];
    w[kk][2] = q[2];
  }
}

template <typename T2, int EPT, int NT, bool TWID>
__device__ __forceinline__ void fft_stage4(T2* lds, int RP, int r, int log2ncol, int log2ns,
                                           const T2 (&w)[EPT / 4][3], int inverse) {
  // Butterfly indices past the tile (partial tiles) are clamped to the last butterfly, whose
  // thread stores the same values: no per-butterfly branches, so every LDS read of the thread
  // is in flight together.  TWID: ns > 1 (twiddles w from stage4_twiddles).
  const int tid = threadIdx.x;
  const int Rq = 1 << (r - 2);
  const int nbf = (1 << log2ncol) * Rq;
  const int ns = 1 << log2ns;
  T2 v[EPT];
#pragma unroll
  for (int kk = 0; kk < EPT / 4; ++kk) {
    const int bi = min(tid + kk * NT, nbf - 1);
    const int c = bi >> (r - 2);
    const int j = bi & (Rq - 1);
    const T2* col = lds + c * RP;
    T2 a0 = col[LPAD(j)], a1 = col[LPAD(j + Rq)], a2 = col[LPAD(j + 2 * Rq)],
       a3 = col[LPAD(j + 3 * Rq)];
    if (TWID) {
      a1 = cmul(a1, w[kk][0]);
      a2 = cmul(a2, w[kk][1]);
      a3 = cmul(a3, w[kk][2]);
    }
    bfly4(a0, a1, a2, a3, inverse);
    v[4 * kk + 0] = a0;
    v[4 * kk + 1] = a1;
    v[4 * kk + 2] = a2;
    v[4 * kk + 3] = a3;
  }
  __syncthreads();
#pragma unroll
  for (int kk = 0; kk < EPT / 4; ++kk) {
    const int bi = min(tid + kk * NT, nbf - 1);
    const int c = bi >> (r - 2);
    const int j = bi & (Rq - 1);
    T2* col = lds + c * RP;
    const int base = ((j >> log2ns) << (log2ns + 2)) + (j & (ns - 1));
    col[LPAD(base)] = v[4 * kk + 0];
    col[LPAD(base + ns)] = v[4 * kk + 1];
    col[LPAD(base + 2 * ns)] = v[4 * kk + 2];
    col[LPAD(base + 3 * ns)] = v[4 * kk + 3];
  }
  __syncthreads();
}

// Two radix-4 stages (spans ns and 4ns) in registers: task (column c, tix = a0*ns + jm), one
// per thread, reads the 16 elements tix + u*R/16 (u = t + 4m: input m of the first stage's
// butterfly t, whose index is tix + t*R/16), runs the four first-stage butterflies (twiddles
// W_{4ns}^{m*jm}, the same for every t), then the four second-stage butterflies (butterfly m
// takes the first stage's outputs m of t = 0..3; twiddles W_{16ns}^{t*(m*ns + jm)}) and writes
// output m'' of butterfly m to a0*16ns + jm + (m + 4m'')*ns.  These are the two stages' own
// operations in their own order (the same bits), with one LDS round trip instead of two.
// the two stages of a radix-16 step on its 16 elements in registers (see fft_stage16)
template <typename T2, bool TW1>
__device__ __forceinline__ void stage16_regs(T2 (&x)[16], int jm, int ns,
                                             const T2* __restrict__ tw4, int inverse) {
  if (TW1) {
    const T2* w = tw4 + 4 * ((ns - 4) / 3 + jm);
    const T2 w1 = w[0], w2 = w[1], w3 = w[2];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      x[t + 4] = cmul(x[t + 4], w1);
      x[t + 8] = cmul(x[t + 8], w2);
      x[t + 12] = cmul(x[t + 12], w3);
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) bfly4(x[t], x[t + 4], x[t + 8], x[t + 12], inverse);
  // second stage: butterfly m takes x[4m' ... ] -> inputs m' = t: x[t + 4m]
  const T2* q2 = tw4 + 4 * ((4 * ns - 4) / 3 + jm);
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const T2* w = q2 + 4 * m * ns;
    x[1 + 4 * m] = cmul(x[1 + 4 * m], w[0]);
    x[2 + 4 * m] = cmul(x[2 + 4 * m], w[1]);
    x[3 + 4 * m] = cmul(x[3 + 4 * m], w[2]);
    bfly4(x[4 * m], x[1 + 4 * m], x[2 + 4 * m], x[3 + 4 * m], inverse);
  }
}

template <typename T2, int NT, bool TW1>
__device__ __forceinline__ void fft_stage16(T2* lds, int RP, int r, int log2ncol, int log2ns,
                                            const T2* __restrict__ tw4, int inverse) {
  const int tid = threadIdx.x;
  const int R16 = 1 << (r - 4);
  const int ntask = (1 << log2ncol) * R16;
  const int ns = 1 << log2ns;
  T2 x[16];
  int base = 0, c = 0;
  if (tid < ntask) {
    c = tid >> (r - 4);
    const int tix = tid & (R16 - 1);
    const int jm = tix & (ns - 1);
    base = ((tix >> log2ns) << (log2ns + 4)) + jm;
    const T2* col = lds + c * RP;
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = col[LPAD(tix + u * R16)];
    stage16_regs<T2, TW1>(x, jm, ns, tw4, inverse);
  }
  __syncthreads();
  if (tid < ntask) {
    T2* col = lds + c * RP;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int m2 = 0; m2 < 4; ++m2) col[LPAD(base + (m + 4 * m2) * ns)] = x[m2 + 4 * m];
  }
  __syncthreads();
}

// The last radix-4 stage (span ns = R/8) and the radix-2 stage after it (span R/2) in
// registers: task (column c, jm < R/8) reads the 8 elements jm + i*R/8, runs the radix-4
// butterflies j = jm (inputs i = 0, 2, 4, 6) and j = jm + R/8 (inputs i = 1, 3, 5, 7, with the
// same twiddles W_{4ns}^{m*jm}), whose outputs k belong at jm + k*R/8 and R/2 + jm + k*R/8,
// then the four radix-2 butterflies j' = jm + k*R/8 (twiddle W_R^{j'}) on those pairs, whose
// outputs belong at j' and j' + R/2.  The two stages' own operations in their own order (the
// same bits), with one LDS round trip instead of two.  A task writes exactly the 8 elements it
// read, so it stores each output as soon as it has it (no barrier between its reads and its
// writes).  So every task runs exactly once: a second thread on the same elements (a clamped
// duplicate) could read them after their owner has rewritten them.  A thread takes up to
// EPT/8 tasks (one when EPT < 8; threads past the tasks idle, whole waves at a time).
template <typename T2, int EPT, int NT, bool TW1>
__device__ __forceinline__ void fft_stage8(T2* lds, int RP, int r, int log2ncol,
                                           const T2* __restrict__ tw4,
                                           const T2* __restrict__ twR, int inverse) {
  constexpr int TPT = EPT >= 8 ? EPT / 8 : 1;
  const int tid = threadIdx.x;
  const int R8 = 1 << (r - 3);
  const int ntask = (1 << log2ncol) * R8;
#pragma unroll
  for (int kk = 0; kk < TPT; ++kk) {
    const int ti = tid + kk * NT;
    if (ti < ntask) {
      const int jm = ti & (R8 - 1);
      T2* col = lds + (ti >> (r - 3)) * RP;
      T2 x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = col[LPAD(jm + i * R8)];
      if (TW1) {
        const T2* w = tw4 + 4 * ((R8 - 4) / 3 + jm);
        const T2 w1 = w[0], w2 = w[1], w3 = w[2];
        x[2] = cmul(x[2], w1);
        x[4] = cmul(x[4], w2);
        x[6] = cmul(x[6], w3);
        x[3] = cmul(x[3], w1);
        x[5] = cmul(x[5], w2);
        x[7] = cmul(x[7], w3);
      }
      bfly4(x[0], x[2], x[4], x[6], inverse);
      bfly4(x[1], x[3], x[5], x[7], inverse);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const T2 a1 = cmul(x[2 * k + 1], twR[jm + k * R8]);
        col[LPAD(jm + k * R8)] = cadd(x[2 * k], a1);
        col[LPAD(jm + (4 + k) * R8)] = csub(x[2 * k], a1);
      }
    }
  }
  __syncthreads();
}

template <typename T2, int EPT, int NT>
__device__ __forceinline__ void fft_stage2(T2* lds, int RP, int r, int log2ncol, int log2ns,
                                           const T2* __restrict__ twR) {
  // (clamped butterfly indices as in fft_stage4)
  const int tid = threadIdx.x;
  const int Rh = 1 << (r - 1);
  const int nbf = (1 << log2ncol) * Rh;
  const int ns = 1 << log2ns;
  const int tstep = 1 << (r - log2ns - 1);
  T2 v[EPT];
  if (ns > 1) {
#pragma unroll
    for (int kk = 0; kk < EPT / 2; ++kk) {
      const int bi = min(tid + kk * NT, nbf - 1);
      const int c = bi >> (r - 1);
      const int j = bi & (Rh - 1);
      const T2* col = lds + c * RP;
      T2 a0 = col[LPAD(j)], a1 = col[LPAD(j + Rh)];
      a1 = cmul(a1, twR[(j & (ns - 1)) * tstep]);
      v[2 * kk + 0] = cadd(a0, a1);
      v[2 * kk + 1] = csub(a0, a1);
    }
  } else {
#pragma unroll
    for (int kk = 0; kk < EPT / 2; ++kk) {
      const int bi = min(tid + kk * NT, nbf - 1);
      const int c = bi >> (r - 1);
      const int j = bi & (Rh - 1);
      const T2* col = lds + c * RP;
      const T2 a0 = col[LPAD(j)], a1 = col[LPAD(j + Rh)];
      v[2 * kk + 0] = cadd(a0, a1);
      v[2 * kk + 1] = csub(a0, a1);
    }
  }
  __syncthreads();
#pragma unroll
  for (int kk = 0; kk < EPT / 2; ++kk) {
    const int bi = min(tid + kk * NT, nbf - 1);
    const int c = bi >> (r - 1);
    const int j = bi & (Rh - 1);
    T2* col = lds + c * RP;
    const int base = ((j >> log2ns) << (log2ns + 1)) + (j & (ns - 1));
    col[LPAD(base)] = v[2 * kk + 0];
    col[LPAD(base + ns)] = v[2 * kk + 1];
  }
  __syncthreads();
}

// TW: the pass's outer twiddles, known at compile time so that the load phase is straight-line
// code: none (the first pass) or products of a high and a low table entry
enum PassTw { kTwNone = 0, kTwSplit = 1 };

// (bx, by) of nbx: the workgroup's tile and batch (comb gathers: tile and batch in bx alone)
template <typename Real, int LOADX, int STORE, int TW>
__device__ __forceinline__ void fft_pass_body(const PassArgs& A, int bx, int nbx, int by) {
  constexpr int LOAD = LOADX & ~kSmallTile;
  using T2 = typename CT<Real>::T2;
  using KT = typename CT<Real>::K;
  constexpr int CAP = Tile<Real, LOADX>::cap, EPT = Tile<Real, LOADX>::ept;
  constexpr int NT = Tile<Real, LOADX>::nt;
  __shared__ T2 lds[CAP + CAP / 16 + FFT_QMAX];
  const int tid = threadIdx.x;
  // The comb-gathering pass runs all comb loops in one grid dimension, loop index fastest,
  // so the same tile of every loop is handled back to back on one XCD: comb loops whose
  // offsets fall in the same 128-byte window read the same lines, fetched once.
  int tile;
  long long b;
  if (LOAD == kLoadComb) {
    const int s = xcd_tile(bx, nbx);
    b = s % A.nbatch;
    tile = s / A.nbatch;
  } else {
    tile = xcd_tile(bx, nbx);
    b = by;
  }
  const int r = A.r;
  const int R = 1 << r;
  // padded column stride (see LPAD); rows of 16 points and more: no skew slot, so that any
  // number of them fits the tile
  const int RP = R + (R >> 4) + ((LOAD == kLoadRows && R >= 16) ? 0 : 1);
  const int log2Lprev = A.log2Lprev;
  const int log2Lcur = log2Lprev + r;
  const long long Lprev = 1LL << log2Lprev;
  const long long nq = 1LL << (A.log2N - log2Lcur);
  constexpr bool first = (TW == kTwNone);   // log2Lprev == 0
  int log2ncol;
  long long q0 = 0, q = 0, t0 = 0;
  // kLoadCombRowsG (comb rows with nq = 2^d * nlo sub-FFTs, d > 0): sub-FFT q reads every
  // 2^d-th element of row q mod nlo, interleaved with its siblings q + j*nlo (j < 2^d).  A tile
  // then takes 2^d sibling groups of ncol/2^d adjacent sub-FFTs, or ncol adjacent siblings of one
  // row where there are more than it has columns, so that it reads whole lines: tile column c is
  // sub-FFT q0 + qoff(c) (the same sub-FFTs and values, grouped differently).
  constexpr bool rows = (LOAD == kLoadCombRows || LOAD == kLoadCombRowsG);
  int log2cpj = 0;
  if (LOAD == kLoadRows) {
    log2ncol = A.log2Q;   // tile column c is row (tile << log2Q) + c
    log2cpj = log2ncol;
  } else if (first) {
    log2ncol = min(A.log2Q, A.log2N - log2Lcur);
    log2cpj = log2ncol;
    if (LOAD == kLoadCombRowsG) {
      const int d = (A.log2N - log2Lcur) - A.log2nlo;
      log2cpj = max(log2ncol - d, 0);
      const int part = max(d - log2ncol, 0);   // 2^part tiles share a row
      q0 = ((long long)(tile >> part) << log2cpj) +
           ((long long)(tile & ((1 << part) - 1)) << (A.log2nlo + log2ncol));
    } else {
      q0 = (long long)tile << log2cpj;
    }
  } else {
    log2ncol = A.log2Q;
    const int log2tpq = log2Lprev - A.log2Q;
    q = (long long)tile >> log2tpq;
    t0 = ((long long)tile & ((1LL << log2tpq) - 1)) << A.log2Q;
  }
  const int ncol = 1 << log2ncol;
  const int TE = ncol << r;
  // element (c, v) of the tile: first pass g = q0 + c + nq*v, later passes
  // g = (q + nq*v)*Lprev + t0 + c -- both gbase + c + vstride*v (no per-element branches)
  const long long gbase = first ? q0 : q * Lprev + t0;
  const long long vstride = first ? nq : nq * Lprev;
  auto qoff = [&](int c) __attribute__((always_inline)) {
    return (long long)(c & ((1 << log2cpj) - 1)) + ((long long)(c >> log2cpj) << A.log2nlo);
  };

  // ---- load (+ outer twiddle) into LDS, column c at lds[c*RP + v].  Every element load of
  // the thread (and every twiddle load) is issued before any is used: in one basic block,
  // with out-of-tile elements clamped to a valid address, so the loads are in flight together
  // (guarding each load with its own branch made the compiler wait for each one in turn).
  using V2 = typename NV<Real>::type;
  const T2* __restrict__ in = (const T2*)A.in + b * A.in_bstride;
  const T2* __restrict__ cx =
      (LOAD == kLoadComb) ? (const T2*)A.comb_x + A.comb_offs[b] : (const T2*)nullptr;
  // kLoadPerm: tile column c takes the input positions p = q0 + c + nq*X (X < R), so that the
  // tile's ncol columns read whole lines.  Position p holds element g = p * pinv mod N of the
  // canonical order (perm[b] * pinv = 1 mod N), which is element v = g / nq of sub-FFT
  // g mod nq = (q0 + c) * pinv mod nq: the column is that sub-FFT, its elements land at their
  // own v (the same sub-FFTs and values as loading g at g * perm[b], grouped differently).
  const uint32_t pinv = (LOAD == kLoadPerm) ? (uint32_t)A.perm_inv[b] : 0u;
  const uint32_t nmask = (1u << A.log2N) - 1u;
  const int log2nq = A.log2N - log2Lcur;
  auto perm_v = [&](int e) __attribute__((always_inline)) {
    const uint32_t pos = (uint32_t)q0 + (uint32_t)(e & (ncol - 1)) +
                         ((uint32_t)(e >> log2ncol) << log2nq);
    return (int)(((pos * pinv) & nmask) >> log2nq);
  };
  // loads in flight per batch: the plain tiles take batches of 8 bytes x 4 (FP32, 512
  // threads) or 16 bytes x 2 (FP64, 1024 threads: within 64 registers); the comb-gathering
  // pass issues all of its loads together
  constexpr int LB = (LOAD == kLoadComb) ? EPT : (sizeof(Real) == 8 ? 2 : 4);
  const T2* __restrict__ twR = (const T2*)A.twR;
  const T2* __restrict__ tw4 = (const T2*)A.tw4;
  // batch kb: loads elements e = tid + (kb + k)*NT (k < LB), with the outer twiddle applied
  auto load_batch = [&](int kb, T2 (&val)[LB]) __attribute__((always_inline)) {
    V2 vv[LB];
#pragma unroll
    for (int k = 0; k < LB; ++k) {
      const int e = min(tid + (kb + k) * NT, TE - 1);
      const int c = e & (ncol - 1);
      const int v = e >> log2ncol;
      const long long g = gbase + c + vstride * v;
      const T2* src;
      if (LOAD == kLoadRows)   // (a row past the last one reads the last one)
        src = in + (min(((long long)tile << (log2ncol + r)) + e, ((long long)A.nbatch << r) - 1));
      else if (LOAD == kLoadComb)
        src = cx + g * (long long)A.comb_sigma;
      else if (rows) {
        const long long gr = (LOAD == kLoadCombRowsG) ? gbase + qoff(c) + vstride * v : g;
        src = in + (((gr & ((1LL << A.log2nlo) - 1)) << A.log2m) | (gr >> A.log2nlo));
      }
      else if (LOAD == kLoadPerm)
        src = in + ((uint32_t)q0 + (uint32_t)c + ((uint32_t)v << log2nq));
      else
        src = in + g;
      if constexpr (LOAD == kLoadWiden) {
        const NV<float>::type s = ((const NV<float>::type*)A.in)[b * A.in_bstride + g];
        vv[k].x = (Real)s.x;
        vv[k].y = (Real)s.y;
      } else if constexpr (LOAD == kLoadTaps) {
        // (a point outside the taps reads the first one and becomes zero: no branch)
        const long long h = A.taps / 2, tail = (1LL << A.log2N) - h;
        const bool lo = g < h, hi = g >= tail;
        vv[k] = *(const V2*)(in + (lo ? h + g : (hi ? g - tail : 0)));
        if (!lo && !hi) vv[k] = (V2)(Real)0;
      } else {
        vv[k] = *(const V2*)src;
      }
    }
#pragma unroll
    for (int k = 0; k < LB; ++k) {
      val[k].x = vv[k].x;
      val[k].y = vv[k].y;
    }
    if constexpr (!first) {
      // outer twiddles W_Lcur^((t0+c)*v): the product of a high and a low table entry (every
      // table load of the batch issued first, as for the data)
      V2 tw[LB], tl[LB];
      const V2* __restrict__ thi = (const V2*)A.thi;
      const V2* __restrict__ tlo = (const V2*)A.tlo;
      const uint32_t lmask = (1u << A.s) - 1u;
#pragma unroll
      for (int k = 0; k < LB; ++k) {
        const int e = min(tid + (kb + k) * NT, TE - 1);
        const uint32_t ex = (uint32_t)((t0 + (e & (ncol - 1))) * (e >> log2ncol));
        tw[k] = thi[ex >> A.s];
        tl[k] = tlo[ex & lmask];
      }
#pragma unroll
      for (int k = 0; k < LB; ++k) {
        T2 hi, lo;
        hi.x = tw[k].x;
        hi.y = tw[k].y;
        lo.x = tl[k].x;
        lo.y = tl[k].y;
        const T2 w = cmul(hi, lo);
        tw[k].x = w.x;
        tw[k].y = w.y;
      }
#pragma unroll
      for (int k = 0; k < LB; ++k) {
        const int e = min(tid + (kb + k) * NT, TE - 1);
        T2 w;
        w.x = tw[k].x;
        w.y = tw[k].y;
        const T2 tv = cmul(val[k], w);
        if ((e >> log2ncol) > 0) val[k] = tv;
      }
    }
  };
  // A full plain tile (TE == NT*EPT): the thread's elements e = tid + k*NT are the elements
  // v = j + k*R/EPT of column c = tid mod ncol (j = tid / ncol), the inputs of one task of the
  // first stage -- FP32 (EPT 16): the radix-16 step of fft_stage16 (its task (c, tix = j));
  // FP64 (EPT 4): the radix-4 butterfly j of fft_stage4.  The thread runs that task on the
  // loaded values in registers and writes only its outputs to LDS: the same operations on the
  // same values as storing the loads and running the stage, with one LDS round trip fewer.
  constexpr int FR = sizeof(Real) == 4 ? 16 : 4;
  constexpr bool can_fuse = (LOAD == kLoadPlain || LOAD == kLoadWiden || LOAD == kLoadTaps ||
                             rows) && EPT == FR;
  int log2ns0 = 0;
  bool fused = false;
  if constexpr (can_fuse) {
    if (TE == NT * EPT && (1 << r) >= FR) {
      fused = true;
      T2 x[EPT];
#pragma unroll
      for (int kb = 0; kb < EPT; kb += LB) {
        T2 val[LB];
        load_batch(kb, val);
#pragma unroll
        for (int k = 0; k < LB; ++k) x[kb + k] = val[k];
      }
      const int j = tid >> log2ncol;
      T2* col = lds + (tid & (ncol - 1)) * RP;
      if constexpr (EPT == 16) {
        stage16_regs<T2, false>(x, 0, 1, tw4, A.inverse);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int m2 = 0; m2 < 4; ++m2) col[LPAD((j << 4) + m + 4 * m2)] = x[m2 + 4 * m];
        log2ns0 = 4;
      } else {
        bfly4(x[0], x[1], x[2], x[3], A.inverse);
#pragma unroll
        for (int m = 0; m < 4; ++m) col[LPAD((j << 2) + m)] = x[m];
        log2ns0 = 2;
      }
    }
  }
  if (!fused) {
#pragma unroll
    for (int kb = 0; kb < EPT; kb += LB) {
      T2 val[LB];
      load_batch(kb, val);
#pragma unroll
      for (int k = 0; k < LB; ++k) {
        // (a clamped element is stored again with its own value: no branch)
        const int e = min(tid + (kb + k) * NT, TE - 1);
        const int c = (LOAD == kLoadRows) ? e >> r : e & (ncol - 1);
        const int v = (LOAD == kLoadPerm) ? perm_v(e)
                                          : (LOAD == kLoadRows ? e & (R - 1) : e >> log2ncol);
        lds[c * RP + LPAD(v)] = val[k];
      }
    }
  }
  __syncthreads();

  // ---- sub-FFT of every column: radix-4 stages, then one radix-2 stage if r is odd
  // FP32: pairs of radix-4 stages as radix-16 steps in registers; FP64: radix-4 stages.  Then
  // the remaining radix-4 stages, the last one fused with the radix-2 stage when r is odd (the
  // same stages in the same order), after the stage run at load time on a full tile
  int log2ns = log2ns0;
  int rem = r - log2ns0;
  while (sizeof(Real) == 4 && rem >= 4) {
    if (log2ns == 0)
      fft_stage16<T2, NT, false>(lds, RP, r, log2ncol, 0, tw4, A.inverse);
    else
      fft_stage16<T2, NT, true>(lds, RP, r, log2ncol, log2ns, tw4, A.inverse);
    log2ns += 4;
    rem -= 4;
  }
  while (rem >= 2) {
    if (rem == 3) {   // the last radix-4 stage with the radix-2 stage: one LDS round trip
      if (log2ns > 0)
        fft_stage8<T2, EPT, NT, true>(lds, RP, r, log2ncol, tw4, twR, A.inverse);
      else
        fft_stage8<T2, EPT, NT, false>(lds, RP, r, log2ncol, tw4, twR, A.inverse);
      log2ns += 3;
      rem = 0;
      break;
    }
    T2 wc[EPT / 4][3];
    if (log2ns > 0) {
      stage4_twiddles<T2, EPT, NT>(wc, r, log2ncol, log2ns, tw4);
      fft_stage4<T2, EPT, NT, true>(lds, RP, r, log2ncol, log2ns, wc, A.inverse);
    } else {
      fft_stage4<T2, EPT, NT, false>(lds, RP, r, log2ncol, 0, wc, A.inverse);
    }
    log2ns += 2;
    rem -= 2;
  }
  if (rem == 1) fft_stage2<T2, EPT, NT>(lds, RP, r, log2ncol, log2ns, twR);

  // ---- store: out[q*Lcur + t + Lprev*k]
  T2* __restrict__ out = (T2*)A.out + b * A.out_bstride;
  KT* __restrict__ keys = (KT*)A.keys + b * A.keys_bstride;
  const bool wkeys = (STORE == kStoreKeys || STORE == kStoreBoth) && (b < A.key_batches);
  uint32_t dg[EPT];   // the first digits of the thread's keys
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int e = tid + k * NT;
    if (e < TE) {
      int c, kk;
      long long g;
      if (first) {
        c = e >> r;
        kk = e & (R - 1);
        // kLoadPerm: column c is sub-FFT (q0 + c) * pinv mod nq; kLoadCombRowsG: q0 + qoff(c)
        const long long qc =
            (LOAD == kLoadPerm)
                ? (long long)(((uint32_t)(q0 + c) * pinv) & (((uint32_t)nq) - 1u))
                : (LOAD == kLoadCombRowsG ? q0 + qoff(c) : q0 + c);
        g = qc * R + kk;
        if (LOAD == kLoadRows) {
          g = ((long long)tile << (log2ncol + r)) + e;
          if (g >= ((long long)A.nbatch << r)) continue;
        }
      } else {
        c = e & (ncol - 1);
        kk = e >> log2ncol;
        g = (q << log2Lcur) + t0 + c + Lprev * kk;
      }
      const T2 val = lds[c * RP + LPAD(kk)];
      if constexpr (STORE == kStoreHead) {
        T2 sv;
        sv.x = val.x * (Real)A.scale;
        sv.y = val.y * (Real)A.scale;
        if (g < A.head) out[g] = sv;
      } else if (STORE != kStoreKeys) {
        out[g] = val;
      }
      if (wkeys) {
        const long long kpos = A.keys_tiled ? (long long)tile * TE + e : g;
        const KT key = sample_key(val);
        keys[kpos] = key;
        dg[k] = sel_first_digit(key);
        if (A.digits) A.digits[b * A.keys_bstride + kpos] = (uint16_t)dg[k];
      }
    }
  }
  // ---- the cutoff's histogram of the tile's first digits: counted in LDS (two 16-bit counts per
  // word, over the tile's values once they are read), then the bins that are not empty added to
  // one of the segment's global histograms: the cutoff needs no launch that reads every digit and
  // none that sums a row of counts per block (n = 2^27, k = 16000: a transform 841 -> 829 us FP64,
  // 487 -> 479 FP32; k = 40000 FP32 1106 -> 1093).
  if constexpr (STORE == kStoreKeys || STORE == kStoreBoth) {
    if (wkeys && A.hist) {
      uint32_t* cnt = reinterpret_cast<uint32_t*>(lds);
      __syncthreads();
      for (int i = tid; i < kSelBins / 2; i += NT) cnt[i] = 0u;
      __syncthreads();
#pragma unroll
      for (int k = 0; k < EPT; ++k)
        if (tid + k * NT < TE) atomicAdd(&cnt[dg[k] >> 1], 1u << ((dg[k] & 1u) * 16u));
      __syncthreads();
      uint32_t* g = A.hist + ((size_t)b * kSelCopies + (size_t)(tile & (kSelCopies - 1))) * kSelBins;
      for (int i = tid; i < kSelBins / 2; i += NT) {
        const uint32_t w = cnt[i];
        if (w & 0xFFFFu) atomicAdd(&g[2 * i], w & 0xFFFFu);
        if (w >> 16) atomicAdd(&g[2 * i + 1], w >> 16);
      }
    }
  }
}

template <typename Real, int LOADX, int STORE, int TW>
__global__ __launch_bounds__((Tile<Real, LOADX>::nt), (Tile<Real, LOADX>::waves)) void
fft_pass_kernel(PassArgs A) {
  fft_pass_body<Real, LOADX, STORE, TW>(A, blockIdx.x, gridDim.x, blockIdx.y);
}

// the same pass of many signals (jobs of tiles x batch workgroups)
template <typename Real, int LOADX, int STORE, int TW>
__global__ __launch_bounds__((Tile<Real, LOADX>::nt), (Tile<Real, LOADX>::waves)) void
fft_jobs_kernel(JobsDev t) {
  const FftJob* j = job_here<FftJob>(t);
  if (!j) return;
  const PassArgs A = j->a;
  const int i = (int)blockIdx.x - j->block0;
  if constexpr (LOADX == kLoadComb) {
    fft_pass_body<Real, LOADX, STORE, TW>(A, i, j->tiles * A.nbatch, 0);
  } else {
    fft_pass_body<Real, LOADX, STORE, TW>(A, i % j->tiles, j->tiles, i / j->tiles);
  }
}

template <typename Real, int LOADX, int STORE, int TW>
static hipError_t launch_tile(const PassArgs& A, int tiles, int batch, hipStream_t st) {
  const dim3 grid = (LOADX == kLoadComb) ? dim3(tiles * batch, 1) : dim3(tiles, batch);
  hipLaunchKernelGGL((fft_pass_kernel<Real, LOADX, STORE, TW>), grid,
                     dim3(Tile<Real, LOADX>::nt), 0, st, A);
  return hipGetLastError();
}

// the loads that have a quarter tile
static constexpr bool has_small(int load, int store) {
  return store != kStoreHead && (load == kLoadPlain || load == kLoadPerm ||
                                 load == kLoadCombRows || load == kLoadCombRowsG);
}

template <typename Real, int LOAD, int STORE, int TW>
static hipError_t launch_pass(const PassArgs& A, int tiles, int batch, hipStream_t st) {
  if constexpr (has_small(LOAD, STORE)) {
    if (A.small_tile)
      return launch_tile<Real, LOAD | kSmallTile, STORE, TW>(A, tiles, batch, st);
  }
  if (A.small_tile) return hipErrorInvalidValue;
  return launch_tile<Real, LOAD, STORE, TW>(A, tiles, batch, st);
}

// the stores that a special load occurs with: combs give keys alone, buckets spectra and keys
static constexpr bool occurs(int load, int store) {
  if (load == kLoadPerm) return store != kStoreKeys;
  if (load == kLoadComb || load == kLoadCombRows || load == kLoadCombRowsG)
    return store != kStoreBoth;
  return true;
}

template <typename Real, int LOAD, int TW>
static hipError_t dispatch_store(const PassArgs& A, int store, int tiles, int batch,
                                 hipStream_t st) {
  if (store == kStoreCplx) return launch_pass<Real, LOAD, kStoreCplx, TW>(A, tiles, batch, st);
  if constexpr (occurs(LOAD, kStoreKeys)) {
    if (store == kStoreKeys) return launch_pass<Real, LOAD, kStoreKeys, TW>(A, tiles, batch, st);
  }
  if constexpr (occurs(LOAD, kStoreBoth)) {
    if (store == kStoreBoth) return launch_pass<Real, LOAD, kStoreBoth, TW>(A, tiles, batch, st);
  }
  return hipErrorInvalidValue;
}

// the FP64-only loads and stores (truth spectra, filter design)
static hipError_t dispatch_fp64(const PassArgs& A, int load, int store, int tw, int tiles,
                                int batch, hipStream_t st) {
  if (load == kLoadTaps)
    return store == kStoreCplx
               ? launch_pass<double, kLoadTaps, kStoreCplx, kTwNone>(A, tiles, batch, st)
               : hipErrorInvalidValue;
  if (load == kLoadWiden) {
    if (store == kStoreCplx)
      return launch_pass<double, kLoadWiden, kStoreCplx, kTwNone>(A, tiles, batch, st);
    return store == kStoreHead
               ? launch_pass<double, kLoadWiden, kStoreHead, kTwNone>(A, tiles, batch, st)
               : hipErrorInvalidValue;
  }
  if (load != kLoadPlain) return hipErrorInvalidValue;
  if (tw == kTwSplit)
    return launch_pass<double, kLoadPlain, kStoreHead, kTwSplit>(A, tiles, batch, st);
  return launch_pass<double, kLoadPlain, kStoreHead, kTwNone>(A, tiles, batch, st);
}

// the special loads only occur in first passes (no outer twiddles)
template <typename Real>
static hipError_t dispatch_pass(const PassArgs& A, int load, int store, int tw, int tiles,
                                int batch, hipStream_t st) {
  if (load == kLoadCombRows)
    return dispatch_store<Real, kLoadCombRows, kTwNone>(A, store, tiles, batch, st);
  if (load == kLoadCombRowsG)
    return dispatch_store<Real, kLoadCombRowsG, kTwNone>(A, store, tiles, batch, st);
  if (load == kLoadPerm)
    return dispatch_store<Real, kLoadPerm, kTwNone>(A, store, tiles, batch, st);
  if (load == kLoadComb)
    return dispatch_store<Real, kLoadComb, kTwNone>(A, store, tiles, batch, st);
  if (load == kLoadRows)
    return launch_pass<Real, kLoadRows, kStoreCplx, kTwNone>(A, tiles, 1, st);
  if (tw == kTwSplit)
    return dispatch_store<Real, kLoadPlain, kTwSplit>(A, store, tiles, batch, st);
  return dispatch_store<Real, kLoadPlain, kTwNone>(A, store, tiles, batch, st);
}

// Columns per tile (log2) of pass p, and whether it takes quarter tiles: where a full tile's
// columns would not fill more than a quarter anyway; where they would not fill all of it and a
// quarter still holds whole lines of 128 bytes per row (complex64 sub-FFTs of up to 128 points,
// complex128 of up to 64; 2^24 points as transforms of 2^12, complex64 256 -> 101 us,
// complex128 274 -> 208; of 2^13 and 2^14, complex64 211 -> 111 and 145 -> 111; a complex128 tile
// that 128-point sub-FFTs fill stays full: 215 against 223 at 2^14), unless the pass counts its keys'
// histogram, whose 4096 bins are cleared and added up once per tile (two combs of 2^23 complex64
// points: 167 us in quarter tiles, 119 in full ones); and, with half lines, where the launch
// would be fewer than 128 full tiles, half the CUs.
struct PassShape {
  int log2q, small_tile;
};
static PassShape pass_shape(const FftTables& T, const FftLaunch& L, int p, int r, int log2Lprev) {
  const int load = (p == 0) ? L.load : kLoadPlain;
  // a kLoadPerm pass takes as many columns as fit: whole lines of its input per tile
  const int qmax = (load != kLoadPerm && L.qmax > 0 && L.qmax <= FFT_QMAX) ? L.qmax : FFT_QMAX;
  const int cap = tile_cap(T.is_fp32, load);
  const int limit = p > 0 ? log2Lprev : T.log2n - r;   // columns there are
  auto cols = [&](int elems) {
    int q = 0;
    while ((1 << (q + 1)) <= qmax && ((1 << (q + 1)) << r) <= elems) ++q;
    return (p > 0 && q > log2Lprev) ? log2Lprev : q;
  };
  const int full = cols(cap), quarter = cols(cap / 4);
  const int store = (p == T.npass - 1) ? L.store : kStoreCplx;
  if (!has_small(load, store) || (1 << r) > cap / 4) return {full, 0};
  const int nf = full < limit ? full : limit, nq = quarter < limit ? quarter : limit;
  const int line = T.is_fp32 ? 4 : 3;
  const long long tiles = ((long long)L.batch << T.log2n) >> (nf + r);
  const bool fits = ((1 << nf) << r) <= cap / 4;
  const bool counts = p == T.npass - 1 && L.hist;
  const bool lines = !counts && ((1 << nf) << r) < cap && nq >= (line < nf ? line : nf);
  const bool idle = tiles < 128 && nq >= (line - 1 < nf ? line - 1 : nf);
  if (fits || lines || idle) return {quarter, 1};
  return {full, 0};
}

// Single-pass transforms of adjacent rows: rows per tile (log2), or -1 where the plain pass runs
// them (one row per workgroup and batch index).  As many rows as fill a tile, while at least
// 512 tiles are left (two workgroups per CU).  2^24 complex64 points in all, one row per workgroup,
// then rows filling tiles: rows of 16 points 6158 -> 42 us, 128 points 904 -> 53 us, 512 points
// 387 -> 60 us, 2048 points 94 -> 62 us.
static int rows_log2q(const FftTables& T, const FftLaunch& L) {
  const long long N = 1LL << T.log2n;
  if (T.npass != 1 || L.load != kLoadPlain || L.store != kStoreCplx || L.batch < 2 ||
      L.in_bstride != N || L.out_bstride != N)
    return -1;
  const int r = T.log2n, cap = tile_cap(T.is_fp32, kLoadRows);
  const int R = 1 << r, RP = R + (R >> 4) + (R >= 16 ? 0 : 1);
  int q = 0;
  while ((2LL << q) * R <= cap && (2LL << q) * RP <= cap + cap / 16 &&
         (L.batch >> (q + 1)) >= 512)
    ++q;
  return q;
}

KeyMap fft_keys_map(const FftLaunch& L) {
  KeyMap m;
  const FftTables& T = *L.tab;
  m.log2n = T.log2n;
  if (!L.keys_tiled || T.npass < 2) return m;
  const int last = T.npass - 1;
  const int r = T.logs[last];
  m.mid = r;
  m.lo = pass_shape(T, L, last, r, T.log2n - r).log2q;
  return m;
}

// calls fn(p, args, load, store, tw, tiles) for each pass of L in order
template <typename F>
static hipError_t each_pass(const FftLaunch& L, F&& fn) {
  const FftTables& T = *L.tab;
  const int log2N = T.log2n;
  const long long N = 1LL << log2N;
  const int np = T.npass;
  if (np == 0) {
    // N == 1: the DFT is the identity (copy / keys)
    return hipErrorInvalidValue;
  }
  int log2Lprev = 0;
  const void* cur_in = L.in;
  long long cur_in_stride = L.in_bstride;
  for (int p = 0; p < np; ++p) {
    const int r = T.logs[p];
    const int log2Lcur = log2Lprev + r;
    const bool last = (p == np - 1);
    // pass p writes to out (or mid, before the last) when (np - 1 - p) is even, else to scratch
    void* even = (last || !L.mid) ? L.out : L.mid;
    void* dst = (((np - 1 - p) & 1) == 0) ? even : L.scratch;
    const long long dst_stride = (dst == L.out) ? L.out_bstride : N;
    PassArgs A;
    A.in = cur_in;
    A.in_bstride = cur_in_stride;
    A.out = dst;
    A.out_bstride = dst_stride;
    A.keys = L.keys;
    A.keys_bstride = L.keys_bstride;
    A.key_batches = L.key_batches;
    A.log2N = log2N;
    A.r = r;
    A.log2Lprev = log2Lprev;
    int load = (p == 0) ? L.load : kLoadPlain;
    const PassShape shape = pass_shape(T, L, p, r, log2Lprev);
    int log2Q = shape.log2q;
    A.small_tile = shape.small_tile;
    const int rq = rows_log2q(T, L);
    int tiles;
    if (rq >= 0) {
      load = kLoadRows;
      A.small_tile = 0;
      log2Q = rq;
      tiles = (int)(((long long)L.batch + (1LL << rq) - 1) >> rq);
    } else if (p == 0) {
      const int lnq = log2N - log2Lcur;
      const int lq = log2Q < lnq ? log2Q : lnq;
      tiles = 1 << (lnq - lq);
      // comb rows holding 2^d sibling sub-FFTs per row: grouped (one column of each of ncol rows
      // reads a line per element; two combs of 2^26 complex64 points of a signal of 2^26, rows of
      // 2^14, where a tile has 16 columns of 32 siblings: 2618 -> 458 us)
      const int d = lnq - L.comb_log2nlo;
      if (load == kLoadCombRows && d > 0) load = kLoadCombRowsG;
    } else {
      tiles = (int)((1LL << (log2N - log2Lcur)) << (log2Lprev - log2Q));
    }
    A.log2Q = log2Q;
    A.inverse = T.inverse;
    A.twR = T.twR[p];
    A.tw4 = T.tw4[p];
    A.thi = T.thi[p];
    A.tlo = T.tlo[p];
    A.s = T.s[p];
    A.comb_x = L.comb_x;
    A.comb_offs = L.comb_offs;
    A.comb_sigma = L.comb_sigma;
    A.log2nlo = L.comb_log2nlo;
    A.log2m = L.comb_log2m;
    A.perm = L.perm;
    A.perm_inv = L.perm_inv;
    if (load == kLoadPerm && (!L.perm || !L.perm_inv)) return hipErrorInvalidValue;
    A.nbatch = L.batch;
    A.taps = L.taps;
    A.head = L.head;
    A.scale = L.scale;
    A.keys_tiled = (last && p > 0 && L.keys_tiled) ? 1 : 0;
    A.digits = last ? L.digits : nullptr;
    A.hist = last ? L.hist : nullptr;
    const int store = last ? L.store : kStoreCplx;
    const int tw = (p == 0) ? kTwNone : kTwSplit;
    if (load != kLoadPlain && tw != kTwNone) return hipErrorInvalidValue;
    const hipError_t e = fn(p, A, load, store, tw, tiles);
    if (e != hipSuccess) return e;
    cur_in = dst;
    cur_in_stride = dst_stride;
    log2Lprev = log2Lcur;
  }
  return hipSuccess;
}

hipError_t fft_run(const FftLaunch& L, hipStream_t st) {
  const int fp32 = L.tab->is_fp32;
  return each_pass(L, [&](int, const PassArgs& A, int load, int store, int tw, int tiles) {
    if (load == kLoadWiden || load == kLoadTaps || store == kStoreHead)
      return fp32 ? hipErrorInvalidValue : dispatch_fp64(A, load, store, tw, tiles, L.batch, st);
    return fp32 ? dispatch_pass<float>(A, load, store, tw, tiles, L.batch, st)
                : dispatch_pass<double>(A, load, store, tw, tiles, L.batch, st);
  });
}

// ---- the comb FFT and the bucket FFTs of a short transform, pass by pass in one launch --------
// Where both FFTs run quarter tiles a pass is a few workgroups and some 5 us, most of it the
// launch: side by side on two streams they cost two launches per pass and the events that fork
// and join the streams.
struct OnePass {
  PassArgs a;
  int load, store, tw, tiles, batch;
  int blocks() const { return tiles * batch; }
};

// (half the waves of a pass alone: both bodies' tiles are in the workgroup's LDS)
template <typename Real, int LA, int SA, int LB, int SB, int TW>
__global__ __launch_bounds__((Tile<Real, LA>::nt), (Tile<Real, LA>::waves / 2)) void
fft_pair_kernel(PassArgs A, PassArgs B, int tiles_a, int blocks_a, int tiles_b) {
  static_assert(Tile<Real, LA>::nt == Tile<Real, LB>::nt, "one block size");
  const int i = blockIdx.x;
  if (i < blocks_a) {
    fft_pass_body<Real, LA, SA, TW>(A, i % tiles_a, tiles_a, i / tiles_a);
  } else {
    const int k = i - blocks_a;
    fft_pass_body<Real, LB, SB, TW>(B, k % tiles_b, tiles_b, k / tiles_b);
  }
}

template <typename Real, int LA, int SA, int LB, int SB, int TW>
static hipError_t pair_go(const OnePass& a, const OnePass& b, hipStream_t st) {
  hipLaunchKernelGGL((fft_pair_kernel<Real, LA | kSmallTile, SA, LB | kSmallTile, SB, TW>),
                     dim3(a.blocks() + b.blocks()), dim3(Tile<Real, LA | kSmallTile>::nt), 0, st,
                     a.a, b.a, a.tiles, a.blocks(), b.tiles);
  return hipGetLastError();
}

// first passes: the last ones too (keys out) or not
template <typename Real, int LA>
static hipError_t pair_first(const OnePass& a, const OnePass& b, hipStream_t st) {
  const bool ka = a.store == kStoreKeys, kb = b.store == kStoreBoth;
  if (ka && kb) return pair_go<Real, LA, kStoreKeys, kLoadPerm, kStoreBoth, kTwNone>(a, b, st);
  if (ka) return pair_go<Real, LA, kStoreKeys, kLoadPerm, kStoreCplx, kTwNone>(a, b, st);
  if (kb) return pair_go<Real, LA, kStoreCplx, kLoadPerm, kStoreBoth, kTwNone>(a, b, st);
  return pair_go<Real, LA, kStoreCplx, kLoadPerm, kStoreCplx, kTwNone>(a, b, st);
}

template <typename Real>
static hipError_t pair_pass(const OnePass& a, const OnePass& b, hipStream_t st) {
  if (a.load == kLoadCombRows) return pair_first<Real, kLoadCombRows>(a, b, st);
  if (a.load == kLoadCombRowsG) return pair_first<Real, kLoadCombRowsG>(a, b, st);
  return pair_go<Real, kLoadPlain, kStoreKeys, kLoadPlain, kStoreBoth, kTwSplit>(a, b, st);
}

// the passes of L (two at most), or fewer than L has where one of them has no quarter tile
static int short_passes(const FftLaunch& L, OnePass* out) {
  int n = 0;
  if (L.tab->npass > 2) return -1;
  const hipError_t e = each_pass(L, [&](int, const PassArgs& A, int load, int store, int tw,
                                        int tiles) {
    if (!A.small_tile) return hipErrorNotSupported;
    out[n++] = OnePass{A, load, store, tw, tiles, L.batch};
    return hipSuccess;
  });
  return e == hipSuccess ? n : -1;
}

// a comb FFT of the copied comb rows (keys out) and the bucket FFTs of column-ordered sums
// (spectra and keys out), every pass of both in quarter tiles
static bool pair_passes(const FftLaunch& comb, const FftLaunch& bucket, OnePass (&a)[2],
                        OnePass (&b)[2], int& na, int& nb) {
  if (comb.load != kLoadCombRows || comb.store != kStoreKeys || bucket.load != kLoadPerm ||
      bucket.store != kStoreBoth || comb.tab->is_fp32 != bucket.tab->is_fp32)
    return false;
  na = short_passes(comb, a);
  nb = short_passes(bucket, b);
  return na > 0 && nb > 0;
}

bool fft_pair_applies(const FftLaunch& comb, const FftLaunch& bucket) {
  OnePass a[2], b[2];
  int na, nb;
  return pair_passes(comb, bucket, a, b, na, nb);
}

hipError_t fft_run_pair(const FftLaunch& comb, const FftLaunch& bucket, hipStream_t st) {
  OnePass a[2], b[2];
  int na, nb;
  if (!pair_passes(comb, bucket, a, b, na, nb)) return hipErrorInvalidValue;
  const int fp32 = comb.tab->is_fp32;
  auto one = [&](const OnePass& p) {
    return fp32 ? dispatch_pass<float>(p.a, p.load, p.store, p.tw, p.tiles, p.batch, st)
                : dispatch_pass<double>(p.a, p.load, p.store, p.tw, p.tiles, p.batch, st);
  };
  for (int p = 0; p < 2; ++p) {
    hipError_t e = hipSuccess;
    if (p < na && p < nb && a[p].tw == b[p].tw) {
      e = fp32 ? pair_pass<float>(a[p], b[p], st) : pair_pass<double>(a[p], b[p], st);
    } else {
      if (p < na) e = one(a[p]);
      if (e == hipSuccess && p < nb) e = one(b[p]);
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t fft_jobs_add(std::vector<FftGroup>& g, const FftLaunch& L) {
  const int fp32 = L.tab->is_fp32;
  return each_pass(L, [&](int p, const PassArgs& A, int load, int store, int tw, int tiles) {
    if (load == kLoadWiden || load == kLoadTaps || load == kLoadRows || store == kStoreHead)
      return hipErrorInvalidValue;
    auto it = std::find_if(g.begin(), g.end(), [&](const FftGroup& x) {
      return x.pass == p && x.load == load && x.store == store && x.tw == tw &&
             x.small_tile == A.small_tile && x.fp32 == fp32;
    });
    if (it == g.end()) {
      FftGroup n;
      n.pass = p;
      n.load = load;
      n.store = store;
      n.tw = tw;
      n.small_tile = A.small_tile;
      n.fp32 = fp32;
      // in the order of the passes
      it = g.insert(std::find_if(g.begin(), g.end(),
                                 [&](const FftGroup& x) { return x.pass > p; }), n);
    }
    FftJob j;
    j.a = A;
    j.tiles = tiles;
    j.block0 = 0;
    it->t.add(j, tiles * L.batch);
    return hipSuccess;
  });
}

template <typename Real, int LOADX, int STORE, int TW>
static hipError_t launch_jobs_tile(const JobsDev& d, hipStream_t st) {
  hipLaunchKernelGGL((fft_jobs_kernel<Real, LOADX, STORE, TW>), dim3(d.blocks),
                     dim3(Tile<Real, LOADX>::nt), 0, st, d);
  return hipGetLastError();
}

template <typename Real, int LOAD, int STORE, int TW>
static hipError_t launch_jobs(const FftGroup& g, hipStream_t st) {
  if constexpr (has_small(LOAD, STORE)) {
    if (g.small_tile) return launch_jobs_tile<Real, LOAD | kSmallTile, STORE, TW>(g.t.dev, st);
  }
  if (g.small_tile) return hipErrorInvalidValue;
  return launch_jobs_tile<Real, LOAD, STORE, TW>(g.t.dev, st);
}

template <typename Real, int LOAD, int TW>
static hipError_t jobs_store(const FftGroup& g, hipStream_t st) {
  // (a batch's combs never start with a plain load)
  constexpr bool keys = occurs(LOAD, kStoreKeys) && !(LOAD == kLoadPlain && TW == kTwNone);
  if (g.store == kStoreCplx) return launch_jobs<Real, LOAD, kStoreCplx, TW>(g, st);
  if constexpr (keys) {
    if (g.store == kStoreKeys) return launch_jobs<Real, LOAD, kStoreKeys, TW>(g, st);
  }
  if constexpr (occurs(LOAD, kStoreBoth)) {
    if (g.store == kStoreBoth) return launch_jobs<Real, LOAD, kStoreBoth, TW>(g, st);
  }
  return hipErrorInvalidValue;
}

template <typename Real>
static hipError_t jobs_pass(const FftGroup& g, hipStream_t st) {
  if (g.load == kLoadComb) return jobs_store<Real, kLoadComb, kTwNone>(g, st);
  if (g.load == kLoadCombRows) return jobs_store<Real, kLoadCombRows, kTwNone>(g, st);
  if (g.load == kLoadCombRowsG) return jobs_store<Real, kLoadCombRowsG, kTwNone>(g, st);
  if (g.load == kLoadPerm) return jobs_store<Real, kLoadPerm, kTwNone>(g, st);
  if (g.load != kLoadPlain) return hipErrorInvalidValue;
  if (g.tw == kTwSplit) return jobs_store<Real, kLoadPlain, kTwSplit>(g, st);
  return jobs_store<Real, kLoadPlain, kTwNone>(g, st);
}

hipError_t fft_jobs_launch(std::vector<FftGroup>& groups, hipStream_t st) {
  for (const FftGroup& g : groups) {
    const hipError_t e = g.fp32 ? jobs_pass<float>(g, st) : jobs_pass<double>(g, st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// ============================================================================================
// permutation + filtering (bucket-owner fold)
// ============================================================================================
// The term as the reference writes it (innerLoop.cu:740-741, 770-771): both products
// rounded, combined, then added to the bucket sum.
// fold_term(x, f) is the tap's product, accumulate() adds a term: add() = both, in that order.
__device__ __forceinline__ double2 fold_term(double2 x, double2 f) {
  return make_double2(x.x * f.x - x.y * f.y, x.x * f.y + x.y * f.x);
}
__device__ __forceinline__ float2 fold_term(float2 x, float2 f) {
  return make_float2(x.x * f.x - x.y * f.y, x.x * f.y + x.y * f.x);
}

struct Acc64 {
  double2 s;
  __device__ __forceinline__ void init() { s = make_double2(0.0, 0.0); }
  __device__ __forceinline__ void accumulate(double2 t) {
    s.x = s.x + t.x;
    s.y = s.y + t.y;
  }
  __device__ __forceinline__ void add(double2 x, double2 f) { accumulate(fold_term(x, f)); }
  __device__ __forceinline__ double2 get() const { return s; }
};

struct Acc32 {  // Kahan-compensated FP32 fold
  float sx, cx, sy, cy;
  __device__ __forceinline__ void init() { sx = cx = sy = cy = 0.f; }
  __device__ __forceinline__ static void kahan(float& sum, float& comp, float term) {
    const float y = term - comp;
    const float t = sum + y;
    comp = (t - sum) - y;
    sum = t;
  }
  __device__ __forceinline__ void accumulate(float2 t) {
    kahan(sx, cx, t.x);
    kahan(sy, cy, t.y);
  }
  __device__ __forceinline__ void add(float2 x, float2 f) { accumulate(fold_term(x, f)); }
  __device__ __forceinline__ float2 get() const { return make_float2(sx, sy); }
};

template <typename Real>
struct AccOf;
template <>
struct AccOf<double> {
  using A = Acc64;
};
template <>
struct AccOf<float> {
  using A = Acc32;
};

constexpr int PF_NT = 256;

// bins[l*B + r] = sum over the taps id of bucket r (canonical order) of v_l(id) * f[id], where
// v_l(id) = x[(id * ai_l) mod n] gathered from the signal (TAPS = false), or read from the
// tap-ordered staging array T[l*w + id] that the streaming pass filled (TAPS = true; same
// values, coalesced reads).  One thread owns bucket r of LPT loops l0 .. l0+LPT-1.  Every
// launch shape (single transform, batch, any LPT or block size) runs this body, so the sums
// are the same bits whatever the shape.
template <typename Real, int LPT, bool TAPS>
__device__ __forceinline__ void pf_body(const typename CT<Real>::T2* __restrict__ x,
                                        const typename CT<Real>::T2* __restrict__ f,
                                        typename CT<Real>::T2* __restrict__ bins,
                                        const int* __restrict__ ai_dev, uint32_t mask, int B,
                                        int w, int loops, int tiled, int r, int l0) {
  using T2 = typename CT<Real>::T2;
  using AC = typename AccOf<Real>::A;
  if (r >= B) return;
  uint32_t ai[LPT];
  const T2* __restrict__ src[LPT];
  AC acc[LPT];
#pragma unroll
  for (int li = 0; li < LPT; ++li) {
    ai[li] = (l0 + li < loops) ? (uint32_t)ai_dev[l0 + li] : 0u;
    src[li] = x + (size_t)min(l0 + li, loops - 1) * (size_t)w;   // staging rows (TAPS)
    acc[li].init();
  }
  auto tap = [&](uint32_t id) {
    const T2 fv = f[id];
    T2 xv[LPT];
#pragma unroll
    for (int li = 0; li < LPT; ++li) xv[li] = TAPS ? src[li][id] : x[(id * ai[li]) & mask];
#pragma unroll
    for (int li = 0; li < LPT; ++li) acc[li].add(xv[li], fv);
  };
  if (tiled) {
    const int T = w / B;
#pragma unroll 2
    for (int t = 0; t < T; ++t) tap((uint32_t)(t * B + r));
    if (r < w - T * B) tap((uint32_t)(r * T + B));
  } else {
#pragma unroll 2
    for (uint32_t id = (uint32_t)r; id < (uint32_t)w; id += (uint32_t)B) tap(id);
  }
#pragma unroll
  for (int li = 0; li < LPT; ++li)
    if (l0 + li < loops) bins[(long long)(l0 + li) * B + r] = acc[li].get();
}

template <typename Real, int LPT, bool TAPS>
__global__ __launch_bounds__(PF_NT) void perm_filter_kernel(
    const typename CT<Real>::T2* __restrict__ x, const typename CT<Real>::T2* __restrict__ f,
    typename CT<Real>::T2* __restrict__ bins, const int* __restrict__ ai_dev, uint32_t mask,
    int B, int w, int loops, int tiled) {
  pf_body<Real, LPT, TAPS>(x, f, bins, ai_dev, mask, B, w, loops, tiled,
                           blockIdx.x * PF_NT + threadIdx.x, blockIdx.y * LPT);
}

template <int LPT, bool TAPS>
static hipError_t pf_launch_lpt(int is_fp32, const void* src, const void* f, void* bins,
                                const int* ai_dev, int n, int B, int w, int loops, int tiled,
                                hipStream_t st) {
  dim3 grid((B + PF_NT - 1) / PF_NT, (loops + LPT - 1) / LPT);
  const uint32_t mask = (uint32_t)n - 1u;
  if (is_fp32)
    hipLaunchKernelGGL((perm_filter_kernel<float, LPT, TAPS>), grid, dim3(PF_NT), 0, st,
                       (const float2*)src, (const float2*)f, (float2*)bins, ai_dev, mask, B, w,
                       loops, tiled);
  else
    hipLaunchKernelGGL((perm_filter_kernel<double, LPT, TAPS>), grid, dim3(PF_NT), 0, st,
                       (const double2*)src, (const double2*)f, (double2*)bins, ai_dev, mask, B,
                       w, loops, tiled);
  return hipGetLastError();
}

// Loops per thread: as many as possible up to 9, split evenly.  One thread then reads each
// filter tap once for all its loops and keeps up to 18 independent gathers in flight (the tap
// loop is unrolled twice); at n = 2^27, k = 16000 (9 loops) this is 7% faster than 3 loops per
// thread.  The sums do not depend on the split.
static int pf_loops_per_thread(int loops) {
  const int groups = (loops + 8) / 9;
  return (loops + groups - 1) / groups;
}

template <bool TAPS>
static hipError_t pf_launch(int is_fp32, const void* src, const void* f, void* bins,
                            const int* ai_dev, int n, int B, int w, int loops, int tiled,
                            hipStream_t st) {
  switch (pf_loops_per_thread(loops)) {
#define SFFT_PF_LPT(k) \
  case k:              \
    return pf_launch_lpt<k, TAPS>(is_fp32, src, f, bins, ai_dev, n, B, w, loops, tiled, st);
    SFFT_PF_LPT(1) SFFT_PF_LPT(2) SFFT_PF_LPT(3) SFFT_PF_LPT(4) SFFT_PF_LPT(5)
    SFFT_PF_LPT(6) SFFT_PF_LPT(7) SFFT_PF_LPT(8) SFFT_PF_LPT(9)
#undef SFFT_PF_LPT
    default:
      return hipErrorInvalidValue;
  }
}

// Batch: the permute+filter of every signal of a batch in one persistent launch.  Work item
// i of job j (item0_j <= i < item0_{j+1}) is bucket block i % nbx of loop group i / nbx;
// the workgroups walk the items with a grid stride (every workgroup runs the same number of
// items +-1, whatever the signal sizes).
template <typename Real, int LPT, int NT>
__global__ __launch_bounds__(NT) void perm_filter_batch_kernel(const PfJob* __restrict__ jobs,
                                                               int njobs, int total) {
  using T2 = typename CT<Real>::T2;
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (jobs[mid].item0 <= item) lo = mid;
      else hi = mid - 1;
    }
    const PfJob& J = jobs[lo];
    const int local = item - J.item0;
    const int bx = local % J.nbx, gy = local / J.nbx;
    pf_body<Real, LPT, false>((const T2*)J.x, (const T2*)J.f, (T2*)J.bins, J.ai, J.mask, J.B,
                              J.w, J.loops, J.tiled, bx * NT + threadIdx.x, gy * LPT);
  }
}

int pf_batch_items(int B, int loops, int lpt, int nt, int* nbx) {
  *nbx = (B + nt - 1) / nt;
  return *nbx * ((loops + lpt - 1) / lpt);
}

template <typename Real, int LPT>
static hipError_t pfb_nt(const PfJob* jobs, int njobs, int total, int nt, int grid,
                         hipStream_t st) {
  if (nt == 128)
    hipLaunchKernelGGL((perm_filter_batch_kernel<Real, LPT, 128>), dim3(grid), dim3(128), 0, st,
                       jobs, njobs, total);
  else if (nt == 256)
    hipLaunchKernelGGL((perm_filter_batch_kernel<Real, LPT, 256>), dim3(grid), dim3(256), 0, st,
                       jobs, njobs, total);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <typename Real>
static hipError_t pfb_lpt(const PfJob* jobs, int njobs, int total, int lpt, int nt, int grid,
                          hipStream_t st) {
  switch (lpt) {
    case 1: return pfb_nt<Real, 1>(jobs, njobs, total, nt, grid, st);
    case 2: return pfb_nt<Real, 2>(jobs, njobs, total, nt, grid, st);
    case 3: return pfb_nt<Real, 3>(jobs, njobs, total, nt, grid, st);
    case 4: return pfb_nt<Real, 4>(jobs, njobs, total, nt, grid, st);
    case 5: return pfb_nt<Real, 5>(jobs, njobs, total, nt, grid, st);
    case 6: return pfb_nt<Real, 6>(jobs, njobs, total, nt, grid, st);
    case 7: return pfb_nt<Real, 7>(jobs, njobs, total, nt, grid, st);
    case 8: return pfb_nt<Real, 8>(jobs, njobs, total, nt, grid, st);
    case 9: return pfb_nt<Real, 9>(jobs, njobs, total, nt, grid, st);
  }
  return hipErrorInvalidValue;
}

hipError_t perm_filter_batch_launch(int is_fp32, const PfJob* d_jobs, int njobs, int total,
                                    int lpt, int nt, int grid, hipStream_t st) {
  if (njobs <= 0 || total <= 0) return hipSuccess;
  if (grid > total) grid = total;
  return is_fp32 ? pfb_lpt<float>(d_jobs, njobs, total, lpt, nt, grid, st)
                 : pfb_lpt<double>(d_jobs, njobs, total, lpt, nt, grid, st);
}

hipError_t perm_filter_launch(int is_fp32, const void* x, const void* f, void* bins,
                              const int* ai_dev, int n, int B, int w, int loops, int tiled,
                              hipStream_t st) {
  return pf_launch<false>(is_fp32, x, f, bins, ai_dev, n, B, w, loops, tiled, st);
}

hipError_t fold_taps_launch(int is_fp32, const void* T, const void* f, void* bins,
                            const int* ai_dev, int n, int B, int w, int loops, int tiled,
                            hipStream_t st) {
  return pf_launch<true>(is_fp32, T, f, bins, ai_dev, n, B, w, loops, tiled, st);
}

// ============================================================================================
// column-ordered fold
//
// View x as m = n/B rows of B columns (x[row*B + col]).  Every tap id = t*B + r of bucket r in
// loop l gathers x[(id*ai_l) mod n], whose column is (id*ai_l) mod B = (r*ai_l) mod B: all the
// taps of a bucket lie in ONE column, c = r*ai_l mod B, and conversely column c holds bucket
// r = c*a_l mod B of loop l.  A workgroup that owns a block of adjacent columns for every loop
// therefore gathers only from the 128-byte lines of those columns, and the taps of different
// loops that land in the same line share one fetch (at n = 2^27, k = 16000: 20.1 M taps over
// 8.4 M lines of complex64, 16.8 M of complex128).  The filter taps of bucket r are read from
// a bucket-major copy fT[r*P + t] (one contiguous row per bucket, built by filter_rows_kernel
// when the filter is set), since the buckets of one column block are scattered over r.
// Each thread owns one (loop, column) pair and sums its bucket's taps in the canonical order
// (t ascending, then the reference's tail tap when tiled), so the sums are the bits of
// pf_body.
// The comb samples y_r[j] = x[off_r + j*sigma] (sigma = n/W divides B) are the columns
// c = off_r mod sigma + lo*sigma of the same view: sample j = row*(B/sigma) + lo.  The threads
// of a column block also copy the comb columns that fall in it, while its lines are being
// fetched for the taps, into column-major rows yc[r*W + lo*m + row] (m contiguous samples per
// comb column); the comb FFT's first pass loads them with kLoadCombRows.
// ============================================================================================
constexpr int FC_NT = 256;
constexpr int FC_CHUNK = 8;   // taps whose loads are issued together

// fT[r*P + t]: row r holds the taps of bucket r in summation order: t*B + r for t < T, then at
// t = T the tiled fold's tail tap r*T + B (tiled, r < w - T*B) or the last full-fold tap T*B + r
// (r < w - T*B); zero elsewhere.  T = w / B.
template <typename T2>
__global__ void filter_rows_kernel(const T2* __restrict__ f, T2* __restrict__ fT, int B, int w,
                                   int T, int P, int tiled) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)B * P) return;
  const int r = (int)(i / P), t = (int)(i % P);
  const int residue = w - T * B;
  long long id = -1;
  if (t < T) id = (long long)t * B + r;
  else if (t == T && r < residue) id = tiled ? (long long)r * T + B : (long long)T * B + r;
  T2 v;
  v.x = 0;
  v.y = 0;
  fT[i] = (id >= 0) ? f[id] : v;
}

template <typename Real>
__global__ __launch_bounds__(FC_NT) void fold_columns_kernel(
    const typename CT<Real>::T2* __restrict__ x, const typename CT<Real>::T2* __restrict__ fT,
    typename CT<Real>::T2* __restrict__ bins, const int* __restrict__ a_dev,
    const int* __restrict__ ai_dev, uint32_t mask, int log2B, int w, int loops, int tiled,
    int T, int P, int log2lw, int remap, typename CT<Real>::T2* __restrict__ yc,
    const int* __restrict__ offs, int Rl, int log2sigma, int log2m) {
  using T2 = typename CT<Real>::T2;
  using AC = typename AccOf<Real>::A;
  const int blk = remap ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const uint32_t item = (uint32_t)blk * FC_NT + threadIdx.x;
  const uint32_t B = 1u << log2B;
  if (item >= (uint32_t)loops * B) return;
  // item = ((column block * loops + l) << log2lw) | column within the block
  const uint32_t lw = 1u << log2lw;
  const uint32_t cc = item & (lw - 1u), rest = item >> log2lw;
  const uint32_t l = rest % (uint32_t)loops, cb = rest / (uint32_t)loops;
  const uint32_t c = (cb << log2lw) | cc;
  const uint32_t ai = (uint32_t)ai_dev[l];
  const uint32_t r = (c * (uint32_t)a_dev[l]) & (B - 1u);
  const int residue = w - T * (int)B;
  // main taps t*B + r: T of them, T+1 for the full fold's r < residue
  const int nmain = (!tiled && (int)r < residue) ? T + 1 : T;
  const uint32_t base = (r * ai) & mask, step = (B * ai) & mask;
  const T2* __restrict__ frow = fT + (size_t)r * (size_t)P;
  AC acc;
  acc.init();
  for (int t0 = 0; t0 < nmain; t0 += FC_CHUNK) {
    T2 xv[FC_CHUNK], fv[FC_CHUNK];
#pragma unroll
    for (int k = 0; k < FC_CHUNK; ++k) {
      const int t = t0 + k;
      if (t < nmain) {
        xv[k] = x[(base + (uint32_t)t * step) & mask];
        fv[k] = frow[t];
      }
    }
#pragma unroll
    for (int k = 0; k < FC_CHUNK; ++k)
      if (t0 + k < nmain) acc.add(xv[k], fv[k]);
  }
  if (tiled && (int)r < residue) {   // the reference's tail tap of its tiled fold (n < 2^27): another column
    const uint32_t id = r * (uint32_t)T + B;
    acc.add(x[(id * ai) & mask], frow[T]);
  }
  bins[(size_t)l * B + r] = acc.get();
  // comb columns of this column block: rank-strided rows, contiguous stores
  const uint32_t rank = (l << log2lw) | cc, G = (uint32_t)loops << log2lw;
  const uint32_t c0 = cb << log2lw, smask = (1u << log2sigma) - 1u, m = 1u << log2m;
  const size_t W = (size_t)B << log2m >> log2sigma;
  for (int rr = 0; rr < Rl; ++rr) {
    const uint32_t o = (uint32_t)offs[rr];
    for (uint32_t col = c0 + ((o - c0) & smask); col < c0 + lw; col += smask + 1u) {
      T2* __restrict__ dst = yc + (size_t)rr * W + ((size_t)(col >> log2sigma) << log2m);
#pragma unroll 4
      for (uint32_t row = rank; row < m; row += G) dst[row] = x[((size_t)row << log2B) | col];
    }
  }
}

// LDS-staged column fold.  A slab is SC adjacent columns (SC * e = 256 bytes, two 128-byte
// lines per row: narrower slabs read at a power-of-two row stride reach only half the bandwidth
// on MI355X) over all m rows of the view.  A workgroup streams its slabs (s, s + G, s + 2G, ...
// for a grid of G resident workgroups) through LDS in chunks of SL_ROWS rows with 16-byte loads;
// the next chunk's loads, also across a slab boundary, are in flight in registers while the
// current chunk is used, so the stream does not stop between slabs: across the grid the whole
// signal is read once.  For each slab the workgroup holds the filter rows of the buckets of its
// (loop, column) pairs in an LDS tap array (slot t of pair p at t * pairs + p; the next slab's
// rows are fetched while the current slab is finished).  As the rows of its taps pass (tap t
// lies in row ((r*ai + t*B*ai) mod n) / B), the thread of pair p replaces slot t by the tap's
// product term x * f; after the slab's last chunk it adds its slots up in the canonical order.
// The bucket sums are written in column order (bins[l*B + c] for the bucket r = c*a_l mod B of
// column c: whole segments instead of scattered 8/16-byte stores); the bucket FFT reads them
// back through that permutation (kLoadPerm).  The comb columns of the slab are copied out of
// each chunk.  Same per-bucket terms and order as pf_body: the same bits.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int SL_ROWS = 128;  // rows per chunk
constexpr int SL_PITCH = 17;  // 16-byte units per chunk row: 256 bytes + 16 of padding (banks)
constexpr int SL_U = 4;       // 16-byte loads per thread for one chunk (512 threads)
constexpr int SL_TABLE = 128; // LDS ints after the slots: a [0,32), ai [32,64), comb offsets [64,128)
template <typename Real>
struct SlabFetch {            // filter-row loads per thread per slab (all in flight together)
  static constexpr int fb = sizeof(Real) == 8 ? 8 : 16;
};

// (workgroup bx of the G that share the signal's slabs; DV: the draws are dv's, else in memory)
template <typename Real, int PMAX, int NT, bool DV>
__device__ __forceinline__ void fold_slab_body(const SlabArgs& A, const DrawVals& dv, uint32_t bx,
                                               uint32_t G) {
  using T2 = typename CT<Real>::T2;
  using V2 = typename NV<Real>::type;
  using AC = typename AccOf<Real>::A;
  const T2* __restrict__ x = (const T2*)A.x;
  const T2* __restrict__ fT = (const T2*)A.fT;
  T2* __restrict__ bins = (T2*)A.bins;
  T2* __restrict__ yc = (T2*)A.yc;
  const uint32_t mask = A.mask;
  const int log2B = A.log2B, log2m = A.log2m, w = A.w, loops = A.loops, tiled = A.tiled, T = A.T,
            P = A.P, log2sc = A.log2sc, Rl = A.Rl, log2sigma = A.log2sigma;
  const FoldClear& clr = A.clr;
  constexpr int EPU = 16 / (int)sizeof(T2);             // elements per 16-byte unit
  constexpr int FB = SlabFetch<Real>::fb;
  extern __shared__ u32x4 dyn16[];
  u32x4* chunk16 = dyn16;                              // SL_ROWS x SL_PITCH units
  const V2* ldsv = (const V2*)dyn16;                   // element (row, k): row*PITCH*EPU + k
  V2* slotv = (V2*)(dyn16 + SL_ROWS * SL_PITCH);       // P x pairs slots
  const int pairs = loops << log2sc;
  int* atab = (int*)(slotv + (size_t)P * pairs);       // SL_TABLE ints
  const int tid = threadIdx.x;
  const uint32_t B = 1u << log2B, SC = 1u << log2sc;
  const uint32_t nslabs = B >> log2sc;
  const bool active = tid < pairs;
  const uint32_t cc = (uint32_t)tid & (SC - 1u), l = (uint32_t)tid >> log2sc;
  const int residue = w - T * (int)B;
  const int log2rows = log2m < 7 ? log2m : 7;          // SL_ROWS = 2^7
  const int rows = 1 << log2rows;
  const int nchunks = 1 << (log2m - log2rows);
  const int units = rows * 16;                         // 16-byte units of x per chunk
  const u32x4* __restrict__ x16 = (const u32x4*)x;
  const uint32_t row16 = (uint32_t)(((size_t)B * sizeof(T2)) / 16);
  const uint32_t smask = (1u << log2sigma) - 1u;
  const size_t W = (size_t)B << log2m >> log2sigma;
  // comb columns of a slab per comb loop: SC / sigma when sigma < SC, else at most one
  const int log2ncs = log2sc > log2sigma ? log2sc - log2sigma : 0;
  const int ncopy = (Rl << log2ncs) << log2rows;       // comb copy elements per chunk
  const int total = P * pairs;                         // filter slots (at most FB * NT)
  const uint32_t magic = P > 1 ? 0xFFFFFFFFu / (uint32_t)P + 1u : 0u;   // k / P = umulhi(k, magic)
  const V2* __restrict__ fTv = (const V2*)fT;

  // The chunks of the workgroup in order: chunk q is chunk (q mod nchunks) of its slab
  // q / nchunks (slab bx + (q / nchunks) * G).  The next chunk is in flight in
  // registers (xa) while one is used from LDS.  q past the last chunk is clamped to it.
  const int log2nch = log2m - log2rows;
  const int nsl = (int)((nslabs - bx + G - 1) / G);   // slabs of this workgroup
  const int Q = nsl << log2nch;
  u32x4 xa[SL_U];
  // the loads of a chunk in one basic block (clamped addresses): in flight together.  Unit
  // indices in 32 bits (n * e / 16 < 2^32).
  auto load = [&](u32x4* buf, int q) __attribute__((always_inline)) {
    const int qq = min(q, Q - 1);
    const uint32_t c0 = (bx + (uint32_t)(qq >> log2nch) * G) << log2sc;
    const int ch = qq & (nchunks - 1);
    const uint32_t col16 = (uint32_t)(((size_t)c0 * sizeof(T2)) / 16);
#pragma unroll
    for (int u = 0; u < SL_U; ++u) {
      const int i = min(u * NT + tid, units - 1);
      const uint32_t unit =
          ((uint32_t)(ch * rows) + (uint32_t)(i >> 4)) * row16 + col16 + (uint32_t)(i & 15);
      buf[u] = __builtin_nontemporal_load(&x16[unit]);
    }
  };
  // every thread stores every one of its units (a clamped one again, with the same value), so
  // that all of the chunk's loads are known to be complete here
  auto store = [&](const u32x4* buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < SL_U; ++u) {
      const int i = min(u * NT + tid, units - 1);
      chunk16[(i >> 4) * SL_PITCH + (i & 15)] = buf[u];
    }
  };
  // the filter rows of a slab's pairs: entry k = p * P + t of the fetch (entry t of pair p's
  // row; neighbouring threads read neighbouring entries of a row) goes to slot t * pairs + p;
  // any thread any entry (clamped addresses; the loads in flight together)
  V2 fv[FB];
  auto entry = [&](int u, int tv, int& p, int& t) __attribute__((always_inline)) {
    const int k = min(u * NT + tv, total - 1);
    p = P > 1 ? (int)__umulhi((uint32_t)k, magic) : k;
    t = k - p * P;
  };
  auto fetch_rows = [&](uint32_t c0) __attribute__((always_inline)) {
    int tv = tid;
    asm volatile("" : "+v"(tv));   // entry indices recomputed here, not kept in registers
#pragma unroll
    for (int u = 0; u < FB; ++u) {
      int p, t;
      entry(u, tv, p, t);
      const uint32_t rp =
          ((c0 + ((uint32_t)p & (SC - 1u))) * (uint32_t)atab[p >> log2sc]) & (B - 1u);
      fv[u] = fTv[(size_t)rp * (size_t)P + (size_t)t];
    }
  };
  // (a clamped entry is stored again with its own value: every load is known complete here)
  auto put_rows = [&]() __attribute__((always_inline)) {
    int tv = tid;
    asm volatile("" : "+v"(tv));
#pragma unroll
    for (int u = 0; u < FB; ++u) {
      int p, t;
      entry(u, tv, p, t);
      slotv[t * pairs + p] = fv[u];
    }
  };
  uint32_t r = 0, ai = 0, base = 0, step = 0;
  int nmain = 0;
  auto pair_state = [&](uint32_t c0) __attribute__((always_inline)) {
    if (active) {
      ai = (uint32_t)atab[32 + l];
      r = ((c0 + cc) * (uint32_t)atab[l]) & (B - 1u);
      nmain = (!tiled && (int)r < residue) ? T + 1 : T;
      base = (r * ai) & mask;
      step = (B * ai) & mask;
    }
  };

  // (a, ai) of every loop and the comb offsets into LDS: their loads go out before the first
  // chunk's, so that waiting for them does not wait for the chunk
  // the caller's clear, spread over the grid (one 4-byte store per thread at n = 2^27)
  for (size_t i = (size_t)bx * NT + tid; i < clr.nbm; i += (size_t)G * NT)
    clr.bm[i] = 0u;
  if (bx == 0 && tid < clr.nmax) clr.maxf[tid] = 0xFFFFFFFFu;
  int av = 0, aiv = 0, ov = 0;
  if (tid < loops) {
    av = DV && dv.count ? dv.v[tid] : A.a_dev[tid];
    aiv = DV && dv.count ? dv.v[loops + tid] : A.ai_dev[tid];
  }
  if (tid < Rl) ov = DV && dv.count ? dv.v[2 * loops + tid] : A.offs[tid];
  if (DV && bx == 0 && tid < dv.count) dv.out[tid] = dv.v[tid];
  load(xa, 0);
  if (tid < loops) {
    atab[tid] = av;
    atab[32 + tid] = aiv;
  }
  if (tid < Rl) atab[64 + tid] = ov;
  __syncthreads();
  fetch_rows(bx << log2sc);
  put_rows();
  pair_state(bx << log2sc);
  store(xa);
  __syncthreads();

  // chunk q from LDS while chunk q + 1 is on its way.  Every load and store is issued on every
  // call (the clamped chunk past the end again): no path on which a load could still be in
  // flight, so the compiler adds no waits for one.
  auto body = [&](int q) __attribute__((always_inline)) {
    const int ch = q & (nchunks - 1);
    const int sl = q >> log2nch;
    const uint32_t c0 = (bx + (uint32_t)sl * G) << log2sc;
    const uint32_t cnext = (bx + (uint32_t)min(sl + 1, nsl - 1) * G) << log2sc;
    const uint32_t r0 = (uint32_t)(ch * rows);
    // comb columns of the slab: this chunk's rows
    for (int e = tid; e < ncopy; e += NT) {
      const int row = e & (rows - 1);
      const int ci = e >> log2rows;
      const int rr = ci >> log2ncs;
      const uint32_t col = c0 + (((uint32_t)atab[64 + rr] - c0) & smask) +
                           ((uint32_t)(ci & ((1 << log2ncs) - 1)) << log2sigma);
      if (col < c0 + SC) {
        V2* __restrict__ dst = (V2*)yc + (size_t)rr * W +
                               ((size_t)(col >> log2sigma) << log2m) + r0 + (uint32_t)row;
        *dst = ldsv[row * (SL_PITCH * EPU) + (int)(col - c0)];
      }
    }
    load(xa, q + 1);
    if (active) {
      // the taps whose rows fall in this chunk (a bit per tap): slot t becomes x * f (tap
      // rows recomputed per chunk, not kept in registers)
      uint32_t bs = base, sp = step;
      int nm = nmain;
      asm volatile("" : "+v"(bs), "+v"(sp), "+v"(nm));
      uint32_t hits = 0;   // built from the top tap down (no per-tap bit constants)
#pragma unroll
      for (int t = PMAX - 1; t >= 0; --t) {
        const uint32_t row = ((bs + (uint32_t)t * sp) & mask) >> log2B;
        hits = (hits << 1) | (uint32_t)(t < nm && row - r0 < (uint32_t)rows);
      }
      while (hits) {
        const int t = __ffs(hits) - 1;
        hits &= hits - 1u;
        const uint32_t row = ((bs + (uint32_t)t * sp) & mask) >> log2B;
        const V2 xv = ldsv[(row - r0) * (SL_PITCH * EPU) + cc];
        const V2 fw = slotv[t * pairs + tid];
        T2 xt, ft;
        xt.x = xv.x;
        xt.y = xv.y;
        ft.x = fw.x;
        ft.y = fw.y;
        const T2 term = fold_term(xt, ft);
        V2 tv;
        tv.x = term.x;
        tv.y = term.y;
        slotv[t * pairs + tid] = tv;
      }
    }
    __syncthreads();
    if (ch == nchunks - 1) {
      // the slab is done: the next slab's filter rows go out (the current slab's again after
      // the workgroup's last slab), this slab's buckets are summed and written while they
      // arrive
      fetch_rows(cnext);
      if (active) {
        int tv = tid;
        asm volatile("" : "+v"(tv));   // slot addresses recomputed here
        AC acc;
        acc.init();
        // the slots in batches of SB reads in flight together (clamped), added up in order
        constexpr int SB = sizeof(Real) == 8 ? 4 : 8;
#pragma unroll
        for (int t0 = 0; t0 < PMAX; t0 += SB) {
          V2 sv[SB];
#pragma unroll
          for (int j = 0; j < SB; ++j) sv[j] = slotv[min(t0 + j, P - 1) * pairs + tv];
#pragma unroll
          for (int j = 0; j < SB; ++j) {
            if (t0 + j < nmain) {
              T2 term;
              term.x = sv[j].x;
              term.y = sv[j].y;
              acc.accumulate(term);
            }
          }
        }
        if (tiled && (int)r < residue) {   // the reference's tail tap of its tiled fold (n < 2^27): another column
          const uint32_t id = r * (uint32_t)T + B;
          acc.add(x[(id * ai) & mask], fT[(size_t)r * (size_t)P + T]);
        }
        bins[(size_t)l * B + c0 + cc] = acc.get();   // column order: whole segments
      }
      __syncthreads();   // every slot read
      put_rows();
      pair_state(cnext);
    }
    store(xa);
    __syncthreads();
  };
#pragma unroll 1
  for (int q = 0; q < Q; ++q) body(q);
}

template <typename Real, int PMAX, int NT>
__global__ __launch_bounds__(NT, 4) void fold_slab_kernel(SlabArgs A, DrawVals dv) {
  fold_slab_body<Real, PMAX, NT, true>(A, dv, blockIdx.x, gridDim.x);
}

// the slabs of many signals: a signal's workgroups stream its slabs, as in a launch of their own
template <typename Real, int PMAX, int NT>
__global__ __launch_bounds__(NT, 4) void fold_slab_jobs_kernel(JobsDev t) {
  const SlabJob* j = job_here<SlabJob>(t);
  if (!j) return;
  const SlabArgs A = j->a;
  fold_slab_body<Real, PMAX, NT, false>(A, DrawVals(), blockIdx.x - (uint32_t)j->block0,
                                        (uint32_t)j->groups);
}

int fold_rows_pitch(int B, int w) { return w / B + 1; }

static size_t slab_lds_bytes(int is_fp32, int loops, int lsc, int P) {
  return (size_t)SL_ROWS * SL_PITCH * 16 + (size_t)P * ((size_t)loops << lsc) * (is_fp32 ? 8 : 16) +
         SL_TABLE * sizeof(int);   // chunk, tap slots, (a, ai) of up to 32 loops, comb offsets
}

// columns per slab (log2) for the LDS-staged fold, or -1 when it does not apply: 256-byte row
// segments, at most 512 (loop, column) threads, at most 32 taps per bucket, at most 96 KB of
// LDS (chunk + tap slots)
static int slab_log2sc(int is_fp32, int log2B, int log2m, int loops, int P) {
  const int lsc = is_fp32 ? 5 : 4;
  (void)log2m;
  if (lsc > log2B) return -1;
  if ((loops << lsc) > 512 || P > 32) return -1;
  // every filter slot of a slab fetched by one round of loads
  const int fb = is_fp32 ? SlabFetch<float>::fb : SlabFetch<double>::fb;
  if (P * (loops << lsc) > fb * 512) return -1;
  if (slab_lds_bytes(is_fp32, loops, lsc, P) > 96 * 1024) return -1;
  return lsc;
}

// resident workgroups of a slab kernel on the current device: asked of the runtime once per
// (kernel, device, LDS size) and kept; 0 where it cannot be asked
static int slab_resident(const void* kernel, int nt, size_t lds) {
  static std::mutex mu;
  static std::map<std::pair<const void*, std::pair<int, size_t>>, int> resident;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(mu);
  const std::pair<const void*, std::pair<int, size_t>> key(kernel, {dev, lds});
  auto it = resident.find(key);
  if (it == resident.end()) {
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, nt, lds) != hipSuccess)
      cus = per_cu = 0;
    it = resident.emplace(key, cus * per_cu).first;
  }
  return it->second;
}

// 512 threads per workgroup: two chunks of loads in flight per workgroup at 4 loads per thread
constexpr int SL_NT = 512;

// taps per bucket of the kernel variant that takes P
static int slab_pmax(int P) { return P <= 16 ? 16 : P <= 24 ? 24 : 32; }

// f(kernel of one signal, kernel of many) for the taps per bucket
template <typename Real, typename F>
static hipError_t with_pmax(int pmax, F&& f) {
  if (pmax == 16)
    return f(fold_slab_kernel<Real, 16, SL_NT>, fold_slab_jobs_kernel<Real, 16, SL_NT>);
  if (pmax == 24)
    return f(fold_slab_kernel<Real, 24, SL_NT>, fold_slab_jobs_kernel<Real, 24, SL_NT>);
  return f(fold_slab_kernel<Real, 32, SL_NT>, fold_slab_jobs_kernel<Real, 32, SL_NT>);
}

static size_t slab_lds(int is_fp32, const SlabArgs& A) {
  return slab_lds_bytes(is_fp32, A.loops, A.log2sc, A.P);
}

// one workgroup per resident slot (each streams nslabs / grid slabs); any grid is correct
template <typename Real>
static hipError_t slab_launch(const SlabArgs& A, const DrawVals& dv, hipStream_t st) {
  const unsigned nslabs = 1u << (A.log2B - A.log2sc);
  const size_t lds = slab_lds(sizeof(Real) == 4, A);
  return with_pmax<Real>(slab_pmax(A.P), [&](auto one, auto) {
    const int res = slab_resident(reinterpret_cast<const void*>(one), SL_NT, lds);
    const unsigned blocks = res > 0 ? std::min(nslabs, (unsigned)res) : nslabs;
    hipLaunchKernelGGL(one, dim3(blocks), dim3(SL_NT), lds, st, A, dv);
    return hipGetLastError();
  });
}

int fold_slab_applies(int is_fp32, int n, int B, int w, int loops) {
  int log2B = 0, log2n = 0;
  while ((1 << log2B) < B) ++log2B;
  while ((1LL << log2n) < n) ++log2n;
  return slab_log2sc(is_fp32, log2B, log2n - log2B, loops, fold_rows_pitch(B, w)) >= 0;
}

hipError_t filter_rows_launch(int is_fp32, const void* f, void* fT, int B, int w, int tiled,
                              hipStream_t st) {
  const int T = w / B, P = fold_rows_pitch(B, w);
  const long long total = (long long)B * P;
  const unsigned blocks = (unsigned)((total + 255) / 256);
  if (is_fp32)
    hipLaunchKernelGGL(filter_rows_kernel<float2>, dim3(blocks), dim3(256), 0, st,
                       (const float2*)f, (float2*)fT, B, w, T, P, tiled);
  else
    hipLaunchKernelGGL(filter_rows_kernel<double2>, dim3(blocks), dim3(256), 0, st,
                       (const double2*)f, (double2*)fT, B, w, T, P, tiled);
  return hipGetLastError();
}

// the slab fold's arguments; false where the slab does not apply
static bool slab_args(SlabArgs& A, int is_fp32, const void* x, const void* fT, void* bins,
                      const int* a_dev, const int* ai_dev, int n, int B, int w, int loops,
                      int tiled, void* yc, const int* offs, int Rl, int W, const FoldClear& clr) {
  int log2B = 0, log2n = 0, log2W = 0;
  while ((1 << log2B) < B) ++log2B;
  while ((1LL << log2n) < n) ++log2n;
  while ((1 << log2W) < W) ++log2W;
  A = SlabArgs();
  A.x = x;
  A.fT = fT;
  A.bins = bins;
  A.a_dev = a_dev;
  A.ai_dev = ai_dev;
  A.mask = (uint32_t)n - 1u;
  A.log2B = log2B;
  A.log2m = log2n - log2B;
  A.w = w;
  A.loops = loops;
  A.tiled = tiled;
  A.T = w / B;
  A.P = fold_rows_pitch(B, w);
  A.yc = yc;
  A.offs = offs;
  A.log2sigma = log2n - log2W;
  A.Rl = (!yc || A.log2sigma > log2B) ? 0 : Rl;   // no comb columns to copy (sigma must divide B)
  A.clr = clr;
  const int lsc = A.Rl <= 64 ? slab_log2sc(is_fp32, log2B, A.log2m, loops, A.P) : -1;
  A.log2sc = lsc;
  return lsc >= 0;
}

hipError_t slab_jobs_add(std::vector<SlabGroup>& groups, int is_fp32, const void* x,
                         const void* fT, void* bins, const int* a_dev, const int* ai_dev, int n, int B, int w, int loops,
                         int tiled, void* yc, const int* offs, int Rl, int W,
                         const FoldClear& clr) {
  SlabArgs A;
  if (!slab_args(A, is_fp32, x, fT, bins, a_dev, ai_dev, n, B, w, loops, tiled, yc, offs, Rl, W,
                 clr))
    return hipErrorInvalidValue;
  // (signals whose slabs are over half a CU's LDS apart: they would leave every signal of the
  // launch one workgroup per CU)
  const size_t lds = slab_lds(is_fp32, A);
  const int wide = lds > 80 * 1024;
  auto it = std::find_if(groups.begin(), groups.end(),
                         [&](const SlabGroup& g) { return g.wide == wide; });
  if (it == groups.end()) {
    groups.emplace_back();
    it = groups.end() - 1;
    it->wide = wide;
    it->fp32 = is_fp32;
  }
  it->pmax = std::max(it->pmax, slab_pmax(A.P));
  it->lds = std::max(it->lds, lds);
  it->args.push_back(A);
  return hipSuccess;
}

// Workgroups of a quarter of a resident slot's even share each (a slab at least), the longest
// streams first: the card deals the rest to the slots that come free, so that slabs of 16 KB
// (2^18 points) and of 4 MB (2^24) leave no slot with a long tail.  (As many workgroups as slots,
// shared out by bytes: signals of 32 slabs on 28 workgroups stream two slabs on some, 64 complex64
// signals of 2^18..2^24 1571 us, now 763.)
static void share_group(SlabGroup& g) {
  const int n = (int)g.args.size();
  if (!n) return;
  int res = 0;
  auto ask = [&](auto, auto many) {
    res = slab_resident(reinterpret_cast<const void*>(many), SL_NT, g.lds);
    return hipSuccess;
  };
  (void)(g.fp32 ? with_pmax<float>(g.pmax, ask) : with_pmax<double>(g.pmax, ask));
  auto slabs = [&](int i) { return 1LL << (g.args[i].log2B - g.args[i].log2sc); };
  auto rows = [&](int i) { return 1LL << g.args[i].log2m; };   // of 256 bytes per slab
  long long total = 0;
  for (int i = 0; i < n; ++i) total += slabs(i) * rows(i);
  const long long part = total / (4 * (res > 0 ? res : 512)) + 1;
  std::vector<long long> per(n);   // slabs per workgroup
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) {
    per[i] = std::max(1LL, part / rows(i));
    order[i] = i;
  }
  std::stable_sort(order.begin(), order.end(),
                   [&](int i, int j) { return per[i] * rows(i) > per[j] * rows(j); });
  for (int i : order) {
    SlabJob j;
    j.a = g.args[i];
    j.groups = (int)((slabs(i) + per[i] - 1) / per[i]);
    j.block0 = 0;
    g.t.add(j, j.groups);
  }
}

void slab_jobs_share(std::vector<SlabGroup>& groups) {
  for (SlabGroup& g : groups) share_group(g);
}

hipError_t slab_jobs_launch(const std::vector<SlabGroup>& groups, hipStream_t st) {
  for (const SlabGroup& g : groups) {
    auto go = [&](auto, auto many) {
      hipLaunchKernelGGL(many, dim3(g.t.dev.blocks), dim3(SL_NT), g.lds, st, g.t.dev);
      return hipGetLastError();
    };
    const hipError_t e = g.fp32 ? with_pmax<float>(g.pmax, go) : with_pmax<double>(g.pmax, go);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t fold_columns_launch(int is_fp32, const void* x, const void* fT, void* bins,
                               const int* a_dev, const int* ai_dev, int n, int B, int w,
                               int loops, int tiled, int by_column, int remap, void* yc,
                               const int* offs, int Rl, int W, const FoldClear& clr,
                               const DrawVals& dv, hipStream_t st) {
  SlabArgs A;
  const bool slab = slab_args(A, is_fp32, x, fT, bins, a_dev, ai_dev, n, B, w, loops, tiled, yc,
                              offs, Rl, W, clr);
  if (by_column) {
    if (!slab || (dv.count && dv.count != 2 * loops + A.Rl)) return hipErrorInvalidValue;
    return is_fp32 ? slab_launch<float>(A, dv, st) : slab_launch<double>(A, dv, st);
  }
  const int log2B = A.log2B, log2m = A.log2m, log2sigma = A.log2sigma, T = A.T, P = A.P;
  const uint32_t mask = A.mask;
  Rl = A.Rl;
  // only the slab fold clears and takes the draws
  if (clr.nbm || clr.nmax || dv.count) return hipErrorInvalidValue;
  // columns per block: one 128-byte line of x (8 complex128 / 16 complex64), fewer if B is
  // smaller
  int log2lw = is_fp32 ? 4 : 3;
  if (log2lw > log2B) log2lw = log2B;
  const long long total = (long long)loops * B;
  const unsigned blocks = (unsigned)((total + FC_NT - 1) / FC_NT);
  if (remap < 0) remap = 1;
  if (is_fp32)
    hipLaunchKernelGGL(fold_columns_kernel<float>, dim3(blocks), dim3(FC_NT), 0, st,
                       (const float2*)x, (const float2*)fT, (float2*)bins, a_dev, ai_dev, mask,
                       log2B, w, loops, tiled, T, P, log2lw, remap, (float2*)yc, offs, Rl,
                       log2sigma, log2m);
  else
    hipLaunchKernelGGL(fold_columns_kernel<double>, dim3(blocks), dim3(FC_NT), 0, st,
                       (const double2*)x, (const double2*)fT, (double2*)bins, a_dev, ai_dev,
                       mask, log2B, w, loops, tiled, T, P, log2lw, remap, (double2*)yc, offs,
                       Rl, log2sigma, log2m);
  return hipGetLastError();
}

// ============================================================================================
// streaming pass: read the signal once in address order and route every element to the tap
// slots and comb samples that use it:
//   T[l*w + i] = x[m]  for each loop l with i = (m * a_l) mod n < w   (i.e. m = i * ai_l)
//   y[r*W + j] = x[m]  for each comb r with m = off_r + j * sigma
// Each thread handles SS_EPT consecutive elements; i advances by a_l per element (no multiply).
// ============================================================================================
constexpr int SS_NT = 256;
constexpr int SS_EPT = 4;

template <typename T2>
__global__ __launch_bounds__(SS_NT) void stream_scatter_kernel(
    const T2* __restrict__ x, T2* __restrict__ T, T2* __restrict__ y,
    const int* __restrict__ a_dev, const int* __restrict__ offs, uint32_t n, uint32_t w,
    int loops, int Rl, int log2sigma, uint32_t W) {
  const uint32_t mask = n - 1u;
  const uint32_t m0 = (blockIdx.x * SS_NT + threadIdx.x) * SS_EPT;
  if (m0 >= n) return;
  T2 v[SS_EPT];
#pragma unroll
  for (int e = 0; e < SS_EPT; ++e) v[e] = x[m0 + e];
  for (int l = 0; l < loops; ++l) {
    const uint32_t a = (uint32_t)a_dev[l];
    uint32_t i = m0 * a;
    T2* __restrict__ Tl = T + (size_t)l * w;
#pragma unroll
    for (int e = 0; e < SS_EPT; ++e) {
      const uint32_t ii = i & mask;
      if (ii < w) Tl[ii] = v[e];
      i += a;
    }
  }
  const uint32_t smask = (1u << log2sigma) - 1u;
  for (int r = 0; r < Rl; ++r) {
    const uint32_t d0 = m0 - (uint32_t)offs[r];   // wraps for m < off: never a multiple
#pragma unroll
    for (int e = 0; e < SS_EPT; ++e) {
      const uint32_t d = d0 + (uint32_t)e;
      if ((d & smask) == 0u) y[(size_t)r * W + (d >> log2sigma)] = v[e];
    }
  }
}

hipError_t stream_scatter_launch(int is_fp32, const void* x, void* T, void* y, const int* a_dev,
                                 const int* offs, int n, int w, int loops, int Rl, int W,
                                 hipStream_t st) {
  int log2sigma = 0;
  while ((W << log2sigma) < n) ++log2sigma;
  const unsigned blocks = (unsigned)(((long long)n / SS_EPT + SS_NT - 1) / SS_NT);
  if (is_fp32)
    hipLaunchKernelGGL((stream_scatter_kernel<float2>), dim3(blocks), dim3(SS_NT), 0, st,
                       (const float2*)x, (float2*)T, (float2*)y, a_dev, offs, (uint32_t)n,
                       (uint32_t)w, loops, Rl, log2sigma, (uint32_t)W);
  else
    hipLaunchKernelGGL((stream_scatter_kernel<double2>), dim3(blocks), dim3(SS_NT), 0, st,
                       (const double2*)x, (double2*)T, (double2*)y, a_dev, offs, (uint32_t)n,
                       (uint32_t)w, loops, Rl, log2sigma, (uint32_t)W);
  return hipGetLastError();
}

}  // namespace sfft
