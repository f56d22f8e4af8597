// sfft_hash.hip -- hand-written CDNA4 (gfx950) kernels of the sparse-FFT hot path, part 2.
//
//  * hash_*_kernel        reverse hash: approved-residue bitmaps, hit masks; the votes of earlier
//                         loops are tested directly from their bucket selections (no vote table)
//  * nodes_kernel         deterministic hit list (loop, bucket, walk order) and per-location FP64
//                         filter division and stable lower median
//
// Floating-point operations that must match the CPU oracle bit for bit are written out
// explicitly (fma where fused); the library is built with -ffp-contract=off.
#include <algorithm>

#include "sfft_jobs.h"

namespace sfft {

template <typename R>
struct CT;
template <>
struct CT<double> {
  using T2 = double2;
};
template <>
struct CT<float> {
  using T2 = float2;
};

// ============================================================================================
// block helpers
// ============================================================================================
// exclusive scan over a block of up to 1024 threads (wave64)
__device__ __forceinline__ int block_excl_scan(int v, int* sh) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  int off = 0;
  for (int i = 0; i < wid; ++i) off += sh[i];
  __syncthreads();
  return off + x - v;
}

__device__ __forceinline__ int block_sum(int v, int* sh) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  int x = v;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  if (lane == 0) sh[wid] = x;
  __syncthreads();
  int tot = 0;
  const int nw = (blockDim.x + 63) >> 6;
  for (int i = 0; i < nw; ++i) tot += sh[i];
  __syncthreads();
  return tot;
}

// ============================================================================================
// reverse hash
// ============================================================================================
__global__ void fill_u32_kernel(uint32_t* __restrict__ p, uint32_t v, size_t words) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t s = (size_t)gridDim.x * blockDim.x;
  for (; i < words; i += s) p[i] = v;
}

hipError_t fill_u32(void* p, uint32_t v, size_t words, hipStream_t st) {
  if (words == 0) return hipSuccess;
  size_t blocks = (words + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (uint32_t*)p, v,
                     words);
  return hipGetLastError();
}

// the per-transform clear in one launch: approved-residue bitmaps (and what lies behind them:
// the cutoffs' histograms) to 0, the largest approved
// residue of each location loop to -1 (the bucket selection bitmaps are rewritten whole by the
// cutoff)
__global__ void hash_clear_kernel(uint32_t* __restrict__ bm, size_t nbm,
                                  uint32_t* __restrict__ maxfirst, int nmax, DrawVals dv) {
  const size_t s = (size_t)gridDim.x * blockDim.x;
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t i = i0; i < nbm; i += s) bm[i] = 0u;
  if (i0 < (size_t)nmax) maxfirst[i0] = 0xFFFFFFFFu;
  if (i0 < (size_t)dv.count) dv.out[i0] = dv.v[i0];   // (block 0: 256 threads, 128 draws at most)
}

static int clear_blocks(const HashArgs& h) {
  const size_t blocks = (h.clear_words + 255) / 256;
  return (int)(blocks > 4096 ? 4096 : blocks < 1 ? 1 : blocks);
}

// the same for the signals of a batch
__global__ void hash_clear_jobs_kernel(JobsDev t) {
  const HashJob* j = job_here<HashJob>(t);
  if (!j) return;
  const HashArgs& h = j->h;
  const size_t nbm = h.clear_words, s = (size_t)j->blocks * 256;
  const size_t i0 = (size_t)((int)blockIdx.x - j->block0) * 256 + threadIdx.x;
  for (size_t i = i0; i < nbm; i += s) h.bitmap[i] = 0u;
  if (i0 < (size_t)h.loops_loc) h.maxfirst[i0] = -1;
}
void hash_jobs_clear(JobTable<HashJob>& t, const HashArgs& h) {
  HashJob j{h, clear_blocks(h), 0};
  t.add(j, j.blocks);
}
hipError_t hash_clear_jobs(const JobTable<HashJob>& t, hipStream_t st) {
  if (!t.dev.blocks) return hipSuccess;
  hipLaunchKernelGGL(hash_clear_jobs_kernel, dim3(t.dev.blocks), dim3(256), 0, st, t.dev);
  return hipGetLastError();
}

hipError_t hash_clear_launch(const HashArgs& h, const DrawVals& dv, hipStream_t st) {
  hipLaunchKernelGGL(hash_clear_kernel, dim3(clear_blocks(h)), dim3(256), 0, st,
                     (uint32_t*)h.bitmap, h.clear_words, (uint32_t*)h.maxfirst, h.loops_loc, dv);
  return hipGetLastError();
}

// approved residue first = J2 * ai mod W of every comb location, as a bitmap per location
// loop, and the largest one (reduced across the block first: one atomic per block on the
// loop's single max word -- same-address atomics serialise)
constexpr int BM_NT = 1024;
__device__ __forceinline__ void hash_bitmap_body(const HashArgs& h, int bx, int l) {
  __shared__ int wmax[BM_NT / 64];
  const int i = bx * BM_NT + threadIdx.x;
  int v = -1;
  if (i < h.nJ2) {
    const uint64_t j2 = (uint64_t)h.J2[i];
    const uint32_t first =
        (uint32_t)((j2 * (uint64_t)(uint32_t)h.ai_dev[l]) & (uint64_t)(h.W - 1));
    atomicOr(&h.bitmap[(size_t)l * h.bm_words + (first >> 5)], 1u << (first & 31));
    v = (int)first;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int m = -1;
    for (int w = 0; w < BM_NT / 64; ++w) m = max(m, wmax[w]);
    if (m >= 0) atomicMax(&h.maxfirst[l], m);
  }
}

__global__ __launch_bounds__(BM_NT) void hash_bitmap_kernel(HashArgs h) {
  hash_bitmap_body(h, blockIdx.x, blockIdx.y);
}
__global__ __launch_bounds__(BM_NT) void hash_bitmap_jobs_kernel(JobsDev t) {
  const HashJob* j = job_here<HashJob>(t);
  if (!j) return;
  const int i = (int)blockIdx.x - j->block0, nx = (j->h.nJ2 + BM_NT - 1) / BM_NT;
  hash_bitmap_body(j->h, i % nx, i / nx);
}
void hash_jobs_bitmap(JobTable<HashJob>& t, const HashArgs& h) {
  HashJob j{h, (h.nJ2 + BM_NT - 1) / BM_NT * h.loops_loc, 0};
  t.add(j, j.blocks);
}
hipError_t hash_bitmap_jobs(const JobTable<HashJob>& t, hipStream_t st) {
  if (!t.dev.blocks) return hipSuccess;
  hipLaunchKernelGGL(hash_bitmap_jobs_kernel, dim3(t.dev.blocks), dim3(BM_NT), 0, st, t.dev);
  return hipGetLastError();
}

hipError_t hash_bitmap_launch(const HashArgs& h, hipStream_t st) {
  dim3 grid((h.nJ2 + BM_NT - 1) / BM_NT, h.loops_loc);
  hipLaunchKernelGGL(hash_bitmap_kernel, grid, dim3(BM_NT), 0, st, h);
  return hipGetLastError();
}

// Lanes per bucket window (a power of two that divides 64 and m = n/B): one per 128 positions
// where the windows are many, so that a lane's table reads overlap its neighbours'; where they
// are few, more of them, down to 8 positions each, until the walk has HASH_LANES lanes: a lane
// tests its positions one after the other, each waiting for its table reads (n = 2^20, k = 1000,
// FP64: a transform 108 -> 92 us; n = 2^22, k = 2000, FP32: 141 -> 120, with 2^16 lanes 128).
constexpr long long HASH_LANES = 1 << 18;
__host__ __device__ __forceinline__ int hash_lpj(int loops_loc, int K, long long m) {
  long long l = m / 128;
  if (l < 1) l = 1;
  if (l > 64) l = 64;
  while (l < 64 && m / l > 8 && 2 * l * loops_loc * K <= HASH_LANES) l *= 2;
  return (int)l;
}

// Enumerate, in increasing circular order, the approved permuted positions p in the slice
// [low + d_begin, low + d_begin + d_len) of bucket J's window [J m - m/2, J m + m/2) (mod n);
// the whole window is empty when (low mod W) exceeds the largest approved residue (the
// reference's findUpperBound returns the last entry and the walk stops without wrapping).
// Calls fn(loc, rel) with loc = p * a mod n and rel = p - (low + d_begin), the position in
// the slice.
template <typename F>
__device__ __forceinline__ void hash_walk(const HashArgs& h, int l, int i, long long d_begin,
                                          long long d_len, F&& fn) {
  const long long n = h.n;
  const long long m = n / h.B;
  const long long J = h.J[(long long)l * h.K + i];
  long long low = J * m - (m >> 1);
  low = (low + n) & (n - 1);
  const int key = (int)(low & (h.W - 1));
  if (key > h.maxfirst[l]) return;
  const unsigned* bm = h.bitmap + (size_t)l * h.bm_words;
  const uint64_t a = (uint64_t)(uint32_t)h.a_dev[l];
  const uint64_t nmask = (uint64_t)n - 1;
  const long long d_end = d_begin + d_len;
  for (long long d = d_begin; d < d_end;) {
    const uint64_t p = (uint64_t)((low + d) & (n - 1));
    const uint32_t bpos = (uint32_t)(p & (uint64_t)(h.W - 1));
    const int off = (int)(bpos & 31u);
    const long long left = d_end - d;
    const int take = (left < 32 - off) ? (int)left : (32 - off);
    uint32_t word = bm[bpos >> 5] >> off;
    if (take < 32) word &= (1u << take) - 1u;
    while (word) {
      const int bit = __ffs(word) - 1;
      word &= word - 1u;
      const uint64_t pp = p + (uint64_t)bit;
      fn((uint32_t)((pp * a) & nmask), (int)(d - d_begin) + bit);
    }
    d += take;
  }
}

constexpr int HASH_NT = 256;

int hash_blocks(int loops, int loops_loc, int K, long long m) {
  return (int)(((long long)loops * K * hash_lpj(loops_loc, K, m) + HASH_NT - 1) / HASH_NT);
}

// 32-bit words of one slice's hit mask (a slice covers m / lpj window positions)
__host__ __device__ __forceinline__ int hash_slice_words(int loops_loc, int K, long long m) {
  return (int)((m / hash_lpj(loops_loc, K, m) + 31) / 32);
}
size_t hash_mask_bytes(int loops_loc, int K, long long m) {
  return (size_t)hash_blocks(loops_loc, loops_loc, K, m) * HASH_NT *
         hash_slice_words(loops_loc, K, m) * 4;
}

// A location is voted at most once per loop (the J windows of a loop are disjoint), so its
// vote count after loop l is the number of loops 0..l that walked it.  Hence (1) only loops
// l >= loops_thresh-1 can produce hits, and (2) the hit test of loop l needs only whether each
// loop l' < l walked the location (its own walk is implied).  Loop l' walked loc exactly when
// loc's position p = loc * ai_l' mod n lies in the window of a bucket J that l' selected,
// J = ((p + m/2) mod n) / m, that window is not cut off by the largest approved residue (the
// walk's early exit), and p's residue p mod W is approved: three table reads instead of a
// vote pass over every window and a vote table.  The walk covers the loops
// [thresh-1, loops_loc) (loops_thresh >= 1 is checked when the plan is made).
static int hash_hit_blocks(const HashArgs& h) {
  return hash_blocks(h.loops_loc - (h.loops_thresh - 1), h.loops_loc, h.K, (long long)h.n / h.B);
}

// thread -> (location loop l, bucket index i, slice sub of lpj)
struct HashSlot {
  int l, i, sub, lpj;
  long long jidx, d0, dl;
  bool valid;
};

__device__ __forceinline__ int hash_hit_first_d(const HashArgs& h) { return h.loops_thresh - 1; }
__device__ __forceinline__ int hash_hit_count_d(const HashArgs& h) {
  return h.loops_loc - (h.loops_thresh - 1);
}

// threads cover loops [l_first, l_first + nloops)
__device__ __forceinline__ HashSlot hash_slot(const HashArgs& h, int l_first, int nloops, int bx) {
  HashSlot s;
  const long long m = (long long)h.n / h.B;
  s.lpj = hash_lpj(h.loops_loc, h.K, m);
  const long long gid = (long long)bx * HASH_NT + threadIdx.x;
  const long long local = gid / s.lpj;
  s.sub = (int)(gid % s.lpj);
  s.valid = local < (long long)nloops * h.K;
  s.jidx = local + (long long)l_first * h.K;
  s.l = (int)(s.jidx / h.K);
  s.i = (int)(s.jidx - (long long)s.l * h.K);
  s.dl = m / s.lpj;
  s.d0 = s.sub * s.dl;
  return s;
}

// whether location loop lp walked loc: its bucket J was selected, J's window is not cut off
// by the largest approved residue, and loc's residue is approved
__device__ __forceinline__ bool hash_walked(const HashArgs& h, int lp, uint32_t loc) {
  const long long n = h.n;
  const long long m = n / h.B;
  const uint64_t p = ((uint64_t)loc * (uint64_t)(uint32_t)h.ai_dev[lp]) & (uint64_t)(n - 1);
  const int lm = 63 - __clzll(m);   // m = n / B, both powers of two
  const uint32_t J = (uint32_t)((((long long)p + (m >> 1)) & (n - 1)) >> lm);
  const long long low = ((long long)J * m - (m >> 1) + n) & (n - 1);
  const uint32_t r = (uint32_t)(p & (uint64_t)(h.W - 1));
  // the three table reads are independent: issued together, tested together
  const unsigned js = h.jsel[(size_t)lp * h.jsel_words + (J >> 5)];
  const int mf = h.maxfirst[lp];
  const unsigned bw = h.bitmap[(size_t)lp * h.bm_words + (r >> 5)];
  return (((js >> (J & 31)) & (bw >> (r & 31))) & 1u) && (int)(low & (h.W - 1)) <= mf;
}

// a location walked by loop l is a hit of loop l when exactly loops_thresh of the loops 0..l
// voted for it, loop l included (the loop in which the reference's count reaches the
// threshold, innerLoop.cu:809-814): loops_thresh - 1 of the loops before l
__device__ __forceinline__ bool hash_is_hit(const HashArgs& h, int l, uint32_t loc) {
  int v = 1;   // loop l's own walk
  for (int lp = 0; lp < l; ++lp) v += hash_walked(h, lp, loc) ? 1 : 0;
  return v == h.loops_thresh;
}

// hit count of a slot's slice, and its hit mask (bit rel of word rel/32 set for a hit at
// slice position rel) into mk[0 .. words)
__device__ __forceinline__ int hash_count_slice(const HashArgs& h, const HashSlot& s,
                                                unsigned* __restrict__ mk, int words) {
  int c = 0;
  if (!s.valid) return 0;
  unsigned cur = 0u;
  int cw = 0;
  hash_walk(h, s.l, s.i, s.d0, s.dl, [&](uint32_t loc, int rel) {
    if (hash_is_hit(h, s.l, loc)) {
      for (; cw < (rel >> 5); ++cw) {
        mk[cw] = cur;
        cur = 0u;
      }
      cur |= 1u << (rel & 31);
      ++c;
    }
  });
  for (; cw < words; ++cw) {
    mk[cw] = cur;
    cur = 0u;
  }
  return c;
}

// ============================================================================================
// estimation
// ============================================================================================
__device__ __forceinline__ double2 to_d2(double2 v) { return v; }
__device__ __forceinline__ double2 to_d2(float2 v) {
  return make_double2((double)v.x, (double)v.y);
}

// The value of location I: the lower medians over the loops of the real and the imaginary parts
// (rr, ri) and the loops they came from (sr, si).  EXACT: the loop count is the template constant
// MAXL (every address first, then every load, so the 2*MAXL reads of a hit are in flight
// together); otherwise loops <= MAXL at run time.  The arithmetic per loop is the same either way.
template <typename Real, int MAXL, bool EXACT>
__device__ __forceinline__ void estimate_one(uint32_t I,
                                             const typename CT<Real>::T2* __restrict__ bins,
                                             int loops_rt, uint32_t n,
                                             const int* __restrict__ ai_dev, int B,
                                             const double2* __restrict__ win, double& rr,
                                             double& ri, int& sr, int& si) {
  const int loops = EXACT ? MAXL : loops_rt;
  const long long m = (long long)(n / (uint32_t)B);
  const int lm = 63 - __clzll(m);   // m = n / B, both powers of two
  const long long nn = n;
  const int med = (loops - 1) / 2;
  long long bidx[MAXL], widx[MAXL];
#pragma unroll
  for (int l = 0; l < MAXL; ++l) {
    const int lc = (EXACT || l < loops) ? l : 0;   // a valid address past the loop count
    const long long p = (long long)(((uint64_t)(uint32_t)ai_dev[lc] * I) & (uint64_t)(n - 1));
    long long hashed = p >> lm;
    long long dist = p & (m - 1);
    if (dist > m / 2) {
      hashed = (hashed + 1) & (B - 1);
      dist -= m;
    }
    dist = (nn - dist) & (nn - 1);
    widx[l] = (dist + m / 2) & (nn - 1);
    bidx[l] = (long long)lc * B + hashed;
  }
  double2 F[MAXL], bb[MAXL];
#pragma unroll
  for (int l = 0; l < MAXL; ++l) {
    F[l] = win[widx[l]];
    bb[l] = to_d2(bins[bidx[l]]);
  }
  double vr[MAXL], vi[MAXL];
#pragma unroll
  for (int l = 0; l < MAXL; ++l) {
    // innerLoop.cu:848-852: products rounded, then combined
    const double abs2 = F[l].x * F[l].x + F[l].y * F[l].y;
    const double mr = bb[l].x * F[l].x + bb[l].y * F[l].y;
    const double mi = bb[l].y * F[l].x - bb[l].x * F[l].y;
    vr[l] = mr / abs2;
    vi[l] = mi / abs2;
  }
  // stable rank selection: position of j in an insertion sort = #(v_i < v_j) + #(i<j, v_i==v_j)
  rr = ri = 0.0;
  sr = si = 0;
#pragma unroll
  for (int j = 0; j < MAXL; ++j) {
    if (j < loops) {
      int pr = 0, pi = 0;
#pragma unroll
      for (int i = 0; i < MAXL; ++i) {
        if (i < loops) {
          pr += (vr[i] < vr[j]) || (i < j && vr[i] == vr[j]);
          pi += (vi[i] < vi[j]) || (i < j && vi[i] == vi[j]);
        }
      }
      if (pr == med) {
        rr = vr[j];
        sr = j;
      }
      if (pi == med) {
        ri = vi[j];
        si = j;
      }
    }
  }
}

// `count` nodes staged in LDS stored as consecutive 8-byte words (coalesced, also when out is
// pinned host memory written over the bus)
constexpr int EST_NT = 256;
static_assert(sizeof(Node) == 24, "Node: key, 4 bytes of padding, two doubles");
__device__ __forceinline__ void stage_node(unsigned long long* stage, uint32_t I, double rr,
                                           double ri) {
  stage[3 * threadIdx.x] = (unsigned long long)I;   // key, then 4 zero bytes of padding
  stage[3 * threadIdx.x + 1] = (unsigned long long)__double_as_longlong(rr);
  stage[3 * threadIdx.x + 2] = (unsigned long long)__double_as_longlong(ri);
}
__device__ __forceinline__ void store_nodes(const unsigned long long* stage, int count,
                                            Node* __restrict__ out) {
  unsigned long long* o = reinterpret_cast<unsigned long long*>(out);
  for (int j = threadIdx.x; j < 3 * count; j += EST_NT) o[j] = stage[j];
}

// One thread per hit of a list (the reference's estimation entry point).
constexpr int EST_GRID = 512;   // blocks of the estimation launch (grid-stride over the hits)
template <typename Real, int MAXL, bool EXACT>
__global__ __launch_bounds__(EST_NT) void estimate_kernel(EstArgs j) {
  __shared__ unsigned long long stage[EST_NT * 3];
  const int total = min(*j.count, j.capacity);
  for (int h0 = blockIdx.x * EST_NT; h0 < total; h0 += gridDim.x * EST_NT) {
    const int h = h0 + (int)threadIdx.x;
    const uint32_t I = (uint32_t)j.hits[h < total ? h : h0];
    double rr, ri;
    int sr, si;
    estimate_one<Real, MAXL, EXACT>(I, (const typename CT<Real>::T2*)j.bins, j.loops,
                                    (uint32_t)j.n, j.ai, j.B, j.win, rr, ri, sr, si);
    stage_node(stage, I, rr, ri);
    __syncthreads();
    store_nodes(stage, min(EST_NT, total - h0), j.out + h0);
    __syncthreads();
  }
}

// The hits of the places before bx, one wave (the decoupled look-back of Merrill and Garland's
// single-pass prefix scan): publishes this place's total, adds up the totals of
// the 64 places before it at a time until it meets one whose sum with all before it is published,
// and publishes its own such sum.  A place is taken by a running block, which publishes its total
// before it waits for anything but its own threads, so every wait ends whatever the order or
// number of resident blocks.
constexpr unsigned long long PLACE_TOTAL = 1ull << 32, PLACE_SUM = 2ull << 32;   // | hits; 0: neither
__device__ __forceinline__ int walk_prefix(unsigned long long* place, int bx, int tot) {
  const int lane = threadIdx.x & 63;
  auto publish = [&](unsigned long long v) __attribute__((always_inline)) {
    if (lane == 0)
      __hip_atomic_store(&place[bx], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (bx > 0) publish(PLACE_TOTAL | (unsigned)tot);
  int before = 0;
  bool summed = bx == 0;
  for (int b0 = bx - 1; !summed; b0 -= 64) {   // (place 0 always holds a sum)
    const int b = b0 - lane;
    unsigned long long v, none, sums;
    int last;   // the nearest place with a sum, or 63
    for (;;) {
      v = b >= 0 ? __hip_atomic_load(&place[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                 : PLACE_SUM;
      none = __ballot(v == 0ull);
      sums = __ballot((v & PLACE_SUM) != 0ull);
      last = sums ? __ffsll((long long)sums) - 1 : 63;
      if (!none || __ffsll((long long)none) - 1 > last) break;
      __builtin_amdgcn_s_sleep(1);
    }
    int x = lane <= last ? (int)(unsigned)v : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    before += x;
    summed = sums != 0ull;
  }
  publish(PLACE_SUM | (unsigned)(before + tot));
  return before;
}

// A walk's hit masks, and each block's hit total into its place, as a launch before nodes_kernel.
__global__ __launch_bounds__(HASH_NT) void hash_count_kernel(HashArgs h) {
  __shared__ int sh[16];
  const HashSlot s = hash_slot(h, hash_hit_first_d(h), hash_hit_count_d(h), blockIdx.x);
  const int words = hash_slice_words(h.loops_loc, h.K, (long long)h.n / h.B);
  const long long gid = (long long)blockIdx.x * HASH_NT + threadIdx.x;
  const int tot = block_sum(hash_count_slice(h, s, h.hmask + gid * words, words), sh);
  if (threadIdx.x == 0) h.place[blockIdx.x] = PLACE_TOTAL | (unsigned)tot;
}

// Walks of up to this many blocks run in the nodes' launch (WALK).  Walk and nodes as two
// launches -> one: n = 2^14, k = 20 (3 blocks) 58 -> 52 us, n = 2^20, k = 1000 (125) FP32
// 61 -> 57, FP64 76 -> 69, 64 signals (places of their own) 1804 -> 1750; but n = 2^24, k = 2503
// (313) 137 -> 143, n = 2^27, k = 16000 (1000) FP32 470 -> 477, k = 40000 (2500) 1078 -> 1089:
// the blocks' turns at one ticket cost more than the launch.
constexpr int WALK_BLOCKS = 256;

// The located indices of one signal in (loop, bucket, walk) order and their values.  A block
// lists the hits of its slices in LDS in window order and estimates one per thread, so the hits
// are consecutive threads' work however the windows hold them.  WALK: it takes the next place in
// the walk and walks its slices itself; else hash_count_kernel has, and the totals of the blocks
// before it are summed (a few KB, read by every block in parallel: no scan launch).
constexpr int ND_LIST = 1024;   // hits listed at a time
template <typename Real, int MAXL, bool EXACT, bool WALK>
__device__ __forceinline__ void nodes_body(const NodeJob& j, int nb) {
  static_assert(HASH_NT == EST_NT, "a hit per thread of the walk's block");
  __shared__ unsigned long long stage[EST_NT * 3];
  __shared__ int list[ND_LIST];
  __shared__ int sh[16];
  __shared__ int s_bx, s_tot, s_pre;
  const HashArgs& h = j.h;
  const int tid = threadIdx.x;
  int bx = blockIdx.x;
  if (WALK) {
    if (tid == 0) s_bx = (int)atomicAdd(h.ticket, 1u);
    __syncthreads();
    bx = s_bx;
  }
  const HashSlot s = hash_slot(h, hash_hit_first_d(h), hash_hit_count_d(h), bx);
  const int words = hash_slice_words(h.loops_loc, h.K, (long long)h.n / h.B);
  const long long gid = (long long)bx * HASH_NT + tid;
  unsigned* mk = h.hmask + gid * words;
  int c = 0;
  if (WALK) {
    c = hash_count_slice(h, s, mk, words);
  } else if (s.valid) {
    for (int w = 0; w < words; ++w) c += __popc(mk[w]);
  }
  // the threads of a block are its slices in walk order
  const int first = block_excl_scan(c, sh);
  if (tid == HASH_NT - 1) s_tot = first + c;
  __syncthreads();
  const int tot = s_tot;
  int boff;
  if (WALK) {
    if (tid < 64) {
      const int before = walk_prefix(h.place, bx, tot);
      if (tid == 0) s_pre = before;
    }
    __syncthreads();
    boff = s_pre;
  } else {
    int pre = 0;
    for (int b = tid; b < bx; b += HASH_NT) pre += (int)(unsigned)h.place[b];
    boff = block_sum(pre, sh);
  }
  if (bx == nb - 1 && tid == 0) {
    *h.count = boff + tot;
    if (j.count_copy) *j.count_copy = boff + tot;
  }
  if (tot == 0) return;
  const long long n = h.n;
  const long long m = n / h.B;
  long long start = 0;
  uint64_t a = 0;
  if (c) {
    const long long J = h.J[(long long)s.l * h.K + s.i];
    start = ((J * m - (m >> 1)) + n + s.d0) & (n - 1);   // low + d0
    a = (uint64_t)(uint32_t)h.a_dev[s.l];
  }
  for (int r0 = 0; r0 < tot; r0 += ND_LIST) {
    if (c) {
      int pos = first - r0;
      for (int w = 0; w < words; ++w) {
        unsigned word = mk[w];
        while (word) {
          const int rel = w * 32 + __ffs(word) - 1;
          word &= word - 1u;
          const uint64_t p = (uint64_t)((start + rel) & (n - 1));
          if (pos >= 0 && pos < ND_LIST) list[pos] = (int)((p * a) & ((uint64_t)n - 1));
          ++pos;
        }
      }
    }
    __syncthreads();
    const int o0 = boff + r0;   // (hits past the capacity are counted only)
    const int lim = min(min(ND_LIST, tot - r0), h.capacity - o0);
    for (int h0 = 0; h0 < lim; h0 += EST_NT) {
      const int i = h0 + tid;
      if (h0 + (tid & ~63) < lim) {   // (waves without a hit leave)
        const uint32_t I = (uint32_t)list[i < lim ? i : h0];
        double rr, ri;
        int sr, si;
        estimate_one<Real, MAXL, EXACT>(I, (const typename CT<Real>::T2*)j.bins, j.loops,
                                        (uint32_t)h.n, h.ai_dev, h.B, j.win, rr, ri, sr, si);
        stage_node(stage, I, rr, ri);
        if (i < lim) {
          h.hits[o0 + i] = (int)I;
          if (j.sel) {
            j.sel[2 * (size_t)(o0 + i)] = (uint8_t)sr;
            j.sel[2 * (size_t)(o0 + i) + 1] = (uint8_t)si;
          }
        }
      }
      __syncthreads();
      const int k = min(EST_NT, lim - h0);
      store_nodes(stage, k, j.out + o0 + h0);
      if (j.copy) store_nodes(stage, k, j.copy + o0 + h0);
      __syncthreads();
    }
    __syncthreads();   // (lim <= 0: the list is read no more before it is written again)
  }
}

template <typename Real, int MAXL, bool EXACT, bool WALK>
__global__ __launch_bounds__(EST_NT) void nodes_kernel(NodeJob j) {
  nodes_body<Real, MAXL, EXACT, WALK>(j, (int)gridDim.x);
}
template <typename Real, int MAXL, bool EXACT>
__global__ __launch_bounds__(EST_NT) void nodes_jobs_kernel(JobsDev t) {
  const NodeJob* p = job_here<NodeJob>(t);
  if (!p) return;
  const NodeJob j = *p;
  nodes_body<Real, MAXL, EXACT, true>(j, j.blocks);
}

// f(the loop count as a template constant, whether it is exact)
template <int V>
struct IntC {
  static constexpr int v = V;
};
template <typename F>
static hipError_t with_loops(int loops, F&& f) {
#define SFFT_EST(L) \
  case L:           \
    return f(IntC<L>(), IntC<1>());
  switch (loops) {
    SFFT_EST(1) SFFT_EST(2) SFFT_EST(3) SFFT_EST(4) SFFT_EST(5) SFFT_EST(6) SFFT_EST(7)
    SFFT_EST(8) SFFT_EST(9) SFFT_EST(10) SFFT_EST(11) SFFT_EST(12) SFFT_EST(13) SFFT_EST(14)
    SFFT_EST(15) SFFT_EST(16)
    default:
      return f(IntC<32>(), IntC<0>());
  }
#undef SFFT_EST
}

hipError_t estimate_launch(const EstArgs& a, hipStream_t st) {
  return with_loops(a.loops, [&](auto L, auto E) {
    hipLaunchKernelGGL((estimate_kernel<double, decltype(L)::v, decltype(E)::v != 0>),
                       dim3(EST_GRID), dim3(EST_NT), 0, st, a);
    return hipGetLastError();
  });
}

template <typename Real>
static hipError_t nodes_go(const NodeJob& j, hipEvent_t between, hipStream_t st) {
  const int blocks = hash_hit_blocks(j.h);
  const bool walk = blocks <= WALK_BLOCKS && !between;
  if (!walk) hipLaunchKernelGGL(hash_count_kernel, dim3(blocks), dim3(HASH_NT), 0, st, j.h);
  if (between) {
    const hipError_t e = hipEventRecord(between, st);
    if (e != hipSuccess) return e;
  }
  return with_loops(j.loops, [&](auto L, auto E) {
    constexpr int l = decltype(L)::v;
    constexpr bool e = decltype(E)::v != 0;
    if (walk)
      hipLaunchKernelGGL((nodes_kernel<Real, l, e, true>), dim3(blocks), dim3(EST_NT), 0, st, j);
    else
      hipLaunchKernelGGL((nodes_kernel<Real, l, e, false>), dim3(blocks), dim3(EST_NT), 0, st, j);
    return hipGetLastError();
  });
}
hipError_t nodes_launch(int is_fp32, const NodeJob& j, hipEvent_t between, hipStream_t st) {
  return is_fp32 ? nodes_go<float>(j, between, st) : nodes_go<double>(j, between, st);
}

void nodes_jobs_add(std::vector<NodeGroup>& g, int is_fp32, NodeJob j) {
  const int key = j.loops <= 16 ? j.loops : 32;   // one kernel takes every count above 16
  auto it = std::find_if(g.begin(), g.end(), [&](const NodeGroup& x) { return x.loops == key; });
  if (it == g.end()) {
    g.emplace_back();
    it = g.end() - 1;
    it->loops = key;
    it->fp32 = is_fp32;
  }
  j.blocks = hash_hit_blocks(j.h);
  it->t.add(j, j.blocks);
}

hipError_t nodes_jobs_launch(const std::vector<NodeGroup>& groups, hipStream_t st) {
  for (const NodeGroup& g : groups) {
    const hipError_t r = with_loops(g.loops, [&](auto L, auto E) {
      constexpr int l = decltype(L)::v;
      constexpr bool e = decltype(E)::v != 0;
      if (g.fp32)
        hipLaunchKernelGGL((nodes_jobs_kernel<float, l, e>), dim3(g.t.dev.blocks), dim3(EST_NT),
                           0, st, g.t.dev);
      else
        hipLaunchKernelGGL((nodes_jobs_kernel<double, l, e>), dim3(g.t.dev.blocks), dim3(EST_NT),
                           0, st, g.t.dev);
      return hipGetLastError();
    });
    if (r != hipSuccess) return r;
  }
  return hipSuccess;
}

}  // namespace sfft
