// sfft_select.hip -- top-K cutoff on the GPU: the K largest |X|^2 of each segment, ties broken
// by the lower index (the reference's cutoff, innerLoop.cu:551-642), without sorting.
//
// Every element gets a unique composite key  c = (key without sign bit) . (N-1-index)  so that
// "larger c" means "larger |X|^2, or equal and lower index"; the top-K set is {c >= T}.
//   1. hist0   : histogram of the top 12 bits of c, one row per block (wave-aggregated LDS
//                atomics), then colsum: the column sums of the rows.  A transform's cutoffs skip
//                both: the last FFT pass leaves the histogram (FftLaunch::hist).
//   2. split   : every block picks the digit d0 holding the K-th largest from the
//                sums, then one pass over N: digit > d0 -> selected (emitted at once in
//                unordered mode), digit == d0 -> appended to a candidate list (typically ~1%
//                of N).
//   3. refine  : one workgroup per segment: MSD radix select on the remaining bits of c over
//                the candidates only, with early exit once a digit bin fills the remainder;
//                yields T and (unordered mode) emits the selected candidates.
//   4. ordered mode only: write, an order-preserving compaction of {c >= T} that produces
//                the ascending index list the reverse hash walks in order.  The selected
//                count of each block (its digit > d0 count from the split plus its candidates
//                >= T) and their exclusive prefix come out of the refine.
// Short segments (select_in_block) take one launch instead: sel_block_kernel.
#include "sfft_jobs.h"

namespace sfft {

typedef unsigned __int128 u128;

struct SelState {
  unsigned long long thr_hi, thr_lo;   // T as two 64-bit halves
  int d0;                              // top digit holding the K-th largest
  int need0;                           // K - #(digit > d0)
  int cand_count;
  int out_count;
};

constexpr int SEL_NT = 1024;   // threads of the streaming select kernels (512: +11 us comb
                               // cutoff, +3 us bucket cutoff at n = 2^27, k = 16000)
constexpr int SEL_DIG = kSelDigit;
constexpr int SEL_BINS = kSelBins;

template <typename K>
struct KeyBits;
template <>
struct KeyBits<unsigned long long> {
  static constexpr int KB = 63;  // bits below the (always zero) sign bit
  // the first digit is not the key's top bits (sel_first_digit): the refine starts at bit 0
  static constexpr bool digit_is_prefix = false;
};
template <>
struct KeyBits<unsigned int> {
  static constexpr int KB = 31;
  static constexpr bool digit_is_prefix = true;
};

// bits of the index field of a composite key: enough for N - 1 (any N, not only powers of 2)
__device__ __forceinline__ int index_bits(int N) { return N > 1 ? 32 - __clz(N - 1) : 0; }


constexpr int SPLIT_ROUND = 8 * SEL_NT;   // keys whose loads the split keeps in flight together

// elements per block: about 256 blocks per segment for large N, at least 2048
static int sel_chunk(int N) {
  int c = 2048;
  while ((long long)c * 256 < N) c <<= 1;
  return c;
}

static size_t hist_words(int segs, int nch, bool counted) {
  return counted ? 0 : (size_t)segs * (nch + 1) * SEL_BINS;
}

size_t select_work_bytes(int segs, int N, bool counted) {
  const int nch = (N + sel_chunk(N) - 1) / sel_chunk(N);
  return (size_t)segs * sizeof(SelState) + hist_words(segs, nch, counted) * 4 +
         (size_t)segs * nch * 4 * 3 + (size_t)segs * N * 8 * 2 + (size_t)segs * N * 4 * 3 + 4096;
}

void select_work_bind(SelectWork* w, void* base, int segs, int N, bool counted) {
  const int nch = (N + sel_chunk(N) - 1) / sel_chunk(N);
  char* p = (char*)base;
  auto take = [&](size_t bytes) {
    char* r = p;
    p += (bytes + 255) / 256 * 256;
    return r;
  };
  w->state = take((size_t)segs * sizeof(SelState));
  w->hist = counted ? nullptr : (unsigned*)take(hist_words(segs, nch, false) * 4);
  w->cnt = (int*)take((size_t)segs * nch * 4);
  w->cand_key = take((size_t)segs * N * 8);
  w->cand_idx = (int*)take((size_t)segs * N * 4);
  w->emit_idx = (int*)take((size_t)segs * N * 4);
  w->blk_key = take((size_t)segs * N * 8);
  w->blk_idx = (int*)take((size_t)segs * N * 4);
  w->ccnt = (int*)take((size_t)segs * nch * 4);
  w->ecnt = (int*)take((size_t)segs * nch * 4);
  w->max_segs = segs;
  w->max_chunks = nch;
}

__device__ __forceinline__ int block_excl_scan_s(int v, int* sh) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
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

// increment h[bin] for the active lanes: one atomic for the whole wave when every active lane
// holds the same bin (flat or tied data), else one LDS atomic per lane (spread data, where
// per-bin aggregation would loop once per distinct bin)
__device__ __forceinline__ void wave_hist_add(unsigned* h, unsigned bin, bool active) {
  const int lane = threadIdx.x & 63;
  const unsigned long long act = __ballot(active);
  if (!act) return;
  const int first = __ffsll((long long)act) - 1;
  const unsigned b0 = __shfl(bin, first, 64);
  const unsigned long long same = __ballot(active && bin == b0);
  if (same == act) {
    if (lane == first) atomicAdd(&h[b0], (unsigned)__popcll(act));
  } else if (active) {
    atomicAdd(&h[bin], 1u);
  }
}

// wave-aggregated append: returns the slot of this lane (valid only where pred)
__device__ __forceinline__ int wave_append(int* counter, bool pred) {
  const int lane = threadIdx.x & 63;
  const unsigned long long m = __ballot(pred);
  if (!m) return -1;
  const int leader = __ffsll((long long)m) - 1;
  int base = 0;
  if (lane == leader) base = atomicAdd(counter, __popcll(m));
  base = __shfl(base, leader, 64);
  return base + __popcll(m & ((1ull << lane) - 1ull));
}

template <typename K>
__device__ __forceinline__ unsigned top_digit(K key) {
  return sel_first_digit(key);
}

template <typename K>
__device__ __forceinline__ u128 composite(K key, unsigned idx, int N, int IB) {
  const K km = key & (K)(~((K)1 << KeyBits<K>::KB));
  return ((u128)km << IB) | (u128)(unsigned)((unsigned)(N - 1) - idx);
}

// ---- 1. top-digit histogram: one row of SEL_BINS counts per block (plain stores) ---------
// (each stage's body takes its block bx and segment seg: a launch of one select, or of many)
template <typename K>
__device__ __forceinline__ void sel_hist0_body(const K* __restrict__ keys, long long seg_stride,
                                               int N, int chunk, int nchunks,
                                               unsigned* __restrict__ rows,
                                               const uint16_t* __restrict__ digits, int bx,
                                               int seg) {
  __shared__ unsigned h[SEL_BINS];
  const int tid = threadIdx.x;
  for (int i = tid; i < SEL_BINS; i += SEL_NT) h[i] = 0u;
  __syncthreads();
  const K* kp = keys + (long long)seg * seg_stride;
  const int begin = bx * chunk, end = min(N, begin + chunk);
  constexpr int U = 8;   // independent loads in flight per thread
  if (digits) {          // the first digits only (2 bytes per key instead of 4 or 8)
    const uint16_t* dp = digits + (long long)seg * seg_stride;
    for (int base = begin; base < end; base += SEL_NT * U) {
      unsigned dd[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = base + u * SEL_NT + tid;
        dd[u] = i < end ? (unsigned)dp[i] : 0u;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = base + u * SEL_NT + tid;
        wave_hist_add(h, dd[u], i < end);
      }
    }
  } else {
    for (int base = begin; base < end; base += SEL_NT * U) {
      K kk[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = base + u * SEL_NT + tid;
        kk[u] = i < end ? kp[i] : (K)0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = base + u * SEL_NT + tid;
        wave_hist_add(h, top_digit<K>(kk[u]), i < end);
      }
    }
  }
  __syncthreads();
  unsigned* row = rows + ((size_t)seg * nchunks + bx) * SEL_BINS;
  for (int i = tid; i < SEL_BINS; i += SEL_NT) row[i] = h[i];
}

// ---- 1b. column sums of the block rows ----------------------------------------------------
// a block sums 16 bins, 16 threads per bin each over every 16th row, then reduces in LDS
constexpr int PICK_NT = 256;
constexpr int PICK_BINS = 16;
__device__ __forceinline__ void sel_colsum_body(int nchunks, const unsigned* __restrict__ rows,
                                                unsigned* __restrict__ ghist, int bx, int seg) {
  __shared__ unsigned part[PICK_NT / PICK_BINS][PICK_BINS];
  const int tid = threadIdx.x;
  const int bl = tid % PICK_BINS, g = tid / PICK_BINS;
  constexpr int G = PICK_NT / PICK_BINS;
  const int bin0 = bx * PICK_BINS;
  const unsigned* r = rows + (size_t)seg * nchunks * SEL_BINS + bin0 + bl;
  unsigned a = 0u;
#pragma unroll 4
  for (int c = g; c < nchunks; c += G) a += r[(size_t)c * SEL_BINS];
  part[g][bl] = a;
  __syncthreads();
  if (tid < PICK_BINS) {
    unsigned acc = 0u;
#pragma unroll
    for (int j = 0; j < G; ++j) acc += part[j][tid];
    ghist[(size_t)seg * SEL_BINS + bin0 + tid] = acc;
  }
}

// ---- 2. split: collect digit == d0 (candidates), count digit > d0 (and emit them, unordered
// mode) ---------------------------------------------------------------------------------------
// Block b writes its candidates to [b*chunk, b*chunk + count) of the segment's candidate
// arrays, its emitted indices to the same range of the emitted array, and the two counts to
// ccnt/ecnt[seg][b]: no global atomics (the refine pass compacts).  Keys stored in a KeyMap
// order are recorded with their natural indices (the tie rule and the output use those).
template <typename K>
__device__ __forceinline__ void sel_split_body(const K* __restrict__ keys, long long seg_stride,
                                               int N, int chunk, int nchunks, int emit, int Ksel,
                                               const unsigned* __restrict__ ghist, int nsum,
                                               SelState* __restrict__ st, K* __restrict__ ckey,
                                               int* __restrict__ cidx, int* __restrict__ eidx,
                                               int* __restrict__ ccnt, int* __restrict__ ecnt,
                                               KeyMap km, const uint16_t* __restrict__ digits,
                                               int bx, int seg) {
  static_assert(SEL_NT * 4 == SEL_BINS, "the pick gives each thread four bins");
  __shared__ int s_nc, s_ne, s_d0;
  __shared__ int sh[16];
  const int tid = threadIdx.x;
  if (tid == 0) {
    s_nc = 0;
    s_ne = 0;
    s_d0 = 0;
  }
  // the top digit d0 holding the K-th largest key, from the column sums: every block finds
  // the same one (16 KB of sums, or the FFT's kSelCopies histograms of 16 KB each: no separate
  // pick launch); block 0 records it and the count still needed inside it for the refine
  {
    const unsigned* gh = ghist + (size_t)seg * nsum * SEL_BINS;
    unsigned v[4];
    int S = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = gh[SEL_BINS - 1 - (4 * tid + j)];
    if (nsum == kSelCopies) {   // the FFT's histograms (their loads in flight together)
#pragma unroll
      for (int c = 1; c < kSelCopies; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += gh[c * SEL_BINS + SEL_BINS - 1 - (4 * tid + j)];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) S += (int)v[j];
    const int E = block_excl_scan_s(S, sh);   // (its barriers also publish the defaults)
    if (E < Ksel && Ksel <= E + S) {
      int cum = E;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (cum + (int)v[j] >= Ksel) {
          const int dd = SEL_BINS - 1 - (4 * tid + j);
          s_d0 = dd;
          if (bx == 0) {
            st[seg].d0 = dd;
            st[seg].need0 = Ksel - cum;
          }
          break;
        }
        cum += (int)v[j];
      }
    }
  }
  __syncthreads();
  const unsigned d0 = (unsigned)s_d0;
  const K* kp = keys + (long long)seg * seg_stride;
  const long long rb = (long long)seg * N + (long long)bx * chunk;
  K* ck = ckey + rb;
  int* ci = cidx + rb;
  int* ce = eidx + rb;
  const int begin = bx * chunk, end = min(N, begin + chunk);
  const uint16_t* dp = digits ? digits + (long long)seg * seg_stride : nullptr;
  // SU elements per thread at a time: their digit (or key) loads are in flight together, then
  // the candidates' key loads, so that the loop waits twice per SU elements, not twice per
  // element (the order of a block's candidates and winners is set by the wave appends either
  // way; every later pass is independent of it)
  constexpr int SU = SPLIT_ROUND / SEL_NT;
  for (int base = begin; base < end; base += SPLIT_ROUND) {
    unsigned d[SU];
    K k[SU];
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      const int i = base + u * SEL_NT + tid;
      const bool ok = i < end;
      if (dp) {
        d[u] = ok ? (unsigned)dp[i] : 0u;
      } else {
        k[u] = ok ? kp[i] : (K)0;
        d[u] = top_digit<K>(k[u]);
      }
    }
    // with the first digits at hand, a key is read only when it is a candidate
    if (dp) {
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const int i = base + u * SEL_NT + tid;
        k[u] = (i < end && d[u] == d0) ? kp[i] : (K)0;
      }
    }
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      const int i = base + u * SEL_NT + tid;
      const bool ok = i < end;
      const bool isc = ok && d[u] == d0;
      const int pc = wave_append(&s_nc, isc);
      if (isc) {
        ck[pc] = k[u];
        ci[pc] = (int)key_natural(km, i);
      }
      const bool ise = ok && d[u] > d0;
      const int pe = wave_append(&s_ne, ise);
      if (emit && ise) ce[pe] = (int)key_natural(km, i);
    }
  }
  __syncthreads();
  if (tid == 0) {
    ccnt[(long long)seg * nchunks + bx] = s_nc;
    ecnt[(long long)seg * nchunks + bx] = s_ne;
  }
}

constexpr int SEL_MAX_CHUNKS = 1024;   // blocks per segment
constexpr int CMP_NT = 256;

// ---- 2b. compaction: block b of the split moves its candidates to the contiguous list at
// the sum of the counts of blocks < b, and (unordered mode) its emitted indices to out --------
template <typename K>
__device__ __forceinline__ void sel_compact_body(int N, int Ksel, int chunk, int nchunks, int emit,
                                                 SelState* __restrict__ st,
                                                 const K* __restrict__ bkey,
                                                 const int* __restrict__ bidx,
                                                 const int* __restrict__ eidx,
                                                 const int* __restrict__ ccnt,
                                                 const int* __restrict__ ecnt,
                                                 K* __restrict__ ckey, int* __restrict__ cidx,
                                                 int* __restrict__ out, int bx, int seg) {
  __shared__ int sh[16];
  const int tid = threadIdx.x, b = bx;
  const int* cc = ccnt + (long long)seg * nchunks;
  const int* ec = ecnt + (long long)seg * nchunks;
  int pc = 0, pe = 0;
  for (int c = tid; c < b; c += CMP_NT) {
    pc += cc[c];
    pe += ec[c];
  }
  const int oc = block_excl_scan_s(pc, sh), oe = block_excl_scan_s(pe, sh);
  // the block totals: exclusive scan of the last thread plus its own value
  __shared__ int s_oc, s_oe;
  if (tid == CMP_NT - 1) {
    s_oc = oc + pc;
    s_oe = oe + pe;
  }
  __syncthreads();
  const int offc = s_oc, offe = s_oe;
  const int nc = cc[b], ne = ec[b];
  const long long src = (long long)seg * N + (long long)b * chunk;
  const long long dst = (long long)seg * N + offc;
  for (int j = tid; j < nc; j += CMP_NT) {
    ckey[dst + j] = bkey[src + j];
    cidx[dst + j] = bidx[src + j];
  }
  if (emit) {
    int* o = out + (long long)seg * Ksel;
    for (int j = tid; j < ne; j += CMP_NT)
      if (offe + j < Ksel) o[offe + j] = eidx[src + j];
  }
  if (b == nchunks - 1 && tid == 0) {
    st[seg].cand_count = offc + nc;
    st[seg].out_count = offe + ne;
  }
}

// minimum of v over a 1024-thread block (every thread gets it); s: 16 entries of LDS
__device__ __forceinline__ u128 block_min_u128(u128 v, u128* s) {
  unsigned long long hi = (unsigned long long)(v >> 64), lo = (unsigned long long)v;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long h2 = __shfl_xor(hi, o, 64), l2 = __shfl_xor(lo, o, 64);
    if (h2 < hi || (h2 == hi && l2 < lo)) {
      hi = h2;
      lo = l2;
    }
  }
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s[w] = ((u128)hi << 64) | (u128)lo;
  __syncthreads();
  u128 m = s[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i)
    if (s[i] < m) m = s[i];
  __syncthreads();
  return m;
}

// ---- 3. refine over the candidates (one workgroup per segment) ----------------------------
// The first level scans the candidate list; from then on only the survivors of the previous
// level (the composite keys under the chosen prefix, usually a handful) are scanned, from LDS
// (back to the full list if they outgrow RF_CAP).  With ccnt set the candidates are read
// where the split left them (block b's at [b*chunk, b*chunk + ccnt[b])) instead of from the
// compacted list: the ordered mode needs no compaction launch.  With base set (ordered mode),
// base[b] = the number of selected elements in blocks < b, from the split's digit > d0 counts
// ecnt and the candidates >= T of each block: the write pass needs no count pass.
constexpr int RF_CAP = 2048;
template <typename K>
__device__ __forceinline__ void sel_refine_body(int N, int Ksel, int emit,
                                                SelState* __restrict__ st,
                                                const K* __restrict__ ckey,
                                                const int* __restrict__ cidx,
                                                int* __restrict__ out,
                                                const int* __restrict__ ccnt, int nchunks,
                                                int chunk, const int* __restrict__ ecnt,
                                                int* __restrict__ base, int seg) {
  __shared__ unsigned h[SEL_BINS];
  __shared__ u128 lst[2][RF_CAP];
  __shared__ int s_len[2];
  __shared__ int sh[16];
  __shared__ int s_digit, s_above, s_exit;
  __shared__ u128 s_min[16];
  __shared__ int s_out;
  __shared__ int s_pre[SEL_MAX_CHUNKS + 1];
  __shared__ int s_bc[SEL_MAX_CHUNKS];
  const int tid = threadIdx.x;
  const int IB = index_bits(N);
  const int TB = KeyBits<K>::KB + IB;
  int nc;
  if (ccnt) {   // exclusive prefix of the per-block candidate counts (nchunks <= 1024)
    const int v = tid < nchunks ? ccnt[(long long)seg * nchunks + tid] : 0;
    const int ex = block_excl_scan_s(v, sh);
    if (tid < nchunks) s_pre[tid] = ex;
    if (tid == nchunks - 1) s_pre[nchunks] = ex + v;
    __syncthreads();
    nc = s_pre[nchunks];
  } else {
    nc = st[seg].cand_count;
  }
  // storage position of candidate j: the last block b with s_pre[b] <= j holds it
  auto at = [&](int j) -> long long {
    if (!ccnt) return j;
    int lo = 0, hi = nchunks - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_pre[mid] <= j) lo = mid;
      else hi = mid - 1;
    }
    return (long long)lo * chunk + (j - s_pre[lo]);
  };
  const K* ck = ckey + (long long)seg * N;
  const int* ci = cidx + (long long)seg * N;
  if (tid == 0) s_out = 0;
  int r = st[seg].need0;
  // the candidates share the first digit d0; where it is the top SEL_DIG bits of c the radix
  // continues below it, else it starts over at the top of c (one more level)
  u128 prefix = KeyBits<K>::digit_is_prefix ? (u128)(unsigned)st[seg].d0 : (u128)0;
  int consumed = KeyBits<K>::digit_is_prefix ? SEL_DIG : 0;
  u128 T = 0;
  bool done = false;
  int cur = -1;   // survivors: -1 = the candidate list, else lst[cur][0 .. s_len[cur])
  // at most ceil(TB / SEL_DIG) levels; the bound only guards against a broken invariant
  for (int level = 0; !done && level < (TB + SEL_DIG - 1) / SEL_DIG; ++level) {
    const int width = min(SEL_DIG, TB - consumed);
    const int shift = TB - consumed - width;
    for (int i = tid; i < SEL_BINS; i += 1024) h[i] = 0u;
    if (tid == 0) {
      s_digit = 0;
      s_above = 0;
      s_exit = 1;
    }
    __syncthreads();
    const unsigned dmask = (1u << width) - 1u;
    if (cur < 0) {
      for (int j = tid; j < nc; j += 1024) {
        const long long q = at(j);
        const u128 c = composite<K>(ck[q], (unsigned)ci[q], N, IB);
        if ((c >> (shift + width)) == prefix) atomicAdd(&h[(unsigned)(c >> shift) & dmask], 1u);
      }
    } else {
      for (int j = tid; j < s_len[cur]; j += 1024)
        atomicAdd(&h[(unsigned)(lst[cur][j] >> shift) & dmask], 1u);
    }
    __syncthreads();
    const int nb = 1 << width;
    unsigned v[4];
    int S = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int rank = 4 * tid + j;
      v[j] = rank < nb ? h[nb - 1 - rank] : 0u;
      S += (int)v[j];
    }
    const int E = block_excl_scan_s(S, sh);   // (contains the barrier after the defaults)
    if (E < r && r <= E + S) {
      int cum = E;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (cum + (int)v[j] >= r) {
          s_digit = nb - 1 - (4 * tid + j);
          s_above = cum;
          s_exit = ((cum + (int)v[j] == r) || (shift == 0)) ? 1 : 0;
          break;
        }
        cum += (int)v[j];
      }
    }
    __syncthreads();
    const unsigned d = (unsigned)s_digit;
    prefix = (prefix << width) | (u128)d;
    r -= s_above;
    consumed += width;
    if (s_exit) {
      T = prefix << shift;
      if (!KeyBits<K>::digit_is_prefix && shift > 0) {
        // keys outside the candidate list can share these top bits (their first digit is
        // below d0, so they are smaller than every candidate): the threshold is the smallest
        // candidate under the prefix instead of the prefix's lower bound
        u128 mn = ~(u128)0;
        if (cur < 0) {
          for (int j = tid; j < nc; j += 1024) {
            const long long q = at(j);
            const u128 c = composite<K>(ck[q], (unsigned)ci[q], N, IB);
            if ((c >> shift) == prefix && c < mn) mn = c;
          }
        } else {
          for (int j = tid; j < s_len[cur]; j += 1024) {
            const u128 c = lst[cur][j];
            if ((c >> shift) == prefix && c < mn) mn = c;
          }
        }
        T = block_min_u128(mn, s_min);
      }
      done = true;
    } else {
      // keep the survivors: the keys whose bits above `shift` equal the new prefix
      const int nxt = (cur < 0) ? 0 : 1 - cur;
      if (tid == 0) s_len[nxt] = 0;
      __syncthreads();
      if (cur < 0) {
        for (int j = tid; j < nc; j += 1024) {
          const long long q = at(j);
          const u128 c = composite<K>(ck[q], (unsigned)ci[q], N, IB);
          if ((c >> shift) == prefix) {
            const int p = atomicAdd(&s_len[nxt], 1);
            if (p < RF_CAP) lst[nxt][p] = c;
          }
        }
      } else {
        for (int j = tid; j < s_len[cur]; j += 1024) {
          const u128 c = lst[cur][j];
          if ((c >> shift) == prefix) {
            const int p = atomicAdd(&s_len[nxt], 1);
            if (p < RF_CAP) lst[nxt][p] = c;
          }
        }
      }
      __syncthreads();
      cur = (s_len[nxt] <= RF_CAP) ? nxt : -1;
      if (cur >= 0 && s_len[cur] <= 1024) {
        // few survivors: the r-th largest of them directly, by rank (composites are distinct)
        const int S = s_len[cur];
        if (tid < S) {
          const u128 c = lst[cur][tid];
          int above = 0;
          for (int j = 0; j < S; ++j) above += lst[cur][j] > c ? 1 : 0;
          if (above == r - 1) s_min[0] = c;
        }
        __syncthreads();
        T = s_min[0];
        done = true;
      }
    }
    __syncthreads();
  }
  if (tid == 0) {
    st[seg].thr_hi = (unsigned long long)(T >> 64);
    st[seg].thr_lo = (unsigned long long)T;
  }
  if (base) {
    // selected per block: digit > d0 (split) + candidates >= T; then the exclusive prefix
    for (int b = tid; b < nchunks; b += 1024) s_bc[b] = 0;
    __syncthreads();
    for (int j = tid; j < nc; j += 1024) {
      const long long q = at(j);
      if (composite<K>(ck[q], (unsigned)ci[q], N, IB) >= T) atomicAdd(&s_bc[(int)(q / chunk)], 1);
    }
    __syncthreads();
    const int v = tid < nchunks ? s_bc[tid] + ecnt[(long long)seg * nchunks + tid] : 0;
    const int ex = block_excl_scan_s(v, sh);
    if (tid < nchunks) base[(long long)seg * nchunks + tid] = ex;
  }
  if (emit) {
    // after the emitted indices (placed by the compaction): the candidates >= T
    int* o = out + (long long)seg * Ksel;
    const int ne = st[seg].out_count;
    for (int j0 = 0; j0 < nc; j0 += 1024) {
      const int j = j0 + tid;
      const long long q = j < nc ? at(j) : 0;
      const bool sel = j < nc && composite<K>(ck[q], (unsigned)ci[q], N, IB) >= T;
      const int po = ne + wave_append(&s_out, sel);
      if (sel && po < Ksel) o[po] = ci[q];
    }
  }
}

// ---- 4. ordered compaction of {c >= T} -----------------------------------------------------
template <typename K>
__device__ __forceinline__ bool sel_pred(K k, int i, int N, int IB, u128 T) {
  return composite<K>(k, (unsigned)i, N, IB) >= T;
}

template <typename K>
__device__ __forceinline__ void sel_write_body(const K* __restrict__ keys, long long seg_stride,
                                               int N, int chunk, int nchunks, int Ksel,
                                               const SelState* __restrict__ st,
                                               const int* __restrict__ base0,
                                               int* __restrict__ out,
                                               unsigned* __restrict__ bits, int bx, int seg) {
  __shared__ int sh[16];
  __shared__ int s_tot;
  const int tid = threadIdx.x;
  const int IB = index_bits(N);
  const u128 T = ((u128)st[seg].thr_hi << 64) | (u128)st[seg].thr_lo;
  const K* kp = keys + (long long)seg * seg_stride;
  int base = base0[(long long)seg * nchunks + bx];
  int* o = out + (long long)seg * Ksel;
  const int begin = bx * chunk, end = min(N, begin + chunk);
  for (int b0 = begin; b0 < end; b0 += SEL_NT) {
    const int i = b0 + tid;
    const bool p = i < end && sel_pred<K>(kp[i], i, N, IB, T);
    if (bits) {
      // selection bitmap: each wave owns the two words of its 64 indices (b0 is a multiple of
      // 64), so every word of the segment is stored once, with plain stores
      const unsigned long long bal = __ballot(p);
      const int lane = tid & 63;
      const int i0 = i - lane;
      unsigned* bw = bits + (long long)seg * ((N + 31) / 32);
      if (lane == 0 && i0 < N) bw[i0 >> 5] = (unsigned)bal;
      if (lane == 32 && i0 + 32 < N) bw[(i0 + 32) >> 5] = (unsigned)(bal >> 32);
    }
    const int ex = block_excl_scan_s(p ? 1 : 0, sh);
    if (p && base + ex < Ksel) o[base + ex] = i;
    if (tid == SEL_NT - 1) s_tot = ex + (p ? 1 : 0);   // total of this round
    __syncthreads();
    base += s_tot;
    __syncthreads();
  }
}

// ---- one workgroup per segment -------------------------------------------------------------
// The whole select of a short segment in one launch.  Thread t owns the PER elements from
// t*PER on (storage order), their first digits packed in registers: histogram, the digit d0
// holding the K-th largest, a mask of the digit > d0 elements per thread, the digit == d0
// candidates in an LDS list narrowed by the 12 bits below the first digit (of the value
// rounded to FP32, as the first digit) and then by rank, and the selected indices written at
// the scan of the masks' counts (storage order, so ascending where that is the natural one).
// For the comb cutoff the same loop marks the approved-residue bitmaps.
// One CU does the work, so what bounds it is instructions per element: no ballots or index
// maps per element, only for the selected ones.
constexpr int SB_CAP = 2048;   // candidates kept in LDS
constexpr int SB_RANK = 64;    // survivors ranked against each other

// composite key: FP32 keys and their index fit 64 bits
template <typename K>
struct CompOf {
  using type = u128;
};
template <>
struct CompOf<unsigned int> {
  using type = unsigned long long;
};
template <typename K>
__device__ __forceinline__ typename CompOf<K>::type composite_n(K key, unsigned idx, int N,
                                                                int IB) {
  using CT = typename CompOf<K>::type;
  const K km = key & (K)(~((K)1 << KeyBits<K>::KB));
  return ((CT)km << IB) | (CT)(unsigned)((unsigned)(N - 1) - idx);
}

// the 12 bits below the first digit, of the same (rounded) value: non-decreasing in the key
// among keys of one first digit
__device__ __forceinline__ unsigned second_digit(unsigned key) { return (key >> 7) & 0xFFFu; }
__device__ __forceinline__ unsigned second_digit(unsigned long long key) {
  const float f = __double2float_rn(__longlong_as_double((long long)key));
  return (__float_as_uint(f) >> 7) & 0xFFFu;
}

// The bin of h[0, nb) holding the r-th largest element, the count above it and the bin's own
// count, to s_pick[0..2] (every thread calls; nb <= SEL_BINS, 1024 threads).
__device__ __forceinline__ void sb_pick(const unsigned* h, int nb, int r, int* sh, int* s_pick) {
  const int tid = threadIdx.x;
  unsigned v[4];
  int S = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int rank = 4 * tid + j;
    v[j] = rank < nb ? h[nb - 1 - rank] : 0u;
    S += (int)v[j];
  }
  const int E = block_excl_scan_s(S, sh);
  if (E < r && r <= E + S) {
    int cum = E;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (cum + (int)v[j] >= r) {
        s_pick[0] = nb - 1 - (4 * tid + j);
        s_pick[1] = cum;
        s_pick[2] = (int)v[j];
        break;
      }
      cum += (int)v[j];
    }
  }
  __syncthreads();
}

// a workgroup's LDS
template <typename K>
struct SelBlockLds {
  using CT = typename CompOf<K>::type;
  unsigned h[SEL_BINS];
  K lkey[SB_CAP];
  int lpos[SB_CAP];
  unsigned picked[SEL_NT];   // candidates selected, as their owners' bits
  CT rkey[SB_RANK];
  int rpos[SB_RANK];
  int sh[16];
  int s_pick[3];
  int s_nc;
  int ai[32], top[32];       // per location loop marked: its factor, its largest residue
};

template <typename K, int PER>
__device__ __forceinline__ void sel_block_body(const K* __restrict__ keys, long long seg_stride,
                                               int N, int Ksel, int* __restrict__ out,
                                               unsigned* __restrict__ bits, KeyMap km,
                                               const uint16_t* __restrict__ digits, int vec,
                                               const SelMark& mark, int seg,
                                               SelBlockLds<K>& lds) {
  using CT = typename CompOf<K>::type;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  auto& h = lds.h;
  auto& lkey = lds.lkey;
  auto& lpos = lds.lpos;
  auto& picked = lds.picked;
  auto& rkey = lds.rkey;
  auto& rpos = lds.rpos;
  auto& sh = lds.sh;
  auto& s_pick = lds.s_pick;
  int& s_nc = lds.s_nc;
  const int tid = threadIdx.x;
  const int IB = index_bits(N), TB = KeyBits<K>::KB + IB;
  const K* kp = keys + (long long)seg * seg_stride;
  const int i0 = tid * PER;
  auto comp_at = [&](K key, int i) __attribute__((always_inline)) {
    return composite_n<K>(key, (unsigned)key_natural(km, i), N, IB);
  };
  auto pick_one = [&](int i) __attribute__((always_inline)) {
    atomicOr(&picked[i / PER], 1u << (i % PER));
  };

  // 1. the first digits of the thread's elements, two per register; past N: 0xFFFF (no digit)
  unsigned pd[PER / 2];
  if (digits) {
    const uint16_t* dp = digits + (long long)seg * seg_stride;
#pragma unroll
    for (int j = 0; j < PER; j += 8) {
      if (vec && i0 + j + 8 <= N) {
        const u32x4 v = *(const u32x4*)(dp + i0 + j);
        pd[j / 2] = v.x;
        pd[j / 2 + 1] = v.y;
        pd[j / 2 + 2] = v.z;
        pd[j / 2 + 3] = v.w;
      } else {
#pragma unroll
        for (int u = 0; u < 8; u += 2) {
          const int i = i0 + j + u;
          const unsigned a = i < N ? dp[i] : 0xFFFFu, b = i + 1 < N ? dp[i + 1] : 0xFFFFu;
          pd[(j + u) / 2] = a | (b << 16);
        }
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < PER; j += 8) {
      K k[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) k[u] = kp[min(i0 + j + u, N - 1)];
#pragma unroll
      for (int u = 0; u < 8; u += 2) {
        const int i = i0 + j + u;
        const unsigned a = i < N ? top_digit<K>(k[u]) : 0xFFFFu;
        const unsigned b = i + 1 < N ? top_digit<K>(k[u + 1]) : 0xFFFFu;
        pd[(j + u) / 2] = a | (b << 16);
      }
    }
  }
  auto digit = [&](int j) __attribute__((always_inline)) {
    return (pd[j / 2] >> ((j & 1) * 16)) & 0xFFFFu;
  };
  for (int i = tid; i < SEL_BINS; i += SEL_NT) h[i] = 0u;
  picked[tid] = 0u;
  if (tid == 0) s_nc = 0;
  if (tid < mark.loops) {
    lds.ai[tid] = mark.ai[tid];
    lds.top[tid] = -1;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const unsigned d = digit(j);
    if (d < (unsigned)SEL_BINS) atomicAdd(&h[d], 1u);
  }
  __syncthreads();
  sb_pick(h, SEL_BINS, Ksel, sh, s_pick);
  const unsigned d0 = (unsigned)s_pick[0];
  int r = Ksel - s_pick[1];      // still to select among the candidates
  int nc = s_pick[2];
  unsigned sel = 0u, cand = 0u;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const unsigned d = digit(j);
    sel |= (unsigned)(d > d0 && d < (unsigned)SEL_BINS) << j;
    cand |= (unsigned)(d == d0) << j;
  }

  // 2. the r largest of the nc candidates
  if (nc == r) {
    sel |= cand;
  } else {
    bool small = nc <= SB_CAP;
    if (small) {
      for (unsigned m = cand; m; m &= m - 1) {
        const int i = i0 + __ffs(m) - 1;
        const int q = atomicAdd(&s_nc, 1);
        lkey[q] = kp[i];
        lpos[q] = i;
      }
      __syncthreads();   // (also: every thread has read s_pick and h)
      for (int i = tid; i < SEL_BINS; i += SEL_NT) h[i] = 0u;
      __syncthreads();
      for (int j = tid; j < nc; j += SEL_NT) atomicAdd(&h[second_digit(lkey[j])], 1u);
      __syncthreads();
      const int nc1 = nc;
      sb_pick(h, SEL_BINS, r, sh, s_pick);
      const int alive = s_pick[2], r1 = r - s_pick[1];
      if (alive == r1 || alive <= SB_RANK) {
        const unsigned d1 = (unsigned)s_pick[0];
        if (tid == 0) s_nc = 0;
        __syncthreads();
        for (int j = tid; j < nc1; j += SEL_NT) {
          const K key = lkey[j];
          const unsigned d = second_digit(key);
          if (d > d1 || (d == d1 && alive == r1)) {
            pick_one(lpos[j]);
          } else if (d == d1) {
            const int q = atomicAdd(&s_nc, 1);
            rkey[q] = comp_at(key, lpos[j]);
            rpos[q] = lpos[j];
          }
        }
        r = r1;
        nc = alive;
      } else {
        small = false;
      }
    }
    if (!small) {
      // many candidates share what was looked at (flat or tied data): narrow them by the
      // digits of the composite, whose index bits all differ, reading the keys again
      CT prefix = 0;
      int consumed = 0;
      do {
        const int width = min(SEL_DIG, TB - consumed), shift = TB - consumed - width;
        __syncthreads();
        for (int i = tid; i < SEL_BINS; i += SEL_NT) h[i] = 0u;
        __syncthreads();
        for (unsigned m = cand; m; m &= m - 1) {
          const int i = i0 + __ffs(m) - 1;
          const CT c = comp_at(kp[i], i);
          if (consumed == 0 || (c >> (shift + width)) == prefix)
            atomicAdd(&h[(unsigned)(c >> shift) & ((1u << width) - 1u)], 1u);
        }
        __syncthreads();
        sb_pick(h, 1 << width, r, sh, s_pick);
        prefix = (prefix << width) | (CT)(unsigned)s_pick[0];
        r -= s_pick[1];
        nc = s_pick[2];
        consumed += width;
      } while (nc > SB_RANK && nc != r);
      if (tid == 0) s_nc = 0;
      __syncthreads();
      for (unsigned m = cand; m; m &= m - 1) {
        const int i = i0 + __ffs(m) - 1;
        const CT c = comp_at(kp[i], i), pre = c >> (TB - consumed);
        if (pre > prefix || (pre == prefix && nc == r)) {
          pick_one(i);
        } else if (pre == prefix) {
          const int q = atomicAdd(&s_nc, 1);
          rkey[q] = c;
          rpos[q] = i;
        }
      }
    }
    __syncthreads();
    if (nc != r && tid < nc) {   // by rank: the composites are distinct
      const CT c = rkey[tid];
      int above = 0;
      for (int j = 0; j < nc; ++j) above += rkey[j] > c ? 1 : 0;
      if (above < r) pick_one(rpos[tid]);
    }
    __syncthreads();
    sel |= picked[tid];
  }

  // 3. the selection: as a bitmap, and as the index list in storage order
  if (bits) {
    unsigned* bw = bits + (long long)seg * ((N + 31) / 32);
    const int nb = (N + 31) / 32 * 32;   // every bit of every word is written
    if (i0 < nb) {
      if (PER == 8) ((uint8_t*)bw)[tid] = (uint8_t)sel;
      if (PER == 16) ((uint16_t*)bw)[tid] = (uint16_t)sel;
      if (PER == 32) bw[tid] = sel;
    }
  }
  int pos = block_excl_scan_s(__popc(sel), sh);
  int* o = out + (long long)seg * Ksel;
  for (unsigned m = sel; m; m &= m - 1) o[pos++] = (int)key_natural(km, i0 + __ffs(m) - 1);
  // the approved residues of each location loop and the largest one (the loops' factors from LDS:
  // a load of theirs per selected index waited for the atomics before it, n = 2^20, k = 1000: the
  // two cutoffs' launch 18.2 -> 15.1 us)
  for (int l = 0; l < mark.loops; ++l) {
    const unsigned a = (unsigned)lds.ai[l];
    unsigned* bm = mark.bitmap + (size_t)l * mark.bm_words;
    int v = -1;
    for (unsigned m = sel; m; m &= m - 1) {
      const unsigned f = ((unsigned)key_natural(km, i0 + __ffs(m) - 1) * a) & mark.wmask;
      atomicOr(&bm[f >> 5], 1u << (f & 31));
      v = max(v, (int)f);
    }
#pragma unroll
    for (int q = 32; q > 0; q >>= 1) v = max(v, __shfl_xor(v, q, 64));
    if ((tid & 63) == 0) atomicMax(&lds.top[l], v);
  }
  __syncthreads();
  if (tid < mark.loops && lds.top[tid] >= 0) atomicMax(&mark.maxfirst[tid], lds.top[tid]);
}

// ---- kernels: every workgroup of a launch belongs to a job (sfft_jobs.h); one select is a
// launch of one job, its workgroups in the grid's (x, y) ---------------------------------------
struct SelOne {   // one select: its job, by value
  SelJob j;
  __device__ __forceinline__ bool get(SelJob& out, int& bx, int& seg, int) const {
    out = j;
    bx = blockIdx.x;
    seg = blockIdx.y;
    return true;
  }
};
struct SelMany {  // many selects: per x workgroups of a job (0: its chunks) and segment
  JobsDev t;
  __device__ __forceinline__ bool get(SelJob& out, int& bx, int& seg, int per) const {
    const SelJob* j = job_here<SelJob>(t);
    if (!j) return false;
    out = *j;
    const int i = (int)blockIdx.x - j->block0, nx = per ? per : j->nchunks;
    bx = i % nx;
    seg = i / nx;
    return true;
  }
};

template <typename K, typename From>
__global__ __launch_bounds__(SEL_NT) void sel_hist0_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (!f.get(j, bx, seg, 0)) return;
  sel_hist0_body<K>((const K*)j.keys, j.seg_stride, j.N, j.chunk, j.nchunks, j.rows, j.digits, bx,
                    seg);
}
template <typename From>
__global__ __launch_bounds__(PICK_NT) void sel_colsum_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (!f.get(j, bx, seg, SEL_BINS / PICK_BINS)) return;
  sel_colsum_body(j.nchunks, j.rows, const_cast<unsigned*>(j.sums), bx, seg);
}
template <typename K, typename From>
__global__ __launch_bounds__(SEL_NT) void sel_split_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (!f.get(j, bx, seg, 0)) return;
  sel_split_body<K>((const K*)j.keys, j.seg_stride, j.N, j.chunk, j.nchunks, j.ordered ? 0 : 1, j.K,
                    j.sums, j.nsum, (SelState*)j.state, (K*)j.blk_key, j.blk_idx, j.emit_idx, j.ccnt,
                    j.ecnt, j.map, j.digits, bx, seg);
}
// unordered: the candidates of the split's blocks side by side, its winners to the output
template <typename K, typename From>
__global__ __launch_bounds__(CMP_NT) void sel_compact_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (!f.get(j, bx, seg, 0)) return;
  sel_compact_body<K>(j.N, j.K, j.chunk, j.nchunks, 1, (SelState*)j.state, (const K*)j.blk_key,
                      j.blk_idx, j.emit_idx, j.ccnt, j.ecnt, (K*)j.cand_key, j.cand_idx, j.out, bx,
                      seg);
}
// ordered: the refine reads the candidates from the split's per-block regions
template <typename K, typename From>
__global__ __launch_bounds__(1024) void sel_refine_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (!f.get(j, bx, seg, 1)) return;
  const bool o = j.ordered != 0;
  sel_refine_body<K>(j.N, j.K, o ? 0 : 1, (SelState*)j.state,
                     (const K*)(o ? j.blk_key : j.cand_key), o ? j.blk_idx : j.cand_idx, j.out,
                     o ? j.ccnt : nullptr, j.nchunks, j.chunk, o ? j.ecnt : nullptr,
                     o ? j.cnt : nullptr, seg);
}
template <typename K, typename From>
__global__ __launch_bounds__(SEL_NT) void sel_write_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (!f.get(j, bx, seg, 0)) return;
  sel_write_body<K>((const K*)j.keys, j.seg_stride, j.N, j.chunk, j.nchunks, j.K,
                    (const SelState*)j.state, j.cnt, j.out, j.bits, bx, seg);
}
// a segment that one workgroup does: 8, 16 or 32 elements per thread
template <typename K>
__device__ __forceinline__ void sel_block_any(const SelJob& j, int seg) {
  __shared__ SelBlockLds<K> lds;
  const K* keys = (const K*)j.keys;
  if (j.N <= 8 * SEL_NT)
    sel_block_body<K, 8>(keys, j.seg_stride, j.N, j.K, j.out, j.bits, j.map, j.digits, j.vec,
                         j.mark, seg, lds);
  else if (j.N <= 16 * SEL_NT)
    sel_block_body<K, 16>(keys, j.seg_stride, j.N, j.K, j.out, j.bits, j.map, j.digits, j.vec,
                          j.mark, seg, lds);
  else
    sel_block_body<K, 32>(keys, j.seg_stride, j.N, j.K, j.out, j.bits, j.map, j.digits, j.vec,
                          j.mark, seg, lds);
}
template <typename K, typename From>
__global__ __launch_bounds__(SEL_NT) void sel_block_kernel(From f) {
  SelJob j;
  int bx, seg;
  if (f.get(j, bx, seg, 1)) sel_block_any<K>(j, seg);
}
// two selects, a workgroup per segment of either
template <typename K>
__global__ __launch_bounds__(SEL_NT) void sel_pair_kernel(SelJob a, SelJob b) {
  const bool first = (int)blockIdx.x < a.segs;
  sel_block_any<K>(first ? a : b, first ? (int)blockIdx.x : (int)blockIdx.x - a.segs);
}

// Up to 32768 keys one workgroup beats the chain of launches, in both precisions; at 65536 its
// one CU takes as long as the launches it saves (whole graph transforms, chain -> one workgroup:
// comb of 8192 keys FP64 128 -> 95 us, FP32 128 -> 96; 16384: 151 -> 117, 150 -> 115; 32768:
// 143 -> 112, 139 -> 113; 65536: 153.4 -> 158.5, 141 -> 153).
constexpr int SB_MAX_N = 32768;
bool select_in_block(int N) { return N <= SB_MAX_N; }

// the job of one select_topk call
static hipError_t select_job(SelJob& j, const void* keys, long long seg_stride, int N,
                             int K, int segs, int* out, int ordered, const SelectWork& w,
                             unsigned* bits, const KeyMap* map, const uint16_t* digits,
                             const SelMark* mark, const unsigned* hist) {
  // the write pass reads the keys
  if (ordered && digits && !select_in_block(N)) return hipErrorInvalidValue;
  if (mark && !select_in_block(N)) return hipErrorInvalidValue;   // the one-workgroup select marks
  if (N < 2 || K < 1 || K > N || segs < 1) return hipErrorInvalidValue;
  if (!hist && !w.hist && !select_in_block(N)) return hipErrorInvalidValue;
  j = SelJob();
  j.chunk = sel_chunk(N);
  j.nchunks = (N + j.chunk - 1) / j.chunk;
  if (j.nchunks > SEL_MAX_CHUNKS || j.nchunks > w.max_chunks || segs > w.max_segs)
    return hipErrorInvalidValue;
  if (map && map->mid != 0) {
    // the ordered compaction walks storage order: natural order only
    if (ordered || (1LL << map->log2n) != (long long)N) return hipErrorInvalidValue;
    j.map = *map;
  }
  j.keys = keys;
  j.seg_stride = seg_stride;
  j.N = N;
  j.K = K;
  j.ordered = ordered;
  j.segs = segs;
  j.vec = ((uintptr_t)digits & 15) == 0 && (seg_stride & 7) == 0;   // 16-byte loads of digits
  // work layout: column sums, then the per-block histogram rows
  j.sums = hist ? hist : w.hist;
  j.nsum = hist ? kSelCopies : 1;
  j.rows = w.hist ? w.hist + (size_t)segs * SEL_BINS : nullptr;
  j.state = w.state;
  j.blk_key = w.blk_key;
  j.blk_idx = w.blk_idx;
  j.emit_idx = w.emit_idx;
  j.ccnt = w.ccnt;
  j.ecnt = w.ecnt;
  j.cand_key = w.cand_key;
  j.cand_idx = w.cand_idx;
  j.cnt = w.cnt;
  j.out = out;
  j.bits = bits;
  j.digits = digits;
  if (mark) j.mark = *mark;
  return hipSuccess;
}

template <typename K>
static hipError_t select_one(const SelJob& j, hipStream_t st) {
  const SelOne f{j};
  const dim3 wide(j.nchunks, j.segs);
  if (select_in_block(j.N)) {
    hipLaunchKernelGGL((sel_block_kernel<K, SelOne>), dim3(1, j.segs), dim3(SEL_NT), 0, st, f);
    return hipGetLastError();
  }
  if (j.nsum == 1) {   // no histograms at hand
    hipLaunchKernelGGL((sel_hist0_kernel<K, SelOne>), wide, dim3(SEL_NT), 0, st, f);
    hipLaunchKernelGGL((sel_colsum_kernel<SelOne>), dim3(SEL_BINS / PICK_BINS, j.segs),
                       dim3(PICK_NT), 0, st, f);
  }
  // (the split blocks pick d0 from the sums themselves)
  hipLaunchKernelGGL((sel_split_kernel<K, SelOne>), wide, dim3(SEL_NT), 0, st, f);
  if (!j.ordered)
    hipLaunchKernelGGL((sel_compact_kernel<K, SelOne>), wide, dim3(CMP_NT), 0, st, f);
  hipLaunchKernelGGL((sel_refine_kernel<K, SelOne>), dim3(1, j.segs), dim3(1024), 0, st, f);
  if (j.ordered)
    hipLaunchKernelGGL((sel_write_kernel<K, SelOne>), wide, dim3(SEL_NT), 0, st, f);
  return hipGetLastError();
}

hipError_t select_topk(int is_fp32, const void* keys, long long seg_stride, int N, int K,
                       int segs, int* out, int ordered, const SelectWork& w, hipStream_t st,
                       unsigned* bits, const KeyMap* map, const uint16_t* digits,
                       const SelMark* mark, const unsigned* hist) {
  SelJob j;
  const hipError_t e = select_job(j, keys, seg_stride, N, K, segs, out, ordered, w, bits,
                                  map, digits, mark, hist);
  if (e != hipSuccess) return e;
  return is_fp32 ? select_one<unsigned int>(j, st) : select_one<unsigned long long>(j, st);
}

hipError_t select_pair(int is_fp32, const SelectArgs& comb, const SelectArgs& bucket,
                       hipStream_t st) {
  SelJob j[2];
  const SelectArgs* args[2] = {&comb, &bucket};
  for (int i = 0; i < 2; ++i) {
    const SelectArgs& s = *args[i];
    if (!select_in_block(s.N)) return hipErrorInvalidValue;
    const hipError_t e = select_job(j[i], s.keys, s.seg_stride, s.N, s.K, s.segs, s.out, i,
                                    *s.w, s.bits, s.map, s.digits, s.mark, nullptr);
    if (e != hipSuccess) return e;
  }
  const dim3 grid(comb.segs + bucket.segs);
  if (is_fp32)
    hipLaunchKernelGGL((sel_pair_kernel<unsigned int>), grid, dim3(SEL_NT), 0, st, j[0], j[1]);
  else
    hipLaunchKernelGGL((sel_pair_kernel<unsigned long long>), grid, dim3(SEL_NT), 0, st, j[0],
                       j[1]);
  return hipGetLastError();
}

hipError_t select_jobs_add(SelGroup& g, int is_fp32, const void* keys, long long seg_stride, int N,
                           int K, int segs, int* out, int ordered, const SelectWork& w,
                           unsigned* bits, const KeyMap* map, const uint16_t* digits,
                           const SelMark* mark, const unsigned* hist) {
  SelJob j;
  const hipError_t e = select_job(j, keys, seg_stride, N, K, segs, out, ordered, w, bits,
                                  map, digits, mark, hist);
  if (e != hipSuccess) return e;
  // a whole round of the split's loads per workgroup: many segments fill the chip by themselves,
  // and each workgroup first reads the segment's histograms (64 KB), which shorter chunks do not
  // pay for (64 signals' comb cutoffs of 2^16..2^18 keys: split 117 -> 43 us)
  if (j.chunk < SPLIT_ROUND) {
    j.chunk = SPLIT_ROUND;
    j.nchunks = (N + j.chunk - 1) / j.chunk;
  }
  g.fp32 = is_fp32;
  if (select_in_block(N)) {
    g.block.add(j, segs);
  } else {
    g.wide.add(j, j.nchunks * segs);
    g.refine.add(j, segs);
  }
  return hipSuccess;
}

// every select of the group is ordered, or none is (a batch's bucket cutoffs, or its combs')
template <typename K>
static hipError_t select_many(const SelGroup& g, hipStream_t st) {
  if (g.block.dev.blocks)
    hipLaunchKernelGGL((sel_block_kernel<K, SelMany>), dim3(g.block.dev.blocks), dim3(SEL_NT), 0,
                       st, SelMany{g.block.dev});
  if (g.wide.dev.blocks) {
    const SelMany wide{g.wide.dev}, refine{g.refine.dev};
    const dim3 nw(wide.t.blocks);
    const bool ordered = g.wide.jobs[0].ordered != 0;
    hipLaunchKernelGGL((sel_split_kernel<K, SelMany>), nw, dim3(SEL_NT), 0, st, wide);
    if (!ordered)
      hipLaunchKernelGGL((sel_compact_kernel<K, SelMany>), nw, dim3(CMP_NT), 0, st, wide);
    hipLaunchKernelGGL((sel_refine_kernel<K, SelMany>), dim3(refine.t.blocks), dim3(1024), 0, st,
                       refine);
    if (ordered)
      hipLaunchKernelGGL((sel_write_kernel<K, SelMany>), nw, dim3(SEL_NT), 0, st, wide);
  }
  return hipGetLastError();
}

hipError_t select_jobs_launch(const SelGroup& g, hipStream_t st) {
  return g.fp32 ? select_many<unsigned int>(g, st) : select_many<unsigned long long>(g, st);
}

}  // namespace sfft
