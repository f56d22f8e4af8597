// sfft_jobs.h -- one launch of a kernel for the jobs of many signals.
//
// A batch runs every stage of all its signals as one launch: a table of jobs (one signal's
// arguments for the stage) and, per workgroup of the launch, the job it belongs to.  The
// kernels call the single transform's own device bodies with the job's arguments and the
// workgroup's index within the job, so a batch computes the single transform's bits.
#pragma once
#include <cstring>
#include <vector>

#include "sfft_internal.h"

namespace sfft {

// device side of a table
struct JobsDev {
  const void* jobs = nullptr;
  const int* map = nullptr;   // job of each workgroup, or -1 (padding)
  int blocks = 0;
};

// the bytes of every table of a batch, uploaded together
struct JobPack {
  std::vector<char> bytes;
  size_t put(const void* p, size_t n) {
    const size_t at = (bytes.size() + 255) / 256 * 256;
    bytes.resize(at + (n ? n : 1));
    if (n) memcpy(&bytes[at], p, n);
    return at;
  }
};

// Job: a plain struct with an int block0, its first workgroup.  Jobs start at multiples of 8
// workgroups, so that a workgroup's index within its job modulo 8 names its XCD, as in a launch
// of the job alone.
template <typename Job>
struct JobTable {
  std::vector<Job> jobs;
  std::vector<int> map;
  JobsDev dev;
  size_t at_jobs = 0, at_map = 0;
  void add(Job j, int blocks) {
    map.resize((map.size() + 7) / 8 * 8, -1);
    j.block0 = (int)map.size();
    map.resize(map.size() + (size_t)blocks, (int)jobs.size());
    jobs.push_back(j);
  }
  void pack(JobPack& p) {
    at_jobs = p.put(jobs.data(), jobs.size() * sizeof(Job));
    at_map = p.put(map.data(), map.size() * sizeof(int));
  }
  void bind(const char* base) {
    dev.jobs = base + at_jobs;
    dev.map = (const int*)(base + at_map);
    dev.blocks = (int)map.size();
  }
};

#if defined(__HIPCC__)
// this workgroup's job, or nullptr; the same for every lane, so its fields load as scalars
template <typename Job>
__device__ __forceinline__ const Job* job_here(const JobsDev& t) {
  const int j = __builtin_amdgcn_readfirstlane(t.map[blockIdx.x]);
  return j < 0 ? nullptr : (const Job*)t.jobs + j;
}
#endif

// ---- FFT passes ----------------------------------------------------------------------------
struct PassArgs {
  const void* in;
  long long in_bstride;
  void* out;
  long long out_bstride;
  void* keys;
  long long keys_bstride;
  int key_batches;
  int log2N, r, log2Lprev, log2Q;
  int small_tile;   // a tile of a quarter of the elements and threads (pass_shape)
  int inverse;
  const void* twR;
  const void* tw4;      // radix-4 stage twiddle quads (see fft_tables_create)
  const void* thi;
  const void* tlo;
  int s;
  const void* comb_x;
  const int* comb_offs;
  int comb_sigma;
  int nbatch;
  int keys_tiled;   // store keys at tile * TE + e (the tile's own contiguous range)
  uint16_t* digits; // optional first digits of the keys (same positions)
  unsigned* hist;   // optional histograms of the first digits (FftLaunch::hist)
  int log2nlo, log2m;   // kLoadCombRows: g at in[(g mod 2^log2nlo) << log2m | g >> log2nlo]
  const int* perm;      // kLoadPerm: g of batch b at in[g * perm[b] mod 2^log2N]
  const int* perm_inv;  // kLoadPerm: the inverse of perm[b] mod 2^log2N
  int taps;             // kLoadTaps
  long long head;       // kStoreHead
  double scale;         // kStoreHead
};
struct FftJob {
  PassArgs a;
  int tiles, block0;
};
// the jobs of one kernel variant, run in the order of their pass
struct FftGroup {
  int pass = 0, load = 0, store = 0, tw = 0, small_tile = 0, fp32 = 0;
  JobTable<FftJob> t;
};
// appends the passes of L to their groups (comb gathers, plain, comb rows and column-permuted
// first passes; every pass of a smaller index is to run first)
hipError_t fft_jobs_add(std::vector<FftGroup>& g, const FftLaunch& L);
hipError_t fft_jobs_launch(std::vector<FftGroup>& g, hipStream_t st);

// ---- slab fold -----------------------------------------------------------------------------
struct SlabArgs {
  const void* x;
  const void* fT;       // bucket-major filter rows
  void* bins;
  const int* a_dev;
  const int* ai_dev;
  uint32_t mask;
  int log2B, log2m, w, loops, tiled, T, P, log2sc;
  void* yc;             // comb samples
  const int* offs;
  int Rl, log2sigma;
  FoldClear clr;
};
struct SlabJob {
  SlabArgs a;
  int groups, block0;   // workgroups that share the signal's slabs
};
// the signals of a batch whose slabs fit two workgroups per CU, or the others (one launch each):
// the kernel variant of the most taps per bucket, with the LDS of the largest
struct SlabGroup {
  int pmax = 0, fp32 = 0, wide = 0;
  size_t lds = 0;
  std::vector<SlabArgs> args;
  JobTable<SlabJob> t;
};
// the arguments of fold_columns_launch with by_column = 1
hipError_t slab_jobs_add(std::vector<SlabGroup>& groups, int is_fp32, const void* x, const void* fT, void* bins,
                         const int* a_dev, const int* ai_dev, int n, int B, int w, int loops,
                         int tiled, void* yc, const int* offs, int Rl, int W,
                         const FoldClear& clr);
// shares the card's resident workgroups out among the signals (after the last add)
void slab_jobs_share(std::vector<SlabGroup>& groups);
hipError_t slab_jobs_launch(const std::vector<SlabGroup>& groups, hipStream_t st);

// ---- top-K select --------------------------------------------------------------------------
struct SelJob {
  const void* keys;
  long long seg_stride;
  int N, K, chunk, nchunks, ordered, vec, segs;
  unsigned* rows;
  const unsigned* sums; // nsum histograms per segment, summed by the split
  int nsum;
  void* state;
  void* blk_key;
  int* blk_idx;
  int* emit_idx;
  int* ccnt;
  int* ecnt;
  void* cand_key;
  int* cand_idx;
  int* cnt;
  int* out;
  unsigned* bits;
  KeyMap map;
  const uint16_t* digits;
  SelMark mark;
  int block0;
};
struct SelGroup {
  int fp32 = 0;
  JobTable<SelJob> block;      // one workgroup does a segment
  JobTable<SelJob> wide;       // nchunks x segs workgroups: split, compact / write
  JobTable<SelJob> refine;     // one workgroup per segment
  void pack(JobPack& p) {
    block.pack(p);
    wide.pack(p);
    refine.pack(p);
  }
  void bind(const char* base) {
    block.bind(base);
    wide.bind(base);
    refine.bind(base);
  }
};
// the arguments of select_topk (hist: where one workgroup does not do a segment)
hipError_t select_jobs_add(SelGroup& g, int is_fp32, const void* keys, long long seg_stride, int N,
                           int K, int segs, int* out, int ordered, const SelectWork& w,
                           unsigned* bits, const KeyMap* map, const uint16_t* digits,
                           const SelMark* mark, const unsigned* hist);
hipError_t select_jobs_launch(const SelGroup& g, hipStream_t st);

// ---- reverse hash, estimation --------------------------------------------------------------
struct HashJob {
  HashArgs h;
  int blocks, block0;
};
void hash_jobs_clear(JobTable<HashJob>& t, const HashArgs& h);
void hash_jobs_bitmap(JobTable<HashJob>& t, const HashArgs& h);
hipError_t hash_clear_jobs(const JobTable<HashJob>& t, hipStream_t st);
hipError_t hash_bitmap_jobs(const JobTable<HashJob>& t, hipStream_t st);

struct NodeGroup {
  int loops = 0, fp32 = 0;
  JobTable<NodeJob> t;
};
void nodes_jobs_add(std::vector<NodeGroup>& g, int is_fp32, NodeJob j);
hipError_t nodes_jobs_launch(const std::vector<NodeGroup>& g, hipStream_t st);

}  // namespace sfft
