// sfft_batch.hip -- many signals of uneven n and k transformed as one batch.
//
// Each signal keeps its own plan (parameters, workspace).  One batch execution runs every stage
// of ALL its signals as one launch (sfft_jobs.h: a table of the signals' arguments, and each
// workgroup's signal), so
// small and large signals share the chip and a batch of any size takes about twenty launches.
// (One launch per signal and stage took 16-25 launches of a few us per signal: 64 complex64
// signals of 2^18..2^24, 6.3 ms on four streams, 2.6 ms as one launch per stage.)
// Signals whose plan takes the column front end (AUTO, where the slab applies) are folded by one
// slab launch, which also copies their comb samples; the others are gathered by one persistent
// permute+filter launch (all 64 gathered: permute+filter 1074 us, comb gather 363 us; slab
// 763 us and comb first passes 150 us, the whole batch 2.57 -> 2.04 ms).
// Two chains run beside each other, as in a single transform: the comb chain (comb FFT, comb
// cutoff, approved bitmaps) on a second stream, and bucket FFT and bucket cutoff (after the
// permute+filter) on the batch stream; joined there, the reverse hash and the estimation follow.
// The draws of all signals go up in one copy.  With graphs the two chains are captured once as
// one graph and replayed (buffers are cleared by kernels, so it holds no memset nodes).  New
// signal or node pointers change the tables' contents alone: they are built again in pinned memory
// and uploaded in stream order, without a wait and under the same graph; new filters or tuned
// shapes drop the graph as well.
//
// Autotuner: times, on the batch itself, only launch shapes that compute the same bits --
// the permute+filter loops per thread, block size and persistent grid (every shape runs the
// same per-bucket body in the same tap order), and the FFT columns per tile of the comb and
// bucket FFTs (columns are independent transforms) -- and keeps the fastest.
#include <algorithm>
#include <cstring>
#include <vector>

#include "sfft_plan_impl.h"
#include "sfft_jobs.h"

struct sfft_batch {
  int count = 0;
  int fp32 = 0;
  hipStream_t st = nullptr;
  int own_st = 0;                    // st created here (a graph cannot capture stream 0)
  hipStream_t st2 = nullptr;         // the comb chain
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  std::vector<sfft_plan*> plans;
  // job tables of every stage, in one device buffer
  std::vector<PfJob> jobs;           // gathering signals
  std::vector<SlabGroup> slab;                    // signals with the column front end
  int total_items = 0;
  int lpt = 3, nt = 256, grid = 2048;
  std::vector<FftGroup> comb, comb_slab, bucket;   // combs gathered, combs the slab fold copied
  SelGroup sel_comb, sel_bucket;
  JobTable<HashJob> clear, bitmap;
  std::vector<NodeGroup> est;
  char* d_tab = nullptr;
  char* h_tab = nullptr;             // pinned
  size_t tab_bytes = 0;              // of either
  hipEvent_t tab_ev = nullptr;       // last upload out of h_tab
  int tab_pending = 0;
  const PfJob* d_jobs = nullptr;
  bool tab_shape = false;            // the tables are those of the current filters and shapes
  std::vector<const void*> tab_x;    // the pointers the tables hold: signals, nodes
  std::vector<Node*> tab_nodes;
  // the draws of all signals: signal i's (a, ai, offsets) at draw_at[i]
  int* d_draws = nullptr;
  int* h_draws = nullptr;            // pinned
  std::vector<size_t> draw_at;
  size_t draw_ints = 0;
  hipEvent_t up_ev = nullptr;        // last upload out of h_draws
  int up_pending = 0;
  // per-signal hit counts, contiguous; the estimation also stores them into h_counts (pinned)
  int* d_counts = nullptr;
  int* h_counts = nullptr;
  int* h_counts_dev = nullptr;
  int use_graph = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

static void drop_graph(sfft_batch* b) {
  if (b->exec) {
    (void)hipStreamSynchronize(b->st);   // (it may still run)
    (void)hipGraphExecDestroy(b->exec);
  }
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
}

// filters or launch shapes change: tables of another layout, and other launches
static void drop_tables(sfft_batch* b) {
  drop_graph(b);
  b->tab_x.clear();
  b->tab_shape = false;
}

extern "C" void sfft_batch_destroy(sfft_batch* b) {
  if (!b) return;
  (void)hipStreamSynchronize(b->st);
  if (b->st2) (void)hipStreamSynchronize(b->st2);
  drop_graph(b);
  for (auto p : b->plans) sfft_plan_destroy(p);
  if (b->st2) (void)hipStreamDestroy(b->st2);
  if (b->ev_fork) (void)hipEventDestroy(b->ev_fork);
  if (b->ev_join) (void)hipEventDestroy(b->ev_join);
  if (b->up_ev) (void)hipEventDestroy(b->up_ev);
  if (b->own_st && b->st) (void)hipStreamDestroy(b->st);
  if (b->tab_ev) (void)hipEventDestroy(b->tab_ev);
  if (b->d_tab) (void)hipFree(b->d_tab);
  if (b->h_tab) (void)hipHostFree(b->h_tab);
  if (b->d_draws) (void)hipFree(b->d_draws);
  if (b->h_draws) (void)hipHostFree(b->h_draws);
  if (b->d_counts) (void)hipFree(b->d_counts);
  if (b->h_counts) (void)hipHostFree(b->h_counts);
  delete b;
}

static sfft_status pack_tables(sfft_batch* b, const void* const* d_x, Node* const* nodes,
                               JobPack& pack, size_t* at_jobs);
static sfft_status reserve_tables(sfft_batch* b, size_t bytes);

extern "C" sfft_status sfft_batch_create(const sfft_params* params, int count,
                                         sfft_precision prec, void* stream, sfft_batch** out) {
  if (!params || count <= 0 || !out) return SFFT_ERR_INVALID;
  *out = nullptr;
  for (int i = 0; i < count; ++i) {
    const sfft_status s = sfft_params_validate(&params[i]);
    if (s != SFFT_OK) return s;
    // AUTO: the column slab fold where it applies, else gathers
    if (params[i].front_end != SFFT_FRONT_AUTO && params[i].front_end != SFFT_FRONT_GATHER)
      return SFFT_ERR_INVALID;
  }
  sfft_batch* b = new sfft_batch();
  b->count = count;
  b->fp32 = prec == SFFT_FP32;
  b->st = (hipStream_t)stream;
  if (!b->st) {
    if (hipStreamCreateWithFlags(&b->st, hipStreamNonBlocking) != hipSuccess) {
      delete b;
      return SFFT_ERR_HIP;
    }
    b->own_st = 1;
  }
  for (int i = 0; i < count; ++i) {
    sfft_plan* p = nullptr;
    const sfft_status s = sfft_plan_create(&params[i], prec, b->st, &p);
    if (s != SFFT_OK) {
      sfft_batch_destroy(b);
      return s;
    }
    b->plans.push_back(p);
  }
  for (int i = 0; i < count; ++i) {
    b->draw_at.push_back(b->draw_ints);
    const size_t ints = (size_t)(2 * params[i].loops + params[i].RLFC_loops);
    b->draw_ints += (ints + 15) / 16 * 16;
  }
  const bool ok =
      hipStreamCreateWithFlags(&b->st2, hipStreamNonBlocking) == hipSuccess &&   // default priority
      hipEventCreateWithFlags(&b->ev_fork, hipEventDisableTiming) == hipSuccess &&
      hipEventCreateWithFlags(&b->ev_join, hipEventDisableTiming) == hipSuccess &&
      hipEventCreateWithFlags(&b->up_ev, hipEventDisableTiming) == hipSuccess &&
      hipEventCreateWithFlags(&b->tab_ev, hipEventDisableTiming) == hipSuccess &&
      dev_alloc((void**)&b->d_draws, sizeof(int) * b->draw_ints) == hipSuccess &&
      hipHostMalloc((void**)&b->h_draws, sizeof(int) * b->draw_ints, hipHostMallocDefault) ==
          hipSuccess &&
      dev_alloc((void**)&b->d_counts, sizeof(int) * (size_t)count) == hipSuccess &&
      hipHostMalloc((void**)&b->h_counts, sizeof(int) * (size_t)count, hipHostMallocDefault) ==
          hipSuccess &&
      hipHostGetDevicePointer((void**)&b->h_counts_dev, b->h_counts, 0) == hipSuccess;
  if (!ok) {
    sfft_batch_destroy(b);
    return SFFT_ERR_ALLOC;
  }
  memset(b->h_draws, 0, sizeof(int) * b->draw_ints);
  for (int i = 0; i < count; ++i) {   // the plans read their draws from the batch's block
    sfft_plan* P = b->plans[i];
    P->d_a = b->d_draws + b->draw_at[i];
    P->d_ai = P->d_a + P->p.loops;
    P->d_offs = P->d_a + 2 * P->p.loops;
  }
  // the tables' memory: their size is known from the shapes
  const std::vector<const void*> no_x(count, nullptr);
  const std::vector<Node*> no_nodes(count, nullptr);
  JobPack pack;
  size_t at_jobs = 0;
  if (pack_tables(b, no_x.data(), no_nodes.data(), pack, &at_jobs) == SFFT_OK &&
      reserve_tables(b, pack.bytes.size()) != SFFT_OK) {
    sfft_batch_destroy(b);
    return SFFT_ERR_ALLOC;
  }
  *out = b;
  return SFFT_OK;
}

extern "C" sfft_plan* sfft_batch_plan(sfft_batch* b, int i) {
  return (b && i >= 0 && i < b->count) ? b->plans[i] : nullptr;
}

extern "C" sfft_status sfft_batch_set_filter(sfft_batch* b, int i, const void* d_filter_time,
                                             const complex_t* h_filter_win) {
  if (!b || i < 0 || i >= b->count) return SFFT_ERR_INVALID;
  drop_tables(b);   // (they hold the taps pointer)
  return sfft_plan_set_filter(b->plans[i], d_filter_time, h_filter_win);
}

// (re)builds every stage's job table for the current shapes and pointers: signal i reads d_x[i]
// and its nodes go to nodes[i] (the device view of pinned host memory, with a copy in the plan's
// buffer; nullptr: the plan's buffer alone).  Where only pointers differ from the tables before,
// every table keeps its size and place, so a captured graph of the launches stays valid.
static sfft_status pack_tables(sfft_batch* b, const void* const* d_x, Node* const* nodes,
                               JobPack& pack, size_t* at_jobs) {
  b->jobs.clear();
  b->slab.clear();
  b->comb.clear();
  b->comb_slab.clear();
  b->bucket.clear();
  b->est.clear();
  b->sel_comb = SelGroup();
  b->sel_bucket = SelGroup();
  b->clear = b->bitmap = JobTable<HashJob>();
  int item = 0;
  for (int i = 0; i < b->count; ++i) {
    const sfft_plan* P = b->plans[i];
    const sfft_params& p = P->p;
    const int tiled = (p.fold_mode == SFFT_FOLD_REFERENCE) && (p.n < (1 << 27));
    const HashArgs h = hash_args(P, b->d_counts + i);
    if (P->columns) {
      FoldClear clr;   // the slab fold clears for the transform, as a single one's does
      clr.bm = h.bitmap;
      clr.nbm = h.clear_words;
      clr.maxf = (uint32_t*)h.maxfirst;
      clr.nmax = h.loops_loc;
      HIPCK(slab_jobs_add(b->slab, b->fp32, d_x[i], P->frows, P->bins_t, P->d_a, P->d_ai, p.n, p.B,
                          p.w, p.loops, tiled, P->comb_y, P->d_offs, p.RLFC_loops, p.W_RLFC,
                          clr));
    } else {
      PfJob J;
      J.x = d_x[i];
      J.f = P->d_ft;
      J.bins = P->bins_t;
      J.ai = P->d_ai;
      J.mask = (uint32_t)p.n - 1u;
      J.B = p.B;
      J.w = p.w;
      J.loops = p.loops;
      J.tiled = tiled;
      J.item0 = item;
      item += pf_batch_items(J.B, J.loops, b->lpt, b->nt, &J.nbx);
      b->jobs.push_back(J);
      hash_jobs_clear(b->clear, h);
    }
    const FftLaunch comb = comb_fft(P, d_x[i]);
    HIPCK(fft_jobs_add(P->columns ? b->comb_slab : b->comb, comb));
    HIPCK(fft_jobs_add(b->bucket, bucket_fft(P)));
    const KeyMap km = fft_keys_map(comb);
    const SelMark mk = comb_mark(h);
    const bool marks = select_in_block(p.W_RLFC);
    HIPCK(select_jobs_add(b->sel_comb, b->fp32, P->comb_keys, p.W_RLFC, p.W_RLFC, p.B_thresh,
                          p.RLFC_loops, P->J2, 0, P->selW, nullptr, &km, P->comb_digits,
                          marks ? &mk : nullptr, P->hist_W));
    HIPCK(select_jobs_add(b->sel_bucket, b->fp32, P->bkeys, p.B, p.B, p.B_thresh, p.loops_loc,
                          P->J, 1, P->selB, P->jsel, nullptr, P->bucket_digits, nullptr,
                          P->hist_B));
    if (!marks) hash_jobs_bitmap(b->bitmap, h);
    NodeJob e = {};
    e.h = h;
    e.bins = P->bins_f;
    e.loops = p.loops;
    e.win = P->win;
    e.out = nodes[i] ? nodes[i] : P->nodes;
    e.copy = nodes[i] ? P->nodes : nullptr;
    e.sel = P->sel;
    e.count_copy = b->h_counts_dev + i;
    nodes_jobs_add(b->est, b->fp32, e);
  }
  b->total_items = item;
  slab_jobs_share(b->slab);
  *at_jobs = pack.put(b->jobs.data(), sizeof(PfJob) * b->jobs.size());
  for (auto& g : b->slab) g.t.pack(pack);
  for (auto& g : b->comb) g.t.pack(pack);
  for (auto& g : b->comb_slab) g.t.pack(pack);
  for (auto& g : b->bucket) g.t.pack(pack);
  for (auto& g : b->est) g.t.pack(pack);
  b->sel_comb.pack(pack);
  b->sel_bucket.pack(pack);
  b->clear.pack(pack);
  b->bitmap.pack(pack);
  return SFFT_OK;
}

// room for tables of `bytes` (no graph of the old ones, none in use)
static sfft_status reserve_tables(sfft_batch* b, size_t bytes) {
  if (b->d_tab) (void)hipFree(b->d_tab);
  if (b->h_tab) (void)hipHostFree(b->h_tab);
  b->d_tab = b->h_tab = nullptr;
  b->tab_bytes = 0;
  if (dev_alloc((void**)&b->d_tab, bytes) != hipSuccess ||
      hipHostMalloc((void**)&b->h_tab, bytes, hipHostMallocDefault) != hipSuccess)
    return SFFT_ERR_ALLOC;
  b->tab_bytes = bytes;
  return SFFT_OK;
}

static sfft_status build_tables(sfft_batch* b, const void* const* d_x, Node* const* nodes) {
  if (!b->tab_shape) drop_graph(b);
  b->tab_shape = false;
  b->tab_x.clear();
  JobPack pack;
  size_t at_jobs = 0;
  sfft_status v = pack_tables(b, d_x, nodes, pack, &at_jobs);
  if (v != SFFT_OK) return v;
  const size_t bytes = pack.bytes.size();
  if (b->tab_pending) HIPCK(hipEventSynchronize(b->tab_ev));
  b->tab_pending = 0;
  if (bytes > b->tab_bytes) {
    drop_graph(b);
    HIPCK(hipStreamSynchronize(b->st));   // an earlier batch may still read the old tables
    if ((v = reserve_tables(b, bytes)) != SFFT_OK) return v;
  }
  memcpy(b->h_tab, pack.bytes.data(), bytes);
  HIPCK(hipMemcpyAsync(b->d_tab, b->h_tab, bytes, hipMemcpyHostToDevice, b->st));
  HIPCK(hipEventRecord(b->tab_ev, b->st));
  b->tab_pending = 1;
  b->d_jobs = (const PfJob*)(b->d_tab + at_jobs);
  for (auto& g : b->slab) g.t.bind(b->d_tab);
  for (auto& g : b->comb) g.t.bind(b->d_tab);
  for (auto& g : b->comb_slab) g.t.bind(b->d_tab);
  for (auto& g : b->bucket) g.t.bind(b->d_tab);
  for (auto& g : b->est) g.t.bind(b->d_tab);
  b->sel_comb.bind(b->d_tab);
  b->sel_bucket.bind(b->d_tab);
  b->clear.bind(b->d_tab);
  b->bitmap.bind(b->d_tab);
  b->tab_x.assign(d_x, d_x + b->count);
  b->tab_nodes.assign(nodes, nodes + b->count);
  b->tab_shape = true;
  return SFFT_OK;
}

// one batch execution from the batch stream (the draws are up, the tables built).  The gathering
// signals' comb chain starts beside their permute+filter, the others' after the slab fold, which
// copies their comb samples (and clears for them).
static sfft_status enqueue(sfft_batch* b) {
  HIPCK(hash_clear_jobs(b->clear, b->st));
  HIPCK(slab_jobs_launch(b->slab, b->st));
  HIPCK(hipEventRecord(b->ev_fork, b->st));
  HIPCK(hipStreamWaitEvent(b->st2, b->ev_fork, 0));
  HIPCK(fft_jobs_launch(b->comb, b->st2));
  HIPCK(fft_jobs_launch(b->comb_slab, b->st2));
  HIPCK(select_jobs_launch(b->sel_comb, b->st2));
  HIPCK(hash_bitmap_jobs(b->bitmap, b->st2));
  HIPCK(hipEventRecord(b->ev_join, b->st2));
  HIPCK(perm_filter_batch_launch(b->fp32, b->d_jobs, (int)b->jobs.size(), b->total_items, b->lpt,
                                 b->nt, b->grid, b->st));
  HIPCK(fft_jobs_launch(b->bucket, b->st));
  HIPCK(select_jobs_launch(b->sel_bucket, b->st));
  HIPCK(hipStreamWaitEvent(b->st, b->ev_join, 0));
  HIPCK(nodes_jobs_launch(b->est, b->st));
  return SFFT_OK;
}

static sfft_status capture(sfft_batch* b) {
  HIPCK(hipStreamBeginCapture(b->st, hipStreamCaptureModeThreadLocal));
  const sfft_status v = enqueue(b);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(b->st, &g);
  if (v != SFFT_OK || e != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return v != SFFT_OK ? v : SFFT_ERR_HIP;
  }
  b->graph = g;
  if (hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0) != hipSuccess) {
    drop_graph(b);
    return SFFT_ERR_HIP;
  }
  return SFFT_OK;
}

// checks, the draws of every signal up in one copy, the tables for these pointers
static sfft_status prepare(sfft_batch* b, const void* const* d_x, const sfft_draws* draws,
                           Node* const* nodes) {
  for (int i = 0; i < b->count; ++i) {
    if (!d_x[i]) return SFFT_ERR_INVALID;
    if (!b->plans[i]->has_filter) return SFFT_ERR_NO_FILTER;
  }
  for (int i = 0; i < b->count; ++i) {
    const sfft_status v = draws_check(b->plans[i], &draws[i]);
    if (v != SFFT_OK) return v;
  }
  if (b->up_pending) HIPCK(hipEventSynchronize(b->up_ev));
  for (int i = 0; i < b->count; ++i) {
    const sfft_params& p = b->plans[i]->p;
    int* h = b->h_draws + b->draw_at[i];
    memcpy(h, draws[i].a, (size_t)p.loops * 4);
    memcpy(h + p.loops, draws[i].ai, (size_t)p.loops * 4);
    memcpy(h + 2 * p.loops, draws[i].offsets, (size_t)p.RLFC_loops * 4);
  }
  HIPCK(hipMemcpyAsync(b->d_draws, b->h_draws, sizeof(int) * b->draw_ints, hipMemcpyHostToDevice,
                       b->st));
  HIPCK(hipEventRecord(b->up_ev, b->st));
  b->up_pending = 1;
  if (b->tab_x.size() != (size_t)b->count ||
      !std::equal(b->tab_x.begin(), b->tab_x.end(), d_x) ||
      !std::equal(b->tab_nodes.begin(), b->tab_nodes.end(), nodes))
    return build_tables(b, d_x, nodes);
  return SFFT_OK;
}

static sfft_status execute(sfft_batch* b, const void* const* d_x, const sfft_draws* draws,
                           Node* const* nodes) {
  sfft_status v = prepare(b, d_x, draws, nodes);
  if (v != SFFT_OK) return v;
  if (!b->use_graph) return enqueue(b);
  if (!b->exec && (v = capture(b)) != SFFT_OK) return v;
  HIPCK(hipGraphLaunch(b->exec, b->st));
  return SFFT_OK;
}

extern "C" sfft_status sfft_batch_execute_async(sfft_batch* b, const void* const* d_x,
                                                const sfft_draws* draws) {
  if (!b || !d_x || !draws) return SFFT_ERR_INVALID;
  const std::vector<Node*> none(b->count, nullptr);
  return execute(b, d_x, draws, none.data());
}

extern "C" sfft_status sfft_batch_execute(sfft_batch* b, const void* const* d_x,
                                          const sfft_draws* draws, Node* const* h_nodes,
                                          int* h_counts) {
  if (!b || !d_x || !draws) return SFFT_ERR_INVALID;
  // pinned node memory: the estimation stores the nodes straight into it
  std::vector<Node*> view(b->count, nullptr);
  PinnedRange pinned;
  for (int i = 0; h_nodes && i < b->count; ++i)
    if (h_nodes[i])
      view[i] = (Node*)pinned.view(h_nodes[i], (size_t)b->plans[i]->cap * sizeof(Node));
  sfft_status v = execute(b, d_x, draws, view.data());
  if (v != SFFT_OK) return v;
  HIPCK(hipStreamSynchronize(b->st));   // (the estimation stored the counts too)
  sfft_status res = SFFT_OK;
  bool copies = false;
  for (int i = 0; i < b->count; ++i) {
    sfft_plan* P = b->plans[i];
    const int cnt = ((volatile int*)b->h_counts)[i];
    P->last_count = cnt;
    if (h_counts) h_counts[i] = cnt;
    if (cnt > P->cap) res = SFFT_ERR_HIT_OVERFLOW;
    const int ncopy = std::min(cnt, P->cap);
    if (h_nodes && h_nodes[i] && !view[i] && ncopy > 0) {
      HIPCK(hipMemcpyAsync(h_nodes[i], P->nodes, sizeof(Node) * (size_t)ncopy,
                           hipMemcpyDeviceToHost, b->st));
      copies = true;
    }
  }
  if (copies) HIPCK(hipStreamSynchronize(b->st));
  return res;
}

extern "C" sfft_status sfft_batch_set_graph(sfft_batch* b, int on) {
  if (!b) return SFFT_ERR_INVALID;
  if (!on) drop_graph(b);
  b->use_graph = on ? 1 : 0;
  return SFFT_OK;
}

extern "C" const int* sfft_batch_counts_device(const sfft_batch* b) {
  return b ? b->d_counts : nullptr;
}

// mean milliseconds of `reps` runs of fn on the batch stream (one warm-up run first)
template <typename F>
static sfft_status time_ms(sfft_batch* b, int reps, F fn, float* ms) {
  hipEvent_t e0, e1;
  HIPCK(hipEventCreate(&e0));
  HIPCK(hipEventCreate(&e1));
  sfft_status v = fn();
  if (v == SFFT_OK && hipEventRecord(e0, b->st) != hipSuccess) v = SFFT_ERR_HIP;
  for (int r = 0; v == SFFT_OK && r < reps; ++r) v = fn();
  if (v == SFFT_OK && (hipEventRecord(e1, b->st) != hipSuccess ||
                       hipEventSynchronize(e1) != hipSuccess ||
                       hipEventElapsedTime(ms, e0, e1) != hipSuccess))
    v = SFFT_ERR_HIP;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (v == SFFT_OK) *ms /= (float)reps;
  return v;
}

extern "C" sfft_status sfft_batch_tune(sfft_batch* b, const void* const* d_x,
                                       const sfft_draws* draws, int reps, int* choice4) {
  if (!b || !d_x || !draws || reps < 1) return SFFT_ERR_INVALID;
  const std::vector<Node*> none(b->count, nullptr);
  sfft_status v = prepare(b, d_x, draws, none.data());
  if (v != SFFT_OK) return v;
  // 1. permute+filter: loops per thread x block size x persistent grid
  const int lpts[] = {1, 2, 3, 4, 5, 6, 7, 8, 9}, nts[] = {128, 256},
            grids[] = {1024, 2048, 4096};
  float best = 1e30f;
  int bl = b->lpt, bn = b->nt, bg = b->grid;
  for (int lpt : lpts)
    for (int nt : nts) {
      b->lpt = lpt;
      b->nt = nt;
      if (b->jobs.empty()) continue;   // every signal takes the column front end
      drop_tables(b);
      if ((v = build_tables(b, d_x, none.data())) != SFFT_OK) return v;
      for (int grid : grids) {
        float ms = 0;
        v = time_ms(b, reps, [&]() -> sfft_status {
          // (only the gathering signals have a job)
          HIPCK(perm_filter_batch_launch(b->fp32, b->d_jobs, (int)b->jobs.size(),
                                         b->total_items, b->lpt, b->nt, grid, b->st));
          return SFFT_OK;
        }, &ms);
        if (v != SFFT_OK) return v;
        if (ms < best) {
          best = ms;
          bl = lpt;
          bn = nt;
          bg = grid;
        }
      }
    }
  b->lpt = bl;
  b->nt = bn;
  b->grid = bg;
  // 2. FFT columns per tile, bucket FFTs then comb FFTs, one choice for the whole batch
  const int qs[] = {1, 2, 4, 8, 16, 32};
  int best_q[2] = {0, 0};
  for (int which = 0; which < 2; ++which) {
    float bq = 1e30f;
    for (int q : qs) {
      for (auto P : b->plans) (which == 0 ? P->qmax_B : P->qmax_W) = q;
      drop_tables(b);
      if ((v = build_tables(b, d_x, none.data())) != SFFT_OK) return v;
      float ms = 0;
      v = time_ms(b, reps, [&]() -> sfft_status {
        HIPCK(fft_jobs_launch(which == 0 ? b->bucket : b->comb, b->st));
        if (which) HIPCK(fft_jobs_launch(b->comb_slab, b->st));
        return SFFT_OK;
      }, &ms);
      if (v != SFFT_OK) return v;
      if (ms < bq) {
        bq = ms;
        best_q[which] = q;
      }
    }
  }
  for (auto P : b->plans) {
    P->qmax_B = best_q[0];
    P->qmax_W = best_q[1];
  }
  drop_tables(b);   // built again for the chosen shapes
  if (choice4) {
    choice4[0] = b->lpt;
    choice4[1] = b->nt;
    choice4[2] = b->grid;
    choice4[3] = best_q[0] | (best_q[1] << 8);
  }
  return SFFT_OK;
}

// explicit shape (for tests that compare shapes): lpt in 1..9, nt 128/256, grid >= 1,
// FFT columns per tile (0 = default) for the bucket and comb FFTs
extern "C" sfft_status sfft_batch_set_shape(sfft_batch* b, int lpt, int nt, int grid,
                                            int qmax_bucket, int qmax_comb) {
  if (!b || lpt < 1 || lpt > 9 || (nt != 128 && nt != 256) || grid < 1 || qmax_bucket < 0 ||
      qmax_bucket > 32 || qmax_comb < 0 || qmax_comb > 32)
    return SFFT_ERR_INVALID;
  drop_tables(b);
  b->lpt = lpt;
  b->nt = nt;
  b->grid = grid;
  for (auto P : b->plans) {
    P->qmax_B = qmax_bucket;
    P->qmax_W = qmax_comb;
  }
  return SFFT_OK;
}
