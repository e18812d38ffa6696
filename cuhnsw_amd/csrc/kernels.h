// The launched kernels: batch search, and the three phases of a build batch.
//
// search_kernel        replaces GetEntryPointsKernel + SearchGraphKernel
//                      (cpp/include/cuda_search_kernels.cuh:11-165 in the reference):
//                      one launch does the descent through every upper level and the
//                      level-0 ef-search for a whole query batch.
// build_search_kernel, reverse_kernel
//                      replace BuildLevelGraphKernel + SearchHeuristic
//                      (cpp/include/cuda_build_kernels.cuh:68-338) and the per-level host
//                      orchestration (cpp/src/cuhnsw_build.cu:96-208).  The reference builds
//                      level by level, top down, every node of a level concurrently under
//                      per-node spin locks.  Here nodes are inserted in id order, each on all
//                      of its levels at once (hnswlib's order: early nodes leave long-range
//                      links on level 0, which is what keeps strongly clustered sets
//                      navigable), in batches of two lock-free phases separated by a kernel
//                      boundary:
//                        1. every node of the batch descends from the current entry point,
//                           searches each of its levels on the frozen graph, selects its
//                           neighbours there, writes its own rows (which nothing reaches yet)
//                           and leaves itself in the inbox of each neighbour y it chose,
//                        2. one wavefront per touched (y, level) merges inbox and row (append
//                           while there is room, else the selection heuristic).
//                      The result is deterministic for a given batch schedule.
#pragma once
#include "device_core.h"

namespace cuhnsw_amd {

// what the entries of the list of given-up queries hold that never come: the first pass is through
constexpr int kListEnds = -2;
// chiplets with an L2 each
constexpr int kShares = 8;

struct SlotPool {
  uint32_t* bitmaps;
  int bitmap_words;
  uint32_t* undo;
  int undo_cap;
  HeapEnt* cand_glob;
  int cand_glob_cap;
  HeapEnt* log;  // accepted entries of the running search
  int log_cap;
};

struct SearchArgs {
  const float* q;  // nq x D
  int nq, k, ef;
  int* nns;
  float* dists;
  int* found;
  int* stats;    // nq x 4 or null
  int* counter;  // work queue head
  int* status;   // set to 1 when a candidate queue ran out of room
  int* repeats;  // counts the queries that met equal keys in the sorted-set pass
  int* redo;     // their indices, for the literal pass; as input of the literal pass: the queries to answer (null = all)
  int* done;     // queries the sorted-set pass has finished with (answered or given up); done[1] is set to 1
                 // by the first wavefront of that pass to start
  int live;      // literal pass only: 1 = the sorted-set pass is running at the same time and a.redo is
                 // still being filled (entries start at -1); a.nq_total queries will pass through it
  int waiting;   // sorted-set pass only: how many literal wavefronts wait beside it (they are told when it is through)
  int* report;   // sorted-set pass only: host memory that gets the number of given-up queries and of spare trails taken
  int nq_total;
  int spin_limit;  // >= 0: polls of a live literal wavefront before it leaves with status 2 (tests force the
                   // fall-back with 0); < 0: no bound in polls, the two bounds in time below apply
  long long start_ticks;  // ticks of the device's wall clock a live literal wavefront waits for the first
                          // pass to START (done[1] != 0) before it takes the streams to be serialised
  long long stall_ticks;  // and for which it accepts no progress of the first pass once that has started
  const int* nq_dev;      // literal pass: when set, the number of list entries is read from here on the
                          // device (the count the first pass left) instead of taken from nq
  int slot_base;   // first slot of the pool this launch may use (two literal launches can be in flight)
  SlotPool pool;
  int cand_lds, hnswlib_dist;
  int team_bucket_bits;  // sorted-set pass by teams of wavefronts (struct Team)
  int team_turn;         // workgroups after which the next one comes to a CU that has one
  int rcap, lcap;  // ids and keys a row buffer holds: those of a link row; literal pass: those of the answer too
  int vc_bits;  // log2 entries of the LDS visited cache of the literal search, 0 = none
  FilterShape fc;  // the LDS visited filter of the sorted-set search (no sets: that search is off)
  int fast_path;  // 0 = literal queues only (exact evaluation counters)
  int reverse;    // expand the farthest waiting candidate (reverse_cand); sorted-set pass only
  const uint32_t* deleted;  // one bit per element (hnswlib's delete marks) or null; literal queues in LDS only (NS == 0)
  FilterShape lean;  // literal pass: result set = sorted set with ids, visited = an LDS filter of this shape
                     // (no bitmap, evaluation counters include repeats); no sets = exact bitmap
  // Sorted-set pass with its queries taken longest first (entry_kernel and the two order kernels below); all
  // null = queries in the caller's order, each descending from the top level itself.
  uint4* entry;     // per query: level-0 entry point, its key (bits), evaluations and sweeps of the descent
  int* order_hist;  // kOrderBuckets counters, then cursors
  int* order;       // nq query indices, in the order they are taken
  // Large batches besides: all but the longest queries by region (see below); null / 0 = largest entry key first throughout
  int* regions;      // the region each query falls into
  int region_level;  // the level at which the node its descent leaves says so
  int* shares;       // kShares + 1 work queue heads, 32 words apart: one over the longest queries, then one over each share of
                     // the others; behind them, how many the longest are
  // Trails of the sorted-set pass (device_core.h, struct Trail), all null / 0 = none are kept.  Buffer b holds
  // trail_cap records from trail + b * trail_cap on; wavefront w of the sorted-set pass starts on buffer w and,
  // each time it hands over a query whose trail the literal pass is to read, goes on with the next unused one
  // of the trail_spares buffers behind those (trail_next counts them; none left: it keeps no more trails).
  uint4* trail;
  int trail_cap, trail_first_spare, trail_spares;
  int* trail_next;
  int4* redo_trail;  // per entry of a.redo: (buffer or -1, records, expansions covered, evaluations up to there)
};

struct BuildArgs {
  int begin, count;        // batch = nodes begin .. begin+count-1
  const int* upper;        // the batch's nodes with upper levels (highest first, offsets from begin): handed out before
  int n_upper;             // the others (they take several searches, and a launch ends when its last node does); 0 = by id
  int cur_ep, cur_max;     // entry point and top level of the graph before this batch (cur_max < 0: empty)
  int efc, nn_num0, nn_numU, save_remains;
  int reverse;   // expand the farthest waiting candidate (reverse_cand)
  int own_cap0;  // how many links a new node may choose for itself on level 0 (<= max_m0)
  int* counter;
  int* status;
  SlotPool pool;
  int cand_lds, lcap;
  int vc_bits;
  FilterShape fc;
  int team_bucket_bits, team_turn;  // a team of wavefronts per node: as in SearchArgs
  HeapEnt* inbox0;  // N x cap_in
  int* inbox0_cnt;  // N
  HeapEnt* inboxU;  // upper rows x cap_in
  int* inboxU_cnt;  // upper rows
  int cap_in;
  unsigned long long* dirty;  // node | level << 32
  int* dirty_cnt;
  int* dropped;  // reverse links that found no room in an inbox (kept: the cap_in closest newcomers)
  // Per link row (N level-0 rows, then the upper rows): 1 = the row as it stands is an output of the selection
  // rule (written by a selection, not appended to since), so that a later re-selection may take the shortcut
  // for newcomers.  The reference keeps the same fact per node and level as went_through_heuristic
  // (cpp/include/cuda_build_kernels.cuh:277,322).  Null = no shortcut.
  unsigned char* selected0;
  unsigned char* selectedU;
  // optional work counters of a build (null = off), level 0 in [0..4], upper levels in [5..9]:
  //   +0 distance evaluations of the searches and descents (one vector row each)
  //   +1 link rows read (expanded candidates, descent sweeps, rows merged with their inbox)
  //   +2 pair tests of the selection heuristic (one vector row each)
  //   +3 picks the heuristic loaded to test candidates against them (one vector row each)
  //   +4 link rows written
  unsigned long long* counters;
};


__host__ __device__ inline size_t align16(size_t x) { return (x + 15) & ~(size_t)15; }

// elements per stored row: D rounded up so that every fp32 row starts on a 128-byte line (32 elements), or —
// `tight` — only to whole 16-byte chunks (4 elements), which shrinks the footprint and gives up the alignment
inline int padded_dims(int D, bool tight = false) { return tight ? (D + 3) / 4 * 4 : (D + 31) / 32 * 32; }
// float4 registers per lane that hold a query of Dp elements spread over 16 lanes (template parameter QR
// of the kernels); 0 = the query does not fit registers and is staged in LDS
inline int query_regs(int Dp) {
  const int chunks16 = ((Dp >> 2) + 15) / 16;
  return chunks16 <= 1 ? 1 : (chunks16 <= 2 ? 2 : (chunks16 <= 4 ? 4 : 0));
}

// LDS layout of one wavefront (shared by host sizing and device carving).  In the build's
// search kernel the visited filter of the sorted-set search (fcache) takes the place of the
// candidate queue and the literal search's visited cache.
struct LdsPlan {
  size_t qlds, top, cand, sorted_id, sorted_key, out_id, out_key, nbuf, dbuf, vcache, fcache, lfilter, total;
};
// fc: filter lying over the queue (build); lf: filter of its own beside the queue (the
// literal search on the sorted set)
__host__ __device__ inline LdsPlan plan_lds(int qr, int Dp, int ef, int cand_lds, int lcap, int n_sorted, int n_out,
                                            int vc_bits = 0, FilterShape fc = FilterShape(), FilterShape lf = FilterShape()) {
  LdsPlan p;
  size_t o = 0;
  p.qlds = o;
  if (qr == 0) o += (size_t)query_lds_chunks(Dp) * 16;
  p.top = o; o = align16(o + (size_t)(ef + 1) * 8);
  p.cand = o; o = align16(o + (size_t)cand_lds * 8);
  p.vcache = o; o = align16(o + (vc_bits > 0 ? ((size_t)2 << vc_bits) : 0));
  p.fcache = p.cand;
  const size_t fend = p.fcache + fc.bytes();
  if (fend > o) o = align16(fend);
  p.sorted_id = o; o = align16(o + (size_t)n_sorted * 4);
  p.sorted_key = o; o = align16(o + (size_t)n_sorted * 4);
  p.out_id = o; o = align16(o + (size_t)n_out * 4);
  p.out_key = o; o = align16(o + (size_t)n_out * 4);
  p.nbuf = o; o = align16(o + (size_t)nbuf_words(lcap) * 4);
  p.dbuf = o; o = align16(o + (size_t)lcap * 4);
  p.lfilter = o; o = align16(o + lf.bytes());
  p.total = o;
  return p;
}

__device__ __forceinline__ void bind_slot(Scratch& s, const SlotPool& pool, int slot) {
  s.bitmap = pool.bitmaps + (size_t)slot * pool.bitmap_words;
  s.bitmap_words = pool.bitmap_words;
  s.undo = pool.undo + (size_t)slot * pool.undo_cap;
  s.undo_cap = pool.undo_cap;
  s.cand_glob = pool.cand_glob + (size_t)slot * pool.cand_glob_cap;
  s.cand_glob_cap = pool.cand_glob_cap;
  s.log = pool.log + (size_t)slot * pool.log_cap;
  s.log_cap = pool.log_cap;
}

// LDS of the sorted-set search: query copy (long rows only), visited filter, row buffers.  The answer (ids, keys, and a copy of
// the ids where equal keys are put in order) lies over the filter, which is done with by then: a wavefront's LDS is handed out
// in steps of 1 280 bytes, and with topk 100 in buffers of its own the filter of 28 wavefronts on a CU is a tenth smaller.
struct FastLdsPlan {
  size_t qlds, fcache, nbuf, dbuf, total;
};
__host__ __device__ inline FastLdsPlan plan_fast_lds(int qr, int Dp, int rcap, FilterShape fc, int k) {
  FastLdsPlan p;
  size_t o = 0;
  p.qlds = o;
  if (qr == 0) o += (size_t)query_lds_chunks(Dp) * 16;
  p.fcache = o; o = align16(o + (fc.bytes() > 12u * (uint32_t)k ? (size_t)fc.bytes() : (size_t)12 * (size_t)k));
  p.nbuf = o; o = align16(o + (size_t)nbuf_words(rcap) * 4);
  p.dbuf = o; o = align16(o + (size_t)rcap * 4);
  p.total = o;
  return p;
}

// ---- longest queries first -------------------------------------------------------------------------------
// A batch of a few rounds of wavefronts ends when its last query does, and the work of a query has a long
// tail (1.18 M x 50, ef 300: median 300 expansions and 1 190 evaluations, one query in a hundred 440 and
// 2 350, the largest 690 and 4 370).  How far the level-0 entry point is from the query predicts most of it
// (correlation 0.67 with the work; the twenty heaviest of 10 000 queries are all within the fifth with the
// largest entry keys): the level-0 search has to walk that distance, accepting and evicting on its way.  So
// the greedy descent through the upper levels is done for the whole batch first (entry_kernel: what every
// query would do anyway), the queries are put in descending order of their entry key (a counting sort on the
// key's leading bits: order_prefix_kernel, order_scatter_kernel) and the first pass takes them in that order.
// The answers do not depend on the order in which queries are taken.
//
// Neighbours together: a batch of three rounds and more is bound by the rows its searches fetch (1 M x 96, 100 000
// queries, longest first: 60 GB in 9.6 ms, two L2 requests in a hundred hits), and queries next to each other search among
// the same rows (by region: 51 GB in 9.0 ms, 17 in a hundred).  So only the fifth with the largest entry keys goes first and
// longest first; the others go by region -- the node at which their descent leaves an upper level -- and every chiplet,
// which has an L2 of its own, takes them from an eighth of its own, then helps the others.  (Which batches: launch_search,
// with both sides.  A tenth first instead of a fifth: 1.18 M x 50, 40 000 queries 3.92 -> 4.11 ms, 10 M x 96, ef 256, 100 000 13.56 ->
// 13.80, 500 000 x 128, 30 000 5.46 -> 5.70; a third: 300 000 x 128, ef 200, 50 000 5.14 -> 5.29, 100 000 x 960, 8 000 4.62 ->
// 4.79, but 1.18 M x 80, 60 000 6.69 -> 6.51.  1.18 M x 50, 10 000 queries, 1.4 rounds, by region: 1.32 -> 1.48.)
constexpr int kLongestOf = 5;
constexpr int kOrderBits = 14;
constexpr int kOrderBuckets = 1 << kOrderBits;
// counters of the keys and of the regions, the work queue heads, and where the longest queries end (bucket, number)
constexpr int kOrderWords = 2 * kOrderBuckets + 32 * (kShares + 1) + 32;
// bucket 0 holds the largest keys (the float's bits made monotone, leading bits, reversed)
__device__ __forceinline__ int order_bucket(uint32_t key_bits) {
  const uint32_t u = key_bits ^ ((key_bits >> 31) ? 0xFFFFFFFFu : 0x80000000u);
  return (kOrderBuckets - 1) - (int)(u >> (32 - kOrderBits));
}
// neighbouring queries in neighbouring places: any order of the regions will do
__device__ __forceinline__ int region_bucket(uint32_t node) { return (int)((node * 2654435761u) >> (32 - kOrderBits)); }
template <int DT, int QR>
__global__ void __launch_bounds__(64) entry_kernel(DevIndex ix, SearchArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x;
  const FastLdsPlan lp = plan_fast_lds(QR, ix.Dp, a.rcap, FilterShape(), 0);
  Scratch s;
  s.vcache = nullptr;
  s.vc_bits = 0;
  s.qlds = reinterpret_cast<float4*>(smem + lp.qlds);
  s.nbuf = reinterpret_cast<uint32_t*>(smem + lp.nbuf);
  s.dbuf = reinterpret_cast<float*>(smem + lp.dbuf);
  for (int qi = blockIdx.x; qi < a.nq; qi += gridDim.x) {
    QVec<QR> qv;
    load_query<QR>(qv, s.qlds, a.q + (size_t)qi * ix.D, ix.D, ix.Dp, lane);
    SearchState st;
    st.n_dist_upper = 0; st.n_sweeps = 0;
    uint32_t cur = ix.enterpoint;
    float dcur = dist_single<DT, QR>(ix, qv, cur, s, lane);
    const int region_level = a.region_level < ix.maxlevel ? a.region_level : ix.maxlevel;
    descend<DT, QR>(ix, qv, ix.maxlevel, region_level > 0 ? region_level - 1 : 0, cur, dcur, s, st, lane);
    const uint32_t region = cur;
    if (region_level > 1) descend<DT, QR>(ix, qv, region_level - 1, 0, cur, dcur, s, st, lane);
    if (lane == 0) {
      const uint32_t bits = __float_as_uint(dcur);
      a.entry[qi] = make_uint4(cur, bits, (uint32_t)st.n_dist_upper, (uint32_t)st.n_sweeps);
      if (a.regions) a.regions[qi] = region_bucket(region);
      atomicAdd(a.order_hist + order_bucket(bits), 1);
    }
    wave_sync();
  }
}
// The same descents, FOUR queries per wavefront, one per group of 16 lanes (rows of up to 128 elements: the
// query in one or two float4 registers per lane).  A descent is a chain of dependent fetches with a dozen
// evaluations each; on its own in a kernel it is bound by their latency, and a group of 16 lanes is what one
// evaluation occupies anyway: the four groups walk their own queries' levels side by side, each evaluating
// the ids of its current link row one after the other (eight or sixteen rows in flight per lane), with the same
// arithmetic, the same strict first minimum and the same counters as `descend`.
template <int DT, int QR, bool HALF>
__device__ __forceinline__ float entry4_key(const void* rows, uint32_t rowlen, uint32_t used, const QVec<QR>& qv,
                                            const float* neg, uint32_t id, int sub) {
  constexpr int R = QR > 0 ? QR : 1;
  const uint64_t first = (uint64_t)id * rowlen;
  float ax = 0.f, ay = 0.f, az = 0.f, aw = 0.f;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const uint32_t c = sub + 16 * k;
    const uint64_t at = first + (c < used ? c : 0);  // (as in dist_pass: one unconditional load, padding replaced)
    const float4 v = HALF ? load_chunk_f16(rows, at) : load_chunk_f32(rows, at);
    if (DT == DIST_DOT || k < R / 2) acc4<DT>(qv.q[k], v, ax, ay, az, aw);
    else acc4_l2_if(qv.q[k], v, neg[k], ax, ay, az, aw);
  }
  return finish16<DT, false>(ax, ay, az, aw);
}
template <int DT, int QR, bool HALF>
__device__ __forceinline__ void entry4_body(const DevIndex& ix, const SearchArgs& a) {
  const int lane = threadIdx.x, g = lane >> 4, sub = lane & 15;
  const uint32_t rowlen = (uint32_t)ix.Dp >> 2, used = (uint32_t)(ix.D + 3) >> 2;
  const void* rows = ix.vectors;
  float neg[QR > 0 ? QR : 1];  // (as in dist_pass)
#pragma unroll
  for (int k = 0; k < (QR > 0 ? QR : 1); ++k) neg[k] = minus_one_if((uint32_t)(sub + 16 * k) < used);
  for (int q0 = blockIdx.x * 4; q0 < a.nq; q0 += gridDim.x * 4) {
    const int qi = q0 + g;
    const bool have = qi < a.nq;
    QVec<QR> qv;
    load_query<QR>(qv, nullptr, a.q + (size_t)(have ? qi : 0) * ix.D, ix.D, ix.Dp, lane);
    uint32_t cur = ix.enterpoint;
    float dcur = entry4_key<DT, QR, HALF>(rows, rowlen, used, qv, neg, cur, sub);
    int level = ix.maxlevel;
    bool active = have && level > 0;
    int sweeps = 0, evals = 0;
    uint32_t region = cur;
    long long first = ix.upper_off[cur];
    while (__ballot(active) != 0ull) {
      const uint32_t* row = ix.linksU + (size_t)((active ? first : 0) + (active ? level : 1) - 1) * ix.SU;
      float best = INFINITY;
      uint32_t best_id = cur;
      int n = 0;
      for (int base = 0; base < ix.SU; base += 16) {
        const uint32_t got = row[base + sub < ix.SU ? base + sub : 0];
        const uint32_t id = (active && base + sub < ix.SU) ? got : kEmpty;
        const unsigned long long valid = __ballot(id != kEmpty);
        n += __popc((uint32_t)(valid >> (16 * g)) & 0xFFFFu);
        constexpr int B = QR == 1 ? 16 : 8;  // rows in flight per lane: 16 float4 registers' worth
#pragma unroll
        for (int p0 = 0; p0 < 16; p0 += B) {
          if (((valid >> p0) & (0x0001000100010001ull * ((1u << B) - 1u))) == 0ull) continue;  // no id in these slots
          uint32_t ids[B];
          float keys[B];
#pragma unroll
          for (int j = 0; j < B; ++j) ids[j] = (uint32_t)__shfl((int)id, 16 * g + p0 + j, 64);
#pragma unroll
          for (int j = 0; j < B; ++j)
            keys[j] = entry4_key<DT, QR, HALF>(rows, rowlen, used, qv, neg, ids[j] != kEmpty ? ids[j] : cur, sub);
#pragma unroll
          for (int j = 0; j < B; ++j)
            if (ids[j] != kEmpty && keys[j] < best) {  // strictly closer: the first occurrence of the minimum wins
              best = keys[j];
              best_id = ids[j];
            }
        }
      }
      if (active) {
        sweeps += 1;
        evals += n;
        if (n > 0 && best < dcur) {
          dcur = best;
          cur = best_id;  // and sweep again on this level
          first = ix.upper_off[best_id];
        } else {
          if (level == a.region_level) region = cur;
          level -= 1;
          active = level > 0;
        }
      }
    }
    if (have && sub == 0) {
      const uint32_t bits = __float_as_uint(dcur);
      a.entry[qi] = make_uint4(cur, bits, (uint32_t)evals, (uint32_t)sweeps);
      if (a.regions) a.regions[qi] = region_bucket(region);
      atomicAdd(a.order_hist + order_bucket(bits), 1);
    }
  }
}
// (Where the neighbours' rows are, asked for beside their vectors as in descend, is not worth it here, for a wavefront per SIMD less:
// 10 000 / 16 000 queries with it and without, us: 1.18 M x 50 67, 90 and 65, 90; 600 000 x 96 77, 106 and 78, 104; 300 000 x 128 L2 76,
// 107 and 71, 101.)
template <int DT, int QR>
__global__ void __launch_bounds__(64) entry4_kernel(DevIndex ix, SearchArgs a) {
  if (uni(ix.half) != 0) entry4_body<DT, QR, true>(ix, a);
  else entry4_body<DT, QR, false>(ix, a);
}
// counters -> first position of every bucket (exclusive prefix sum over `from` and what lies before; one workgroup of 1024).
// cut: the longest queries end with the first bucket at which there are `most` of them or more; set to that bucket and to
// their number.
__device__ __forceinline__ void order_prefix(int* hist, int from, int most, int* cut) {
  __shared__ int part[1024];
  constexpr int per = kOrderBuckets / 1024;
  const int t = threadIdx.x;
  int local[per];
  int sum = 0;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    local[i] = hist[t * per + i];
    sum += local[i];
  }
  part[t] = sum;
  __syncthreads();
  for (int step = 1; step < 1024; step <<= 1) {
    const int add = t >= step ? part[t - step] : 0;
    __syncthreads();
    part[t] += add;
    __syncthreads();
  }
  const int first = part[t] - sum + from;
  int run = first;
#pragma unroll
  for (int i = 0; i < per; ++i) {
    hist[t * per + i] = run;
    run += local[i];
  }
  // (one thread's business, and apart from the loop above, whose stores it would take apart: 6 us in it, 11 there)
  if (cut && first < most && run >= most) {
    run = first;
#pragma unroll
    for (int i = 0; i < per; ++i) {
      if (run < most && run + local[i] >= most) {
        cut[0] = t * per + i;
        cut[1] = run + local[i];
      }
      run += local[i];
    }
  }
}
static __global__ void __launch_bounds__(1024) order_prefix_kernel(int* hist, int most, int* cut) { order_prefix(hist, 0, most, cut); }
static __global__ void __launch_bounds__(1024) region_prefix_kernel(int* hist, const int* cut) { order_prefix(hist, cut[1], 0, nullptr); }
// how many queries that are not among the longest each region has
static __global__ void __launch_bounds__(1024) region_count_kernel(const uint4* entry, const int* regions, int nq, const int* cut, int* hist) {
  const int qi = blockIdx.x * 1024 + threadIdx.x;
  if (qi < nq && order_bucket(entry[qi].y) > cut[0]) atomicAdd(hist + regions[qi], 1);
}
// Queries to their places: by entry key, or (regions) only the longest of them and the others by region.
static __global__ void __launch_bounds__(1024) order_scatter_kernel(const uint4* entry, const int* regions, const int* cut, int nq, int* cursor,
                                                                    int* region_cursor, int* order) {
  // The keys of a batch fall into a few dozen buckets: a workgroup ranks its 1024 queries in LDS and takes one
  // range per bucket it met from the global cursors (the order inside a bucket is free).
  __shared__ int cnt[kOrderBuckets];
  const int t = threadIdx.x;
  const int qi = blockIdx.x * 1024 + t;
  const int last = regions ? cut[0] : kOrderBuckets;
  for (int part = 0; part < (regions ? 2 : 1); ++part) {
    int* from = part == 0 ? cursor : region_cursor;
    for (int i = t; i < kOrderBuckets; i += 1024) cnt[i] = 0;
    __syncthreads();
    int bucket = 0, rank = 0;
    bool mine = false;
    if (qi < nq) {
      bucket = order_bucket(entry[qi].y);
      mine = (bucket <= last) == (part == 0);
      if (part == 1) bucket = regions[qi];
      if (mine) rank = atomicAdd(&cnt[bucket], 1);
    }
    __syncthreads();
    for (int i = t; i < kOrderBuckets; i += 1024) {
      const int c = cnt[i];
      if (c > 0) cnt[i] = atomicAdd(from + i, c);
    }
    __syncthreads();
    if (mine) order[cnt[bucket] + rank] = qi;
    __syncthreads();
  }
}

// The LDS that the wavefronts of a workgroup share to search together (device_core.h, team_help), set up by all of them; returns this
// one's part: 0 searches, the others help.
template <int NS>
__device__ __forceinline__ int gather_team(Scratch& s, unsigned char* lds, int stride, int level, int bucket_bits, int turn) {
  s.team.base = reinterpret_cast<uint32_t*>(lds);
  s.team.bucket_bits = bucket_bits;
  s.team.stride = stride;
  s.team.lists = Team::lists_at(NS);
  for (int i = (int)threadIdx.x; i < Team::kRoom; i += (int)blockDim.x)
    s.team.base[i] = i < (4 << bucket_bits) ? kNobody : (i == Team::kOver ? 0u : (i == Team::kOver + 1 ? (uint32_t)level << 16 : kEmpty));
  filter_reset(s, (int)threadIdx.x, (int)blockDim.x);
  __syncthreads();
  // (the workgroups that share a CU have their first wavefronts on the same SIMD: another one of each searches)
  const int waves = (int)blockDim.x >> 6;
  return (uni((int)threadIdx.x >> 6) + waves - ((int)blockIdx.x / turn) % waves) % waves;
}

// A kernel's arguments read afresh from where the launch put them.  The compiler loads every argument once, when the
// kernel starts, and keeps it: fifty scalar registers for what is needed once per query, and what does not fit is parked
// in lanes of vector registers.  Through a pointer it cannot see through the fields are loaded where they are used.
// (Kernels here take a DevIndex, then their own arguments.)
template <typename T>
__device__ __forceinline__ const T& fresh_kernel_args(size_t offset) {
  typedef const __attribute__((address_space(4))) char* kernarg_t;
  kernarg_t p = (kernarg_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const T*)(const __attribute__((address_space(4))) T*)(p + offset);
}
__device__ __forceinline__ const DevIndex& fresh_index() { return fresh_kernel_args<DevIndex>(0); }
template <typename Args>
__device__ __forceinline__ const Args& fresh_args() {
  static_assert(alignof(Args) == 8 && alignof(DevIndex) == 8, "second argument right after the first");
  return fresh_kernel_args<Args>((sizeof(DevIndex) + 7) / 8 * 8);
}

// First pass of a search batch: every query on the sorted set in registers (ef <= 64*NS).
// A query in which two equal keys meet is not answered here: its index is appended to
// a.redo (a.repeats counts them) and the literal search_kernel answers it afterwards.
// (with at most six keys per lane and the query in at most two float4 registers the kernel is
// held to 72 registers, seven wavefronts per SIMD, at the price of up to nine spilled registers, none of them
// touched inside a hop loop; eight wavefronts are no faster.  Six keys per lane spill up to 19, and where their reloads are
// in the loop six wavefronts are the better ones, fast_waves_of_six: 400 000 x 50, ef 330, 40 000 queries 4.05 -> 3.92 ms,
// 10 000 with trails 1.66 -> 1.63, 300 000 x 60 L2 1.59 -> 1.44, x 100 1.92 -> 1.86; seven stay where they are not, 300 000 x
// 60 L2, 40 000 3.33 against 3.50, 200 000 x 128 L2 7.51 against 8.05, or are few, 400 000 x 96 4.64 against 4.69 and, with
// trails, 1.67 against 1.72.
// With seven and eight keys per lane it fits 96 registers, five wavefronts per SIMD: with six of them ef 430 is 2 % slower
// to 5 % faster and ef 512 a fifth slower; the other shapes would spill heavily.  129 to 256 elements in L2 with five keys
// per lane would take one register too many for five wavefronts: 100 000 x 180 in fp16, ef 300, 40 000 queries 5.43 -> 4.87
// ms, in fp32 5.33 -> 4.94, 150 000 x 250 6.26 -> 6.34.  Not with two keys, six wavefronts or seven: 4.73 and 4.77 at ef 128.)
// TRAILS: the pass leaves trails for the literal pass (a.trail set; 2 to 3 % more instructions: the host launches
// this instance for batches of a round or two of wavefronts, where a query handed over late is a good part of the
// batch's time, and the instance without the trail code otherwise).
// FEW: for batches that leave the machine idle, at most a wavefront per SIMD: twice the rows in flight and more
// candidates at a time, with the registers that takes (100 000 x 50, ef 300, one query: 0.290 -> 0.278 ms; 100 000 x 960,
// ef 300, 1 000 queries: 1.35 -> 1.29).
// TEAM: FEW, and the other wavefronts of the workgroup help the one that searches (device_core.h, team_help; which batches:
// launch_teams).  Held to 128 registers, four of its wavefronts on a SIMD, on rows of up to 256 elements.
constexpr int kMostTeam = 8;  // wavefronts per query
constexpr int fast_waves_of_six(int dt, int qr, bool trails) { return (dt == DIST_DOT ? qr == 1 : trails) ? 6 : 7; }
template <int DT, int QR, int NS, bool TRAILS, bool FEW = false, bool TEAM = false>
__global__ void __launch_bounds__(TEAM ? 64 * kMostTeam : 64, TEAM ? (QR != 0 && NS <= 8 ? 4 : 2) : FEW ? 1 : (QR >= 1 && QR <= 2) ? (NS <= 5 ? 7 : NS == 6 ? fast_waves_of_six(DT, QR, TRAILS) : (NS <= 8 ? 5 : 1)) : (QR == 4 && NS == 5 && DT == DIST_L2) ? 5 : 1) search_fast_kernel(DevIndex ix0, SearchArgs a0) {
  extern __shared__ __align__(16) unsigned char smem[];
  const FastLdsPlan lp = plan_fast_lds(QR, ix0.Dp, a0.rcap, a0.fc, a0.k);
  Scratch s;
  s.vcache = reinterpret_cast<uint16_t*>(smem + lp.fcache);
  s.filter = a0.fc;
  s.qlds = reinterpret_cast<float4*>(smem + lp.qlds);
  s.nbuf = reinterpret_cast<uint32_t*>(smem + lp.nbuf);
  s.dbuf = reinterpret_cast<float*>(smem + lp.dbuf);
  if (TEAM) {
    // a workgroup per query: one wavefront searches (gather_team says which), the others help
    const int wave = gather_team<NS>(s, smem + lp.total, ix0.S0, 0, a0.team_bucket_bits, a0.team_turn);
    if (wave > 0) {
      const int lane = (int)threadIdx.x & 63;
      QVec<QR> qv;
      load_query<QR>(qv, s.qlds, a0.q + (size_t)blockIdx.x * ix0.D, ix0.D, ix0.Dp, lane);
      team_help<DT, QR>(ix0, qv, s, wave - 1, lane);
      return;
    }
    __builtin_amdgcn_s_setprio(3);
  }
  // tells a literal pass waiting beside this one that the two kernels do run at the same time
  if (blockIdx.x == 0 && threadIdx.x == 0) __hip_atomic_store(a0.done + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  int trail_buf = (TRAILS && a0.trail) ? (int)blockIdx.x : -1;  // the buffer this wavefront's trails go to
  int share_at = 0;  // the queue this wavefront is at (a.shares)

  for (;;) {
    int lane = fresh((int)threadIdx.x & 63);
    const SearchArgs& in = fresh_args<SearchArgs>();
    const DevIndex& from = fresh_index();
    int qi = 0;
    if (!FEW && !TRAILS && in.shares) {
      // the longest queries, then this chiplet's share of the others, then what is left of the other chiplets'
      const int longest = in.shares[32 * (kShares + 1) + 1];
      qi = in.nq;
      while (share_at <= kShares) {
        const int share = (int)(__builtin_amdgcn_s_getreg(20 | (31 << 11)) + share_at) & (kShares - 1);  // (XCC_ID, all 32 bits)
        const long long others = in.nq - longest;
        const int begin = share_at == 0 ? 0 : longest + (int)(others * share / kShares);
        const int end = share_at == 0 ? longest : longest + (int)(others * (share + 1) / kShares);
        int at = 0;
        if (lane == 0) at = begin + atomicAdd(in.shares + 32 * (share_at == 0 ? 0 : share + 1), 1);
        at = uni(at);
        if (at < end) {
          qi = in.order[at];
          break;
        }
        share_at += 1;
      }
    } else if (TEAM) {
      qi = share_at++ == 0 ? (int)blockIdx.x : in.nq;
    } else if (lane == 0) {
      qi = atomicAdd(in.counter, 1);
      if (qi < in.nq && in.order) qi = in.order[qi];
    }
    qi = __builtin_amdgcn_readfirstlane(qi);
    if (qi >= in.nq) break;
    Trail tr;
    if (TRAILS && trail_buf >= 0) {
      tr.rec = in.trail + (size_t)trail_buf * in.trail_cap;
      tr.cap = in.trail_cap;
      tr.on = true;
    }
    QVec<QR> qv;
    load_query<QR>(qv, s.qlds, in.q + (size_t)qi * from.D, from.D, from.Dp, lane);
    SearchState st;
    st.top_size = 0; st.cand_size = 0; st.n_acc = 0; st.lower = 0.f; st.maxkey = -INFINITY; st.undo_cnt = 0;
    st.n_dist = 0; st.n_hops = 0; st.n_dist_upper = 0; st.n_sweeps = 0; st.fail = 0; st.ahead = 1;

    uint32_t cur = from.enterpoint;
    if (in.entry) {  // the descent through the upper levels has been done for the whole batch
      const uint4 en = in.entry[qi];
      cur = (uint32_t)__builtin_amdgcn_readfirstlane((int)en.x);
      st.n_dist_upper = __builtin_amdgcn_readfirstlane((int)en.z);
      st.n_sweeps = __builtin_amdgcn_readfirstlane((int)en.w);
    } else {
      float dcur = dist_single<DT, QR>(from, qv, cur, s, lane);
      descend<DT, QR>(from, qv, from.maxlevel, 0, cur, dcur, s, st, lane);
    }

    lane = fresh(lane);
    if (TEAM) {
      // (the first candidate: its list can be made while this wavefront gets ready)
      HeapEnt e;
      e.key = INFINITY;
      e.id = cur;
      if (lane == 0) s.team.line()[8] = e;
      __builtin_amdgcn_wave_barrier();
    }
    Frontier<NS> fr;
    frontier_init<NS>(fr, a0.ef, lane);
    if (!TEAM) filter_reset(s, lane);
    visit_lossy_single(s, cur, lane);
    if (lane == 0) s.nbuf[0] = cur;
    wave_sync();
    // (the flag is made wavefront-uniform explicitly and both outcomes are plain branches)
    const int how =
        __builtin_amdgcn_readfirstlane(search_level_fast<DT, QR, NS, false, TRAILS, FEW, TEAM>(ix0, qv, 0, a0.ef, s, st, fr, 1, lane, a0.reverse != 0, a0.k >= a0.ef, TRAILS ? &tr : nullptr));
    if (TEAM) {
      if (lane == 0) lds_tell(s.team.over(), 1u);
      __builtin_amdgcn_wave_barrier();
    }
    lane = fresh(lane);
    const SearchArgs& a = fresh_args<SearchArgs>();
    const DevIndex& ix = fresh_index();
    const int T0 = st.top_size < a.k ? st.top_size : a.k;
    // Equal keys across the cut at k: which of them stays is up to the result heap, which the
    // literal search reproduces.  Equal keys among the k best: the answer lists them by label.
    const bool cut_tie = how == 2 && !a.reverse && frontier_tie_within<NS>(fr, a.ef, T0, st.top_size, lane, T0 - 1);
    const int inner_tie = __builtin_amdgcn_readfirstlane(
        (how == 2 && !a.reverse && frontier_tie_within<NS>(fr, a.ef, T0 - 1, st.top_size, lane)) ? 1 : 0);
    const bool gave_up = how == 1 || cut_tie;
    if (gave_up) {
      // (the trail's records are written by many lanes: all of them out before lane 0 publishes the entry)
      const bool with_trail = TRAILS && a.redo_trail && trail_buf >= 0 && tr.n > 0 && tr.hops > 0;
      // a search that went all the way (only the cut at k is open) and whose trail covers every hop: the literal
      // pass needs no search at all, only the result heap replayed from the trail (hops stored negative)
      const bool whole = how != 1 && tr.hops == st.n_hops;
      if (with_trail) __threadfence();
      int spare = 0;
      if (lane == 0) {
        const int slot = atomicAdd(a.repeats, 1);
        if (a.redo_trail) a.redo_trail[slot] = make_int4(with_trail ? trail_buf : -1, tr.n, whole ? -tr.hops : tr.hops, tr.n_dist);
        __hip_atomic_store(&a.redo[slot], qi, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        if (with_trail) spare = atomicAdd(a.trail_next, 1);
      }
      // (the lanes meet again HERE: threaded through to the loop's end, lane 0's way out of the branch above
      // would make everything the next lines set look lane-dependent to the compiler)
      __builtin_amdgcn_wave_barrier();
      if (with_trail) {
        // that buffer belongs to the literal pass now
        spare = __builtin_amdgcn_readfirstlane(spare);
        trail_buf = spare < a.trail_spares ? a.trail_first_spare + spare : -1;
      }
    } else {
      const int T = __builtin_amdgcn_readfirstlane(st.top_size < a.k ? st.top_size : a.k);
      uint32_t* const ids = reinterpret_cast<uint32_t*>(s.vcache);
      float* const keys = reinterpret_cast<float*>(ids + a.k);
      wave_sync();
      frontier_dump<NS>(fr, a.ef, T, ids, keys, lane);
      wave_sync();
      if (inner_tie) order_equal_keys(ix, ids, keys, T, ids + 2 * a.k, lane);
      if (!a.hnswlib_dist && T > 0) {
        dist_list<DT, QR, true>(ix, qv, s.qlds, ids, T, keys, lane);
        wave_sync();
      }
      for (int r = lane; r < a.k; r += 64) {
        int out_id = -1;
        float out_d = INFINITY;
        if (r < T) {
          const uint32_t id = ids[r];
          out_id = ix.labels ? (int)ix.labels[id] : (int)id;
          out_d = a.hnswlib_dist ? answer_key(keys[r]) : keys[r];
        }
        a.nns[(size_t)qi * a.k + r] = out_id;
        a.dists[(size_t)qi * a.k + r] = out_d;
      }
      if (lane == 0) {
        a.found[qi] = T;
        if (a.stats) {
          a.stats[(size_t)qi * 4 + 0] = st.n_dist;
          a.stats[(size_t)qi * 4 + 1] = st.n_hops;
          a.stats[(size_t)qi * 4 + 2] = st.n_dist_upper;
          a.stats[(size_t)qi * 4 + 3] = st.n_sweeps;
        }
      }
    }
    // The count the literal pass watches.  Only a query that was handed over has published something that pass
    // reads (its list entry, its trail): there the count is raised with release order, after them; an answered
    // query's results are the host's to read, after the kernel.
    if (lane == 0) {
      const int before = gave_up ? __hip_atomic_fetch_add(a.done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT)
                                 : __hip_atomic_fetch_add(a.done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (before == a.nq - 1) {
        // the batch's last query: the list is complete.  The wavefronts that wait for further entries are told through
        // the entries they poll (at most a.waiting of them), the host through its own memory.
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        const int n_list = __hip_atomic_load(a.repeats, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a.report) {
          a.report[0] = n_list;
          a.report[1] = a.trail_next ? __hip_atomic_load(a.trail_next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
        }
        for (int i = n_list; i < a.nq && i < n_list + a.waiting; ++i)
          __hip_atomic_store(&a.redo[i], kListEnds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    wave_sync();
  }
}

// The accepted entries of a search through hnswlib's result heap.  (64 of the log's records per fetch, handed out lane by lane, and
// the next 64 fetched meanwhile: one by one each is a trip to memory, a third of what an entry takes.)
__device__ __forceinline__ void replay_log(const Scratch& s, LdsHeap& top, int& size, int n, int ef, int lane) {
  HeapEnt next = s.log[lane < n ? lane : 0];
  for (int base = 0; base < n; base += 64) {
    const HeapEnt mine = next;
    const int cnt = n - base < 64 ? n - base : 64;
    next = s.log[base + 64 + lane < n ? base + 64 + lane : 0];
    for (int j = 0; j < cnt; ++j) {
      HeapEnt e;
      e.key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.key), j));
      e.id = (uint32_t)__builtin_amdgcn_readlane((int)mine.id, j);
      coop_push<false>(top, size, e, lane);
      if (size > ef) coop_pop<false>(top, size, s.tree, lane);
    }
  }
}
// Search with literal hnswlib priority queues: the only pass for ef beyond the sorted set's
// capacity, the second pass (over a.redo) otherwise.
// NS > 0: result keys in registers (ef <= 64*NS); NS == 0: literal result heap in LDS.
// (held to 96 registers, five wavefronts per SIMD, where the query fits two float4 registers: a
// batch answered by the literal queues alone runs 7-10 % faster for a dozen spilled registers)
template <int DT, int QR, int NS>
__global__ void __launch_bounds__(64, (QR >= 1 && QR <= 2 && NS > 0 && NS <= 5) ? 5 : 1) search_kernel(DevIndex ix, SearchArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x;
  const bool lean = NS > 0 && a.lean.sets() > 0;
  const LdsPlan lp = plan_lds(QR, ix.Dp, NS > 0 ? -1 : a.ef, a.cand_lds, a.lcap, 0, 0, lean ? 0 : a.vc_bits, FilterShape(), a.lean);
  Scratch s;
  if (lean) {
    s.vcache = reinterpret_cast<uint16_t*>(smem + lp.lfilter);
    s.filter = a.lean;
  } else {
    s.vcache = a.vc_bits > 0 ? reinterpret_cast<uint16_t*>(smem + lp.vcache) : nullptr;
    s.vc_bits = a.vc_bits;
  }
  s.qlds = reinterpret_cast<float4*>(smem + lp.qlds);
  s.top = reinterpret_cast<HeapEnt*>(smem + lp.top);
  s.cand = reinterpret_cast<HeapEnt*>(smem + lp.cand);
  s.cand_lds = a.cand_lds;
  s.nbuf = reinterpret_cast<uint32_t*>(smem + lp.nbuf);
  s.dbuf = reinterpret_cast<float*>(smem + lp.dbuf);
  s.tree = make_stage_tree(lane);
  bind_slot(s, a.pool, a.slot_base + blockIdx.x);
  // after the search the candidate queue is dead: its LDS share (>= ef + 1 entries) then
  // holds the collected results, or the literal heap when a tie has to be replayed
  if (NS > 0) s.top = s.cand;

  for (;;) {
    int qi = 0;
    int entry = 0;  // which entry of the list this is
    if (lane == 0) {
      qi = atomicAdd(a.counter, 1);
      if (a.live) {
        entry = qi;
        // entry qi of the list appears once the sorted-set pass has given up that many
        // queries; it never will if that pass has finished them all and the entry is still
        // empty.  The wait is bounded in wall-clock time: if the first pass has not even started
        // after start_ticks (the two streams are being serialised, as under a counter-collecting
        // profiler), or has made no progress for stall_ticks, the wavefront leaves with status 2
        // and the host answers the rest after the first pass.
        int got = kListEnds;
        if (qi < a.nq_total) {
          const long long t_begin = wall_clock64();
          long long t_progress = t_begin;
          int seen_done = -1;
          // (relaxed agent-scope loads: they read the L2 and, unlike acquire loads, do not
          // invalidate this CU's vector cache on every poll; the list entry is the only thing
          // read from the other pass, and it is read after the count that vouches for it)
          // every waiter polls its own list entry, which is where it also learns that the first pass
          // is through (kListEnds); the shared count is looked at only now and then, for the bounds
          // in time, so that the waiting does not crowd the memory channel of the counters the other
          // pass is working with
          for (int spins = 0;; ++spins) {
            got = __hip_atomic_load(&a.redo[qi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (got != -1) break;
            if (a.spin_limit >= 0 && spins >= a.spin_limit) {
              atomicOr(a.status, 2);
              break;
            }
            if ((spins & 15) == 15) {
              const int done_now = __hip_atomic_load(a.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              if (done_now >= a.nq_total) {
                got = __hip_atomic_load(&a.redo[qi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
              }
              const long long now = wall_clock64();
              if (done_now != seen_done) {
                seen_done = done_now;
                t_progress = now;
              }
              const bool started = __hip_atomic_load(a.done + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
              if (started ? (now - t_progress > a.stall_ticks) : (now - t_begin > a.start_ticks)) {
                atomicOr(a.status, 2);
                break;
              }
            }
            if (spins < 16) __builtin_amdgcn_s_sleep(32);  // 0.9 us
            else __builtin_amdgcn_s_sleep(127);            // 3.5 us
          }
        }
        qi = got;
      } else if (qi >= (a.nq_dev ? *a.nq_dev : a.nq)) {
        qi = -1;
      } else if (a.redo) {
        entry = qi;
        qi = a.redo[qi];  // second pass: only the queries the sorted-set pass gave up
      }
    }
    qi = __builtin_amdgcn_readfirstlane(qi);
    if (qi < 0) break;
    // the trail the sorted-set pass left for this query, if any (its records were written by another
    // wavefront before the list entry was: read them from memory, not from this CU's cache)
    int4 tmeta = make_int4(-1, 0, 0, 0);
    if (lean && a.redo_trail) {
      entry = __builtin_amdgcn_readfirstlane(entry);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      const int4 m = a.redo_trail[entry];
      tmeta = make_int4(__builtin_amdgcn_readfirstlane(m.x), __builtin_amdgcn_readfirstlane(m.y),
                        __builtin_amdgcn_readfirstlane(m.z), __builtin_amdgcn_readfirstlane(m.w));
    }
    // beside the first pass a literal wavefront is one among a few dozen on its CU and its query
    // is on the batch's critical path: it goes first whenever it has an instruction ready
    if (a.live) __builtin_amdgcn_s_setprio(3);
    QVec<QR> qv;
    load_query<QR>(qv, s.qlds, a.q + (size_t)qi * ix.D, ix.D, ix.Dp, lane);
    SearchState st;
    st.top_size = 0; st.cand_size = 0; st.n_acc = 0; st.lower = 0.f; st.maxkey = -INFINITY; st.undo_cnt = 0;
    st.n_dist = 0; st.n_hops = 0; st.n_dist_upper = 0; st.n_sweeps = 0; st.fail = 0; st.ahead = 1;
    TopKeys<NS> tk;
    topkeys_init<NS>(tk, a.ef, lane);

    uint32_t cur = ix.enterpoint;
    float dcur;
    if (a.entry) {  // the descent through the upper levels has been done for the whole batch
      const uint4 en = a.entry[qi];
      cur = (uint32_t)__builtin_amdgcn_readfirstlane((int)en.x);
      dcur = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane((int)en.y));
      st.n_dist_upper = __builtin_amdgcn_readfirstlane((int)en.z);
      st.n_sweeps = __builtin_amdgcn_readfirstlane((int)en.w);
    } else {
      dcur = dist_single<DT, QR>(ix, qv, cur, s, lane);
      descend<DT, QR>(ix, qv, ix.maxlevel, 0, cur, dcur, s, st, lane);
    }

    int T;
    bool literal = NS == 0;
    bool have_result = false;  // s.nbuf / s.dbuf already hold the T answers in order
    if (lean) {
      Frontier<NS> fr;
      frontier_init<NS>(fr, a.ef, lane);
      filter_reset(s, lane);
      visit_lossy_single(s, cur, lane);
      if (lane == 0) s.nbuf[0] = cur;
      wave_sync();
      bool ambiguous = false;
      // A trail that covers a whole search (the first pass went all the way: only the cut at k is open) IS
      // hnswlib's sequence of accepted entries wherever it sets no stretch apart.  From its last marker on
      // nothing but the result heap needs replaying: the search below stops there (with no marker at all it
      // is not even started), and the heap is fed from the log of what the search accepted so far and then
      // from the rest of the trail — no queue, no set, no rows.
      const uint4* trail = tmeta.x >= 0 ? a.trail + (size_t)tmeta.x * a.trail_cap : nullptr;
      const bool whole = trail != nullptr && tmeta.z < 0;
      const int trail_hops = tmeta.z < 0 ? -tmeta.z : tmeta.z;
      int last_marker = -1;
      if (whole) {
        for (int base = 0; base < tmeta.y; base += 64) {
          const int i = base + lane;
          const unsigned long long m = __ballot(i < tmeta.y && trail[i < tmeta.y ? i : 0].x >= kTrailBack);
          if (m != 0ull) last_marker = base + 63 - __builtin_clzll(m);
        }
      }
      int rest_from = (whole && last_marker < 0) ? 0 : -1;  // >= 0: the trail's records from here on are the rest of the accepted sequence
      if (rest_from < 0)
        search_level_lean<DT, QR, NS>(ix, qv, a.ef, s, st, fr, 1, lane, &ambiguous, trail, tmeta.y,
                                      trail != nullptr ? trail_hops : 0, tmeta.w, whole ? last_marker : -1, &rest_from);
      if (rest_from >= 0 && !st.fail) {
        __threadfence_block();
        LdsHeap top{s.top};
        int size = 0;
        if (st.n_acc == 0) {  // (no search was made: the entry point is the first accepted entry)
          HeapEnt seed;
          seed.key = dcur;
          seed.id = cur;
          coop_push<false>(top, size, seed, lane);
        }
        replay_log(s, top, size, st.n_acc, a.ef, lane);
        for (int base = rest_from; base < tmeta.y; base += 64) {
          const int cnt = tmeta.y - base < 64 ? tmeta.y - base : 64;
          const uint4 r = trail[base + (lane < cnt ? lane : 0)];   // 64 records per fetch, handed out lane by lane
          for (int j = 0; j < cnt; ++j) {
            HeapEnt e;
            e.key = __builtin_bit_cast(float, __builtin_amdgcn_readlane((int)r.z, j));
            e.id = (uint32_t)__builtin_amdgcn_readlane((int)r.y, j);
            coop_push<false>(top, size, e, lane);
            if (size > a.ef) coop_pop<false>(top, size, s.tree, lane);
          }
        }
        st.top_size = size;
        st.n_hops = trail_hops;
        if (st.n_acc == 0) st.n_dist = tmeta.w;
        literal = true;
        T = 0;  // (set below, once the heap is down to k entries)
      } else {
      T = st.top_size < a.k ? st.top_size : a.k;
      // The first T entries of the set (equal keys among them in label order) are hnswlib's
      // answer unless equal keys sit across the cut, or the whole set is returned after an
      // eviction had twins to choose from; then the result heap is replayed from the log, as below.
      const bool inner_tie = !st.fail && frontier_tie_within<NS>(fr, a.ef, T - 1, st.top_size, lane);
      const bool replay = !st.fail && (frontier_tie_within<NS>(fr, a.ef, T, st.top_size, lane, T - 1) ||
                                       (ambiguous && T == st.top_size) || (inner_tie && T > 2 * a.lean.sets()));
      if (!st.fail && !replay) {
        wave_sync();
        frontier_dump<NS>(fr, a.ef, T, s.nbuf, s.dbuf, lane);
        wave_sync();
        if (inner_tie) order_equal_keys(ix, s.nbuf, s.dbuf, T, reinterpret_cast<uint32_t*>(s.vcache), lane);
        have_result = true;
      } else if (replay) {
        __threadfence_block();
        literal = true;
        LdsHeap top{s.top};
        int size = 0;
        replay_log(s, top, size, st.n_acc, a.ef, lane);
        st.top_size = size;
      }
      }
    } else if (NS == 0 && a.reverse) {
      // reverse_cand beyond the register set's capacity: a sorted list in LDS; the answer is its first k entries
      vcache_reset(s, lane);
      visit_single(s, st, cur, lane);
      if (lane == 0) s.nbuf[0] = cur;
      wave_sync();
      search_level_far_lds<DT, QR>(ix, qv, 0, a.ef, s, st, 1, lane);
      literal = false;
      T = st.top_size < a.k ? st.top_size : a.k;
      wave_sync();
      for (int e = lane; e < T; e += 64) {  // (the list has its own LDS: NS == 0)
        s.nbuf[e] = s.top[e].id & ~kExpanded;
        s.dbuf[e] = s.top[e].key;
      }
      have_result = true;
    } else {
    vcache_reset(s, lane);
    visit_single(s, st, cur, lane);
    if (lane == 0) s.nbuf[0] = cur;
    wave_sync();
    search_level<DT, QR, NS, false>(ix, qv, 0, a.ef, s, st, tk, 1, lane, NS == 0 ? a.deleted : nullptr);

    // the k best.  With the keys in registers: the entries of the log at or below the k-th
    // key are the answer unless equal keys straddle the cut; then (and for NS == 0) the
    // literal heap decides: replay every accepted entry through it, pop down to k.
    T = st.top_size < a.k ? st.top_size : a.k;
    if (NS > 0 && !st.fail) {
      __threadfence_block();
      const float bound = topkeys_at<NS>(tk, T - 1, a.ef, reinterpret_cast<float*>(s.cand), lane);
      const int cnt = collect_le(s.log, st.n_acc, bound, s.top, a.lcap, lane);
      if (cnt != T) {
        literal = true;
        LdsHeap top{s.top};
        int size = 0;
        replay_log(s, top, size, st.n_acc, a.ef, lane);
        st.top_size = size;
      }
    }
    }
    if (literal) {
      LdsHeap top{s.top};
      while (st.top_size > a.k) coop_pop<false>(top, st.top_size, s.tree, lane);
      T = st.top_size;
    }
    wave_sync();
    if (!have_result) {
      uint64_t* tie = nullptr;
      if (ix.labels) {
        // labels of the T survivors; with the keys in registers s.top aliases the queue's share,
        // whose first lcap entries hold the survivors themselves
        tie = reinterpret_cast<uint64_t*>(s.cand + (NS > 0 ? a.lcap : 0));
        for (int e = lane; e < T; e += 64) tie[e] = ix.labels[s.top[e].id];
        wave_sync();
      }
      rank_sort(s.top, tie, T, s.nbuf, s.dbuf, lane);
      wave_sync();
    }
    if (!a.hnswlib_dist && T > 0) {
      dist_list<DT, QR, true>(ix, qv, s.qlds, s.nbuf, T, s.dbuf, lane);
      wave_sync();
    }
    for (int r = lane; r < a.k; r += 64) {
      int out_id = -1;
      float out_d = INFINITY;
      if (r < T) {
        uint32_t id = s.nbuf[r];
        out_id = ix.labels ? (int)ix.labels[id] : (int)id;
        out_d = a.hnswlib_dist ? answer_key(s.dbuf[r]) : s.dbuf[r];
      }
      a.nns[(size_t)qi * a.k + r] = out_id;
      a.dists[(size_t)qi * a.k + r] = out_d;
    }
    if (lane == 0) {
      a.found[qi] = st.fail ? -1 : T;
      if (st.fail) atomicOr(a.status, 1);
      if (a.stats) {
        a.stats[(size_t)qi * 4 + 0] = st.n_dist;
        a.stats[(size_t)qi * 4 + 1] = st.n_hops;
        a.stats[(size_t)qi * 4 + 2] = st.n_dist_upper;
        a.stats[(size_t)qi * 4 + 3] = st.n_sweeps;
      }
    }
    if (!lean) undo_visited(s, st, lane);
    wave_sync();
    if (a.live) __builtin_amdgcn_s_setprio(0);  // waiting for the next query is nobody's critical path
  }
}

// loads the (zero padded, 128-byte aligned) vector of a stored node as the "query"
template <int QR, bool HALF>
__device__ __forceinline__ void load_node_query_t(QVec<QR>& qv, float4* qlds, const DevIndex& ix, uint32_t node, int lane) {
  const int rowlen = ix.Dp >> 2;
  const int used = (ix.D + 3) >> 2;  // chunks that hold data (the last one zero padded)
  const uint64_t first = (uint64_t)node * (uint32_t)rowlen;
  if (QR > 0) {
    const int sub = lane & 15;
#pragma unroll
    for (int k = 0; k < (QR > 0 ? QR : 1); ++k) {
      const int c = sub + 16 * k;
      const uint64_t at = first + (c < used ? c : 0);  // unconditional load
      const float4 t = HALF ? load_chunk_f16(ix.vectors, at) : load_chunk_f32(ix.vectors, at);
      qv.q[k] = masked(t, mask_if(c < used));
    }
  } else {
    const int chunks = query_lds_chunks(ix.Dp);
    wave_sync();
    for (int c = lane; c < chunks; c += 64) {
      const uint64_t at = first + (c < used ? c : 0);
      const float4 t = HALF ? load_chunk_f16(ix.vectors, at) : load_chunk_f32(ix.vectors, at);
      qlds[c] = masked(t, mask_if(c < used));
    }
    wave_sync();
  }
}
template <int QR>
__device__ __forceinline__ void load_node_query(QVec<QR>& qv, float4* qlds, const DevIndex& ix, uint32_t node, int lane) {
  if (uni(ix.half) != 0) load_node_query_t<QR, true>(qv, qlds, ix, node, lane);
  else load_node_query_t<QR, false>(qv, qlds, ix, node, lane);
}

// Neighbour selection (HNSW Alg. 4 / hnswlib getNeighborsByHeuristic2) with the two
// extras of the reference's SearchHeuristic (cpp/include/cuda_build_kernels.cuh:68-162):
// the first nn_num candidates pass unconditionally, and with save_remains pruned
// candidates fill the row from the tail.  Candidates sid/skey[0..T) are ascending.
// Returns the degree; oid/okey[0..degree) is the new row.
//
// new_from > 0 is the reference's new_comer shortcut (cuda_build_kernels.cuh:109-110,122-125,137-138) in the
// form that is exact for any number of newcomers: the candidates with an id below new_from are a row that
// this very rule produced before (each of them was tested against every pick before it and passed), the
// others are newcomers.  A newcomer is tested against every pick before it, as always; an old candidate only
// against the NEWCOMERS picked before it — the old picks before it are a subset of those it has passed
// already.  Same row as the full rule, at a fraction of its pair tests.  (Only with nn_num = 0 and without
// save_remains: free picks and tail fill make a row that the rule's own tests do not vouch for.)
//
// The rule asks, candidate after candidate, whether any pick before it is closer to it than the node is.  Here the
// PICK asks: 64 candidates at a time, one per lane, and each pick strikes out at once those after it that are closer
// to it than to the node; the first one left standing is the next pick.  Same outcome (a candidate falls to any pick
// before it, whatever the order of the tests; a distance has the same bits from either end), but a struck-out
// candidate is tested no further, and the chain of dependent steps is one per pick (a dozen, each over all rows still
// standing: sixteen in flight) instead of one per candidate (ef_construction of them, each waiting for its own vector
// and its few rows): latency is what bounds this part.  Blocks of 64 rather than the whole list: where next to nothing
// is struck out the row is full before the later candidates come up, and tests on them would have been for nothing.
// (From array to index file, candidate by candidate -> pick by pick: 1 183 514 x 50 with 110 candidates 197 -> 167 ms,
// 200 003 x 128 with 200 candidates 110 -> 80 ms, 20 000 x 50 12.9 -> 10.3 ms.)
template <int DT, int QR>
__device__ __forceinline__ int select_neighbors(const DevIndex& ix, const uint32_t* sid, const float* skey, int T, int m,
                                                int nn_num, int save_remains, uint32_t* oid, float* okey, Scratch& s,
                                                int lane, unsigned int* work = nullptr, uint32_t new_from = 0u) {
  int head = 0, rejected = 0;
  const int tail = (m < T ? m : T) - 1;
  for (int base = 0; base < T && head < m; base += 64) {
    const int cnt = T - base < 64 ? T - base : 64;
    const int at = base + (lane < cnt ? lane : cnt - 1);
    const uint32_t my_id = sid[at];
    const float my_key = skey[at];
    const unsigned long long block = cnt < 64 ? (1ull << cnt) - 1ull : ~0ull;
    // candidates that pass untested (nn_num free picks), and those that only newcomers may strike out
    const int free_here = nn_num - base;
    const unsigned long long tested = free_here <= 0 ? block : (free_here >= 64 ? 0ull : block & ~((1ull << free_here) - 1ull));
    const unsigned long long newcomers = __ballot(my_id >= new_from);  // (new_from = 0: all of them)
    unsigned long long standing = block;
    unsigned long long todo = block;  // standing candidates that are not picks yet
    int h = 0;                        // the pick whose turn it is: first those of the blocks before, then this block's
    while (true) {
      uint32_t p;
      if (h == head) {
        if (todo == 0ull || head >= m) break;
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        if (lane == j) {
          oid[head] = my_id;
          okey[head] = my_key;
        }
        __builtin_amdgcn_wave_barrier();
        head += 1;
        if (head >= m) break;
        p = (uint32_t)__builtin_amdgcn_readlane((int)my_id, j);
      } else {
        p = (uint32_t)uni((int)oid[h]);
      }
      h += 1;
      const unsigned long long ask = todo & tested & (p >= new_from ? ~0ull : newcomers);
      if (ask != 0ull) {
        const int n = __popcll(ask);
        const int pos = lanes_below(ask);
        const bool mine = __builtin_amdgcn_inverse_ballot_w64(ask);
        QVec<QR> pv;
        load_node_query<QR>(pv, s.qlds, ix, p, lane);
        if (mine) s.nbuf[pos] = my_id;
        __builtin_amdgcn_wave_barrier();
        if (work && lane == 0) {  // (LDS: +2 pair tests, +3 rows of the picks of this level's counters)
          work[2] += (unsigned int)n;
          work[3] += 1u;
        }
        wave_sync();
        dist_list<DT, QR, false>(ix, pv, s.qlds, s.nbuf, n, s.dbuf, lane);
        wave_sync();
        const float d = s.dbuf[pos < n ? pos : 0];
        const unsigned long long out = __ballot(mine && my_key > d);
        standing &= ~out;
        todo &= ~out;
        wave_sync();
      }
    }
    if (save_remains && head < m) {
      // the r-th candidate turned away goes r places before the row's end, unless a pick ends up there
      const unsigned long long out = block & ~standing;
      const int slot = tail - rejected - lanes_below(out);
      if (__builtin_amdgcn_inverse_ballot_w64(out) && slot >= head) {
        oid[slot] = my_id;
        okey[slot] = my_key;
      }
      __builtin_amdgcn_wave_barrier();
      rejected += __popcll(out);
      wave_sync();
    }
  }
  wave_sync();
  return save_remains ? tail + 1 : head;
}

__device__ __forceinline__ uint32_t* link_row_mut(const DevIndex& ix, uint32_t node, int level) {
  return level == 0 ? ix.links0 + (size_t)node * ix.S0 : ix.linksU + (size_t)(ix.upper_off[node] + level - 1) * ix.SU;
}
__device__ __forceinline__ float* dist_row_mut(const DevIndex& ix, uint32_t node, int level) {
  return level == 0 ? ix.dists0 + (size_t)node * ix.S0 : ix.distsU + (size_t)(ix.upper_off[node] + level - 1) * ix.SU;
}

// A new node's row of one level, chosen by the selection (LDS): written in its place, and the node left in the inbox of
// each neighbour it chose, which goes on the list of touched rows with its first one.  Nothing reads either before the
// batch's next phase.  (As a kernel of its own, a thread per slot of every row, this was 7 of the 104 ms that 1 183 514 x
// 50 take to build: one counter for the touched rows, asked by every wavefront at once.  Here the searches of other nodes
// run while the atomics are under way.)
__device__ __forceinline__ void write_row_and_post(const DevIndex& ix, const BuildArgs& a, uint32_t x, int level, const uint32_t* oid,
                                                   const float* okey, int deg, int lane) {
  const int m_cap = level == 0 ? ix.max_m0 : ix.max_m;
  uint32_t* row = link_row_mut(ix, x, level);
  float* drow = dist_row_mut(ix, x, level);
  for (int base = 0; base < m_cap; base += 64) {
    const int j = base + lane;
    const bool link = j < deg;
    const uint32_t y = link ? oid[j] : kEmpty;
    const float key = link ? okey[j] : 0.f;
    if (j < m_cap) {
      row[j] = y;
      drow[j] = key;
    }
    bool first = false;
    if (link) {
      const size_t r = level == 0 ? (size_t)y : (size_t)(ix.upper_off[y] + level - 1);
      const int slot = atomicAdd((level == 0 ? a.inbox0_cnt : a.inboxU_cnt) + r, 1);
      first = slot == 0;
      if (slot < a.cap_in) {
        HeapEnt e;
        e.key = key;
        e.id = x;
        (level == 0 ? a.inbox0 : a.inboxU)[r * a.cap_in + slot] = e;
      }
    }
    const unsigned long long touched = __ballot(first);
    if (touched != 0ull) {
      int at = 0;
      if (lane == 0) at = atomicAdd(a.dirty_cnt, __popcll(touched));
      at = uni(at);
      if (first) a.dirty[at + lanes_below(touched)] = (unsigned long long)y | ((unsigned long long)level << 32);
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (lane == 0 && a.selected0) {
    // (with free picks or the tail fill the row holds entries the rule's tests do not vouch for)
    const unsigned char pure = (level == 0 ? a.nn_num0 : a.nn_numU) == 0 && !a.save_remains;
    if (level == 0) a.selected0[x] = pure;
    else a.selectedU[(size_t)(ix.upper_off[x] + level - 1)] = pure;
  }
  __builtin_amdgcn_wave_barrier();
}

// Phase 1 of a build batch: search, select, write the new rows, post the reverse links.
// (held to six / five wavefronts per SIMD where the query fits one / two float4 registers: a few
// spilled registers, 3-4 % off the build time of the 1.18 M x 50 and 10 M x 96 sets)
// TEAM: a batch that leaves the machine idle, a workgroup per node (team_help), those of the list first; sorted set only.
template <int DT, int QR, int NS, bool TEAM = false>
__global__ void __launch_bounds__(TEAM ? 64 * kMostTeam : 64, TEAM ? (QR != 0 && NS <= 8 ? 4 : 2) : (NS <= 5 && QR == 1) ? 6 : ((NS <= 5 && QR == 2) ? 5 : 1)) build_search_kernel(DevIndex ix, BuildArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  int lane = threadIdx.x & 63;
  const int m_max = ix.max_m0 > ix.max_m ? ix.max_m0 : ix.max_m;
  const bool sorted_set = TEAM || (NS > 0 && a.fc.sets() > 0);
  const LdsPlan lp = plan_lds(QR, ix.Dp, sorted_set ? -1 : a.efc, a.cand_lds, a.lcap, a.efc, m_max, a.vc_bits, a.fc);
  Scratch s;
  s.vcache = sorted_set ? reinterpret_cast<uint16_t*>(smem + lp.fcache)
                        : (a.vc_bits > 0 ? reinterpret_cast<uint16_t*>(smem + lp.vcache) : nullptr);
  s.vc_bits = a.vc_bits;
  s.filter = a.fc;
  s.qlds = reinterpret_cast<float4*>(smem + lp.qlds);
  s.top = reinterpret_cast<HeapEnt*>(smem + lp.top);
  s.cand = reinterpret_cast<HeapEnt*>(smem + lp.cand);
  s.cand_lds = a.cand_lds;
  s.nbuf = reinterpret_cast<uint32_t*>(smem + lp.nbuf);
  s.dbuf = reinterpret_cast<float*>(smem + lp.dbuf);
  uint32_t* sid = reinterpret_cast<uint32_t*>(smem + lp.sorted_id);
  float* skey = reinterpret_cast<float*>(smem + lp.sorted_key);
  uint32_t* oid = reinterpret_cast<uint32_t*>(smem + lp.out_id);
  float* okey = reinterpret_cast<float*>(smem + lp.out_key);
  s.tree = make_stage_tree(lane);
  bind_slot(s, a.pool, blockIdx.x);
  // this wavefront's share of a.counters (LDS, so that counting costs the kernel no registers when it is off)
  __shared__ unsigned int work[16];
  if (threadIdx.x < 16) work[threadIdx.x] = 0u;
  wave_sync();
  int taken = 0;  // (TEAM) nodes this workgroup has dealt with
  if (TEAM) {
    const int at = (int)blockIdx.x < a.n_upper ? a.upper[blockIdx.x] : (int)blockIdx.x - a.n_upper;
    const uint32_t x = (uint32_t)(a.begin + uni(at < a.count ? at : 0));
    const int lx = ix.levels[x];
    const int top_level = uni(lx < a.cur_max ? lx : a.cur_max);
    const bool here = uni(((int)blockIdx.x < a.n_upper || a.n_upper == 0 || lx <= 0) ? 1 : 0) != 0;
    // (a row that lies in LDS: there before gather_team's barrier, all wavefronts write the same.  The selection puts its picks in its
    // place, and a helper that came to write it only then would have the picks' tests made against the node.)
    QVec<QR> qv;
    if (QR == 0) load_node_query<QR>(qv, s.qlds, ix, x, lane);
    const int wave = gather_team<NS>(s, smem + lp.total, ix.S0 > ix.SU ? ix.S0 : ix.SU, top_level > 0 ? top_level : 0, a.team_bucket_bits, a.team_turn);
    if (wave > 0) {
      if (here && top_level >= 0) {
        if (QR != 0) load_node_query<QR>(qv, s.qlds, ix, x, lane);
        team_help<DT, QR, true>(ix, qv, s, wave - 1, lane);
      }
      return;
    }
    __builtin_amdgcn_s_setprio(3);
  }

  for (;;) {
    // first the n_upper nodes of the list, then all by id, the ones of the list passed over
    lane = fresh(lane);
    int b = 0;
    if (TEAM) {
      b = (int)blockIdx.x;
      b = b < a.n_upper ? a.upper[b] : b - a.n_upper + (1 << 30);
      if (taken++ > 0) b = a.count + (1 << 30);
    } else if (lane == 0) {
      b = atomicAdd(a.counter, 1);
      b = b < a.n_upper ? a.upper[b] : b - a.n_upper + (1 << 30);
    }
    b = __builtin_amdgcn_readfirstlane(b);
    const bool listed = b < (1 << 30);
    b &= (1 << 30) - 1;
    if (b >= a.count) break;
    const uint32_t x = (uint32_t)(a.begin + b);
    const int lx = ix.levels[x];
    const int top_level = lx < a.cur_max ? lx : a.cur_max;  // levels x shares with the graph so far
    const bool here = listed || a.n_upper == 0 || lx <= 0;
    // (the very first node has nothing to link to)
    if (here && top_level >= 0) {
      QVec<QR> qv;
      load_node_query<QR>(qv, s.qlds, ix, x, lane);
      SearchState st;
      st.undo_cnt = 0; st.n_dist = 0; st.n_hops = 0; st.n_dist_upper = 0; st.n_sweeps = 0; st.fail = 0; st.ahead = 1;

      // hnswlib addPoint: greedy descent from the entry point down to the node's top level,
      // then search + select on every level it has, entering each level at the closest
      // neighbour chosen one level up
      uint32_t cur = (uint32_t)a.cur_ep;
      if (a.cur_max > lx) {
        float dcur = dist_single<DT, QR>(ix, qv, cur, s, lane);
        descend<DT, QR>(ix, qv, a.cur_max, lx, cur, dcur, s, st, lane);
      }
      for (int level = top_level; level >= 0; --level) {
        lane = fresh(lane);
        const int m_cap = level == 0 ? ix.max_m0 : ix.max_m;
        st.top_size = 0; st.cand_size = 0; st.n_acc = 0; st.lower = 0.f; st.maxkey = -INFINITY; st.ahead = 1;
        const int evals_before = st.n_dist, hops_before = st.n_hops;
        int T;
        if (sorted_set) {
          if (!TEAM || level < top_level) filter_reset(s, lane);
          if (TEAM) {
            if (level < top_level) team_open(s.team, level, lane);
            HeapEnt e;
            e.key = INFINITY;
            e.id = cur;
            if (lane == 0) s.team.line()[8] = e;
            __builtin_amdgcn_wave_barrier();
          }
          // sorted set in registers: the efc best come out in order (equal keys in the order
          // the set placed them, which is deterministic).  The new node itself cannot turn up:
          // nothing links to it before the batch's later phases.
          visit_lossy_single(s, cur, lane);
          if (lane == 0) s.nbuf[0] = cur;
          wave_sync();
          Frontier<NS> fr;
          frontier_init<NS>(fr, a.efc, lane);
          search_level_fast<DT, QR, NS, true, false, TEAM, TEAM>(ix, qv, level, a.efc, s, st, fr, 1, lane, a.reverse != 0);
          T = st.top_size;
          if (TEAM) {
            if (level > 0) team_close(s.team, lane);
            else if (lane == 0) lds_tell(s.team.over(), 1u);
            __builtin_amdgcn_wave_barrier();
          }
          wave_sync();
          frontier_dump<NS>(fr, a.efc, T, sid, skey, lane);
          wave_sync();
        } else if (NS == 0 && a.reverse) {
          // reverse_cand beyond the register set's capacity: a sorted list in LDS, already in order
          vcache_reset(s, lane);
          visit_single(s, st, x, lane);  // a node never links to itself
          visit_single(s, st, cur, lane);
          if (lane == 0) s.nbuf[0] = cur;
          wave_sync();
          search_level_far_lds<DT, QR>(ix, qv, level, a.efc, s, st, 1, lane);
          T = st.top_size;
          wave_sync();
          for (int e = lane; e < T; e += 64) {
            sid[e] = s.top[e].id & ~kExpanded;
            skey[e] = s.top[e].key;
          }
          wave_sync();
        } else {
          vcache_reset(s, lane);
          visit_single(s, st, x, lane);  // a node never links to itself
          visit_single(s, st, cur, lane);
          if (lane == 0) s.nbuf[0] = cur;
          wave_sync();
          TopKeys<NS> tk;
          topkeys_init<NS>(tk, a.efc, lane);
          search_level<DT, QR, NS, true>(ix, qv, level, a.efc, s, st, tk, 1, lane);
          T = st.top_size;
          if (NS > 0 && T > 0) {
            __threadfence_block();
            const float bound = topkeys_at<NS>(tk, T - 1, a.efc, reinterpret_cast<float*>(s.cand), lane);
            T = collect_best(s.log, st.n_acc, bound, T, s.top, lane);
          }
          wave_sync();
          rank_sort(s.top, nullptr, T, sid, skey, lane);
          wave_sync();
        }
        lane = fresh(lane);
        unsigned int* level_work = a.counters ? work + (level == 0 ? 0 : 5) : nullptr;
        const int deg = select_neighbors<DT, QR>(ix, sid, skey, T, level == 0 ? a.own_cap0 : m_cap,
                                                 level == 0 ? a.nn_num0 : a.nn_numU, a.save_remains, oid, okey, s, lane,
                                                 level_work);
        if (level_work && lane == 0) {
          level_work[0] += (unsigned int)(st.n_dist - evals_before);
          level_work[1] += (unsigned int)(st.n_hops - hops_before);
          level_work[4] += 1u;
        }
        if (QR == 0) load_node_query<QR>(qv, s.qlds, ix, x, lane);  // the LDS query copy was reused by the selection
        write_row_and_post(ix, a, x, level, oid, okey, deg, lane);
        if (deg > 0) cur = oid[0];  // closest selected neighbour: entry for the level below
        wave_sync();
        if (!sorted_set) {
          undo_visited(s, st, lane);
          wave_sync();
        }
      }
      if (lane == 0 && st.fail) *a.status = 1;
      if (a.counters && lane == 0) {
        work[5] += (unsigned int)st.n_dist_upper + (a.cur_max > lx ? 1u : 0u);  // the descent and its entry point
        work[6] += (unsigned int)st.n_sweeps;
      }
    }
  }
  wave_sync();
  if (a.counters && lane < 10 && work[lane] != 0u) atomicAdd(a.counters + lane, (unsigned long long)work[lane]);
}

// More newcomers chose node y on this level than its inbox holds (a hub of a clustered set, late in a
// large batch).  Which of them reached the inbox depends on the order of the atomics, so the inbox is
// not used: the rows of the batch's nodes are scanned for y and the cap closest newcomers by (key, id) are
// collected into obox (LDS, cap entries) — the same set in every run.  Returns how many newcomers chose
// y in all.  Rare; one wavefront reads the rows of the whole batch.
__device__ __forceinline__ int gather_overflowed_inbox(const DevIndex& ix, const BuildArgs& a, uint32_t y, int level,
                                                       HeapEnt* obox, int cap, int lane) {
  int size = 0, total = 0;
  for (int base = 0; base < a.count; base += 64) {
    const int b = base + lane;
    bool hit = false;
    float my_key = 0.f;
    uint32_t my_id = kEmpty;
    if (b < a.count) {
      const uint32_t x = (uint32_t)(a.begin + b);
      const int lx = ix.levels[x];
      const int top_level = lx < a.cur_max ? lx : a.cur_max;
      if (level <= top_level) {
        const uint32_t* ids = link_row(ix, x, level);  // (no row of a batch's node is touched in its own batch)
        const float* keys = dist_row_mut(ix, x, level);
        const int m_cap = level == 0 ? ix.max_m0 : ix.max_m;
        for (int j = 0; j < m_cap && ids[j] != kEmpty; ++j) {
          if (ids[j] == y) {
            hit = true;
            my_key = keys[j];
            my_id = x;
          }
        }
      }
    }
    unsigned long long todo = __ballot(hit);
    total += __popcll(todo);
    while (todo != 0ull) {
      const int j = __builtin_ctzll(todo);
      todo &= todo - 1ull;
      const float key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_key), j));
      const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)my_id, j);
      if (size < cap) {
        if (lane == 0) {
          obox[size].key = key;
          obox[size].id = id;
        }
        size += 1;
      } else {
        // the farthest entry of the list by (key, id) gives way if the newcomer is closer
        const HeapEnt m = obox[lane < cap ? lane : 0];
        const bool in = lane < cap;
        const float far_key = -least_of_all(in ? -m.key : INFINITY);
        const bool at_far = in && m.key == far_key;
        uint32_t far_id = at_far ? m.id : 0u;
#pragma unroll
        for (int sh = 32; sh >= 1; sh >>= 1) {
          const uint32_t o = (uint32_t)__shfl_xor((int)far_id, sh, 64);
          far_id = o > far_id ? o : far_id;
        }
        const bool closer = key < far_key || (key == far_key && id < far_id);
        if (closer && at_far && m.id == far_id) {
          obox[lane].key = key;
          obox[lane].id = id;
        }
      }
      wave_sync();
    }
  }
  return total;
}

// Phase 2: one wavefront per (node, level) that received reverse links.
template <int DT, int QR>
__global__ void __launch_bounds__(64) reverse_kernel(DevIndex ix, BuildArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x;
  const int s_max = ix.S0 > ix.SU ? ix.S0 : ix.SU;
  const int m_max = ix.max_m0 > ix.max_m ? ix.max_m0 : ix.max_m;
  const int ncand = s_max + a.cap_in;
  // plan: "top" region holds the merged candidates, sorted_* their ranking
  const LdsPlan lp = plan_lds(QR, ix.Dp, ncand, 0, a.lcap, ncand, m_max > a.cap_in ? m_max : a.cap_in);
  Scratch s;
  s.qlds = reinterpret_cast<float4*>(smem + lp.qlds);
  HeapEnt* cbuf = reinterpret_cast<HeapEnt*>(smem + lp.top);
  s.nbuf = reinterpret_cast<uint32_t*>(smem + lp.nbuf);
  s.dbuf = reinterpret_cast<float*>(smem + lp.dbuf);
  uint32_t* sid = reinterpret_cast<uint32_t*>(smem + lp.sorted_id);
  float* skey = reinterpret_cast<float*>(smem + lp.sorted_key);
  uint32_t* oid = reinterpret_cast<uint32_t*>(smem + lp.out_id);
  float* okey = reinterpret_cast<float*>(smem + lp.out_key);
  const int n_dirty = *a.dirty_cnt;
  __shared__ unsigned int work[16];
  if (lane < 16) work[lane] = 0u;
  wave_sync();

  // What a touched row is made of, lane by lane: the row itself (its first 64 slots), its keys, its inbox and how many were
  // posted there.  All of it is asked for at once (an inbox is read whole, whatever is in it), and for the next row before
  // this one is dealt with: one after the other these are four trips to memory, which is what most rows' time was.
  struct Touched {
    uint32_t y, id;
    int level, posted;
    float key;
    HeapEnt in;
  };
  auto fetch = [&](unsigned long long entry) __attribute__((always_inline)) {
    Touched t;
    t.y = (uint32_t)uni((int)(uint32_t)(entry & 0xffffffffull));
    t.level = uni((int)(entry >> 32));
    const size_t r = t.level == 0 ? (size_t)t.y : (size_t)(ix.upper_off[t.y] + t.level - 1);
    const int S = row_stride(ix, t.level);
    t.posted = (t.level == 0 ? a.inbox0_cnt : a.inboxU_cnt)[r];
    t.id = link_row(ix, t.y, t.level)[lane < S ? lane : 0];
    t.key = dist_row_mut(ix, t.y, t.level)[lane < S ? lane : 0];
    t.in = ((t.level == 0 ? a.inbox0 : a.inboxU) + r * a.cap_in)[lane < a.cap_in ? lane : 0];
    return t;
  };
  const int step = (int)gridDim.x;
  Touched next;
  unsigned long long entry_after = 0ull;
  if ((int)blockIdx.x < n_dirty) {
    next = fetch(a.dirty[blockIdx.x]);
    entry_after = a.dirty[(int)blockIdx.x + step < n_dirty ? (int)blockIdx.x + step : 0];
  }
  for (int di = blockIdx.x; di < n_dirty; di += step) {
    const Touched t = next;
    if (di + step < n_dirty) {
      next = fetch(entry_after);
      entry_after = a.dirty[di + 2 * step < n_dirty ? di + 2 * step : 0];
    }
    const uint32_t y = t.y;
    const int level = t.level;
    const int S = row_stride(ix, level);
    const int m_cap = level == 0 ? ix.max_m0 : ix.max_m;
    int* cnt = level == 0 ? a.inbox0_cnt + y : a.inboxU_cnt + (size_t)(ix.upper_off[y] + level - 1);
    const int posted = uni(t.posted);
    const int n_new = posted < a.cap_in ? posted : a.cap_in;
    HeapEnt in = t.in;
    if (posted > a.cap_in) {
      // (the overflow list takes the LDS of the selection's output rows, which are not in use yet; the
      // host sizes them for cap_in entries)
      HeapEnt* obox = reinterpret_cast<HeapEnt*>(smem + lp.out_id);
      const int total = gather_overflowed_inbox(ix, a, y, level, obox, a.cap_in, lane);
      if (lane == 0) atomicAdd(a.dropped, total - a.cap_in);
      wave_sync();
      in = obox[lane < a.cap_in ? lane : 0];
    }
    uint32_t* row = link_row_mut(ix, y, level);
    float* drow = dist_row_mut(ix, y, level);
    // the links there are, in front of the candidate list (a newcomer cannot be among them: it was in no row before)
    int n0 = 0;
    for (int base = 0; base < S; base += 64) {
      uint32_t id = t.id;
      float key = t.key;
      if (base > 0) {
        id = row[base + lane < S ? base + lane : 0];
        key = drow[base + lane < S ? base + lane : 0];
      }
      const unsigned long long mask = __ballot(base + lane < S && id != kEmpty);
      if (__builtin_amdgcn_inverse_ballot_w64(mask)) {
        HeapEnt e;
        e.key = key;
        e.id = id;
        cbuf[n0 + lanes_below(mask)] = e;
      }
      __builtin_amdgcn_wave_barrier();
      n0 += __popcll(mask);
    }
    const int T = n0 + n_new;
    unsigned char* selected = !a.selected0 ? nullptr
                              : (level == 0 ? a.selected0 + y : a.selectedU + (size_t)(ix.upper_off[y] + level - 1));
    if (T <= m_cap) {
      // room for all: the newcomers go behind the row, ordered by (key, id)
      int before = 0;
      for (int i = 0; i < n_new; ++i) {
        const float key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, in.key), i));
        const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)in.id, i);
        before += key < in.key || (key == in.key && id < in.id) ? 1 : 0;
      }
      if (lane < n_new) {
        row[n0 + before] = in.id;
        drow[n0 + before] = in.key;
      }
      if (selected && lane == 0) *selected = 0;  // no longer what the selection rule alone would leave
    } else {
      if (lane < n_new) cbuf[n0 + lane] = in;
      wave_sync();
      rank_sort(cbuf, nullptr, T, sid, skey, lane);
      wave_sync();
      // A row that is an output of the rule is re-selected with the shortcut for newcomers: the nodes of this
      // batch (ids from a.begin on; everything the row held before has a smaller id).
      const int nn_num = level == 0 ? a.nn_num0 : a.nn_numU;
      const bool pure = nn_num == 0 && !a.save_remains;
      const bool shortcut = pure && selected && uni((int)*selected) != 0;
      const int deg = select_neighbors<DT, QR>(ix, sid, skey, T, m_cap, nn_num, a.save_remains, oid, okey, s, lane,
                                               a.counters ? work + (level == 0 ? 0 : 5) : nullptr,
                                               shortcut ? (uint32_t)a.begin : 0u);
      for (int j = lane; j < m_cap; j += 64) {
        row[j] = j < deg ? oid[j] : kEmpty;
        drow[j] = j < deg ? okey[j] : 0.f;
      }
      if (selected && lane == 0) *selected = pure ? 1 : 0;
    }
    if (lane == 0) *cnt = 0;
    if (a.counters && lane == 0) {
      unsigned int* level_work = work + (level == 0 ? 0 : 5);
      level_work[1] += 1u;
      level_work[4] += 1u;
    }
    wave_sync();
  }
  wave_sync();
  if (a.counters && lane < 10 && work[lane] != 0u) atomicAdd(a.counters + lane, (unsigned long long)work[lane]);
}

// Measurement aid: nothing but the search's memory access pattern.  Every 16-lane group fetches pseudo-random
// vector rows of the resident index, U rows per group in flight, each lane one 16-byte chunk per 64 elements,
// exactly as the distance passes do; `dependent` makes each batch of loads wait for the one before, as a hop
// waits for its rows.  Gives the rate at which this GPU's memory system delivers random rows of THIS index.
template <int U>
__global__ void __launch_bounds__(64) gather_probe_kernel(DevIndex ix, int batches, int dependent, float* sink) {
  const int lane = threadIdx.x, g = lane >> 4, sub = lane & 15;
  const uint32_t rowlen = (uint32_t)ix.Dp >> 2, used = ((uint32_t)ix.D + 3u) >> 2;
  const int nk = (int)((used + 15u) >> 4);
  uint32_t x = (uint32_t)(blockIdx.x * 4 + g) * 2654435761u + 12345u;
  float acc = 0.f;
  uint32_t chain = 0u;
  for (int b = 0; b < batches; ++b) {
    for (int k = 0; k < nk; ++k) {
      float4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        uint32_t y = x + (uint32_t)u * 0x9E3779B9u;
        y ^= y >> 15; y *= 0x2C1B3C6Du; y ^= y >> 12; y *= 0x297A2D39u; y ^= y >> 15;
        const uint32_t id = (uint32_t)(((unsigned long long)y * (unsigned long long)ix.N) >> 32) + chain;
        const uint32_t c = sub + 16u * (uint32_t)k;
        const unsigned long long at = (unsigned long long)id * rowlen + (c < used ? c : 0u);
        v[u] = ix.half ? load_chunk_f16(ix.vectors, at) : load_chunk_f32(ix.vectors, at);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) acc += (v[u].x + v[u].y) + (v[u].z + v[u].w);
    }
    x = x * 1664525u + 1013904223u;
    if (dependent) chain = acc == 1234567.0f ? 1u : 0u;  // (never true: the next addresses just have to wait for this sum)
  }
  if (acc == 7654321.0f) sink[blockIdx.x] = acc;
}

// Upload helper: N rows of D floats into rows of Dp elements, zero padded; a thread writes four of them.  (fp16: to
// nearest even.)
template <typename T>
__global__ void __launch_bounds__(256) pad_rows_kernel(const float* src, T* dst, long long n, int D, int Dp) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int chunks = Dp >> 2;
  if (i >= n * chunks) return;
  const long long row = i / chunks;
  const int col = 4 * (int)(i - row * chunks);
  const float* from = src + row * D + col;
  struct __attribute__((aligned(4 * sizeof(T)))) Four { T v[4]; } out;
#pragma unroll
  for (int j = 0; j < 4; ++j) out.v[j] = col + j < D ? (T)from[j] : (T)0.f;
  *reinterpret_cast<Four*>(dst + row * Dp + col) = out;
}

// ---- level-0 records of an index file: [count | max_m0 ids | D floats | label], 32-bit words ------------------------
// One wavefront per record, four per workgroup: a record is read and written in whole lines whatever its length.
static __global__ void __launch_bounds__(256) pack_records_kernel(DevIndex ix, int first, int rows, const uint32_t* deleted,
                                                                  uint32_t* out) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int i = first + r;
  uint32_t* rec = out + (size_t)r * (size_t)(1 + ix.max_m0 + ix.D + 2);
  const uint32_t* row = ix.links0 + (size_t)i * ix.S0;
  uint32_t deg = 0;
  for (int base = 0; base < ix.max_m0; base += 64) {
    const int k = base + lane;
    const uint32_t id = k < ix.max_m0 ? row[k] : kEmpty;
    deg += (uint32_t)__popcll(__ballot(id != kEmpty));
    if (k < ix.max_m0) rec[1 + k] = id != kEmpty ? id : 0u;  // unused link slots are zeros in the file
  }
  float* vec = reinterpret_cast<float*>(rec + 1 + ix.max_m0);
  const size_t at = (size_t)i * ix.Dp;
  for (int k = lane; k < ix.D; k += 64)
    vec[k] = ix.half ? (float)reinterpret_cast<const _Float16*>(ix.vectors)[at + k] : reinterpret_cast<const float*>(ix.vectors)[at + k];
  if (lane == 0) {
    const uint64_t label = ix.labels ? ix.labels[i] : (uint64_t)i;
    const bool marked = deleted && ((deleted[i >> 5] >> (i & 31)) & 1u) != 0u;
    rec[0] = deg | (marked ? kDeleteMark : 0u);
    rec[1 + ix.max_m0 + ix.D] = (uint32_t)label;
    rec[2 + ix.max_m0 + ix.D] = (uint32_t)(label >> 32);
  }
}
// status[0]: 1 = a link count above max_m0, 2 = a link id out of range; status[1] counts the delete marks (marks: one
// byte per record).  hnswlib keeps the count in the low 16 bits of its word and flags above: markDelete sets bit 0 of
// the third byte, the others are unknown and dropped.
static __global__ void __launch_bounds__(256) check_records_kernel(const uint32_t* raw, int n, int D, int max_m0,
                                                                   unsigned char* marks, int* status) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= n) return;
  const uint32_t* rec = raw + (size_t)i * (size_t)(1 + max_m0 + D + 2);
  const uint32_t word = rec[0];
  const uint32_t deg = word & 0xffffu;
  int wrong = deg > (uint32_t)max_m0 ? 1 : 0;
  for (int k = lane; k < max_m0; k += 64) wrong |= ((uint32_t)k < deg && rec[1 + k] >= (uint32_t)n) ? 2 : 0;
  if (wrong) atomicOr(status, wrong);
  if (lane == 0) {
    const bool marked = (word & kDeleteMark) != 0u;
    marks[i] = marked ? 1 : 0;
    if (marked) atomicAdd(status + 1, 1);
  }
}
static __global__ void __launch_bounds__(256) unpack_records_kernel(const uint32_t* raw, DevIndex ix, uint64_t* labels) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= ix.N) return;
  const uint32_t* rec = raw + (size_t)i * (size_t)(1 + ix.max_m0 + ix.D + 2);
  const int deg = (int)(rec[0] & 0xffffu);
  for (int k = lane; k < ix.S0; k += 64) ix.links0[(size_t)i * ix.S0 + k] = k < deg ? rec[1 + k] : kEmpty;
  const float* vec = reinterpret_cast<const float*>(rec + 1 + ix.max_m0);
  const size_t at = (size_t)i * ix.Dp;
  for (int k = lane; k < ix.Dp; k += 64) {
    const float x = k < ix.D ? vec[k] : 0.f;
    if (ix.half) const_cast<_Float16*>(reinterpret_cast<const _Float16*>(ix.vectors))[at + k] = (_Float16)x;
    else const_cast<float*>(reinterpret_cast<const float*>(ix.vectors))[at + k] = x;
  }
  if (lane == 0) labels[i] = (uint64_t)rec[1 + ix.max_m0 + ix.D] | ((uint64_t)rec[2 + ix.max_m0 + ix.D] << 32);
}

}  // namespace cuhnsw_amd
