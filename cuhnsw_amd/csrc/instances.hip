// Launches of the templated kernels, compiled once per distance and row width: the build passes CUHNSW_DT (DistType),
// CUHNSW_QR (kernels.h, query_regs) and CUHNSW_PART (0: searches, 1: index builds), so that the objects compile side by side.
#include "engine.h"

namespace cuhnsw_amd {

// (the no-allocation search clears its control words with this kernel: it issues no memset)
static __global__ void __launch_bounds__(128) fill_ints_kernel(int* p, int n, int value) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}
// Everything a two-pass search needs cleared, in one launch: the control words (0), the list the first pass
// appends to (-1 = "no entry yet", which the literal wavefronts poll for) and, for a batch taken longest
// first, the counters of the counting sort (0).
static __global__ void __launch_bounds__(256) prepare_search_kernel(int* ctl, int n_ctl, int* redo, int n_redo, int* hist, int n_hist) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_ctl) ctl[i] = 0;
  if (i < n_redo) redo[i] = -1;
  if (i < n_hist) hist[i] = 0;
}

// Two passes: every query on the sorted set in registers (search_fast_kernel); the queries
// in which equal keys met, and every query when ef exceeds the set's capacity, with the
// literal priority queues (search_kernel).  The literal pass normally runs at the same time
// on a second stream, on one wavefront per SIMD, and picks the given-up queries off a list
// as the first pass appends them; should it report a problem (its bounded wait ran out, or a
// queue overflowed) the list is answered again after the first pass.  ms covers everything.
template <int DT, int QR, int NS>
void Engine::launch_search(const DevIndex& ix, SearchArgs& a, int max_slots_override, float* ms) {
  a.counter = d_ctl.p;
  a.status = d_ctl.p + 1;
  a.repeats = d_ctl.p + 32;   // the counters of the two passes sit in separate 128-byte lines
  a.done = d_ctl.p + 64;
  a.redo = nullptr;
  a.live = 0;
  a.nq_total = a.nq;
  a.slot_base = 0;
  // a literal wavefront beside the first pass waits at most 2 ms for that pass to start (it is launched
  // microseconds later unless something serialises the two streams) and accepts no progress of a
  // started first pass for 100 ms (its queries finish every few microseconds)
  a.spin_limit = spin_limit_override;
  a.start_ticks = 2 * wall_clock_khz;
  a.stall_ticks = 100 * wall_clock_khz;
  a.nq_dev = nullptr;
  a.entry = nullptr;
  a.order_hist = nullptr;
  a.regions = nullptr;
  a.region_level = 0;
  a.shares = nullptr;
  a.order = nullptr;
  a.trail = nullptr;
  a.redo_trail = nullptr;
  a.trail_next = nullptr;
  a.trail_cap = a.trail_first_spare = a.trail_spares = 0;
  a.waiting = 0;
  a.report = nullptr;
  last_repeats = 0;
  last_trails = 0;
  last_side_by_side = last_team = 0;
  if (use_static) {
    launch_search_static<DT, QR, NS>(ix, a, ms);
    return;
  }
  if (ms) HIP_CHECK(hipEventRecord(ev0, stream));
  // The literal pass runs on the sorted set with ids and the LDS filter (no bitmap) where the first pass leaves it trails
  // (which only that variant replays), and else unless the caller asked for literal queues only, which also means exact
  // evaluation counters, or the visited bitmaps of the wavefronts at work fit the L2 caches (32 MB) together: there the
  // bitmap's atomics are cheap and a search from the entry point with them is the faster one.
  auto choose_variant = [&](bool with_trails) {
    const size_t bitmap_bytes = (size_t)std::min(num_cus * 24, a.nq) * ((host.N + 31) / 32) * 4;
    const bool want_lean = lean_literal == 1 ? with_trails || bitmap_bytes > ((size_t)32 << 20) : lean_literal > 1;
    a.lean = (NS > 0 && fast_path != 0 && want_lean) ? least_filter(a.ef) : FilterShape();
    if (a.lean.sets() && filter_entries <= 0) {
      int sets = 256;
      while (sets < a.lean.sets()) sets *= 2;
      a.lean = filter_shape(std::min(sets, 4096), host.N);
      // a batch of few queries leaves most of each CU's LDS unused: give the filter what is there
      // (up to 32 KB), so that it forgets next to nothing
      const int per_cu = (a.nq + num_cus - 1) / num_cus;
      const size_t room = per_cu > 0 ? (size_t)(150 * 1024) / per_cu : 0;
      const size_t other = plan_lds(QR, ix.Dp, NS > 0 ? -1 : a.ef, a.cand_lds, a.lcap, 0, 0).total + 256;
      while (a.lean.sets() < 4096 && other + 2 * a.lean.bytes() <= std::min<size_t>(room, 60 * 1024))
        a.lean = filter_shape(std::min(2 * a.lean.sets(), 4096), host.N);
    }
  };
  auto literal_lds = [&](int cand_lds) -> size_t {
    return plan_lds(QR, ix.Dp, NS > 0 ? -1 : a.ef, cand_lds, a.lcap, 0, 0, a.lean.sets() ? 0 : a.vc_bits, FilterShape(), a.lean).total;
  };
  auto kernel = search_kernel<DT, QR, NS>;
  int glob_cap = spill_cap > 0 ? spill_cap : std::max(4096, 8 * a.ef);
  int n_literal = a.nq;
  bool answered = false;
  bool timed = false;  // ev1 has been recorded after the last kernel of this search
  // The first pass takes every batch, however small: it needs half the literal search's time per expanded candidate
  // (100 000 x 50, ef 300: one query 0.81 -> 0.33 ms, 1 000 queries 1.03 -> 0.55).  A query that is handed over ends
  // later than it would have on the literal queues alone, though, replayed from its trail or not (1.23 ms there; 200 000
  // x 128 integers, ef 300: 1.2 ms without a hand-over, 1.9 with one, literal queues alone 1.78).  So where 1.5 or more
  // hand-overs are to be expected of a batch, three batches in four have one, and the batch is one round of literal
  // wavefronts whose bitmaps fit the L2, it goes to the literal queues alone (there, 1 000 queries of which 12 are handed
  // over: 2.27 -> 1.99 ms; 256 with 3: 1.89 -> 1.78; 32 with 0.4 stay, 1.46 against 1.60).  Not at ef <= 128, where a
  // replay is short (1 000 queries with 2.7: 0.80 ms, 0.86 on the literal queues), and not on rows that are read from
  // memory as long as the queues are busy (QR == 0).  One batch in sixteen takes the first pass all the same, so that the
  // share is not taken for known forever.
  bool literal_alone = false;
  if (NS > 2 && QR > 0 && fast_path == 1 && a.fast_path == 1 && a.fc.sets() > 0 && max_slots_override <= 0 &&
      cautious_share() * a.nq >= 1.5) {
    choose_variant(false);
    if (!a.lean.sets() && a.nq <= resident_slots(kernel, literal_lds(a.cand_lds))) {
      literal_alone = literal_streak < kLiteralStreak;
      literal_streak = literal_alone ? literal_streak + 1 : 0;
    }
  }
  const bool first_pass = NS > 0 && a.fast_path && a.fc.sets() > 0 && !literal_alone;  // (reverse_cand: fast_path is 2)
  if (!first_pass) choose_variant(false);
  if constexpr (NS > 0) if (first_pass) {
    d_redo.reserve((size_t)a.nq);
    a.redo = d_redo.p;
    auto fast_kernel = search_fast_kernel<DT, QR, NS, false>;
    auto fast_lds = [&](FilterShape f) -> size_t { return plan_fast_lds(QR, ix.Dp, a.rcap, f, a.k).total; };
    a.fc = fit_filter(fast_kernel, a.fc, fast_lds);
    const size_t fast_lds_bytes = fast_lds(a.fc);
    int slots = resident_slots(fast_kernel, fast_lds_bytes);
    // A batch of at most one wavefront per SIMD that is not expected to hand anything over does without the second
    // stream: its events and the wait for the waiting wavefronts are 60 us of a search of a few hundred.
    const bool alone = fast_path == 1 && !a.reverse && a.nq <= std::min(4 * num_cus, slots) && first_pass_waves == 0 &&
                       max_slots_override <= 0 && repeat_share * a.nq < 0.5;
    const bool side = concurrent_literal && sequential_left == 0 && max_slots_override <= 0 && !alone;
    last_side_by_side = side ? 1 : 0;
    int side_slots = 0;
    // few queries need the literal pass: one wavefront per CU serves them without taking room from
    // the first pass; two when the last search handed over 2 % and more (a literal wavefront's LDS
    // is that of one and a half wavefronts of the first pass, so more of them cost more than they serve)
    const int per_cu = side_per_cu > 0 ? side_per_cu : (repeat_share < 0.02 ? 1 : 2);
    if (side) {
      side_slots = std::min(num_cus * per_cu, a.nq);
      // an index that hands over next to nothing (the last search: under one query in a thousand) gets one
      // literal wavefront per four CUs, and the first pass the room of the others
      if (side_per_cu <= 0 && share_known && repeat_share < 0.001) side_slots = std::min(std::max(num_cus / 4, 1), a.nq);
      ensure_pool(std::max(side_slots, 1), glob_cap, 2 * glob_cap);
      slots = std::max(num_cus, slots - std::min(side_slots, num_cus * per_cu));  // leave the literal wavefronts their room
    }
    if (max_slots_override > 0) slots = max_slots_override;
    if (first_pass_waves > 0) slots = std::min(slots, first_pass_waves * num_cus);
    slots = std::max(1, std::min(slots, a.nq));
    // (every allocation before the literal pass is launched: growing a buffer frees the old one, and
    // hipFree waits for the device, on which that pass would be waiting for the first pass to start)
    const long long resident = slots;  // queries at work at a time
    // A handed-over query is not searched again from its entry point: the first pass leaves the entries it
    // accepted, hop by hop, and the literal pass (on the sorted set with ids: it needs no visited bitmap
    // brought up to date) replays its queue operations from them up to where the two may part.  One query per
    // wavefront, link rows of one pass of 64 lanes, and batches of under three rounds of wavefronts: keeping
    // the trail costs the first pass 9 % (the kernel instance with the trail code 4 %, writing the records the
    // rest), which only a batch short enough to wait for its last hand-over gets back.  trails = 2: whatever
    // the batch.  (Nor where the batch runs alone: one query in a hundred or fewer is handed over there, and the records
    // would cost every one of them 10 %, 0.383 -> 0.428 ms for a single query on 100 000 x 50 at ef 300.)
    bool keep_trails = !alone && (QR == 1 || QR == 2) && trails && !a.reverse && host.S0 <= 63 &&
                       (trails > 1 || 4 * (long long)a.nq <= 11 * resident);
    choose_variant(keep_trails);
    keep_trails = keep_trails && a.lean.sets() > 0;
    if (keep_trails) {
      // (normally there since the index became resident; a changed trail_cap / trail_spares asks again)
      if (d_trail.n < trail_records_wanted(slots)) {
        trails_unavailable = false;
        reserve_trails(slots);
      }
      keep_trails = !trails_unavailable && d_trail.n >= trail_records_wanted(slots);
    }
    // (with trails a late hand-over costs less, and the order pays from one round on)
    const bool in_order = query_order && (query_order == 2 ? a.nq > resident
                                                           : (keep_trails ? a.nq > resident : 2 * a.nq >= 3 * resident) &&
                                                                 a.nq <= 32 * resident);
    // Three rounds and more: all but the longest of them by region (kernels.h).  The level whose nodes stand for the regions
    // is the lowest that has four queries a node (of 1, 2, 3, 4: 2 is the best or next to it on 1 M x 96 with 100 000
    // queries, 1.18 M x 50 with 40 000, 500 000 x 128 with 30 000 and 100 000 x 960 with 8 000, that is 25, 5, 15 and 20).
    // Not on an index of which every chiplet's 4 MB of L2 holds a good part anyway: 20 000 x 30 (5 MB) 1.68 -> 1.75 ms,
    // 40 000 x 50 (15 MB) 1.98 -> 2.00 and 2.70 -> 2.61, 40 000 x 128 (26 MB) 2.56 -> 2.33.
    // Nor, on rows of up to 128 elements, where the queries that a chiplet has at work lie so far apart that its L2 holds
    // little of what they search: their share of the index is the measure, twice the L2, and four times for the short
    // searches (ef <= 128) of rows of more than 64 elements: hand-overs late in a batch, the price of not going longest
    // first, are short there as well.
    // Longest first throughout / by region, means over 5 to 40 draws: 1 M x 96, 100 000 queries, ef 256 (4.6 MB) 9.64 /
    // 9.03 ms; 500 000 x 128, 60 000, ef 100 (4.8 MB) 5.56 / 4.87; 1.18 M x 50, ef 300, 100 000 (4 MB) 8.27 / 8.29, 40 000
    // (10 MB) 3.93 / 3.90, 4.04 / 4.16 and 4.11 / 4.00; 1.18 M x 80, ef 300, 25 000 (22 MB) 3.42 / 3.56; 2 M x 96, 22 000, ef 256
    // (41 MB) 3.42 / 3.72; 10 M x 96, ef 256, 100 000 (46 MB) 13.6 / 14.9, 30 000 (153 MB) 5.21 / 5.83; at ef 128 50 000 on
    // 1 M x 96 (9 MB) 4.47 / 4.15, 100 000 on 3 M x 96 (14 MB) 8.89 / 8.50, but 30 000 there (46 MB) 3.36 / 3.42, and 40 000 on
    // 1.18 M x 50 (11 MB) 2.48 / 2.49, at ef 64 1.62 / 1.64.  Longer rows gain however far apart: 1 M x 960, 8 000, ef 300 (135 MB) 11.2 / 10.6.
    constexpr size_t kRegionIndexFrom = (size_t)12 << 20;
    constexpr size_t kRegionAtWork = (size_t)(NS == 2 && QR == 2 ? 16 : 8) << 20;
    const size_t index_bytes = (size_t)host.N * ((size_t)Dp * (storage_half ? 2 : 4) + (size_t)host.S0 * 4);
    const bool near_by = !(QR == 1 || QR == 2) || (double)index_bytes * resident <= (double)kRegionAtWork * kShares * a.nq;
    const bool by_region = query_order == 2 || (query_order == 1 && index_bytes > kRegionIndexFrom && near_by);
    int region_level = 0;
    if (in_order && !keep_trails && a.nq >= 3 * resident && by_region) {
      // (a level has this share of the nodes of the one below it: so many upper rows are there for so many nodes)
      const double share = (double)host.upper_rows / ((double)host.upper_rows + host.N);
      double nodes = host.N;
      for (int level = 1; level <= host.maxlevel && region_level == 0; ++level) {
        nodes *= share;
        if (a.nq >= 4.0 * nodes) region_level = level;
      }
    }
    if (in_order) {
      d_entry.reserve((size_t)a.nq);
      d_order.reserve((size_t)a.nq * (region_level > 0 ? 2 : 1));
      d_order_hist.reserve(kOrderWords);
    }
    if (keep_trails) {
      d_redo_trail.reserve((size_t)a.nq);
      a.trail = d_trail.p;
      a.trail_cap = trail_cap;
      a.trail_first_spare = slots;
      a.trail_spares = trail_spares;
      a.trail_next = d_ctl.p + 48;
      a.redo_trail = d_redo_trail.p;
    }
    a.waiting = side_slots;
    a.report = side ? nullptr : h_ctl;  // (beside a literal pass the host needs that pass's status as well)
    if (alone) {
      // control words of its own, cleared with those of the next searches of this kind (the list is not: nobody polls it)
      int* ctl = next_control_block();
      a.counter = ctl;
      a.repeats = ctl + 32;
      a.done = ctl + 64;
    } else {
      const int n_hist = in_order ? kOrderWords : 0;
      const int n_fill = std::max(std::max(a.nq, n_hist), 128);
      hipLaunchKernelGGL(prepare_search_kernel, dim3((unsigned)((n_fill + 255) / 256)), dim3(256), 0, stream, d_ctl.p, 128,
                         d_redo.p, a.nq, in_order ? d_order_hist.p : nullptr, n_hist);
      HIP_CHECK(hipGetLastError());
    }
    if (side) {
      SearchArgs b = a;
      b.live = 1;
      b.entry = in_order ? d_entry.p : nullptr;  // (a query reaches that pass after the batch's descents are done)
      b.counter = d_ctl.p + 96;
      b.pool = pool;
      // one or two of these wavefronts per CU: LDS for a candidate queue that never spills costs the first
      // pass nothing (the queue of a long search outgrows 2 * ef entries)
      if (NS > 0) b.cand_lds = std::max(a.cand_lds, 1024);
      // (the first pass starts after the batch's descents when its queries are put in order: 0.1 ms per
      // 10 000 queries of the 1.18 M x 50 set; allow ten times that on top of the usual 2 ms)
      b.start_ticks += (long long)wall_clock_khz * (a.nq / 10000 + 1);
      HIP_CHECK(hipEventRecord(ev_side0, stream));
      HIP_CHECK(hipStreamWaitEvent(stream2, ev_side0, 0));
      hipLaunchKernelGGL(kernel, dim3(side_slots), dim3(64), literal_lds(b.cand_lds), stream2, ix, b);
      HIP_CHECK(hipGetLastError());
      HIP_CHECK(hipEventRecord(ev_side1, stream2));
    }
    // more than one round of wavefronts: the batch's descents first, then its queries longest first.  (The
    // literal pass has been launched by now: launched after the first pass it would find no room until the
    // first of that pass's wavefronts leave, a third of the way through the batch.)
    if (in_order) {
      a.entry = d_entry.p;
      a.order = d_order.p;
      a.order_hist = d_order_hist.p;
      int* const cut = d_order_hist.p + 2 * kOrderBuckets + 32 * (kShares + 1);
      if (region_level > 0) {
        a.regions = d_order.p + a.nq;
        a.region_level = region_level;
        a.shares = d_order_hist.p + 2 * kOrderBuckets;
      }
      if constexpr (QR == 1 || QR == 2) {
        // four queries per wavefront, one per group of 16 lanes
        auto k_entry = entry4_kernel<DT, QR>;
        const int groups = std::max(1, (a.nq + 3) / 4);
        // Two rounds of wavefronts are of equal length: a full one and a short one take as long, and the full one's wavefronts are
        // in each other's way.  More than two, of longer L2 rows: four wavefronts on a SIMD instead of the five it holds.
        // Every batch by four wavefronts / this, us: 1 M x 50 dot, 20 000 queries 104 / 101, 24 000 113 / 118, 33 000 161 / 139,
        // 60 000 256 / 240, 100 000 435 / 394; 600 000 x 96 dot 131 / 127, 142 / 140 (a full and a short round: 155), 202 / 179,
        // 314 / 298, 528 / 490; 300 000 x 128 L2 135 / 127, 147 / 137, 178 / 178, 285 / 285 (five wavefronts: 294), 454 / 454 (478).
        const int entry_slots = resident_slots(k_entry, 0);
        int entry_grid = groups <= entry_slots ? groups : groups <= 2 * entry_slots ? (groups + 1) / 2 : entry_slots;
        if (DT == DIST_L2 && QR == 2 && groups > 2 * entry_slots) entry_grid = std::min(entry_grid, 4 * 4 * num_cus);
        hipLaunchKernelGGL(k_entry, dim3(entry_grid), dim3(64), 0, stream, ix, a);
      } else {
        auto k_entry = entry_kernel<DT, QR>;
        const size_t entry_lds = plan_fast_lds(QR, ix.Dp, a.rcap, FilterShape(), 0).total;
        const int entry_grid = std::max(1, std::min(a.nq, resident_slots(k_entry, entry_lds)));
        hipLaunchKernelGGL(k_entry, dim3(entry_grid), dim3(64), entry_lds, stream, ix, a);
      }
      HIP_CHECK(hipGetLastError());
      const dim3 per_query((unsigned)((a.nq + 1023) / 1024));
      int* const region_hist = d_order_hist.p + kOrderBuckets;
      hipLaunchKernelGGL(order_prefix_kernel, dim3(1), dim3(1024), 0, stream, d_order_hist.p, std::max(1, a.nq / kLongestOf),
                         a.regions ? cut : nullptr);
      HIP_CHECK(hipGetLastError());
      if (a.regions) {
        hipLaunchKernelGGL(region_count_kernel, per_query, dim3(1024), 0, stream, d_entry.p, a.regions, a.nq, cut, region_hist);
        HIP_CHECK(hipGetLastError());
        hipLaunchKernelGGL(region_prefix_kernel, dim3(1), dim3(1024), 0, stream, region_hist, cut);
        HIP_CHECK(hipGetLastError());
      }
      hipLaunchKernelGGL(order_scatter_kernel, per_query, dim3(1024), 0, stream, d_entry.p, a.regions, cut, a.nq, d_order_hist.p, region_hist,
                         d_order.p);
      HIP_CHECK(hipGetLastError());
    }
    if (alone) {
      if (!launch_teams(search_fast_kernel<DT, QR, NS, false, true, true>, QR, NS, fast_lds, ix, a))
        hipLaunchKernelGGL((search_fast_kernel<DT, QR, NS, false, true>), dim3(slots), dim3(64), fast_lds_bytes, stream, ix, a);
    } else if constexpr (QR == 1 || QR == 2) {
      if (keep_trails) hipLaunchKernelGGL((search_fast_kernel<DT, QR, NS, true>), dim3(slots), dim3(64), fast_lds_bytes, stream, ix, a);
      else hipLaunchKernelGGL(fast_kernel, dim3(slots), dim3(64), fast_lds_bytes, stream, ix, a);
    } else {
      hipLaunchKernelGGL(fast_kernel, dim3(slots), dim3(64), fast_lds_bytes, stream, ix, a);
    }
    HIP_CHECK(hipGetLastError());
    if (side) {
      HIP_CHECK(hipStreamWaitEvent(stream, ev_side1, 0));
    }
    if (ms) HIP_CHECK(hipEventRecord(ev1, stream));  // (recorded again further down if the list has to be answered after all)
    timed = true;
    int* ctl = h_ctl;  // pinned
    if (side) HIP_CHECK(hipMemcpyAsync(ctl, d_ctl.p, 49 * sizeof(int), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    n_literal = last_repeats = side ? ctl[32] : ctl[0];
    last_trails = side ? ctl[48] : ctl[1];
    if (!side && sequential_left > 0) --sequential_left;
    learn_share(a.nq, n_literal);
    if (side) {
      answered = ctl[1] == 0;
      if (!answered) {
        scrub_pool();
        if (ctl[1] & 1) glob_cap *= 4;
        // the wait ran out: the streams of this process do not run side by side at present (a profiler
        // collecting counters, a saturated device); the next searches run one pass after the other
        if (ctl[1] & 2) {
          sequential_left = kSequentialSearches;
          ++literal_fallbacks;
        }
      }
    }
  }
  if (n_literal > 0 && !answered) {
    timed = false;
    SearchArgs b = a;
    b.nq = n_literal;
    const size_t lds = literal_lds(a.cand_lds);
    const int lit_slots = max_slots_override > 0 ? max_slots_override : resident_slots(kernel, lds);
    int slots = std::max(1, std::min(lit_slots, b.nq));
    bool done = false;
    for (int attempt = 0; attempt < 8 && !done; ++attempt) {
      ensure_pool(slots, glob_cap, 2 * glob_cap);
      b.pool = pool;
      b.counter = d_ctl.p;
      b.status = d_ctl.p + 1;
      HIP_CHECK(hipMemsetAsync(d_ctl.p, 0, 3 * sizeof(int), stream));
      hipLaunchKernelGGL(kernel, dim3(slots), dim3(64), lds, stream, ix, b);
      HIP_CHECK(hipGetLastError());
      int ctl[2];
      HIP_CHECK(hipMemcpyAsync(ctl, d_ctl.p, sizeof(ctl), hipMemcpyDeviceToHost, stream));
      HIP_CHECK(hipStreamSynchronize(stream));
      done = ctl[1] == 0;
      if (!done) {
        scrub_pool();
        glob_cap *= 4;  // a candidate queue or accept log overflowed its global area: retry with more room
      }
    }
    if (!done) throw std::runtime_error("search: candidate queue overflow");
  }
  if (!timed && ms) {
    HIP_CHECK(hipEventRecord(ev1, stream));
    HIP_CHECK(hipEventSynchronize(ev1));
  }
  if (ms) HIP_CHECK(hipEventElapsedTime(ms, ev0, ev1));
}
// The search of the entry point that allocates nothing: the sorted-set pass over every query, then the
// literal pass over the list it left, one after the other on the engine's stream.  The length of the
// list stays on the device (the literal kernel reads it there), so nothing is read back in between;
// control words, list and the literal wavefronts' queue overflow and log areas live in this device's
// copy of the static scratch array.  No hipMalloc, no hipFree, no memset: a fill kernel clears the
// control words, the list needs no clearing (the pass after reads only the entries the count vouches
// for).  Calls that overlap on one GPU would share the array and race.
template <int DT, int QR, int NS>
void Engine::launch_search_static(const DevIndex& ix, SearchArgs& a, float* ms) {
  if constexpr (NS > 0) {
    StaticScratchLease lease(device_ordinal);  // released on every way out of this function
    StaticScratch* sc = static_scratch;
    a.counter = sc->ctl;
    a.status = sc->ctl + 1;
    a.repeats = sc->ctl + 32;
    a.done = sc->ctl + 64;
    a.redo = sc->redo;
    a.fast_path = 2;
    a.lean = a.fc;  // literal searches keep the LDS filter and the sorted set with ids: no bitmap in HBM
    auto kernel = search_kernel<DT, QR, NS>;
    auto fast_kernel = search_fast_kernel<DT, QR, NS, false>;
    a.fc = fit_filter(fast_kernel, a.fc, [&](FilterShape f) { return plan_fast_lds(QR, ix.Dp, a.rcap, f, a.k).total; });
    const FastLdsPlan fp = plan_fast_lds(QR, ix.Dp, a.rcap, a.fc, a.k);
    const LdsPlan lp = plan_lds(QR, ix.Dp, -1, a.cand_lds, a.lcap, 0, 0, 0, FilterShape(), a.lean);
    const int slots = std::max(1, std::min(resident_slots(fast_kernel, fp.total), a.nq));
    const int lit_slots = std::max(1, std::min(std::min(resident_slots(kernel, lp.total), kStaticSlots), a.nq));
    if (ms) HIP_CHECK(hipEventRecord(ev0, stream));
    hipLaunchKernelGGL(fill_ints_kernel, dim3(1), dim3(128), 0, stream, sc->ctl, 128, 0);
    HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(fast_kernel, dim3(slots), dim3(64), fp.total, stream, ix, a);
    HIP_CHECK(hipGetLastError());
    SearchArgs b = a;
    b.nq = 0;
    b.nq_dev = sc->ctl + 32;
    b.counter = sc->ctl + 96;
    b.pool = SlotPool{};
    b.pool.cand_glob = sc->cand_glob;
    b.pool.cand_glob_cap = kStaticGlobCap;
    b.pool.log = sc->log;
    b.pool.log_cap = kStaticLogCap;
    hipLaunchKernelGGL(kernel, dim3(lit_slots), dim3(64), lp.total, stream, ix, b);
    HIP_CHECK(hipGetLastError());
    if (ms) HIP_CHECK(hipEventRecord(ev1, stream));
    HIP_CHECK(hipMemcpyAsync(h_ctl, sc->ctl, 33 * sizeof(int), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    last_repeats = h_ctl[32];
    if (ms) HIP_CHECK(hipEventElapsedTime(ms, ev0, ev1));
    if (h_ctl[1] != 0)
      throw std::runtime_error("search_knn (no allocation): a literal search outgrew its share of the static scratch "
                               "(candidate queue or accept log); use cuhnsw_search_knn_device for this batch");
  } else {
    (void)ix; (void)a; (void)ms;
    throw std::runtime_error("search_knn (no allocation): ef_search beyond the sorted set's capacity");
  }
}

template <int DT, int QR>
void Engine::launch_search_ns(int ns, const DevIndex& ix, SearchArgs& a, float* ms) {
  switch (ns) {
    case 2: launch_search<DT, QR, 2>(ix, a, search_slots, ms); break;
    case 3: launch_search<DT, QR, 3>(ix, a, search_slots, ms); break;
    case 4: launch_search<DT, QR, 4>(ix, a, search_slots, ms); break;
    case 5: launch_search<DT, QR, 5>(ix, a, search_slots, ms); break;
    case 6: launch_search<DT, QR, 6>(ix, a, search_slots, ms); break;
    case 7: launch_search<DT, QR, 7>(ix, a, search_slots, ms); break;
    case 8: launch_search<DT, QR, 8>(ix, a, search_slots, ms); break;
    case 16: launch_search<DT, QR, 16>(ix, a, search_slots, ms); break;
    default: launch_search<DT, QR, 0>(ix, a, search_slots, ms); break;
  }
}

// ---- build ---------------------------------------------------------------------------------
template <int DT, int QR, int NS>
void Engine::build_levels() {
  const int N = host.N;
  const int cap_in = 32;
  const int bmax = build_batch > 0 ? build_batch : std::min(std::max(N, 1), 65536);
  const int m_max = std::max(host.max_m, host.max_m0);
  const size_t up_rows = std::max<size_t>((size_t)host.upper_rows, 1);
  // Batches: the nodes go in by ascending id, batch_at(in) of them at a time (below).
  auto batch_at = [&](int in) {
    if (build_batch > 0) return std::max(1, std::min(build_batch, in / 4));
    return std::max(1, std::min(in / 4, std::max(16384, std::min(65536, in / 32))));
  };
  int n_batches = 0;
  for (int p0 = 0; p0 < N; p0 += batch_at(p0)) ++n_batches;
  // All of it is carved from the engine's workspace, which the next build (or a save) finds allocated: taking and giving
  // back half a gigabyte is 4 ms of a build of a million nodes and 0.9 of the 7.7 ms of one of twenty thousand.
  workspace.begin();
  auto p_dists0 = workspace.part<float>((size_t)N * host.S0);
  auto p_distsU = workspace.part<float>(up_rows * host.SU);
  // a batch node posts at most max_m0 links on level 0 and max_m on each upper level
  auto p_dirty = workspace.part<unsigned long long>((size_t)bmax * ((size_t)host.max_m0 + (size_t)std::max(host.maxlevel, 1) * host.max_m));
  auto p_inbox0 = workspace.part<HeapEnt>((size_t)N * cap_in);
  auto p_inboxU = workspace.part<HeapEnt>(up_rows * cap_in);
  auto p_upper = workspace.part<int>((size_t)N);
  auto p_work = workspace.part<unsigned long long>(10);
  // (from here on: cleared below, in one go)
  auto p_inbox0_cnt = workspace.part<int>((size_t)N);
  auto p_inboxU_cnt = workspace.part<int>(up_rows);
  auto p_selected = workspace.part<unsigned char>((size_t)N + up_rows);  // per link row: the row is an output of the selection rule (kernels.h, BuildArgs)
  // work counter and number of touched rows of each batch, which all wavefronts of its search ask for all the time: in one
  // memory line they wait for each other (300 000 x 8 indexed 17.4 -> 19.6 ms, x 30 22.3 -> 23.8, 1 183 514 x 50 from array
  // to file 125.6 -> 128.1)
  auto p_batch_ctl = workspace.part<int>((size_t)n_batches);
  auto p_dirty_cnt = workspace.part<int>((size_t)n_batches);
  workspace.reserve();
  HIP_CHECK(hipMemsetAsync(workspace.at(p_inbox0_cnt), 0, workspace.bytes_from(p_inbox0_cnt), stream));
  HIP_CHECK(hipMemsetAsync(workspace.at(p_work), 0, 10 * sizeof(unsigned long long), stream));
  HIP_CHECK(hipMemsetAsync(d_links0.p, 0xFF, (size_t)N * host.S0 * 4, stream));
  if (host.upper_rows > 0) HIP_CHECK(hipMemsetAsync(d_linksU.p, 0xFF, (size_t)host.upper_rows * host.SU * 4, stream));

  DevIndex ix = dev_index(workspace.at(p_dists0), workspace.at(p_distsU));
  auto k_search = build_search_kernel<DT, QR, NS>;
  auto k_reverse = reverse_kernel<DT, QR>;
  const int efc = opt.ef_construction;
  const int glob_cap = std::max(4096, 8 * efc);

  BuildArgs a{};
  a.efc = efc;
  // (the reference multiplies in single precision: `const int nn_num = max_m * heuristic_coef` with a
  // float coefficient, cpp/include/cuda_build_kernels.cuh:77,101)
  a.nn_num0 = (int)((float)host.max_m0 * (float)opt.heuristic_coef);
  a.nn_numU = (int)((float)host.max_m * (float)opt.heuristic_coef);
  a.save_remains = opt.save_remains ? 1 : 0;
  a.reverse = opt.reverse_cand ? 1 : 0;
  a.own_cap0 = own_links0 > 0 ? std::min(own_links0, host.max_m0) : host.max_m0;
  a.status = d_ctl.p + 1;
  a.inbox0 = workspace.at(p_inbox0); a.inbox0_cnt = workspace.at(p_inbox0_cnt);
  a.inboxU = workspace.at(p_inboxU); a.inboxU_cnt = workspace.at(p_inboxU_cnt);
  a.cap_in = cap_in;
  a.dirty = workspace.at(p_dirty);
  a.dropped = d_ctl.p + 3;
  a.selected0 = newcomer_shortcut ? workspace.at(p_selected) : nullptr;
  a.selectedU = newcomer_shortcut ? workspace.at(p_selected) + N : nullptr;
  a.counters = count_build_work ? workspace.at(p_work) : nullptr;
  const int s_max = std::max(host.S0, host.SU);
  a.lcap = (std::max(s_max, 64) + 63) / 64 * 64;
  size_t fixed = (size_t)a.lcap * 8 + (size_t)efc * 8 + (size_t)m_max * 8 + 64 +
                 (QR == 0 ? (size_t)query_lds_chunks(Dp) * 16 : 0);
  a.fc = NS > 0 ? least_filter(efc) : FilterShape();
  const bool sorted_set = NS > 0 && a.fc.sets() > 0;  // then neither queue nor literal cache is needed
  if (a.reverse && NS > 0 && !sorted_set) throw std::runtime_error("build_graph: reverse_cand needs fewer than 2^28 points");
  a.cand_lds = sorted_set ? 0 : auto_cand_lds(efc, NS, 64, fixed);
  a.vc_bits = sorted_set ? 0 : auto_vc_bits();
  auto search_lds = [&](FilterShape f) { return plan_lds(QR, Dp, sorted_set ? -1 : efc, a.cand_lds, a.lcap, efc, m_max, a.vc_bits, f).total; };
  a.fc = fit_filter(k_search, a.fc, search_lds);
  const size_t lds1 = search_lds(a.fc);
  const LdsPlan lp3 = plan_lds(QR, Dp, s_max + cap_in, 0, a.lcap, s_max + cap_in, std::max(m_max, cap_in));
  const int slots1 = resident_slots(k_search, lds1);
  last_team_batches = 0;
  // Batches that leave the machine idle: a workgroup of wavefronts per node (kernels.h, TEAM), eight or four as in launch_teams.
  // (A batch of 58 / 222 / 543 nodes of 20 000 x 50: 126 -> 88 us, 203 -> 128, 220 -> 183; the 44 batches 6.70 -> 5.81 ms, 20 003 x 128
  // 12.6 -> 10.9, 8 000 x 300 12.2 -> 10.8, 6 000 x 960 15.8 -> 14.2, 100 000 x 50 13.0 -> 12.3.)
  auto k_team = build_search_kernel<DT, QR, (NS > 0 ? NS : 2), true>;
  const bool teams = NS > 0 && sorted_set && !a.reverse && s_max <= 64 && filter_entries <= 0;
  auto launch_team = [&](BuildArgs b) {
    if (!teams || b.count > 4 * num_cus) return false;
    const int per_cu = (b.count + num_cus - 1) / num_cus;
    const size_t room = (size_t)160 * 1024 / per_cu / kLdsStep * kLdsStep - 64;  // (the kernel has 64 bytes of its own)
    const FilterShape least = least_filter(efc);
    b.fc = filter_shape(std::min(8 * least.sets(), 4096), N);
    b.team_turn = num_cus;
    b.team_bucket_bits = 5;
    auto bytes = [&] { return search_lds(b.fc) + (size_t)Team::words(NS, b.team_bucket_bits, s_max) * 4; };
    while (b.fc.sets() > 2 * least.sets() && bytes() > room) b.fc = filter_shape(b.fc.sets() / 2, N);
    while (b.team_bucket_bits > 3 && bytes() > room) --b.team_bucket_bits;
    if (bytes() > room) return false;
    for (int waves = kMostTeam; waves >= kMostTeam / 2; waves /= 2) {
      if (resident_slots(k_team, bytes(), waves) < per_cu * num_cus) continue;
      hipLaunchKernelGGL(k_team, dim3(b.count + b.n_upper), dim3(64 * waves), bytes(), stream, ix, b);
      last_team_batches += 1;
      return true;
    }
    return false;
  };
  const int slots3 = resident_slots(k_reverse, lp3.total);
  // the sorted-set search needs no per-wavefront global memory (no bitmap, no undo list, no log)
  if (!sorted_set) ensure_pool(slots1, glob_cap, 2 * glob_cap);
  a.pool = pool;

  // Nodes go in by ascending id, as hnswlib inserts them.  The graph a batch sees is the
  // one of all earlier batches: its entry point is the first node that reached the highest
  // level so far.  Batches grow with the graph — a quarter of what is already in, up to 16 384 nodes, so
  // that early nodes, which wire the long-range links, see each other; beyond half a million nodes a
  // thirty-second of the graph, up to 65 536 — because the nodes of a batch do not see each other (recall
  // falls when the share of new nodes grows), and a launch of several rounds of wavefronts loses less to
  // its last, partly filled round.
  // build_batch > 0 replaces the two caps by one.
  // Within a batch the nodes with upper levels are handed out first (highest level first, then by id).
  std::vector<int> upper, upper_end;
  if (level_first) {
    upper.reserve((size_t)host.upper_rows);
    upper_end.reserve((size_t)n_batches);
    std::vector<int> mine;
    for (int p0 = 0; p0 < N;) {
      const int b = std::min(batch_at(p0), N - p0);
      mine.clear();
      int top = 0;
      for (int i = 0; i < b; ++i)
        if (host.levels[p0 + i] > 0) {
          mine.push_back(i);
          top = std::max(top, host.levels[p0 + i]);
        }
      for (int lv = top; lv > 0; --lv)
        for (const int i : mine)
          if (host.levels[p0 + i] == lv) upper.push_back(i);
      upper_end.push_back((int)upper.size());
      p0 += b;
    }
    if (!upper.empty())
      HIP_CHECK(hipMemcpyAsync(workspace.at(p_upper), upper.data(), upper.size() * sizeof(int), hipMemcpyHostToDevice, stream));
  }
  int cur_ep = 0, cur_max = -1;
  int pos = 0, batch = 0;
  while (pos < N) {
    int b = batch_at(pos);
    b = std::min(b, N - pos);
    a.begin = pos;
    a.count = b;
    a.cur_ep = cur_ep;
    a.cur_max = cur_max;
    a.counter = workspace.at(p_batch_ctl) + batch;
    a.dirty_cnt = workspace.at(p_dirty_cnt) + batch;
    if (level_first) {
      const int from = batch > 0 ? upper_end[batch - 1] : 0;
      a.upper = workspace.at(p_upper) + from;
      a.n_upper = upper_end[batch] - from;
    }
    ++batch;
    if (!launch_team(a)) hipLaunchKernelGGL(k_search, dim3(std::min(b, slots1)), dim3(64), lds1, stream, ix, a);
    HIP_CHECK(hipGetLastError());
    if (cur_max >= 0) {
      long long work = (long long)b * m_max;
      hipLaunchKernelGGL(k_reverse, dim3((unsigned)std::min<long long>(work, slots3)), dim3(64), lp3.total, stream, ix, a);
      HIP_CHECK(hipGetLastError());
    }
    for (int i = pos; i < pos + b; ++i)
      if (host.levels[i] > cur_max) {
        cur_max = host.levels[i];
        cur_ep = i;
      }
    pos += b;
  }
  int ctl[4];
  HIP_CHECK(hipMemcpyAsync(ctl, d_ctl.p, sizeof(ctl), hipMemcpyDeviceToHost, stream));
  HIP_CHECK(hipStreamSynchronize(stream));
  if (ctl[1] != 0) {
    scrub_pool();
    throw std::runtime_error("build_graph: candidate queue overflow");
  }
  last_build_dropped = ctl[3];
  std::memset(build_counters, 0, sizeof(build_counters));
  if (count_build_work) {
    HIP_CHECK(hipMemcpyAsync(build_counters, workspace.at(p_work), sizeof(build_counters), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
  }
  if (keep_link_keys) {
    // debugging aid: the key stored with every level-0 link, for a validator to recompute
    std::vector<float> strided((size_t)N * host.S0);
    HIP_CHECK(hipMemcpyAsync(strided.data(), workspace.at(p_dists0), strided.size() * 4, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    link_keys0.assign((size_t)N * host.max_m0, 0.f);
    for (int i = 0; i < N; ++i)
      std::memcpy(&link_keys0[(size_t)i * host.max_m0], &strided[(size_t)i * host.S0], (size_t)host.max_m0 * 4);
  }
}

template <int DT, int QR>
void Engine::build_ns(int ns) {
  switch (ns) {
    case 2: build_levels<DT, QR, 2>(); break;
    case 3: build_levels<DT, QR, 3>(); break;
    case 4: build_levels<DT, QR, 4>(); break;
    case 5: build_levels<DT, QR, 5>(); break;
    case 6: build_levels<DT, QR, 6>(); break;
    case 7: build_levels<DT, QR, 7>(); break;
    case 8: build_levels<DT, QR, 8>(); break;
    case 16: build_levels<DT, QR, 16>(); break;
    default: build_levels<DT, QR, 0>(); break;
  }
}

#if CUHNSW_PART == 0
template void Engine::launch_search_ns<CUHNSW_DT, CUHNSW_QR>(int, const DevIndex&, SearchArgs&, float*);
#else
template void Engine::build_ns<CUHNSW_DT, CUHNSW_QR>(int);
#endif

}  // namespace cuhnsw_amd
