// Host engine of libcuhnsw_amd.so: options, data, index files and what surrounds the kernel launches.  (The C ABI is
// in engine.hip, the launches of the templated kernels are in instances.hip.)
//
// Counterpart of the reference's host class cuhnsw::CuHNSW
// (cpp/include/cuhnsw.hpp:61-112, cpp/src/cuhnsw_base.cu, cpp/src/cuhnsw_build.cu).
// Differences by design: the whole multi-level index stays resident in HBM in flat
// fixed-stride rows (the reference re-flattens and re-uploads the graph on every
// search call, cpp/src/cuhnsw_build.cu:226-253, and once per upper level for the
// descent, :25-94); there is no per-level host graph container; HIP runtime calls
// are made directly (no Thrust).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "host_staging.h"
#include "index_file.h"
#include "kernels.h"
#include "options.h"

namespace cuhnsw_amd {

inline bool device_present() {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return n > 0;
}

// ---- scratch of the entry point that allocates nothing (cuhnsw_search_knn_device_noalloc) ----------
// Everything the two search kernels need beyond the caller's buffers, at fixed maximum sizes, in one
// array that lives in the code object: each GPU the library runs on holds its own copy from the moment
// the code object is loaded there until the process ends.  Host code never uses the array's name as an
// address (it is a host-side stand-in); the device address is looked up once per device
// (static_scratch_for_current_device) and handed to the kernels like any other buffer.
constexpr int kStaticMaxQueries = 131072;  // entries of the list of queries the first pass gives up
constexpr int kStaticMaxEf = 512;          // the sorted set in registers holds up to 512 entries
constexpr int kStaticSlots = 128;          // wavefronts of the literal pass
constexpr int kStaticGlobCap = 4096;       // per wavefront: overflow of its candidate queue beyond the LDS share
constexpr int kStaticLogCap = 8192;        // per wavefront: log of accepted entries
struct StaticScratch {
  int ctl[128];
  int redo[kStaticMaxQueries];
  HeapEnt cand_glob[(size_t)kStaticSlots * kStaticGlobCap];
  HeapEnt log[(size_t)kStaticSlots * kStaticLogCap];
};
constexpr int kMaxDevices = 64;
extern std::atomic_flag g_static_busy[kMaxDevices];  // set while a no-allocation search uses the device's array
// device address of this device's copy of the array; looked up on first use, then kept
StaticScratch* static_scratch_for_current_device(int* device = nullptr);
// One no-allocation search at a time per GPU: every engine of the process shares that GPU's array.
struct StaticScratchLease {
  int dev;
  explicit StaticScratchLease(int d) : dev(d) {
    if (g_static_busy[dev].test_and_set(std::memory_order_acquire))
      throw std::runtime_error("search_knn (no allocation): another no-allocation search is running on this GPU "
                               "(all engines of a process share the GPU's scratch array; serialise the calls)");
  }
  ~StaticScratchLease() { g_static_busy[dev].clear(std::memory_order_release); }
  StaticScratchLease(const StaticScratchLease&) = delete;
  StaticScratchLease& operator=(const StaticScratchLease&) = delete;
};

template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  // grows (never shrinks); contents are not preserved
  void reserve(size_t want) {
    if (want <= n) return;
    release();
    HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&p), want * sizeof(T)));
    n = want;
  }
  // the same for a buffer the caller can do without: false (and an empty buffer) when the memory is not there
  bool try_reserve(size_t want) {
    if (want <= n) return true;
    release();
    if (hipMalloc(reinterpret_cast<void**>(&p), want * sizeof(T)) != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      return false;
    }
    n = want;
    return true;
  }
  ~DevBuf() { release(); }
};

// Device memory that a build, a save or a load needs while it runs, in one allocation that the engine keeps for the next
// of them: parts are asked for one after the other, reserve() makes room for all of them.
class Workspace {
 public:
  template <typename T>
  struct Part {
    size_t offset;
  };
  void begin() { used_ = 0; }
  template <typename T>
  Part<T> part(size_t n) {
    const Part<T> p{used_};
    used_ += (n * sizeof(T) + 255) & ~(size_t)255;
    return p;
  }
  void reserve() { memory_.reserve(std::max<size_t>(used_, 256)); }
  template <typename T>
  T* at(Part<T> p) const {
    return reinterpret_cast<T*>(memory_.p + p.offset);
  }
  template <typename T>
  size_t bytes_from(Part<T> p) const {
    return used_ - p.offset;
  }
  // The call that needed it is over: what the next one may use stays.  (More than kKept does not: the largest builds need
  // a tenth of the GPU's memory, which a search may want.  Nor does what goes beyond the process's bound, nor anything
  // with keep = false.)
  void end(bool keep) {
    if (keep && memory_.n == counted_) return;
    kept_device_memory.give_back(counted_);
    counted_ = 0;
    if (keep && memory_.n <= kKept && kept_device_memory.take(memory_.n)) counted_ = memory_.n;
    else memory_.release();
  }
  ~Workspace() { kept_device_memory.give_back(counted_); }

 private:
  static constexpr size_t kKept = (size_t)2 << 30;
  DevBuf<unsigned char> memory_;
  size_t used_ = 0;
  size_t counted_ = 0;  // bytes of it that count as kept
};

class Engine {
 public:
  Options opt;
  int dist_type = DIST_DOT;
  HostIndex host;
  bool have_data = false, have_levels = false, have_graph = false;
  bool has_device = false;
  int num_cus = 0;
  hipStream_t stream = nullptr;
  hipStream_t stream2 = nullptr;  // the literal pass, while the sorted-set pass runs on `stream`
  hipEvent_t ev_side0 = nullptr, ev_side1 = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::string err;
  double last_build_seconds = 0.0;

  // tunables
  int level_first = 1;     // build: a batch hands out its nodes with upper levels first
  int build_literal = 0;   // build: 1 = the literal search (queues / sorted list in LDS) whatever ef_construction (tests)
  int build_batch = 0;     // nodes inserted per batch at most; 0 = by the size of the graph (batch_at)
  int search_slots = 0;
  int cand_lds_override = 0;
  int hnswlib_dist = 0;
  int spin_limit_override = -1;  // polls a waiting literal wavefront may spend (-1 = automatic)
  static constexpr int kLiteralStreak = 15;  // batches that go to the literal queues alone before one asks the first pass again
  int literal_streak = 0;
  // the share of queries given up over the last few searches, cautiously: as if 750 more had been answered without (two of
  // a thousand may be an accident)
  double recent_queries = 0.0, recent_repeats = 0.0;
  double cautious_share() const { return recent_repeats / (recent_queries + 750.0); }
  int side_per_cu = 0;         // its wavefronts per CU (0 = from the share of queries the last search gave up)
  bool share_known = false;               // repeat_share comes from searches of this index
  double repeat_share = 0.0;              // share of the last queries (256 or more, once there are so many) that were given up
  long long share_queries = 0, share_repeats = 0;  // the batches too small to judge by, taken together
  int concurrent_literal = 1;  // run the literal pass beside the sorted-set pass (0: after it)
  // A literal wavefront whose bounded wait ran out (the two streams did not run side by side: a profiler that
  // serialises kernels, a saturated device) makes the next kSequentialSearches searches run their passes one
  // after the other; then the concurrent schedule is tried again.  The caller's setting above is left alone.
  static constexpr int kSequentialSearches = 8;
  int sequential_left = 0;       // searches still to run one pass after the other
  int literal_fallbacks = 0;     // how often that happened on this index
  int last_side_by_side = 0;     // the last search ran its literal pass beside the first pass
  int last_team = 0;             // wavefronts that searched each of its queries together (launch_teams); 0 = one alone
  int last_team_batches = 0;     // batches of the last build whose nodes were searched so
  bool trails_unavailable = false;  // the trail buffers could not be allocated: searches go on without trails
  int filter_entries = 0;  // entries of the sorted-set search's visited filter (0 = automatic)
  int first_pass_waves = 0;  // wavefronts per CU of the first pass (0 = as many as fit)
  int query_order = 1;     // first pass of 1.5 to 32 rounds of wavefronts: longest queries first, those of large batches by
                           // region (3: not those; 2: both whatever the sizes; 0: caller's order)
  bool fast_suspended = false;  // this index ties too often for the sorted-set search to pay (integer data)
  int lean_literal = 1;  // literal pass: 0 = always the exact visited bitmap, 1 = automatic, 2 = always the LDS filter
  bool storage_half = false;  // vectors live in HBM as fp16 (set before set_data / load_index)
  bool tight_rows = false;    // rows padded to 16-byte chunks only, not to 128-byte lines (set before set_data / load_index)
  int fast_path = 1;     // 0: search with the literal queues only; 1: sorted-set pass first, unless the index is known
                         // to hand over too many of such a batch's queries; 2: always
  int last_repeats = 0;  // queries of the last search that were repeated with the literal queues
  int last_trails = 0;   // how many of them came with the first pass's trail
  int count_build_work = 0;    // count the work of a build on the device (cuhnsw_last_build_counters)
  unsigned long long build_counters[10] = {};
  int last_build_dropped = 0;  // reverse links of the last build that found no room in an inbox
  int keep_link_keys = 0;      // keep the keys stored with the level-0 links after a build (debugging aid)
  std::vector<float> link_keys0;  // N x max_m0, only with keep_link_keys
  int newcomer_shortcut = 1;  // build: a link row that the selection rule produced is re-selected with the shortcut for newcomers
  int own_links0 = 0;  // links a new node selects for itself on level 0: 0 = max_m0 (as the reference), else min(value, max_m0); hnswlib uses max_m
  int spill_cap = 0;  // first size of the per-slot queue overflow area (0 = automatic); the accept log is twice that
  int visited_cache = 0;  // entries of the LDS visited cache: 0 = automatic, < 0 = none

  // resident index
  int Dp = 0;
  DevBuf<float> d_vectors;
  DevBuf<uint64_t> d_labels;
  DevBuf<uint32_t> d_deleted;  // one bit per element: hnswlib's delete marks of a loaded file (used while host.n_deleted > 0)
  DevBuf<uint32_t> d_links0, d_linksU;
  DevBuf<int64_t> d_upper_off;
  DevBuf<int> d_levels;
  // per-wavefront slots
  DevBuf<uint32_t> d_bitmaps, d_undo;
  DevBuf<HeapEnt> d_cand_glob, d_log;
  SlotPool pool{};
  int pool_slots = 0;
  DevBuf<int> d_ctl;  // [0] work counter, [1] status, [2] dirty count, [32] queries given up by the
                      // sorted-set pass, [64] queries it has finished with, [96] work counter of a concurrent literal pass
  DevBuf<int> d_redo;  // their indices
  DevBuf<uint4> d_trail;      // trails of the sorted-set pass: one buffer per wavefront and the spares,
  DevBuf<int4> d_redo_trail;  // and which of them goes with which entry of d_redo
  int trails = 1;             // 0 = the literal pass searches every handed-over query from its entry point
  int trail_cap = 2048;       // records (accepted entries) per trail; a search that outgrows it leaves none
  int trail_spares = 1024;    // hand-overs with a trail per batch; the ones after that leave none
  DevBuf<uint4> d_entry;      // longest queries first: level-0 entry of every query of the batch,
  DevBuf<int> d_order_hist;   // bucket counters,
  DevBuf<int> d_order;        // and the order the first pass takes the queries in
  // staging for the host-pointer search entry point
  DevBuf<float> d_q, d_dist;
  DevBuf<int> d_nns, d_found;
  HostStaging staging;
  Workspace workspace;
  int keep_workspace = 1;  // 0: neither stays allocated after the call that needed it
  struct CallEnd {         // (also where the call ends with an exception)
    Engine& e;
    explicit CallEnd(Engine& engine) : e(engine) {}
    ~CallEnd() { e.give_back_workspace(); }
  };
  void give_back_workspace() {
    workspace.end(keep_workspace != 0);
    staging.end(keep_workspace != 0);
  }
  // Pinned memory that small batches are read from and answered into (kernels address it).  How small was measured on
  // searches of next to no work (ef 8, 20 000 rows), through copies -> directly:
  //   queries 128 KB 84 -> 72 us (128 x 256), 256 KB 95 -> 80 us (128 x 512), 125 -> 113 us (960 x 66), 750 KB 261 -> 229 us
  //           (32 x 6 000), 1 MB 171 -> 147 us (960 x 266), 194 -> 177 us (128 x 2 000);
  //   answers 0.1 MB 272 -> 196 us (128 x topk 100), 0.5 MB 285 -> 240 us, 1 MB 450 -> 395 us, 2 MB 532 -> 456 us,
  //           3.9 MB 728 -> 633 us.
  // Beyond, the copies run at the bus's rate while a search's own reads and writes wait for it.
  static constexpr size_t kDirectQueries = (size_t)1 << 20, kDirectAnswers = (size_t)4 << 20;
  static constexpr size_t kQueryBlock = (size_t)1 << 20;
  unsigned char* h_io = nullptr;
  size_t h_io_bytes = 0;
  void reserve_io(size_t bytes) {
    if (bytes <= h_io_bytes) return;
    // (at least doubled: batches that grow by a query at a time do not allocate each time)
    bytes = std::max({bytes, (size_t)64 << 10, std::min(2 * h_io_bytes, kDirectQueries + kDirectAnswers)});
    if (h_io) HIP_CHECK(hipHostFree(h_io));
    h_io = nullptr;
    h_io_bytes = 0;
    HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&h_io), bytes, hipHostMallocDefault));
    h_io_bytes = bytes;
  }
  static constexpr size_t kPiece = (size_t)512 << 20;  // device memory an index file is packed in, piece by piece
  StaticScratch* static_scratch = nullptr;  // this device's copy (device address)
  int device_ordinal = 0;
  int* h_ctl = nullptr;                     // pinned: control words read back without staging
  long long wall_clock_khz = 100000;        // ticks of wall_clock64() per millisecond

  Engine() {
    has_device = device_present();
    if (has_device) {
      int dev = 0;
      HIP_CHECK(hipGetDevice(&dev));
      hipDeviceProp_t prop;
      HIP_CHECK(hipGetDeviceProperties(&prop, dev));
      num_cus = prop.multiProcessorCount;
      int khz = 0;
      if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess && khz > 0) wall_clock_khz = khz;
      else (void)hipGetLastError();
      static_scratch = static_scratch_for_current_device(&device_ordinal);
      HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&h_ctl), 64 * sizeof(int), hipHostMallocDefault));
      HIP_CHECK(hipStreamCreate(&stream));
      HIP_CHECK(hipEventCreate(&ev0));
      HIP_CHECK(hipEventCreate(&ev1));
      d_ctl.reserve(128);
      HIP_CHECK(hipStreamCreate(&stream2));
      HIP_CHECK(hipEventCreate(&ev_side0));
      HIP_CHECK(hipEventCreate(&ev_side1));
    }
  }
  ~Engine() {
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (ev_side0) (void)hipEventDestroy(ev_side0);
    if (ev_side1) (void)hipEventDestroy(ev_side1);
    if (stream2) (void)hipStreamDestroy(stream2);
    if (stream) (void)hipStreamDestroy(stream);
    if (h_ctl) (void)hipHostFree(h_ctl);
    if (h_io) (void)hipHostFree(h_io);
  }

  void need_device() const {
    if (!has_device) throw std::runtime_error("no HIP device available: this call needs a GPU");
  }

  int qr() const { return query_regs(Dp); }

  DevIndex dev_index(float* dists0 = nullptr, float* distsU = nullptr) const {
    DevIndex ix;
    ix.vectors = d_vectors.p;
    ix.labels = host.labelled ? d_labels.p : nullptr;
    ix.links0 = d_links0.p;
    ix.linksU = d_linksU.p;
    ix.upper_off = d_upper_off.p;
    ix.levels = d_levels.p;
    ix.dists0 = dists0;
    ix.distsU = distsU;
    ix.half = storage_half ? 1 : 0;
    ix.N = host.N; ix.D = host.D; ix.Dp = Dp; ix.S0 = host.S0; ix.SU = host.SU;
    ix.max_m = host.max_m; ix.max_m0 = host.max_m0; ix.maxlevel = host.maxlevel;
    ix.enterpoint = host.enterpoint;
    return ix;
  }

  // ---- option / data / level plumbing -------------------------------------------------
  int init(const char* path) {
    Options o;
    int dt = DIST_DOT;
    std::string why;
    int rc = load_options(path ? path : "", o, dt, why);
    if (rc == 0) {
      opt = o;
      dist_type = dt;
    }
    err = why;  // empty after a successful call
    return rc;
  }

  // Between host memory and device memory everything large goes through the pinned blocks of `staging`
  // (host_staging.h), filled and emptied by several threads while the copy engine runs.  Vectors, links and labels live
  // in device memory only; an index file is packed and unpacked there.
  void reserve_vectors() {
    Dp = padded_dims(host.D, tight_rows);
    const size_t n = (size_t)host.N * Dp;
    d_vectors.reserve(storage_half ? (n + 1) / 2 : n);
  }
  // (with fp16 storage the rows are rounded to nearest even on their way into the index: everything downstream,
  // the saved file and a CPU search of that file, then sees exactly the vectors the kernels see)
  void upload_vectors(const float* rows) {
    reserve_vectors();
    const size_t row_bytes = (size_t)host.D * sizeof(float), total = (size_t)host.N * row_bytes;
    const bool plain = Dp == host.D && !storage_half;
    staging.reserve(row_bytes, !plain);
    const size_t block = staging.block() / row_bytes * row_bytes;  // whole rows
    const unsigned char* src = reinterpret_cast<const unsigned char*>(rows);
    unsigned char* dst = reinterpret_cast<unsigned char*>(d_vectors.p);
    staging.send(stream, total, block, [&](unsigned char* to, size_t at, size_t n) { std::memcpy(to, src + at, n); },
                 [&](size_t at, size_t) { return plain ? dst + at : nullptr; },
                 [&](unsigned char* there, size_t at, size_t n) {
                   if (plain) return;
                   const long long first = (long long)(at / row_bytes), count = (long long)(n / row_bytes);
                   const dim3 grid((unsigned)((count * (Dp / 4) + 255) / 256));
                   const float* from = reinterpret_cast<const float*>(there);
                   if (storage_half)
                     hipLaunchKernelGGL(pad_rows_kernel<_Float16>, grid, dim3(256), 0, stream, from,
                                        reinterpret_cast<_Float16*>(d_vectors.p) + first * Dp, count, host.D, Dp);
                   else
                     hipLaunchKernelGGL(pad_rows_kernel<float>, grid, dim3(256), 0, stream, from, d_vectors.p + first * Dp,
                                        count, host.D, Dp);
                   HIP_CHECK(hipGetLastError());
                 });
    HIP_CHECK(hipStreamSynchronize(stream));
  }

  void set_data(const float* data, int n, int d) {
    if (!data || n <= 0 || d <= 0) throw std::runtime_error("set_data: empty data");
    const CallEnd at_end(*this);
    // (a call that fails leaves nothing behind that a later one could mistake for data or a graph)
    have_data = have_levels = have_graph = false;
    host = HostIndex();
    host.N = n;
    host.D = d;
    forget_search_history();
    pool_slots = 0;  // the slot pool is sized by N: rebuild it lazily
    pool = SlotPool{};
    try {
      if (has_device) upload_vectors(data);
      else host.vectors.assign(data, data + (size_t)n * d);  // without a GPU only the host-side calls remain usable
    } catch (...) {
      host = HostIndex();
      throw;
    }
    have_data = true;
  }

  void upload_structure() {
    d_levels.reserve((size_t)host.N);
    d_upper_off.reserve((size_t)host.N);
    d_links0.reserve((size_t)host.N * host.S0);
    d_linksU.reserve(std::max<size_t>((size_t)host.upper_rows * host.SU, 1));
    HIP_CHECK(hipMemcpyAsync(d_levels.p, host.levels.data(), (size_t)host.N * 4, hipMemcpyHostToDevice, stream));
    HIP_CHECK(hipMemcpyAsync(d_upper_off.p, host.upper_off.data(), (size_t)host.N * 8, hipMemcpyHostToDevice, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
  }
  void set_random_levels(const int* levels, int n) {
    if (!have_data) throw std::runtime_error("set_random_levels: call set_data first");
    if (n != host.N) throw std::runtime_error("set_random_levels: length differs from the number of data rows");
    if (std::any_of(levels, levels + n, [](int l) { return l < 0; })) throw std::runtime_error("levels must be non-negative");
    host.max_m = opt.max_m;
    host.max_m0 = opt.max_m0;
    host.M = opt.max_m;
    host.ef_construction = opt.ef_construction;
    host.mult = opt.level_mult;
    have_levels = have_graph = false;
    host.set_levels(levels, n);
    if (has_device) host.layout_upper();
    else host.layout_links();
    host.labelled = false;
    host.labels.clear();
    host.deleted.clear();  // a graph built anew holds every element
    host.n_deleted = 0;
    if (has_device) upload_structure();
    have_levels = true;
  }

  // What a search learns about an index (how many of its queries tie, whether the two passes ran side by
  // side) belongs to that index: forgotten whenever another one takes its place.
  void forget_search_history() {
    fast_suspended = false;
    share_known = false;
    repeat_share = 0.0;
    share_queries = share_repeats = 0;
    literal_streak = 0;
    recent_queries = recent_repeats = 0.0;
    sequential_left = 0;
    literal_fallbacks = 0;
    last_side_by_side = last_team = 0;
    last_repeats = last_trails = 0;
  }

  // An index whose distances tie all the time (integer-valued data) sends most queries through both passes: where more
  // than a third of 256 or more queries were given up the sorted set is tried no more.  Smaller batches are judged
  // together (not where the caller asked for the first pass whatever the batch).
  void learn_share(long long nq, long long given_up) {
    recent_queries = 0.75 * recent_queries + (double)nq;
    recent_repeats = 0.75 * recent_repeats + (double)given_up;
    if (nq < 256 && fast_path == 1) {
      nq = share_queries += nq;
      given_up = share_repeats += given_up;
      if (nq >= 256) share_queries = share_repeats = 0;
    }
    repeat_share = (double)given_up / (double)nq;
    share_known = true;
    if (nq >= 256 && given_up * 3 > nq) fast_suspended = true;
  }
  // control words (as d_ctl) of a search that needs nothing else cleared: cleared kControlBlocks at a time
  static constexpr int kControlBlocks = 64;
  DevBuf<int> d_ctl_blocks;
  int ctl_block = kControlBlocks;
  int* next_control_block() {
    if (ctl_block == kControlBlocks) {
      d_ctl_blocks.reserve((size_t)kControlBlocks * 128);
      HIP_CHECK(hipMemsetAsync(d_ctl_blocks.p, 0, (size_t)kControlBlocks * 128 * sizeof(int), stream));
      ctl_block = 0;
    }
    return d_ctl_blocks.p + (size_t)128 * ctl_block++;
  }

  // Buffers of a search that do not depend on the batch are allocated when the index becomes resident, not
  // inside the first search that wants them: the trails of the sorted-set pass (one buffer per wavefront the
  // GPU can hold plus the spares).  They are an optimisation: if the memory is not there the searches go on
  // without trails.
  size_t trail_records_wanted(int slots) const { return (size_t)(slots + trail_spares) * (size_t)trail_cap; }
  void reserve_trails(int slots) {
    if (!trails || trails_unavailable) return;
    if (!d_trail.try_reserve(trail_records_wanted(slots))) trails_unavailable = true;
  }
  void prepare_search_buffers() {
    if (!has_device) return;
    trails_unavailable = false;
    reserve_trails(28 * num_cus);  // seven wavefronts per SIMD: what the sorted-set pass holds at most where it keeps trails
  }

  // ---- slots -----------------------------------------------------------------------------
  void ensure_pool(int slots, int cand_glob_cap, int log_cap) {
    const int words = (host.N + 31) / 32;
    const int undo_cap = std::min(32768, std::max(host.N, 64));
    if (slots <= pool_slots && words == pool.bitmap_words && cand_glob_cap <= pool.cand_glob_cap &&
        log_cap <= pool.log_cap && undo_cap == pool.undo_cap)
      return;
    slots = std::max(slots, pool_slots);
    cand_glob_cap = std::max(cand_glob_cap, pool.cand_glob_cap);
    log_cap = std::max(log_cap, pool.log_cap);
    d_bitmaps.release();
    d_bitmaps.reserve((size_t)slots * words);
    HIP_CHECK(hipMemsetAsync(d_bitmaps.p, 0, (size_t)slots * words * 4, stream));
    d_undo.reserve((size_t)slots * undo_cap);
    d_cand_glob.reserve((size_t)slots * cand_glob_cap);
    d_log.reserve((size_t)slots * log_cap);
    pool.log = d_log.p;
    pool.log_cap = log_cap;
    pool.bitmaps = d_bitmaps.p;
    pool.bitmap_words = words;
    pool.undo = d_undo.p;
    pool.undo_cap = undo_cap;
    pool.cand_glob = d_cand_glob.p;
    pool.cand_glob_cap = cand_glob_cap;
    pool_slots = slots;
  }
  // a failed kernel may leave bits set: start over with clean bitmaps
  void scrub_pool() {
    HIP_CHECK(hipMemsetAsync(d_bitmaps.p, 0, (size_t)pool_slots * pool.bitmap_words * 4, stream));
  }

  // slots of sorted result keys per lane: as few as hold the result set (an insert costs five instructions a slot), two at
  // least (one for ef <= 64 is 0 to 2 % slower than two), eight for ef <= 512, sixteen beyond; 0 selects the literal LDS heap.
  // (Against 2, 5 and 8 only: 300 000 x 50, 20 000 queries, ef 180 1.66 -> 1.52 ms, ef 250 1.74 -> 1.66, ef 350 3.13 -> 2.64,
  // ef 430 2.87 -> 2.74; 300 000 x 96, 30 000 queries, ef 350 4.64 -> 3.91; 200 003 x 128 indexed at 200 66.6 -> 64.8 ms.)
  static int key_slots(int ef) {
    const int slots = (ef + 63) / 64;
    return slots <= 8 ? std::max(slots, 2) : (ef < 1024 ? 16 : 0);
  }

  // LDS entries of the candidate queue.  With the result keys in registers the queue is the
  // only large LDS user: 2*ef entries hold it in nearly every query (the rest spills to the
  // slot's global area) and keep ~30 wavefronts per CU resident at ef = 300.
  int auto_cand_lds(int ef, int ns, int floor_entries, size_t fixed_bytes) const {
    if (cand_lds_override > 0) return std::max(cand_lds_override, floor_entries);
    if (ns > 0) return std::max(floor_entries, std::min(std::max(2 * ef, 128), 1024));
    const size_t budget = 10240;  // ~16 resident wavefronts per CU out of 160 KB LDS
    size_t used = fixed_bytes + (size_t)(ef + 1) * 8;
    int c = used < budget ? (int)((budget - used) / 8) : 0;
    return std::max(c, std::max(floor_entries, 128));
  }

  // log2 entries of the LDS visited cache (16-bit tags: usable while N >> bits fits 16 bits
  // with 0xFFFF to spare)
  int auto_vc_bits() const {
    if (visited_cache < 0) return 0;
    int want = visited_cache > 0 ? visited_cache : 1024;
    int bits = 8;
    while ((1 << bits) < want && bits < 14) ++bits;
    if (((unsigned)host.N >> bits) >= 0xFFFFu) return 0;
    return bits;
  }

  // The visited filter (visited_filter.h) a search on the sorted set should have at least.  A search at ef = 300 evaluates
  // 1 100 to 1 300 distinct nodes on the million-point sets (max_m0 24 and 32 alike), about 800 at ef = 100; the filter gets
  // 4 * ef + 512 entries, and twice as many when a repeated evaluation is expensive (rows of 2 KB and more).  Without sets
  // when ids do not fit the tags of a filter of that many entries, rounded up to a power of two.
  FilterShape least_filter(int ef) const {
    long long want = filter_entries > 0 ? filter_entries : 4ll * ef + 512;
    if (filter_entries <= 0 && Dp >= 512) want *= 2;
    int bits = 8;
    while ((2ll << bits) < want && bits < 13) ++bits;
    if (((unsigned)host.N >> (bits - 1)) >= 0xFFFFu) return FilterShape();  // tags are 16 bits wide, sets 64
    return filter_shape((int)std::min<long long>((want + 3) / 4, 1 << (bits - 1)), host.N);
  }
  // ... and the one it gets: what the wavefronts that the kernel's registers allow leave of LDS is the filter's, as far as it
  // needs it (four times the least: next to nothing is forgotten then).  Nor must it be what limits the wavefronts: half the
  // filter repeats more evaluations, but is the faster choice wherever it buys 15 % more of them.
  // (Against the next power of two above the least: 500 000 x 128 at ef 128, 256 -> 568 sets, 10 000 queries 1.93 -> 1.81 ms; 150 000
  // x 100 L2, 1 500 to 6 500 queries, ef 180 0.92 to 0.96 of the time, ef 300 0.95 to 0.98; dot rows of 64 elements 1.0 to 1.03.)
  // (Worked out once per kernel, filter to begin with -- and so to end with -- and LDS beside it, which the sizes without a
  // filter, with the first and with the last tell: the answer lies over the filter and counts as far as it is longer.)
  struct Fitted {
    const void* kernel;
    uint32_t first;
    size_t lds_none, lds_first, lds_last;
    int sets;
  };
  std::vector<Fitted> filters_known;
  template <typename K, typename Lds>
  FilterShape fit_filter(K kernel, FilterShape f, Lds&& lds_of) {
    if (filter_entries > 0 || f.sets() == 0) return f;
    const void* const id = reinterpret_cast<const void*>(kernel);
    const int most = std::min(4 * f.sets(), kMostFilterSets);
    Fitted now{id, f.code, lds_of(FilterShape()), lds_of(f), lds_of(filter_shape(most, host.N)), 0};
    for (const Fitted& k : filters_known)
      if (k.kernel == id && k.first == now.first && k.lds_none == now.lds_none && k.lds_first == now.lds_first && k.lds_last == now.lds_last)
        return filter_shape(k.sets, host.N);
    while (true) {
      const FilterShape half = filter_shape(f.sets() / 2, host.N);
      if (half.sets() >= f.sets() || resident_slots(kernel, lds_of(half)) * 20 < resident_slots(kernel, lds_of(f)) * 23) break;
      f = half;
    }
    const int waves = resident_slots(kernel, lds_of(f));
    for (int low = f.sets(), high = most; high - low >= 8;) {
      const FilterShape mid = filter_shape((low + high) / 2, host.N);
      if (mid.sets() > low && mid.sets() < high && resident_slots(kernel, lds_of(mid)) >= waves) low = (f = mid).sets();
      else high = (low + high) / 2;
    }
    if (filters_known.size() >= 64) filters_known.clear();
    now.sets = f.sets();
    filters_known.push_back(now);
    return f;
  }

  // How many workgroups (of one wavefront, or of `waves`) of a kernel the GPU holds.  A workgroup's LDS is handed out in whole steps of
  // kLdsStep bytes, which the runtime's answer leaves out (measured with workgroups that count each other, 160 KB per CU:
  // 5 120 bytes 32 on a CU, 5 184 25, 6 464 21, 7 744 18; the runtime says 32, 31, 25 and 21).  (Asked once per kernel and LDS
  // size: a search wants to know half a dozen of them.)
  static constexpr size_t kLdsStep = 1280;
  struct Resident {
    const void* kernel;
    size_t lds;
    int waves;
    int slots;
  };
  std::vector<Resident> resident_known;
  template <typename K>
  int resident_slots(K kernel, size_t lds, int waves = 1) {
    const void* const id = reinterpret_cast<const void*>(kernel);
    for (const Resident& r : resident_known)
      if (r.kernel == id && r.lds == lds && r.waves == waves) return r.slots;
    hipFuncAttributes attr;
    HIP_CHECK(hipFuncGetAttributes(&attr, id));
    const size_t fixed = attr.sharedSizeBytes, whole = (fixed + lds + kLdsStep - 1) / kLdsStep * kLdsStep;
    int per_cu = 0;
    HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64 * waves, std::max(whole, fixed) - fixed));
    per_cu = std::max(waves > 1 ? 0 : 1, std::min(per_cu, 32));
    if (resident_known.size() >= 256) resident_known.clear();
    resident_known.push_back({id, lds, waves, per_cu * num_cus});
    return per_cu * num_cus;
  }

  // Whether teams of `waves` wavefronts are faster than a wavefront alone per query: what helpers evaluate ahead must be what the search
  // comes to.  A short search ends before it has got to most of the 32 candidates in line, and the less the rows and the other teams
  // leave of a CU the longer a search it takes to make up for that.  A long one on a CU that teams share has its wavefronts busy and its
  // memory as well; rows of 129 to 256 elements spill in teams on top.  Bounds of ef by row (up to 64, 128, 256 elements, longer) and
  // load (a team of eight for every fourth CU or fewer, for every CU or fewer, two on a CU; teams of four).
  // Time by teams over time alone, 100 000 to 1 M elements, fp32 and fp16, dot and L2 -- inside the bounds 0.6 to 1.03.  Outside:
  // x 50 ef 16 1.02 to 1.1, ef 1 000 256 queries 0.95 and 1.09, fours 0.97 to 1.19; 500 000 x 96 ef 30 64 to 1 024 queries 1.04 to
  // 1.13, ef 500 fours 1.07 and 1.12; 400 000 x 200 ef 20 1.06 to 1.46, ef 64 400 to 1 024 queries 1.1 to 1.2, fours at ef 128 0.96 to
  // 1.1, 440 1.01 to 1.13, 512 1.07 to 1.16, x 180 in fp16 0.98 to 1.04, 1.09 to 1.15, 1.09 to 1.18; 300 000 x 200 L2, 1 024 queries 1.0 to
  // 1.3; 90 000 x 960 ef 20 128 and more 1.09 to 1.19.
  static bool teams_pay(int qr, int ef, int nq, int cus, int waves, bool half) {
    struct Bounds { int from, to; };
    constexpr Bounds bounds[4][4] = {{{32, 960}, {32, 928}, {40, 512}, {40, 704}},
                                     {{40, 960}, {48, 928}, {56, 512}, {72, 640}},
                                     {{48, 960}, {72, 704}, {100, 512}, {128, 320}},
                                     {{40, 960}, {48, 928}, {48, 512}, {48, 640}}};
    const bool fours = waves < kMostTeam;
    const int row = qr == 0 ? 3 : qr >> 1;
    const Bounds b = bounds[row][fours ? 3 : 4 * nq <= cus ? 0 : nq <= cus ? 1 : 2];
    if (fours && qr == 4 && (half || nq > 3 * cus)) return false;
    if (fours && qr == 2 && nq > 2 * cus && ef > 448) return false;
    return ef >= b.from && (ef <= b.to || 32 * nq <= cus);  // (few enough, and the longest search of the batch is an ordinary one)
  }

  // A batch that leaves the machine idle by teams of wavefronts, a workgroup of eight or four per query (kernels.h, team_help);
  // false: not such a batch.  Eight where the GPU holds them for all queries at once, else four (a number in between puts two of
  // a workgroup's wavefronts on one SIMD as eight do: 345 678 x 101 in fp16, 400 queries, 5 to 7 of them 319 us, four 229).
  // A wavefront alone -> by teams, ef 300, us, 1 / 32 / 256 / 512 / 768 / 1 000 queries: 100 000 x 50 264 -> 182, 320 -> 232, 451 -> 323,
  // 512 -> 377, 554 -> 454, 584 -> 538; 500 000 x 96 273 -> 191, 386 -> 284, 507 -> 408, 542 -> 420, 558 -> 501, 580 -> 560; 100 000 x 180
  // 275 -> 204, 348 -> 258, 393 -> 314, 444 -> 367, 468 -> 436.  On long rows the GPU holds no teams for more than 512 queries:
  // x 300 343 -> 239, 424 -> 305, 493 -> 374, 517 -> 455; x 512 317 -> 226, 397 -> 301, 666 -> 542, 705 -> 639.
  // Alone as well: long rows where the batch has the memory busy, to which helpers add a quarter (100 000 x 960, 32 queries 551 -> 366
  // us; 256 646, in eights 618, in fours 582; 400 667, in fours 687; 512 710, in fours 817).
  template <typename K, typename Lds>
  bool launch_teams(K kernel, int qr, int ns, Lds&& search_lds, const DevIndex& ix, SearchArgs a) {
    constexpr size_t kBusyFrom = (size_t)1100 << 10, kHalfBusyFrom = (size_t)700 << 10;  // bytes of one row for every query
    const int per_cu = (a.nq + num_cus - 1) / num_cus;
    const size_t rows = qr == 0 ? (size_t)a.nq * Dp * (storage_half ? 2 : 4) : 0;
    if (ix.S0 > 64 || filter_entries > 0 || rows > kBusyFrom) return false;
    const size_t lds = (size_t)160 * 1024 / per_cu / kLdsStep * kLdsStep;
    const FilterShape least = least_filter(a.ef);
    a.fc = filter_shape(std::min(8 * least.sets(), 4096), host.N);  // (a forgotten node keeps candidates back)
    a.team_turn = num_cus;
    a.team_bucket_bits = 5;
    auto bytes = [&] { return search_lds(a.fc) + (size_t)Team::words(ns, a.team_bucket_bits, ix.S0) * 4; };
    while (a.fc.sets() > 2 * least.sets() && bytes() > lds) a.fc = filter_shape(a.fc.sets() / 2, host.N);
    while (a.team_bucket_bits > 3 && bytes() > lds) --a.team_bucket_bits;
    if (bytes() > lds) return false;
    for (int waves = rows > kHalfBusyFrom ? kMostTeam / 2 : kMostTeam; waves >= kMostTeam / 2; waves /= 2) {
      if (!teams_pay(qr, a.ef, a.nq, num_cus, waves, storage_half) || resident_slots(kernel, bytes(), waves) < per_cu * num_cus) continue;
      hipLaunchKernelGGL(kernel, dim3(a.nq), dim3(64 * waves), bytes(), stream, ix, a);
      HIP_CHECK(hipGetLastError());
      last_team = waves;
      return true;
    }
    return false;
  }

  // ---- search ------------------------------------------------------------------------------
  // (defined in instances.hip, two objects per distance and row width)
  template <int DT, int QR, int NS>
  void launch_search(const DevIndex& ix, SearchArgs& a, int max_slots_override, float* ms);
  template <int DT, int QR, int NS>
  void launch_search_static(const DevIndex& ix, SearchArgs& a, float* ms);
  template <int DT, int QR>
  void launch_search_ns(int ns, const DevIndex& ix, SearchArgs& a, float* ms);
  template <int DT>
  void launch_search_qr(int q, int ns, const DevIndex& ix, SearchArgs& a, float* ms) {
    switch (q) {
      case 1: launch_search_ns<DT, 1>(ns, ix, a, ms); break;
      case 2: launch_search_ns<DT, 2>(ns, ix, a, ms); break;
      case 4: launch_search_ns<DT, 4>(ns, ix, a, ms); break;
      default: launch_search_ns<DT, 0>(ns, ix, a, ms); break;
    }
  }

  bool use_static = false;  // the running search is the one that allocates nothing

  void search_device(const float* d_qdata, int nq, int k, int ef, int* d_nns_out, float* d_dist_out, int* d_found_out,
                     int* d_stats, float* ms, bool no_alloc = false) {
    need_device();
    if (!have_graph) throw std::runtime_error("search_knn: no index (call build_graph or load_index first)");
    if (nq <= 0) return;
    if (k <= 0) throw std::runtime_error("search_knn: topk must be positive");
    ef = std::max(ef, k);
    use_static = no_alloc;
    if (no_alloc) {
      if (nq > kStaticMaxQueries)
        throw std::runtime_error("search_knn (no allocation): at most " + std::to_string(kStaticMaxQueries) + " queries per call");
      if (ef > kStaticMaxEf)
        throw std::runtime_error("search_knn (no allocation): max(topk, ef_search) must not exceed " + std::to_string(kStaticMaxEf));
      if (least_filter(ef).sets() == 0)
        throw std::runtime_error("search_knn (no allocation): the index has too many points for the LDS visited filter");
    }
    DevIndex ix = dev_index();
    SearchArgs a{};
    a.q = d_qdata; a.nq = nq; a.k = k; a.ef = ef;
    a.nns = d_nns_out; a.dists = d_dist_out; a.found = d_found_out; a.stats = d_stats;
    a.hnswlib_dist = hnswlib_dist;
    a.rcap = (std::max(std::max(host.S0, host.SU), 64) + 63) / 64 * 64;
    a.lcap = std::max(a.rcap, (k + 63) / 64 * 64);
    const int q = qr();
    size_t fixed = (size_t)a.lcap * 8 + (q == 0 ? (size_t)query_lds_chunks(Dp) * 16 : 0);
    int ns = key_slots(ef);
    a.vc_bits = auto_vc_bits();
    a.fast_path = no_alloc ? 2 : (fast_suspended ? 0 : fast_path);
    a.reverse = opt.reverse_cand ? 1 : 0;
    // An index with deleted elements (hnswlib's marks in a loaded file) is searched by hnswlib's rule for them:
    // walked through, never returned.  Only the search on the literal queues in LDS states that rule; it takes
    // every query of such an index.
    if (host.n_deleted > 0) {
      if (no_alloc) throw std::runtime_error("search_knn (no allocation): the index holds deleted elements");
      if (a.reverse) throw std::runtime_error("search_knn: reverse_cand is not defined on an index with deleted elements");
      ns = 0;
      a.fast_path = 0;
      a.deleted = d_deleted.p;
    }
    // reverse_cand: the sorted set in registers expands its farthest entry; beyond its capacity (ef >= 1024) the
    // literal pass does, on a sorted list in LDS
    if (a.reverse) a.fast_path = ns > 0 ? 2 : 0;
    if (a.reverse && no_alloc && ns == 0) throw std::runtime_error("search_knn (no allocation): reverse_cand needs ef_search below 1024");
    a.fc = (ns > 0 && a.fast_path) ? least_filter(ef) : FilterShape();
    if (a.reverse && ns > 0 && a.fc.sets() == 0)
      throw std::runtime_error("search_knn: reverse_cand needs fewer than 2^28 points");
    // with the keys in registers the queue's LDS share doubles as result buffer (lcap entries,
    // then lcap label slots) and as the replay heap (ef + 1 entries)
    const int floor_entries = ns > 0 ? std::max(ef + 1, 2 * a.lcap) : std::max(k, 64);
    a.cand_lds = auto_cand_lds(ef, ns, floor_entries, fixed);
    if (dist_type == DIST_DOT) launch_search_qr<DIST_DOT>(q, ns, ix, a, ms);
    else launch_search_qr<DIST_L2>(q, ns, ix, a, ms);
  }

  // taken() is called once the queries have been read for the last time
  template <typename Taken>
  void search_host(const float* q, int nq, int k, int ef, int* nns, float* dists, int* found, Taken&& taken) {
    need_device();
    if (nq <= 0) return;
    if (!q || !nns || !dists || !found) throw std::runtime_error("search_knn: null argument");
    if (k <= 0) throw std::runtime_error("search_knn: topk must be positive");
    // Small traffic skips the copy engine, of which every copy is 15 to 40 us with what surrounds it: the kernels read
    // few queries where they lie in pinned memory, and write the answers there (each is written once).
    const size_t q_bytes = (size_t)nq * host.D * 4, out_bytes = ((size_t)nq * k * 2 + nq) * 4;
    const bool direct_q = q_bytes <= kDirectQueries, direct_out = out_bytes <= kDirectAnswers;
    if (direct_q || direct_out) reserve_io((direct_q ? q_bytes : 0) + (direct_out ? out_bytes : 0));
    int* out = reinterpret_cast<int*>(h_io + (direct_q ? q_bytes : 0));
    const float* q_there;
    if (direct_q) {
      std::memcpy(h_io, q, q_bytes);
      q_there = reinterpret_cast<const float*>(h_io);
    } else {
      d_q.reserve((size_t)nq * host.D);
      q_there = d_q.p;
      if (staging.block() > 0) {
        const unsigned char* src = reinterpret_cast<const unsigned char*>(q);
        unsigned char* dst = reinterpret_cast<unsigned char*>(d_q.p);
        // (each copy is 15 us, whatever its size; threads pay from a megabyte each on.  Up to 2 MB: 4 000 x 128 in blocks of
        // 0.5 / 1 / 2 MB 303 / 303 / 320 us, 5 003 x 101 in fp16 682 / 669 / 667, out of the caller's memory 666.  10 000 x 128: 0.60 ms, 0.63 on one
        // thread, 0.61 to 0.67 in blocks of 1 or 0.5 MB; out of the caller's own memory in one copy that is waited for
        // 0.63; 100 000 x 128: 3.46, 3.89, 3.77 to 4.45 and 3.98 ms)
        const bool small = q_bytes <= staging.block();
        staging.send(stream, q_bytes, small ? kQueryBlock : staging.block(), [&](unsigned char* to, size_t at, size_t n) { std::memcpy(to, src + at, n); },
                     [&](size_t at, size_t) { return dst + at; }, [](unsigned char*, size_t, size_t) {}, [] {},
                     small ? 1 : (int)std::min<size_t>(q_bytes >> 20, HostStaging::kBlocks / 2), true);
      } else {  // (no pinned blocks are kept: one copy out of the caller's memory, waited for)
        HIP_CHECK(hipMemcpyAsync(d_q.p, q, q_bytes, hipMemcpyHostToDevice, stream));
        HIP_CHECK(hipStreamSynchronize(stream));
      }
    }
    taken();
    if (direct_out) {
      search_device(q_there, nq, k, ef, out, reinterpret_cast<float*>(out + (size_t)nq * k), out + (size_t)nq * k * 2, nullptr, nullptr);
      std::memcpy(nns, out, (size_t)nq * k * 4);
      std::memcpy(dists, out + (size_t)nq * k, (size_t)nq * k * 4);
      std::memcpy(found, out + (size_t)nq * k * 2, (size_t)nq * 4);
      return;
    }
    d_nns.reserve((size_t)nq * k);
    d_dist.reserve((size_t)nq * k);
    d_found.reserve((size_t)nq);
    search_device(q_there, nq, k, ef, d_nns.p, d_dist.p, d_found.p, nullptr, nullptr);
    HIP_CHECK(hipMemcpyAsync(nns, d_nns.p, (size_t)nq * k * 4, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipMemcpyAsync(dists, d_dist.p, (size_t)nq * k * 4, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipMemcpyAsync(found, d_found.p, (size_t)nq * 4, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
  }

  // ---- build ---------------------------------------------------------------------------------
  // (defined in instances.hip)
  template <int DT, int QR, int NS>
  void build_levels();
  template <int DT, int QR>
  void build_ns(int ns);
  template <int DT>
  void build_qr(int q, int ns) {
    switch (q) {
      case 1: build_ns<DT, 1>(ns); break;
      case 2: build_ns<DT, 2>(ns); break;
      case 4: build_ns<DT, 4>(ns); break;
      default: build_ns<DT, 0>(ns); break;
    }
  }

  void build_graph() {
    need_device();
    if (!have_data || !have_levels) throw std::runtime_error("build_graph: call set_data and set_random_levels first");
    const CallEnd at_end(*this);
    HIP_CHECK(hipMemsetAsync(d_ctl.p, 0, 4 * sizeof(int), stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    auto t0 = std::chrono::steady_clock::now();
    const int q = qr();
    const int ns = build_literal ? 0 : key_slots(opt.ef_construction);
    have_graph = false;
    if (dist_type == DIST_DOT) build_qr<DIST_DOT>(q, ns);
    else build_qr<DIST_L2>(q, ns);
    last_build_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    have_graph = true;
    forget_search_history();
    prepare_search_buffers();
  }

  // ---- measurement aid --------------------------------------------------------------------------------
  // random row gathers over the resident vectors (gather_probe_kernel): returns rows fetched, ms taken
  void gather_probe(int waves_per_cu, int rows_in_flight, int dependent, double* rows, float* ms) {
    need_device();
    if (!have_data) throw std::runtime_error("gather probe: no vectors (call set_data or load_index first)");
    const int waves = std::max(1, std::min(waves_per_cu, 32)) * num_cus;
    const int batches = 2048;
    const int U = rows_in_flight >= 16 ? 4 : (rows_in_flight >= 8 ? 2 : 1);
    DevBuf<float> sink;
    sink.reserve((size_t)waves);
    DevIndex ix = dev_index();
    float best = 0.f;
    for (int it = 0; it < 3; ++it) {
      HIP_CHECK(hipEventRecord(ev0, stream));
      if (U == 4) hipLaunchKernelGGL(gather_probe_kernel<4>, dim3(waves), dim3(64), 0, stream, ix, batches, dependent, sink.p);
      else if (U == 2) hipLaunchKernelGGL(gather_probe_kernel<2>, dim3(waves), dim3(64), 0, stream, ix, batches, dependent, sink.p);
      else hipLaunchKernelGGL(gather_probe_kernel<1>, dim3(waves), dim3(64), 0, stream, ix, batches, dependent, sink.p);
      HIP_CHECK(hipGetLastError());
      HIP_CHECK(hipEventRecord(ev1, stream));
      HIP_CHECK(hipEventSynchronize(ev1));
      float t = 0.f;
      HIP_CHECK(hipEventElapsedTime(&t, ev0, ev1));
      if (it == 0 || t < best) best = t;
    }
    if (rows) *rows = (double)waves * 4.0 * U * batches;
    if (ms) *ms = best;
  }

  // ---- index file --------------------------------------------------------------------------------
  // The level-0 block leaves device memory as the file's own bytes: packed by pack_records_kernel, piece by piece,
  // copied into the pinned blocks and from there into the file by the threads that wait for them.
  void save_index(const char* path) {
    if (!have_graph) throw std::runtime_error("save_index: no index to save");
    if (!has_device) {
      write_index_file(host, path);
      return;
    }
    const size_t rec = (size_t)FileLayout((uint64_t)host.max_m, (uint64_t)host.max_m0, (uint64_t)host.D).record;
    const size_t piece_rows = std::max<size_t>(1, std::min<size_t>((size_t)host.N, kPiece / rec));
    const CallEnd at_end(*this);
    workspace.begin();
    const auto p_packed = workspace.part<unsigned char>(piece_rows * rec);
    workspace.reserve();
    unsigned char* const packed = workspace.at(p_packed);
    staging.reserve(0, false);
    if (host.n_deleted > 0) upload_marks();
    std::vector<uint32_t> up((size_t)host.upper_rows * host.SU);
    if (!up.empty()) HIP_CHECK(hipMemcpyAsync(up.data(), d_linksU.p, up.size() * 4, hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    const DevIndex ix = dev_index();
    IndexWriter out(host, path);  // (after everything that may find no memory: the file that is there goes with it)
    for (size_t first = 0; first < (size_t)host.N; first += piece_rows) {
      const size_t rows = std::min(piece_rows, (size_t)host.N - first);
      hipLaunchKernelGGL(pack_records_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, ix, (int)first, (int)rows,
                         host.n_deleted > 0 ? d_deleted.p : nullptr, reinterpret_cast<uint32_t*>(packed));
      HIP_CHECK(hipGetLastError());
      const uint64_t file_at = FileLayout::kHeader + (uint64_t)first * rec;
      staging.fetch(stream, packed, rows * rec, out.parallel(),
                    [&](const unsigned char* from, size_t at, size_t n) { out.write(file_at + at, from, n); },
                    [&] {  // (beside the others, where the file may be written in any order)
                      if (out.parallel() && first + rows == (size_t)host.N) out.write_upper(host, up.data());
                    });
    }
    HIP_CHECK(hipStreamSynchronize(stream));
    if (!out.parallel()) out.write_upper(host, up.data());
    out.finish();
  }
  void upload_marks() {
    std::vector<uint32_t> marks(((size_t)host.N + 31) / 32, 0u);
    for (int i = 0; i < host.N; ++i)
      if (host.deleted[i]) marks[(size_t)i >> 5] |= 1u << (i & 31);
    d_deleted.reserve(marks.size());
    HIP_CHECK(hipMemcpyAsync(d_deleted.p, marks.data(), marks.size() * 4, hipMemcpyHostToDevice, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
  }
  // The way back: the level-0 block goes up as it stands in the file and is checked there; only once the whole file
  // has been found good do its records take the place of the index that was resident before.
  void load_index(const char* path) {
    HostIndex fresh;
    if (!has_device) {
      read_index_file(fresh, path);
      if (fresh.N <= 0) throw std::runtime_error("load_index: empty index");
      host = std::move(fresh);
      have_data = have_levels = have_graph = true;
      forget_search_history();
      return;
    }
    IndexReader in(fresh, path);
    const size_t rec = (size_t)in.layout.record, n = (size_t)fresh.N;
    const CallEnd at_end(*this);
    workspace.begin();
    const auto p_raw = workspace.part<unsigned char>(n * rec);
    const auto p_marks = workspace.part<unsigned char>(n);
    workspace.reserve();
    unsigned char *const raw = workspace.at(p_raw), *const marks = workspace.at(p_marks);
    staging.reserve(0, false);
    std::string upper_error;
    HIP_CHECK(hipMemsetAsync(d_ctl.p, 0, 2 * sizeof(int), stream));
    staging.send(stream, n * rec, staging.block(),
                 [&](unsigned char* to, size_t at, size_t len) { in.read(FileLayout::kHeader + at, to, len, "level-0 block"); },
                 [&](size_t at, size_t) { return raw + at; }, [](unsigned char*, size_t, size_t) {},
                 [&] {  // (on this thread, beside the others)
                   try {
                     in.read_upper(fresh);
                   } catch (const std::exception& ex) {
                     upper_error = ex.what();
                   }
                 });
    if (n > 0) {
      hipLaunchKernelGGL(check_records_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream,
                         reinterpret_cast<const uint32_t*>(raw), (int)n, fresh.D, fresh.max_m0, marks, d_ctl.p);
      HIP_CHECK(hipGetLastError());
    }
    HIP_CHECK(hipMemcpyAsync(h_ctl, d_ctl.p, 2 * sizeof(int), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    if (h_ctl[0] & 1) throw std::runtime_error("index file: link count above max_m0");
    if (h_ctl[0] & 2) throw std::runtime_error("index file: link id out of range");
    if (!upper_error.empty()) throw std::runtime_error(upper_error);
    in.check_unchanged();
    if (n == 0) throw std::runtime_error("load_index: empty index");
    fresh.n_deleted = h_ctl[1];
    if (fresh.n_deleted > 0) {
      fresh.deleted.resize(n);
      HIP_CHECK(hipMemcpyAsync(fresh.deleted.data(), marks, n, hipMemcpyDeviceToHost, stream));
      HIP_CHECK(hipStreamSynchronize(stream));
    }
    have_data = have_levels = have_graph = false;  // until all of it is there
    host = std::move(fresh);
    forget_search_history();
    reserve_vectors();
    upload_structure();
    d_labels.reserve(n);
    hipLaunchKernelGGL(unpack_records_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream,
                       reinterpret_cast<const uint32_t*>(raw), dev_index(), d_labels.p);
    HIP_CHECK(hipGetLastError());
    if (!host.linksU.empty())
      HIP_CHECK(hipMemcpyAsync(d_linksU.p, host.linksU.data(), host.linksU.size() * 4, hipMemcpyHostToDevice, stream));
    if (host.n_deleted > 0) upload_marks();
    HIP_CHECK(hipStreamSynchronize(stream));
    std::vector<uint32_t>().swap(host.linksU);
    pool_slots = 0;  // N may have changed: rebuild the slot pool lazily
    pool = SlotPool{};
    have_data = have_levels = have_graph = true;
    prepare_search_buffers();
  }
};


// every instance has an object of its own (instances.hip)
#define CUHNSW_EXTERN(DT, QR)                                                                                  \
  extern template void Engine::launch_search_ns<DT, QR>(int, const DevIndex&, SearchArgs&, float*);            \
  extern template void Engine::build_ns<DT, QR>(int);
CUHNSW_EXTERN(DIST_DOT, 0) CUHNSW_EXTERN(DIST_DOT, 1) CUHNSW_EXTERN(DIST_DOT, 2) CUHNSW_EXTERN(DIST_DOT, 4)
CUHNSW_EXTERN(DIST_L2, 0) CUHNSW_EXTERN(DIST_L2, 1) CUHNSW_EXTERN(DIST_L2, 2) CUHNSW_EXTERN(DIST_L2, 4)
#undef CUHNSW_EXTERN

}  // namespace cuhnsw_amd
