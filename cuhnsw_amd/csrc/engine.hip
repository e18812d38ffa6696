// C ABI of libcuhnsw_amd.so.
#include "engine.h"

#include "../../include/cuhnsw_amd.h"

namespace cuhnsw_amd {

static __device__ __align__(256) unsigned char scratch[sizeof(StaticScratch)];  // 12.5 MB

static StaticScratch* g_static_scratch[kMaxDevices] = {};
static std::mutex g_static_scratch_mutex;             // guards the table above
std::atomic_flag g_static_busy[kMaxDevices];
StaticScratch* static_scratch_for_current_device(int* device) {
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device ordinal beyond the table of static scratch addresses");
  if (device) *device = dev;
  std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
  if (!g_static_scratch[dev]) {
    void* ptr = nullptr;
    HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_static_scratch[dev] = static_cast<StaticScratch*>(ptr);
  }
  return g_static_scratch[dev];
}

}  // namespace cuhnsw_amd

// ---------------------------------------------------------------------------------------------- C ABI
using cuhnsw_amd::Engine;

struct cuhnsw_engine {
  Engine impl;
  std::mutex mutex;  // calls on one engine are serialised: they share its staging buffers, slot pool and streams
};

namespace {
thread_local std::string g_create_error;

template <typename F>
int locked(cuhnsw_engine* e, F&& f) {  // (the engine's lock is held)
  try {
    e->impl.err.clear();
    f(e->impl);
    return 0;
  } catch (const std::exception& ex) {
    e->impl.err = ex.what();
    return -1;
  } catch (...) {
    e->impl.err = "unknown error";
    return -1;
  }
}
template <typename F>
int guarded(cuhnsw_engine* e, F&& f) {
  if (!e) return -1;
  std::lock_guard<std::mutex> lock(e->mutex);
  return locked(e, f);
}
}  // namespace

extern "C" {

int cuhnsw_create(cuhnsw_engine** out) {
  if (!out) return -1;
  try {
    *out = new cuhnsw_engine();
    return 0;
  } catch (const std::exception& ex) {
    g_create_error = ex.what();
    *out = nullptr;
    return -1;
  }
}
void cuhnsw_destroy(cuhnsw_engine* e) { delete e; }
const char* cuhnsw_last_error(cuhnsw_engine* e) { return e ? e->impl.err.c_str() : g_create_error.c_str(); }

int cuhnsw_init(cuhnsw_engine* e, const char* opt_path) {
  if (!e) return -1;
  std::lock_guard<std::mutex> lock(e->mutex);
  return e->impl.init(opt_path);
}
int cuhnsw_set_data(cuhnsw_engine* e, const float* data, int num_data, int num_dims) {
  return guarded(e, [&](Engine& g) { g.set_data(data, num_data, num_dims); });
}
int cuhnsw_set_random_levels(cuhnsw_engine* e, const int* levels, int num_levels) {
  return guarded(e, [&](Engine& g) {
    if (!levels) throw std::runtime_error("set_random_levels: null levels");
    g.set_random_levels(levels, num_levels);
  });
}
int cuhnsw_build_graph(cuhnsw_engine* e) { return guarded(e, [&](Engine& g) { g.build_graph(); }); }
int cuhnsw_save_index(cuhnsw_engine* e, const char* fpath) {
  return guarded(e, [&](Engine& g) { g.save_index(fpath ? fpath : ""); });
}
int cuhnsw_load_index(cuhnsw_engine* e, const char* fpath) {
  return guarded(e, [&](Engine& g) { g.load_index(fpath ? fpath : ""); });
}
int cuhnsw_search_knn(cuhnsw_engine* e, const float* qdata, int num_queries, int topk, int ef_search, int* nns,
                      float* distances, int* found_cnt) {
  return guarded(e, [&](Engine& g) { g.search_host(qdata, num_queries, topk, ef_search, nns, distances, found_cnt, [] {}); });
}
int cuhnsw_search_knn_taking(cuhnsw_engine* e, const float* qdata, int num_queries, int num_dims, int topk, int ef_search,
                             int* nns, float* distances, int* found_cnt, void (*taken)(void*), void* arg) {
  if (!e || !taken) return -1;
  // (an engine that is at work is not waited for with the queries still in the caller's memory)
  std::vector<float> own;
  bool told = false;
  std::unique_lock<std::mutex> lock(e->mutex, std::try_to_lock);
  if (!lock.owns_lock()) {
    try {
      if (qdata && num_queries > 0 && num_dims > 0) own.assign(qdata, qdata + (size_t)num_queries * num_dims);
    } catch (const std::exception&) {
      return -1;
    }
    if (qdata) qdata = own.data();
    taken(arg);
    told = true;
    lock.lock();
  }
  return locked(e, [&](Engine& g) {
    if (num_dims != g.host.D) throw std::runtime_error("query dimension differs from the index dimension");
    g.search_host(qdata, num_queries, topk, ef_search, nns, distances, found_cnt, [&] {
      if (!told) taken(arg);
    });
  });
}
int cuhnsw_search_knn_device(cuhnsw_engine* e, const float* d_qdata, int num_queries, int topk, int ef_search, int* d_nns,
                             float* d_distances, int* d_found_cnt, int* d_stats, float* kernel_ms) {
  return guarded(e, [&](Engine& g) {
    g.search_device(d_qdata, num_queries, topk, ef_search, d_nns, d_distances, d_found_cnt, d_stats, kernel_ms);
  });
}
int cuhnsw_search_knn_device_noalloc(cuhnsw_engine* e, const float* d_qdata, int num_queries, int topk, int ef_search,
                                     int* d_nns, float* d_distances, int* d_found_cnt, float* kernel_ms) {
  return guarded(e, [&](Engine& g) {
    g.search_device(d_qdata, num_queries, topk, ef_search, d_nns, d_distances, d_found_cnt, nullptr, kernel_ms, true);
  });
}
int cuhnsw_debug_gather_probe(cuhnsw_engine* e, int waves_per_cu, int rows_in_flight, int dependent, double* rows,
                              float* ms) {
  return guarded(e, [&](Engine& g) { g.gather_probe(waves_per_cu, rows_in_flight, dependent, rows, ms); });
}
int cuhnsw_last_build_dropped_links(cuhnsw_engine* e) { return e ? e->impl.last_build_dropped : 0; }
int cuhnsw_last_build_counters(cuhnsw_engine* e, unsigned long long* out, int n) {
  if (!e || !out || n < 10) return -1;
  std::memcpy(out, e->impl.build_counters, sizeof(e->impl.build_counters));
  return 0;
}
int cuhnsw_debug_link_keys0(cuhnsw_engine* e, float* out, long long capacity) {
  return guarded(e, [&](Engine& g) {
    if (g.link_keys0.empty()) throw std::runtime_error("link keys were not kept: set tunable keep_link_keys before build_graph");
    if (!out || capacity < (long long)g.link_keys0.size()) throw std::runtime_error("link keys: output buffer too small");
    std::memcpy(out, g.link_keys0.data(), g.link_keys0.size() * sizeof(float));
  });
}
int cuhnsw_num_data(cuhnsw_engine* e) { return e ? e->impl.host.N : 0; }
int cuhnsw_num_dims(cuhnsw_engine* e) { return e ? e->impl.host.D : 0; }
int cuhnsw_max_level(cuhnsw_engine* e) { return e ? e->impl.host.maxlevel : 0; }
int cuhnsw_enter_point(cuhnsw_engine* e) { return e ? (int)e->impl.host.enterpoint : 0; }
int cuhnsw_has_device(void) { return cuhnsw_amd::device_present() ? 1 : 0; }
double cuhnsw_last_build_seconds(cuhnsw_engine* e) { return e ? e->impl.last_build_seconds : 0.0; }
int cuhnsw_num_deleted(cuhnsw_engine* e) { return e ? e->impl.host.n_deleted : 0; }
int cuhnsw_last_search_repeats(cuhnsw_engine* e) { return e ? e->impl.last_repeats : 0; }
int cuhnsw_last_search_trails(cuhnsw_engine* e) { return e ? e->impl.last_trails : 0; }
int cuhnsw_last_search_side_by_side(cuhnsw_engine* e) { return e ? e->impl.last_side_by_side : 0; }
int cuhnsw_last_search_team(cuhnsw_engine* e) { return e ? e->impl.last_team : 0; }
int cuhnsw_last_build_team_batches(cuhnsw_engine* e) { return e ? e->impl.last_team_batches : 0; }
int cuhnsw_literal_fallbacks(cuhnsw_engine* e) { return e ? e->impl.literal_fallbacks : 0; }
int cuhnsw_trails_available(cuhnsw_engine* e) { return e ? (e->impl.trails_unavailable ? 0 : 1) : 0; }
int cuhnsw_set_tunable(cuhnsw_engine* e, const char* name, double value) {
  if (!e || !name) return -1;
  std::lock_guard<std::mutex> lock(e->mutex);
  std::string n(name);
  if (n == "build_batch") e->impl.build_batch = (int)value;
  else if (n == "level_first") e->impl.level_first = (int)value;
  else if (n == "build_literal") e->impl.build_literal = (int)value;
  else if (n == "search_slots") e->impl.search_slots = (int)value;
  else if (n == "cand_lds") e->impl.cand_lds_override = (int)value;
  else if (n == "hnswlib_dist") e->impl.hnswlib_dist = (int)value;
  else if (n == "visited_cache") e->impl.visited_cache = (int)value;
  else if (n == "own_links0") e->impl.own_links0 = (int)value;
  else if (n == "newcomer_shortcut") e->impl.newcomer_shortcut = value != 0.0;
  else if (n == "fast_path") e->impl.fast_path = (int)value;
  else if (n == "lean_literal") e->impl.lean_literal = (int)value;
  else if (n == "trails") e->impl.trails = (int)value;
  else if (n == "trail_cap") e->impl.trail_cap = std::max(1, (int)value);
  else if (n == "trail_spares") e->impl.trail_spares = std::max(0, (int)value);
  else if (n == "filter_entries") e->impl.filter_entries = (int)value;
  else if (n == "query_order") e->impl.query_order = (int)value;
  else if (n == "first_pass_waves") e->impl.first_pass_waves = (int)value;
  else if (n == "concurrent_literal") e->impl.concurrent_literal = value != 0.0;
  else if (n == "literal_spin_limit") e->impl.spin_limit_override = (int)value;
  else if (n == "literal_per_cu") e->impl.side_per_cu = std::max(0, std::min(8, (int)value));
  else if (n == "spill_cap") e->impl.spill_cap = (int)value;
  else if (n == "keep_workspace") {
    e->impl.keep_workspace = value != 0.0;
    e->impl.give_back_workspace();
  }
  else if (n == "keep_link_keys") e->impl.keep_link_keys = value != 0.0;
  else if (n == "build_counters") e->impl.count_build_work = value != 0.0;
  else if (n == "tight_rows") {
    if (e->impl.have_data && e->impl.tight_rows != (value != 0.0)) return -2;  // only before the vectors are there
    e->impl.tight_rows = value != 0.0;
  }
  else if (n == "fp16_storage") {
    if (e->impl.have_data && e->impl.storage_half != (value != 0.0)) return -2;  // only before the vectors are there
    e->impl.storage_half = value != 0.0;
  }
  else return -1;
  return 0;
}

}  // extern "C"
