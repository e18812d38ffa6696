// Wavefront-level building blocks shared by the search and build kernels (gfx950,
// 64-lane wavefronts, one wavefront per query / inserted node).
//
//   * distances: a 64-lane wavefront works on FOUR rows at a time, 16 lanes per row,
//     each lane loading float4 (dwordx4) chunks of the row, so one load instruction
//     of the wavefront fetches 4 x 256 contiguous bytes.  The 16 lanes are reduced
//     with DPP (quad_perm, row_half_mirror, row_mirror); no LDS, no barrier.
//     Replaces dot / squaresum / GetDistanceByVec of the reference
//     (cpp/include/cuda_dist_kernels.cuh:13-124), which reduce over a 32-thread
//     block through shared memory.
//   * the search runs on ONE sorted set of (key, id, expanded) kept in registers
//     (Frontier, search_level_fast): result set and candidate set of hnswlib at once, which
//     is exact unless the layout of hnswlib's heaps would decide between equal keys; its
//     visited filter is a four-way tag cache in LDS only (visit_lossy).  Replaces the
//     global-memory, thread-0 heap of the reference (cpp/include/cuda_heap_kernels.cuh:13-49),
//     its GetCand / CheckAlreadyExists scans (cpp/include/cuda_utils_kernels.cuh:50-151) and
//     its lossy visited table (cpp/include/cuda_utils_kernels.cuh:185-210).
//   * where equal keys do decide, the search is repeated with hnswlib's two priority queues
//     reproduced move for move: candidate queue in LDS as a libstdc++ heap, each push / pop
//     executed cooperatively by the wavefront (heap_coop.h), result set as sorted keys in
//     registers plus a log (search_level), or as the sorted set with ids (search_level_lean);
//     visited set either an exact bitmap per wavefront in global memory, cleared through an
//     undo list, or the LDS filter.
//
// Canonical fp32 distance arithmetic: element i is accumulated with one fused
// multiply-add into partial sum (i mod 64) in increasing i; the 64 partials are
// combined by a pairwise adjacent tree (s = 1,2 inside a lane, s = 4..32 across the
// 16 lanes).  The key used for ordering is 1 - dot (hnswlib) or the squared L2.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "heap_coop.h"
#include "index_file.h"
#include "options.h"
#include "team_slots.h"
#include "visited_filter.h"

namespace cuhnsw_amd {

struct DevIndex {
  const void* vectors;       // N x Dp, rows zero padded to Dp (multiple of 32 elements); fp32, or fp16 when half != 0
  const uint64_t* labels;    // N, or null when labels are the internal ids
  uint32_t* links0;          // N x S0
  uint32_t* linksU;          // upper rows x SU
  const int64_t* upper_off;  // N
  const int* levels;         // N
  float* dists0;             // build only: key of every level-0 link
  float* distsU;             // build only
  int N, D, Dp, S0, SU, max_m, max_m0, maxlevel;
  uint32_t enterpoint;
  int half;                  // vectors are stored as fp16 (all arithmetic stays fp32 on the stored values)
};

// What the wavefronts of a team share in LDS beside the visited filter (team_help): whose list is in which slot, four slots to a bucket;
// the candidates that come next; whether the search is over; room to work in for the wavefront that searches; the lists.
constexpr int kTeamSlots = 128;  // at most
struct Team {
  uint32_t* base = nullptr;
  int bucket_bits = 0;  // log2 of the buckets
  int stride = 0;       // ids (and keys) a list holds
  int lists = 0;        // where they begin
  static constexpr int kInLine = 32;
  static constexpr int kLine = kTeamSlots, kOver = kLine + 2 * (kInLine + 1), kRoom = kOver + 2;
  __host__ __device__ static int lists_at(int ns) { return kRoom + 128 * (ns + 1); }
  __host__ __device__ static int words(int ns, int bucket_bits, int stride) { return lists_at(ns) + (8 << bucket_bits) * stride; }
  __device__ __forceinline__ uint32_t* owner() const { return base; }
  // the closest candidates; behind them a place that nobody reads
  __device__ __forceinline__ HeapEnt* line() const { return reinterpret_cast<HeapEnt*>(base + kLine); }
  __device__ __forceinline__ uint32_t* over() const { return base + kOver; }
  // the level that is searched (from bit 16 on), and a number that changes with it: odd while no list may be begun
  __device__ __forceinline__ uint32_t* level() const { return base + kOver + 1; }
  __device__ __forceinline__ uint32_t* room() const { return base + kRoom; }
  __device__ __forceinline__ uint32_t bucket(uint32_t id) const { return (id * 2654435761u) >> (32 - bucket_bits); }
  __device__ __forceinline__ uint32_t* ids(int slot) const { return base + lists + 2 * slot * stride; }
  __device__ __forceinline__ float* keys(int slot) const { return reinterpret_cast<float*>(ids(slot) + stride); }
};

// per resident wavefront scratch: LDS pointers + this wavefront's global slot
struct Scratch {
  HeapEnt* top;        // LDS, ef + 1 entries
  HeapEnt* cand;       // LDS, cand_lds entries
  HeapEnt* cand_glob;  // global overflow of the candidate queue
  int cand_lds, cand_glob_cap;
  uint32_t* nbuf;      // LDS, lcap ids
  float* dbuf;         // LDS, lcap keys
  float4* qlds;        // LDS copy of the query (only when the query is not kept in registers)
  uint16_t* vcache;    // LDS, direct-mapped cache of ids known to be visited (null = none)
  int vc_bits;         // log2 of its size: slot = id & (size-1), tag = id >> vc_bits
  FilterShape filter;  // where vcache is the sorted-set search's filter instead (visit_lossy)
  uint32_t* bitmap;    // global, one bit per node
  uint32_t* undo;      // global, ids whose bit is set
  int undo_cap;
  int bitmap_words;
  HeapEnt* log;        // global, every accepted (key, id) in acceptance order
  int log_cap;
  StageTree tree;      // per-lane constants of the cooperative heap pop
  Team team;           // LDS, shared with the wavefronts that help this one (sorted-set search of a batch that leaves the machine idle)
};

// The candidates a search expands at a time (tie_free_phase) lie in LDS behind the 64 ids that search lists in s.nbuf.
constexpr int kAhead = 8;
__host__ __device__ inline int nbuf_words(int lcap) { return lcap > 64 + 2 * kAhead ? lcap : 64 + 2 * kAhead; }
__device__ __forceinline__ HeapEnt* batch_candidates(const Scratch& s) { return reinterpret_cast<HeapEnt*>(s.nbuf + 64); }

struct SearchState {
  int top_size, cand_size;  // top_size: entries of the result set = min(accepted, ef)
  int n_acc;                // accepted so far (= log entries)
  float maxkey;             // largest accepted key
  float lower;
  int undo_cnt;
  int n_dist, n_hops, n_dist_upper, n_sweeps;
  int fail;
  int ahead;  // tie-free loop on a full set: candidates it expands at a time (tie_free_phase)
};

struct LdsHeap {
  HeapEnt* a;
  __device__ __forceinline__ HeapEnt get(int i) const { return a[i]; }
  __device__ __forceinline__ void set(int i, HeapEnt e) { a[i] = e; }
};
struct SplitHeap {
  HeapEnt* lds;
  HeapEnt* glob;
  int nlds;
  // The global branch waits for its own load at once (s_waitcnt vmcnt(0)).  It is the rare
  // path; without the explicit wait the compiler merges both branches into one flat load
  // and then has to drain ALL outstanding vector-memory traffic (the fire-and-forget log and
  // undo stores too) before unrelated instructions of the hot loop.
  __device__ __forceinline__ HeapEnt get(int i) const {
    if (i < nlds) return lds[i];
    HeapEnt r = glob[i - nlds];
    __builtin_amdgcn_s_waitcnt(0x0F70);
    return r;
  }
  __device__ __forceinline__ void set(int i, HeapEnt e) {
    if (i < nlds) {
      lds[i] = e;
    } else {
      glob[i - nlds] = e;
      __builtin_amdgcn_s_waitcnt(0x0F70);
    }
  }
};

template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// sum over each group of 16 consecutive lanes; every lane of the group gets the same bits.
// Must be executed with all 64 lanes active.
__device__ __forceinline__ float reduce16(float x) {
  x = x + dpp_move<0xB1>(x);   // quad_perm [1,0,3,2]
  x = x + dpp_move<0x4E>(x);   // quad_perm [2,3,0,1]
  x = x + dpp_move<0x141>(x);  // row_half_mirror
  x = x + dpp_move<0x140>(x);  // row_mirror
  return x;
}
// Tells the compiler that a value is the same in all lanes (it is then kept in a scalar register
// and branches on it are scalar branches instead of exec-mask juggling).
__device__ __forceinline__ float uni(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
// The same number, which the compiler takes for a new one: what is computed from it is computed here, not ahead of the
// loops around and kept in registers through them.
__device__ __forceinline__ int fresh(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
// how many lanes below this one have their bit set in a wavefront-uniform mask (v_mbcnt: no lane masks in registers)
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned int)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)mask, 0u));
}
__device__ __forceinline__ unsigned long long first_lanes(int n) { return n < 64 ? (1ull << (n & 63)) - 1ull : ~0ull; }  // (n <= 64)

// Smallest value of all lanes, wavefront-uniform.  (Through neighbours' registers: as exchanges through LDS it took 720 cycles, a
// quarter of a step of a descent.)
__device__ __forceinline__ float least_of_all(float x) {
  auto take = [&](int from) __attribute__((always_inline)) { x = fminf(x, __builtin_bit_cast(float, from)); };
  const auto bits = [&]() __attribute__((always_inline)) { return __builtin_bit_cast(int, x); };
  take(__builtin_amdgcn_update_dpp(bits(), bits(), 0x111, 0xF, 0xF, false));  // (lane 63 has seen all in the end)
  take(__builtin_amdgcn_update_dpp(bits(), bits(), 0x112, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(bits(), bits(), 0x114, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(bits(), bits(), 0x118, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(bits(), bits(), 0x142, 0xA, 0xF, false));
  take(__builtin_amdgcn_update_dpp(bits(), bits(), 0x143, 0xC, 0xF, false));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits(), 63));
}
template <int DT>
__device__ __forceinline__ void acc4(const float4 q, const float4 v, float& ax, float& ay, float& az, float& aw) {
  if (DT == DIST_DOT) {
    ax = __builtin_fmaf(q.x, v.x, ax);
    ay = __builtin_fmaf(q.y, v.y, ay);
    az = __builtin_fmaf(q.z, v.z, az);
    aw = __builtin_fmaf(q.w, v.w, aw);
  } else {
    float tx = q.x - v.x, ty = q.y - v.y, tz = q.z - v.z, tw = q.w - v.w;
    ax = __builtin_fmaf(tx, tx, ax);
    ay = __builtin_fmaf(ty, ty, ay);
    az = __builtin_fmaf(tz, tz, az);
    aw = __builtin_fmaf(tw, tw, aw);
  }
}
// One chunk (four consecutive elements) of stored vectors: 16 bytes of fp32, or 8 bytes of fp16
// widened to fp32 (exact).  `chunk` counts chunks from the start of the array.
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 load_chunk_f32(const void* base, uint64_t chunk) {
  return reinterpret_cast<const float4*>(base)[chunk];
}
__device__ __forceinline__ float4 widen(const half4_t h) {
  const floatx4_t f = __builtin_convertvector(h, floatx4_t);
  return make_float4(f.x, f.y, f.z, f.w);
}
__device__ __forceinline__ float4 widen(const float4 v) { return v; }
__device__ __forceinline__ float4 load_chunk_f16(const void* base, uint64_t chunk) {
  return widen(reinterpret_cast<const half4_t*>(base)[chunk]);
}
template <bool HALF>
struct StoredChunk {
  using type = float4;
};
template <>
struct StoredChunk<true> {
  using type = half4_t;
};

// Chunks past a row's end are fetched all the same (chunk 0 in their place) and do not count.  Not by a select: a load
// whose only use is a select is moved into a branch on the select's condition, split into words there and waited for
// before the next row's is issued (200 000 x 128, L2, 32 queries: 5 300 cycles for the 15 rows of a step).  These numbers
// are made where the compiler does not see what they are (AGAIN: anew each time, else once if registers allow).
__device__ __forceinline__ uint32_t mask_if(bool inside) {  // for masked(): the same bits, or zeros
  uint32_t m = inside ? ~0u : 0u;
  asm("" : "+v"(m));
  return m;
}
template <bool AGAIN = false>
__device__ __forceinline__ float minus_one_if(bool inside) {
  float m = inside ? -1.0f : -0.0f;
  if (AGAIN) asm volatile("" : "+v"(m));
  else asm("" : "+v"(m));
  return m;
}
__device__ __forceinline__ float4 masked(const float4 t, uint32_t m) {
  return make_float4(__uint_as_float(__float_as_uint(t.x) & m), __uint_as_float(__float_as_uint(t.y) & m),
                     __uint_as_float(__float_as_uint(t.z) & m), __uint_as_float(__float_as_uint(t.w) & m));
}
// acc4 where v counts only where `neg` is -1 (L2; elsewhere it is -0, and q is zero there).  q + (-1) * v is q - v to the
// bit.  (An infinite element makes 0 * v a NaN: only for ordering keys, which stop at the largest number either way.)
__device__ __forceinline__ void acc4_l2_if(const float4 q, const float4 v, float neg, float& ax, float& ay, float& az, float& aw) {
  const float tx = __builtin_fmaf(neg, v.x, q.x), ty = __builtin_fmaf(neg, v.y, q.y);
  const float tz = __builtin_fmaf(neg, v.z, q.z), tw = __builtin_fmaf(neg, v.w, q.w);
  ax = __builtin_fmaf(tx, tx, ax);
  ay = __builtin_fmaf(ty, ty, ay);
  az = __builtin_fmaf(tz, tz, az);
  aw = __builtin_fmaf(tw, tw, aw);
}

// RAW = false: ordering key (1 - dot | squared L2); RAW = true: API value (-dot | squared L2)
//
// The distance of two finite vectors can overflow to an infinity.  An ordering key never is one: it stops at the largest
// finite number, so that no entry of a set is ever equal to the set's padding (-inf below, +inf above), which keeps its
// place by comparisons alone -- an infinite key would be lost among the padding and the padding's id taken for its
// node's.  The order is the same (only a key that is exactly the largest number is no longer told from an overflow), and
// what a search returns is computed without the stop, or freed of it (answer_key).
constexpr float kLargestKey = 3.402823466e+38f;
// (written out: with both bounds in operands of its own the compiler keeps one of them in a vector register throughout)
__device__ __forceinline__ float bounded_key(float x) {
  float r;
  asm("v_med3_f32 %0, %1, -%2, %2" : "=v"(r) : "v"(x), "s"(kLargestKey));
  return r;
}
template <int DT, bool RAW>
__device__ __forceinline__ float finish_sum(float s) {
  if (DT == DIST_DOT) return RAW ? -s : bounded_key(1.0f - s);
  return RAW ? s : fminf(s, kLargestKey);
}
__device__ __forceinline__ float answer_key(float key) {
  return __builtin_fabsf(key) < kLargestKey ? key : __builtin_copysignf(INFINITY, key);
}
template <int DT, bool RAW>
__device__ __forceinline__ float finish16(float ax, float ay, float az, float aw) {
  float s = (ax + ay) + (az + aw);
  s = reduce16(s);
  return finish_sum<DT, RAW>(s);
}

// The same for U rows at once (s[u]: this lane's partial sum of row u): lane `sub` < U of each group of 16 gets row sub's
// value, the other lanes garbage.  The rows share the steps: each of the first two folds two of them into one register
// (even lanes go on with one, odd lanes with the other), so that four rows take 11 additions and selections instead of
// 16 plus what spreading the results over the lanes would take.  Same pairs in the same tree, hence the same bits.
template <int CTRL>
__device__ __forceinline__ float dpp_move_zero(float x) {  // (lanes without a source: 0)
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
template <int DT, bool RAW, int U>
__device__ __forceinline__ float finish_rows(const float* s, int sub) {
  static_assert(U == 1 || U == 2 || U == 4, "rows per lane group");
  float x;
  if (U == 1) {
    x = s[0] + dpp_move<0xB1>(s[0]);  // quad_perm [1,0,3,2]
    x = x + dpp_move<0x4E>(x);        // quad_perm [2,3,0,1]
  } else {
    const bool odd = (sub & 1) != 0;
    float y[2];
#pragma unroll
    for (int p = 0; p < U / 2; ++p) {
      const float own = odd ? s[2 * p + (U > 1 ? 1 : 0)] : s[2 * p], other = odd ? s[2 * p] : s[2 * p + (U > 1 ? 1 : 0)];
      y[p] = own + dpp_move<0xB1>(other);
    }
    if (U == 2) {
      x = y[0] + dpp_move<0x4E>(y[0]);
    } else {
      const bool high = (sub & 2) != 0;
      const float own = high ? y[1] : y[0], other = high ? y[0] : y[1];
      x = own + dpp_move<0x4E>(other);
    }
  }
  x = x + dpp_move_zero<0x104>(x);  // row_shl:4 (from the lane four above)
  x = x + dpp_move_zero<0x108>(x);  // row_shl:8
  return finish_sum<DT, RAW>(x);
}

// Query kept in registers: lane `sub` of each 16-lane group holds float4 chunks
// sub, sub+16, ... (QR of them).  QR == 0 selects the LDS copy instead.
template <int QR>
struct QVec {
  float4 q[QR > 0 ? QR : 1];
};

// Long rows (the query is read from LDS): 16 lanes own a row, so a lane fetches every 16th chunk of it,
// kLongB of them per round.  The LDS copy of the query is zero-padded to whole rounds (kLongB * 16 chunks),
// so that a round reads it without guards.
constexpr int kLongB = 8;
__host__ __device__ inline int query_lds_chunks(int Dp) {
  const int chunk_rows = ((Dp >> 2) + 15) / 16;
  return (chunk_rows + kLongB - 1) / kLongB * kLongB * 16;
}

// fills the query holder from a row of D floats (any alignment)
template <int QR>
__device__ __forceinline__ void load_query(QVec<QR>& qv, float4* qlds, const float* src, int D, int Dp, int lane) {
  if (QR > 0) {
    const int sub = lane & 15;
#pragma unroll
    for (int k = 0; k < (QR > 0 ? QR : 1); ++k) {
      int i = 4 * (sub + 16 * k);
      float4 t;
      t.x = i + 0 < D ? src[i + 0] : 0.0f;
      t.y = i + 1 < D ? src[i + 1] : 0.0f;
      t.z = i + 2 < D ? src[i + 2] : 0.0f;
      t.w = i + 3 < D ? src[i + 3] : 0.0f;
      qv.q[k] = t;
    }
  } else {
    const int chunks = query_lds_chunks(Dp);
    for (int c = lane; c < chunks; c += 64) {
      int i = 4 * c;
      float4 t;
      t.x = i + 0 < D ? src[i + 0] : 0.0f;
      t.y = i + 1 < D ? src[i + 1] : 0.0f;
      t.z = i + 2 < D ? src[i + 2] : 0.0f;
      t.w = i + 3 < D ? src[i + 3] : 0.0f;
      qlds[c] = t;
    }
    wave_sync();
  }
}

// one pass over 4*U rows starting at ids[r]: loads first, arithmetic after.  SELECT: chunks past the data are left out by a
// select after all (literal_select)
template <int DT, int R, int U, bool RAW, bool HALF, bool SELECT = false>
__device__ __forceinline__ void dist_pass(const void* rows, uint32_t rowlen, uint32_t used, const float4* q,
                                          const uint32_t* ids, int r, int n, float* out, int g, int sub) {
  if (DT != DIST_DOT && R == 2) sub = fresh(sub);  // (these are short of registers where the set is large)
  float4 v[U][R];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int idx = r + 4 * u + g;
    const uint32_t id = ids[idx < n ? idx : n - 1];
    const uint64_t first = (uint64_t)id * rowlen;  // one 32x32->64 multiply-add
#pragma unroll
    for (int k = 0; k < R; ++k) {
      // always one unconditional load; a chunk past
      // the row's data (`used` chunks; the row's stride may be longer) re-reads chunk 0, which costs no
      // further memory line.  The query holds zeros there, which is all a dot product needs (finite
      // data); for L2 the chunk does not count (acc4_l2_if).  The data is longer than
      // 16 * (R / 2) chunks, so only the upper half of k can be past its end.
      const uint32_t c = sub + 16 * k;
      const uint64_t at = first + (c < used ? c : 0);
      const float4 t = HALF ? load_chunk_f16(rows, at) : load_chunk_f32(rows, at);
      v[u][k] = SELECT && DT != DIST_DOT && k >= R / 2 && !(c < used) ? q[k] : t;
    }
  }
  float neg[R];
  uint32_t keep[R];
#pragma unroll
  for (int k = R / 2; k < R; ++k) {
    if (DT != DIST_DOT && !RAW) neg[k] = minus_one_if<(U * R < 8)>((uint32_t)(sub + 16 * k) < used);
    if (DT != DIST_DOT && RAW) keep[k] = mask_if((uint32_t)(sub + 16 * k) < used);
  }
  float s[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float ax = 0.f, ay = 0.f, az = 0.f, aw = 0.f;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      if (DT == DIST_DOT || k < R / 2 || SELECT) acc4<DT>(q[k], v[u][k], ax, ay, az, aw);
      else if (RAW) acc4<DT>(q[k], masked(v[u][k], keep[k]), ax, ay, az, aw);
      else acc4_l2_if(q[k], v[u][k], neg[k], ax, ay, az, aw);
    }
    s[u] = (ax + ay) + (az + aw);
  }
#pragma unroll
  for (int u = 0; u < U; u += 4) {
    constexpr int H = U < 4 ? U : 4;
    const float key = finish_rows<DT, RAW, H>(s + u, sub);
    const int mine = r + 4 * (u + sub) + g;
    if (sub < H && mine < n) out[mine] = key;
  }
  // (the lanes meet again here, not at the caller's loop end: see trail_mark)
  __builtin_amdgcn_wave_barrier();
}

// long rows: 16 lanes still own one row (the summation order is tied to 16 lanes), so a lane
// has rowlen/16 chunks to fetch; they are issued B at a time for each of U groups of four rows, to keep
// U * B loads per lane in flight; the query chunks come from LDS, one read for all U groups.  Rounds that
// lie wholly inside the rows' data carry no guards; the last one re-reads chunk 0 for chunks past the end
// and multiplies zeros there (the LDS copy of the query is zero-padded to whole rounds).
template <int DT, bool RAW, bool HALF, int U, int B>
__device__ __forceinline__ void dist_long_pass(const void* rows, int rowlen, int used, const float4* qlds, const uint32_t* ids,
                                               int r, int n, float* out, int g, int sub) {
  static_assert(B == kLongB, "the LDS copy of the query is padded to rounds of kLongB chunk rows");
  const int nk = (used + 15) >> 4;  // chunk rows that hold data
  const int nfull = used >> 4;      // chunk rows that hold nothing else
  uint64_t first[U];
  float ax[U], ay[U], az[U], aw[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int idx = r + 4 * u + g;
    const uint32_t id = ids[idx < n ? idx : n - 1];
    first[u] = (uint64_t)id * (uint32_t)rowlen;
    ax[u] = ay[u] = az[u] = aw[u] = 0.f;
  }
  // (fp16 chunks are widened where they are used, all of them asked for by then: short of registers the compiler widens each
  // on arrival otherwise, and waits for it before it asks for the next.  1 000 queries in fp16: 60 000 x 960, ef 400 2.49 ->
  // 1.16 ms, ef 300 1.03 -> 0.98; 60 000 x 300, ef 400 1.61 -> 1.02)
  using Stored = typename StoredChunk<HALF>::type;
  const Stored* chunks = reinterpret_cast<const Stored*>(rows);
  int k0 = 0;
  for (; k0 + B <= nfull; k0 += B) {
    Stored v[U][B];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int b = 0; b < B; ++b) v[u][b] = chunks[first[u] + (uint32_t)(sub + 16 * (k0 + b))];
    }
    // (the round's query chunks are read in one go, ahead of the arithmetic: read one by one each would be
    // waited for in turn, which is what a lone wavefront's time goes to)
    float4 qq[B];
#pragma unroll
    for (int b = 0; b < B; ++b) qq[b] = qlds[sub + 16 * (k0 + b)];
    if (HALF) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
      for (int u = 0; u < U; ++u) acc4<DT>(qq[b], widen(v[u][b]), ax[u], ay[u], az[u], aw[u]);
    }
  }
  if (k0 < nk) {  // (k0 + B > nfull >= nk - 1: one more round reaches the end)
    Stored v[U][B];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int c = sub + 16 * (k0 + b);
        v[u][b] = chunks[first[u] + (uint32_t)(c < used ? c : 0)];  // unconditional load (chunk 0 past the end)
      }
    }
    float4 qq[B];
#pragma unroll
    for (int b = 0; b < B; ++b) qq[b] = qlds[sub + 16 * (k0 + b)];  // zeros past the end
    if (HALF) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const uint32_t inside = mask_if(sub + 16 * (k0 + b) < used);
#pragma unroll
      for (int u = 0; u < U; ++u) acc4<DT>(qq[b], masked(widen(v[u][b]), inside), ax[u], ay[u], az[u], aw[u]);
    }
  }
  float s[U];
#pragma unroll
  for (int u = 0; u < U; ++u) s[u] = (ax[u] + ay[u]) + (az[u] + aw[u]);
  const float key = finish_rows<DT, RAW, U>(s, sub);
  const int mine = r + 4 * sub + g;
  if (sub < U && mine < n) out[mine] = key;
  __builtin_amdgcn_wave_barrier();  // (the lanes meet again here, not at the loop's end: see trail_mark)
}
// U = 2: eight rows at a time while more than four are left (twice the loads in flight, 64 more registers:
// for the search of few queries at a time, where a wavefront waits for its own loads and arithmetic in turn)
template <int DT, bool RAW, bool HALF, int U>
__device__ __forceinline__ void dist_long(const void* rows, int rowlen, int used, const float4* qlds, const uint32_t* ids,
                                          int n, float* out, int g, int sub) {
  int r = 0;
  while (r < n) {
    if (U >= 4 && n - r > 8) {
      dist_long_pass<DT, RAW, HALF, (U >= 4 ? 4 : 1), kLongB>(rows, rowlen, used, qlds, ids, r, n, out, g, sub);
      r += 16;
    } else if (U >= 2 && n - r > 4) {
      dist_long_pass<DT, RAW, HALF, (U >= 2 ? 2 : 1), kLongB>(rows, rowlen, used, qlds, ids, r, n, out, g, sub);
      r += 8;
    } else {
      dist_long_pass<DT, RAW, HALF, 1, kLongB>(rows, rowlen, used, qlds, ids, r, n, out, g, sub);
      r += 4;
    }
  }
}

// keys of ids[0..n) (LDS) against the query -> out[0..n) (LDS).  n is wavefront-uniform.
template <int DT, int QR, bool RAW, bool HALF, int WIDE = 1, bool SELECT = false>
__device__ __forceinline__ void dist_list_t(const DevIndex& ix, const QVec<QR>& qv, const float4* qlds, const uint32_t* ids,
                                            int n, float* out, int lane) {
  const int g = lane >> 4, sub = lane & 15;
  const int rowlen = ix.Dp >> 2;
  const int used = (ix.D + 3) >> 2;  // chunks of a row that hold data
  const void* rows = ix.vectors;
  if (QR > 0) {
    constexpr int R = QR > 0 ? QR : 1;
    // groups of 4 rows in flight
    constexpr int UMAX = R == 1 ? (WIDE >= 4 ? 8 : 4) : (R == 2 ? (WIDE >= 4 ? 8 : (WIDE >= 2 ? 4 : (WIDE >= 1 ? 2 : 1))) : (WIDE >= 4 ? 4 : (WIDE >= 3 ? 2 : 1)));
    int r = 0;
    while (r < n) {
      const int rem = n - r;
      if (UMAX >= 8 && rem > 16) {
        dist_pass<DT, R, (UMAX >= 8 ? 8 : 1), RAW, HALF, SELECT>(rows, rowlen, used, qv.q, ids, r, n, out, g, sub);
        r += 32;
      } else if (UMAX >= 4 && rem > 8) {
        dist_pass<DT, R, (UMAX >= 4 ? 4 : 1), RAW, HALF, SELECT>(rows, rowlen, used, qv.q, ids, r, n, out, g, sub);
        r += 16;
      } else if (UMAX >= 2 && rem > 4) {
        dist_pass<DT, R, (UMAX >= 2 ? 2 : 1), RAW, HALF, SELECT>(rows, rowlen, used, qv.q, ids, r, n, out, g, sub);
        r += 8;
      } else {
        dist_pass<DT, R, 1, RAW, HALF, SELECT>(rows, rowlen, used, qv.q, ids, r, n, out, g, sub);
        r += 4;
      }
    }
  } else {
    dist_long<DT, RAW, HALF, WIDE>(rows, rowlen, used, qlds, ids, n, out, g, sub);
  }
}
// (the element type of the stored vectors is a property of the index: one scalar branch per list.  In the wide instances the
// code for fp16 goes out of the way, which is 1 % of a search of one query; elsewhere it costs spills.)
// WIDE: how many rows are in flight; 1 = as many as registers allow beside a full machine's wavefronts, 4 = as a
// wavefront with a SIMD to itself can have, 0 = four
template <int DT, int QR, bool RAW, int WIDE = 1, bool SELECT = false>
__device__ __forceinline__ void dist_list(const DevIndex& ix, const QVec<QR>& qv, const float4* qlds,
                                          const uint32_t* ids, int n, float* out, int lane) {
  const bool half = uni(ix.half) != 0;
  if (WIDE >= 4 ? __builtin_expect(half, 0) : half) dist_list_t<DT, QR, RAW, true, WIDE, SELECT>(ix, qv, qlds, ids, n, out, lane);
  else dist_list_t<DT, QR, RAW, false, WIDE, SELECT>(ix, qv, qlds, ids, n, out, lane);
}

// The same for the searches on the literal queues: long rows eight at a time (dist_long), L2 rows of two chunks per lane
// four at a time -- a hop of theirs has four new nodes, and eight in flight spill in the loop (100 000 x 128, ef 300, 200
// queries on the literal queues alone: 1.38 -> 1.30 ms).
template <int DT, int QR, int NS>
constexpr int literal_wide() {
  return QR == 0 && NS <= 8 ? 2 : (DT == DIST_L2 && QR == 2 ? 0 : 1);
}
// And there L2 rows of up to 64 elements leave chunks past the data out by a select, where the result set is larger than five
// keys per lane or a heap in LDS (60 000 x 40 integers: 100 queries at ef 600 1.87 -> 1.78 ms, 2 000 at 1 100 6.11 -> 5.84; at
// ef 300 no difference, at 128 0.87 against 0.88).
template <int DT, int QR, int NS>
constexpr bool literal_select() {
  return DT == DIST_L2 && QR == 1 && (NS == 0 || NS > 5);
}

__device__ __forceinline__ const uint32_t* link_row(const DevIndex& ix, uint32_t node, int level) {
  return level == 0 ? ix.links0 + (size_t)node * ix.S0 : ix.linksU + (size_t)(ix.upper_off[node] + level - 1) * ix.SU;
}
// A wavefront-uniform pointer whose making the compiler cannot see: an access through it then takes its address from a
// scalar pair and a lane offset, where it would otherwise keep base + lane offset, two registers, through the whole search.
__device__ __forceinline__ const uint32_t* scalar_base(const uint32_t* p) {
  asm volatile("" : "+s"(p));
  return p;
}
__device__ __forceinline__ int row_stride(const DevIndex& ix, int level) { return level == 0 ? ix.S0 : ix.SU; }

// The visited bitmap of a slot is touched by one wavefront only; the atomic is there because
// two lanes of that wavefront may hit the same word.  Workgroup scope is therefore enough
// and lets the read-modify-write complete in the XCD's own L2 instead of being pushed out
// to device-coherent memory as an agent-scope atomic (atomicOr) is.
__device__ __forceinline__ uint32_t visited_fetch_or(uint32_t* word, uint32_t bit) {
  return __hip_atomic_fetch_or(word, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// In front of the bitmap sits a small direct-mapped cache in LDS of ids already known to be
// visited (16-bit tags, slot = low id bits).  Most neighbours of an expanded node were seen
// a few hops earlier; a cache hit answers "visited" exactly (tags are only written for ids
// whose bit is set) and saves the global atomic — on the 1.18M-point benchmark the atomics
// were more than half of all L2 requests and nearly all of the DRAM write traffic.
__device__ __forceinline__ void vcache_reset(Scratch& s, int lane) {
  if (s.vcache == nullptr) return;
  uint4* c4 = reinterpret_cast<uint4*>(s.vcache);
  const int n4 = (1 << s.vc_bits) >> 3;  // 8 tags per 16 bytes
  for (int i = lane; i < n4; i += 64) c4[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
  wave_sync();
}

// marks one id visited (lane 0 does it); returns nothing, logs it for the undo
__device__ __forceinline__ void visit_single(Scratch& s, SearchState& st, uint32_t id, int lane) {
  if (lane == 0) {
    visited_fetch_or(&s.bitmap[id >> 5], 1u << (id & 31));
    if (st.undo_cnt < s.undo_cap) s.undo[st.undo_cnt] = id;
    if (s.vcache != nullptr) s.vcache[id & ((1u << s.vc_bits) - 1u)] = (uint16_t)(id >> s.vc_bits);
  }
  st.undo_cnt += 1;
}

// Reads a link row, marks its ids visited and compacts the ones seen for the first
// time into s.nbuf (stored order kept).  Returns how many.
__device__ __forceinline__ int visit_row(const uint32_t* row, int S, Scratch& s, SearchState& st, int lane) {
  int n = 0;
  for (int base = 0; base < S; base += 64) {
    uint32_t id = (base + lane < S) ? row[base + lane] : kEmpty;
    bool ask = id != kEmpty;
    uint32_t slot = 0;
    uint16_t tag = 0;
    if (s.vcache != nullptr && ask) {
      slot = id & ((1u << s.vc_bits) - 1u);
      tag = (uint16_t)(id >> s.vc_bits);
      ask = s.vcache[slot] != tag;  // hit: visited for sure
    }
    bool newly = false;
    if (ask) {
      uint32_t bit = 1u << (id & 31);
      uint32_t old = visited_fetch_or(&s.bitmap[id >> 5], bit);
      newly = (old & bit) == 0;
      if (s.vcache != nullptr) s.vcache[slot] = tag;
    }
    unsigned long long mask = __ballot(newly);
    int pos = n + lanes_below(mask);
    if (newly) {
      s.nbuf[pos] = id;
      int u = st.undo_cnt + pos;
      if (u < s.undo_cap) s.undo[u] = id;
    }
    n += __popcll(mask);
    wave_sync();
  }
  st.undo_cnt += n;
  return n;
}

// The same for rows of at most 64 slots, split in two so that the vector rows of the
// neighbours can be fetched WHILE the visited atomics are in flight instead of after them:
// visit_issue() starts the atomics for every neighbour the cache does not vouch for and
// compacts those ids into s.nbuf; the caller computes their distances; visit_commit() then
// reads the atomics' answers, blanks the entries that turn out to have been visited before
// (kEmpty in s.nbuf; their distances are discarded) and logs the new ones for the undo.
// The speculative rows are few: after the cache most remaining neighbours are new.
struct VisitPending {
  uint32_t id, bit, old;
  int pos, n_ask;
  bool ask;
};
__device__ __forceinline__ VisitPending visit_issue(const uint32_t* row, int S, Scratch& s, int lane) {
  VisitPending v;
  v.id = lane < S ? row[lane] : kEmpty;
  v.ask = v.id != kEmpty;
  uint32_t slot = 0;
  uint16_t tag = 0;
  if (s.vcache != nullptr && v.ask) {
    slot = v.id & ((1u << s.vc_bits) - 1u);
    tag = (uint16_t)(v.id >> s.vc_bits);
    v.ask = s.vcache[slot] != tag;
  }
  const unsigned long long mask = __ballot(v.ask);
  v.pos = lanes_below(mask);
  v.n_ask = __popcll(mask);
  v.bit = 1u << (v.id & 31);
  v.old = 0u;
  if (v.ask) {
    v.old = visited_fetch_or(&s.bitmap[v.id >> 5], v.bit);
    s.nbuf[v.pos] = v.id;
    if (s.vcache != nullptr) s.vcache[slot] = tag;
  }
  return v;
}
__device__ __forceinline__ int visit_commit(const VisitPending& v, Scratch& s, SearchState& st, int lane) {
  const bool newly = v.ask && (v.old & v.bit) == 0u;
  const unsigned long long mask = __ballot(newly);
  if (v.ask && !newly) s.nbuf[v.pos] = kEmpty;
  if (newly) {
    const int u = st.undo_cnt + lanes_below(mask);
    if (u < s.undo_cap) s.undo[u] = v.id;
  }
  const int n_new = __popcll(mask);
  st.undo_cnt += n_new;
  return n_new;
}

// Reads a link row and compacts its valid ids into s.nbuf without touching the visited set.
__device__ __forceinline__ int load_row(const uint32_t* row, int S, Scratch& s, int lane) {
  int n = 0;
  for (int base = 0; base < S; base += 64) {
    uint32_t id = (base + lane < S) ? row[base + lane] : kEmpty;
    bool valid = id != kEmpty;
    unsigned long long mask = __ballot(valid);
    int pos = n + lanes_below(mask);
    if (valid) s.nbuf[pos] = id;
    n += __popcll(mask);
  }
  return n;
}

// clears the bits this wavefront set; leaves the slot's bitmap all zero
__device__ __forceinline__ void undo_visited(Scratch& s, SearchState& st, int lane) {
  if (st.undo_cnt <= s.undo_cap) {
    for (int i = lane; i < st.undo_cnt; i += 64) s.bitmap[s.undo[i] >> 5] = 0u;
  } else {
    for (int w = lane; w < s.bitmap_words; w += 64) s.bitmap[w] = 0u;
  }
  // (the bitmap belongs to this wavefront alone: its clearing stores only have to be done before its next
  // atomics are issued.  An agent-scope fence here would write the L2 back and invalidate the L1 once per query.)
  __threadfence_block();
  st.undo_cnt = 0;
}

// The result set's KEYS, kept sorted in registers: lane L holds sorted positions
// [L*NS, L*NS + NS).  hnswlib's search uses top_candidates only through its size and its
// largest key (lowerBound), and both depend on the multiset of accepted keys alone, not on
// the heap's layout — so during the search the ids are not needed and the eviction
// "push, then pop the maximum" becomes one sorted insert (about 35 vector instructions, no
// LDS).  Which ids survive is decided at the end from the log of accepted entries; only a
// tie exactly at the k-th key needs the literal heap, which is then replayed from the log.
// Unused positions hold +inf; when the set is full the evicted key falls off the end.
template <int NS>
struct TopKeys {
  float k[NS > 0 ? NS : 1];
};
// The keys are kept right-aligned: sorted position p lives in physical slot p + 64*NS - ef,
// the slots below hold -inf and never move.  The largest key of a FULL set then always sits
// in the last slot of lane 63 — a fixed register, which matters: indexing the register
// array with a run-time position would push it through scratch memory.
template <int NS>
__device__ __forceinline__ void topkeys_init(TopKeys<NS>& t, int ef, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
#pragma unroll
  for (int j = 0; j < N; ++j) t.k[j] = (lane * N + j < 64 * N - ef) ? -INFINITY : INFINITY;
}
template <int NS>
__device__ __forceinline__ void topkeys_insert(TopKeys<NS>& t, float v, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  int c = 0;  // keys of this lane below v
#pragma unroll
  for (int j = 0; j < N; ++j) c += t.k[j] < v ? 1 : 0;
  // previous lane's count and last key (lane 0: "all below", nothing to take over)
  const int prev_c = __builtin_amdgcn_update_dpp(N, c, 0x138, 0xF, 0xF, false);  // wave_shr:1
  const float prev_last = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, t.k[N - 1]), 0x138, 0xF, 0xF, false));
  const bool shifted = prev_c < N;         // the insertion happened in an earlier lane
  const int pos = shifted ? 0 : c;         // c == N: this lane is untouched
  const float incoming = shifted ? prev_last : v;
#pragma unroll
  for (int j = N - 1; j >= 0; --j) {
    const float below = j > 0 ? t.k[j - 1] : incoming;
    t.k[j] = j > pos ? below : (j == pos ? incoming : t.k[j]);
  }
}
// largest key of a full set
template <int NS>
__device__ __forceinline__ float topkeys_max(const TopKeys<NS>& t) {
  constexpr int N = NS > 0 ? NS : 1;
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, t.k[N - 1]), 63));
}
// key at sorted position pos (wavefront-uniform, once per search): through an LDS copy
template <int NS>
__device__ __forceinline__ float topkeys_at(const TopKeys<NS>& t, int pos, int ef, float* lds_tmp, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  wave_sync();
#pragma unroll
  for (int j = 0; j < N; ++j) lds_tmp[lane * N + j] = t.k[j];
  wave_sync();
  const float x = lds_tmp[pos + 64 * N - ef];
  wave_sync();
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}

// Offers nbuf/dbuf[0..n) in stored order (hnswlib's accept rule, identical to the
// reference's, cpp/include/cuda_utils_kernels.cuh:220-225).  Wavefront-uniform: every lane
// runs it, the heap moves are cooperative.  NS > 0: result keys in registers (TopKeys);
// NS == 0: literal result heap in LDS (s.top), for ef beyond the register capacity.
// deleted (NS == 0 only): one bit per element, hnswlib's delete marks (hnswlib searchBaseLayerST, has_deletions):
// a marked element is queued as a candidate like any other and never enters the result heap; the bound moves
// only while that heap holds something.
template <int NS>
__device__ __forceinline__ void accept_list(Scratch& s, SearchState& st, TopKeys<NS>& tk, int n, int ef, int lane,
                                            const uint32_t* deleted = nullptr) {
  SplitHeap cand{s.cand, s.cand_glob, s.cand_lds};
  const int cand_cap = s.cand_lds + s.cand_glob_cap;
  for (int base = 0; base < n; base += 64) {
    // every lane takes one offer; blanked entries (speculatively fetched neighbours that had
    // been visited before) and offers that already fail against the current bound are
    // dropped at once (the bound never rises once the set is full), the others are taken in
    // stored order and re-checked against the bound as it moves
    const int mine = base + lane;
    const float my_key = mine < n ? s.dbuf[mine] : INFINITY;
    const uint32_t my_id = mine < n ? s.nbuf[mine] : 0u;
    unsigned long long todo = __ballot(mine < n && my_id != kEmpty && (st.top_size < ef || st.lower > my_key));
    unsigned long long marked = 0ull;
    if (NS == 0 && deleted != nullptr)
      marked = __ballot(mine < n && my_id != kEmpty && ((deleted[my_id >> 5] >> (my_id & 31u)) & 1u) != 0u);
    while (todo != 0ull) {
      const int j = __builtin_ctzll(todo);
      todo &= todo - 1ull;
      HeapEnt e;
      e.key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_key), j));
      e.id = (uint32_t)__builtin_amdgcn_readlane((int)my_id, j);
      // (if/else nesting with one way out of the loops, as in search_level_fast)
      if (st.top_size < ef || st.lower > e.key) {
        if (st.cand_size >= cand_cap || (NS > 0 && st.n_acc >= s.log_cap)) {
          st.fail = 1;
          todo = 0ull;
        } else {
          if (NS > 0 && lane == 0) s.log[st.n_acc] = e;
          st.n_acc += 1;
          // the candidate queue normally fits its LDS share: keep that case on pure LDS
          // instructions (the split accessor compiles to flat loads)
          if (st.cand_size < s.cand_lds) {
            LdsHeap cand_fast{s.cand};
            coop_push<true>(cand_fast, st.cand_size, e, lane);
          } else {
            coop_push<true>(cand, st.cand_size, e, lane);
          }
          if (NS > 0) {
            topkeys_insert<NS>(tk, e.key, lane);
            st.top_size = st.n_acc < ef ? st.n_acc : ef;
            st.maxkey = fmaxf(st.maxkey, e.key);
            st.lower = st.n_acc >= ef ? topkeys_max<NS>(tk) : st.maxkey;  // hnswlib's lowerBound
          } else {
            LdsHeap top{s.top};
            if (((marked >> j) & 1ull) == 0ull) {
              coop_push<false>(top, st.top_size, e, lane);
              if (st.top_size > ef) coop_pop<false>(top, st.top_size, s.tree, lane);
            }
            wave_sync();
            if (st.top_size > 0)
              st.lower = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, s.top[0].key)));
          }
        }
      }
    }
    if (st.fail) base = n;
  }
}

// Best-first search of one level (hnswlib searchBaseLayerST / searchBaseLayer).
// On entry s.nbuf[0..n_seed) holds seed ids that are already marked visited.  On exit
// the accepted entries are in s.log[0..st.n_acc) and tk holds the result keys (NS > 0), or
// s.top[0..st.top_size) is the literal result max-heap (NS == 0).  BUILD selects hnswlib's
// construction-time stop rule; so do delete marks (see accept_list): a result heap short of ef never stops
// the search, marked candidates beyond the bound are walked through.
template <int DT, int QR, int NS, bool BUILD>
__device__ __forceinline__ void search_level(const DevIndex& ix, const QVec<QR>& qv, int level, int ef, Scratch& s,
                                             SearchState& st, TopKeys<NS>& tk, int n_seed, int lane,
                                             const uint32_t* deleted = nullptr) {
  SplitHeap cand{s.cand, s.cand_glob, s.cand_lds};
  const int S = row_stride(ix, level);
  constexpr int kWide = BUILD ? 1 : literal_wide<DT, QR, NS>();
  constexpr bool kSelect = !BUILD && literal_select<DT, QR, NS>();
  int n = n_seed;
  if (n > 0) {
    dist_list<DT, QR, false, 1, kSelect>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
    st.n_dist += n;
  }
  while (true) {
    wave_sync();
    int cid = -1;
    accept_list<NS>(s, st, tk, n, ef, lane, deleted);
    if (!st.fail && st.cand_size > 0) {
      wave_sync();
      const HeapEnt c = uniform_ent(s.cand[0]);
      const bool stop = (BUILD || (NS == 0 && deleted != nullptr)) ? (c.key > st.lower && st.top_size == ef) : (c.key > st.lower);
      if (!stop) {
        cid = (int)c.id;
        if (st.cand_size <= s.cand_lds) {
          LdsHeap cand_fast{s.cand};
          coop_pop<true>(cand_fast, st.cand_size, s.tree, lane);
        } else {
          coop_pop<true>(cand, st.cand_size, s.tree, lane);
        }
      }
    }
    wave_sync();
    if (cid < 0) break;
    st.n_hops += 1;
    const uint32_t* row = link_row(ix, (uint32_t)cid, level);
    if (S <= 64) {
      const VisitPending vp = visit_issue(row, S, s, lane);
      wave_sync();
      n = vp.n_ask;
      if (n > 0) dist_list<DT, QR, false, kWide, kSelect>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
      wave_sync();
      st.n_dist += visit_commit(vp, s, st, lane);
    } else {
      n = visit_row(row, S, s, st, lane);
      wave_sync();
      if (n > 0) dist_list<DT, QR, false, kWide, kSelect>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
      st.n_dist += n;
    }
  }
}

// ---- the tie-free fast path -------------------------------------------------------------
// hnswlib expands a candidate only while its key is <= lowerBound, the largest key of the
// result set, and once an entry has been evicted from the result set its key stays >= every
// later lowerBound.  So the candidates that are ever expanded are exactly the not yet
// expanded members of the result set, and ONE sorted set of (key, id, expanded) does the work
// of both priority queues (the reference's kernel uses the same view of the algorithm,
// cpp/include/cuda_search_kernels.cuh:99-164).  The equivalence is exact as long as no two
// keys that are in the set at the same time are equal: then the order of expansion, the
// evicted entry and the final order do not depend on how a heap lays equal keys out.  The set
// lives in registers, sorted, lane L holding positions [L*NS, L*NS + NS) (right-aligned like
// TopKeys); an insert is a shift through one DPP exchange, the next candidate is the first
// entry without the expanded mark.  An insert that meets an equal key reports it; the search
// kernel then repeats the query with the literal queues, the build (where any deterministic
// choice among equal keys is as good) carries on.
template <int NS>
struct Frontier {
  float k[NS > 0 ? NS : 1];
  uint32_t v[NS > 0 ? NS : 1];  // id; bit 31 = expanded (also set on the padding)
};
constexpr uint32_t kExpanded = 0x80000000u;
template <int NS>
__device__ __forceinline__ void frontier_init(Frontier<NS>& f, int ef, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    f.k[j] = (lane * N + j < 64 * N - ef) ? -INFINITY : INFINITY;
    f.v[j] = kEmpty;
  }
}
// is there an entry with exactly this key?
template <int NS>
__device__ __forceinline__ bool frontier_has_key(const Frontier<NS>& f, float v) {
  constexpr int N = NS > 0 ? NS : 1;
  unsigned long long eq = 0ull;  // (masks ORed in scalar registers: a bool per lane would be made a number and compared again)
#pragma unroll
  for (int j = 0; j < N; ++j) eq |= __ballot(f.k[j] == v);
  return eq != 0ull;
}
// ... and with this id?
template <int NS>
__device__ __forceinline__ bool frontier_has(const Frontier<NS>& f, float v, uint32_t id) {
  constexpr int N = NS > 0 ? NS : 1;
  unsigned long long same = 0ull;
#pragma unroll
  for (int j = 0; j < N; ++j) same |= __ballot(f.k[j] == v) & __ballot((f.v[j] & ~kExpanded) == id);
  return same != 0ull;
}
// Inserts (v, id) unless the id is already in the set (a neighbour met again after the lossy
// visited filter forgot it).  Returns 0 = inserted, 1 = inserted next to an equal key of
// another id, 2 = already present, nothing done.  Wavefront-uniform.
// With a[-1] the last key of the lane below, the new key at sorted position j is the median
// of (a[j-1], v, a[j]): a[j] where v is not below it, a[j-1] where v is below that too, else
// v itself; the ids follow the same two comparisons.  Equal keys keep their order of arrival.
template <int NS>
__device__ __forceinline__ int frontier_insert(Frontier<NS>& f, float v, uint32_t id, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  const bool any_eq = frontier_has_key<NS>(f, v);
  const bool dup = any_eq && frontier_has<NS>(f, v, id);
  // (one exit: early returns out of an inlined function inside the caller's loops cost the
  // caller a good deal of scalar control flow)
  if (!dup) {
    // last entry of the lane below (lane 0: "-inf", never taken over)
    const float prev_k = __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp((int)0xFF800000u, __builtin_bit_cast(int, f.k[N - 1]), 0x138, 0xF, 0xF, false));
    const uint32_t prev_v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)f.v[N - 1], 0x138, 0xF, 0xF, false);
    bool below[N + 1];  // below[j + 1]: v sorts before a[j]; below[0]: before the lane below's last
    below[0] = v < prev_k;
#pragma unroll
    for (int j = 0; j < N; ++j) below[j + 1] = v < f.k[j];
#pragma unroll
    for (int j = N - 1; j >= 0; --j) {
      const float lo_k = j > 0 ? f.k[j - 1] : prev_k;
      const uint32_t lo_v = j > 0 ? f.v[j - 1] : prev_v;
      f.k[j] = __builtin_amdgcn_fmed3f(lo_k, v, f.k[j]);
      f.v[j] = below[j + 1] ? (below[j] ? lo_v : id) : f.v[j];
    }
  }
  return dup ? 2 : (any_eq ? 1 : 0);
}
// The same shift for a key that is known to differ from every key of the set (the caller has looked).
template <int NS>
__device__ __forceinline__ void frontier_insert_distinct(Frontier<NS>& f, float v, uint32_t id) {
  constexpr int N = NS > 0 ? NS : 1;
  const float prev_k = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp((int)0xFF800000u, __builtin_bit_cast(int, f.k[N - 1]), 0x138, 0xF, 0xF, false));
  const uint32_t prev_v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)f.v[N - 1], 0x138, 0xF, 0xF, false);
#pragma unroll
  for (int j = N - 1; j >= 0; --j) {
    const float lo_k = j > 0 ? f.k[j - 1] : prev_k;
    const uint32_t lo_v = j > 0 ? f.v[j - 1] : prev_v;
    const bool before_this = v < f.k[j], before_lower = v < lo_k;
    f.k[j] = __builtin_amdgcn_fmed3f(lo_k, v, f.k[j]);
    f.v[j] = before_this ? (before_lower ? lo_v : id) : f.v[j];
  }
}
// Largest value of this lane and those below.
__device__ __forceinline__ int max_so_far(int x) {
  auto take = [&](int from) __attribute__((always_inline)) { x = from > x ? from : x; };
  take(__builtin_amdgcn_update_dpp(x, x, 0x111, 0xF, 0xF, false));  // row_shr:1 (lanes without a source keep their own)
  take(__builtin_amdgcn_update_dpp(x, x, 0x112, 0xF, 0xF, false));  // row_shr:2
  take(__builtin_amdgcn_update_dpp(x, x, 0x114, 0xF, 0xF, false));  // row_shr:4
  take(__builtin_amdgcn_update_dpp(x, x, 0x118, 0xF, 0xF, false));  // row_shr:8
  take(__builtin_amdgcn_update_dpp(x, x, 0x142, 0xA, 0xF, false));  // row_bcast:15 into rows 1 and 3
  take(__builtin_amdgcn_update_dpp(x, x, 0x143, 0xC, 0xF, false));  // row_bcast:31 into rows 2 and 3
  return x;
}
__device__ __forceinline__ int least_of_all_ints(int x) {
  auto take = [&](int from) __attribute__((always_inline)) { x = from < x ? from : x; };
  take(__builtin_amdgcn_update_dpp(x, x, 0x111, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(x, x, 0x112, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(x, x, 0x114, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(x, x, 0x118, 0xF, 0xF, false));
  take(__builtin_amdgcn_update_dpp(x, x, 0x142, 0xA, 0xF, false));
  take(__builtin_amdgcn_update_dpp(x, x, 0x143, 0xC, 0xF, false));
  return __builtin_amdgcn_readlane(x, 63);
}
// Several offers of a list at once: those of the lanes in `offers` (fewer than 64; not SPARSE: the first lanes, and +inf in
// the others), whose list lies in ids / keys (LDS), into a set of `size` entries; what does not fit behind ef entries falls off its end.  The offers are put
// in order (in ids / keys), every entry finds by halving how many of them go before it, and entries and offers go to their
// new places through LDS.  `room`: 64 * (NS + 1) words of LDS, whose contents are put back.  Returns false, with nothing
// done, if an offer has the key of another or of an entry (or its node is in the set already), also if one of the two is the
// set's last then and the other the first to fall off (hnswlib expands both, and its heap says which one leaves), or if the
// set's largest key would not stay above `above`: those go in one by one, by the rules for them.  last_key: the set's largest
// key afterwards.
// (An insert of its own is 39 instructions at ef 300 and 0.2 us of latency, this 200 for 14 offers.  Counting for each entry
// and each offer what goes before it, offer by offer, was 45 instructions an offer: one query on 100 000 x 50 284 -> 272 us,
// 1 000 queries there 636 -> 607, of which the full set's share below is half; 1 M x 96, ef 256, 100 000 queries 9.92 ->
// 9.80 ms.)
template <int NS, bool SPARSE>
__device__ __forceinline__ bool frontier_insert_all(Frontier<NS>& f, unsigned long long offers, int size, int ef, float my_key, uint32_t my_id,
                                                    uint32_t* ids, float* keys, uint32_t* room, float above, float& last_key, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  lane = fresh(lane);
  const int n = __popcll(offers);
  if (SPARSE) {  // the offers first, in their order
    const int pos = lanes_below(offers);
    wave_sync();
    if (__builtin_amdgcn_inverse_ballot_w64(offers)) {
      keys[pos] = my_key;
      ids[pos] = my_id;
    }
    wave_sync();
  }
  const float listed_key = SPARSE ? (lane < n ? keys[lane] : INFINITY) : my_key;
  const uint32_t listed_id = SPARSE ? ids[lane] : my_id;
  int less = 0;  // offers before this lane's
  for (int i = 0; i < n; i += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // (past the last offer: +inf, which goes before nothing)
      const float key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, listed_key), i + u));
      less += key < listed_key ? 1 : 0;
    }
  }
  uint32_t kept[N + 1];
#pragma unroll
  for (int j = 0; j <= N; ++j) kept[j] = room[64 * j + lane];
  wave_sync();
  keys[lane] = lane < n ? -INFINITY : INFINITY;
  room[lane] = 0u;
  wave_sync();
  if (lane < n) {
    keys[less] = listed_key;
    ids[less] = listed_id;
  }
  wave_sync();
  const float offer_key = keys[lane];  // in order from here on: lane r has the r-th
  bool done = __ballot(offer_key == -INFINITY) == 0ull;  // (two equal offers went to one place and left another empty)
  if (done) {
    int before[N];  // offers that go before each of this lane's entries
#pragma unroll
    for (int j = 0; j < N; ++j) before[j] = 0;
    for (int half = 1 << (31 - __builtin_clz(n)); half > 0; half >>= 1) {
      float probe[N];
#pragma unroll
      for (int j = 0; j < N; ++j) probe[j] = keys[before[j] + half - 1];
#pragma unroll
      for (int j = 0; j < N; ++j) before[j] += probe[j] < f.k[j] ? half : 0;
    }
    // an offer's place: as many entries go before it as have no more offers before them than it has.  The last entry of
    // each such number says how many there are up to it (the others write where nobody looks).
    const int next_first = __builtin_amdgcn_update_dpp(-1, before[0], 0x130, 0xF, 0xF, false);  // wave_shl:1
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int after = j + 1 < N ? before[j + 1 < N ? j + 1 : 0] : next_first;
      room[after != before[j] ? before[j] : 64 + lane] = (uint32_t)(lane * N + j + 1);
    }
    wave_sync();
    const int place = max_so_far((int)room[lane]) + lane;
    wave_sync();
#pragma unroll
    for (int j = 0; j < N; ++j) room[lane * N + j + before[j]] = __float_as_uint(f.k[j]);
    if (lane < n) room[place] = __float_as_uint(offer_key);
    wave_sync();
    // an offer equal to an entry comes right beside it (the padding on both sides is infinite)
    unsigned long long twins = 0ull;
#pragma unroll
    for (int j = 0; j < N; ++j) f.k[j] = __uint_as_float(room[lane * N + j]);
    const float last = uni(__uint_as_float(room[64 * N - ef + (size + n < ef ? size + n : ef) - 1]));
    if (SPARSE) {
      // (those that fall off included, as far as they are no farther than the set's last: candidates all the same.  Equal
      // entries that were there before are none of its business.)
      twins = __ballot(lane < n && offer_key <= last && place > 0 && __uint_as_float(room[place > 0 ? place - 1 : 0]) == offer_key);
    } else {
      const float prev_last = __builtin_bit_cast(
          float, __builtin_amdgcn_update_dpp((int)0xFF800000u, __builtin_bit_cast(int, f.k[N - 1]), 0x138, 0xF, 0xF, false));  // wave_shr:1
#pragma unroll
      for (int j = 0; j < N; ++j)
        twins |= __ballot(f.k[j] == (j > 0 ? f.k[j > 0 ? j - 1 : 0] : prev_last)) & __ballot(__builtin_fabsf(f.k[j]) < INFINITY);
    }
    // (the comparison holds wherever `above` is -inf; without it the instances for six keys a lane and rows of 65 to 128
    // elements spill five registers more and reload some in the hop loop: 200 000 x 128, ef 330, 40 000 queries 7.51 -> 7.85 ms)
    done = twins == 0ull && last > above;
    if (!done) {
#pragma unroll
      for (int j = 0; j < N; ++j) f.k[j] = __uint_as_float(room[lane * N + j + before[j]]);
    } else {
      wave_sync();
#pragma unroll
      for (int j = 0; j < N; ++j) room[lane * N + j + before[j]] = f.v[j];
      if (lane < n) room[place] = ids[lane];
      wave_sync();
#pragma unroll
      for (int j = 0; j < N; ++j) f.v[j] = room[lane * N + j];
      last_key = last;
    }
  }
  wave_sync();
#pragma unroll
  for (int j = 0; j <= N; ++j) room[64 * j + lane] = kept[j];
  if (!done) {  // (the list as it was)
    keys[lane] = my_key;
    ids[lane] = my_id;
  }
  wave_sync();
  return done;
}
template <int NS>
__device__ __forceinline__ float frontier_max(const Frontier<NS>& f) {
  constexpr int N = NS > 0 ? NS : 1;
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f.k[N - 1]), 63));
}
// closest (far: farthest) entry not yet expanded: marks it and returns its id, or -1 when none
// is left.  The farthest one is what the reference expands with its reverse_cand option
// (GetCand, cpp/include/cuda_utils_kernels.cuh:104-151).
template <int NS>
__device__ __forceinline__ int frontier_take(Frontier<NS>& f, int lane, bool far = false) {
  constexpr int N = NS > 0 ? NS : 1;
  uint32_t vf = kEmpty;
  int L;
  if (!far) {
#pragma unroll
    for (int j = N - 1; j >= 0; --j) vf = (f.v[j] & kExpanded) == 0u ? f.v[j] : vf;
    const unsigned long long mask = __ballot((vf & kExpanded) == 0u);
    if (mask == 0ull) return -1;
    L = __builtin_ctzll(mask);
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) vf = (f.v[j] & kExpanded) == 0u ? f.v[j] : vf;
    const unsigned long long mask = __ballot((vf & kExpanded) == 0u);
    if (mask == 0ull) return -1;
    L = 63 - __builtin_clzll(mask);
  }
  const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)vf, L);
  // (an id is in the set once: the entry that holds it is the one taken, whichever lane that is)
#pragma unroll
  for (int j = 0; j < N; ++j) f.v[j] = f.v[j] == id ? (id | kExpanded) : f.v[j];
  return (int)id;
}
// The (at most `want`) closest entries not yet expanded, all at once: marks them and writes them to out (LDS), closest
// first.  Returns how many there are.
template <int NS>
__device__ __forceinline__ int frontier_take_many(Frontier<NS>& f, int want, HeapEnt* out, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  int rank = 0;  // waiting entries in the lanes below, then in this lane's slots below
  int total = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const unsigned long long open = __ballot((int)f.v[j] >= 0);
    total += __popcll(open);
    rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned int)(open >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)open, (unsigned int)rank));
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const bool open = (int)f.v[j] >= 0;
    if (open && rank < want) {
      HeapEnt e;
      e.key = f.k[j];
      e.id = f.v[j];
      out[rank] = e;
      f.v[j] |= kExpanded;
    }
    rank += open ? 1 : 0;
  }
  wave_sync();
  return total < want ? total : want;
}
// frontier_insert_all<SPARSE> for the wavefront that searches in a team, where latency is all that counts and LDS there is: every entry and
// every offer is compared with all offers, four keys to an LDS read (halving, a trip to LDS per step, or reading the
// keys from lanes, a scalar hazard each, takes twice as long); keys and ids move together, and the set stays as it is in its
// registers until the outcome is known.  Of several offers of one node one counts.  room: 128 * (NS + 1) words.
template <int NS>
__device__ __forceinline__ bool frontier_merge(Frontier<NS>& f, unsigned long long offers, int size, int ef, float my_key, uint32_t my_id,
                                               uint32_t* room, float above, int& count, float& last_key, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  int less = 0;   // offers before this lane's
  int before[N];  // offers before each of this lane's entries
  int n, entries;
  bool mine, equal;
  while (true) {
    n = __popcll(offers);
    mine = __builtin_amdgcn_inverse_ballot_w64(offers);
    float* const keys = reinterpret_cast<float*>(room);
    keys[lane] = INFINITY;
    wave_sync();
    if (mine) keys[lanes_below(offers)] = my_key;
    wave_sync();
    less = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) before[j] = 0;
    for (int i = 0; i < n; i += 4) {
      const float4 k = reinterpret_cast<const float4*>(keys)[i >> 2];
      less += k.x < my_key ? 1 : 0;
      less += k.y < my_key ? 1 : 0;
      less += k.z < my_key ? 1 : 0;
      less += k.w < my_key ? 1 : 0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        before[j] += k.x < f.k[j] ? 1 : 0;
        before[j] += k.y < f.k[j] ? 1 : 0;
        before[j] += k.z < f.k[j] ? 1 : 0;
        before[j] += k.w < f.k[j] ? 1 : 0;
      }
    }
    wave_sync();
    // how many entries go before an offer that has so many offers before it (as in frontier_insert_all); and the offers in order,
    // where one of two equal ones leaves a place empty
    const int next_first = __builtin_amdgcn_update_dpp(-1, before[0], 0x130, 0xF, 0xF, false);  // wave_shl:1
    uint32_t* const nth = room + 128;
    room[lane] = 0u;
    nth[lane] = 64u;
    wave_sync();
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int after = j + 1 < N ? before[j + 1 < N ? j + 1 : 0] : next_first;
      room[after != before[j] ? before[j] : 64 + lane] = (uint32_t)(lane * N + j + 1);
    }
    if (mine) nth[less] = (uint32_t)lane;
    wave_sync();
    entries = max_so_far((int)room[lane]);
    const uint32_t at_place = nth[lane], first = nth[mine ? less : 0];
    equal = __ballot(lane < n && at_place == 64u) != 0ull;
    if (__builtin_expect(!equal, 1)) break;
    const uint32_t first_id = (uint32_t)__shfl((int)my_id, (int)first, 64);
    const unsigned long long again = __ballot(first != (uint32_t)lane && first_id == my_id) & offers;
    if (again == 0ull) break;
    offers &= ~again;
    wave_sync();
  }
  bool done = false;
  if (!equal && n < 64) {
    const int place = __shfl(entries, less, 64) + less;
    wave_sync();
    HeapEnt* const to = reinterpret_cast<HeapEnt*>(room);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      HeapEnt e;
      e.key = f.k[j];
      e.id = f.v[j];
      to[lane * N + j + before[j]] = e;
    }
    if (mine) {
      HeapEnt e;
      e.key = my_key;
      e.id = my_id;
      to[place] = e;
    }
    wave_sync();
    HeapEnt now[N];
#pragma unroll
    for (int j = 0; j < N; ++j) now[j] = to[lane * N + j];
    const float last = uni(to[64 * N - ef + (size + n < ef ? size + n : ef) - 1].key);
    const float next_to = to[mine && place > 0 ? place - 1 : 0].key;
    // (an offer equal to an entry comes right behind it; those that fall off count as far as they are no farther than the last)
    done = __ballot(mine && my_key <= last && place > 0 && next_to == my_key) == 0ull && last > above;
    if (done) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        f.k[j] = now[j].key;
        f.v[j] = now[j].id;
      }
      last_key = last;
      count = n;
    }
    wave_sync();
  }
  return done;
}
// For a team (team_help): the eight closest entries not yet expanded to the first places of its line, the 24 next
// ones behind them.  None is marked; returns how many there are in all, rank: waiting entries in the lanes below.  (All
// writes are unconditional, to a place that nobody reads where there is nothing to write: no exec-mask branches.)
template <int NS>
__device__ __forceinline__ int frontier_line_up(const Frontier<NS>& f, const Team& team, int& rank, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  HeapEnt* const line = team.line();
  int total = 0;
  rank = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const unsigned long long open = __ballot((int)f.v[j] >= 0);
    total += __popcll(open);
    rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned int)(open >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)open, (unsigned int)rank));
  }
  int at = rank;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const bool open = (int)f.v[j] >= 0;
    HeapEnt e;
    e.key = f.k[j];
    e.id = f.v[j];
    line[open && at < Team::kInLine ? at : Team::kInLine] = e;
    at += open ? 1 : 0;
  }
  if (total < Team::kInLine && lane >= total && lane < Team::kInLine) {
    HeapEnt none;
    none.key = INFINITY;
    none.id = kEmpty;
    line[lane] = none;
  }
  wave_sync();
  return total;
}
// marks the `count` closest entries not yet expanded
template <int NS>
__device__ __forceinline__ void frontier_take_first(Frontier<NS>& f, int count, int rank) {
  constexpr int N = NS > 0 ? NS : 1;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const bool open = (int)f.v[j] >= 0;
    f.v[j] |= open && rank < count ? kExpanded : 0u;
    rank += open ? 1 : 0;
  }
}
// key of the entry with this id (which is in the set)
template <int NS>
__device__ __forceinline__ float frontier_key_of(const Frontier<NS>& f, uint32_t id) {
  constexpr int N = NS > 0 ? NS : 1;
  float kf = 0.f;
  bool hit = false;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const bool h = (f.v[j] & ~kExpanded) == id;
    kf = h ? f.k[j] : kf;
    hit = hit || h;
  }
  const unsigned long long mask = __ballot(hit);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, kf), __builtin_ctzll(mask | (1ull << 63))));
}
// is there an entry not yet expanded with exactly this key?
template <int NS>
__device__ __forceinline__ bool frontier_open_key(const Frontier<NS>& f, float key) {
  constexpr int N = NS > 0 ? NS : 1;
  bool hit = false;
#pragma unroll
  for (int j = 0; j < N; ++j) hit = hit || ((f.v[j] & kExpanded) == 0u && f.k[j] == key);
  return __ballot(hit) != 0ull;
}
// do the two largest keys of a full set coincide?
template <int NS>
__device__ __forceinline__ bool frontier_max_twice(const Frontier<NS>& f) {
  constexpr int N = NS > 0 ? NS : 1;
  const float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f.k[N - 1]), 63));
  const float b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f.k[N > 1 ? N - 2 : 0]), 63));
  return a == b;
}
// do two neighbouring keys coincide among sorted positions p, p+1 with from <= p < upto and p+1 < count?
template <int NS>
__device__ __forceinline__ bool frontier_tie_within(const Frontier<NS>& f, int ef, int upto, int count, int lane,
                                                    int from = 0) {
  constexpr int N = NS > 0 ? NS : 1;
  const float next_first = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, f.k[0]), 0x130, 0xF, 0xF, false));  // wave_shl:1
  bool hit = false;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int pos = lane * N + j - (64 * N - ef);
    const float nxt = j + 1 < N ? f.k[j + 1 < N ? j + 1 : 0] : next_first;
    hit = hit || (pos >= from && pos < upto && pos + 1 < count && f.k[j] == nxt);
  }
  return __ballot(hit) != 0ull;
}
// The waiting (not yet expanded) entries whose key coincides with a neighbour's: while the tie-free loop runs on a
// set that holds equal keys, these are the entries it must not expand or push out by itself.
struct TieWatch {
  int id0 = -1, id1 = -1, id2 = -1, id3 = -1;  // (-1: unused; no taken candidate compares equal)
  float hi = -INFINITY;                        // their largest key
};
// Fills w; false when there are more than four such entries.
template <int NS>
__device__ __forceinline__ bool frontier_watch_list(const Frontier<NS>& f, TieWatch& w) {
  constexpr int N = NS > 0 ? NS : 1;
  const float prev_last = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp((int)0xFF800000u, __builtin_bit_cast(int, f.k[N - 1]), 0x138, 0xF, 0xF, false));  // wave_shr:1
  const float next_first = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp((int)0xFF800000u, __builtin_bit_cast(int, f.k[0]), 0x130, 0xF, 0xF, false));  // wave_shl:1
  unsigned long long m[N];
  int total = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float below = j > 0 ? f.k[j > 0 ? j - 1 : 0] : prev_last;
    const float above = j + 1 < N ? f.k[j + 1 < N ? j + 1 : 0] : next_first;
    m[j] = __ballot((f.v[j] & kExpanded) == 0u && (f.k[j] == below || f.k[j] == above));
    total += __popcll(m[j]);
  }
  w = TieWatch();
  if (total > 4) return false;
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    while (m[j] != 0ull) {
      const int L = __builtin_ctzll(m[j]);
      m[j] &= m[j] - 1ull;
      const int id = __builtin_amdgcn_readlane((int)f.v[j], L);
      const float key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f.k[j]), L));
      if (cnt == 0) w.id0 = id;
      else if (cnt == 1) w.id1 = id;
      else if (cnt == 2) w.id2 = id;
      else w.id3 = id;
      w.hi = uni(fmaxf(w.hi, key));
      cnt += 1;
    }
  }
  return true;
}
// takes the expanded mark off an entry again
template <int NS>
__device__ __forceinline__ void frontier_untake(Frontier<NS>& f, uint32_t id) {
  constexpr int N = NS > 0 ? NS : 1;
#pragma unroll
  for (int j = 0; j < N; ++j) f.v[j] = f.v[j] == (id | kExpanded) ? id : f.v[j];
}
// writes the sorted entries [0, count) to out_id / out_key (LDS)
template <int NS>
__device__ __forceinline__ void frontier_dump(const Frontier<NS>& f, int ef, int count, uint32_t* out_id, float* out_key,
                                              int lane) {
  constexpr int N = NS > 0 ? NS : 1;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int pos = lane * N + j - (64 * N - ef);
    if (pos >= 0 && pos < count) {
      out_id[pos] = f.v[j] & ~kExpanded;
      out_key[pos] = f.k[j];
    }
  }
}

// The reference's reverse_cand search (expand the farthest waiting candidate, GetCand(..., reverse),
// cpp/include/cuda_utils_kernels.cuh:104-151) for result sets beyond the register set's capacity: one sorted list in
// LDS (s.top, ef entries, ascending; bit 31 of the id = expanded), equal keys in order of arrival, the last entry
// leaves a full list.  An insert counts the keys not above the new one (the list is sorted: whole chunks of 64
// until the first that is not) and moves the tail up one place, 64 entries at a time from the top; the next
// candidate is the last entry without the mark.  Exact visited bitmap.  A list of a thousand entries makes an
// insert a few dozen LDS round trips: the option is there for completeness, not for speed.  On entry
// s.nbuf[0..n_seed) holds the seeds (marked visited); on exit s.top[0..st.top_size) is the result in order.
template <int DT, int QR>
__device__ __forceinline__ void search_level_far_lds(const DevIndex& ix, const QVec<QR>& qv, int level, int ef, Scratch& s,
                                                     SearchState& st, int n_seed, int lane) {
  HeapEnt* set = s.top;
  const int S = row_stride(ix, level);
  int size = 0;
  int n = n_seed;
  while (true) {
    if (n > 0) dist_list<DT, QR, false>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
    st.n_dist += n;
    wave_sync();
    for (int j = 0; j < n; ++j) {
      const float key = s.dbuf[j];   // (the same address in every lane)
      const uint32_t id = s.nbuf[j];
      const float last_key = size > 0 ? set[size - 1].key : INFINITY;
      if (size < ef || last_key > key) {
        // where it goes: after every entry whose key is not above it
        int p = 0;
        for (int base = 0; base < size; base += 64) {
          const int i = base + lane;
          const unsigned long long le = __ballot(i < size && set[i < size ? i : 0].key <= key);
          p += __popcll(le);
          if (__popcll(le) < (size - base < 64 ? size - base : 64)) break;
        }
        const int new_size = size < ef ? size + 1 : ef;
        // entries [p, new_size - 1) move up one place, the topmost chunk first (each chunk is read whole
        // before it is written)
        for (int hi = new_size - 1; hi > p; hi -= 64) {
          const int dst = hi - lane;
          HeapEnt e = set[dst > p ? dst - 1 : p];
          wave_sync();
          if (dst > p) set[dst] = e;
          wave_sync();
        }
        if (lane == 0) {
          HeapEnt e;
          e.key = key;
          e.id = id;
          set[p] = e;
        }
        wave_sync();
        size = new_size;
      }
    }
    // the farthest entry still waiting
    int pick = -1;
    for (int hi = size - 1; hi >= 0 && pick < 0; hi -= 64) {
      const int i = hi - lane;
      const unsigned long long open = __ballot(i >= 0 && (set[i >= 0 ? i : 0].id & kExpanded) == 0u);
      if (open != 0ull) pick = hi - __builtin_ctzll(open);
    }
    if (pick < 0) break;
    const uint32_t cid = set[pick].id;
    wave_sync();
    if (lane == 0) set[pick].id = cid | kExpanded;
    st.n_hops += 1;
    n = visit_row(link_row(ix, cid, level), S, s, st, lane);
    wave_sync();
  }
  st.top_size = size;
}

// The sorted-set search's visited filter: a four-way set-associative tag cache in LDS alone, no
// bitmap.  A set is one 64-bit word holding four 16-bit tags (set = low id bits, tag = the
// rest; 0xFFFF = empty); a new tag pushes the oldest of the four out.  A hit is exact ("seen
// before"), a miss may be a node whose tag has been pushed out since: it is then evaluated
// again, which changes nothing — if it is still in the set the insert finds it, and if it was
// rejected or evicted its key is still not below the bound.  No atomics, no global memory,
// nothing to undo.  s.vcache / s.filter hold the table and its shape.
// (Four ways rather than two at the same size: on the 1.18 M-point set the neighbourhoods
// overlap so much that most forgotten nodes were victims of set conflicts, not of capacity —
// repeated evaluations fell from 31 % to 12 % of the distinct ones.)
__device__ __forceinline__ void filter_reset(Scratch& s, int lane, int lanes = 64) {
  uint4* c4 = reinterpret_cast<uint4*>(s.vcache);
  const int n4 = (s.filter.sets() + 1) >> 1;  // 2 sets per 16 bytes
  for (int i = lane; i < n4; i += lanes) {
    const uint32_t a = filter_empty_tag(s.filter, 2u * (uint32_t)i) * 0x10001u, b = filter_empty_tag(s.filter, 2u * (uint32_t)i + 1u) * 0x10001u;
    c4[i] = make_uint4(a, a, b, b);
  }
  wave_sync();
}
__device__ __forceinline__ uint2 filter_push(uint2 w, uint32_t place) {
  return make_uint2(__builtin_amdgcn_alignbit(w.x, place << 16, 16), (w.y << 16) | (w.x >> 16));
}
// the lanes whose tag is not among the four of their set
__device__ __forceinline__ unsigned long long filter_misses(uint2 w, uint32_t place) {
  const uint16_t tag = (uint16_t)place;
  return __ballot((uint16_t)w.x != tag) & __ballot((uint16_t)(w.x >> 16) != tag) & __ballot((uint16_t)w.y != tag) &
         __ballot((uint16_t)(w.y >> 16) != tag);
}
// Compacts the ids of a link row that the filter does not know into s.nbuf; returns how many.
template <bool WIDE>
__device__ __forceinline__ int visit_lossy_t(const uint32_t* row, int S, Scratch& s, int lane) {
  int n = 0;
  uint2* sets = reinterpret_cast<uint2*>(s.vcache);
  for (int base = 0; base < S; base += 64) {
    const uint32_t got = row[base + lane < S ? base + lane : 0];  // unconditional load, then a select
    const uint32_t id = (base + lane < S) ? got : kEmpty;
    // (every lane looks its set up — an empty slot's "id" has some set too — so that the only predicated part is the two
    // LDS writes at the end)
    const uint32_t place = filter_place<WIDE>(id);
    const uint32_t slot = filter_set<WIDE>(s.filter, place);
    const uint2 w = sets[slot];
    const unsigned long long mask = __ballot(id != kEmpty) & filter_misses(w, place);
    if (__builtin_amdgcn_inverse_ballot_w64(mask)) {
      sets[slot] = filter_push(w, place);
      s.nbuf[n + lanes_below(mask)] = id;
    }
    n += __popcll(mask);
  }
  return n;
}
__device__ __forceinline__ int visit_lossy(const uint32_t* row, int S, Scratch& s, int lane) {
  if (__builtin_expect(s.filter.more_bits() != 0, 0)) return visit_lossy_t<true>(row, S, s, lane);
  return visit_lossy_t<false>(row, S, s, lane);
}
// an id's place and its set
__device__ __forceinline__ uint32_t filter_find(FilterShape f, uint32_t id, uint32_t& slot) {
  const uint32_t place = f.more_bits() != 0 ? filter_place<true>(id) : filter_place<false>(id);
  slot = filter_set<true>(f, place);
  return place;
}
// the lanes whose id the filter does not know; enters the ids of the lanes in `which` (where two of them fall into one set one is forgotten)
__device__ __forceinline__ unsigned long long filter_unknown(const Scratch& s, uint32_t id) {
  uint32_t set;
  const uint32_t place = filter_find(s.filter, id, set);
  return filter_misses(reinterpret_cast<const uint2*>(s.vcache)[set], place);
}
__device__ __forceinline__ void filter_enter(Scratch& s, uint32_t id, unsigned long long which) {
  uint2* sets = reinterpret_cast<uint2*>(s.vcache);
  uint32_t set;
  const uint32_t place = filter_find(s.filter, id, set);
  const uint2 w = sets[set];
  if (__builtin_amdgcn_inverse_ballot_w64(which)) sets[set] = filter_push(w, place);
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void visit_lossy_single(Scratch& s, uint32_t id, int lane) {
  if (lane == 0) {
    uint2* sets = reinterpret_cast<uint2*>(s.vcache);
    uint32_t slot;
    const uint32_t place = filter_find(s.filter, id, slot);
    sets[slot] = filter_push(sets[slot], place);
  }
}

// The link rows of `rows` (at most K) candidates, lane r of `cands` holding the r-th one's id, looked up and entered in
// the filter one after the other -- so that a node two of them link to is in the first one's list only -- with all of
// their fetches in flight at once.  Compacts like visit_lossy; ends gets the end of each row's list, eight bits each.  At
// most 64 ids in all: the rows that do not fit are left out (returns how many are in).  S <= 64.
template <int K, bool WIDE>
__device__ __forceinline__ int visit_lossy_rows_t(const DevIndex& ix, uint32_t cands, int rows, int level, int S, Scratch& s,
                                                  int& n_ids, unsigned long long& ends, int lane) {
  static_assert(K <= 8, "eight ends in 64 bits");
  uint2* sets = reinterpret_cast<uint2*>(s.vcache);
  uint32_t got[K];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    got[r] = kEmpty;
    if (r < rows) got[r] = scalar_base(link_row(ix, (uint32_t)__builtin_amdgcn_readlane((int)cands, r), level))[lane < S ? lane : 0];
  }
  int n = 0, in = rows;
  ends = 0ull;
#pragma unroll
  for (int r = 0; r < K; ++r) {
    if (r < in) {
      const uint32_t id = lane < S ? got[r] : kEmpty;
      const uint32_t place = filter_place<WIDE>(id);
      const uint32_t slot = filter_set<WIDE>(s.filter, place);
      const uint2 w = sets[slot];
      const unsigned long long mask = __ballot(id != kEmpty) & filter_misses(w, place);
      const int more = __popcll(mask);
      if (r > 0 && n + more > 64) {
        in = r;
      } else {
        if (__builtin_amdgcn_inverse_ballot_w64(mask)) {
          sets[slot] = filter_push(w, place);
          s.nbuf[n + lanes_below(mask)] = id;
        }
        __builtin_amdgcn_wave_barrier();
        n += more;
        ends |= (unsigned long long)n << (8 * r);
      }
    }
  }
  n_ids = n;
  return in;
}
template <int K>
__device__ __forceinline__ int visit_lossy_rows(const DevIndex& ix, uint32_t cands, int rows, int level, int S, Scratch& s,
                                                int& n_ids, unsigned long long& ends, int lane) {
  if (__builtin_expect(s.filter.more_bits() != 0, 0)) return visit_lossy_rows_t<K, true>(ix, cands, rows, level, S, s, n_ids, ends, lane);
  return visit_lossy_rows_t<K, false>(ix, cands, rows, level, S, s, n_ids, ends, lane);
}
// ---- a query that a team of wavefronts searches ---------------------------------------------------------------
// A batch that leaves the machine idle is bound by the chain of its slowest search: fetch the next candidates' link rows, fetch the
// vectors of their new nodes, put those into the set, choose the next candidates.  The first two are memory latency and
// arithmetic that nothing but the choice of the candidates waits for, and the choice is mostly known ahead: of the 300
// candidates that a search expands at ef 300, 274 are among the next sixteen in line two steps before their turn (60 000 x 50; 102 of
// 128 at ef 128 on integers).  So one wavefront of a workgroup makes the search; in every step it says which candidates are the next
// in line, and the others fetch their link rows and evaluate the nodes that have not been dealt with, ahead of time.  A
// candidate whose list is there when its turn comes costs neither fetch; one whose list is not is evaluated by the
// search itself.  The search's decisions, and what it returns, are its own either way: a list holds every node of the link
// row but those whose offers it has dealt with for good, with the keys it would have computed.  A helper that
// finds a node closer than the candidate it came from goes on with that node, which will be the next candidate.
// (Cycles of a step of one query on 100 000 x 50 at ef 300, a wavefront alone: distances 1 150, the set 2 200, candidates, links and
// filter 2 090, 112 steps; the search by a team has 69 of them, of which 13 evaluate nodes of their own.)
//
// Slots: team_slots.h.  (Ids are below 2^28 where there is a visited filter.)  A helper takes a free slot of the candidate's
// bucket by compare-and-swap, then looks whether the candidate is still in line and in no other slot (the search writes the line
// before it looks for lists: one of the two sees the other), and gives the slot back otherwise.  Only the search frees a slot
// whose list is there.  LDS operations of a wavefront are carried out in order.
static_assert(kSlotMaking == kExpanded && kNoSlot == kEmpty, "as the ids in the line and in link rows");
__device__ __forceinline__ void lds_done() {  // everything this wavefront wrote to LDS is there
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint32_t lds_now(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void lds_tell(uint32_t* p, uint32_t x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
// The slots of a node's bucket.  there: the slot its list is in, or -1; eights: of nodes there; making: its list is being made;
// room: a free slot, or -1.
struct TeamPlace {
  int there, eights, room;
  bool making;
};
__device__ __forceinline__ TeamPlace team_look(const Team& team, uint32_t id) {
  const int first = 4 * (int)team.bucket(id);
  wave_sync();
  const uint4 now = *reinterpret_cast<const uint4*>(team.owner() + first);
  const uint32_t o[4] = {now.x, now.y, now.z, now.w};
  TeamPlace t;
  t.there = t.room = -1;
  t.eights = 0;
  t.making = false;
#pragma unroll
  for (int w = 3; w >= 0; --w) {
    const bool mine = slot_is_of(o[w], id);
    t.there = mine ? first + w : t.there;
    t.eights = mine ? slot_eights(o[w]) : t.eights;
    t.making = t.making || o[w] == (id | kSlotMaking);
    t.room = o[w] == kNobody ? first + w : t.room;
  }
  return t;
}

// Frees the slots of candidates that are not in the line (pushed out of the set, or back in it).
__device__ __forceinline__ void team_tidy(const Team& team, int lane) {
  static_assert(kTeamSlots == 128, "two slots per lane");
  const TeamPlace t = team_look(team, lane < Team::kInLine ? team.line()[lane < Team::kInLine ? lane : 0].id : kEmpty);
  uint32_t* const kept = team.room();
  kept[lane] = kept[lane + 64] = 0u;
  wave_sync();
  if (t.there >= 0) kept[t.there] = 1u;
  wave_sync();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t owner = lds_now(team.owner() + lane + 64 * i);
    if (slot_holds_list(owner) && kept[lane + 64 * i] == 0u) lds_tell(team.owner() + lane + 64 * i, kNobody);
    __builtin_amdgcn_wave_barrier();
  }
  wave_sync();
}
// rows in flight (dist_list): sixteen, eight long ones (of 65 to 128 elements thirty-two would take the registers of a wavefront per SIMD)
template <int QR>
constexpr int team_wide() {
  return QR == 4 ? 3 : (QR == 1 ? 1 : 2);
}
// The search of one level is over and another's begins (LEVELS): nobody begins a list any more, those under way are waited
// for (a helper looks at the level again once it has its slot: it is seen here, or sees that it may not) -- and all slots are free.
__device__ __forceinline__ void team_close(const Team& team, int lane) {
  if (lane == 0) lds_tell(team.level(), lds_now(team.level()) | 1u);
  wave_sync();
  for (int i = 0; i < 2; ++i) {
    while (true) {
      const uint32_t owner = lds_now(team.owner() + lane + 64 * i);
      if (__ballot(slot_being_made(owner)) == 0ull) {
        if (slot_holds_list(owner)) lds_tell(team.owner() + lane + 64 * i, kNobody);
        __builtin_amdgcn_wave_barrier();
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
}
__device__ __forceinline__ void team_open(const Team& team, int level, int lane) {
  HeapEnt none;
  none.key = INFINITY;
  none.id = kEmpty;
  if (lane < Team::kInLine) team.line()[lane < Team::kInLine ? lane : 0] = none;
  wave_sync();
  if (lane == 0) lds_tell(team.level(), ((uint32_t)level << 16) | (((lds_now(team.level()) & 0xFFFFu) + 1u) & 0xFFFEu));
  wave_sync();
}
template <int DT, int QR, bool LEVELS = false>
__device__ __forceinline__ void team_help(const DevIndex& ix, const QVec<QR>& qv, const Scratch& s, int helper, int lane) {
  const Team& team = s.team;
  uint32_t next_at = 0u;  // and the level it was found on
  uint32_t next = kEmpty;  // the node to go on with, whose list nobody has asked for yet
  float next_key = 0.f;
  while (uni((int)lds_now(team.over())) == 0) {
    const uint32_t at = LEVELS ? (uint32_t)uni((int)lds_now(team.level())) : 0u;
    if (LEVELS && (at != next_at || (at & 1u) != 0u)) next = kEmpty;
    next_at = at;
    const int S = LEVELS ? row_stride(ix, (int)(at >> 16)) : ix.S0;
    uint32_t id = next;
    float key = next_key;
    int slot;
    if (LEVELS && (at & 1u) != 0u) {
      slot = -1;
    } else if (next == kEmpty) {
      const uint32_t* const wish = reinterpret_cast<const uint32_t*>(team.line() + (lane < Team::kInLine ? lane : 0));
      const float wish_key = __uint_as_float(lds_now(wish));
      const uint32_t wish_id = lds_now(wish + 1);
      const TeamPlace t = team_look(team, wish_id);
      unsigned long long open = __ballot(lane < Team::kInLine && wish_id != kEmpty && t.there < 0 && !t.making && t.room >= 0);
      // (helpers that look at the same time choose different wishes, as far as there are several)
      if (open != 0ull) {
        for (int skip = helper % __popcll(open); skip > 0; --skip) open &= open - 1ull;
        const int i = __builtin_ctzll(open);
        id = (uint32_t)__builtin_amdgcn_readlane((int)wish_id, i);
        key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wish_key), i));
        slot = __builtin_amdgcn_readlane(t.room, i);
      } else {
        slot = -1;
      }
    } else {
      const TeamPlace t = team_look(team, next);
      slot = uni(t.there < 0 && !t.making ? t.room : -1);
    }
    const bool asked = next == kEmpty;
    next = kEmpty;
    bool mine = false;
    if (slot >= 0) {
      if (lane == 0) {
        uint32_t was = kNobody;
        mine = __hip_atomic_compare_exchange_strong(team.owner() + slot, &was, id | kSlotMaking, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (uni(mine ? 1 : 0) != 0) {
      lds_done();
      const bool wished = __ballot(lane < Team::kInLine && lds_now(reinterpret_cast<const uint32_t*>(team.line() + (lane < Team::kInLine ? lane : 0)) + 1) == id) != 0ull;
      const int other = 4 * (int)team.bucket(id) + (lane & 3);
      const uint32_t there = lds_now(team.owner() + other);
      const bool twice = __ballot(other != slot && (slot_is_of(there, id) || there == (id | kSlotMaking))) != 0ull;
      const bool still = !LEVELS || (uint32_t)uni((int)lds_now(team.level())) == at;
      uint32_t say = kNobody;
      if ((wished || !asked) && !twice && still) {
        uint32_t* const ids = team.ids(slot);
        const uint32_t got = scalar_base(LEVELS ? link_row(ix, id, (int)(at >> 16)) : ix.links0 + (size_t)id * S)[lane < S ? lane : 0];
        const uint32_t node = lane < S ? got : kEmpty;
        const unsigned long long mask = __ballot(node != kEmpty) & filter_unknown(s, node);
        const int n = __popcll(mask);
        if (lane < S) ids[lane] = kEmpty;
        wave_sync();
        if (__builtin_amdgcn_inverse_ballot_w64(mask)) ids[lanes_below(mask)] = node;
        wave_sync();
        dist_list<DT, QR, false, team_wide<QR>()>(ix, qv, s.qlds, ids, n, team.keys(slot), lane);
        lds_done();
        say = slot_word(id, n);
        if (n > 0) {
          const float my_key = lane < n ? team.keys(slot)[lane < n ? lane : 0] : INFINITY;
          const float least = least_of_all(my_key);
          const unsigned long long at = __ballot(my_key == least);
          if (least < key && at != 0ull) {
            next = (uint32_t)uni((int)ids[__builtin_ctzll(at)]);
            next_key = least;
          }
        }
      }
      if (lane == 0) lds_tell(team.owner() + slot, say);
      __builtin_amdgcn_wave_barrier();
    } else if (slot < 0) {
      __builtin_amdgcn_s_sleep(1);
    }
  }
}

// Compacts the ids of a link row (of at most 64) that the filter does not know into s.nbuf, without telling it; returns how many.
__device__ __forceinline__ int visit_unmarked(const uint32_t* row, int S, Scratch& s, int lane) {
  const uint32_t got = row[lane < S ? lane : 0];
  const uint32_t id = lane < S ? got : kEmpty;
  const unsigned long long mask = __ballot(id != kEmpty) & filter_unknown(s, id);
  if (__builtin_amdgcn_inverse_ballot_w64(mask)) s.nbuf[lanes_below(mask)] = id;
  __builtin_amdgcn_wave_barrier();
  return __popcll(mask);
}
// The list of a candidate whose turn has come, if there is one: the nodes that the filter does not know, and their keys, to s.nbuf
// and s.dbuf, their number to n.
__device__ __forceinline__ bool visit_listed(Scratch& s, uint32_t cid, int S, int& n, int lane) {
  TeamPlace t = team_look(s.team, cid);
  for (int polls = 0; polls < 4096 && uni(t.there < 0 && t.making ? 1 : 0) != 0; ++polls) t = team_look(s.team, cid);
  const int where = uni(t.there);
  if (where >= 0) {
    const uint32_t got = s.team.ids(where)[lane < S ? lane : 0];
    const float key = s.team.keys(where)[lane < S ? lane : 0];
    const uint32_t id = lane < S ? got : kEmpty;
    uint2* sets = reinterpret_cast<uint2*>(s.vcache);
    uint32_t set;
    const uint32_t place = filter_find(s.filter, id, set);
    const uint2 w = sets[set];
    const unsigned long long mask = __ballot(id != kEmpty) & filter_misses(w, place);
    if (__builtin_amdgcn_inverse_ballot_w64(mask)) {
      sets[set] = filter_push(w, place);
      s.nbuf[lanes_below(mask)] = id;
      s.dbuf[lanes_below(mask)] = key;
    }
    __builtin_amdgcn_wave_barrier();
    n = __popcll(mask);
    if (lane == 0) lds_tell(s.team.owner() + where, kNobody);
    __builtin_amdgcn_wave_barrier();
  }
  return where >= 0;
}
// Takes the ids of the lanes that say so out of the filter again.  (Two of them may share a word: each makes its own half the
// set's empty tag with two atomics -- which may come twice for one id, listed twice where the filter lost it in between.)
__device__ __forceinline__ void filter_forget(Scratch& s, uint32_t id, bool mine) {
  uint2* sets = reinterpret_cast<uint2*>(s.vcache);
  if (mine) {
    uint32_t slot;
    const uint32_t tag = filter_find(s.filter, id, slot) & 0xFFFFu, empty = filter_empty_tag(s.filter, slot) * 0x10001u;
    const uint2 w = sets[slot];
    const uint32_t x = ((w.x & 0xFFFFu) == tag ? 0xFFFFu : 0u) | ((w.x >> 16) == tag ? 0xFFFF0000u : 0u);
    const uint32_t y = ((w.y & 0xFFFFu) == tag ? 0xFFFFu : 0u) | ((w.y >> 16) == tag ? 0xFFFF0000u : 0u);
    if (x) {
      __hip_atomic_fetch_and(&sets[slot].x, ~x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      __hip_atomic_fetch_or(&sets[slot].x, empty & x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
    if (y) {
      __hip_atomic_fetch_and(&sets[slot].y, ~y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      __hip_atomic_fetch_or(&sets[slot].y, empty & y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
  }
  __builtin_amdgcn_wave_barrier();
}

// The trail of a sorted-set search: the entries it accepted, hop by hop, wherever its course is certainly
// hnswlib's own.  A query that is given up afterwards is not searched again from its entry point: the
// literal pass takes the accepted entries of those hops from the trail — no link rows, no vectors, no
// arithmetic, only its queue and set operations in hnswlib's order — and searches on from where the trail
// ends.  One 16-byte record per accepted entry: (expanded node, accepted node, key bits, number of the hop);
// hops without an accepted entry leave none.  While equal keys wait side by side (a group that is followed
// through) the order of expansion may differ from hnswlib's and with it what each hop accepts: those hops are
// not recorded, two markers (kTrailOwn from hop h on, kTrailBack from hop h on) tell the literal pass to make
// them itself, in its own order; after such a group the set, the bound and the nodes met are the same again
// under either order, and so is what every later hop accepts.  The trail ends for good when the twins of an
// eviction come up (a node outside the set is expanded there).
constexpr uint32_t kTrailOwn = 0xFFFFFFFFu;
constexpr uint32_t kTrailBack = 0xFFFFFFFEu;
struct Trail {
  uint4* rec = nullptr;  // this search's records, or null: no trail is kept
  int cap = 0;
  int n = 0;         // records written; -1: the trail outgrew its buffer and is void
  int hops = 0;      // expansions the trail covers (all of them completed)
  int n_dist = 0;    // evaluations up to there
  bool on = false;   // still recording
  bool own = false;  // inside a stretch the literal pass makes itself
};
// (The wave barriers after the one-lane and some-lanes stores below emit nothing; they keep the end of such a
// branch a block of its own.  Merged into the join of the surrounding wavefront-uniform branches, it makes the
// compiler take every value that differs between those for lane-dependent -- the trail's state then sits in
// vector registers, of which the pass has none to spare.)
__device__ __forceinline__ void trail_mark(Trail& tr, uint32_t kind, int hop, int lane) {
  if (tr.on) {
    if (tr.n + 1 > tr.cap) {
      tr.on = false;
      tr.n = -1;
    } else {
      if (lane == 0) tr.rec[tr.n] = make_uint4(kind, 0u, 0u, (uint32_t)hop);
      __builtin_amdgcn_wave_barrier();
      tr.n += 1;
      tr.own = kind == kTrailOwn;
    }
  }
}
__device__ __forceinline__ void trail_hop(Trail& tr, unsigned long long accepted, int cid, int hop, uint32_t my_id,
                                          float my_key, int lane) {
  if (tr.on && !tr.own && accepted != 0ull && cid >= 0) {
    const int cnt = __popcll(accepted);
    if (tr.n + cnt > tr.cap) {
      tr.on = false;
      tr.n = -1;
    } else {
      if (__builtin_amdgcn_inverse_ballot_w64(accepted)) {  // (the lanes whose bit is set)
        tr.rec[tr.n + lanes_below(accepted)] = make_uint4((uint32_t)cid, my_id, __float_as_uint(my_key), (uint32_t)hop);
      }
      __builtin_amdgcn_wave_barrier();
      tr.n += cnt;
    }
  }
}
// the trail ends here: `hops` expansions are complete
__device__ __forceinline__ void trail_stop(Trail& tr, int hops, int n_dist) {
  if (tr.on) {
    tr.on = false;
    tr.hops = hops;
    tr.n_dist = n_dist;
  }
}

// The offers of one evaluation (the lanes of `todo`), in order, into a set that holds no equal keys that matter.  SEVERAL:
// they are those of a batch of candidates (tie_free_phase), each one's ending at its byte of `ends`; r and row_end follow
// the one under way, good is how many of them are expanded for good.  resume_at: the offer the rules for equal keys apply
// from.  (The search of a query far from its entry point accepts several offers per hop and is the last of its batch to end:
// what an accepted offer costs is latency, and a taken branch is twenty cycles of it -- hence the hints, and the insert in
// both arms.)
template <int NS, bool FULL, bool TRAILS, bool WATCH, bool BUILD, bool SEVERAL>
__device__ __forceinline__ void tie_free_offers(SearchState& st, Frontier<NS>& fr, unsigned long long todo, float my_key, uint32_t my_id,
                                                int ef, float w_hi, const HeapEnt& cand, unsigned long long ends, int hop_cid, int& r, int& row_end,
                                                int& good, int& resume_at, unsigned long long& accepted, Trail& tr, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  while (todo != 0ull) {
    const int j = __builtin_ctzll(todo);
    todo &= todo - 1ull;
    if (SEVERAL) {
      while (__builtin_expect(j >= row_end, 0)) {
        if (TRAILS) {
          trail_hop(tr, accepted, r == 0 ? hop_cid : __builtin_amdgcn_readlane((int)cand.id, r), st.n_hops + r, my_id, my_key, lane);
          accepted = 0ull;
        }
        r += 1;
        row_end = (int)((ends >> (8 * r)) & 0xFFu);
      }
    }
    const float key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_key), j));
    const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)my_id, j);
    if (FULL ? st.lower > key : (st.n_acc < ef || st.lower > key)) {
      auto enter = [&]() __attribute__((always_inline)) {
        frontier_insert_distinct<NS>(fr, key, id);
        if (TRAILS) accepted |= 1ull << j;
        st.n_acc = st.n_acc + 1;
        if (!FULL && st.n_acc < ef) {
          st.maxkey = uni(fmaxf(st.maxkey, key));
          st.lower = st.maxkey;
        } else {
          st.lower = frontier_max<NS>(fr);  // hnswlib's lowerBound
        }
        if (SEVERAL) {
          // the first candidate after this one that the new entry is closer than: its turn does not come now
          const int upto = r + 1 + __builtin_ctzll(__ballot(cand.key > key) >> (r + 1));  // (lanes past the batch: +inf)
          if (__builtin_expect(upto < good, 0)) {
            good = upto;
            const int end = (int)((ends >> (8 * (upto - 1))) & 0xFFu);
            todo &= end < 64 ? (1ull << end) - 1ull : ~0ull;
          }
        }
      };
      unsigned long long eq = 0ull;
#pragma unroll
      for (int t = 0; t < N; ++t) eq |= __ballot(fr.k[t] == key);
      // (WATCH: an eviction that would reach a watched entry, or its equal, is the general loop's as well)
      // (while the set is not full its last key is the padding's +inf)
      if (WATCH) eq |= __ballot(fr.k[N - 1] <= w_hi) >> 63;
      if (__builtin_expect(eq == 0ull, 1)) {
        enter();
      } else if (!frontier_has<NS>(fr, key, id)) {
        if constexpr (BUILD) {
          enter();  // the build takes equal keys as they come (order of arrival): any deterministic choice is as good
        } else {
          resume_at = j;  // an equal key of another node (WATCH: or a watched eviction): the rules for equal keys apply from this offer on
          todo = 0ull;
        }
      }
      // (else: a node met again after the visited filter forgot it; it is in the set already)
    }
  }
}
// One phase of the tie-free loop of search_level_fast (below).  Nine searches in ten never hold two equal keys in
// their set; until the first such pair turns up the search runs here, with none of the bookkeeping that equal keys
// need.  FULL = false: while the set fills (the bound is the largest key accepted so far, every offer is accepted);
// FULL = true: the set holds ef entries (the bound is its last key, an accepted offer pushes one out) — two
// instantiations, so that the hot one carries neither the fill test nor the running maximum.  TRAILS: the hop's
// accepted entries go on the search's trail (a kernel instance of its own: a pass that keeps no trails pays
// nothing for them).  WATCH: the set holds equal keys that do no harm as long as the waiting entries on the watch
// list (those with an equal in the set) are neither expanded nor pushed out here -- the loop hands back to the
// general one when that is about to happen.  BUILD: equal keys are taken in order of arrival and nothing is ever
// handed back.  Returns 0: no waiting entry is left, the search is over; 1: an offer met an equal key of another
// node, or its eviction would reach a watched entry (resume_at = which offer of the list in s.nbuf / s.dbuf);
// 2 (FULL = false only): the set is full now, the other phase goes on; 3 (WATCH only): the next candidate is a
// watched entry (its expanded mark has been taken off again, n = 0).  n = ids waiting in s.nbuf on entry.
//
// FULL: several candidates at a time.  Once the set is full seven expansions in ten bring in nothing, and the next
// candidate is nearly always one that is waiting already.  So the st.ahead closest waiting entries are expanded
// together: their link rows are fetched at once, the new nodes of all of them evaluated in one go (a pass of sixteen rows
// is filled instead of started for three or four), and their offers dealt with candidate by candidate, as if each had been
// expanded at its turn.  That is the same search as long as no accepted offer is closer than the next candidate of the
// batch: where one is, that candidate and those after it are put back (unmarked, and their nodes out of the visited
// filter; what they evaluated was for nothing) and the search goes on from the closer one.  st.ahead doubles up to
// kAhead after a batch in which nothing was accepted and falls to what was good of one that did not hold.  Counted on
// 100 000 x 50 at ef 300 with up to four: 127 batches instead of 301 hops per search, 2 % more evaluations, 40 % fewer
// passes over rows (growing after every batch that held: 104 batches, but 10 % more evaluations).  Not in searches of
// ef <= 128: with as many accepted offers as hops a batch seldom holds (40 000 queries on 1.18 M x 50, ef 64: 1.77 ms
// without, 1.81 with).  1.18 M x 50, ef 300, 10 000 / 40 000 queries: 1.76 -> 1.53, 5.08 -> 4.54 ms; 1 M x 96, topk 100,
// ef 256, 100 000 queries: 11.06 -> 9.99 ms; 100 000 x 960, ef 300, 1 000 queries: 1.44 -> 1.36 ms.
template <int DT, int QR, int NS, bool FULL, bool TRAILS, bool WATCH, bool BUILD = false, bool FEW = false>
__device__ __forceinline__ int tie_free_phase(const DevIndex& ix, const QVec<QR>& qv, int level, int ef, int S, Scratch& s,
                                              SearchState& st, Frontier<NS>& fr, int& n, int& hop_cid, int& resume_at,
                                              unsigned long long& accepted, Trail& tr, const TieWatch& watch, int lane) {
  constexpr int N = NS > 0 ? NS : 1;
  // shorter lists go in one by one (2, 4 or 8 are the same within the runs' spread: 1.18 M x 50, ef 300, 10 000 queries
  // 1.322 / 1.321 / 1.323 ms, one query on 100 000 x 50 0.279 each, 20 000 x 50 indexed 7.82 / 7.78 / 7.81 ms)
  constexpr int kInsertAllFrom = 4;
  // On a full set most steps bring in nothing and the others a dozen offers: those of one evaluation enter it together from
  // six on, in the instances that have the registers (a trail wants to know of each whether it was accepted when its turn
  // came; sets of two registers take their offers one by one as fast).  Also beside equal keys, as long as none of the offers
  // has one (one query on 200 000 x 128 integers, ef 300: 0.493 ms, refused for any equal keys in the set 0.504; not tried
  // beside them 0.495, but 1 000 queries on 100 000 x 50, one in eight of which meets two by accident, 0.539 instead of 0.528).
  constexpr bool kMerge = FEW && !TRAILS && NS > 2;
  constexpr int kMergeFrom = 6;
  // more rows in flight: the search on long rows (dist_long), and small sets, which leave the registers for it (56 of 72;
  // 345 678 x 101 in fp16, ef 77, 5 003 queries: 0.85 -> 0.71 ms)
  constexpr int kWide = FEW ? 4 : (!BUILD && ((QR == 0 && NS <= 8) || (QR == 2 && NS == 2)) ? 2 : 1);
  // candidates at a time at most, 8 / 6 / 4: 1.18 M x 50, ef 300, 10 000 queries 1.319 / 1.326 / 1.397 ms, one query on
  // 100 000 x 50 0.280 / 0.287 / 0.295 ms; 1 M x 96, ef 256, 100 000 queries 9.74 / 9.83 / 9.90 ms (longer rows: registers)
  constexpr int K = FULL && (BUILD || FEW || NS > 2) ? (QR == 1 || FEW ? kAhead : 6) : 1;
  // (said to be wavefront-uniform, so that they sit in scalar registers through the loop)
  const int w0 = WATCH ? uni(watch.id0) : -1, w1 = WATCH ? uni(watch.id1) : -1;
  const int w2 = WATCH ? uni(watch.id2) : -1, w3 = WATCH ? uni(watch.id3) : -1;
  const float w_hi = WATCH ? uni(watch.hi) : -INFINITY;
  int rows = 1;                  // candidates of the batch under way
  HeapEnt* const cands = batch_candidates(s);
  unsigned long long ends = (uint32_t)n;   // end of each one's offers in s.nbuf / s.dbuf, eight bits each
  while (true) {
    if ((QR == 2 || (QR == 1 && (TRAILS || NS == 6) )) && NS > 2 && !BUILD && !FEW) lane = fresh(lane);  // (these are the instances short of registers)
    if (n > 0) dist_list<DT, QR, false, kWide>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
    st.n_dist += n;
    wave_sync();
    // (unconditional LDS reads at a clamped index, then a select: no exec-mask branches)
    const int last = n > 0 ? n - 1 : 0;
    const int at = lane < last ? lane : last;
    const float got_key = s.dbuf[at];
    const uint32_t my_id = s.nbuf[at];
    const float my_key = lane < n ? got_key : INFINITY;
    unsigned long long todo = FULL ? __ballot(st.lower > my_key) : __ballot(lane < n);
    HeapEnt cand;  // lane r: the batch's r-th candidate (in LDS meanwhile: two registers less where rows are in flight)
    cand.key = INFINITY;
    cand.id = kEmpty;
    if (K > 1 && rows > 1) {
      const HeapEnt c = cands[lane < rows ? lane : 0];
      cand.key = lane < rows ? c.key : INFINITY;
      cand.id = c.id;
    }
    int r = 0;                                              // the candidate whose offers are being dealt with
    int row_end = K > 1 ? (int)(ends & 0xFFu) : n;
    int good = rows;                                        // candidates of the batch that are expanded for good
    const int acc_before = st.n_acc;
    if (!FULL && (BUILD || FEW || NS > 2) && n >= kInsertAllFrom && n < 64 && st.n_acc + n <= ef && 32 * (N + 1) <= s.filter.sets()) {
      float last_key = 0.f;
      if (frontier_insert_all<NS, false>(fr, todo, st.n_acc, ef, my_key, my_id, s.nbuf, s.dbuf, reinterpret_cast<uint32_t*>(s.vcache), -INFINITY,
                                         last_key, lane)) {
        if (TRAILS) accepted |= todo;
        st.n_acc = st.n_acc + n;
        st.maxkey = last_key;
        st.lower = last_key;
        todo = 0ull;
      }
    }
    if (FULL && kMerge && __popcll(todo) >= kMergeFrom && __popcll(todo) < 64 && 32 * (N + 1) <= s.filter.sets()) {
      // the first candidate that an offer of those before it is closer than: its turn does not come now (tie_free_offers)
      int upto = rows;
      for (int c = rows - 1; c > 0; --c) {
        const float next_key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cand.key), c));
        const int end = (int)((ends >> (8 * (c - 1))) & 0xFFu);
        if ((__ballot(my_key < next_key) & todo & (end < 64 ? (1ull << end) - 1ull : ~0ull)) != 0ull) upto = c;
      }
      const int end = (int)((ends >> (8 * (upto - 1))) & 0xFFu);
      const unsigned long long now = todo & (end < 64 ? (1ull << end) - 1ull : ~0ull);
      float last_key = 0.f;
      if (__popcll(now) >= kMergeFrom &&
          frontier_insert_all<NS, true>(fr, now, ef, ef, my_key, my_id, s.nbuf, s.dbuf, reinterpret_cast<uint32_t*>(s.vcache), w_hi, last_key, lane)) {
        st.n_acc = st.n_acc + 1;  // (a full set only asks whether there were any)
        st.lower = last_key;
        good = upto;
        todo = 0ull;
      }
    }
    if (K > 1)
      tie_free_offers<NS, FULL, TRAILS, WATCH, BUILD, true>(st, fr, todo, my_key, my_id, ef, w_hi, cand, ends, hop_cid, r, row_end, good,
                                                            resume_at, accepted, tr, lane);
    else
      tie_free_offers<NS, FULL, TRAILS, WATCH, BUILD, false>(st, fr, todo, my_key, my_id, ef, w_hi, cand, ends, hop_cid, r, row_end, good,
                                                             resume_at, accepted, tr, lane);
    int start = 0;
    if (K > 1) {
      if (resume_at >= 0) {
        good = r + 1;
        start = r > 0 ? (int)((ends >> (8 * (r - 1))) & 0xFFu) : 0;
      }
      if (good < rows) {
        const int end = (int)((ends >> (8 * (good - 1))) & 0xFFu);
        filter_forget(s, my_id, lane >= end && lane < n);
        for (int b = good; b < rows; ++b) frontier_untake<NS>(fr, (uint32_t)__builtin_amdgcn_readlane((int)cand.id, b));
        st.ahead = good;
      } else if (st.n_acc == acc_before) {
        st.ahead = 2 * st.ahead < K ? 2 * st.ahead : K;
      }
    }
    if (resume_at >= 0) {
      if (K > 1) {
        // the general loop goes on with this candidate's offers, at the front of the list
        st.n_hops += r;
        if (r > 0) hop_cid = __builtin_amdgcn_readlane((int)cand.id, r);
        n = row_end - start;
        if (start > 0) {
          resume_at -= start;
          accepted >>= start;
          const int from = start + (lane < n ? lane : 0);
          const float k0 = s.dbuf[from];
          const uint32_t i0 = s.nbuf[from];
          wave_sync();
          if (lane < n) {
            s.dbuf[lane] = k0;
            s.nbuf[lane] = i0;
          }
          wave_sync();
        }
      }
      return 1;
    }
    if (TRAILS) trail_hop(tr, accepted, r == 0 ? hop_cid : __builtin_amdgcn_readlane((int)cand.id, r), st.n_hops + r, my_id, my_key, lane);
    accepted = 0ull;
    if (K > 1) st.n_hops += good - 1;
    wave_sync();
    if (K == 1 || st.ahead == 1) {
      const int cid = frontier_take<NS>(fr, lane, false);
      if (cid < 0) return 0;
      if (WATCH && (cid == w0 || cid == w1 || cid == w2 || cid == w3)) {
        frontier_untake<NS>(fr, (uint32_t)cid);  // a watched entry's turn: the general loop takes it, with its bookkeeping
        n = 0;
        return 3;
      }
      hop_cid = cid;
      rows = 1;
      n = visit_lossy(scalar_base(link_row(ix, (uint32_t)cid, level)), S, s, lane);
      ends = (uint32_t)n;
    } else {
      rows = frontier_take_many<NS>(fr, st.ahead, cands, lane);
      if (rows == 0) return 0;
      const uint32_t cand_id = cands[lane < rows ? lane : 0].id;
      if (WATCH) {
        // a watched entry's turn is the general loop's business: the batch ends before it
        const unsigned long long hit = __ballot(lane < rows && ((int)cand_id == w0 || (int)cand_id == w1 || (int)cand_id == w2 || (int)cand_id == w3));
        if (hit != 0ull) {
          const int first = __builtin_ctzll(hit);
          for (int b = first; b < rows; ++b) frontier_untake<NS>(fr, (uint32_t)__builtin_amdgcn_readlane((int)cand_id, b));
          rows = first;
          if (rows == 0) {
            n = 0;
            return 3;
          }
        }
      }
      hop_cid = __builtin_amdgcn_readlane((int)cand_id, 0);
      const int in = visit_lossy_rows<K>(ix, cand_id, rows, level, S, s, n, ends, lane);
      for (int b = in; b < rows; ++b) frontier_untake<NS>(fr, (uint32_t)__builtin_amdgcn_readlane((int)cand_id, b));
      rows = in;
    }
    st.n_hops += 1;
    wave_sync();
    if (!FULL && st.n_acc >= ef) return 2;
  }
}

// The tie-free loop where a team helps: as tie_free_phase, but while the set fills and afterwards, and with up to eight candidates
// considered in every step.  Their lists are there already (the first one may have none: its nodes are evaluated here; the step
// ends before another without); of the eight, as many are expanded as surely come next whatever their offers do: those before the
// first one that an offer of an earlier one is closer than.  The others stay where they are, with their lists.  So a step
// costs no evaluation that a later one repeats, and a search has 60 of them at ef 300 where batches that grow and shrink took 100
// (CPU model, 60 000 x 50).
template <int DT, int QR, int NS, bool WATCH, bool BUILD = false>
__device__ __forceinline__ int team_phase(const DevIndex& ix, const QVec<QR>& qv, int level, int ef, int S, Scratch& s, SearchState& st, Frontier<NS>& fr,
                                          int& n, bool have_keys, int& hop_cid, int& resume_at, const TieWatch& watch, int lane) {
  constexpr int kMergeFrom = 6;  // fewer offers enter the set one by one
  const int w0 = WATCH ? uni(watch.id0) : -1, w1 = WATCH ? uni(watch.id1) : -1;
  const int w2 = WATCH ? uni(watch.id2) : -1, w3 = WATCH ? uni(watch.id3) : -1;
  const float w_hi = WATCH ? uni(watch.hi) : -INFINITY;
  int rows = 1;                     // candidates considered
  bool taken = true;                // (the one whose n nodes come first is marked already)
  int rank = 0, steps = 0;
  HeapEnt cand;                     // lane r: the r-th; +inf behind the last
  cand.key = INFINITY;
  cand.id = kEmpty;
  float cand_keys[8];               // all of their keys, in each lane
#pragma unroll
  for (int c = 0; c < 8; ++c) cand_keys[c] = INFINITY;
  int row_ends = 64;                // lane r: the first lane behind its nodes
  int from = 0;                     // each lane: the number of the candidate whose node it holds
  int slot = -1;                    // lane r: where its list is
  uint32_t listed_id = kEmpty;      // nodes that came from lists, lane by lane behind the n ids whose keys are still to be computed
  float listed_key = INFINITY;
  unsigned long long listed = 0ull; // the lanes that hold one
  uint2* listed_set = nullptr;      // where the filter has it, what it says there, and what it is to say
  uint2 listed_word = make_uint2(0u, 0u);
  uint32_t listed_place = 0u;
  Trail no_trail;
  unsigned long long accepted = 0ull;
  while (true) {
    if (n > 0 && !have_keys) dist_list<DT, QR, false, team_wide<QR>()>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
    have_keys = false;
    wave_sync();
    float my_key = listed_key;
    uint32_t my_id = listed_id;
    unsigned long long valid = listed;
    if (n > 0) {
      const int at = lane < n ? lane : n - 1;
      const float got_key = s.dbuf[at];
      const uint32_t got_id = s.nbuf[at];
      my_key = lane < n ? got_key : my_key;
      my_id = lane < n ? got_id : my_id;
      valid |= first_lanes(n);
    }
    unsigned long long todo = st.n_acc < ef ? valid : valid & __ballot(st.lower > my_key);
    int good = rows;  // candidates that are expanded now
    if (todo != 0ull && rows > 1) {
      // (an offer keeps back the candidates after its own that it is closer than)
      int kept_back = 0;
#pragma unroll
      for (int c = 0; c < 8; ++c) kept_back += cand_keys[c] <= my_key ? 1 : 0;
      kept_back = kept_back > from ? kept_back : from + 1;
      const int first_kept = least_of_all_ints(__builtin_amdgcn_inverse_ballot_w64(todo) ? kept_back : 8);
      good = first_kept < rows ? first_kept : rows;
    }
    const unsigned long long now_lanes = good < rows ? first_lanes(__builtin_amdgcn_readlane(row_ends, good - 1)) : ~0ull;
    todo &= now_lanes;
    if (!taken) frontier_take_first<NS>(fr, good, rank);
    const int most = good;
    if (__popcll(todo) >= kMergeFrom) {
      int offers = 0;
      float last_key = 0.f;
      if (frontier_merge<NS>(fr, todo, st.n_acc < ef ? st.n_acc : ef, ef, my_key, my_id, s.team.room(), w_hi, offers, last_key, lane)) {
        st.n_acc = st.n_acc + offers;
        st.maxkey = last_key;
        st.lower = last_key;
        todo = 0ull;
      }
    }
    int r = 0, row_end = 64;
    unsigned long long ends = 64ull;  // row_ends, eight bits each
    if (todo != 0ull && rows > 1) {
      ends = 0ull;
      for (int c = 0; c < good; ++c) ends |= (unsigned long long)(uint32_t)__builtin_amdgcn_readlane(row_ends, c) << (8 * c);
      row_end = (int)(ends & 0xFFu);
    }
    if (todo != 0ull)
      tie_free_offers<NS, false, false, WATCH, BUILD, true>(st, fr, todo, my_key, my_id, ef, w_hi, cand, ends, hop_cid, r, row_end, good,
                                                            resume_at, accepted, no_trail, lane);
    if (resume_at >= 0) {
      // an equal key: the general loop goes on with this candidate's offers, at the front of the list
      for (int b = r + 1; b < most; ++b) frontier_untake<NS>(fr, (uint32_t)__builtin_amdgcn_readlane((int)cand.id, b));
      if (lane <= r && slot >= 0) lds_tell(s.team.owner() + slot, kNobody);
      __builtin_amdgcn_wave_barrier();
      if (!taken) {
        st.n_hops += r + 1;
        hop_cid = __builtin_amdgcn_readlane((int)cand.id, r);
      }
      const int start = r > 0 ? (int)((ends >> (8 * (r - 1))) & 0xFFu) : 0;
      const unsigned long long of = valid & first_lanes(row_end) & ~first_lanes(start);
      const unsigned long long before = valid & first_lanes(start);
      n = __popcll(of);
      st.n_dist += __popcll(before | of);
      resume_at = __popcll(of & first_lanes(resume_at));
      wave_sync();
      if (__builtin_amdgcn_inverse_ballot_w64(of)) {
        s.nbuf[lanes_below(of)] = my_id;
        s.dbuf[lanes_below(of)] = my_key;
      }
      filter_enter(s, my_id, before | of);
      wave_sync();
      return 1;
    }
    // the lists of the candidates that have been expanded are done with, and their nodes dealt with
    if (lane < good && slot >= 0) lds_tell(s.team.owner() + slot, kNobody);
    __builtin_amdgcn_wave_barrier();
    const unsigned long long done = valid & now_lanes;
    st.n_dist += __popcll(done);
    if (n > 0) {
      filter_enter(s, my_id, done);
    } else if (__builtin_amdgcn_inverse_ballot_w64(done)) {  // (nothing has been entered since)
      *listed_set = filter_push(listed_word, listed_place);
    }
    __builtin_amdgcn_wave_barrier();
    // every eighth step the lists of candidates that are no longer among the next go
    if ((++steps & 7) == 0) team_tidy(s.team, lane);
    if (!taken) st.n_hops += good;
    taken = false;

    n = 0;
    const int total = frontier_line_up<NS>(fr, s.team, rank, lane);
    if (total == 0) return 0;
    rows = total < 8 ? total : 8;
    const int nth = lane & 7;
    cand = s.team.line()[nth];
#pragma unroll
    for (int c = 0; c < 8; ++c) cand_keys[c] = s.team.line()[c].key;
    if (WATCH) {
      // a watched entry's turn is the general loop's business: the batch ends before it
      const unsigned long long hit = __ballot(lane < rows && ((int)cand.id == w0 || (int)cand.id == w1 || (int)cand.id == w2 || (int)cand.id == w3));
      if (hit != 0ull) rows = __builtin_ctzll(hit);
      if (rows == 0) return 3;
    }
    TeamPlace t = team_look(s.team, cand.id);
    // (lists that are just being made are waited for: each was begun a step ago or earlier)
    for (int polls = 0; polls < 4096 && __ballot(lane < rows && t.there < 0 && t.making) != 0ull; ++polls) t = team_look(s.team, cand.id);
    const unsigned long long there = __ballot(lane < rows && t.there >= 0);
    const unsigned long long stop = first_lanes(rows) & ~there & ~1ull;
    rows = stop != 0ull ? __builtin_ctzll(stop) : rows;
    hop_cid = uni((int)cand.id);
    if ((there & 1ull) == 0ull) {  // the first one has no list: its nodes are the search's own to evaluate
      n = visit_unmarked(scalar_base(link_row(ix, (uint32_t)hop_cid, level)), S, s, lane);
      t.eights = lane == 0 ? (n > 0 ? (n + 7) >> 3 : 1) : t.eights;
    }
    // Eight lanes, or more of them, to a list: lane r gets the first eight behind its nodes.
    const int own = (there & 1ull) == 0ull ? 1 : 0;
    int upto = lane < rows ? t.eights : 0;
    const int eights = upto;
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x111, 0xF, 0xF, true);  // row_shr:1
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x112, 0xF, 0xF, true);  // row_shr:2
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x114, 0xF, 0xF, true);  // row_shr:4
    const unsigned long long over = __ballot(upto > 8) & first_lanes(rows);
    rows = over != 0ull ? __builtin_ctzll(over) : rows;
    row_ends = 8 * upto;
    // whose nodes each eight of lanes holds: the lists' first eights, one bit each, from all of them
    int begins = lane < rows ? 1 << (upto - eights) : 0;
    begins |= __builtin_amdgcn_update_dpp(0, begins, 0x111, 0xF, 0xF, true);
    begins |= __builtin_amdgcn_update_dpp(0, begins, 0x112, 0xF, 0xF, true);
    begins |= __builtin_amdgcn_update_dpp(0, begins, 0x114, 0xF, 0xF, true);
    const uint32_t starts = (uint32_t)__builtin_amdgcn_readlane(begins, 7);
    const int used = __builtin_amdgcn_readlane(upto, rows - 1);
    const int eight = lane >> 3;
    const uint32_t mine = starts & ((2u << eight) - 1u);
    from = __popc(mine) - 1;
    const int part = eight - (31 - __builtin_clz(mine | 1u));
    const bool in = eight < used && (own == 0 || from > 0);
    slot = lane < rows ? t.there : -1;
    const int where = __shfl(t.there, in ? from : 0, 64);
    const int place = in ? 8 * part + nth : 0;
    const uint32_t got = s.team.ids(in ? where : 0)[place];
    const float got_key = s.team.keys(in ? where : 0)[place];
    const uint32_t id = in ? got : kEmpty;
    uint32_t set;
    listed_place = filter_find(s.filter, id, set);
    listed_set = reinterpret_cast<uint2*>(s.vcache) + set;
    listed_word = *listed_set;
    listed = __ballot(id != kEmpty) & filter_misses(listed_word, listed_place);
    listed_id = id;
    listed_key = __builtin_amdgcn_inverse_ballot_w64(listed) ? got_key : INFINITY;
    cand.key = lane < rows ? cand.key : INFINITY;
    wave_sync();
  }
}

// Best-first search of one level on the sorted set (needs the LDS tag filter).  On entry
// s.nbuf[0..n_seed) holds the seeds, already entered into the filter.  Returns 0: fr holds the
// result (st.top_size entries, ascending), all keys were distinct; 2: the same, but equal keys
// met on the way (the caller has to look at the cut at k); 1: given up — the outcome would
// depend on how hnswlib's heaps lay equal keys out.  st.n_dist counts the evaluations
// performed, repeated ones included.
//
// When do equal keys matter?  (a) Several waiting candidates share the smallest key d: hnswlib
// expands them in its heap's order.  If none of their expansions produces a key below d the
// order is immaterial — every node evaluated on the way is evaluated once whichever member
// meets it first, a key below d would be accepted under any order (d is within the bound), so
// none exists under any order, the whole group is expanded back to back and the set afterwards
// is the ef smallest of old set and offers either way — up to entries whose key equals the
// bound the set ends up with: whether such an offer is accepted or turned away, and which of
// several such entries is evicted, does depend on the order.  So a group during which an offer was turned
// away or an entry evicted whose key equals the bound at the group's end gives the query up.  A key below d
// turning up during the group does not by itself: such a candidate (and whatever closer ones it leads to) is
// expanded before the rest of the group under any order, and by the same argument the set after the last
// member is the same — provided every member does get expanded under any order, i.e. the bound is still at
// or above d when the group is through and no member was pushed out of the set before its turn; a second group
// of equal keys among those closer candidates is not followed (given up).  (b) An eviction finds equal largest keys: which one leaves is the heap's
// choice, and the one that leaves stays a live candidate of hnswlib as long as that key is
// within the bound.  The search goes on, but gives up if it comes to expand an entry with such
// a key, or ends while such a key is still within the bound — except in the one case that covers most of
// them: a single such eviction, out of exactly two equal largest keys, with fewer than the whole set asked
// for.  Then the two twins are known (the one the set kept, the one it pushed out: the "ghost", remembered
// with its expanded mark), hnswlib holds both in its candidate queue whichever of them its result heap kept,
// and when their key comes up — last of all, it is the bound — it expands each of them that is not expanded
// yet, in its heap's order.  If neither expansion has an offer accepted, the order is immaterial: nothing
// changes but the visited marks, and the search ends there.  So the twins are expanded one after the other
// (the ghost too, though it is not in the set), and only an accepted offer on the way gives the query up.
// (c) Equal keys across
// the cut at k (the result heap's choice) or among the k best (listed by label): the caller's business.
// far: expand the farthest waiting entry instead of the closest (the reference's
// reverse_cand); that is no hnswlib search any more, equal keys simply keep their order of
// arrival and nothing is ever given up.  BUILD likewise never gives up.
template <int DT, int QR, int NS, bool BUILD, bool TRAILS = false, bool FEW = false, bool TEAM = false>
__device__ __forceinline__ int search_level_fast(const DevIndex& ix, const QVec<QR>& qv, int level, int ef, Scratch& s,
                                                  SearchState& st, Frontier<NS>& fr, int n_seed, int lane,
                                                  bool far = false, bool whole_set = false, Trail* trail = nullptr) {
  const int S = row_stride(ix, level);
  constexpr int kWide = TEAM ? team_wide<QR>() : FEW ? 4 : ((QR == 0 && !BUILD && NS <= 8) ? 2 : 1);  // (rows in flight: dist_list)
  int n = n_seed;
  const bool exact = !BUILD && !far;  // the outcome has to be hnswlib's
  Trail no_trail;
  Trail& tr = trail ? *trail : no_trail;
  unsigned long long accepted = 0ull;  // offers of the current hop that entered the set
  int hop_cid = -1;                    // the node the current hop expanded (-1: the seeds)
  int ghosts = 0;                     // evictions that had equal largest keys to choose from
  uint32_t ghost = kEmpty;            // the entry the (single) such eviction pushed out, with its expanded mark
  bool twin_phase = false;            // the twins of that eviction are being expanded: no offer may be accepted
  bool have_tie = false;              // equal keys have met in the set
  bool in_group = false;              // the entries being expanded share one key with others still waiting
  float group_key = 0.f;
  float group_edge = INFINITY;        // closest key turned away or evicted while the group is expanded
  float ek_min = INFINITY;            // smallest key at which an eviction had equal largest keys to choose from
  bool gave_up = false;
  // Until two equal keys meet in the set the search runs in tie_free_phase — same decisions, half the
  // instructions per accepted candidate — and only then moves on to the general loop below, at the very offer
  // that met the equal key (resume_at).
  int resume_at = -1;
  bool listed = false;  // (TEAM) the keys of the n nodes are there
  bool calm = (exact || (BUILD && !far)) && S <= 64;  // no equal keys are at work (or none matter): the tie-free loop may run
  TieWatch watch;
  while (true) {
    if (calm) {
      int how = st.n_acc >= ef ? 2 : 0;
      if constexpr (BUILD && TEAM) {
        how = team_phase<DT, QR, NS, false, true>(ix, qv, level, ef, S, s, st, fr, n, false, hop_cid, resume_at, watch, lane);
      } else if constexpr (BUILD) {
        if (how == 0) how = tie_free_phase<DT, QR, NS, false, false, false, true>(ix, qv, level, ef, S, s, st, fr, n, hop_cid, resume_at, accepted, tr, watch, lane);
        if (how == 2) how = tie_free_phase<DT, QR, NS, true, false, false, true>(ix, qv, level, ef, S, s, st, fr, n, hop_cid, resume_at, accepted, tr, watch, lane);
      } else if constexpr (TEAM) {  // (other wavefronts help)
        if (!have_tie) how = team_phase<DT, QR, NS, false>(ix, qv, level, ef, S, s, st, fr, n, listed, hop_cid, resume_at, watch, lane);
        else how = team_phase<DT, QR, NS, true>(ix, qv, level, ef, S, s, st, fr, n, listed, hop_cid, resume_at, watch, lane);
      } else if (!have_tie) {
        if (how == 0) how = tie_free_phase<DT, QR, NS, false, TRAILS, false, false, FEW>(ix, qv, level, ef, S, s, st, fr, n, hop_cid, resume_at, accepted, tr, watch, lane);
        if (how == 2) how = tie_free_phase<DT, QR, NS, true, TRAILS, false, false, FEW>(ix, qv, level, ef, S, s, st, fr, n, hop_cid, resume_at, accepted, tr, watch, lane);
      } else {
        // (after equal keys have met, the tie-free loop takes over again only once the set is full: how == 2)
        how = tie_free_phase<DT, QR, NS, true, TRAILS, true, false, FEW>(ix, qv, level, ef, S, s, st, fr, n, hop_cid, resume_at, accepted, tr, watch, lane);
      }
      st.top_size = st.n_acc < ef ? st.n_acc : ef;
      if (how == 0) {
        trail_stop(tr, st.n_hops, st.n_dist);
        return have_tie ? 2 : 0;
      }
      calm = false;
      // (what these were when the tie-free loop took over; said again so that none of them has to live through it)
      ghosts = 0;
      ghost = kEmpty;
      twin_phase = false;
      in_group = false;
      group_key = 0.f;
      group_edge = INFINITY;
      ek_min = INFINITY;
      gave_up = false;
    }
    while (true) {
      if ((QR == 1 || (QR == 2 && DT == DIST_DOT)) && NS == 6 && !BUILD && !FEW) lane = fresh(lane);
      if (resume_at < 0) {
        if (n > 0 && !(TEAM && listed)) dist_list<DT, QR, false, kWide>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
        st.n_dist += n;
        wave_sync();
      }
      for (int base = 0; base < n; base += 64) {
        const int mine = base + lane;
        // unconditional LDS reads at a clamped index, then a select: no exec-mask branches
        const int at = mine < n ? mine : 0;
        const float my_key = mine < n ? s.dbuf[at] : INFINITY;
        const uint32_t my_id = s.nbuf[at];
        const bool pass = mine < n && (st.n_acc < ef || st.lower > my_key);
        unsigned long long todo = __ballot(pass);
        if (resume_at >= 0) {
          todo &= ~((1ull << resume_at) - 1ull);  // the offers before it have been dealt with (one list of at most 64)
          resume_at = -1;
        }
        // offers turned away while a group of equal keys is being expanded: remember the closest
        if (exact && in_group) group_edge = uni(fminf(group_edge, least_of_all((mine < n && !pass) ? my_key : INFINITY)));
        // (plain if/else nesting, one way out of the loop: `continue` and `return` in here make the
        // compiler thread a state variable through a dozen scalar blocks per accepted candidate)
        while (todo != 0ull) {
          const int j = __builtin_ctzll(todo);
          todo &= todo - 1ull;
          const float key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_key), j));
          const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)my_id, j);
          if (st.n_acc < ef || st.lower > key) {
            // an eviction out of several equal largest keys: the heap's choice decides which of
            // them stays in the result set, and the other one stays a live candidate of hnswlib
            const bool twins = exact && have_tie && st.n_acc >= ef && frontier_max_twice<NS>(fr);
            // the entry a full set is about to push out, where somebody will ask for it
            const uint32_t evicted = (twins || (exact && in_group && st.n_acc >= ef && st.lower == group_key))
                                         ? (uint32_t)__builtin_amdgcn_readlane((int)fr.v[(NS > 0 ? NS : 1) - 1], 63)
                                         : kEmpty;
            const int r = frontier_insert<NS>(fr, key, id, lane);
            if (r != 2) {
              accepted |= 1ull << j;
              if (twins) {
                ek_min = uni(fminf(ek_min, st.lower));
                ghost = evicted;
                // (three or more equal largest keys, a second event, the whole set asked for: the plain rule)
                ghosts += (frontier_max_twice<NS>(fr) || whole_set) ? 2 : 1;
              }
              if (exact && twin_phase) {
                gave_up = true;  // which twin hnswlib expands first now decides whether the other one is expanded at all
                todo = 0ull;
              }
              have_tie = have_tie || r == 1;
              if (exact && in_group && st.n_acc >= ef) {
                group_edge = uni(fminf(group_edge, st.lower));  // the entry this insert evicted
                // a member of the group pushed out before its turn: with another order it would have been expanded
                if (st.lower == group_key && (evicted & kExpanded) == 0u) {
                  gave_up = true;
                  todo = 0ull;
                }
              }
              st.n_acc = uni(st.n_acc + 1);
              st.maxkey = uni(fmaxf(st.maxkey, key));
              st.lower = uni(st.n_acc >= ef ? frontier_max<NS>(fr) : st.maxkey);  // hnswlib's lowerBound
            }
          } else if (exact && in_group) {
            group_edge = uni(fminf(group_edge, key));
          }
        }
        if (gave_up) base = n;  // leave the outer loop as well
        else trail_hop(tr, accepted, hop_cid, st.n_hops, my_id, my_key, lane);  // (a trail is kept for rows of one pass only)
        accepted = 0ull;
      }
      if (gave_up) {
        trail_stop(tr, st.n_hops - 1, st.n_dist - n);  // (a trail still recording here: the hop under way, and its evaluations, are not on it)
        break;
      }
      st.top_size = st.n_acc < ef ? st.n_acc : ef;
      int cid = frontier_take<NS>(fr, lane, far);
      const bool was_in_group = in_group;
      if (exact && have_tie) {
        const float d = cid >= 0 ? frontier_key_of<NS>(fr, (uint32_t)cid) : INFINITY;
        if (in_group && cid >= 0 && d < group_key) {
          // a closer candidate turned up inside the group: it is expanded before the rest of the group under any
          // order.  A group within the group is not followed.
          gave_up = frontier_open_key<NS>(fr, d);
        } else if (in_group && d != group_key) {
          // the group is through.  With another order of its members an offer or an entry whose
          // key equals the bound reached now could have ended up on the other side of it; and with the bound
          // below the group's key a member popped late would not have been expanded at all.
          gave_up = st.n_acc >= ef && (group_edge == st.lower || st.lower < group_key);
          in_group = false;
        }
        if (cid >= 0) {
          if (d >= ek_min) {
            // the twin the set kept: it is the set's last entry and its key is the bound
            if (ghosts == 1 && !in_group && !frontier_open_key<NS>(fr, d)) twin_phase = true;
            else gave_up = true;
          }
          if (!in_group && !twin_phase) {
            in_group = frontier_open_key<NS>(fr, d);  // other waiting entries with this very key
            group_key = d;
            group_edge = INFINITY;
          }
        } else if (!gave_up && st.n_acc >= ef && st.lower >= ek_min) {
          // an entry evicted out of equal largest keys that are still within the bound is one
          // hnswlib would go on to expand
          if (ghosts == 1) {
            if ((ghost & kExpanded) == 0u) {
              cid = (int)ghost;  // the twin the set pushed out: expanded like any other, nothing of it may be accepted
              ghost |= kExpanded;
              twin_phase = true;
            }
          } else {
            gave_up = true;
          }
        }
      }
      // the trail: over for good, or the hops of a group of equal keys begin or end with the next one
      if (twin_phase || gave_up || cid < 0) trail_stop(tr, st.n_hops, st.n_dist);
      else if (in_group != was_in_group) trail_mark(tr, in_group ? kTrailOwn : kTrailBack, st.n_hops + 1, lane);
      if (gave_up || cid < 0) break;
      hop_cid = cid;
      st.n_hops += 1;
      wave_sync();
      listed = false;
      if constexpr (TEAM && !BUILD) {
        if (S <= 64) {
          int rank;
          frontier_line_up<NS>(fr, s.team, rank, lane);
          listed = visit_listed(s, (uint32_t)cid, S, n, lane);
          if ((st.n_hops & 7) == 0) team_tidy(s.team, lane);
        }
      }
      if (!listed) n = visit_lossy(scalar_base(link_row(ix, (uint32_t)cid, level)), S, s, lane);
      wave_sync();
      // Equal keys that sit in the set do no harm while none of them that still waits is expanded or pushed out
      // (unless the whole set is the answer): no group can form, and which of two expanded twins an eviction
      // pushes out changes neither the keys of the set nor hnswlib's candidates.  With no group under way and
      // no eviction out of equal largest keys on record whose key is still within the bound (once the bound is
      // below it, the entry such an eviction pushed out is as dead for hnswlib as any other), the tie-free loop
      // takes over again from this hop's offers, with the waiting entries that have an equal (at most four) on
      // its watch list; it comes back at the next offer that meets an equal key, when a watched entry's turn
      // comes, or when an eviction reaches one.
      if (exact && S <= 64 && !whole_set && st.n_acc >= ef && !in_group && !twin_phase && (ghosts == 0 || st.lower < ek_min) &&
          frontier_watch_list<NS>(fr, watch)) {
        calm = true;
        break;
      }
    }
    if (!calm) break;
  }
  return gave_up ? 1 : (have_tie ? 2 : 0);
}

// hnswlib's level-0 search with the literal candidate queue (which alone decides the order of
// expansion among equal keys) but with the sorted set with ids as result set and the LDS-only
// visited filter of the sorted-set search: a neighbour the filter has forgotten is evaluated
// again and then either found in the set by its id, or turned away by the accept rule as it
// was (or would be) the first time — the candidate queue sees exactly hnswlib's sequence of
// pushes and pops.  No bitmap, no atomics, nothing to undo.  Every accepted entry is also
// logged (s.log) for the caller's replay of the result heap.  *ambiguous is set when an
// eviction had equal largest keys to choose from: the set then holds the same keys as
// hnswlib's result heap but possibly another of the twins.  st.n_dist counts the evaluations
// performed, repeated ones included.  On entry s.nbuf[0..n_seed) holds the seeds, already
// entered into the filter.
template <int DT, int QR, int NS>
__device__ __forceinline__ void search_level_lean(const DevIndex& ix, const QVec<QR>& qv, int ef, Scratch& s, SearchState& st,
                                                  Frontier<NS>& fr, int n_seed, int lane, bool* ambiguous,
                                                  const uint4* trail = nullptr, int trail_n = 0, int trail_hops = 0,
                                                  int trail_n_dist = 0, int stop_marker = -1, int* rest_from = nullptr) {
  SplitHeap cand{s.cand, s.cand_glob, s.cand_lds};
  const int cand_cap = s.cand_lds + s.cand_glob_cap;
  const int S = row_stride(ix, 0);
  int n = n_seed;
  bool amb = false;
  // The first trail_hops expansions were made by the sorted-set pass too: outside the stretches its markers
  // set apart, their accepted entries come from its trail (records in hop order, none for a hop that accepted
  // nothing) instead of from link rows and vectors.  Every entry goes through the accept rule again: it
  // passes as it did there.
  int trail_at = 0;
  bool from_trail = false;
  // 64 of its records at a time, lane by lane: a hop has two or three, and fetched for each hop anew they were a trip to
  // memory and back twice per hop
  uint4 win = make_uint4(0u, 0u, 0u, 0u);
  int win_at = -64;
  uint32_t win_last = 0u;  // the hop of the window's last record
  auto window = [&](int hop) __attribute__((always_inline)) {  // from trail_at on, all of this hop's records at least
    if (trail_at < trail_n && trail_at > win_at &&
        (trail_at >= win_at + 64 || (win_at + 64 < trail_n && win_last <= (uint32_t)hop))) {
      win_at = trail_at;
      win = trail[win_at + lane < trail_n ? win_at + lane : trail_n - 1];
      win_last = (uint32_t)__builtin_amdgcn_readlane((int)win.w, 63);
    }
    return trail_at - win_at;
  };
  bool own_stretch = false;  // between two markers: hops this pass makes itself
  if (trail_hops > 0) st.n_dist += trail_n_dist;  // the evaluations that pass made up to the trail's end count as performed
  while (true) {
    if (n > 0 && !from_trail) dist_list<DT, QR, false, literal_wide<DT, QR, NS>(), literal_select<DT, QR, NS>()>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
    st.n_dist += from_trail ? 0 : n;
    wave_sync();
    for (int base = 0; base < n; base += 64) {
      const int mine = base + lane;
      const int at = mine < n ? mine : 0;
      const float my_key = mine < n ? s.dbuf[at] : INFINITY;
      const uint32_t my_id = s.nbuf[at];
      unsigned long long todo = __ballot(mine < n && (st.n_acc < ef || st.lower > my_key));
      while (todo != 0ull) {
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        HeapEnt e;
        e.key = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_key), j));
        e.id = (uint32_t)__builtin_amdgcn_readlane((int)my_id, j);
        if (st.n_acc < ef || st.lower > e.key) {
          const bool twins = st.n_acc >= ef && frontier_max_twice<NS>(fr);
          if (frontier_insert<NS>(fr, e.key, e.id, lane) != 2) {
            amb = amb || twins;
            if (st.cand_size >= cand_cap || st.n_acc >= s.log_cap) {
              st.fail = 1;  // (one way out of the loops: see search_level_fast)
              todo = 0ull;
            } else {
              if (lane == 0) s.log[st.n_acc] = e;
              st.n_acc = uni(st.n_acc + 1);
              if (st.cand_size < s.cand_lds) {
                LdsHeap cand_fast{s.cand};
                coop_push<true>(cand_fast, st.cand_size, e, lane);
              } else {
                coop_push<true>(cand, st.cand_size, e, lane);
              }
              st.maxkey = uni(fmaxf(st.maxkey, e.key));
              st.lower = uni(st.n_acc >= ef ? frontier_max<NS>(fr) : st.maxkey);  // hnswlib's lowerBound
            }
          }
        }
      }
      if (st.fail) base = n;
    }
    if (st.fail) break;
    st.top_size = st.n_acc < ef ? st.n_acc : ef;
    int cid = -1;
    if (st.cand_size > 0) {
      wave_sync();
      const HeapEnt c = uniform_ent(s.cand[0]);
      if (!(c.key > st.lower)) {
        cid = (int)c.id;
        if (st.cand_size <= s.cand_lds) {
          LdsHeap cand_fast{s.cand};
          coop_pop<true>(cand_fast, st.cand_size, s.tree, lane);
        } else {
          coop_pop<true>(cand, st.cand_size, s.tree, lane);
        }
      }
    }
    wave_sync();
    if (cid < 0) break;
    st.n_hops += 1;
    from_trail = false;
    if (st.n_hops <= trail_hops) {
      // markers that take effect with this hop (a group may end and the next begin at the same one)
      while (true) {
        const int off = window(st.n_hops);
        if (trail_at >= trail_n) break;
        const uint32_t kind = (uint32_t)__builtin_amdgcn_readlane((int)win.x, off);
        const uint32_t at_hop = (uint32_t)__builtin_amdgcn_readlane((int)win.w, off);
        if (kind < kTrailBack || at_hop != (uint32_t)st.n_hops) break;
        own_stretch = kind == kTrailOwn;
        trail_at += 1;
      }
      // (stop_marker >= 0: the trail covers the whole search and this is the index of its last marker.  Once past
      // it, every further accepted entry is on the trail: the caller needs no more of this search.)
      if (stop_marker >= 0 && !own_stretch && trail_at > stop_marker) {
        *rest_from = trail_at;
        break;
      }
      if (!own_stretch) {
        // this hop's records: a run from trail_at on (at most one link row's worth: under 64)
        const int off = window(st.n_hops);
        const bool mine = lane >= off && win_at + lane < trail_n && win.x < kTrailBack && win.w == (uint32_t)st.n_hops;
        const unsigned long long run = __ballot(mine);
        if (__ballot(mine && win.x != (uint32_t)cid) != 0ull) {
          trail_hops = 0;  // not the node that pass expanded here: nothing more is taken from the trail
        } else {
          n = __popcll(run);
          // the filter learns the nodes (a later hop this pass makes itself need not evaluate them again; where two of
          // them fall into the same set of tags one is forgotten, as in visit_lossy)
          if (__builtin_amdgcn_inverse_ballot_w64(run)) {
            s.nbuf[lane - off] = win.y;
            s.dbuf[lane - off] = __uint_as_float(win.z);
            uint2* sets = reinterpret_cast<uint2*>(s.vcache);
            uint32_t slot;
            const uint32_t place = filter_find(s.filter, win.y, slot);
            sets[slot] = filter_push(sets[slot], place);
          }
          __builtin_amdgcn_wave_barrier();
          trail_at += n;
          from_trail = true;
        }
      }
    }
    if (!from_trail) n = visit_lossy(link_row(ix, (uint32_t)cid, 0), S, s, lane);
    wave_sync();
  }
  *ambiguous = amb;
}

// Greedy descent through levels from_level .. to_level+1 (hnswlib searchKnn upper
// loop; cpp/include/cuda_search_kernels.cuh:22-66 in the reference): each sweep
// scans the neighbour list captured at its start and moves to the strictly
// closest entry, which for a strict running minimum is the first occurrence of the
// list minimum.
// (A chain of fetches: where a node's upper rows are, its row, the neighbours' vectors.  Where the neighbours' rows are is asked for
// beside their vectors, and so is the node's row one level down, which a sweep that finds nothing closer goes on with.)
template <int DT, int QR>
__device__ __forceinline__ void descend(const DevIndex& ix, const QVec<QR>& qv, int from_level, int to_level,
                                        uint32_t& cur, float& dcur, Scratch& s, SearchState& st, int lane) {
  if (from_level <= to_level) return;
  const int SU = ix.SU;
  const int at = lane < SU ? lane : 0;
  long long first = ix.upper_off[cur];  // the node's row of level 1
  uint32_t below = kEmpty;              // the first 64 slots of its row one level down, where they have been asked for
  bool have_below = false;
  for (int level = from_level; level > to_level; --level) {
    bool changed = true;
    while (changed) {
      changed = false;
      const uint32_t* const row = ix.linksU + (size_t)(first + level - 1) * SU;
      const uint32_t got = have_below ? below : row[at];
      const uint32_t mine = lane < SU ? got : kEmpty;
      have_below = level - 1 > to_level;
      if (have_below) below = (row - SU)[at];
      const unsigned long long mask = __ballot(mine != kEmpty);
      if (mine != kEmpty) s.nbuf[lanes_below(mask)] = mine;
      __builtin_amdgcn_wave_barrier();
      int n = __popcll(mask);
      for (int base = 64; base < SU; base += 64) {
        const uint32_t id = base + lane < SU ? row[base + lane] : kEmpty;
        const unsigned long long more = __ballot(id != kEmpty);
        if (id != kEmpty) s.nbuf[n + lanes_below(more)] = id;
        __builtin_amdgcn_wave_barrier();
        n += __popcll(more);
      }
      wave_sync();
      st.n_sweeps += 1;
      if (n == 0) break;
      const long long firsts = ix.upper_off[mine != kEmpty ? mine : cur];
      dist_list<DT, QR, false>(ix, qv, s.qlds, s.nbuf, n, s.dbuf, lane);
      st.n_dist_upper += n;
      wave_sync();
      float best = INFINITY;
      int bidx = -1;
      for (int base = 0; base < n; base += 64) {
        int t = base + lane;
        float d = t < n ? s.dbuf[t] : INFINITY;
        float m = least_of_all(d);
        if (m < best) {
          best = m;
          unsigned long long mask = __ballot(d == m);
          bidx = base + __ffsll((long long)mask) - 1;
        }
      }
      if (bidx >= 0 && best < dcur) {
        dcur = uni(best);
        cur = (uint32_t)uni((int)s.nbuf[bidx]);
        const unsigned long long holds = __ballot(mine == cur);
        if (holds != 0ull) {
          const int l = __builtin_ctzll(holds);
          first = (long long)(((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(firsts >> 32), l) << 32) |
                              (uint32_t)__builtin_amdgcn_readlane((int)firsts, l));
        } else {
          first = ix.upper_off[cur];
        }
        have_below = false;
        changed = true;
      }
      wave_sync();
    }
  }
}

// key of one node against the query (all lanes return it)
template <int DT, int QR>
__device__ __forceinline__ float dist_single(const DevIndex& ix, const QVec<QR>& qv, uint32_t id, Scratch& s, int lane) {
  if (lane == 0) s.nbuf[0] = id;
  wave_sync();
  dist_list<DT, QR, false>(ix, qv, s.qlds, s.nbuf, 1, s.dbuf, lane);
  wave_sync();
  float d = s.dbuf[0];
  wave_sync();
  return d;
}

// Ascending (key, tie) ranking of n LDS entries into out_id / out_key (rank sort,
// O(n^2 / 64) per lane).  tie[] may be null (then the id breaks ties).
__device__ __forceinline__ void rank_sort(const HeapEnt* in, const uint64_t* tie, int n, uint32_t* out_id, float* out_key,
                                          int lane) {
  for (int e = lane; e < n; e += 64) {
    HeapEnt me = in[e];
    uint64_t mt = tie ? tie[e] : (uint64_t)me.id;
    int rank = 0;
    for (int f = 0; f < n; ++f) {
      HeapEnt o = in[f];
      uint64_t ot = tie ? tie[f] : (uint64_t)o.id;
      rank += (o.key < me.key || (o.key == me.key && ot < mt)) ? 1 : 0;
    }
    out_id[rank] = me.id;
    out_key[rank] = me.key;
  }
}

// ids[0..n) with keys[0..n) ascending (LDS): puts the ids of every run of equal keys into the
// order of their labels, which is how hnswlib's answer orders equal distances (its result queue
// compares (distance, label) pairs).  tmp: n words of LDS.
__device__ __forceinline__ void order_equal_keys(const DevIndex& ix, uint32_t* ids, const float* keys, int n, uint32_t* tmp,
                                                 int lane) {
  for (int e = lane; e < n; e += 64) tmp[e] = ids[e];
  wave_sync();
  for (int e = lane; e < n; e += 64) {
    const float k = keys[e];
    const uint32_t me = tmp[e];
    const uint64_t ml = ix.labels ? ix.labels[me] : (uint64_t)me;
    int rank = e;
    for (int f = e - 1; f >= 0 && keys[f] == k; --f) {
      const uint32_t o = tmp[f];
      rank -= (ix.labels ? ix.labels[o] : (uint64_t)o) > ml ? 1 : 0;
    }
    for (int f = e + 1; f < n && keys[f] == k; ++f) {
      const uint32_t o = tmp[f];
      rank += (ix.labels ? ix.labels[o] : (uint64_t)o) < ml ? 1 : 0;
    }
    ids[rank] = me;
  }
  wave_sync();
}

// Collects from the log the entries that make up the k best: those with key <= bound.
// Returns how many there are (they are stored while they fit cap).  More than `want`
// means equal keys straddle the cut, which only the literal heap can resolve.
__device__ __forceinline__ int collect_le(const HeapEnt* log, int n, float bound, HeapEnt* out, int cap, int lane) {
  int cnt = 0;
  for (int base = 0; base < n; base += 64) {
    const int i = base + lane;
    HeapEnt e;
    e.key = INFINITY;
    e.id = 0;
    if (i < n) e = log[i];
    const bool keep = i < n && e.key <= bound;
    const unsigned long long mask = __ballot(keep);
    const int pos = cnt + lanes_below(mask);
    if (keep && pos < cap) out[pos] = e;
    cnt += __popcll(mask);
  }
  return cnt;
}
// Same with a strict bound first and ties filling up to `want` in log order (build: any
// deterministic choice among equal keys is fine).
__device__ __forceinline__ int collect_best(const HeapEnt* log, int n, float bound, int want, HeapEnt* out, int lane) {
  int cnt = 0;
  for (int pass = 0; pass < 2; ++pass) {
    for (int base = 0; base < n && cnt < want; base += 64) {
      const int i = base + lane;
      HeapEnt e;
      e.key = INFINITY;
      e.id = 0;
      if (i < n) e = log[i];
      const bool keep = i < n && (pass == 0 ? e.key < bound : e.key == bound);
      const unsigned long long mask = __ballot(keep);
      const int pos = cnt + lanes_below(mask);
      if (keep && pos < want) out[pos] = e;
      cnt += __popcll(mask);
    }
  }
  return cnt < want ? cnt : want;
}

}  // namespace cuhnsw_amd
