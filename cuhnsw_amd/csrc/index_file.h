// Host model of an HNSW index and its hnswlib-compatible file format.
// Replaces CuHNSW::SaveIndex / LoadIndex (cpp/src/cuhnsw_base.cu:159-365 in the
// reference) and the host graph container LevelGraph
// (cpp/include/level_graph.hpp:23-89): adjacency is kept in the same flat,
// fixed-stride rows the GPU uses, so upload and download are plain copies.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

namespace cuhnsw_amd {

constexpr uint32_t kEmpty = 0xFFFFFFFFu;  // unused link slot

struct HostIndex {
  int N = 0, D = 0;
  int max_m = 12, max_m0 = 24, M = 12, ef_construction = 150;
  double mult = 0.0;
  int maxlevel = 0;
  uint32_t enterpoint = 0;
  bool labelled = false;               // labels came from a file
  std::vector<float> vectors;          // N x D
  std::vector<uint64_t> labels;        // N
  std::vector<int> levels;             // N, number of upper levels of a node
  int S0 = 32, SU = 16;                // row strides (uint32 slots) of level 0 / upper levels
  std::vector<uint32_t> links0;        // N x S0, first deg slots hold ids, the rest kEmpty
  std::vector<int64_t> upper_off;      // N: index of the node's level-1 row in linksU, -1 if none
  std::vector<uint32_t> linksU;        // (sum of levels) x SU; row of (node, level) = upper_off[node] + level - 1
  int64_t upper_rows = 0;
  // hnswlib's delete marks (markDelete: bit 0 of the third byte of an element's level-0 count word), one
  // byte per element, or empty when nothing is marked.  A marked element is searched through like any
  // other and never returned.  The reference keeps no such mark: it reads the count word as a plain count
  // (cpp/src/cuhnsw_base.cu:311-312).
  std::vector<uint8_t> deleted;
  int n_deleted = 0;

  static int stride0(int max_m0) { return (max_m0 + 31) / 32 * 32; }
  static int strideU(int max_m) { return (max_m + 15) / 16 * 16; }
  // strides, offsets and number of upper rows from N, levels, max_m, max_m0
  void layout_upper();
  // the same, and empty link tables on the host (an engine with a GPU keeps its links there)
  void layout_links();
  // max level and entry point from levels: the first node that reaches the
  // maximal level (cpp/src/cuhnsw_base.cu:133-141; node 0 if every level is 0)
  void set_levels(const int* lv, int n);
};

constexpr uint32_t kDeleteMark = 0x00010000u;  // hnswlib's DELETE_MARK as a bit of the level-0 count word

// Where things sit in an index file: a header, N level-0 records, the upper block.
struct FileLayout {
  static constexpr uint64_t kHeader = 96;
  uint64_t links0_bytes = 0;  // bytes of a record's link part = offset of its vector
  uint64_t linksU_bytes = 0;  // bytes of one upper-level link list
  uint64_t label_offset = 0;  // offset of a record's label
  uint64_t record = 0;        // bytes of a record
  FileLayout() {}
  FileLayout(uint64_t max_m, uint64_t max_m0, uint64_t D)
      : links0_bytes(max_m0 * 4 + 4), linksU_bytes(max_m * 4 + 4), label_offset(links0_bytes + D * 4), record(label_offset + 8) {}
};

// An index file opened for reading.  The constructor checks the header; read() is safe to call from several
// threads and throws "index file: truncated <what>" where the file ends early.
class IndexReader {
 public:
  IndexReader(HostIndex& ix, const std::string& path);  // fills the header's fields of ix
  ~IndexReader();
  IndexReader(const IndexReader&) = delete;
  IndexReader& operator=(const IndexReader&) = delete;
  void read(uint64_t offset, void* dst, size_t n, const char* what) const;
  // levels, offsets and upper links (on the host) of ix from the block behind the records; links are checked
  void read_upper(HostIndex& ix) const;
  // Once everything has been read: throws if the file was written to meanwhile (a save goes over a file in place: what
  // was read may be part of one index and part of another).
  void check_unchanged() const;
  FileLayout layout;

 private:
  int fd_ = -1;
  std::vector<unsigned char> memory_;  // the whole file where it cannot be read by position (a pipe)
  bool in_memory_ = false;
  uint64_t size_ = 0;
  uint64_t upper_at_ = 0;
  long long seconds_ = 0, nanoseconds_ = 0;  // when the file was last written, as it was opened
  unsigned char header_[FileLayout::kHeader];
};

// An index file opened for writing; its size is known from the start.  write() may be called from several threads
// where parallel() says so, else in ascending order without gaps.  A regular file has no header until finish() puts it
// there, as the last thing of all: a save that does not get that far, for whatever reason, leaves nothing that loads (and
// an empty file where the destructor still runs).
class IndexWriter {
 public:
  IndexWriter(const HostIndex& ix, const std::string& path);
  ~IndexWriter();
  IndexWriter(const IndexWriter&) = delete;
  IndexWriter& operator=(const IndexWriter&) = delete;
  bool parallel() const { return regular_; }
  void write(uint64_t offset, const void* src, size_t n);
  // the upper block from ix.levels / upper_off and the link rows given (upper_rows x SU)
  void write_upper(const HostIndex& ix, const uint32_t* linksU);
  void finish();
  FileLayout layout;

 private:
  int fd_ = -1;
  bool regular_ = false;
  unsigned char* map_ = nullptr;
  uint64_t size_ = 0, upper_at_ = 0;
  unsigned char header_[FileLayout::kHeader];
  std::string path_;
};

// Both throw std::runtime_error with a message on I/O or format errors.  (Host tables only: an engine with a GPU
// moves records between the file and device memory itself, engine.h.)
void write_index_file(const HostIndex& ix, const std::string& path);
void read_index_file(HostIndex& ix, const std::string& path);

}  // namespace cuhnsw_amd
