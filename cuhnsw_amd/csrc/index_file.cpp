// hnswlib index file reader / writer (byte layout: 96-byte header, N level-0
// records [count | max_m0 ids | D floats | label], then per node a uint32 byte
// size followed by its upper-level link lists).  Same layout as the reference's
// CuHNSW::SaveIndex / LoadIndex (cpp/src/cuhnsw_base.cu:159-365).
#include "index_file.h"

#include <errno.h>
#include <fcntl.h>
#include <linux/magic.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <sys/uio.h>
#include <sys/vfs.h>
#include <unistd.h>

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>

namespace cuhnsw_amd {

void HostIndex::layout_upper() {
  S0 = stride0(max_m0);
  SU = strideU(max_m);
  upper_off.resize(N);
  int64_t rows = 0;
  for (int i = 0; i < N; ++i) {
    upper_off[i] = levels[i] > 0 ? rows : -1;
    rows += levels[i];
  }
  upper_rows = rows;
}

void HostIndex::layout_links() {
  layout_upper();
  links0.assign((size_t)N * S0, kEmpty);
  linksU.assign((size_t)upper_rows * SU, kEmpty);
}

void HostIndex::set_levels(const int* lv, int n) {
  levels.assign(lv, lv + n);
  maxlevel = 0;
  enterpoint = 0;
  for (int i = 0; i < n; ++i) {
    if (lv[i] < 0) throw std::runtime_error("levels must be non-negative");
    if (lv[i] > maxlevel) {
      maxlevel = lv[i];
      enterpoint = (uint32_t)i;
    }
  }
}

namespace {

// the header's fields by their place in the file (the layout must not depend on a compiler's padding)
struct HeaderField {
  unsigned char bytes[FileLayout::kHeader];
  template <typename T>
  T get(size_t at) const {
    T v;
    std::memcpy(&v, bytes + at, sizeof(T));
    return v;
  }
  template <typename T>
  void put(size_t at, T v) {
    std::memcpy(bytes + at, &v, sizeof(T));
  }
};
enum : size_t {  // byte offsets: eight-byte fields but for maxlevel and enterpoint
  kOffsetLevel0 = 0, kMaxElements = 8, kCount = 16, kRecord = 24, kLabelOffset = 32, kOffsetData = 40,
  kMaxLevel = 48, kEnterPoint = 52, kMaxM = 56, kMaxM0 = 64, kM = 72, kMult = 80, kEfConstruction = 88
};

int row_degree(const uint32_t* row, int cap) {
  int d = 0;
  while (d < cap && row[d] != kEmpty) ++d;
  return d;
}

void write_at(int fd, uint64_t offset, const void* src, size_t n) {
  const unsigned char* p = static_cast<const unsigned char*>(src);
  while (n > 0) {
    const ssize_t got = ::pwrite(fd, p, n, (off_t)offset);
    if (got < 0 && errno == EINTR) continue;
    if (got <= 0) throw std::runtime_error("index file: write failed");
    p += got;
    offset += (uint64_t)got;
    n -= (size_t)got;
  }
}

void write_all(int fd, const void* src, size_t n) {
  const unsigned char* p = static_cast<const unsigned char*>(src);
  while (n > 0) {
    const ssize_t got = ::write(fd, p, n);
    if (got < 0 && errno == EINTR) continue;
    if (got <= 0) throw std::runtime_error("index file: write failed");
    p += got;
    n -= (size_t)got;
  }
}

}  // namespace

// ---- reading -------------------------------------------------------------------------------------------
IndexReader::IndexReader(HostIndex& ix, const std::string& path) {
  fd_ = ::open(path.c_str(), O_RDONLY | O_CLOEXEC);
  if (fd_ < 0) throw std::runtime_error("cannot open index file: " + path);
  try {
    struct stat st;
    if (::fstat(fd_, &st) == 0 && S_ISREG(st.st_mode)) {
      size_ = (uint64_t)st.st_size;
      seconds_ = st.st_mtim.tv_sec;
      nanoseconds_ = st.st_mtim.tv_nsec;
    } else {
      in_memory_ = true;
      size_t have = 0;
      for (;;) {
        memory_.resize(have + ((size_t)1 << 20));
        const ssize_t got = ::read(fd_, memory_.data() + have, (size_t)1 << 20);
        if (got < 0 && errno == EINTR) continue;
        if (got <= 0) break;
        have += (size_t)got;
      }
      memory_.resize(have);
      size_ = have;
    }
    HeaderField h;
    read(0, h.bytes, sizeof(h.bytes), "header");
    std::memcpy(header_, h.bytes, sizeof(header_));
    const uint64_t count = h.get<uint64_t>(kCount), max_elements = h.get<uint64_t>(kMaxElements);
    const uint64_t max_m = h.get<uint64_t>(kMaxM), max_m0 = h.get<uint64_t>(kMaxM0);
    const uint64_t offset_data = h.get<uint64_t>(kOffsetData), label_offset = h.get<uint64_t>(kLabelOffset);
    const uint64_t record = h.get<uint64_t>(kRecord);
    const int32_t maxlevel = h.get<int32_t>(kMaxLevel);
    if (count > 0x7fffffffull || max_m == 0 || max_m0 == 0 || max_m > 65535 || max_m0 > 65535 ||
        offset_data != max_m0 * 4 + 4 || label_offset <= offset_data || (label_offset - offset_data) % 4 != 0 ||
        record != label_offset + 8 || count > max_elements || maxlevel < 0)
      throw std::runtime_error("index file: inconsistent header");
    ix.N = (int)count;
    ix.D = (int)((label_offset - offset_data) / 4);
    ix.max_m = (int)max_m;
    ix.max_m0 = (int)max_m0;
    ix.M = (int)h.get<uint64_t>(kM);
    ix.mult = h.get<double>(kMult);
    ix.ef_construction = (int)h.get<uint64_t>(kEfConstruction);
    ix.maxlevel = maxlevel;
    ix.enterpoint = h.get<uint32_t>(kEnterPoint);
    if (ix.N > 0 && ix.enterpoint >= (uint32_t)ix.N) throw std::runtime_error("index file: entry point out of range");
    ix.labelled = true;
    layout = FileLayout(max_m, max_m0, (uint64_t)ix.D);
    // (a header may promise more room than any file has: the block's end is looked at, never computed past 2^64)
    if (size_ < FileLayout::kHeader || (size_ - FileLayout::kHeader) / record < count)
      throw std::runtime_error("index file: truncated level-0 block");
    if ((size_ - FileLayout::kHeader) / record < max_elements) upper_at_ = size_;  // the block behind it is missing
    else upper_at_ = FileLayout::kHeader + max_elements * record;
  } catch (...) {
    ::close(fd_);
    throw;
  }
}

IndexReader::~IndexReader() { ::close(fd_); }

void IndexReader::read(uint64_t offset, void* dst, size_t n, const char* what) const {
  if (offset > size_ || n > size_ - offset) throw std::runtime_error(std::string("index file: truncated ") + what);
  if (in_memory_) {
    if (n > 0) std::memcpy(dst, memory_.data() + offset, n);
    return;
  }
  unsigned char* p = static_cast<unsigned char*>(dst);
  while (n > 0) {
    const ssize_t got = ::pread(fd_, p, n, (off_t)offset);
    if (got < 0 && errno == EINTR) continue;
    if (got <= 0) throw std::runtime_error(std::string("index file: truncated ") + what);
    p += got;
    offset += (uint64_t)got;
    n -= (size_t)got;
  }
}

void IndexReader::check_unchanged() const {
  if (in_memory_) return;
  struct stat st;
  unsigned char now[FileLayout::kHeader];
  const bool same = ::fstat(fd_, &st) == 0 && (uint64_t)st.st_size == size_ && st.st_mtim.tv_sec == seconds_ &&
                    st.st_mtim.tv_nsec == nanoseconds_ && ::pread(fd_, now, sizeof(now), 0) == (ssize_t)sizeof(now) &&
                    std::memcmp(now, header_, sizeof(now)) == 0;
  if (!same) throw std::runtime_error("index file: written to while it was read");
}

void IndexReader::read_upper(HostIndex& ix) const {
  std::vector<unsigned char> block(size_ - upper_at_);
  read(upper_at_, block.data(), block.size(), "upper block");
  const size_t per_list = (size_t)layout.linksU_bytes;
  // where each node's lists start; the lists are checked once every level is known
  ix.levels.assign(ix.N, 0);
  std::vector<size_t> start(ix.N);
  size_t at = 0;
  for (int i = 0; i < ix.N; ++i) {
    uint32_t bytes;
    if (block.size() - at < 4) throw std::runtime_error("index file: truncated upper block");
    std::memcpy(&bytes, block.data() + at, 4);
    at += 4;
    start[i] = at;
    if (bytes == 0) continue;
    if (bytes % per_list != 0) throw std::runtime_error("index file: bad upper list size");
    ix.levels[i] = (int)(bytes / per_list);
    if (ix.levels[i] > ix.maxlevel) throw std::runtime_error("index file: node level above maxlevel");
    if (block.size() - at < bytes) throw std::runtime_error("index file: truncated upper block");
    at += bytes;
  }
  ix.layout_upper();
  ix.linksU.assign((size_t)ix.upper_rows * ix.SU, kEmpty);
  for (int i = 0; i < ix.N; ++i)
    for (int l = 1; l <= ix.levels[i]; ++l) {
      const unsigned char* src = block.data() + start[i] + (size_t)(l - 1) * per_list;
      uint32_t deg;
      std::memcpy(&deg, src, 4);
      deg &= 0xffffu;
      if (deg > (uint32_t)ix.max_m) throw std::runtime_error("index file: link count above max_m");
      uint32_t* row = &ix.linksU[(size_t)(ix.upper_off[i] + l - 1) * ix.SU];
      for (uint32_t k = 0; k < deg; ++k) {
        uint32_t id;
        std::memcpy(&id, src + 4 + 4 * (size_t)k, 4);
        if (id >= (uint32_t)ix.N) throw std::runtime_error("index file: link id out of range");
        if (ix.levels[id] < l) throw std::runtime_error("index file: link to a node that lacks that level");
        row[k] = id;
      }
    }
  if (ix.N > 0 && ix.levels[ix.enterpoint] < ix.maxlevel) throw std::runtime_error("index file: entry point below maxlevel");
}

// ---- writing -------------------------------------------------------------------------------------------
IndexWriter::IndexWriter(const HostIndex& ix, const std::string& path)
    : layout((uint64_t)ix.max_m, (uint64_t)ix.max_m0, (uint64_t)ix.D), path_(path) {
  upper_at_ = FileLayout::kHeader + (uint64_t)ix.N * layout.record;
  size_ = upper_at_ + (uint64_t)ix.N * 4 + (uint64_t)ix.upper_rows * layout.linksU_bytes;
  // A file that is there is written over in place and cut to its new length at the end: its pages need not be
  // given back and taken again (364 MB in memory: 20 ms and 60 ms).
  struct stat st;
  const bool special = ::stat(path.c_str(), &st) == 0 && !S_ISREG(st.st_mode);  // a pipe, a device
  if (!special) fd_ = ::open(path.c_str(), O_RDWR | O_CREAT | O_CLOEXEC, 0666);
  const bool readable = fd_ >= 0;
  if (!readable) fd_ = ::open(path.c_str(), O_WRONLY | O_CREAT | O_TRUNC | O_CLOEXEC, 0666);  // (what can be written only)
  if (fd_ < 0) throw std::runtime_error("cannot open index file for writing: " + path);
  regular_ = ::fstat(fd_, &st) == 0 && S_ISREG(st.st_mode);
  if (readable && regular_) {
    // Room first, where the file system can say that there is none: a file that is there stays as it was then.
    const bool there = (uint64_t)st.st_size >= size_ && (uint64_t)st.st_blocks * 512 >= size_;
    int rc = 0;
    if (!there) {
      do rc = ::fallocate(fd_, 0, 0, (off_t)size_);
      while (rc != 0 && errno == EINTR);
      if (rc != 0 && (errno == ENOSPC || errno == EDQUOT || errno == EFBIG)) {
        (void)!::ftruncate(fd_, st.st_size);
        ::close(fd_);
        throw std::runtime_error("index file: write failed");
      }
    }
    // In memory (tmpfs) the file is written through a mapping: write() holds the file's lock, pages of a mapping are
    // filled by several threads side by side (364 MB over a file that is there: 7 ms, 20 to 25 with pwrite on one thread
    // or eight).  On a disk's file system a mapping costs more than it saves (61 ms, 13 with pwrite).
    struct statfs fs;
    if (rc == 0 && ::fstatfs(fd_, &fs) == 0 && fs.f_type == TMPFS_MAGIC) {
      void* p = ::mmap(nullptr, size_, PROT_READ | PROT_WRITE, MAP_SHARED, fd_, 0);
      if (p != MAP_FAILED) map_ = static_cast<unsigned char*>(p);
    }
  }
  HeaderField h;
  h.put<uint64_t>(kOffsetLevel0, 0);
  h.put<uint64_t>(kMaxElements, (uint64_t)ix.N);
  h.put<uint64_t>(kCount, (uint64_t)ix.N);
  h.put<uint64_t>(kRecord, layout.record);
  h.put<uint64_t>(kLabelOffset, layout.label_offset);
  h.put<uint64_t>(kOffsetData, layout.links0_bytes);
  h.put<int32_t>(kMaxLevel, ix.maxlevel);
  h.put<uint32_t>(kEnterPoint, ix.enterpoint);
  h.put<uint64_t>(kMaxM, (uint64_t)ix.max_m);
  h.put<uint64_t>(kMaxM0, (uint64_t)ix.max_m0);
  h.put<uint64_t>(kM, (uint64_t)ix.M);
  h.put<double>(kMult, ix.mult);
  h.put<uint64_t>(kEfConstruction, (uint64_t)ix.ef_construction);
  std::memcpy(header_, h.bytes, sizeof(header_));
  try {
    static const unsigned char none[FileLayout::kHeader] = {};
    if (regular_) write_at(fd_, 0, none, sizeof(none));  // from here on the file is no index, until finish() says so
    else write_all(fd_, header_, sizeof(header_));
  } catch (...) {
    if (map_) ::munmap(map_, size_);
    ::close(fd_);
    throw;
  }
}

IndexWriter::~IndexWriter() {
  if (map_) ::munmap(map_, size_);
  if (fd_ < 0) return;
  if (regular_) (void)!::ftruncate(fd_, 0);  // not finished
  ::close(fd_);
}

void IndexWriter::write(uint64_t offset, const void* src, size_t n) {
  if (map_) {
    // The kernel makes the copy: a page that cannot be had (no room for it, the file cut off by somebody else) is an
    // error there, where a store of this process would end it with a bus error.
    const unsigned char* from = static_cast<const unsigned char*>(src);
    while (n > 0) {
      struct iovec local = {const_cast<unsigned char*>(from), n}, remote = {map_ + offset, n};
      const ssize_t got = ::process_vm_writev(::getpid(), &local, 1, &remote, 1, 0);
      if (got <= 0) {
        if (got < 0 && (errno == EINTR || errno == EAGAIN)) continue;
        if (got < 0 && (errno == ENOSYS || errno == EPERM)) break;  // (not allowed here: pwrite below)
        throw std::runtime_error("index file: write failed");
      }
      from += got;
      offset += (uint64_t)got;
      n -= (size_t)got;
    }
    src = from;
    if (n == 0) return;
  }
  if (regular_) write_at(fd_, offset, src, n);
  else write_all(fd_, src, n);
}

void IndexWriter::write_upper(const HostIndex& ix, const uint32_t* linksU) {
  std::vector<unsigned char> block((size_t)(size_ - upper_at_), 0);
  unsigned char* dst = block.data();
  for (int i = 0; i < ix.N; ++i) {
    const uint32_t bytes = (uint32_t)(layout.linksU_bytes * (uint64_t)ix.levels[i]);
    std::memcpy(dst, &bytes, 4);
    dst += 4;
    for (int l = 1; l <= ix.levels[i]; ++l) {
      const uint32_t* row = linksU + (size_t)(ix.upper_off[i] + l - 1) * ix.SU;
      const uint32_t deg = (uint32_t)row_degree(row, ix.max_m);
      std::memcpy(dst, &deg, 4);
      std::memcpy(dst + 4, row, (size_t)deg * 4);
      dst += layout.linksU_bytes;
    }
  }
  write(upper_at_, block.data(), block.size());
}

void IndexWriter::finish() {
  if (map_) {
    ::munmap(map_, size_);
    map_ = nullptr;
  }
  if (regular_) {
    if (::ftruncate(fd_, (off_t)size_) != 0) throw std::runtime_error("index file: write failed");
    write_at(fd_, 0, header_, sizeof(header_));
  }
  const int fd = fd_;
  fd_ = -1;
  if (::close(fd) != 0) {  // (where what was written leaves for a server only now)
    if (regular_) (void)!::truncate(path_.c_str(), 0);
    throw std::runtime_error("index file: write failed");
  }
}

// ---- host tables <-> file ------------------------------------------------------------------------------
void write_index_file(const HostIndex& ix, const std::string& path) {
  IndexWriter out(ix, path);
  const FileLayout& fl = out.layout;
  const int block = (int)std::max<uint64_t>(1, (1 << 20) / fl.record);
  std::vector<unsigned char> buf;
  for (int i0 = 0; i0 < ix.N; i0 += block) {
    const int n = std::min(block, ix.N - i0);
    buf.assign((size_t)n * fl.record, 0);  // unused link slots are written as zeros
    for (int i = i0; i < i0 + n; ++i) {
      unsigned char* rec = buf.data() + (size_t)(i - i0) * fl.record;
      const uint32_t* row = &ix.links0[(size_t)i * ix.S0];
      uint32_t deg = (uint32_t)row_degree(row, ix.max_m0);
      std::memcpy(rec + 4, row, (size_t)deg * 4);
      if (ix.n_deleted > 0 && ix.deleted[i]) deg |= kDeleteMark;
      std::memcpy(rec, &deg, 4);
      std::memcpy(rec + fl.links0_bytes, &ix.vectors[(size_t)i * ix.D], (size_t)ix.D * 4);
      const uint64_t label = ix.labels.empty() ? (uint64_t)i : ix.labels[i];
      std::memcpy(rec + fl.label_offset, &label, 8);
    }
    out.write(FileLayout::kHeader + (uint64_t)i0 * fl.record, buf.data(), buf.size());
  }
  out.write_upper(ix, ix.linksU.data());
  out.finish();
}

void read_index_file(HostIndex& ix, const std::string& path) {
  IndexReader in(ix, path);
  const FileLayout& fl = in.layout;
  ix.vectors.resize((size_t)ix.N * ix.D);
  ix.labels.resize(ix.N);
  ix.deleted.clear();
  ix.n_deleted = 0;
  const int S0 = HostIndex::stride0(ix.max_m0);
  ix.links0.assign((size_t)ix.N * S0, kEmpty);
  const int block = (int)std::max<uint64_t>(1, (1 << 20) / fl.record);
  std::vector<unsigned char> buf;
  for (int i0 = 0; i0 < ix.N; i0 += block) {
    const int n = std::min(block, ix.N - i0);
    buf.resize((size_t)n * fl.record);
    in.read(FileLayout::kHeader + (uint64_t)i0 * fl.record, buf.data(), buf.size(), "level-0 block");
    for (int i = i0; i < i0 + n; ++i) {
      const unsigned char* rec = buf.data() + (size_t)(i - i0) * fl.record;
      uint32_t word;
      std::memcpy(&word, rec, 4);
      const uint32_t deg = word & 0xffffu;  // hnswlib keeps the count in the low 16 bits, flags above
      // hnswlib's markDelete sets bit 0 of the word's third byte; the other flag bits are unknown and dropped
      // (the reference reads the word as a plain count, cpp/src/cuhnsw_base.cu:311-312, and would index out
      // of its rows)
      if (word & kDeleteMark) {
        if (ix.deleted.empty()) ix.deleted.assign(ix.N, 0);
        ix.deleted[i] = 1;
        ++ix.n_deleted;
      }
      if (deg > (uint32_t)ix.max_m0) throw std::runtime_error("index file: link count above max_m0");
      uint32_t* row = &ix.links0[(size_t)i * S0];
      std::memcpy(row, rec + 4, (size_t)deg * 4);
      for (uint32_t k = 0; k < deg; ++k)
        if (row[k] >= (uint32_t)ix.N) throw std::runtime_error("index file: link id out of range");
      std::memcpy(&ix.vectors[(size_t)i * ix.D], rec + fl.links0_bytes, (size_t)ix.D * 4);
      std::memcpy(&ix.labels[i], rec + fl.label_offset, 8);
    }
  }
  in.read_upper(ix);
  in.check_unchanged();
}

}  // namespace cuhnsw_amd
