// Saves that go wrong, on the host side of the index file alone: file_faults MODE PATH.  An index of 4 000 nodes is
// written; every component of its vectors is the index's number, so that a mixture of two of them can be told.
//   write K      index number K, whole
//   throw K      upper block and half of the records, then an exception (the writer is destroyed)
//   die K        the same, then the process ends without running any destructor
//   cut K        half of the records, then the file is cut to nothing by somebody else, then the other half
//   read         prints the lowest and the highest component found
//   overtaken K  half of the records are read, index number K is saved over the file, the other half is read
// Prints "refused: ..." where the library throws.
#include <fcntl.h>
#include <unistd.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "index_file.h"

using namespace cuhnsw_amd;

static HostIndex make(float number) {
  HostIndex ix;
  ix.N = 4000;
  ix.D = 60;
  ix.max_m = 2;
  ix.max_m0 = 3;
  std::vector<int> levels(ix.N, 0);
  for (int i = 0; i < ix.N; i += 7) levels[i] = 1;
  ix.set_levels(levels.data(), ix.N);
  ix.layout_links();
  for (int i = 0; i < ix.N; ++i) ix.links0[(size_t)i * ix.S0] = (uint32_t)((i + 1) % ix.N);
  ix.vectors.assign((size_t)ix.N * ix.D, number);
  return ix;
}

static std::vector<unsigned char> records(const HostIndex& ix, const FileLayout& fl, int from, int to) {
  std::vector<unsigned char> out((size_t)(to - from) * fl.record, 0);
  for (int i = from; i < to; ++i) {
    unsigned char* rec = out.data() + (size_t)(i - from) * fl.record;
    const uint32_t deg = 1, link = (uint32_t)((i + 1) % ix.N);
    const uint64_t label = (uint64_t)i;
    std::memcpy(rec, &deg, 4);
    std::memcpy(rec + 4, &link, 4);
    std::memcpy(rec + fl.links0_bytes, &ix.vectors[(size_t)i * ix.D], (size_t)ix.D * 4);
    std::memcpy(rec + fl.label_offset, &label, 8);
  }
  return out;
}

static void half(IndexWriter& out, const HostIndex& ix, int which) {
  const int from = which ? ix.N / 2 : 0, to = which ? ix.N : ix.N / 2;
  const std::vector<unsigned char> r = records(ix, out.layout, from, to);
  out.write(FileLayout::kHeader + (uint64_t)from * out.layout.record, r.data(), r.size());
}

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const std::string mode = argv[1], path = argv[2];
  const HostIndex ix = make(argc > 3 ? (float)std::atof(argv[3]) : 0.f);
  try {
    if (mode == "write") {
      write_index_file(ix, path);
    } else if (mode == "throw" || mode == "die") {
      IndexWriter out(ix, path);
      out.write_upper(ix, ix.linksU.data());
      half(out, ix, 0);
      if (mode == "die") _exit(0);
      throw std::runtime_error("the device is gone");
    } else if (mode == "cut") {
      IndexWriter out(ix, path);
      half(out, ix, 0);
      if (::truncate(path.c_str(), 0) != 0) return 3;
      half(out, ix, 1);
      out.write_upper(ix, ix.linksU.data());
      out.finish();
    } else if (mode == "read") {
      HostIndex got;
      read_index_file(got, path);
      const auto ends = std::minmax_element(got.vectors.begin(), got.vectors.end());
      std::printf("%g %g\n", *ends.first, *ends.second);
    } else if (mode == "overtaken") {
      HostIndex got;
      IndexReader in(got, path);
      const size_t bytes = (size_t)got.N / 2 * in.layout.record;
      std::vector<unsigned char> buf(bytes);
      in.read(FileLayout::kHeader, buf.data(), bytes, "level-0 block");
      write_index_file(ix, path);
      in.read(FileLayout::kHeader + bytes, buf.data(), bytes, "level-0 block");
      in.read_upper(got);
      in.check_unchanged();
      std::printf("accepted\n");
    } else {
      return 2;
    }
  } catch (const std::exception& ex) {
    std::printf("refused: %s\n", ex.what());
  }
  return 0;
}
