// TEST-ONLY: which pages of a fresh array the host side's map_pages maps.
// Built by tests/test_map_pages.py.
#include <sys/mman.h>

#include <cstring>
#include <vector>

#include "../../zisafvm_amd/csrc/setup.hpp"

// Maps n doubles at an offset of `skip` doubles into a fresh region of small
// pages, of which the first `keep` hold values; busy answers yes `polls` times.
// mapped[k]: page k of the region is there afterwards.  Returns the region's
// pages, or -1 if a value changed.
extern "C" int pages_mapped(int64_t n, int64_t skip, int64_t keep, int all, int polls, unsigned char *mapped) {
  const size_t page = 4096, bytes = ((skip + n) * 8 + 2 * page) / page * page, pages = bytes / page;
  auto *p = static_cast<double *>(mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
  if (p == MAP_FAILED) return -2;
  (void)madvise(p, bytes, MADV_NOHUGEPAGE);
  for (int64_t k = 0; k < keep * 512; ++k) p[k] = double(k) + 0.5;
  zfv::map_pages(p + skip, size_t(n), all != 0, [&] { return polls-- > 0; });
  std::vector<unsigned char> in(pages);
  int rc = mincore(p, bytes, in.data()) == 0 ? int(pages) : -2;
  for (size_t k = 0; k < pages; ++k) mapped[k] = in[k] & 1;
  for (int64_t k = 0; k < keep * 512; ++k)
    if (p[k] != double(k) + 0.5) rc = -1;
  munmap(p, bytes);
  return rc;
}

extern "C" int64_t map_whole_bytes() { return int64_t(zfv::kMapWhole); }
