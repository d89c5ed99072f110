// From a selected position to its row of the latent cache.  No device code in it, so that a
// CPU test can run it against a page table that ends where the address space does.
#pragma once
#include <stddef.h>
#include <stdint.h>

#ifdef __HIPCC__
#define MK2_HOST_DEV __host__ __device__ __forceinline__
#else
#define MK2_HOST_DEV inline
#endif

namespace mk2 {

// whether a position is one of the table's (a list holds -1 for an unused entry)
MK2_HOST_DEV bool mla_on_page(int pos, int stride) { return pos >= 0 && pos < stride * 64; }

// where row r's line of the page table starts.  A pad row, whose list is all unused, need not
// name a request of the table.
MK2_HOST_DEV ptrdiff_t mla_line(const int32_t* req, int r, int stride) { return (ptrdiff_t)req[r] * stride; }

// the page-table entry of a position.  An unused one reads the table's first entry, whatever
// its row's line is (a read and no branch, which would wait for it).
MK2_HOST_DEV int mla_page(const int32_t* pt, ptrdiff_t line, int stride, int pos) {
  return pt[mla_on_page(pos, stride) ? line + (pos >> 6) : 0];
}

MK2_HOST_DEV int mla_cache_row(int pos, int page, int stride) {
  return mla_on_page(pos, stride) ? page * 64 + (pos & 63) : -1;
}

}  // namespace mk2
