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

// row r's page-table entry for a position.  An unused one reads the table's first entry,
// whatever the row's request id is: a pad row, whose list is all unused, need not name a
// request of the table.  (A read and no branch, which would wait for it.)
MK2_HOST_DEV int mla_page(const int32_t* pt, const int32_t* req, int r, int stride, int pos) {
  const ptrdiff_t at = (ptrdiff_t)req[r] * stride + (pos >> 6);
  return pt[mla_on_page(pos, stride) ? at : 0];
}

MK2_HOST_DEV int mla_cache_row(int pos, int page, int stride) {
  return mla_on_page(pos, stride) ? page * 64 + (pos & 63) : -1;
}

}  // namespace mk2
