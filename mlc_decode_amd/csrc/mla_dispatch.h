// mla_dispatch.h -- which decodes the wide kernel takes (host code, no HIP: the CPU tests compile
// these rules by themselves).
#pragma once
#include <stdint.h>

namespace mla {

// The wide kernel's sparse form multiplies a page id by a 32-bit page stride; the one-ring kernel
// does so in 64 bits.  The C ABI bounds the page strides of a block table below 2^32 elements and
// those of an index list not at all.
inline bool wide_takes_sparse(int64_t kv_stride_page, int64_t kv_rope_stride_page) {
  constexpr int64_t kLimit = int64_t(1) << 32;
  return kv_stride_page < kLimit && kv_rope_stride_page < kLimit;
}

}  // namespace mla
