// Token rows of several tensors copied together (carry.hip: where flags say so; norm.hip: where a token
// halts).
#pragma once
#include "common.h"

namespace vsp {
namespace {

constexpr int kMaxItems = 8;

struct RowItems {
  const uint8_t* src[kMaxItems];
  uint8_t* dst[kMaxItems];
  unsigned row_units[kMaxItems];  // copy units per row
  unsigned unit_log2[kMaxItems];  // a unit is 1 << unit_log2 bytes (1 .. 16)
  int count;
};

template <typename U>
__device__ __forceinline__ void copy_unit(const uint8_t* src, uint8_t* dst, size_t u) {
  reinterpret_cast<U*>(dst)[u] = reinterpret_cast<const U*>(src)[u];
}

// Row `row` of item i by one wave, in units of 1 << unit_log2 bytes.
__device__ __forceinline__ void copy_row_item(const RowItems& items, int i, unsigned row) {
  const unsigned per = items.row_units[i], lane = threadIdx.x & 63;
  const size_t base = (size_t)row * per;
  const uint8_t* s = items.src[i];
  uint8_t* d = items.dst[i];
  for (unsigned u = lane; u < per; u += 64) {
    switch (items.unit_log2[i]) {
      case 4: copy_unit<uint4>(s, d, base + u); break;
      case 3: copy_unit<uint2>(s, d, base + u); break;
      case 2: copy_unit<uint32_t>(s, d, base + u); break;
      case 1: copy_unit<uint16_t>(s, d, base + u); break;
      default: copy_unit<uint8_t>(s, d, base + u); break;
    }
  }
}
__device__ __forceinline__ void copy_row_items(const RowItems& items, unsigned row) {
  for (int i = 0; i < items.count; ++i) copy_row_item(items, i, row);
}

// Fills `items` from host arrays of `count` entries; returns OK or the error it has set.
inline int row_items(RowItems& items, int count, const void* const* src, void* const* dst, const size_t* row_bytes,
                     const char* who) {
  if (count < 0 || count > kMaxItems) return fail(ERR_ARG, "%s: %d tensors (1 .. %d per launch)", who, count, kMaxItems);
  items.count = count;
  if (count > 0 && (!src || !dst || !row_bytes)) return fail(ERR_ARG, "%s: null array", who);
  for (int i = 0; i < count; ++i) {
    if (!src[i] || !dst[i]) return fail(ERR_ARG, "%s: null pointer in tensor %d", who, i);
    if (row_bytes[i] == 0) return fail(ERR_ARG, "%s: tensor %d has empty rows", who, i);
    const uintptr_t mix = reinterpret_cast<uintptr_t>(src[i]) | reinterpret_cast<uintptr_t>(dst[i]) | row_bytes[i];
    unsigned lg = 4;
    while (lg > 0 && (mix & ((1u << lg) - 1)) != 0) --lg;
    const size_t per = row_bytes[i] >> lg;
    if (per > 0xFFFFFFFFu) return fail(ERR_UNSUPPORTED, "%s: rows of %zu bytes", who, row_bytes[i]);
    items.src[i] = static_cast<const uint8_t*>(src[i]);
    items.dst[i] = static_cast<uint8_t*>(dst[i]);
    items.row_units[i] = (unsigned)per;
    items.unit_log2[i] = lg;
  }
  return OK;
}

}  // namespace
}  // namespace vsp
