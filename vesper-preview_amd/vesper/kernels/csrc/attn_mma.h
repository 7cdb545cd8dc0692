// MFMA operand helpers shared by the window attention kernels (window_attn.hip: forward;
// window_attn_backward.hip: gradients).
#pragma once
#include "common.h"

#include <algorithm>

namespace vsp {
namespace {

template <typename T> struct Mma;
template <> struct Mma<__bf16> {
  using V8 = bf16x8;
  using V4 = bf16x4;
  __device__ __forceinline__ static f32x4 run(V8 a, V8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<_Float16> {
  using V8 = f16x8;
  using V4 = f16x4;
  __device__ __forceinline__ static f32x4 run(V8 a, V8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <typename T>
__device__ __forceinline__ typename Mma<T>::V4 read_tr(const T* p) {
  return read_tr16<typename Mma<T>::V4>(p);
}

// IEEE maximum (NaN-propagating): v_maximum3_f32 / v_maximum_f32, which need no operand
// canonicalisation, unlike fmaxf's v_max_f32
__device__ __forceinline__ float fmax_ieee(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// max over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (the four lane groups of one query)
__device__ __forceinline__ float max_over_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmax_ieee(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmax_ieee(__uint_as_float(c[0]), __uint_as_float(c[1]));
}

constexpr size_t kCus = 256;  // of an MI355X

// The order of the query tiles (nqt a head, QT queries each) of a kernel that walks each query's window of
// W keys, as query_tile takes it; decided on the host and a template parameter of the kernels, so that
// the in-order kernels are what they would be without the other order (with the choice in the kernel, even
// of one precomputed value, they ran up to 1.5 % longer: 8 workgroups 4.90 -> 4.96 us, B4 N4096 H8 d256 178.8
// -> 181.7).
// In order (0): a head's tiles run on one XCD one after the other. Their key windows overlap, so most of
// each tile's K and V reads hit that XCD's L2.
// Heavy first (the heads of an XCD): the first tiles see fewer than W keys. Where they are a quarter of a
// head's tiles or more, in order some CUs get several full tiles and others short ones; the full ones
// first, the XCD's heads taking turns, even that out once a CU has more than two workgroups. With exactly
// two, full tiles still meet unless half of them are short. Longer sequences keep the order, whose K and V
// reuse counts for more there. In order / heavy first at D 64, us: plain B16 N1024 H8 31.2 / 27.9, B8 N1024
// H8 over 2 20.8 / 18.8, B9 N1024 M300 H8 26.3 / 23.4, B8 N2048 H8 32.0 / 31.4; cached B9 N1024 M300 26.0 /
// 23.6; carried B16 N1024 H8 45.9 / 35.2; forward and backward B16 N1024 H8 134.7 / 124.7. Other widths, B16
// N1024 H8, plain: 16 23.8 / 19.3, 32 23.4 / 20.3, 128 55.7 / 51.3, 256 167.7 / 144.8. Two a CU and a quarter
// short (B4 N2048 H8): 16 carried 17.0 / 17.4, 256 plain 87.9 / 89.9; 64 the same.
inline int query_order(size_t heads, int nqt, int M, int N, int W, int QT) {
  const int64_t light = (std::max<int64_t>(std::min<int64_t>(W, (int64_t)M + N) - 1 - M, 0) + QT - 1) / QT;
  const size_t workgroups = heads * nqt;
  const bool uneven = workgroups > 2 * kCus ? 4 * light >= nqt : workgroups == 2 * kCus && 2 * light >= nqt;
  return uneven && heads % 8 == 0 ? (int)(heads / 8) : 0;
}
// The workgroup's query tile and (batch, head) in that order (HEAVY: it is not 0).
template <bool HEAVY>
__device__ __forceinline__ void query_tile(int nqt, int order, int& qt, int& bh) {
  if constexpr (HEAVY) {  // the XCD's heads take turns, each from its last tile on
    const int r = (int)blockIdx.x >> 3, rank = r / order;
    bh = (int)(blockIdx.x & 7) * order + (r - rank * order);
    qt = nqt - 1 - rank;
  } else {
    const int lg = xcd_logical_block(blockIdx.x, gridDim.x);
    qt = lg % nqt;
    bh = lg / nqt;
  }
}

}  // namespace
}  // namespace vsp
