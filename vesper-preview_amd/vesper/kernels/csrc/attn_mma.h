// MFMA operand helpers shared by the window attention kernels (window_attn.hip: forward;
// window_attn_backward.hip: gradients).
#pragma once
#include "common.h"

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

// The workgroup's query tile (of nqt of QT queries) and (batch, head) of a kernel that walks each
// query's window of W keys. A head's tiles run on one XCD, in order: their key windows overlap, so most
// of each tile's K and V reads hit that XCD's L2. The first tiles see fewer than W keys. Where they are
// a quarter of a head's tiles or more and a CU holds two workgroups or more, in that order some CUs get
// several heavy tiles and others light ones; there the heavy tiles go first, the XCD's heads taking
// turns (plain attention, in order / heavy first, us: B16 N1024 H8 30.2 / 27.1, B8 N1024 H8 over 2 20.2 /
// 18.7, B9 N1024 M300 H8 24.8 / 21.8, B8 N2048 H8 31.4 / 30.4). Longer sequences keep the order, whose
// K and V reuse counts for more there (B4 N4096 H8 31.5 / 33.2).
__device__ __forceinline__ void query_tile(int nqt, int M, int N, int W, int QT, int& qt, int& bh) {
  const int heads = (int)gridDim.x / nqt;
  const int light = (max(min(W, M + N) - 1 - M, 0) + QT - 1) / QT;
  if (heads % 8 == 0 && gridDim.x >= 512 && 4 * light >= nqt) {
    const int per = heads >> 3, r = (int)blockIdx.x >> 3, rank = r / per;
    bh = (int)(blockIdx.x & 7) * per + (r - rank * per);
    qt = nqt - 1 - rank;
  } else {
    const int lg = xcd_logical_block(blockIdx.x, gridDim.x);
    bh = lg / nqt;
    qt = lg - bh * nqt;
  }
}

}  // namespace
}  // namespace vsp
