// The fp32 matrix instruction v_mfma_f32_16x16x4_f32 as the attention kernels
// use it (lane l, j = l % 16, g = l / 16: A[i][k] has i = j and k = g, B[k][j]
// has k = g, C[i][j] register r is row i = 4 g + r): a [rows, D] operand's
// d are read 16 bytes at a time, and output columns are stored as rows.
#pragma once
#include "cdna4.h"

DEVI f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// the value held by lane l ^ 16
DEVI float other_16(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x),
                                            __builtin_bit_cast(unsigned, x), false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 16) ? r[0] : r[1]);
}
// over the four lanes that share j
DEVI float max_g(float x) {
  x = fmaxf(x, other_16(x));
  return fmaxf(x, other_half(x));
}
DEVI float sum_g(float x) {
  x += other_16(x);
  return x + other_half(x);
}

// global vectors: tensors may start at any float
typedef float f32x4g __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2g __attribute__((ext_vector_type(2), aligned(4)));

template <int D>
struct Geo {
  static constexpr int NC = D < 16 ? 1 : D / 16;     // chunks of 16 d per row
  static constexpr int VW = D >= 64 ? 4 : D == 32 ? 2 : 1;  // d per transposed read
  static constexpr int NH = D < 16 ? 1 : D / (16 * VW);     // groups of VW output tiles
};

// A row-wise A or B operand of one row in global memory: lane g holds d =
// 16 c + 4 g .. + 3 of chunk c (D = 8: zeros past the row)
template <int D>
DEVI void row_regs(const float* row, int g, f32x4* out) {
#pragma unroll
  for (int c = 0; c < Geo<D>::NC; ++c) {
    if constexpr (D == 8) {
      out[c] = g < 2 ? (f32x4)*reinterpret_cast<const f32x4g*>(row + 4 * g)
                     : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    } else {
      out[c] = *reinterpret_cast<const f32x4g*>(row + 16 * c + 4 * g);
    }
  }
}

template <int D>
DEVI void zero_acc(f32x4 (*acc)[Geo<D>::VW]) {
#pragma unroll
  for (int h = 0; h < Geo<D>::NH; ++h)
#pragma unroll
    for (int e = 0; e < Geo<D>::VW; ++e) acc[h][e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
}

// the lane's column of acc, each value through f, to row [D]: output tile e
// of group h holds d = 16 VW h + VW (4 g + r) + e
template <int D, typename F>
DEVI void store_col(float* row, const f32x4 (*acc)[Geo<D>::VW], int g, F&& f) {
  constexpr int VW = Geo<D>::VW;
#pragma unroll
  for (int h = 0; h < Geo<D>::NH; ++h) {
    if constexpr (VW == 1) {
      if (D >= 16 || g < 2)
        *reinterpret_cast<f32x4g*>(row + 4 * g) =
            f32x4g{f(acc[0][0][0]), f(acc[0][0][1]), f(acc[0][0][2]), f(acc[0][0][3])};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* p = row + 16 * VW * h + VW * (4 * g + r);
        if constexpr (VW == 4)
          *reinterpret_cast<f32x4g*>(p) =
              f32x4g{f(acc[h][0][r]), f(acc[h][1][r]), f(acc[h][2][r]), f(acc[h][3][r])};
        else
          *reinterpret_cast<f32x2g*>(p) = f32x2g{f(acc[h][0][r]), f(acc[h][1][r])};
      }
    }
  }
}
