// The end of the decode kernels over 256-channel rows (attend256.hip, attend_tb.hip): the states of the four waves of a
// workgroup are merged through LDS into one partial per (row, split).  gfx950.
//
// Bound by LDS instructions: every wave leaves 16 accumulators of 4 registers.  They go out as 128-bit writes (a lane holds
// runs of 8 consecutive channels) of the rows that exist only - 12 of 16 with two tokens, 6 with one - and come back as
// 128-bit reads, 8 channels a lane, so that a partial row leaves in 16-byte stores.  A 128-bit access of a wave is served 16
// lanes at a time, lanes {0-7, 24-31} first: with 260 floats per row and 32 more from row 8 on those lanes fall into 64
// different banks.  Written a value at a time (64 writes that meet 4 to a bank, 2-byte stores) the merge cost about 1.3 us
// of a decode call: int4 rows, 16 layers, 20,011 tokens 226 us with it and 256 without, 9,000 tokens 206 and 227.
#pragma once
#include "yka_internal.h"

namespace yka {

constexpr int kM256Pitch = 260;
__device__ __forceinline__ int m256_row(int i) { return i * kM256Pitch + 32 * (i >> 3); }
template <int ROWS> constexpr int m256_wave() { return ROWS * kM256Pitch + (ROWS > 8 ? 32 : 0); }      // floats per wave

// o[8 hh + el][r] of lane (row i, group g) is channel 8 (4 g + r + 16 hh) + el of row i; ROWS rows exist (i < ROWS), of which
// the first `rows` belong to tokens of the slice.  pair_of(j): the (token, split) pair of row j.  factor scales the
// normalised row, `mu` (or nullptr) is added to rows that saw a key.  s_acc: 4 * m256_wave<ROWS>() floats, free for use.
template <int ROWS, class V4, class PairOf>
__device__ __forceinline__ void merge_waves256(const V4 (&o)[16], float m_run, float l_run, int wave, int rows, int kvh, int n_heads, float factor,
                                               const float* mu, float (*s_m)[16], float (*s_l)[16], float (*s_wn)[4], float* s_acc,
                                               float* pm, float* pl, uint16_t* pacc16, PairOf pair_of) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  l_run = lane_rows(l_run, LaneAdd{});
  if (g == 0) { s_m[wave][i] = m_run; s_l[wave][i] = l_run; }
  if (i < rows) {
    float* const d = s_acc + wave * m256_wave<ROWS>() + m256_row(i);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* const c = d + 8 * (4 * g + r + 16 * hh);
        *reinterpret_cast<float4*>(c) = make_float4(o[8 * hh][r], o[8 * hh + 1][r], o[8 * hh + 2][r], o[8 * hh + 3][r]);
        *reinterpret_cast<float4*>(c + 4) = make_float4(o[8 * hh + 4][r], o[8 * hh + 5][r], o[8 * hh + 6][r], o[8 * hh + 7][r]);
      }
  }
  __syncthreads();
  // per row: the weight of each wave's accumulator, already divided by the row's sum - computed once per row by 4 lanes,
  // not once per output element
  if (threadIdx.x < 64) {
    const int j = threadIdx.x >> 2, w = threadIdx.x & 3;
    const float mw = s_m[w][j];
    float M2 = fmaxf(mw, lane_xor1(mw));
    M2 = fmaxf(M2, lane_xor2(M2));
    const float ww = exp2f(mw - M2);
    float L = ww * s_l[w][j];
    L += lane_xor1(L);
    L += lane_xor2(L);
    s_wn[j][w] = L > 0.f ? ww * factor / L : 0.f;
    if (w == 0 && j < rows) {
      const size_t p = pair_of(j) * n_heads + kvh * kG + j % kG;
      pm[p] = M2; pl[p] = L;
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < rows * 32; idx += 256) {
    const int j = idx >> 5, c8 = (idx & 31) * 8;
    const float4 w4 = *reinterpret_cast<const float4*>(s_wn[j]);
    const float w[4] = {w4.x, w4.y, w4.z, w4.w};
    float4 a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float* const s = s_acc + k * m256_wave<ROWS>() + m256_row(j) + c8;
      a[k] = *reinterpret_cast<const float4*>(s);
      b[k] = *reinterpret_cast<const float4*>(s + 4);
    }
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = w[0] * (e < 4 ? (&a[0].x)[e] : (&b[0].x)[e - 4]);
#pragma unroll
    for (int k = 1; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] += w[k] * (e < 4 ? (&a[k].x)[e] : (&b[k].x)[e - 4]);
    if (mu && w[0] + w[1] + w[2] + w[3] > 0.f) {
      const float4 m0 = *reinterpret_cast<const float4*>(mu + c8), m1 = *reinterpret_cast<const float4*>(mu + c8 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) { y[e] += (&m0.x)[e]; y[4 + e] += (&m1.x)[e]; }
    }
    const size_t p = pair_of(j) * n_heads + kvh * kG + j % kG;
    *reinterpret_cast<uint4*>(pacc16 + p * 256 + c8) = pack_out8(y, 0);
  }
}

}  // namespace yka
