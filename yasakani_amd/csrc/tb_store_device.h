// The end of the trellis encoder: which of a row's searches it is coded with, and its packed form (trellis.hip, and the
// combiner of decode in attend256.hip, which codes the rows of the pass itself).  gfx950.
#pragma once
#include "yka_internal.h"

namespace yka {

constexpr int kMaxMult = 16;
// word d of a row's MSB-first stream of KB-bit fields: the fields that overlap bits [32 d, 32 d + 32)
template <int KB>
__device__ __forceinline__ uint32_t pack_word(const uint8_t* fld, int d) {
  const int e0 = (32 * d) / KB;                          // first field with bits in the word (division by a constant)
  uint32_t w = 0u;
#pragma unroll
  for (int k = 0; k < 32 / KB + 2; ++k) {
    const int e = e0 + k, sh = 32 * d + 32 - KB * (e + 1);   // distance of the field's last bit from the word's last bit
    if (e < 256 && sh > -KB) w |= sh >= 0 ? (uint32_t)fld[e] << sh : (uint32_t)fld[e] >> -sh;
  }
  return w;
}

// What a row is stored as after the search (cache form), by a wave: the multiplier whose search left the smallest squared error (its 8
// partial sums added in order from 0; the first of equal errors), the four states of elements 4 lane .. 4 lane + 3 it chose, its scale.
__device__ __forceinline__ void pick_job(const TbJobs& A, int row, int lane, uint32_t& states, float& scale) {
  const size_t job0 = (size_t)row * A.nm;
  uint32_t all[kMaxMult];
#pragma unroll
  for (int i = 0; i < kMaxMult; ++i) all[i] = i < A.nm ? reinterpret_cast<const uint32_t*>(A.scr + (job0 + i) * 256)[lane] : 0u;
  float4 e0 = make_float4(0, 0, 0, 0), e1 = e0;
  float s = 0.f;
  if (lane < A.nm) {
    const float4* err = reinterpret_cast<const float4*>(A.scr + A.w_ofs) + (job0 + lane) * 2;
    e0 = err[0]; e1 = err[1];
    s = reinterpret_cast<const float*>(A.scr + A.s_ofs)[job0 + lane];
  }
  float total = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) total = __fadd_rn(total, (&e0.x)[k]);
#pragma unroll
  for (int k = 0; k < 4; ++k) total = __fadd_rn(total, (&e1.x)[k]);
  // the smallest total, the first of equal ones; one that is not a number never wins, except by being the first multiplier's
  const float inf = __builtin_huge_valf(), mine = lane < A.nm && total == total ? total : inf;
  const float least = lane_row16(mine, LaneMinF{});
  const uint64_t at = __ballot(lane < A.nm && mine == least), first_bad = __ballot(lane == 0 && total != total);
  const int keep = __builtin_amdgcn_readfirstlane(first_bad ? 0 : __builtin_ctzll(at));
#pragma unroll
  for (int b = kMaxMult / 2; b; b >>= 1)
#pragma unroll
    for (int i = 0; i < b; ++i) all[i] = (keep & b) ? all[i + b] : all[i];       // uniform over the wave
  states = all[0];
  scale = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s), keep));
}
// packs and stores the fields of those states (fld: 256 bytes of LDS private to the wave)
template <int KB>
__device__ __forceinline__ void store_coded_row(uint8_t* dst, uint8_t* fld, int lane, uint32_t states) {
  reinterpret_cast<uint32_t*>(fld)[lane] = states & (0x01010101u * ((1u << KB) - 1u));
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  if (lane < 8 * KB) reinterpret_cast<uint32_t*>(dst)[lane] = pack_word<KB>(fld, lane);
}

}  // namespace yka
