// The end of the trellis encoder: which of a row's searches it is coded with, and its packed form (trellis.hip, and the
// combiner of decode in attend256.hip, which codes the rows of the pass itself).  gfx950.
#pragma once
#include "yka_internal.h"

namespace yka {

constexpr int kMaxMult = 16;
// What a row is stored as after the search (cache form), by a wave: the multiplier whose search left the smallest squared
// error (its 8 partial sums added in order from 0; the first of equal errors), the four states of elements 4 lane .. 4 lane
// + 3 it chose, its scale.
// choose_job: which job, from what request_errors has asked for.  A wave with one row asks for the states of all jobs
// beside that (pick_job, one trip to memory; no branch stands between the requests, past the last multiplier it is asked
// for again); one with several rows asks for the chosen states only, which are a ninth of the bytes.
typedef uint32_t JobStates __attribute__((ext_vector_type(kMaxMult)));
typedef float JobErrors __attribute__((ext_vector_type(4)));
struct JobTotals { JobErrors e0, e1; float s; };
__device__ __forceinline__ JobTotals request_errors(const TbJobs& A, int row, int lane) {
  const size_t mine = (size_t)row * A.nm + min(lane, A.nm - 1);
  const JobErrors* err = reinterpret_cast<const JobErrors*>(A.scr + A.w_ofs) + mine * 2;
  return JobTotals{err[0], err[1], reinterpret_cast<const float*>(A.scr + A.s_ofs)[mine]};
}
__device__ __forceinline__ uint32_t job_states(const TbJobs& A, int row, int job, int lane) {
  return reinterpret_cast<const uint32_t*>(A.scr + ((size_t)row * A.nm + job) * 256)[lane];
}
__device__ __forceinline__ int choose_job(const TbJobs& A, int lane, const JobTotals& R, float& scale) {
  float total = 0.f;
  total = __fadd_rn(total, R.e0.x); total = __fadd_rn(total, R.e0.y); total = __fadd_rn(total, R.e0.z); total = __fadd_rn(total, R.e0.w);
  total = __fadd_rn(total, R.e1.x); total = __fadd_rn(total, R.e1.y); total = __fadd_rn(total, R.e1.z); total = __fadd_rn(total, R.e1.w);
  // the smallest total, the first of equal ones; one that is not a number never wins, except by being the first multiplier's
  const float inf = __builtin_huge_valf(), mine = lane < A.nm && total == total ? total : inf;
  const float least = lane_row16(mine, LaneMinF{});
  const uint64_t at = __ballot(lane < A.nm && mine == least), first_bad = __ballot(lane == 0 && total != total);
  const int keep = __builtin_amdgcn_readfirstlane(first_bad ? 0 : __builtin_ctzll(at));
  scale = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(R.s), keep));
  return keep;
}
__device__ __forceinline__ void pick_job(const TbJobs& A, int row, int lane, uint32_t& states, float& scale) {
  JobStates all;
#pragma unroll
  for (int i = 0; i < kMaxMult; ++i) all[i] = job_states(A, row, min(i, A.nm - 1), lane);
  const int keep = choose_job(A, lane, request_errors(A, row, lane), scale);
  const auto a8 = (keep & 8) ? all.hi : all.lo;          // uniform over the wave
  const auto a4 = (keep & 4) ? a8.hi : a8.lo;
  const auto a2 = (keep & 2) ? a4.hi : a4.lo;
  states = (keep & 1) ? a2.y : a2.x;
}
// packs the fields of those states and stores the row: 4 fields of a lane are 4 KB bits of the MSB-first stream; a word is
// made of the bits of two lanes (4 bits: lane 2 w and the next) or of up to three (5 bits: 8 lanes are 5 words, word j
// starts in lane 8 j / 5)
template <int KB>
__device__ __forceinline__ void store_coded_row(uint8_t* dst, int lane, uint32_t states) {
  constexpr uint32_t mask = (1u << KB) - 1u;
  const uint32_t own = ((states & mask) << (3 * KB)) | (((states >> 8) & mask) << (2 * KB)) | (((states >> 16) & mask) << KB) | ((states >> 24) & mask);
  uint32_t* const words = reinterpret_cast<uint32_t*>(dst);
  if constexpr (KB == 4) {
    const uint32_t next = lane_xor1(own);
    if ((lane & 1) == 0) words[lane >> 1] = (own << 16) | next;
  } else {
    static_assert(KB == 5, "4 or 5 bits");
    const int j = lane & 7, a = (8 * j) / 5, at = (lane & ~7) + a;
    const uint32_t v0 = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * at, (int)own), v1 = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (at + 1), (int)own),
                   v2 = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * min(at + 2, lane | 7), (int)own);
    const uint64_t bits = ((uint64_t)v0 << 40) | ((uint64_t)v1 << 20) | v2;
    if (j < 5) words[5 * (lane >> 3) + j] = (uint32_t)(bits >> (28 + 20 * a - 32 * j));
  }
}

}  // namespace yka
