// Exchanges between lanes without LDS (gfx950): a __shfl is an LDS instruction with its round trip, on the critical path of a wave
// that has its SIMD to itself (the decode kernels); a DPP move or a row / half swap is one or two vector instructions.
// 16 layers of one token, 128 channels: 1,003 tokens 121 -> 113 us, 8,003 127 -> 122, 32,741 178 -> 171; 256 channels at 9,000
// 177 -> 169; 4 rows at 2,003 tokens 170 -> 162, 64 rows 345 -> 335.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace yka {

typedef unsigned lanes_u32x2 __attribute__((ext_vector_type(2)));

// the value a DPP control names, every lane valid
template <int CTRL, class T>
__device__ __forceinline__ T lane_dpp(T v) {
  static_assert(sizeof(T) == 4, "one register");
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false));
}
template <class T> __device__ __forceinline__ T lane_xor1(T v) { return lane_dpp<0xB1>(v); }     // quad_perm [1,0,3,2]
template <class T> __device__ __forceinline__ T lane_xor2(T v) { return lane_dpp<0x4E>(v); }     // quad_perm [2,3,0,1]
// two shifts inside rows of 16, each into the banks of 4 lanes whose partner lies that way
template <class T> __device__ __forceinline__ T lane_xor4(T v) {
  static_assert(sizeof(T) == 4, "one register");
  const int b = __builtin_bit_cast(int, v);
  const int up = __builtin_amdgcn_update_dpp(b, b, 0x104, 0xf, 0x5, false);                         // row_shl:4 into banks 0 and 2
  return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(up, b, 0x114, 0xf, 0xa, false));         // row_shr:4 into banks 1 and 3
}
template <class T> __device__ __forceinline__ T lane_xor8(T v) { return lane_dpp<0x128>(v); }    // row_ror:8
// op(v, v of lane ^ 16) and op(v, v of lane ^ 32): after swapping a register with a copy of itself the two results hold, in
// every lane, the values of the lane and of its partner (op commutes)
template <class T, class Op>
__device__ __forceinline__ T lane_op16(T v, Op op) {
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const lanes_u32x2 r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  return op(__builtin_bit_cast(T, r0), __builtin_bit_cast(T, r1));
}
template <class T, class Op>
__device__ __forceinline__ T lane_op32(T v, Op op) {
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const lanes_u32x2 r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  return op(__builtin_bit_cast(T, r0), __builtin_bit_cast(T, r1));
}
struct LaneMax { template <class T> __device__ __forceinline__ T operator()(T a, T b) const { if constexpr (__is_same(T, float)) return fmaxf(a, b); else return a > b ? a : b; } };
struct LaneMinF { __device__ __forceinline__ float operator()(float a, float b) const { return fminf(a, b); } };
struct LaneMin { __device__ __forceinline__ int operator()(int a, int b) const { return a < b ? a : b; } };
struct LaneAdd { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };
// over the four lanes l, l ^ 16, l ^ 32, l ^ 48
template <class T, class Op> __device__ __forceinline__ T lane_rows(T v, Op op) { return lane_op32(lane_op16(v, op), op); }
// Stands between the last request of a step and the first use of an answer: left to itself the compiler moves requests behind uses of
// earlier ones to save registers, which makes one trip to memory two or more.
__device__ __forceinline__ void all_requested() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// Sums of eight values over lanes l and l ^ 32, shared out: a swap of a register's half with another's leaves in either half what
// the other needs, so that a fold halves the registers.  The lower half ends with the sums of v[0 .. 3], the upper with v[4 .. 7].
__device__ __forceinline__ float4 fold_halves(const float (&v)[8]) {
  float h[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const lanes_u32x2 r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v[e]), __builtin_bit_cast(unsigned, v[e + 4]), false, false);
    const unsigned r0 = r[0], r1 = r[1];
    h[e] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
  }
  return make_float4(h[0], h[1], h[2], h[3]);
}
// the same over the four lanes l, l ^ 16, l ^ 32, l ^ 48, 12 instructions instead of the 32 of eight butterflies: row g of 16 lanes
// ends with the sums of v[4 (g / 2) + 2 (g % 2)] and of the value after it
__device__ __forceinline__ float2 fold_rows(const float (&v)[8]) {
  const float4 f = fold_halves(v);
  const float h[4] = {f.x, f.y, f.z, f.w};
  float q[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const lanes_u32x2 r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, h[e]), __builtin_bit_cast(unsigned, h[e + 2]), false, false);
    const unsigned r0 = r[0], r1 = r[1];
    q[e] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
  }
  return make_float2(q[0], q[1]);
}
// the butterfly v = op(v, v of lane ^ o), o = 16 .. 1, inside each half of the wave (the reference's reduction of a run of 32
// elements); lane ^ 4 as a rotation by four, since lanes l and l ^ 8 hold one value by then
template <class T, class Op>
__device__ __forceinline__ T lane_run32(T v, Op op) {
  v = lane_op16(v, op);
  v = op(v, lane_xor8(v));
  v = op(v, lane_dpp<0x124>(v));                   // row_ror:4
  v = op(v, lane_xor2(v));
  return op(v, lane_xor1(v));
}
// one stage of a Hadamard transform: a + b in the lane whose bit H is 0, b - a (b: the partner's value) in the other
template <int H>
__device__ __forceinline__ float lane_hadamard(float a, int lane) {
  if constexpr (H >= 16) {
    const unsigned u = __builtin_bit_cast(unsigned, a);
    const lanes_u32x2 r = H == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned r0 = r[0], r1 = r[1];           // in both lanes of a pair: the value of the lower and of the upper one
    const float lo = __builtin_bit_cast(float, r0), hi = __builtin_bit_cast(float, r1);
    return (lane & H) ? __fsub_rn(lo, hi) : __fadd_rn(lo, hi);
  } else {
    const float b = H == 1 ? lane_xor1(a) : H == 2 ? lane_xor2(a) : H == 4 ? lane_xor4(a) : lane_xor8(a);
    return (lane & H) ? __fsub_rn(b, a) : __fadd_rn(a, b);
  }
}
__device__ __forceinline__ float wave_hadamard(float a, int lane) {
  a = lane_hadamard<1>(a, lane); a = lane_hadamard<2>(a, lane); a = lane_hadamard<4>(a, lane);
  a = lane_hadamard<8>(a, lane); a = lane_hadamard<16>(a, lane); return lane_hadamard<32>(a, lane);
}
// over a row of 16 lanes (after two steps a quad holds one value, so the mirrored octet is lane ^ 4); the lanes of a row end with one
// value, sums included: every step adds the same two partial sums in either lane
template <class T, class Op>
__device__ __forceinline__ T lane_row16(T v, Op op) {
  v = op(v, lane_xor1(v));
  v = op(v, lane_xor2(v));
  v = op(v, lane_dpp<0x141>(v));                   // row_half_mirror
  return op(v, lane_xor8(v));
}

}  // namespace yka
