// Split-KV attention for windows of 3..64 query tokens (verify windows) and for prefill chunks cut into slices of up to
// 2048 tokens (one launch per slice, every workgroup 128 rows of it).  gfx950.
//
// Same mathematics as the narrow kernel (reference: src/q35_atxpk4.cuh:71-499 for the window shape, row geometry
// src/q35_atxpk.cu:391-411): every row t of the window runs an online softmax over the keys [0, len(t)) of its
// split and leaves (m, l, acc) partials for the combiner.  What differs is who dequantizes and how the work of a
// compute unit is laid out in time:
//   * one workgroup of 8 waves per compute unit owns up to 128 query rows (token-major, 6 heads per token) and one
//     split of the keys.  The waves form two groups of four; group g walks the tiles tile0 + g, tile0 + g + 2, ... of
//     the split, each with its own softmax state, and the two states are merged through LDS at the end: one partial
//     row per (row, split), half as many splits as workgroups of four waves would need to fill the chip;
//   * a group dequantizes each of its 32-key tiles ONCE into LDS - K as exact integer codes n-8 in fp16, V scaled
//     and transposed (channel-major, the operand shape of the token-contracting MFMA) - and every wave of the group reads
//     its MFMA fragments from there;
//   * a wave owns one tile of 32 rows (MFMA 32x32x16: one K or V fragment read from LDS serves 32 rows) and stays
//     under 256 registers, so the two waves of a SIMD (one of each group) fit and all MFMA results live in ordinary
//     VGPRs (no accumulator-file copies);
//   * a step of a group has two phases: a MATRIX phase (the PV product of the previous tile, the score MFMAs of this tile
//     with the scale multiply-adds in their shadow, fragment reads) and a VECTOR phase (softmax, dequantization of the
//     group's next tile, requests for the tile after that).  The groups run half a step apart - between two workgroup barriers
//     one runs matrix, then vector phase, the other vector, then matrix phase - so the two waves of a SIMD
//     do not compete for the matrix pipe and vector work of one wave runs under the MFMAs of the other.  Two waves
//     left to themselves do not find this arrangement: measured, two independent 4-wave workgroups per compute unit
//     take as long as the same two one after the other;
//   * the group scales of K are applied to the fp32 partial sum of each 32-channel group (two chained MFMAs per
//     group), so K is never rounded; V carries one fp16 rounding.  The scales in LDS carry log2(e)/sqrt(d) and the
//     chain of multiply-adds starts from minus the row's running maximum: a score leaves it as the exponent of its
//     probability.  A lane needs the scales of 16 keys, the same in all 32 lanes of its half: one read gives every lane
//     the four group scales of one key, and the multiply-adds of groups 1 to 3 take the others' by row broadcasts (scale_scores);
//     group 0, whose addend is minus the maximum and no accumulator, reads its 16 scales;
//   * the running maximum of a row is only raised when the probabilities of a tile sum to more than 2^8 in a lane: the sum is
//     there anyway, and accumulators stay in their registers untouched on almost every tile;
//   * LDS is double buffered per group; the raw tile loads run two tiles ahead as explicit load instructions with
//     their own counter waits;
//   * the last split owns the tiles that hold the rows this pass appends and quantizes them itself before reading
//     them (quantize-on-append without a launch of its own).
// The values the instruction-form loads produce must reach their wait in the registers they were loaded into: they are
// loop carried in fixed registers, every request is waited for before the loop's registers are given up, and every
// parity test would fail on a copy made before its wait.
// LDS image of one tile (19584 bytes):
//   K  [32 keys][272 B]   chunk 4m+g of a key = channels 32m+8g..+7 in the order n0,n4,n1,n5,n2,n6,n3,n7; the 272-byte
//                          pitch makes the lanes of a fragment read hit distinct banks
//   V  [128 rows][80 B]   channel 8*dw+c lives in row 16*sigma(c)+dw, sigma(c) = 2*(c&3) + (c>>2): the 16 lanes that
//                          dequantize one byte position write 16 consecutive rows, and an output lane ends up with runs
//                          of 8 consecutive channels.  Inside a row token 16u+8a+4h+b sits at position 16u+8h+4a+b, so
//                          the 8 tokens an MFMA lane needs are 16 contiguous bytes
//   S  [2 h][16 r][4 groups] fp32   K group scales of key 8 (r / 4) + 4 h + r % 4, r being the score register of that key: lane
//                          (h, i) reads the four of r = i % 16.  Converted to fp32 once per workgroup
//   S0 [2 h][16 r] fp32    group 0 once more, read four keys at a time (a broadcast)
// With all 64 scales of a lane read as broadcasts (16 reads of 1 KB a tile and wave, as many as the fragments take) the LDS pipe was
// as busy as the matrix pipe.  us, 16 reads / 5 and row broadcasts / and the maximum raised by the sum (8 max3 fewer): 16 layers of 64
// rows at 32,768 tokens 730 / 716 / 709, of 1,500 rows on an empty cache 703 / 687 / 689, 2 layers of 2,048 rows at 131,072
// 8,240 / 8,020 / 7,710.
// Partial results leave through the same LDS after the last tile so that every store writes whole 256-byte rows.
#include "codec_device.h"
#include <hip/hip_fp16.h>
#include <type_traits>

namespace yka {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

namespace {

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u32(h2 h) { return __builtin_bit_cast(uint32_t, h); }

constexpr uint32_t kMagic = 0x64006400u;
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kKPitch = 272, kVPitch = 80;
constexpr int kLdsK = 0, kLdsV = 32 * kKPitch, kLdsS = kLdsV + 128 * kVPitch, kLdsS0 = kLdsS + 512, kLdsBuf = kLdsS0 + 128;   // 19584
constexpr int NT = 512;                        // threads per workgroup: two groups of four waves
constexpr int NTG = 256;                       // threads per group
constexpr float kRaiseSum = 256.f;             // a tile whose probabilities sum to more than this in a lane raises the running maximum

// what a wave does in a step of its group; a wave that only decodes takes two or all four quarters of the tile
enum { kIdle, kFeed1, kFeed2, kFeed4, kComputeOnly, kComputeFeed };
template <int kRole>
constexpr int quarters() { return kRole == kFeed4 ? 4 : kRole == kFeed2 ? 2 : 1; }

template <int U>
struct Raw {                                   // a lane's share of U quarters of a raw 32-key tile; t = 64 x quarter + lane
  uint32_t kw[U][2];
  uint32_t vw[U][2];
  uint32_t vs[U];
  uint32_t ks[U < 2 ? U : 2];                  // fp16 scale of (key (t & 127) / 4, group t % 4): quarters 2 and 3 repeat 0 and 1
};

// Byte offsets of one thread inside a page, fixed for the whole kernel; the page pointer and the tile's first token
// are wave uniform, so every load is "scalar base + 32-bit lane offset".
struct LaneOffs { uint32_t k, v, vs, ks; };
__device__ __forceinline__ LaneOffs lane_offs(int tid) {
  const uint32_t pair = tid >> 4, dw = tid & 15;
  return LaneOffs{(uint32_t)tid * 4u, kPageVc + pair * 128u + dw * 4u, kPageVs + (dw >> 2) * (kPageTok * 2u) + pair * 4u,
                  kPageKs + ((uint32_t)tid & 127u) * 2u};
}
// The tile loads are written as instructions: they stay in flight across two loop steps, and the counter wait the
// compiler would place at the loop header (it merges the header's predecessors conservatively) drains all of them.
// Every load here is "wave-uniform base in scalar registers + 32-bit lane offset"; wait_raw<N> ties the six registers
// of a tile to a wait that leaves the N younger loads in flight.  Loads return in order and nothing stores in the loop.
template <int U>
__device__ __forceinline__ void load_raw(const uint8_t* pg, int tp, const LaneOffs& L, Raw<U>& R) {
  const uint8_t* kt = pg + (uint32_t)tp * 64u;            // K and V code rows of the tile start here (+ plane offset)
  const uint8_t *vs = pg + (uint32_t)tp * 2u, *ks = pg + (uint32_t)tp * 8u;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "=v"(R.kw[u][0]) : "v"(L.k), "s"(kt), "n"(256 * u));
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "=v"(R.kw[u][1]) : "v"(L.k), "s"(kt), "n"(256 * u + NTG * 4));
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "=v"(R.vw[u][0]) : "v"(L.v), "s"(kt), "n"(512 * u));
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "=v"(R.vw[u][1]) : "v"(L.v), "s"(kt), "n"(512 * u + 64));
    asm volatile("global_load_dword %0, %1, %2 offset:%3" : "=v"(R.vs[u]) : "v"(L.vs), "s"(vs), "n"(16 * u));
    if (u < 2) asm volatile("global_load_ushort %0, %1, %2 offset:%3" : "=v"(R.ks[u]) : "v"(L.ks), "s"(ks), "n"(128 * u));
  }
}
template <int N, int U>
__device__ __forceinline__ void wait_raw(Raw<U>& R) {
  static_assert(U == 1 || U == 2 || U == 4);
#define YKA_RAW(u) "+v"(R.kw[u][0]), "+v"(R.kw[u][1]), "+v"(R.vw[u][0]), "+v"(R.vw[u][1]), "+v"(R.vs[u])
  if constexpr (U == 1) asm volatile("s_waitcnt vmcnt(%6)" : YKA_RAW(0), "+v"(R.ks[0]) : "n"(N));
  else if constexpr (U == 2) asm volatile("s_waitcnt vmcnt(%12)" : YKA_RAW(0), YKA_RAW(1), "+v"(R.ks[0]), "+v"(R.ks[1]) : "n"(N));
  else asm volatile("s_waitcnt vmcnt(%22)" : YKA_RAW(0), YKA_RAW(1), YKA_RAW(2), YKA_RAW(3), "+v"(R.ks[0]), "+v"(R.ks[1]) : "n"(N));
#undef YKA_RAW
}

// (w & mask) | magic as one bit-field insert: `magic` (0x64006400, no bit inside either nibble mask) is kept opaque to
// the optimizer so that the select form survives to instruction selection
__device__ __forceinline__ uint32_t nib(uint32_t w, uint32_t mask, uint32_t magic) { return (w & mask) | (magic & ~mask); }

// t: of the first quarter, as for the loads
template <int U>
__device__ __forceinline__ void dequant_to_lds(uint8_t* buf, int t, const Raw<U>& R, uint32_t magic, float sc_log2) {
  const h2 c1032 = {(_Float16)1032.f, (_Float16)1032.f}, c1152 = {(_Float16)1152.f, (_Float16)1152.f};
  const h2 c16 = {(_Float16)0.0625f, (_Float16)0.0625f}, c72 = {(_Float16)-72.f, (_Float16)-72.f};
#pragma unroll
  for (int n = 0; n < 2 * U; ++n) {
    const int idx = t + 64 * (n >> 1) + (n & 1) * NTG, key = idx >> 4, p = idx & 15;      // physical dword p = 4g+m of the key row
    const uint32_t w = R.kw[n >> 1][n & 1], w8 = w >> 8;
    uint4 o;
    o.x = as_u32(as_h2(nib(w, 0x000f000fu, magic)) - c1032);
    o.y = as_u32(__builtin_elementwise_fma(as_h2(nib(w, 0x00f000f0u, magic)), c16, c72));      // (1024 + 16 n) / 16 - 72 = n - 8, exactly
    o.z = as_u32(as_h2(nib(w8, 0x000f000fu, magic)) - c1032);
    o.w = as_u32(__builtin_elementwise_fma(as_h2(nib(w8, 0x00f000f0u, magic)), c16, c72));
    *reinterpret_cast<uint4*>(buf + kLdsK + key * kKPitch + (4 * (p & 3) + (p >> 2)) * 16) = o;
  }
#pragma unroll
  for (int u = 0; u < (U < 2 ? U : 2); ++u) {                        // K group scales as fp32, [group][a][h][b] for key 8a+4h+b,
    const int key = ((t + 64 * u) & 127) >> 2, m = t & 3;                   // times log2(e)/sqrt(d): scores come out in log2 units
    const int at = ((key >> 2) & 1) * 16 + (key >> 3) * 4 + (key & 3);
    const float sc = (float)as_h2(R.ks[u])[0] * sc_log2;
    reinterpret_cast<float*>(buf + kLdsS)[at * 4 + m] = sc;
    reinterpret_cast<float*>(buf)[m == 0 ? kLdsS0 / 4 + at : kLdsS / 4 + at * 4 + m] = sc;   // waves 2 and 3 repeat waves 0 and 1 (no divergent branch)
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int pair = (t >> 4) + 4 * u, dw = t & 15;
    const int t0 = 2 * pair;                                         // token 16u + 8a + 4h + b -> position 16u + 8h + 4a + b
    const int posn = (t0 & 16) + 8 * ((t0 >> 2) & 1) + 4 * ((t0 >> 3) & 1) + (t0 & 3);
    const h2 s2 = as_h2(R.vs[u]), s2q = s2 * h2{(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t w0 = R.vw[u][0], w1 = R.vw[u][1];
    uint8_t* vb = buf + kLdsV + dw * kVPitch + posn * 2;
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) {
      // byte bb of both tokens side by side (low half = token t0, high half = token t0+1)
      const uint32_t x = __builtin_amdgcn_perm(w1, w0, 0x0c040c00u + bb * 0x00010001u);
      const h2 lo = (as_h2(nib(x, 0x000f000fu, magic)) - c1032) * s2;       // channel c = 2bb
      const h2 hi = (as_h2(nib(x, 0x00f000f0u, magic)) - c1152) * s2q;      // channel c = 2bb+1
      const int c0 = 2 * bb, c1 = 2 * bb + 1;
      *reinterpret_cast<uint32_t*>(vb + 16 * (2 * (c0 & 3) + (c0 >> 2)) * kVPitch) = as_u32(lo);
      *reinterpret_cast<uint32_t*>(vb + 16 * (2 * (c1 & 3) + (c1 >> 2)) * kVPitch) = as_u32(hi);
    }
  }
}

// s[r] += part[r] * scale, where lane i % 16 == r of every row of 16 holds the scale of register r.  The compiler makes a move of its
// own out of every broadcast it is given, so the multiply-adds are written out.  It keeps the wait between the matrix instruction
// that leaves `part` and its first reader only for instructions it knows: that is the first one here, and the written ones
// name its result so that they stay behind it.
template <int R>
__device__ __forceinline__ void scale_scores(float (&s)[16], const f16v& part, float sc) {
  if constexpr (R == 0) s[0] = __builtin_fmaf(part[0], __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sc), 0x150, 0xf, 0xf, true)), s[0]);
  else asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%4 row_mask:0xf bank_mask:0xf" : "+v"(s[R]) : "v"(sc), "v"(part[R]), "v"(s[0]), "n"(R));
  if constexpr (R < 15) scale_scores<R + 1>(s, part, sc);
}

}  // namespace

// Workgroup = (split, kv head, row block), block 512; row wave w of either group owns rows [32 w, 32 (w+1)) of the block.
// The row blocks of one (split, kv head) pair read the same KV tiles, and each of the 8 XCDs has an L2 of its own, so the
// grid is one-dimensional and laid out for the dispatcher's round robin (workgroup i runs on XCD i mod 8, strictly: a
// workgroup waits for a CU of ITS XCD, so the grid holds exactly pairs x n_rb workgroups and no padding).  XCD x gets
// n_x = total / 8 (+1 if x < total mod 8) workgroups.  The first F * n_rb of them, F = (total / 8) / n_rb, are the row
// blocks of F whole pairs (the k-th is row block k mod n_rb of pair x + 8 (k / n_rb)): all row blocks of such a pair run
// on one XCD at about the same time and each tile leaves HBM once.  The workgroups left over on every XCD take the
// remaining pairs in order.
// BF: Q / new K / new V are bf16 rows; a kernel of its own, because a branch around the conversion in this one costs the fp16
// rows 1.5 % (755 against 767 us for 16 layers of 64 rows at 32,768 tokens)
// CHUNK: slice of a prefill chunk, whose rows an append launch has stored: no rows to quantize, the key range cut evenly
// into the number of splits the length found on the device justifies (chunk_splits_used), the other workgroups exit.  A
// slice that uses one split writes its output rows instead of partials.  While the keys of all kv heads fit one XCD's L2
// the longest row blocks start first, spread over the XCDs (on a short context a block's length is its place in the slice).
// FEW: a window whose blocks have three waves of rows at most (the roles below); a slice that one split would give less than half of the
// CUs a workgroup: it mostly uses several, and what the early request of the query adds is instructions fetched cold in front of everything
// else.  us per 4 layers, with the early request / without: one KV head (15 workgroups), 300 rows at 2,000 tokens 86.0 / 80.6, four
// (20), 100 rows there 87 / 84.2, four (40), 200 rows at 500 78.6 / 77.2, four (96), 500 first rows 81.4 / 81.0; per 8 layers, four (132), 700 first rows
// 199.7 / 201.2, four (188), 1,000 first rows 242.2 / 245.5.
template <bool BF, bool CHUNK, bool FEW>
__global__ void __launch_bounds__(NT) attend_wide_kernel(WindowHead head_args, WindowSizes size_args, WindowTail tail_args) {
  AttnArgs A = window_args(head_args, size_args, tail_args);
  __shared__ __align__(16) uint8_t lds[2][2][kLdsBuf];               // [group][buffer]
  __shared__ __align__(16) uint8_t s_q[128 * kKPitch];               // the block's query rows in operand order
  const int n_rb = (kG * A.M + A.rows_per_block - 1) / A.rows_per_block;
  const int tid = threadIdx.x;
  // 16 bytes of four query rows (16 threads a row).  A lane that reads its own row asks for pieces 256 bytes from its neighbours':
  // eight loads of 32 lines a wave, 2,048 line accesses a workgroup, and each in a branch of its own; here a workgroup touches every line
  // once and goes through LDS.  us per 16 layers, before / since (loops aligned, see the Makefile): 64 rows at 32,768 tokens 700 / 682,
  // 1,500 rows on an empty cache 686 / 661, 24 tree rows at 9,000 305 / 286, 32 rows at 3,000 253.5 / 242.5, 12 at 3,000 233.2 / 229.
  // A slice asks for the rows this workgroup takes if the slice uses one split, which is known before the position (1,500 rows 656 / 643.7;
  // 1,000 rows at 9,000 tokens, where it asks twice, 2,685 / 2,693), unless it is FEW.
  uint4 qraw[4];
  auto request_q = [&](int b, int kvh_q) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int Rq = min(b * A.rows_per_block + 32 * u + (tid >> 4), kG * A.M - 1);
      qraw[u] = *reinterpret_cast<const uint4*>(A.q16 + ((size_t)(Rq / kG) * A.n_heads + kvh_q * kG + Rq % kG) * kD + 8 * (tid & 15));
    }
  };
  const int rb_q = n_rb - 1 - min((int)blockIdx.x / A.kv.n_kv, n_rb - 1), kvh_one = (int)blockIdx.x % A.kv.n_kv;
  if constexpr (CHUNK && !FEW) request_q(rb_q, kvh_one);
  const int pos = *A.d_pos;
  if constexpr (CHUNK) { if (A.adapt) A.S = chunk_splits_used(pos, A.tok0, A.M, A.kv.n_kv, A.kv.max_ctx, A.S, A.adapt); }
  const int total = CHUNK ? A.S * A.kv.n_kv * n_rb : (int)gridDim.x;
  if (CHUNK && (int)blockIdx.x >= total) return;
  int pair, rb;
  if (CHUNK && A.adapt && (long long)((min(pos + A.tok0 + A.M, A.kv.max_ctx) + 31) / 32) * 4608 * A.kv.n_kv <= (4 << 20)) {
    const int pairs = A.S * A.kv.n_kv;
    rb = n_rb - 1 - (int)blockIdx.x / pairs; pair = (int)blockIdx.x % pairs;
  } else {
    const int x = blockIdx.x & 7, k = blockIdx.x >> 3, F = (total >> 3) / n_rb;
    if (k < F * n_rb) { pair = x + 8 * (k / n_rb); rb = k % n_rb; }
    else {
      const int base_e = (total >> 3) - F * n_rb;                     // leftover workgroups of an XCD, +1 on the first total mod 8
      const int jj = x * base_e + min(x, total & 7) + (k - F * n_rb);
      pair = 8 * F + jj / n_rb; rb = jj % n_rb;
    }
  }
  const int split = pair % A.S, kvh = pair / A.S;
  if constexpr (CHUNK && !FEW) { if (rb != rb_q || kvh != kvh_one) request_q(rb, kvh); } else request_q(rb, kvh);
  const int gt = tid & (NTG - 1);                  // gt: thread index inside the group
  const int grp = __builtin_amdgcn_readfirstlane(tid >> 8);           // wave uniform
  // waves w and w + 4 share a SIMD: group 1 counts its rows from the third wave, so that in a block of up to 64 rows no SIMD has two
  // waves of rows (16 layers of 32 rows, then 128 + 64, at 12,000 tokens 312 / 304.7 us)
  const int wave = (__builtin_amdgcn_readfirstlane(gt >> 6) + 2 * grp) & 3, lane = tid & 63, j = lane & 31, h = lane >> 5;
  const int nrows = kG * A.M;
  // the rows the window split stores (below) are requested before anything that waits for the position
  // (64 rows at 32,000 tokens, 16 layers: 727 us against 733)
  const bool stores = !CHUNK && A.k16 && split == A.S - 1;
  const int tok_lo = (rb * A.rows_per_block) / kG, tok_hi = min(A.M, (rb * A.rows_per_block + A.rows_per_block + kG - 1) / kG);
  uint4 rawv[8];
  if (stores && grp == 0) {
    const int c = gt & 15, slot = gt >> 4;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int hh = it * 16 + slot, t = hh >> 1;
      const uint16_t* src = ((hh & 1) ? A.v16 : A.k16) + ((size_t)(A.tok0 + t) * A.kv.n_kv + kvh) * kD + 8 * c;
      rawv[it] = t < tok_hi ? *reinterpret_cast<const uint4*>(src) : make_uint4(0, 0, 0, 0);
    }
  }

  // row of this lane: R = rb*rows_per_block + wave*32 + j  ->  token R/6 of the slice, head kvh*6 + R%6
  const int RPB = A.rows_per_block;
  const int row0 = rb * RPB + wave * 32;
  const int R = row0 + j;
  const bool vrow = R < nrows && R < (rb + 1) * RPB;
  const int tl = R / kG, head = kvh * kG + R % kG;
  int dep = A.tok0 + tl, mindep = A.tok0 + tok_lo, maxdep = A.tok0 + tok_hi - 1;
  if (A.depth) {                               // uniform over the grid
    dep = A.depth[min(dep, A.tok0 + A.M - 1)];
    depth_range(A.depth + A.tok0, tok_lo, tok_hi, mindep, maxdep);
    asm volatile("" : "+v"(dep));              // answered here: behind the branch a pass without depths would wait for its query
  }
  const int len = vrow ? min(pos + dep + 1, A.kv.max_ctx) : 0;
  const size_t pidx = ((size_t)tl * A.S + split) * A.n_heads + head;
  {
    if constexpr (BF) rows16_to_f16(qraw);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = 32 * u + (tid >> 4);
      const bool some = r < RPB && rb * RPB + r < nrows;
      const h8 c = __builtin_bit_cast(h8, some ? qraw[u] : make_uint4(0, 0, 0, 0));
      *reinterpret_cast<h8*>(s_q + r * kKPitch + 16 * (tid & 15)) = h8{c[0], c[4], c[1], c[5], c[2], c[6], c[3], c[7]};
    }
  }
  __syncthreads();
  // B operand of S^T = K Q^T, k-step ks: lane (row j, half h) holds chunk 2ks+h = (group ks/2, sub-chunk 2(ks&1)+h)
  h8 qf[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const h8*>(s_q + (32 * wave + j) * kKPitch + 16 * (2 * ks + h));
  const bool has_rows = row0 < min(nrows, (rb + 1) * RPB);             // wave uniform

  // key range of the workgroup: its splits cut [0, maxlen) of the block's longest row into 32-key tiles
  const int maxlen = min(pos + maxdep + 1, A.kv.max_ctx), minlen = min(pos + mindep + 1, A.kv.max_ctx);
  // The last split owns the tiles that hold rows of this slice (from tile Tw on), the other splits share the cached
  // context before them evenly: the rows a pass appends are then read by the workgroups of one split only, which
  // is what lets them be quantized and stored by those workgroups themselves (below) instead of by a launch of
  // their own.
  const int ntiles = (maxlen + 31) >> 5;
  // The window split takes an even share of the cached context as well, less window_cost tiles for the quantization it
  // does first (measured: about the time of 7 tiles for 64 rows): every workgroup of the launch then finishes at about
  // the same time (with the window tiles alone, 12 of the 252 workgroups of a 64-row pass were idle after two tiles and
  // the others walked 51 tiles instead of 49).
  const int kWindowCost = !CHUNK && A.k16 ? 1 + A.M / 10 : 0;
  const int Tnew = min(ntiles, max(0, pos + A.tok0) >> 5);            // first tile that holds a row of this slice
  const int Tw = A.S > 1 ? min(Tnew, (A.S - 1) * ((ntiles + kWindowCost + A.S - 1) / A.S)) : Tnew;
  int tile0, tile1;
  if (A.S == 1) { tile0 = 0; tile1 = ntiles; }
  else if (CHUNK) { const int tps = (ntiles + A.S - 1) / A.S; tile0 = min(ntiles, split * tps); tile1 = min(ntiles, tile0 + tps); }
  else if (split == A.S - 1) { tile0 = Tw; tile1 = ntiles; }
  else { const int tps = (Tw + A.S - 2) / (A.S - 1); tile0 = split * tps; tile1 = min(Tw, tile0 + tps); }
  // ---- fused quantize-on-append: every workgroup of the window split stores the slice's rows up to its own last
  //      token (the row blocks of one kv head write identical bytes: each row is the same sequence of IEEE operations
  //      on the same inputs whoever computes it) and reads them back after a workgroup barrier: writer and readers
  //      are waves of one CU and one write-through L1.  Group 0 quantizes; the barrier is the workgroup's. ----
  if (stores) {
    // 16 lanes per 128-channel row, 16 rows (K and V of 8 tokens) per step, at most 64 tokens
    static_assert(kMaxSlice <= 64, "8 steps of 16 rows cover K and V of a slice");
    if (grp == 0) {
      const int c = gt & 15, slot = gt >> 4;
      if constexpr (BF) rows16_to_f16(rawv);
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int hh = it * 16 + slot, t = hh >> 1, r = pos + A.tok0 + t;
        if (t < tok_hi && r >= 0 && r < A.kv.max_ctx) quant_store_chunk8(A.kv, kvh, r, hh & 1, rawv[it], c);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    asm volatile("" ::: "memory");             // the tile loads below are instructions the compiler does not see as loads
  }

  // tiles of this group: tile0 + grp + 2u, u = 0 .. nu-1; both groups walk nstep steps (idle where they have no tile left) so
  // that every wave of the workgroup meets the same number of barriers
  const int ntl = max(0, tile1 - tile0);
  const int nu = (ntl + 1 - grp) >> 1;
  auto tile_of = [&](int u) __attribute__((always_inline)) { return tile0 + grp + 2 * min(u, nu - 1); };   // past the end: the last tile again

  float m_run = vrow ? -1e30f : 0.f, l_run = 0.f;   // m_run in log2 units, shared by the two lanes of a row; a lane without a row never asks for one
  f16v o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;

  const float sc_log2 = kLog2e / sqrtf((float)kD);
  uint32_t magic = kMagic;
  asm volatile("" : "+v"(magic));
  auto load_tile_raw = [&](int T, const LaneOffs& offs, auto& r) __attribute__((always_inline)) { load_raw(kv_page_uniform(A.kv, kvh, T << 5), (T << 5) % kPageTok, offs, r); };
  if (nu > 0) {                                // the first tile: a quarter a wave
    Raw<1> start;
    load_tile_raw(tile_of(0), lane_offs(gt), start);
    wait_raw<0>(start);
    dequant_to_lds(lds[grp][0], gt, start, magic, sc_log2);
  }

  // The probabilities and the V fragments of a tile stay in registers until the next matrix phase; their eight
  // MFMAs open the NEXT matrix phase.  The first one multiplies zeros; the product of the last tile follows the loop.
  h8 pf[2], vfr[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) { vfr[c][e] = (_Float16)0.f; pf[c & 1][e] = (_Float16)0.f; }
  auto pv = [&]() __attribute__((always_inline)) {                            // O^T += V^T P^T : d-tile dt (32 rows of the V image), k-step u (16 tokens)
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int u = 0; u < 2; ++u) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vfr[2 * dt + u], pf[u], o[dt], 0, 0, 0);
  };
  float s[16];                                 // exponents of the tile in hand: written by the matrix phase, used by the vector phase
  float m_sub = 0.f;
  bool first = true;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = -INFINITY;

  // ---- matrix phase of the group's tile u (buffer cb of the group): PV of the tile before, scores of this one ----
  auto matrix_phase = [&](const int u, const int cb) __attribute__((always_inline)) {
    const uint8_t* buf = lds[grp][cb];
    h8 kfr[8];
#pragma unroll
    for (int c = 0; c < 8; ++c)
      kfr[c] = __builtin_bit_cast(h8, *reinterpret_cast<const uint4*>(buf + kLdsK + j * kKPitch + (4 * (c >> 1) + 2 * (c & 1) + h) * 16));
    pv();
    // scores: per scale group two chained MFMAs (32 channels), then the fp32 sum times the group scale.  A row that has
    // seen no key yet (m_run is the "no keys" marker) starts its chain from 0.
    first = m_run < -1e29f;
    m_sub = first ? 0.f : m_run;
    const float4 sc = *reinterpret_cast<const float4*>(buf + kLdsS + (16 * h + (j & 15)) * 16);
    float4 sc0[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) sc0[a] = *reinterpret_cast<const float4*>(buf + kLdsS0 + 64 * h + 16 * a);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f16v part;
#pragma unroll
      for (int r = 0; r < 16; ++r) part[r] = 0.f;
      part = __builtin_amdgcn_mfma_f32_32x32x16_f16(kfr[2 * m], qf[2 * m], part, 0, 0, 0);
      part = __builtin_amdgcn_mfma_f32_32x32x16_f16(kfr[2 * m + 1], qf[2 * m + 1], part, 0, 0, 0);
      // part[r]: key 8(r/4) + 4h + r%4 of the tile against row j
      if (m == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = __builtin_fmaf(part[r], (&sc0[r >> 2].x)[r & 3], -m_sub);
      } else scale_scores<0>(s, part, (&sc.x)[m]);
    }
    // the V fragments are requested here and used in the next matrix phase: their latency runs under the vector phase
#pragma unroll
    for (int c = 0; c < 8; ++c)
      vfr[c] = __builtin_bit_cast(h8, *reinterpret_cast<const uint4*>(buf + kLdsV + (32 * (c >> 1) + j) * kVPitch + (16 * (c & 1) + 8 * h) * 2));
  };
  // ---- vector phase of tile u: softmax of its scores ----
  auto softmax = [&](const int u) __attribute__((always_inline)) {
    {
      const int t0 = tile_of(u) << 5;
      // online softmax with a lazily raised maximum: a row's offset m_run only moves when the probabilities of a lane
      // sum to more than kRaiseSum (or when the row sees its first keys); they are then taken again.  The row sum is taken from
      // the fp16 probabilities the PV product uses (two per dot2), which hold 2^16.
      if (t0 + 32 > minlen) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = t0 + 8 * (r >> 2) + 4 * h + (r & 3);
          s[r] = key < len ? s[r] : -INFINITY;
        }
      }
      const h2 ones = {(_Float16)1.f, (_Float16)1.f};
      float lsum;
      auto exps = [&]() __attribute__((always_inline)) {
        float lsum0 = 0.f, lsum1 = 0.f;
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const h2 p01 = {(_Float16)__builtin_amdgcn_exp2f(s[r]), (_Float16)__builtin_amdgcn_exp2f(s[r + 1])};
          const h2 p23 = {(_Float16)__builtin_amdgcn_exp2f(s[r + 2]), (_Float16)__builtin_amdgcn_exp2f(s[r + 3])};
          lsum0 = __builtin_amdgcn_fdot2(p01, ones, lsum0, false);
          lsum1 = __builtin_amdgcn_fdot2(p23, ones, lsum1, false);
          pf[r >> 3][r & 7] = p01[0]; pf[r >> 3][(r & 7) + 1] = p01[1]; pf[r >> 3][(r & 7) + 2] = p23[0]; pf[r >> 3][(r & 7) + 3] = p23[1];
        }
        lsum = lsum0 + lsum1;
      };
      exps();
      if (__any(first || lsum > kRaiseSum)) {
        float tmax = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[r]);
        tmax = lane_op32(tmax, LaneMax{});
        const bool seen = tmax > -INFINITY;                       // false: every key of the tile lies past the row's length
        const bool high = lane_op32(lsum, LaneMax{}) > kRaiseSum; // of either lane of the row; a row that is neither first nor high keeps its bits
        const float d = first ? (seen ? tmax : 0.f) : high ? fmaxf(tmax, 0.f) : 0.f;
        const float alpha = first ? 1.f : __builtin_amdgcn_exp2f(-d);   // a first tile finds zeros in l and o
        if (!first || seen) m_run = m_sub + d;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] -= d;
        exps();
      }
      l_run += lsum;
    }
  };
  // ---- the group's tile k + 1, whose raw codes `rs` holds, goes to the buffer that tile k does not occupy (after the last
  //      tile that buffer is read by nobody); the request for tile k + 3 replaces them (past the end: the last tile again, so
  //      that the count of loads in flight is static) ----
  auto feed = [&](const int k, const int cb, const int t4, const LaneOffs& offs, auto& rs) __attribute__((always_inline)) {
    constexpr int kLoads = sizeof(rs) / 4;    // every register is a load of its own
    wait_raw<kLoads>(rs);                      // the loads of the other register set stay in flight
    dequant_to_lds(lds[grp][cb ^ 1], t4, rs, magic, sc_log2);
    load_tile_raw(tile_of(k + 3), offs, rs);
  };
  // One workgroup barrier per step.  Between two barriers group 0 runs the matrix and then the vector phase of its tile k,
  // group 1 the vector phase of its tile k - 1 and then the matrix phase of its tile k: each time one group's MFMAs run
  // under the other's vector work.  Both dequantize tile k + 1 in step k, into the buffer of tile k - 1, which nobody has
  // read since the barrier before.  The wave in its vector phase goes first when both waves of a SIMD have an instruction
  // to issue: at equal priority the older wave (group 0) wins in both of its phases and the younger group sets the pace.
  // With a barrier behind either phase the waves waited 130 cycles behind the matrix phase and 250 behind the vector phase
  // of a step of 2,780.  us, two barriers / one: 16 layers of 1,500 rows on an empty cache 742 / 704, of 64 rows at 32,768
  // tokens 731 / 716.
  // 2,048 rows at 131,072 tokens, 2 layers 8,043 / 8,027: the waves wait in 27 % of their cycles instead of 32, but are in
  // line for an issue slot in 27 instead of 24 (1,401 / 1,384 cycles a tile, at 2.1 GHz) - a long slice is bound by what
  // its two waves a SIMD have to issue.
  // The loads of a group live inside its own branch from the request to the last wait (a join would copy their registers).
  const int nstep = max((ntl + 1) >> 1, (ntl >> 1) + 1);
  auto run = [&](auto role, auto group, const int t4) __attribute__((always_inline)) {
    constexpr int kRole = decltype(role)::value;
    constexpr bool kCompute = kRole >= kComputeOnly, kFeeds = kRole != kIdle && kRole != kComputeOnly;
    const LaneOffs offs = lane_offs(t4);
    Raw<quarters<kRole>()> raw0{}, raw1{};     // raw codes of the group's next two tiles: loads run two tiles ahead of their use
    auto step = [&](const int k, const int cb, auto& rs) __attribute__((always_inline)) {
      if constexpr (decltype(group)::value == 0) {
        if (k < nu) {
          if constexpr (kCompute) {
            matrix_phase(k, cb);
            __builtin_amdgcn_s_setprio(2);
            softmax(k);
          }
          if constexpr (kFeeds) feed(k, cb, t4, offs, rs);
          if constexpr (kCompute) __builtin_amdgcn_s_setprio(0);
        }
      } else {
        if constexpr (kCompute) {
          __builtin_amdgcn_s_setprio(2);
          if (k > 0 && k <= nu) softmax(k - 1);
        }
        if (k < nu) {
          if constexpr (kFeeds) feed(k, cb, t4, offs, rs);
          if constexpr (kCompute) {
            __builtin_amdgcn_s_setprio(0);
            matrix_phase(k, cb);
          }
        }
      }
      __syncthreads();
    };
    if (kFeeds && nu > 0) { load_tile_raw(tile_of(1), offs, raw1); load_tile_raw(tile_of(2), offs, raw0); }
    __syncthreads();
    for (int k = 0; k < nstep; k += 2) {
      step(k, 0, raw1);
      if (k + 1 < nstep) step(k + 1, 1, raw0);
    }
    if constexpr (kFeeds) {
      wait_raw<0>(raw0);                       // every request has been answered before the registers it names are given up
      wait_raw<0>(raw1);
    }
  };
  // Who decodes: a quarter each, or, in a window whose blocks have rows for at most three waves of a group, the waves without rows:
  // all four quarters by one of them or two by each of two; the waves with rows then only compute.  us per 16 layers, a quarter
  // by every wave in blocks of 128 rows / so, in blocks cut at the even share rounded up to whole waves: 24 rows (128 + 16, 96 + 48) at 30,000 tokens
  // 454.5 / 427, with a tree at 9,000 283.6 / 268, 48 (128 + 128 + 32, three of 96) at 9,000 337.5 / 326.3, 16 at 30,000 338 / 328, 11 at
  // 5,000 203.5 / 200.5, 32 at 12,000 312 / 306.  One kernel for both was 1.5 % slower on blocks of four waves.
  const int computing = (min(nrows, (rb + 1) * RPB) - rb * RPB + 31) >> 5, feeder = wave - computing;
  auto play = [&](auto group) __attribute__((always_inline)) {
    if constexpr (CHUNK || !FEW) {
      if (has_rows) run(std::integral_constant<int, kComputeFeed>{}, group, gt);
      else run(std::integral_constant<int, kFeed1>{}, group, gt);
    } else {
      if (has_rows) run(std::integral_constant<int, kComputeOnly>{}, group, lane);
      else if (computing == 3) run(std::integral_constant<int, kFeed4>{}, group, lane);
      else if (feeder < 2) run(std::integral_constant<int, kFeed2>{}, group, 128 * feeder + lane);
      else run(std::integral_constant<int, kIdle>{}, group, lane);
    }
  };
  if (grp == 0) play(std::integral_constant<int, 0>{});
  else play(std::integral_constant<int, 1>{});
  __builtin_amdgcn_s_setprio(0);
  if (has_rows) pv();

  // ---- the two groups' states of a row are merged: group 1 leaves its registers in LDS (the tile buffers are free
  //      after the last barrier), group 0 folds them into its own.  Wave w of either group holds the same rows in the
  //      same registers, so the exchange is a plain register image: [wave][register][lane]. ----
  float* xo = reinterpret_cast<float*>(&lds[0][0][0]);               // 4 waves x 64 registers x 64 lanes = 65536 bytes
  float* xm = xo + 4 * 64 * 64;                                       // then m and l, [wave][lane]: 2048 bytes
  float* xl = xm + 4 * 64;
  static_assert(4 * 64 * 64 * 4 + 2 * 4 * 64 * 4 <= 4 * kLdsBuf, "the register image of group 1 fits the tile buffers");
  if (grp == 1 && has_rows) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) xo[(wave * 64 + dt * 16 + r) * 64 + lane] = o[dt][r];
    xm[wave * 64 + lane] = m_run; xl[wave * 64 + lane] = l_run;
  }
  __syncthreads();
  if (grp == 1 || !has_rows) return;           // no barrier follows
  {
    const float mb = xm[wave * 64 + lane], lb = xl[wave * 64 + lane];
    const float m2 = fmaxf(m_run, mb);
    const float wa = __builtin_amdgcn_exp2f(m_run - m2), wb = __builtin_amdgcn_exp2f(mb - m2);   // both markers: 2^0, sums stay 0
    m_run = m2; l_run = wa * l_run + wb * lb;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = wa * o[dt][r] + wb * xo[(wave * 64 + dt * 16 + r) * 64 + lane];
  }
  // ---- partials: normalised fp16.  o[dt][4a+b] of lane (row j, half h) is V-image row 32dt + 8a + 4h + b, i.e.
  //      channel 64(a&1) + 32h + 8b + 4(a>>1) + dt: for each (a&1, b) the lane owns 8 consecutive channels.
  //      Rows go through LDS so that every store instruction writes whole 256-byte rows: 16 lanes per row instead of
  //      64 scattered 16-byte pieces.  A wave stages its rows inside the part of the register image only it has read. ----
  constexpr int kOPitch = 2 * kD + 16;                       // bytes per staged row
  static_assert(32 * kOPitch <= 64 * 64 * 4, "a wave's staging area lies inside its own part of the register image");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");     // the image has been read before the wave overwrites it
  uint8_t* stage = &lds[0][0][0] + wave * (64 * 64 * 4);     // 4 waves x 8704 bytes, 16384 bytes apart
  float l = l_run;
  l = lane_op32(l, LaneAdd{});
  const bool direct = CHUNK && A.S == 1 && A.out16;          // uniform over the grid
  if (!direct && vrow && h == 0) { A.pm[pidx] = m_run; A.pl[pidx] = l; }
  // a row none of whose scores is a number keeps the marker: the combiner drops its partial and writes zeros, and so does this
  // (behind a branch: 64 selects here, or 32 on the packed rows, are 0.2 us of a slice, as instructions fetched for nothing)
  if (CHUNK && direct && __any(m_run < -1e29f)) {
    const bool none = m_run < -1e29f;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = none ? 0.f : o[dt][r];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int a0 = 0; a0 < 2; ++a0)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      h8 v;
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = (_Float16)(o[c & 3][4 * (2 * (c >> 2) + a0) + b] * inv);
      uint4 packed = __builtin_bit_cast(uint4, v);
      if (CHUNK && BF && direct) {
        float y[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) y[c] = o[c & 3][4 * (2 * (c >> 2) + a0) + b] * inv;
        packed = pack_out8(y, 1);
      }
      *reinterpret_cast<uint4*>(stage + j * kOPitch + (64 * a0 + 32 * h + 8 * b) * 2) = packed;
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");     // the wave reads back what its own lanes wrote
  const int chunk = lane & 15;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int jr = 4 * k + (lane >> 4);
    const int Rr = row0 + jr;
    if (Rr < nrows && Rr < (rb + 1) * RPB) {
      const size_t p = ((size_t)(Rr / kG) * A.S + split) * A.n_heads + kvh * kG + Rr % kG;   // S == 1: also the output row
      const uint4 v = *reinterpret_cast<const uint4*>(stage + jr * kOPitch + chunk * 16);
      if constexpr (CHUNK) *reinterpret_cast<uint4*>((direct ? A.out16 : A.pacc16) + p * kD + chunk * 8) = v;   // a slice in several splits gains nothing from writing through
      else store_partial16(A.pacc16 + p * kD + chunk * 8, v);
    }
  }
}

template <bool CHUNK, bool FEW>
static void launch_wide(const AttnArgs& A, hipStream_t st) {
  const int rows = kG * A.M, rb = (rows + A.rows_per_block - 1) / A.rows_per_block;
  const dim3 grid(A.S * A.kv.n_kv * rb);
  if (A.in_bf16) hipLaunchKernelGGL((attend_wide_kernel<true, CHUNK, FEW>), grid, dim3(NT), 0, st, window_head(A), window_sizes(A), window_tail(A));
  else hipLaunchKernelGGL((attend_wide_kernel<false, CHUNK, FEW>), grid, dim3(NT), 0, st, window_head(A), window_sizes(A), window_tail(A));
}
void launch_attend_wide(const AttnArgs& A, hipStream_t st) {
  if (A.rows_per_block <= 96) launch_wide<false, true>(A, st);       // three waves of rows at most in every block
  else launch_wide<false, false>(A, st);
}
void launch_attend_chunk(const AttnArgs& A, hipStream_t st) {
  if (A.kv.n_kv * ((kG * A.M + A.rows_per_block - 1) / A.rows_per_block) < 128) launch_wide<true, true>(A, st);
  else launch_wide<true, false>(A, st);
}

}  // namespace yka
