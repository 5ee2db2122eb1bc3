// Split-KV attention over the int4 cache for row tiles of at most 2 tokens x 6 heads (single-token decode and the
// building block for any window), plus the split combiner.  gfx950 (wave64, MFMA 16x16x32 f16).
//
// What it computes is the reference's split-KV pass (src/attention_kv4q.cu:71-146, production form
// src/q35_atxpk3.cuh:131-477): for every query row, an online softmax over the keys of one split, written as
// (m, l, acc) partials, merged by a combiner (src/attention_kv4q.cu:325-332).  How it computes it is specific to
// CDNA4:
//   * one wave owns a 32-key tile.  K rows are read as one 16-byte chunk per lane; the page layout puts one dword of
//     every scale group into that chunk, so MFMA step m contracts exactly the 32 channels of group m.  V is read as
//     one dword per (lane, token) so that a lane ends up with 8 tokens of the same 8 channels - the operand shape
//     the token-contracting MFMA needs;
//   * codes become fp16 without integer conversion.  V: a nibble OR-ed into the mantissa of 1024.0 is 1024+n (or
//     1024+16n for the odd nibble of a byte); subtracting 1032 (1152) gives n-8 (16(n-8)) exactly.  K: a nibble left in
//     place in a zero word IS an fp16, the subnormal n * 2^-24, and the matrix pipe takes subnormal inputs unflushed: an
//     AND per pair of codes is the whole conversion, the offset -8 rides in the MFMA's initial accumulator as
//     -8 * 2^-24 * sum(q) per (row, scale group), and the 2^24 is folded into the exponent's scale;
//   * K stays exact: the MFMA multiplies Q by the integer codes, and the fp16 group scale is applied to the fp32
//     partial sum of each group (rounding q*scale to fp16 first costs 7e-4 relative L2 on inputs with outlier
//     channels, most of the 1e-3 budget).  V is scaled in fp16 (one rounding, 2e-4);
//   * scores S^T = K Q^T come out of the MFMA with one query row per lane column, which is already the B-operand
//     layout of O^T += V^T P^T: probabilities never move between lanes;
//   * running maxima are shared by the 4 lane groups of a row through two cross-lane exchanges per tile;
//   * a wave that has more than one tile to walk keeps two raw tiles in registers: the 16 loads of the tile after the
//     one it works on are in flight while it dequantizes and multiplies (2 waves per SIMD, 8 per CU, two tiles each).
//     Against 4 waves per SIMD with one tile each this measures the same at 32k tokens per head, 17 % faster at 262k
//     and 10 % faster with 32 streams in one launch;
//   * quantize-on-append is fused into the decode launch (a launch costs about 2.5 us here, the same order as the
//     whole KV stream): the workgroup whose tiles contain a row appended by this pass quantizes and stores that row
//     before it loads the tile;
//   * the split merge is a second launch by default.  It can ride in the same launch when the caller hands over a
//     ticket array: every workgroup of a (kv head, row tile) column stores its partials with agent-scope stores (written
//     through its XCD's L2, which the other XCDs do not see), waits until they are acknowledged, and takes a ticket; the
//     workgroup that draws the last one reads the column's partials back with agent-scope loads and writes the final
//     rows.  No cache-wide write-back or invalidate is involved (a device-scope release fence in every workgroup measured
//     4x slower than a second launch), but the last workgroup still pays three dependent trips to memory after its
//     tiles - stores acknowledged, ticket, loads - and that measures slower than the gap between two kernels: 14.7
//     against 8.6 us per layer call at 4k tokens, 18.9 against 12.0 at 32k, 34.0 against 24.9 at 131k (one token; two
//     tokens add another 7 to 14 us).
#include <type_traits>
#include "codec_device.h"
#include "sign_device.h"
#include "tile32_device.h"

namespace yka {

// Agent-scope accesses for data that workgroups on different XCDs hand to each other inside one launch: relaxed atomics,
// which the compiler turns into plain stores and loads with the scope bit that makes them go past the XCD-local L2.
__device__ __forceinline__ void st_agent(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float ld_agent(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint4 ld_agent16(const uint16_t* p) {
  const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
  const uint64_t a = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), b = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_uint4((uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32));
}

// The workgroup's partials are out (or its "no keys" markers): wait until the stores are acknowledged, take a ticket of
// the column.  True for the workgroup that drew the last one: every partial of the column is then visible to agent-scope
// loads.  The ticket is an acquire-release operation at agent scope behind a workgroup barrier, so the order "partials,
// then ticket" (writers) and "ticket, then partials" (the merging workgroup) holds by the memory model and not only by
// the explicit wait.  The counter is also put back to zero; the host zeroes it in front of every launch regardless.
__device__ __forceinline__ bool last_of_column(const AttnArgs& A, int* s_ticket) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int* t = A.tickets + blockIdx.y * gridDim.z + blockIdx.z;
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(t, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (old == A.S - 1) __hip_atomic_store(t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *s_ticket = old;
  }
  __syncthreads();
  return *s_ticket == A.S - 1;
}

// The combiner of one column (reference: src/attention_kv4q.cu:325-332), run by its last workgroup: 256 threads, rows =
// the column's tokens x 6 heads.  Per token: thread t weighs split t of each head (w = 2^(m - max m) * l), then 16 split
// lanes x 16 channel lanes sum w * acc/l over the splits, K splits in flight per lane and head; K * 16 >= S.  All six
// heads are in flight at once when K is 4 (one memory round trip: decode up to 64 splits), one head at a time otherwise.
// lds: 6 * 256 + 4 * 6 * 128 + 64 floats.
template <int TPT, int K>
__device__ __forceinline__ void combine_column(const AttnArgs& A, int kvh, int rt, float* lds) {
  constexpr int HB = K <= 4 ? kG : 1;                  // heads per batch of loads
  float* s_w = lds;                                    // [6][256] weights
  float* s_o = lds + kG * 256;                         // [4 waves][6 heads][128]
  float* s_red = s_o + 4 * kG * kD;                    // [4][6] maxima, then [4][6] weight sums
  const int tid = threadIdx.x, wave = tid >> 6, sl = tid >> 4, c8 = (tid & 15) * 8;
  const int ntok = min(TPT, A.M - TPT * rt);
  for (int tk = 0; tk < ntok; ++tk) {
    const int tj = TPT * rt + tk;
    const size_t p0 = (size_t)tj * A.S * A.n_heads + kvh * kG;        // (split s, head h) lives at p0 + s * n_heads + h
    const size_t stride = (size_t)A.n_heads * kD;
    float pmv[kG], plv[kG];
#pragma unroll
    for (int h = 0; h < kG; ++h) {
      pmv[h] = tid < A.S ? ld_agent(A.pm + p0 + (size_t)tid * A.n_heads + h) : -1e30f;
      plv[h] = tid < A.S ? ld_agent(A.pl + p0 + (size_t)tid * A.n_heads + h) : 0.f;
    }
    uint4 u[HB][K];
    auto request = [&](int h0) __attribute__((always_inline)) {
#pragma unroll
      for (int hh = 0; hh < HB; ++hh)
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int sp = sl + 16 * k;
          u[hh][k] = sp < A.S ? ld_agent16(A.pacc16 + (p0 + h0 + hh) * kD + (size_t)sp * stride + c8) : make_uint4(0, 0, 0, 0);
        }
    };
    request(0);
    // maxima over the splits, per head
    float mx[kG];
#pragma unroll
    for (int h = 0; h < kG; ++h) {
      mx[h] = pmv[h];
#pragma unroll
      for (int o = 32; o; o >>= 1) mx[h] = fmaxf(mx[h], __shfl_xor(mx[h], o, 64));
    }
    __syncthreads();                                   // the previous token's readers of s_red / s_w / s_o are done
    if ((tid & 63) == 0)
#pragma unroll
      for (int h = 0; h < kG; ++h) s_red[wave * kG + h] = mx[h];
    __syncthreads();
    float wsum[kG];
#pragma unroll
    for (int h = 0; h < kG; ++h) {
      const float M2 = fmaxf(fmaxf(s_red[h], s_red[kG + h]), fmaxf(s_red[2 * kG + h], s_red[3 * kG + h]));
      const float w = (tid < A.S && pmv[h] > -1e29f) ? exp2f(pmv[h] - M2) * plv[h] : 0.f;
      s_w[h * 256 + tid] = w;
      wsum[h] = w;
#pragma unroll
      for (int o = 32; o; o >>= 1) wsum[h] += __shfl_xor(wsum[h], o, 64);
    }
    __syncthreads();                                   // maxima read by everyone, weights written
    if ((tid & 63) == 0)
#pragma unroll
      for (int h = 0; h < kG; ++h) s_red[wave * kG + h] = wsum[h];
    // weighted sums over the splits
#pragma unroll
    for (int h0 = 0; h0 < kG; h0 += HB) {
      if (h0) request(h0);
#pragma unroll
      for (int hh = 0; hh < HB; ++hh) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int sp = sl + 16 * k;
          const float w = sp < A.S ? s_w[(h0 + hh) * 256 + sp] : 0.f;
          const uint4 r = w != 0.f ? u[hh][k] : make_uint4(0, 0, 0, 0);   // a row of weight 0 may hold anything
          const h8 v = __builtin_bit_cast(h8, r);
#pragma unroll
          for (int c = 0; c < 8; ++c) acc[c] += w * (float)v[c];
        }
        // the wave's 4 split lanes (lane bits 4 and 5), then the 4 waves through LDS
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c] = lane_rows(acc[c], LaneAdd{});
        if ((tid & 48) == 0) {
          float* d = s_o + (wave * kG + h0 + hh) * kD + c8;
          *reinterpret_cast<float4*>(d) = make_float4(acc[0], acc[1], acc[2], acc[3]);
          *reinterpret_cast<float4*>(d + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
        }
      }
    }
    __syncthreads();
    if (tid < kG * 16) {                               // 16 lanes per head, 8 channels each: one 16-byte store
      const int h = tid >> 4;
      const float L = s_red[h] + s_red[kG + h] + s_red[2 * kG + h] + s_red[3 * kG + h];
      const float inv = L > 0.f ? 1.f / L : 0.f;       // a row that saw no key at all (a rejected row of a multi-stream pass)
      float yv[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float o = s_o[(0 * kG + h) * kD + c8 + c] + s_o[(1 * kG + h) * kD + c8 + c] + s_o[(2 * kG + h) * kD + c8 + c] + s_o[(3 * kG + h) * kD + c8 + c];
        yv[c] = o * inv;
      }
      *reinterpret_cast<uint4*>(A.out16 + ((size_t)tj * A.n_heads + kvh * kG + h) * kD + c8) = pack_out8(yv, A.out_bf16);
    }
  }
}

// grid (S, n_kv, ceil(M/TPT)), block 256 (4 waves).  Workgroup = (split, kv head, row tile of TPT tokens x 6 heads):
// TPT = 2 for a single-stream pass; MS (multi-stream pass, reference: src/q35_atxpk_ms.cu:13-33): one token per tile,
// which reads the container and the position its row map names.
template <bool MS>
__global__ void __launch_bounds__(256, 2) attend_narrow_kernel(uint64_t p_pos, uint64_t p_slot, int p_m, AttnArgs A) {
  // multi-stream passes read all three, the others the position alone
  if (MS) { A.rows.pos = head_ptr<const int>(p_pos); A.rows.slot = head_ptr<const int>(p_slot); A.M = p_m; } else A.d_pos = head_ptr<const int>(p_pos);
  __shared__ float s_m[4][16], s_l[4][16];
  __shared__ __align__(16) float s_acc[4][kAccWave];       // 8576 floats; the fused combiner needs 4672 of them
  __shared__ int s_ticket;
  constexpr int TPT = MS ? 1 : 2;
  const bool fused = A.tickets != nullptr;                 // uniform over the grid
  int split = blockIdx.x, rt = blockIdx.z;
  const int kvh = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // a scalar: tile indices and page pointers are wave uniform
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  int pos, slot = 0; bool row_ok = true;
  MsShare share{};
  if (MS) {
    if (A.adapt) {
      const int b = split + A.S * rt;
      share = ms_share(A.rows, A.M, A.kv.max_ctx, A.S * A.M, A.ms_short, b, A.plan, b == 0 && kvh == 0 && wave == 0);
      if (share.row < 0) return;
      split = share.split; rt = share.row; pos = share.pos; slot = share.slot;
    } else { pos = A.rows.pos[rt]; slot = A.rows.slot[rt]; }
    row_ok = pos >= 0 && pos < A.kv.max_ctx && slot >= 0 && slot < A.rows.n_slots;   // a bad row reads nothing and yields zeros
    A.kv = slot_view(A.kv, A.rows, row_ok ? slot : 0);
  } else {
    pos = *A.d_pos;
  }

  // query row of this lane column: j = i -> (token TPT*rt + i/6, head kvh*6 + i%6); the other columns are padding
  const int tl = TPT * rt + i / kG;                // token index inside the slice
  const bool vrow = i < TPT * kG && tl < A.M && row_ok;
  const int head = kvh * kG + i % kG;
  int len = 0;
  if (vrow) {
    if (MS) len = pos + 1;
    else { const int tg = A.tok0 + tl; len = pos + (A.depth ? (int)A.depth[tg] : tg) + 1; }
    len = min(len, A.kv.max_ctx);
  }
  int maxlen = len, minlen = vrow ? len : 0x7fffffff;
  maxlen = lane_row16(maxlen, LaneMax{}); minlen = lane_row16(minlen, LaneMin{});
  maxlen = __builtin_amdgcn_readfirstlane(maxlen); minlen = __builtin_amdgcn_readfirstlane(minlen);
  // The grid is sized for long contexts; how many of its splits a row tile uses follows from the length it finds on the
  // device: at least two 32-key tiles per workgroup.  The other workgroups leave the "no keys" marker and exit, and
  // the combiner does not read their rows.
  const int ntiles = (maxlen + 31) >> 5;
  const int s_used = MS && A.adapt ? share.n : min(A.S, max(1, ntiles >> 1));
  // partials of (token tj, split) start at pair * n_heads
  auto pair_of = [&](int tj) __attribute__((always_inline)) { return MS && A.adapt ? share.base + split : (size_t)tj * A.S + split; };
  if (split >= s_used) {
    const int j = threadIdx.x, tj = TPT * rt + j / kG;
    if (j < TPT * kG && tj < A.M) {
      const size_t p = pair_of(tj) * A.n_heads + kvh * kG + j % kG;
      if (fused) { st_agent(A.pm + p, -1e30f); st_agent(A.pl + p, 0.f); }
      else { A.pm[p] = -1e30f; A.pl[p] = 0.f; }
    }
    if (fused && last_of_column(A, &s_ticket)) {
      if (A.S <= 64) combine_column<TPT, 4>(A, kvh, rt, &s_acc[0][0]); else combine_column<TPT, 16>(A, kvh, rt, &s_acc[0][0]);
    }
    return;
  }
  const int tps = (ntiles + s_used - 1) / s_used;
  const int tile0 = split * tps, tile1 = min(ntiles, tile0 + tps);

  // ---- fused quantize-on-append (decode, M <= 2, one row tile): a row of this pass is written by the one workgroup
  //      whose tile range holds it - the only workgroup of this kv head that will read it in this launch.  Writer and
  //      readers are waves of one workgroup, i.e. of one CU and one (write-through) L1, so workgroup-scope fences
  //      around the barrier order the stores before the loads without any cache maintenance. ----
  if (MS && A.k16 && row_ok) {
    int lane_pos;
    uint64_t todo = ms_new_rows(A.rows, A.M, slot, pos, tile0, tile1, lane_pos);
    if (todo) {                        // uniform over the workgroup
      for (; todo; todo &= todo - 1) {
        const int t = __builtin_ctzll(todo);
        const bool isv = threadIdx.x >= 128;
        quant_store_row(A.kv, kvh, __builtin_amdgcn_readlane(lane_pos, t), isv, (isv ? A.v16 : A.k16) + ((size_t)t * A.kv.n_kv + kvh) * kD, threadIdx.x & 127, A.in_bf16);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  }
  if (!MS && A.k16) {
    bool mine = false;
    for (int t = 0; t < A.M; ++t) {
      const int r = pos + A.tok0 + t;              // k16/v16 point at row 0 of the pass, this slice starts at row tok0
      // A row no query row of this launch can see (a depth table may say so) lies past the last tile when it opens a new
      // one: nobody reads it now, the last workgroup in use stores it.  All conditions are uniform over the workgroup.
      const bool held = (r >> 5) >= tile0 && (r >> 5) < tile1, unseen = (r >> 5) >= ntiles && split == s_used - 1;
      if (r < 0 || r >= A.kv.max_ctx || !(held || unseen)) continue;
      mine = true;
      const bool isv = threadIdx.x >= 128;
      const uint16_t* src = (isv ? A.v16 : A.k16) + ((size_t)(A.tok0 + t) * A.kv.n_kv + kvh) * kD;
      quant_store_row(A.kv, kvh, r, isv, src, threadIdx.x & 127, A.in_bf16);
    }
    if (mine) {                      // uniform over the workgroup
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  }

  // Q fragments: B operand of S^T = K Q^T.  MFMA step m (= scale group m), lane (row i, lane group g), element e
  // <-> channel 32m + 8g + pi(e), pi = [0,4,1,5,2,6,3,7] (the order dq_dword_int produces); odd channels carry 1/4, even ones 4.
  // The four loads are written as instructions and only requested here: the first tiles are requested right behind them
  // and q_ready<N> then waits for the query alone, leaving the N tile loads in flight - one trip to memory before the
  // first MFMA instead of two.  Padding lanes read row 0 of the slice (memory that exists) and drop it.
  // q_ready is called once in every branch below.  It does not name the query registers as operands of its wait (a
  // wait site per branch that redefines them makes the compiler place copies of the registers in front of one of the
  // waits, i.e. copies of registers whose loads are still in flight); instead the wait hands out a zero that is OR-ed
  // into the raw words, so that nothing computed from them can be scheduled ahead of it.
  h8 qf[4];
  f4 kinit[4];                 // initial accumulators of the score MFMAs: the code offset -8, see dq_dword_sub
  u32x4 qraw[4];
  {
    const uint16_t* qrow = A.q16 + (vrow ? ((size_t)tl * A.n_heads + head) * kD : (size_t)0) + 8 * g;
#pragma unroll
    for (int m = 0; m < 4; ++m) asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(qraw[m]) : "v"(qrow + 32 * m));
  }
  auto q_ready = [&](auto n_younger) __attribute__((always_inline)) {
    uint32_t z;
    asm volatile("s_waitcnt vmcnt(%1)\n\tv_mov_b32 %0, 0" : "=v"(z) : "n"(decltype(n_younger)::value));
    // the odd nibble of a byte enters the MFMA as 16 n: its query channels carry 1/4 and the others 4, so that both
    // kinds of products are 4 q n and neither factor costs fp16 range at one end only (a plain 1/16 on the odd channels
    // pushes queries below 1e-3 into the subnormals); the 4 leaves with the softmax scale
    const _Float16 se = (_Float16)4.f, so = (_Float16)0.25f;
    uint4 qw[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) qw[m] = __builtin_bit_cast(uint4, vrow ? (qraw[m] | u32x4{z, z, z, z}) : u32x4{0u, 0u, 0u, 0u});
    rows16_to_f16(qw, A.in_bf16);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const h8 c = __builtin_bit_cast(h8, qw[m]);
      qf[m] = h8{c[0] * se, c[4] * se, c[1] * so, c[5] * so, c[2] * se, c[6] * se, c[3] * so, c[7] * so};
      // -8 * 2^-24 * (sum of the row's 32 query channels of group m): the lane's 8 channels, then its 3 sister lanes
      float qs = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) qs += (float)c[e];
      qs = lane_rows(qs, LaneAdd{});
      const float c0 = -32.f * kTwoM24 * qs;       // -8 per code, in the units of the products: 4 q n 2^-24
      kinit[m] = f4{c0, c0, c0, c0};
    }
  };
  const float sc_log2 = 0.25f * kTwo24 * kLog2e / sqrtf((float)kD);   // scores carry the 2^-24 of the subnormal codes and the 4 of the query fragments

  float m_run = -1e30f, l_run = 0.f;
  f4 o[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) o[b] = f4{0.f, 0.f, 0.f, 0.f};

  const LaneOffs offs = lane_offs(i, g);
  uint32_t magic = kMagic;
  asm volatile("" : "+v"(magic));
  // one 32-key tile: scores, online softmax, O += P V
  auto tile = [&](const int T, const RawTile& cur) __attribute__((always_inline)) {
    const int t0 = T << 5;
    const bool need_mask = t0 + 32 > minlen;         // wave uniform: only the last tiles of a row can hold keys past its length
    // ---- scores: two 16-key MFMA tiles; step m contracts scale group m, its fp32 sum is scaled afterwards ----
    float s[8];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const uint32_t w[4] = {cur.kw[kt][0], cur.kw[kt][1], cur.kw[kt][2], cur.kw[kt][3]};
      f4 part[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        h2 k4[4];
        dq_dword_sub(w[m], k4);
        const h8 kf = h8{k4[0][0], k4[0][1], k4[1][0], k4[1][1], k4[2][0], k4[2][1], k4[3][0], k4[3][1]};
        part[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[m], kinit[m], 0, 0, 0);
      }
      // part[m][r] = sum over group m of q * code for key t0 + 16kt + 4g + r and row i
      const uint32_t sw[8] = {cur.ks[kt][0][0], cur.ks[kt][0][1], cur.ks[kt][0][2], cur.ks[kt][0][3],
                              cur.ks[kt][1][0], cur.ks[kt][1][1], cur.ks[kt][1][2], cur.ks[kt][1][3]};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const h2 s01 = as_h2(sw[2 * r]), s23 = as_h2(sw[2 * r + 1]);
        float dot = __builtin_fmaf(part[0][r], (float)s01[0], 0.f);
        dot = __builtin_fmaf(part[1][r], (float)s01[1], dot);
        dot = __builtin_fmaf(part[2][r], (float)s23[0], dot);
        dot = __builtin_fmaf(part[3][r], (float)s23[1], dot);
        s[4 * kt + r] = dot;                           // raw units; log2(e)/sqrt(d) is folded into the exponent below
      }
    }
    if (need_mask) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { const int key = t0 + 16 * (e >> 2) + 4 * g + (e & 3); s[e] = key < len ? s[e] : -INFINITY; }
    }
    // ---- online softmax (one running maximum per row, shared by its 4 lane groups) ----
    float tmax = s[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) tmax = fmaxf(tmax, s[e]);
    tmax = lane_rows(tmax, LaneMax{});
    const float m_new = fmaxf(m_run, tmax * sc_log2);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);    // 0 on the first tile (m_run = -1e30): nothing to rescale yet
    const bool first = m_run < -1e29f;
    m_run = m_new;
    if (__any(alpha != 1.f && !first)) {
      l_run *= alpha;
#pragma unroll
      for (int b = 0; b < 8; ++b) { o[b][0] *= alpha; o[b][1] *= alpha; o[b][2] *= alpha; o[b][3] *= alpha; }
    }
    h8 pf;
#pragma unroll
    for (int e = 0; e < 8; ++e) { const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], sc_log2, -m_new)); l_run += p; pf[e] = (_Float16)p; }
    // ---- O^T += V^T P^T : 8 MFMAs, MFMA b covers channels 8*i' + b ----
    h2 va[8][4];
#pragma unroll
    for (int pe = 0; pe < 4; ++pe) {
      const uint32_t spk = cur.vs[pe >> 1][pe & 1];                            // scales of tokens (2pe, 2pe+1) of this lane
      const h2 s2 = as_h2(spk), s2q = s2 * h2{(_Float16)0.0625f, (_Float16)0.0625f};
      const h2 c1032 = {(_Float16)1032.f, (_Float16)1032.f}, c1152 = {(_Float16)1152.f, (_Float16)1152.f};
      const uint32_t w0 = cur.vw[2 * pe], w1 = cur.vw[2 * pe + 1];
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        // byte bb of both tokens side by side: low half = token 2pe, high half = token 2pe+1
        const uint32_t x = __builtin_amdgcn_perm(w1, w0, 0x0c040c00u + bb * 0x00010001u);
        va[2 * bb][pe] = (as_h2(nib(x, 0x000f000fu, magic)) - c1032) * s2;
        va[2 * bb + 1][pe] = (as_h2(nib(x, 0x00f000f0u, magic)) - c1152) * s2q;
      }
    }
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const h8 vf = h8{va[b][0][0], va[b][0][1], va[b][1][0], va[b][1][1], va[b][2][0], va[b][2][1], va[b][3][0], va[b][3][1]};
      o[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf, o[b], 0, 0, 0);
    }
  };
  // While the wave works on one of its tiles T0, T0 + stride, ..., the next is in flight in another register set.  Every
  // branch here is wave uniform, so the number of loads in flight at each wait is known: 16 if a younger tile was
  // requested, 0 otherwise.  The wait that names a tile's registers is the only one that does and unconditional (with one per
  // branch, or a conditional one, the compiler merges two versions of those registers, with copies placed before the wait); when
  // there is no younger tile a full wait without operands precedes it.
  // The first tile stands in front of the loop: it finds no sums to rescale.  The tiles of the loop begin where most of their 8-byte
  // instructions begin at a multiple of 8 bytes (wait_tile).  us per 16 layers, all tiles in one loop whose second half lay
  // where it fell / so: one token at 32,741 tokens 161.3 / 157.8, two at 3,000 121.8 / 117.8; 4 layers at 262,100 133.5 / 133.0.
  constexpr int stride = 4;
  const int T0 = tile0 + wave, Tend = tile1;
  auto request = [&](int T, RawTile& r) __attribute__((always_inline)) { load_tile(kv_page_uniform(A.kv, kvh, T << 5), (T << 5) % kPageTok, offs, r); };
  if (T0 + stride < Tend) {                            // two tiles or more: the next tile is always in flight
    RawTile ta, tb, tc;
    int T = T0 + stride;
    request(T0, ta);
    request(T, tb);
    q_ready(std::integral_constant<int, 2 * kTileLoads>{});
    wait_tile<kTileLoads>(ta);
    tile(T0, ta);
    for (;;) {
      if (T + stride < Tend) request(T + stride, tc); else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      wait_tile<kTileLoads, true>(tb);
      tile(T, tb);
      T += stride;
      if (T >= Tend) break;
      if (T + stride < Tend) request(T + stride, tb); else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      wait_tile<kTileLoads, true>(tc);
      tile(T, tc);
      T += stride;
      if (T >= Tend) break;
    }
  } else if (T0 < Tend) {                              // one: code of its own, in which nothing has to be jumped over
    RawTile t1;
    request(T0, t1);
    q_ready(std::integral_constant<int, kTileLoads>{});
    wait_tile<0>(t1);
    tile(T0, t1);
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // a wave without tiles: the requests are answered before their registers are given up
  }
  // ---- merge the 4 waves of the workgroup, write one partial per (row, split) ----
  l_run = lane_rows(l_run, LaneAdd{});
  if (g == 0) { s_m[wave][i] = m_run; s_l[wave][i] = l_run; }
  // o[b][r] of lane (row i, group g) is channel 8 (4g + r) + b: eight consecutive channels per r, two 16-byte writes
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float* d = &s_acc[wave][acc_row(i) + 8 * (4 * g + r)];
    *reinterpret_cast<float4*>(d) = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
    *reinterpret_cast<float4*>(d + 4) = make_float4(o[4][r], o[5][r], o[6][r], o[7][r]);
  }
  __syncthreads();
  // 8 or 4 channels a lane: the rows of two tokens keep 192 threads busy with 8, those of one with 4 (one token, 16 layers at 1,003
  // tokens, 110.5 us with 8 and 109.4 with 4; two tokens, 155,173 tokens, 27.1 and 27.3 a call)
  auto merge = [&](auto channels) __attribute__((always_inline)) {
    constexpr int C = decltype(channels)::value, LANES = kD / C;
    const int j = threadIdx.x / LANES, c0 = (threadIdx.x % LANES) * C;
    const int tj = TPT * rt + j / kG;
    if (j >= TPT * kG || tj >= A.M) return;
    float4 a[4][C / 4];                                     // all reads first: one LDS round trip
#pragma unroll
    for (int wv = 0; wv < 4; ++wv)
#pragma unroll
      for (int k = 0; k < C / 4; ++k) a[wv][k] = *reinterpret_cast<const float4*>(&s_acc[wv][acc_row(j) + c0 + 4 * k]);
    const float m0 = s_m[0][j], m1 = s_m[1][j], m2 = s_m[2][j], m3 = s_m[3][j];
    const float l0 = s_l[0][j], l1 = s_l[1][j], l2 = s_l[2][j], l3 = s_l[3][j];
    const float M2 = fmaxf(fmaxf(m0, m1), fmaxf(m2, m3));
    const float w0 = __builtin_amdgcn_exp2f(m0 - M2), w1 = __builtin_amdgcn_exp2f(m1 - M2), w2 = __builtin_amdgcn_exp2f(m2 - M2), w3 = __builtin_amdgcn_exp2f(m3 - M2);
    const size_t p = pair_of(tj) * A.n_heads + kvh * kG + j % kG;
    const float L = w0 * l0 + w1 * l1 + w2 * l2 + w3 * l3;
    const float inv = L > 0.f ? 1.f / L : 0.f;              // one division per lane, not one per channel
    uint32_t v[C / 2];
#pragma unroll
    for (int k = 0; k < C / 4; ++k) {
      const h2 lo = {(_Float16)((w0 * a[0][k].x + w1 * a[1][k].x + w2 * a[2][k].x + w3 * a[3][k].x) * inv),
                     (_Float16)((w0 * a[0][k].y + w1 * a[1][k].y + w2 * a[2][k].y + w3 * a[3][k].y) * inv)};
      const h2 hi = {(_Float16)((w0 * a[0][k].z + w1 * a[1][k].z + w2 * a[2][k].z + w3 * a[3][k].z) * inv),
                     (_Float16)((w0 * a[0][k].w + w1 * a[1][k].w + w2 * a[2][k].w + w3 * a[3][k].w) * inv)};
      v[2 * k] = as_u32(lo); v[2 * k + 1] = as_u32(hi);
    }
    uint16_t* const dst = A.pacc16 + p * kD + c0;
    if (fused) {
#pragma unroll
      for (int k = 0; k < C / 4; ++k)
        __hip_atomic_store(reinterpret_cast<uint64_t*>(dst + 4 * k), (uint64_t)v[2 * k] | ((uint64_t)v[2 * k + 1] << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (c0 == 0) { st_agent(A.pm + p, M2); st_agent(A.pl + p, L); }
    } else {
      if constexpr (C == 8) *reinterpret_cast<uint4*>(dst) = make_uint4(v[0], v[1], v[2], v[3]);
      else *reinterpret_cast<uint2*>(dst) = make_uint2(v[0], v[1]);
      if (c0 == 0) { A.pm[p] = M2; A.pl[p] = L; }
    }
  };
  if (!MS && A.M - TPT * rt > 1) merge(std::integral_constant<int, 8>{}); else merge(std::integral_constant<int, 4>{});
  if (fused && last_of_column(A, &s_ticket)) {   // the barrier inside also ends every read of s_acc above
    if (A.S <= 64) combine_column<TPT, 4>(A, kvh, rt, &s_acc[0][0]); else combine_column<TPT, 16>(A, kvh, rt, &s_acc[0][0]);
  }
}

void launch_attend_narrow(const AttnArgs& A, hipStream_t st) {
  if (A.rows.pos) hipLaunchKernelGGL(attend_narrow_kernel<true>, dim3(A.S, A.kv.n_kv, A.M), dim3(256), 0, st, (uint64_t)(uintptr_t)A.rows.pos, (uint64_t)(uintptr_t)A.rows.slot, A.M, A);
  else hipLaunchKernelGGL(attend_narrow_kernel<false>, dim3(A.S, A.kv.n_kv, (A.M + 1) / 2), dim3(256), 0, st, (uint64_t)(uintptr_t)A.d_pos, (uint64_t)0, A.M, A);
}

// combiner (reference: src/attention_kv4q.cu:325-332): M2 = max pm; w_s = pm_s > -1e29 ? 2^(pm_s - M2) * pl_s : 0;
// y = sum w_s * (acc_s / l_s) / sum w_s.  grid (n_heads, M), block 256: 16 lanes x 8 channels cover a row, 16 split lanes
// run in parallel.  S <= 64 * SETS.
// What it costs is a launch, that trip and a serial chain of a few hundred instructions, so the chain is what counts: every
// wave finds maximum and weights by itself (a row's weights are in its own 16 lanes, read by row broadcasts), the four split lanes
// of a wave are folded in registers (fold_rows), and one barrier is left where weights and sums through LDS took three.  us
// per 16 layers, before / since: one token at 1,003 tokens 113.7 / 110.4, at 32,741 166.3 / 163.5, 8 rows at 12,037 tokens
// 221.5 / 216.2; 4 layers of one token at 262,100 (128 splits, two sets) 135.0 / 134.7.  Requests without a branch of their own (a
// split past the last asks for the last once more, weight 0), here and in the rows form below: 109.0 / 106.5, 158.4 / 156.3, 203.0 /
// 201.7; 32 rows at 3,000 257.7 / 254.5.  With four sets the compiler then asked for two to seven rows at a time, with waits in between,
// until it was held to one trip (all_requested; 16 layers of one KV head at 20,000 tokens 119.2 / 116.7, 8 layers at 100,000 82.9 / 81.4).  With
// one set it is one by itself; with two, two rows of eight are asked for behind the first answers, and held to one trip the kernel
// takes longer (two KV heads at 20,000 tokens 123.7 / 125.0).
// MS: a stream's share of the splits may exceed what is in flight at once (a loop over sets; 256 splits at most).
// ADAPT: rows of a prefill slice that the rows form below does not take (inverse rotation, or more than 32 splits); as many
// workgroups as the chip holds at once, each walks its share of the tokens, so that the choice of the splits is made 8
// times per CU and not once per row (1,024 rows at 9,000 tokens with the inverse rotation: 42.4 us with a workgroup per
// row, 37.9 so).
template <int SETS, bool MS, bool ADAPT>
__global__ void __launch_bounds__(256) combine_kernel(CombineHead head_args, CombineTail tail_args) {
  CombineArgs A = combine_args(head_args, tail_args);
  __shared__ __align__(16) float s_o[4][kD];
  __shared__ float s_w[kD];
  const int head = blockIdx.x, tid = threadIdx.x;
  int tok = blockIdx.y;
  if constexpr (ADAPT) {
    A.S = chunk_splits_used(*A.d_pos, A.tok0, A.M, A.n_kv, A.max_ctx, A.S, A.adapt);
    if (A.S == 1 && A.direct) return;
  }
  const int wave = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4, c8 = i * 8;
  do {
  size_t pair0 = (size_t)tok * A.S;
  if constexpr (MS) {
    const int2 P = A.plan[tok];
    pair0 = P.y > 0 ? (size_t)P.x : 0; A.S = P.y;  // a rejected row has no splits: its requests go to the first pair, its weights are 0
  }
  const size_t p0 = pair0 * A.n_heads + head;                  // split s lives at p0 + s * n_heads
  // Lane (g, i) of wave w takes channels 8 i .. 8 i + 7 of splits 64 j + 16 g + 4 w + k, k = 0 .. 3, and looks at the (m, l)
  // of split 64 j + 16 g + (i + 4 w) % 16: every wave finds the maximum and the sum of the weights by itself, and the weight
  // of its k-th split is the one lane k of its row of 16 holds.  No request needs another's answer.  A row of weight 0 may be one that no
  // workgroup wrote: it is zeroed before use.
  const int first = 16 * g + 4 * wave, look = 16 * g + ((i + 4 * wave) & 15), last = MS ? max(A.S - 1, 0) : A.S - 1;
  const uint16_t* src = A.pacc16 + p0 * kD + c8;
  const uint32_t stride = (uint32_t)A.n_heads * kD * 2;
  constexpr int LOOK = MS ? 4 : SETS;
  uint4 u[SETS][4];
  auto request = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SETS; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int sp = s0 + 64 * j + first + k;
        u[j][k] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(src) + (uint32_t)min(sp, last) * stride);
      }
  };
  constexpr bool HOLD = SETS == 4;                 // to one trip, see above
  float m[LOOK], wl[LOOK];
#pragma unroll
  for (int j = 0; j < LOOK; ++j) {
    const int sp = 64 * j + look;
    const uint32_t e = (uint32_t)min(sp, last) * A.n_heads;
    const float m1 = A.pm[p0 + e], l1 = A.pl[p0 + e];
    m[j] = HOLD || sp < A.S ? m1 : -1e30f; wl[j] = HOLD || sp < A.S ? l1 : 0.f;
  }
  if constexpr (HOLD) all_requested();
  request(0);
  if constexpr (HOLD) {
    all_requested();
#pragma unroll
    for (int j = 0; j < LOOK; ++j)
      if (64 * j + look >= A.S) { m[j] = -1e30f; wl[j] = 0.f; }
  }
  float M2 = m[0];
#pragma unroll
  for (int j = 1; j < LOOK; ++j) M2 = fmaxf(M2, m[j]);
  M2 = lane_rows(lane_row16(M2, LaneMax{}), LaneMax{});
  float L = 0.f;
#pragma unroll
  for (int j = 0; j < LOOK; ++j) {
    wl[j] = m[j] > -1e29f ? __builtin_amdgcn_exp2f(m[j] - M2) * wl[j] : 0.f;
    L += wl[j];
  }
  L = lane_rows(lane_row16(L, LaneAdd{}), LaneAdd{});
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add = [&](const uint4& row, float w) __attribute__((always_inline)) {
    const uint4 r = w != 0.f ? row : make_uint4(0, 0, 0, 0);
    const h8 v = __builtin_bit_cast(h8, r);
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] += w * (float)v[c];
  };
  auto add_set = [&](int j, float w) __attribute__((always_inline)) {
    add(u[j][0], lane_dpp<0x150>(w)); add(u[j][1], lane_dpp<0x151>(w)); add(u[j][2], lane_dpp<0x152>(w)); add(u[j][3], lane_dpp<0x153>(w));   // row_newbcast:k
  };
#pragma unroll
  for (int j = 0; j < SETS; ++j) add_set(j, wl[j]);
  if constexpr (MS) {
#pragma unroll 1
    for (int j = 1; 64 * j < A.S; ++j) {
      request(64 * j);
      add_set(0, j == 1 ? wl[1] : j == 2 ? wl[2] : wl[3]);
    }
  }
  // The four split lanes of a wave: each fold halves what a lane holds, channels 8 i + 4 (g / 2) + 2 (g % 2) are left
  *reinterpret_cast<float2*>(&s_o[wave][c8 + 4 * (g >> 1) + 2 * (g & 1)]) = fold_rows(acc);
  __syncthreads();
  float y = 0.f;                                   // stays for a row that saw no key (a rejected row of a multi-stream pass) and one without a softmax (scores that are not finite)
  if (tid < kD && L > 0.f) y = (s_o[0][tid] + s_o[1][tid] + s_o[2][tid] + s_o[3][tid]) * (1.f / L);
  if (A.unrot) {                                   // uniform over the grid
    // inverse signed Hadamard rotation over the row's 128 channels (threads 0..127 = two waves)
    y = wave_hadamard(y, tid);
    __syncthreads();
    if (tid < kD) s_w[tid] = y;
    __syncthreads();
    if (tid < kD) {
      const float b = s_w[tid ^ 64];
      y = (tid & 64) ? b - y : y + b;
      y = y * 0.0625f * channel_sign(tid);         // signs last on the way back (src/kvx_codec.cuh:28-32)
    }
  }
  if (tid < kD) A.out16[((size_t)tok * A.n_heads + head) * kD + tid] = A.out_bf16 ? f2bf_bits(y) : __half_as_ushort(__float2half_rn(y));
  if constexpr (ADAPT) __syncthreads();            // the next token reuses the LDS arrays
  } while (ADAPT && (tok += gridDim.y) < A.M);
}
// The combiner for wide passes (many rows, at most 32 splits, no un-rotation): one wave per (token, head) row, four
// waves per workgroup, no LDS and no barrier.  Lane = (split lane 0..3, 8 channels); a split lane takes splits sl, sl + 4,
// ... (at most 8), requests their rows together with the (m, l) pairs - one trip, to which all_requested holds the compiler: it had
// asked for l behind the answers (16 layers of 32 rows at 12,000 tokens 305.3 / 300.6 us, of 64 at 32,768 675.3 / 673.0, 8 layers of 1,000
// at 9,000 1,366.6 / 1,361.7) - and the four split lanes are summed by two cross-lane exchanges.  Same arithmetic as combine_kernel up to the order of the sums.
// ADAPT: rows of a prefill slice; 4 workgroups per CU, each walks its share - most slices on short contexts find nothing to do
// here and should not pay for dispatching thousands of workgroups to find out (16 layers of 1,500 rows on an empty cache 637 us, with
// 8 per CU 644).  A split lane asks for as many partials as there are splits for it, 1, 2, 4 or 8: eight whatever
// their number cost as much as the row's own (4 layers of 300 rows at 2,000 tokens, one KV head, 7 splits 89.8 / 87.2 us; with eight KV heads 100 rows
// there 101.5 / 98.3; 8 layers of 200 rows at 9,000, four heads, 364 / 355).  Several rows a step, so that
// eight pieces are in flight, are slower while waves have few steps (4 layers, four KV heads, 800 rows at 2,000 tokens in 3 splits, 1 / 8 rows
// a step, 221.6 / 231.0, 200 at 500 77.7 / 78.3) and faster where every wave has eight rows of a partial a lane each (4 layers of 2,048 rows at
// 3,000 tokens, 2 splits, 636 / 625, eight KV heads, 800 rows at 2,000 411.5 / 407).
template <bool ADAPT>
__global__ void __launch_bounds__(256) combine_rows_kernel(CombineHead head_args, CombineTail tail_args) {
  CombineArgs A = combine_args(head_args, tail_args);
  if constexpr (ADAPT) {
    A.S = chunk_splits_used(*A.d_pos, A.tok0, A.M, A.n_kv, A.max_ctx, A.S, A.adapt);
    if (A.S == 1 && A.direct) return;
  }
  const int lane = threadIdx.x & 63, sl = lane >> 4, c8 = (lane & 15) * 8, total = A.M * A.n_heads;
  const uint32_t stride = (uint32_t)A.n_heads * kD * 2;
  // RB rows a step, KN partials a split lane: row = tok * n_heads + head
  auto walk = [&](auto kn_tag, auto rb_tag) __attribute__((always_inline)) {
    constexpr int KN = decltype(kn_tag)::value, RB = decltype(rb_tag)::value;
    for (int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RB; row0 < total; row0 += ADAPT ? 4 * (int)gridDim.x * RB : total) {
      float pmv[RB], plv[RB];
      uint4 u[RB][KN];
      // lane t < S looks at split t; the maximum and every weight then come from cross-lane reads
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int row = min(row0 + r, total - 1);
        const size_t p0 = (size_t)(row / A.n_heads) * A.S * A.n_heads + row % A.n_heads;
        const uint32_t e = (uint32_t)min(lane, A.S - 1) * A.n_heads;
        pmv[r] = A.pm[p0 + e]; plv[r] = A.pl[p0 + e];
#pragma unroll
        for (int k = 0; k < KN; ++k)
          u[r][k] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(A.pacc16 + p0 * kD + c8) + (uint32_t)min(sl + 4 * k, A.S - 1) * stride);
      }
      all_requested();
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const float M2 = lane_rows(lane_row16(pmv[r], LaneMax{}), LaneMax{});
        const float wl = (lane < A.S && pmv[r] > -1e29f) ? exp2f(pmv[r] - M2) * plv[r] : 0.f;     // weight of split `lane`
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float wsum = 0.f;
#pragma unroll
        for (int k = 0; k < KN; ++k) {
          const float w = __shfl(wl, sl + 4 * k, 64);                        // < 32: a lane of this wave
          const uint4 x = w != 0.f ? u[r][k] : make_uint4(0, 0, 0, 0);        // a row of weight 0 may be one that no workgroup wrote
          const h8 v = __builtin_bit_cast(h8, x);
#pragma unroll
          for (int c = 0; c < 8; ++c) acc[c] += w * (float)v[c];
          wsum += w;
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c] = lane_rows(acc[c], LaneAdd{});
        wsum = lane_rows(wsum, LaneAdd{});
        if (sl == 0 && row0 + r < total) {
          const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
          float yv[8];
#pragma unroll
          for (int c = 0; c < 8; ++c) yv[c] = acc[c] * inv;
          *reinterpret_cast<uint4*>(A.out16 + (size_t)(row0 + r) * kD + c8) = pack_out8(yv, A.out_bf16);
        }
      }
    }
  };
  const std::integral_constant<int, 1> c1{};
  const std::integral_constant<int, 8> c8_rows{};
  if (ADAPT && A.S <= 4 && total >= 32 * (int)gridDim.x) walk(c1, c8_rows);
  else if (ADAPT && A.S <= 4) walk(c1, c1);
  else if (ADAPT && A.S <= 8) walk(std::integral_constant<int, 2>{}, c1);
  else if (ADAPT && A.S <= 16) walk(std::integral_constant<int, 4>{}, c1);
  else walk(std::integral_constant<int, 8>{}, c1);
}
void launch_combine(const CombineArgs& A, hipStream_t st) {
  if (A.plan) {                                    // a stream may hold any share of the splits (256 at most)
    hipLaunchKernelGGL((combine_kernel<1, true, false>), dim3(A.n_heads, A.M), dim3(256), 0, st, combine_head(A), combine_tail(A));
    return;
  }
  if (A.S <= 32 && !A.unrot && A.M >= 8) {
    const int wgs = (A.M * A.n_heads + 3) / 4;
    if (A.adapt) hipLaunchKernelGGL(combine_rows_kernel<true>, dim3(min(wgs, 1024)), dim3(256), 0, st, combine_head(A), combine_tail(A));
    else hipLaunchKernelGGL(combine_rows_kernel<false>, dim3(wgs), dim3(256), 0, st, combine_head(A), combine_tail(A));
    return;
  }
  if (A.adapt) {                                   // S <= kChunkMaxSplits
    static_assert(kChunkMaxSplits <= 64, "one set");
    hipLaunchKernelGGL((combine_kernel<1, false, true>), dim3(A.n_heads, min(A.M, max(1, 2048 / A.n_heads))), dim3(256), 0, st, combine_head(A), combine_tail(A));
    return;
  }
  if (A.S > 128) hipLaunchKernelGGL((combine_kernel<4, false, false>), dim3(A.n_heads, A.M), dim3(256), 0, st, combine_head(A), combine_tail(A));   // S <= 256
  else if (A.S > 64) hipLaunchKernelGGL((combine_kernel<2, false, false>), dim3(A.n_heads, A.M), dim3(256), 0, st, combine_head(A), combine_tail(A));
  else hipLaunchKernelGGL((combine_kernel<1, false, false>), dim3(A.n_heads, A.M), dim3(256), 0, st, combine_head(A), combine_tail(A));
}

}  // namespace yka
