// The reference's own KV rows on gfx950: head_dim 256, flat int4 with ONE fp32 scale per row, 4-bit fields MSB first in
// 32-bit words (src/kvq_fast.cuh:194-198,226-233; decode src/kvq_attn.cuh:33-37,53-54).  Quantize-on-append, the
// canonical image, split-KV attention for row tiles of 2 tokens x 6 heads, and the combiner.
//
// Page of one (page, kv head): 256 tokens, 67584 bytes
//   +0      K words  [256][32] uint32      +65536  K scales [256] fp32
//   +32768  V words  [256][32] uint32      +66560  V scales [256] fp32
// Attention follows the 128-channel narrow kernel (same MFMA 16x16x32 layouts: S^T = K Q^T leaves one query row per lane
// column, which is the B-operand layout of O^T += V^T P^T), with what one scale per row allows:
//   * the score of a key is (sum over 256 channels of q * code) * scale: 8 chained MFMAs and ONE multiply;
//   * V codes stay exact integers in the MFMA; the V scale of a key is folded into its probability (p * scale, rounded
//     to fp16 once), the softmax denominator uses the unscaled p.
// Nibble -> fp16: ((w >> s) & 0x000f000f) | 0x64006400 is (1024 + n) in both halves; minus 1032 gives n - 8.  Shift s
// selects elements 7 - s/4 (low half) and 3 - s/4 (high half) of the word, so a word yields its 8 codes in the order
// [7,3,6,2,5,1,4,0]; the query fragments are loaded in the same order.
#include "yka_internal.h"
#include "rot256_device.h"
#include "merge256_device.h"
#include "tb_store_device.h"
#include <hip/hip_fp16.h>

namespace yka {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kD2 = 256;
constexpr int kP2Kw = 0, kP2Vw = 32768, kP2Ks = 65536, kP2Vs = 66560;
constexpr uint32_t kMagic = 0x64006400u;
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t nib(uint32_t w, uint32_t magic) { return (w & 0x000f000fu) | (magic & ~0x000f000fu); }

// start of the (page, kv head) block of token t; t uniform over the wave (table entry through the scalar path)
__device__ __forceinline__ uint8_t* page256(const KvView& kv, int kvh, int t) {
  const int lp = t / kPageTok;
  int pp = lp;
  if (kv.table) pp = table_entry_scalar(kv.table, lp);
  return kv.base + (size_t)(pp * kv.n_kv + kvh) * kPage256Bytes;
}

// One row of 256 values (thread d holds channel d) -> 32 words + one fp32 scale at token `pos` of kv head `kvh`.  Called by
// all 256 threads of a workgroup (three barriers inside); red[4] and fld[256] are its LDS scratch.
__device__ __forceinline__ void quant_store_row256(const KvView& kv, int kvh, int pos, bool isv, float x, int d, float* red, uint8_t* fld) {
  float am = fabsf(x);
  am = lane_rows(lane_row16(am, LaneMax{}), LaneMax{});
  __syncthreads();                               // the scratch of a previous row is no longer read
  if ((d & 63) == 0) red[d >> 6] = am;
  __syncthreads();
  am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float s7 = __fdiv_rn(am, 7.f);
  if (s7 == 0.f) s7 = 1.f;
  float q = rintf(__fdiv_rn(x, s7));
  q = fminf(fmaxf(q, -7.f), 7.f);
  fld[d] = (uint8_t)((int)q + 8);
  __syncthreads();
  uint8_t* pg = page256(kv, kvh, pos);
  const int tp = pos % kPageTok;
  if (d < 32) {                                  // word d = fields 8d .. 8d+7, the first in the top nibble
    uint32_t w = 0u;
#pragma unroll
    for (int k = 0; k < 8; ++k) w |= (uint32_t)fld[8 * d + k] << (28 - 4 * k);
    reinterpret_cast<uint32_t*>(pg + (isv ? kP2Vw : kP2Kw))[tp * 32 + d] = w;
  }
  if (d == 0) reinterpret_cast<float*>(pg + (isv ? kP2Vs : kP2Ks))[tp] = s7;
}

// ---- quantize-on-append: grid (M, n_kv * 2), block 256 = one row, thread = channel ----
__global__ void __launch_bounds__(256) append256_kernel(AppendArgs A) {
  __shared__ float red[4];
  __shared__ float buf[256];
  __shared__ uint8_t fld[256];
  const int tok = blockIdx.x, kvh = blockIdx.y >> 1, isv = blockIdx.y & 1, d = threadIdx.x;
  int pos;
  if (A.rows.pos) {                                // multi-stream pass: the row's own container and position
    pos = A.rows.pos[tok];
    const int slot = A.rows.slot[tok];
    if (pos < 0 || pos >= A.kv.max_ctx || slot < 0 || slot >= A.rows.n_slots) return;
    A.kv = slot_view(A.kv, A.rows, slot);
  } else {
    pos = *A.d_pos + tok;
    if (pos < 0 || pos >= A.kv.max_ctx) return;
  }
  const size_t e = ((size_t)tok * A.kv.n_kv + kvh) * kD2 + d;
  float x = A.k32 ? (isv ? A.v32 : A.k32)[e] : row16_value((isv ? A.v16 : A.k16)[e], A.in_bf16);
  if (A.rot) x = rotate256(x, buf, false);
  quant_store_row256(A.kv, kvh, pos, isv, x, d, red, fld);
}

// ---- the step between the QKV projection and the cache for 256-channel heads, fused with quantize-on-append
//      (src/q35_kernels.cu:1030-1065 in the reference's own order of operations, with fp16 in the place of its bf16
//      roundings): the projected value is rounded to 16 bits first (:1030); per-head RMS normalisation (sum of squares:
//      butterfly inside each run of 32 channels, then the 8 run sums folded in sequence, :1051-1056), partial rotary
//      embedding with the rotate-half pairing, optional 256-point signed rotation; Q rows leave as fp16, K and V rows go
//      through the row quantizer as fp32 values; gate rows (if given) leave as the rounded projection (:1048).
//      grid (n_heads + 2 n_kv [+ n_heads gate rows], M), block 256 = one head row. ----
__device__ __forceinline__ float f16r256(float x) { asm volatile("" : "+v"(x)); return __half2float(__float2half_rn(x)); }
__global__ void __launch_bounds__(256) attn_post256_kernel(PostArgs A) {
  __shared__ float buf[256];
  __shared__ float red[8];
  __shared__ uint8_t fld[256];
  const int blk = blockIdx.x, tok = blockIdx.y, d = threadIdx.x;
  const int NH = A.n_heads, KVH = A.kv.n_kv;
  // as in attn_post_kernel: value and weight are requested with the position, the rotary factors as soon as it is known
  const bool gate = blk >= NH + 2 * KVH, isq = blk < NH, isk = !isq && blk < NH + KVH;
  const int head = gate ? blk - NH - 2 * KVH : isq ? blk : (isk ? blk - NH : blk - NH - KVH);
  const float* src = (gate ? A.xgate : isq ? A.xq : isk ? A.xk : A.xv) + ((size_t)tok * (gate || isq ? NH : KVH) + head) * kD2;
  const float raw = __hip_atomic_load(src + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  const uint16_t* weights = isq ? A.qn_w16 : A.kn_w16;
  const uint16_t wraw = isq || isk ? request16(weights + d) : (uint16_t)0;
  const int pos = *A.d_pos + tok;
  if (pos < 0 || pos >= A.kv.max_ctx || (A.rd > 0 && pos >= A.rope_rows)) return;   // rows outside the container are dropped
  if (gate) {                                      // gate rows: the projection rounded to the 16-bit type
    A.gate16[((size_t)tok * NH + head) * kD2 + d] = A.io_bf16 ? f2bf_bits(raw) : __half_as_ushort(__float2half_rn(raw));
    return;
  }
  const int hr = A.rd >> 1;
  float2 cs = make_float2(0.f, 0.f);
  if (d < A.rd && (isq || isk)) cs = reinterpret_cast<const float2*>(A.rope)[(size_t)pos * hr + (d < hr ? d : d - hr)];
  const float y = f16r256(raw);
  float out;
  if (isq || isk) {
    const float ss = lane_run32(__fmul_rn(y, y), [](float a, float b) { return __fadd_rn(a, b); });
    if ((d & 31) == 0) red[d >> 5] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) tot = __fadd_rn(tot, red[w]);
    // sqrtf, not __fsqrt_rn: only the former is correctly rounded on this target
    const float r = __fdiv_rn(1.f, sqrtf(__fadd_rn(__fdiv_rn(tot, 256.f), A.eps)));
    const float w = __half2float(__ushort_as_half(wraw));
    const float xn = f16r256(__fmul_rn(__fmul_rn(y, r), __fadd_rn(1.f, w)));
    out = xn;
    if (hr > 0) {
      buf[d] = xn;
      __syncthreads();
      if (d < A.rd) {
        const float partner = d < hr ? -buf[d + hr] : buf[d - hr];
        out = f16r256(__fadd_rn(f16r256(__fmul_rn(xn, cs.x)), f16r256(__fmul_rn(partner, cs.y))));
      }
    }
    if (A.rot) out = rotate256(out, buf, false);
  } else {
    out = A.rot ? rotate256(y, buf, false) : y;
  }
  if (isq) {
    asm volatile("" : "+v"(out));                  // the rotation's last multiply is rounded to fp32 before the fp16 rounding
    A.q16[((size_t)tok * NH + head) * kD2 + d] = A.io_bf16 ? f2bf_bits(out) : __half_as_ushort(__float2half_rn(out));
  } else if (A.k32_out) {
    (isk ? A.k32_out : A.v32_out)[((size_t)tok * KVH + head) * kD2 + d] = out;
  } else {
    quant_store_row256(A.kv, head, pos, !isk, out, d, red, fld);
  }
}

// ---- canonical image <-> pages: grid (n, n_kv), block 64: lanes 0..31 move K words, 32..63 V words ----
// rotated query rows: grid rows, block 256
__global__ void __launch_bounds__(256) rotate_q256_kernel(const float* x32, uint16_t* q16) {
  __shared__ float buf[256];
  const size_t e = (size_t)blockIdx.x * kD2 + threadIdx.x;
  q16[e] = __half_as_ushort(__float2half_rn(rotate256(x32[e], buf, false)));
}

template <bool IMPORT>
__global__ void __launch_bounds__(64) xfer256_kernel(KvView kv, int pos0, int n, uint32_t* kw, float* ks, uint32_t* vw, float* vs) {
  const int t = blockIdx.x, kvh = blockIdx.y, j = threadIdx.x & 31, isv = threadIdx.x >> 5;
  uint8_t* pg = page256(kv, kvh, pos0 + t);
  const int tp = (pos0 + t) % kPageTok;
  uint32_t* pw = reinterpret_cast<uint32_t*>(pg + (isv ? kP2Vw : kP2Kw)) + tp * 32 + j;
  float* ps = reinterpret_cast<float*>(pg + (isv ? kP2Vs : kP2Ks)) + tp;
  const size_t row = (size_t)kvh * n + t;
  uint32_t* cw = (isv ? vw : kw) + row * 32 + j;
  float* cs = (isv ? vs : ks) + row;
  if (IMPORT) { *pw = *cw; if (j == 0) *ps = *cs; }
  else { *cw = *pw; if (j == 0) *cs = *ps; }
}

struct Raw256 {        // what one lane holds of a 32-key tile
  uint4 kw[2][2];      // K words of key 16kt + (lane & 15): words 8g .. 8g+7 (g = lane >> 4) = channels 64g .. 64g+63
  f4 ksc[2], vsc[2];   // scales of the 4 keys whose scores this lane receives: keys 16kt + 4g + r
  uint32_t vw[2][8];   // V word (lane & 15) + 16 hh of token tau(g, e)
};
struct Offs256 { uint32_t kw, sc, vw; };

// The two halves of a tile are requested apart: each one tile ahead, as soon as the registers it lands in are free.
__device__ __forceinline__ void load_k256(const uint8_t* pg, int tp, const Offs256& L, Raw256& R) {
  const uint8_t* rows = pg + (uint32_t)tp * 128u;          // code rows of the tile (K and V planes)
  const uint8_t* sc = pg + (uint32_t)tp * 4u;              // scale entries of the tile
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    R.kw[kt][0] = *reinterpret_cast<const uint4*>(rows + kP2Kw + L.kw + 2048 * kt);
    R.kw[kt][1] = *reinterpret_cast<const uint4*>(rows + kP2Kw + L.kw + 2048 * kt + 16);
    R.ksc[kt] = *reinterpret_cast<const f4*>(sc + kP2Ks + L.sc + 64 * kt);
  }
}
__device__ __forceinline__ void load_v256(const uint8_t* pg, int tp, const Offs256& L, Raw256& R) {
  const uint8_t* rows = pg + (uint32_t)tp * 128u;
  const uint8_t* sc = pg + (uint32_t)tp * 4u;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) R.vsc[kt] = *reinterpret_cast<const f4*>(sc + kP2Vs + L.sc + 64 * kt);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
#pragma unroll
    for (int e = 0; e < 8; ++e)                             // token tau(g, e) = 16 (e >> 2) + 4 g + (e & 3)
      R.vw[hh][e] = *reinterpret_cast<const uint32_t*>(rows + kP2Vw + L.vw + (16 * (e >> 2) + (e & 3)) * 128 + 64 * hh);
}

}  // namespace

typedef uint32_t Attend256Head __attribute__((ext_vector_type(8)));   // positions, q16 (two words each), M, n_heads, slots (two words)
// grid (S, n_kv, ceil(M/TPT)), block 256 (4 waves; decode launches one workgroup per CU, streams and forced windows two).
// Workgroup = (split, kv head, TPT tokens x 6 heads):
// TPT = 2 for a single-stream pass; MS (multi-stream pass, reference: src/q35_atxpk_ms.cu:13-33): one token per row tile,
// which reads the container and the position its row map names.
// In front of the first score stand three trips to memory (kernel arguments, position, tile): the head brings what the first loads
// need with the wave, the query rows are asked for beside the position (stage_q256), the first tile behind their answers.  16 layers of one
// token at 32,745 tokens 252.1 -> 244.0 us, at 2,000 150.3 -> 149.2; two tokens at 5,000 177.5 -> 175.7; 4 layers at 100,000 114.0 -> 108.9.
template <bool MS>
__global__ void __launch_bounds__(256, 2) attend256_kernel(Attend256Head H, AttnArgs A) {
  A.q16 = head_ptr<const uint16_t>(H[2], H[3]); A.M = (int)H[4]; A.n_heads = (int)H[5];
  if (MS) { A.rows.pos = head_ptr<const int>(H[0], H[1]); A.rows.slot = head_ptr<const int>(H[6], H[7]); } else A.d_pos = head_ptr<const int>(H[0], H[1]);
  constexpr int TPT = MS ? 1 : 2;
  __shared__ float s_m[4][16], s_l[4][16];
  __shared__ __align__(16) float s_acc[4 * m256_wave<TPT * kG>()];
  __shared__ __align__(16) uint8_t s_q[m256_q_row(TPT * kG)];
  int split = blockIdx.x, rt = blockIdx.z;
  const int kvh = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  // 16 bytes of the query rows (32 threads a row), asked for in front of the position where that does not decide which they are
  uint4 qraw[TPT];
  auto request_q = [&](int t0, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < TPT; ++u) {
      const int j = min((int)(threadIdx.x >> 5) + 8 * u, n * kG - 1);          // thread 256 u + t: a row past the last repeats it
      qraw[u] = *reinterpret_cast<const uint4*>(A.q16 + ((size_t)(t0 + j / kG) * A.n_heads + kvh * kG + j % kG) * kD2 + 8 * (threadIdx.x & 31));
    }
  };
  if constexpr (!MS) request_q(TPT * rt, min(TPT, A.M - TPT * rt));
  // channel threadIdx.x of the rows a single-stream pass may have to store (without a branch, at whose end the compiler would
  // wait for what was asked for in it: a pass that stores none asks for query rows, which are more)
  uint16_t fresh_k[2], fresh_v[2];
  if constexpr (!MS) {
    const uint16_t* const k16 = A.k16 ? A.k16 + (size_t)A.tok0 * A.kv.n_kv * kD2 : A.q16;
    const uint16_t* const v16 = A.k16 ? A.v16 + (size_t)A.tok0 * A.kv.n_kv * kD2 : A.q16;
    const size_t e = (size_t)kvh * kD2 + threadIdx.x, e1 = e + (A.M > 1 ? (size_t)A.kv.n_kv * kD2 : 0);
    fresh_k[0] = request16(k16 + e); fresh_v[0] = request16(v16 + e);
    fresh_k[1] = request16(k16 + e1); fresh_v[1] = request16(v16 + e1);
  }
  int pos, slot = 0; bool row_ok = true;
  MsShare share{};
  if (MS) {
    if (A.adapt) {
      const int b = split + A.S * rt;
      share = ms_share(A.rows, A.M, A.kv.max_ctx, A.S * A.M, 0, b, A.plan, b == 0 && kvh == 0 && wave == 0);
      if (share.row < 0) return;
      split = share.split; rt = share.row; pos = share.pos; slot = share.slot;
    } else { pos = A.rows.pos[rt]; slot = A.rows.slot[rt]; }
    row_ok = pos >= 0 && pos < A.kv.max_ctx && slot >= 0 && slot < A.rows.n_slots;   // a bad row reads nothing and yields zeros
    A.kv = slot_view(A.kv, A.rows, row_ok ? slot : 0);
  } else {
    pos = *A.d_pos;
  }
  const int tl = TPT * rt + i / kG;
  const bool vrow = i < TPT * kG && tl < A.M && row_ok;
  if constexpr (MS) request_q(min(rt, A.M - 1), 1);
  int dep = A.tok0 + tl;
  if (!MS && A.depth) {                            // uniform over the grid
    dep = A.depth[min(dep, A.tok0 + A.M - 1)];
    asm volatile("" : "+v"(dep));                  // answered here: behind the branch a pass without depths would wait for its query
  }
  const int len = vrow ? min(pos + (MS ? 0 : dep) + 1, A.kv.max_ctx) : 0;
  int maxlen = len, minlen = vrow ? len : 0x7fffffff;
  maxlen = lane_row16(maxlen, LaneMax{}); minlen = lane_row16(minlen, LaneMin{});
  maxlen = __builtin_amdgcn_readfirstlane(maxlen); minlen = __builtin_amdgcn_readfirstlane(minlen);
  // as many of the launched splits as the length found on the device justifies (two 32-key tiles per workgroup at
  // least); the others leave the "no keys" marker, whose rows the combiner does not read
  const int ntiles = (maxlen + 31) >> 5;
  const int s_used = MS && A.adapt ? share.n : min(A.S, max(1, ntiles >> 1));
  // partials of (token tj, split) start at pair * n_heads
  auto pair_of = [&](int tj) __attribute__((always_inline)) { return MS && A.adapt ? share.base + split : (size_t)tj * A.S + split; };
  if (split >= s_used) {
    const int j = threadIdx.x, tj = TPT * rt + j / kG;
    if (j < TPT * kG && tj < A.M) {
      const size_t p = pair_of(tj) * A.n_heads + kvh * kG + j % kG;
      A.pm[p] = -1e30f; A.pl[p] = 0.f;
    }
    return;
  }
  const int tps = (ntiles + s_used - 1) / s_used;
  const int tile0 = split * tps, tile1 = min(ntiles, tile0 + tps);

  // ---- fused quantize-on-append (rows of at most 2 tokens, one row tile): a row of this pass is written by the one
  //      workgroup whose tile range holds it - the only workgroup of this kv head that reads it in this launch; writer
  //      and readers are waves of one CU and one write-through L1, so workgroup-scope fences order the stores ----
  if (MS && A.k16 && row_ok) {
    __shared__ float a_red[4];
    __shared__ uint8_t a_fld[256];
    int lane_pos;
    uint64_t todo = ms_new_rows(A.rows, A.M, slot, pos, tile0, tile1, lane_pos);
    if (todo) {                        // uniform over the workgroup
      for (; todo; todo &= todo - 1) {
        const int t = __builtin_ctzll(todo), r = __builtin_amdgcn_readlane(lane_pos, t);
        const size_t e = ((size_t)t * A.kv.n_kv + kvh) * kD2 + threadIdx.x;
        quant_store_row256(A.kv, kvh, r, false, row16_value(A.k16[e], A.in_bf16), threadIdx.x, a_red, a_fld);
        quant_store_row256(A.kv, kvh, r, true, row16_value(A.v16[e], A.in_bf16), threadIdx.x, a_red, a_fld);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  }
  if (!MS && A.k16) {
    __shared__ float a_red[4];
    __shared__ uint8_t a_fld[256];
    bool mine = false;
#pragma unroll
    for (int t = 0; t < 2; ++t) {              // a fused pass has at most two rows
      if (t >= A.M) break;
      const int r = pos + A.tok0 + t;
      // A row no query row of this launch can see (a depth table may say so) lies past the last tile when it opens a new
      // one: nobody reads it now, the last workgroup in use stores it.  All conditions are uniform over the workgroup.
      const bool held = (r >> 5) >= tile0 && (r >> 5) < tile1, unseen = (r >> 5) >= ntiles && split == s_used - 1;
      if (r < 0 || r >= A.kv.max_ctx || !(held || unseen)) continue;
      mine = true;
      quant_store_row256(A.kv, kvh, r, false, row16_value(fresh_k[t], A.in_bf16), threadIdx.x, a_red, a_fld);
      quant_store_row256(A.kv, kvh, r, true, row16_value(fresh_v[t], A.in_bf16), threadIdx.x, a_red, a_fld);
    }
    if (mine) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  }

  const float sc_log2 = kLog2e * 0.0625f;          // log2(e) / sqrt(256)
  const h2 c1032 = {(_Float16)1032.f, (_Float16)1032.f};
  uint32_t magic = kMagic;
  asm volatile("" : "+v"(magic));
  const Offs256 offs{(uint32_t)i * 128u + 32u * g, 16u * g, 512u * g + 4u * i};

  float m_run = -1e30f, l_run = 0.f;
  f4 o[16];
#pragma unroll
  for (int b = 0; b < 16; ++b) o[b] = f4{0.f, 0.f, 0.f, 0.f};

  // K words of the wave's next tile are requested behind the scores of this one, V words behind its PV product: no second
  // register set, and every request has half a tile of work to hide under.  Past the end K is the last tile once more (an
  // unconditional request: the compiler then knows how many loads are in flight at each wait).
  Raw256 cur;
  h8 qf[8];
  if (tile0 < tile1) {                             // uniform over the workgroup; a wave without a tile asks for the last one: the compiler
                                                   // then knows how many loads are younger than the query's
    const int t0 = min(tile0 + wave, tile1 - 1) << 5;
    const uint8_t* pg = page256(A.kv, kvh, t0);
    load_k256(pg, t0 % kPageTok, offs, cur);
    load_v256(pg, t0 % kPageTok, offs, cur);
    // Q fragments: k-step t of 8, lane (row i, group g), element e <-> channel 64g + 8t + [7,3,6,2,5,1,4,0][e], through LDS
    stage_q256<TPT * kG, false>(qraw, A.in_bf16, s_q, qf, i, g);
    for (int T = tile0 + wave; T < tile1; T += 4) {
      const int t0 = T << 5;
      const bool need_mask = t0 + 32 > minlen;
      // ---- scores: per 16-key tile 8 chained MFMAs (one per word of the lane), then one multiply by the key's scale ----
      float s[8];
  #pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const uint32_t w[8] = {cur.kw[kt][0].x, cur.kw[kt][0].y, cur.kw[kt][0].z, cur.kw[kt][0].w,
                               cur.kw[kt][1].x, cur.kw[kt][1].y, cur.kw[kt][1].z, cur.kw[kt][1].w};
        f4 part = f4{0.f, 0.f, 0.f, 0.f};
  #pragma unroll
        for (int t = 0; t < 8; ++t) {
          const h2 p0 = as_h2(nib(w[t], magic)) - c1032, p1 = as_h2(nib(w[t] >> 4, magic)) - c1032;
          const h2 p2 = as_h2(nib(w[t] >> 8, magic)) - c1032, p3 = as_h2(nib(w[t] >> 12, magic)) - c1032;
          const h8 kf = h8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
          part = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[t], part, 0, 0, 0);
        }
  #pragma unroll
        for (int r = 0; r < 4; ++r) s[4 * kt + r] = part[r] * cur.ksc[kt][r];      // key t0 + 16kt + 4g + r against row i
      }
      const int tn = min(T + 4, tile1 - 1) << 5;
      const uint8_t* const pgn = page256(A.kv, kvh, tn);
      load_k256(pgn, tn % kPageTok, offs, cur);
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
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      const bool first = m_run < -1e29f;
      m_run = m_new;
      if (__any(alpha != 1.f && !first)) {
        l_run *= alpha;
  #pragma unroll
        for (int b = 0; b < 16; ++b) { o[b][0] *= alpha; o[b][1] *= alpha; o[b][2] *= alpha; o[b][3] *= alpha; }
      }
      h8 pf;
  #pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], sc_log2, -m_new));
        l_run += p;
        pf[e] = (_Float16)(p * cur.vsc[e >> 2][e & 3]);       // the V scale of the key rides on its probability
      }
      // ---- O^T += V^T P^T: word (lane & 15) + 16 hh of 8 tokens; byte bb of those words holds elements 7-2bb (low
      //      nibble) and 6-2bb (high nibble): accumulator hh*8 + element covers channels 8 * word + element ----
  #pragma unroll
      for (int hh = 0; hh < 2; ++hh)
  #pragma unroll
        for (int bb = 0; bb < 4; ++bb) {
          h2 lo[4], hi[4];
  #pragma unroll
          for (int pe = 0; pe < 4; ++pe) {
            const uint32_t x = __builtin_amdgcn_perm(cur.vw[hh][2 * pe + 1], cur.vw[hh][2 * pe], 0x0c040c00u + bb * 0x00010001u);
            lo[pe] = as_h2(nib(x, magic)) - c1032;
            hi[pe] = as_h2(nib(x >> 4, magic)) - c1032;
          }
          const h8 vlo = h8{lo[0][0], lo[0][1], lo[1][0], lo[1][1], lo[2][0], lo[2][1], lo[3][0], lo[3][1]};
          const h8 vhi = h8{hi[0][0], hi[0][1], hi[1][0], hi[1][1], hi[2][0], hi[2][1], hi[3][0], hi[3][1]};
          o[hh * 8 + 7 - 2 * bb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vlo, pf, o[hh * 8 + 7 - 2 * bb], 0, 0, 0);
          o[hh * 8 + 6 - 2 * bb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vhi, pf, o[hh * 8 + 6 - 2 * bb], 0, 0, 0);
        }
      load_v256(pgn, tn % kPageTok, offs, cur);
    }
  }
  merge_waves256<TPT * kG>(o, m_run, l_run, wave, min(TPT, A.M - TPT * rt) * kG, kvh, A.n_heads, 1.f, nullptr, s_m, s_l, s_acc, A.pm, A.pl, A.pacc16,
                           [&](int j) __attribute__((always_inline)) { return pair_of(TPT * rt + j / kG); });
}

// combiner (src/attention_kv4q.cu:325-332) for 256-channel rows: grid (n_heads, M), block 256 = 8 split lanes x 32 channel
// lanes of 8 channels; the split lanes run in parallel.  S <= 8 * K * SETS <= 256: K = 8 covers the 64 splits of decode (two sets
// 128, four 256), K = 4 covers 32 and keeps the register count low where thousands of workgroups run (wide windows).
// MS: a stream's share of the splits may exceed one set (a loop over sets; 256 at most).
// The chain behind the one trip to memory counts, as in the combiner of 128 channels: weights without LDS where a launch
// knows how many splits there are, the split lanes of a wave folded in registers, multiply-adds that take the fp16 value as it
// is.  us per 16 layers, before / since: 24 rows at 9,001 tokens 351.1 / 342.6, one token at 20,011 262.8 / 261.8, 5-bit
// rows: one token at 16,001 282.5 / 277.4, 16 at 16,384 682.1 / 674.3.  Then every request without a branch (past the last
// split it is the last one once more: a branch a request was 8 to 12 changes of the lane mask and jumps) and the requests of the new
// keys in front, whose answers take two more barriers: one token at 20,011 246.2 / 241.0, at 2,000 150.3 / 145.2, 24 rows at 9,001
// 329.0 / 326.3; 5-bit rows, one token at 16,001 266.0 / 256.4 (259.5 with the rows of the partials in front of what is picked
// from), at 300 201 / 192, two at 3,000 212.5 / 204.3, 16 at 16,384 670 / 667.3.  With two sets the compiler then spread the requests over
// several trips until it was held to one (all_requested; two KV heads, one token at 20,000 164.2 / 162.3).  One set with K = 4 is one trip by
// itself; with K = 8 two rows of eight are asked for behind the first answers, which measures the same, and four sets take longer in one
// trip than in the compiler's several (one KV head at 20,000 171.0 / 173.1).
// KB != 0: partials of launch_tb_encode_attend, which leave out the rows of the pass; token t also sees the keys *d_pos +
// u, u <= t, which join the sum as splits of one key each, in fp32 (thread = channel; N names the rows).  The searches have
// left what the rows may be coded with: wave 2 u + v of a workgroup picks the code of the K (v = 0) or V row of token u,
// and the workgroups of a kv head's first query head store them.  Everything that takes is requested with the partials.  5
// bits at 16,001 tokens, 16 layers: 356 us with a launch between that stored the rows and their values read back here, 312
// us so.
template <int KB> struct NewKeyArgs { TbAttnArgs N; TbJobs J; };
template <> struct NewKeyArgs<0> {};
template <int K, int SETS, bool MS, int KB>
__global__ void __launch_bounds__(256) combine256_kernel(CombineArgs A, NewKeyArgs<KB> X) {
  __shared__ __align__(16) float s_o[4][kD2];
  __shared__ float s_w[256];
  __shared__ float s_max[4], s_sum[4];
  const int head = blockIdx.x, tok = blockIdx.y, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, half = lane >> 5, c8 = (lane & 31) * 8;
  // what the new keys take is asked for first: it has the longer way to go (KB != 0)
  JobRequest job; uint32_t tk = 0, tv = 0; uint16_t q16 = 0; float mu = 0.f, gk = 0.f, gv = 0.f;
  if constexpr (KB != 0) {
    const TbAttnArgs& N = X.N;
    const int kvh = head / kG, gK = (N.layer * N.n_kv + kvh) * 2, gV = gK + 1;
    job = request_job(X.J, (2 * min(wave >> 1, tok) + (wave & 1)) * N.n_kv + kvh, lane);
    // entry i of a pair table ends with the value of state i & 255
    tk = N.pairs[((size_t)gK << (8 + KB)) + tid]; tv = N.pairs[((size_t)gV << (8 + KB)) + tid];
    q16 = N.q16[((size_t)tok * A.n_heads + head) * kD2 + tid];
    if (N.mu) mu = N.mu[(size_t)gV * 256 + tid];
    gk = N.gfac[gK]; gv = N.gfac[gV];
  }
  size_t pair0 = (size_t)tok * A.S;
  if constexpr (MS) {
    const int2 P = A.plan[tok];
    pair0 = P.y > 0 ? (size_t)P.x : 0; A.S = P.y;  // a rejected row has no splits: its requests go to the first pair, its weights are 0
  }
  else if (A.s_short) A.S = splits_at(A.S, A.s_short, *A.d_pos);        // the partials keep the distance of the launched splits
  const size_t p0 = pair0 * A.n_heads + head;
  // Half h of wave w takes splits 8 K j + 4 K h + K w + k, k < K, of set j, 8 channels a lane.  A stream may hold any number of
  // sets: its weights go through LDS, thread t looking at split t.  Otherwise both rows of 16 lanes of a half look at the
  // (m, l) of the half's 4 K splits, the wave's own first: every wave finds the maximum and the sum of the weights by itself
  // and has the weight of its k-th split in lane k of either row.  No request needs another's answer.  A row of weight 0 may be one that
  // no workgroup wrote: it is zeroed before use.
  const int first = 4 * K * half + K * wave, last = MS ? max(A.S - 1, 0) : A.S - 1;    // a split past the last asks for the last once more
  const uint16_t* src = A.pacc16 + p0 * kD2 + c8;
  const uint32_t stride = (uint32_t)A.n_heads * kD2 * 2;
  uint4 u[SETS][K];
  auto request = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SETS; ++j)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int sp = s0 + 8 * K * j + first + k;
        u[j][k] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(src) + (uint32_t)min(sp, last) * stride);
      }
  };
  constexpr int LOOK = MS ? 1 : SETS * K / 4;
  constexpr bool HOLD = KB == 0 && SETS == 2;      // to one trip, see above
  float pmv[LOOK], plv[LOOK];
  auto split_of = [&](int n) __attribute__((always_inline)) {
    return MS ? tid : 8 * K * (n / (K / 4)) + 4 * K * half + ((16 * (n % (K / 4)) + (lane & 15) + K * wave) & (4 * K - 1));
  };
#pragma unroll
  for (int n = 0; n < LOOK; ++n) {
    const int sp = split_of(n);
    const uint32_t e = (uint32_t)min(sp, last) * A.n_heads;
    const float m1 = A.pm[p0 + e], l1 = A.pl[p0 + e];
    pmv[n] = HOLD || sp < A.S ? m1 : -1e30f; plv[n] = HOLD || sp < A.S ? l1 : 0.f;
  }
  if constexpr (HOLD) all_requested();
  request(0);
  if constexpr (HOLD) {
    all_requested();
#pragma unroll
    for (int n = 0; n < LOOK; ++n)
      if (split_of(n) >= A.S) { pmv[n] = -1e30f; plv[n] = 0.f; }
  }
  float new_s[2] = {-1e30f, -1e30f}, new_v[2] = {0.f, 0.f};       // score in log2 units and V value (channel tid) of the new keys
  bool seen[2] = {false, false};               // uniform over the workgroup
  float ksc[2] = {0.f, 0.f};
  float kfac = 0.f;
  __shared__ float s_dot[2][4];
  if constexpr (KB != 0) {
    __shared__ float s_tab[2][256];              // K and V table of the kv head
    __shared__ uint32_t s_code[4][64];
    __shared__ float s_scale[4];
    const TbAttnArgs& N = X.N;
    const int kvh = head / kG, u_w = wave >> 1;
    const int pos = *N.d_pos;
    const float q = row16_value(q16, N.in_bf16);
    uint32_t states; float scale;
    pick_job(X.J, lane, job, states, scale);
    if (u_w <= tok) {                            // uniform over the wave
      s_code[wave][lane] = states;
      if (lane == 0) s_scale[wave] = scale;
      const int r = pos + u_w;
      if (tok == A.M - 1 && head % kG == 0 && r >= 0 && r < N.max_ctx) {
        const size_t row = (size_t)kvh * N.max_ctx + r;
        store_coded_row<KB>(const_cast<uint8_t*>((wave & 1) ? N.vpay : N.kpay) + row * N.stride, lane, states);
        if (lane == 0) const_cast<float*>((wave & 1) ? N.vscl : N.kscl)[row] = scale;
      }
    }
    s_tab[0][tid] = __half2float(__ushort_as_half((uint16_t)(tk >> 16)));
    s_tab[1][tid] = __half2float(__ushort_as_half((uint16_t)(tv >> 16)));
    __syncthreads();
    float dot[2] = {0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = pos + u;
      seen[u] = u <= tok && r >= 0 && r < N.max_ctx;
      if (!seen[u]) continue;
      ksc[u] = s_scale[2 * u];
      kfac = kLog2e * 0.0625f * gk;
      dot[u] = q * s_tab[0][reinterpret_cast<const uint8_t*>(s_code[2 * u])[tid]];
      new_v[u] = s_tab[1][reinterpret_cast<const uint8_t*>(s_code[2 * u + 1])[tid]] * s_scale[2 * u + 1] * gv + mu;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      dot[u] = lane_run32(lane_op32(dot[u], LaneAdd{}), LaneAdd{});
      if ((tid & 63) == 0) s_dot[u][tid >> 6] = dot[u];
    }
  }
  float M2 = pmv[0];
#pragma unroll
  for (int n = 1; n < LOOK; ++n) M2 = fmaxf(M2, pmv[n]);
  M2 = lane_rows(lane_row16(M2, LaneMax{}), LaneMax{});
  if (MS && lane == 0) s_max[wave] = M2;
  if constexpr (MS || KB != 0) __syncthreads();
  if constexpr (MS) M2 = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
  if constexpr (KB != 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (seen[u]) new_s[u] = (s_dot[u][0] + s_dot[u][1] + s_dot[u][2] + s_dot[u][3]) * ksc[u] * kfac;
    M2 = fmaxf(M2, fmaxf(new_s[0], new_s[1]));
  }
  float L = 0.f;
#pragma unroll
  for (int n = 0; n < LOOK; ++n) {
    plv[n] = pmv[n] > -1e29f ? __builtin_amdgcn_exp2f(pmv[n] - M2) * plv[n] : 0.f;
    L += plv[n];
  }
  L = lane_op32(lane_row16(L, LaneAdd{}), LaneAdd{});          // the rows of a half hold the same splits
  if constexpr (MS) {
    L = lane_op16(L, LaneAdd{});                               // here every lane has looked at another split
    s_w[tid] = plv[0];
    if (lane == 0) s_sum[wave] = L;
    __syncthreads();
    L = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
  }
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add = [&](const uint4& row, float w) __attribute__((always_inline)) {
    const uint4 r = w != 0.f ? row : make_uint4(0, 0, 0, 0);
    const h8 v = __builtin_bit_cast(h8, r);
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = __builtin_fmaf(w, (float)v[c], acc[c]);   // this file is compiled without contraction
  };
  if constexpr (MS) {
    for (int s0 = 0;;) {                           // one set, except for a stream with more than 8 K splits
#pragma unroll
      for (int k = 0; k < K; ++k) add(u[0][k], s0 + first + k < A.S ? s_w[s0 + first + k] : 0.f);
      s0 += 8 * K;
      if (s0 >= A.S) break;
      request(s0);
    }
  } else {
#pragma unroll
    for (int j = 0; j < SETS; ++j) {
      const float w = plv[j * (K / 4)];
      add(u[j][0], lane_dpp<0x150>(w)); add(u[j][1], lane_dpp<0x151>(w)); add(u[j][2], lane_dpp<0x152>(w)); add(u[j][3], lane_dpp<0x153>(w));   // row_newbcast:k
      if constexpr (K == 8) { add(u[j][4], lane_dpp<0x154>(w)); add(u[j][5], lane_dpp<0x155>(w)); add(u[j][6], lane_dpp<0x156>(w)); add(u[j][7], lane_dpp<0x157>(w)); }
    }
  }
  // the two split lanes of a wave: the fold leaves channels 8 i + 4 h .. + 3 in lane i of half h
  *reinterpret_cast<float4*>(&s_o[wave][c8 + 4 * half]) = fold_halves(acc);
  __syncthreads();
  float o = s_o[0][tid] + s_o[1][tid] + s_o[2][tid] + s_o[3][tid];
  if constexpr (KB != 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float w = seen[u] ? exp2f(new_s[u] - M2) : 0.f;        // a score that is NaN ends in L: no softmax, zeros below
      o += w * new_v[u]; L += w;
    }
  }
  float y = L > 0.f ? __fdiv_rn(o, L) : 0.f;
  if (A.unrot) y = rotate256(y, s_w, true);        // inverse of the rotation of the V rows (src/q35_kernels.cu:1421); s_w is free again
  A.out16[((size_t)tok * A.n_heads + head) * kD2 + tid] = A.out_bf16 ? f2bf_bits(y) : __half_as_ushort(__float2half_rn(y));
}

void launch_attn_post256(const PostArgs& A, hipStream_t st) {
  hipLaunchKernelGGL(attn_post256_kernel, dim3(A.n_heads + 2 * A.kv.n_kv + (A.gate16 ? A.n_heads : 0), A.M), dim3(256), 0, st, A);
}
void launch_append256(const AppendArgs& A, hipStream_t st) {
  hipLaunchKernelGGL(append256_kernel, dim3(A.M, A.kv.n_kv * 2), dim3(256), 0, st, A);
}
void launch_rotate_q256(const float* x32, int rows, uint16_t* q16, hipStream_t st) {
  hipLaunchKernelGGL(rotate_q256_kernel, dim3(rows), dim3(256), 0, st, x32, q16);
}
void launch_attend256(const AttnArgs& A, hipStream_t st) {
  const uint64_t pos = (uint64_t)(uintptr_t)(A.rows.pos ? A.rows.pos : A.d_pos), q = (uint64_t)(uintptr_t)A.q16, slot = (uint64_t)(uintptr_t)A.rows.slot;
  const Attend256Head H{(uint32_t)pos, (uint32_t)(pos >> 32), (uint32_t)q, (uint32_t)(q >> 32), (uint32_t)A.M, (uint32_t)A.n_heads, (uint32_t)slot, (uint32_t)(slot >> 32)};
  if (A.rows.pos) hipLaunchKernelGGL(attend256_kernel<true>, dim3(A.S, A.kv.n_kv, A.M), dim3(256), 0, st, H, A);
  else hipLaunchKernelGGL(attend256_kernel<false>, dim3(A.S, A.kv.n_kv, (A.M + 1) / 2), dim3(256), 0, st, H, A);
}
void launch_combine256(const CombineArgs& A, hipStream_t st) {
  // Streams walk sets of 8 K splits, whatever share of them a stream holds (256 at most); other passes need S <= 8 * K * SETS.  5 streams
  // of up to 3,000 tokens, us a pass: 15.2 with K = 16 (and 198 registers), 12.4 with 4 and splits of 4 tiles.
  if (A.plan) {
    if (A.M < 4) hipLaunchKernelGGL((combine256_kernel<8, 1, true, 0>), dim3(A.n_heads, A.M), dim3(256), 0, st, A, NewKeyArgs<0>{});
    else hipLaunchKernelGGL((combine256_kernel<4, 1, true, 0>), dim3(A.n_heads, A.M), dim3(256), 0, st, A, NewKeyArgs<0>{});
    return;
  }
  if (A.S > 128) hipLaunchKernelGGL((combine256_kernel<8, 4, false, 0>), dim3(A.n_heads, A.M), dim3(256), 0, st, A, NewKeyArgs<0>{});
  else if (A.S > 64) hipLaunchKernelGGL((combine256_kernel<8, 2, false, 0>), dim3(A.n_heads, A.M), dim3(256), 0, st, A, NewKeyArgs<0>{});
  else if (A.S > 32) hipLaunchKernelGGL((combine256_kernel<8, 1, false, 0>), dim3(A.n_heads, A.M), dim3(256), 0, st, A, NewKeyArgs<0>{});
  else hipLaunchKernelGGL((combine256_kernel<4, 1, false, 0>), dim3(A.n_heads, A.M), dim3(256), 0, st, A, NewKeyArgs<0>{});
}
template <int KB>
static void launch_combine_new(const CombineArgs& A, const TbAttnArgs& N, const TbJobs& J, hipStream_t st) {
  const dim3 grid(A.n_heads, A.M);
  const NewKeyArgs<KB> X{N, J};
  if (A.S > 128) hipLaunchKernelGGL((combine256_kernel<8, 4, false, KB>), grid, dim3(256), 0, st, A, X);
  else if (A.S > 64) hipLaunchKernelGGL((combine256_kernel<8, 2, false, KB>), grid, dim3(256), 0, st, A, X);
  else hipLaunchKernelGGL((combine256_kernel<8, 1, false, KB>), grid, dim3(256), 0, st, A, X);
}
void launch_combine256_new(const CombineArgs& A, const TbAttnArgs& N, const TbJobs& J, int kb, hipStream_t st) {
  if (kb == 4) launch_combine_new<4>(A, N, J, st); else launch_combine_new<5>(A, N, J, st);
}
void launch_export_rows256(const KvView& kv, int pos0, int n, uint32_t* kw, float* ks, uint32_t* vw, float* vs, hipStream_t st) {
  hipLaunchKernelGGL(xfer256_kernel<false>, dim3(n, kv.n_kv), dim3(64), 0, st, kv, pos0, n, kw, ks, vw, vs);
}
void launch_import_rows256(const KvView& kv, int pos0, int n, const uint32_t* kw, const float* ks, const uint32_t* vw, const float* vs, hipStream_t st) {
  hipLaunchKernelGGL(xfer256_kernel<true>, dim3(n, kv.n_kv), dim3(64), 0, st, kv, pos0, n, const_cast<uint32_t*>(kw), const_cast<float*>(ks),
                     const_cast<uint32_t*>(vw), const_cast<float*>(vs));
}

}  // namespace yka
