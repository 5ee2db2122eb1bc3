// Quantize-on-append and the codec probes.  Compiled with -ffp-contract=off: the codec is bit-exact by contract,
// and the reference builds with --fmad=false (CMakeLists.txt:60-63).
// The quantizer itself lives in codec_device.h (shared with the fused decode kernel).
#include "codec_device.h"

namespace yka {

// grid (ceil(M / 16), n_kv * 2), block 256: blockIdx.y = kvh * 2 + (0: K, 1: V); 16 lanes per row, 16 consecutive rows of
// one head per workgroup, so that the code rows of a workgroup are one run of 1 KB and its V scales runs of 32 bytes.
// Rows land at *d_pos + tok (reference: q35_kernels.cu:1038,1064 write the pass's rows before attention reads them).
// Bound by latency and by the number of workgroups: with a workgroup per row (8 M of them, one byte stored per lane pair)
// 1,500 rows took 7.8 us, in this form 4.7.
// A16: both row tensors start on a 16-byte boundary; otherwise a lane reads its 8 channels one by one.
template <bool A16>
__global__ void __launch_bounds__(256) append_kernel(AppendArgs A) {
  const int tok = blockIdx.x * 16 + (threadIdx.x >> 4), kvh = blockIdx.y >> 1, isv = blockIdx.y & 1, c = threadIdx.x & 15;
  if (tok >= A.M) return;                          // all 16 lanes of a row agree on every exit
  const uint16_t* src = (isv ? A.v16 : A.k16) + ((size_t)tok * A.kv.n_kv + kvh) * kD + 8 * c;
  uint4 raw[1];
  if constexpr (A16) raw[0] = *reinterpret_cast<const uint4*>(src);
  else {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = src[2 * k] | ((uint32_t)src[2 * k + 1] << 16);
    raw[0] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  KvView kv = A.kv;
  int pos;
  if (A.rows.pos) {                                // multi-stream pass: the row's own container and position
    pos = A.rows.pos[tok];
    const int slot = A.rows.slot[tok];
    if (slot < 0 || slot >= A.rows.n_slots) return;
    kv = slot_view(kv, A.rows, slot);
  } else pos = *A.d_pos + tok;
  if (pos < 0 || pos >= kv.max_ctx) return;
  rows16_to_f16(raw, A.in_bf16);
  quant_store_chunk8(kv, kvh, pos, isv != 0, raw[0], c);
}
void launch_append(const AppendArgs& A, hipStream_t st) {
  const dim3 grid((A.M + 15) / 16, A.kv.n_kv * 2);
  if ((((uintptr_t)A.k16 | (uintptr_t)A.v16) & 15) == 0) hipLaunchKernelGGL(append_kernel<true>, grid, dim3(256), 0, st, A);
  else hipLaunchKernelGGL(append_kernel<false>, grid, dim3(256), 0, st, A);
}

// codec round trip: x16 [rows][128] -> codes [rows][64], scales [rows][4], y [rows][128] fp32
__global__ void __launch_bounds__(128) codec_probe_kernel(const uint16_t* x16, int rows, uint8_t* codes, uint16_t* scales, float* y) {
  const int row = blockIdx.x, d = threadIdx.x;
  if (row >= rows) return;
  const float x = h2f_bits(x16[(size_t)row * kD + d]);
  int code; uint16_t s16;
  quant_lane(x, code, s16);
  const int nb = __shfl_xor(code, 1, 64);
  if ((d & 1) == 0) codes[(size_t)row * (kD / 2) + (d >> 1)] = (uint8_t)((code & 15) | ((nb & 15) << 4));
  if ((d & 31) == 0) scales[(size_t)row * kNG + (d >> 5)] = s16;
  // decode: (nib - 8) * s, exact in fp32 (reference: src/kvq_attn.cuh:52-54)
  y[(size_t)row * kD + d] = __fmul_rn((float)(code - 8), h2f_bits(s16));
}
void launch_codec_probe(const uint16_t* x16, int rows, uint8_t* codes, uint16_t* scales, float* y, hipStream_t st) {
  hipLaunchKernelGGL(codec_probe_kernel, dim3(rows), dim3(128), 0, st, x16, rows, codes, scales, y);
}

// canonical image <-> physical pages.  grid (n, n_kv), block 64: lane j moves byte j of K and V codes; lanes 0..3 the scales.
template <bool IMPORT>
__global__ void __launch_bounds__(64) xfer_rows_kernel(KvView kv, int pos0, int n, uint8_t* kc, uint16_t* ks, uint8_t* vc, uint16_t* vs) {
  const int t = blockIdx.x, kvh = blockIdx.y, j = threadIdx.x;
  uint8_t* pg = kv_page(kv, kvh, pos0 + t);
  const int tp = (pos0 + t) % kPageTok;
  uint8_t* pk = pg + kPageKc + tp * 64 + k_code_byte(j);
  uint8_t* pv = pg + kPageVc + tp * 64 + j;
  uint16_t* pks = reinterpret_cast<uint16_t*>(pg + kPageKs) + tp * kNG + j;      // j < 4 only
  uint16_t* pvs = reinterpret_cast<uint16_t*>(pg + kPageVs) + j * kPageTok + tp; // j < 4 only
  const size_t row = (size_t)kvh * n + t;
  if (IMPORT) {
    *pk = kc[row * 64 + j]; *pv = vc[row * 64 + j];
    if (j < kNG) { *pks = ks[row * kNG + j]; *pvs = vs[row * kNG + j]; }
  } else {
    kc[row * 64 + j] = *pk; vc[row * 64 + j] = *pv;
    if (j < kNG) { ks[row * kNG + j] = *pks; vs[row * kNG + j] = *pvs; }
  }
}
void launch_export_rows(const KvView& kv, int pos0, int n, uint8_t* kc, uint16_t* ks, uint8_t* vc, uint16_t* vs, hipStream_t st) {
  hipLaunchKernelGGL(xfer_rows_kernel<false>, dim3(n, kv.n_kv), dim3(64), 0, st, kv, pos0, n, kc, ks, vc, vs);
}
void launch_import_rows(const KvView& kv, int pos0, int n, const uint8_t* kc, const uint16_t* ks, const uint8_t* vc, const uint16_t* vs, hipStream_t st) {
  hipLaunchKernelGGL(xfer_rows_kernel<true>, dim3(n, kv.n_kv), dim3(64), 0, st, kv, pos0, n,
                     const_cast<uint8_t*>(kc), const_cast<uint16_t*>(ks), const_cast<uint8_t*>(vc), const_cast<uint16_t*>(vs));
}

// decoder probe: k, v [n_kv][n][128] fp32 = (nib - 8) * scale
__global__ void __launch_bounds__(128) dequant_rows_kernel(KvView kv, int pos0, int n, float* k, float* v) {
  const int t = blockIdx.x, kvh = blockIdx.y, d = threadIdx.x;
  const uint8_t* pg = kv_page(kv, kvh, pos0 + t);
  const int tp = (pos0 + t) % kPageTok;
  const size_t o = ((size_t)kvh * n + t) * kD + d;
  const int kb = pg[kPageKc + tp * 64 + k_code_byte(d >> 1)], vb = pg[kPageVc + tp * 64 + (d >> 1)];
  const int kn = (d & 1) ? (kb >> 4) : (kb & 15), vn = (d & 1) ? (vb >> 4) : (vb & 15);
  k[o] = __fmul_rn((float)(kn - 8), h2f_bits(reinterpret_cast<const uint16_t*>(pg + kPageKs)[tp * kNG + (d >> 5)]));
  v[o] = __fmul_rn((float)(vn - 8), h2f_bits(reinterpret_cast<const uint16_t*>(pg + kPageVs)[(d >> 5) * kPageTok + tp]));
}
void launch_dequant_rows(const KvView& kv, int pos0, int n, float* k, float* v, hipStream_t st) {
  hipLaunchKernelGGL(dequant_rows_kernel, dim3(n, kv.n_kv), dim3(128), 0, st, kv, pos0, n, k, v);
}

__global__ void set_int_kernel(int* p, int v) { *p = v; }
__global__ void zero_ints_kernel(int* p, int n) { const int i = blockIdx.x * 256 + threadIdx.x; if (i < n) p[i] = 0; }
void launch_zero_ints(int* p, int n, hipStream_t st) { hipLaunchKernelGGL(zero_ints_kernel, dim3((n + 255) / 256), dim3(256), 0, st, p, n); }
void launch_set_int(int* p, int v, hipStream_t st) { hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, st, p, v); }

}  // namespace yka
