// Internal declarations shared by the translation units of libyka.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include "lanes_device.h"

namespace yka {

// ---- fixed shape of the path ----
constexpr int kD = 128;          // head_dim
constexpr int kG = 6;            // query heads per KV head
constexpr int kGroup = 32;       // channels per scale group
constexpr int kNG = kD / kGroup; // scale groups per row (4)
constexpr int kPageTok = 256;    // tokens per page
// ---- physical page of one (page, kv head): 256 tokens, 36864 bytes, four planes ----
//   +0      K codes  [256][64]  byte j of a row: channel 2j low nibble, 2j+1 high nibble, value q+8; the 16 dwords of a
//                                row are stored in the order physical 4g+m = logical 4m+g, so that the 16-byte chunk g
//                                holds channels {32m + 8g .. 32m + 8g + 7 : m = 0..3} - one dword of every scale group
//   +16384  V codes  [256][64]  plain channel order
//   +32768  K scales [256][4]   fp16, token major
//   +34816  V scales [4][256]   fp16, group major (4 consecutive tokens of one group are 8 contiguous bytes)
constexpr int kPageKc = 0, kPageVc = 16384, kPageKs = 32768, kPageVs = 34816, kPageBytes = 36864;
__host__ __device__ inline int k_phys_dword(int logical) { return 4 * (logical & 3) + (logical >> 2); }
constexpr int kPage256Bytes = 67584;   // page of the 256-channel row format (attend256.hip): 256 x (128 + 128) code bytes + 2 x 256 fp32 scales
constexpr int kMaxSlice = 64;    // rows per attention slice (kVerifyMax of the reference, engine35.hpp:157)

// One layer's container.  The page of token t of kv head h starts at
//   base + (p * n_kv + h) * 36864,   p = table ? table[t / 256] : t / 256
struct KvView {
  uint8_t* base;
  const int32_t* table;  // nullptr in contiguous mode
  int n_kv;
  int max_ctx;
};
__host__ __device__ inline size_t kv_page_bytes(int n_kv) { return (size_t)n_kv * kPageBytes; }

// Multi-stream passes (reference: Q35MsRows, src/q35.hpp:28-35): row t of the pass belongs to the stream whose container
// is slot[t] and sits at position pos[t] of it.  Containers are slot_bytes apart (page tables slot_pages entries apart),
// starting from the view the arguments carry.  pos == nullptr: single-stream pass.
struct RowMap { const int* pos = nullptr; const int* slot = nullptr; int n_slots = 0; size_t slot_bytes = 0; int slot_pages = 0; };
__device__ __forceinline__ KvView slot_view(KvView v, const RowMap& R, int slot) {
  v.base += (size_t)slot * R.slot_bytes;
  if (v.table) v.table += (size_t)slot * R.slot_pages;
  return v;
}

// k32 / v32 / rot: 256-channel rows only (attend256.hip) - fp32 source rows instead of fp16 ones, and the signed Hadamard
// rotation applied to every row before it is quantized (src/q35_kernels.cu:1036,1060 + launch_tb_requant)
struct AppendArgs { KvView kv; const uint16_t* k16; const uint16_t* v16; const int* d_pos; int M; RowMap rows;
                    const float* k32 = nullptr; const float* v32 = nullptr; int rot = 0;
                    int in_bf16 = 0; };   // k16 / v16 are bf16 rows

// partial results of the split-KV kernels (same roles as pm/pl/pacc of the reference, args.hpp:10):
//   pm, pl [rows_tok][S][n_heads] fp32; pacc16 [rows_tok][S][n_heads][128] fp16 = acc / l (normalised, so that fp16
//   costs nothing measurable: every split's row is a convex combination of V rows).  pm is in log2 units; empty
//   split: pm = -1e30, pl = 0, pacc16 = 0.
struct AttnArgs {
  KvView kv; const uint16_t* q16; const int* d_pos; const uint8_t* depth;
  int M;        // rows (tokens) of this slice
  int tok0;     // index of the slice's first row inside the pass (row t sees keys [0, *d_pos + depth(tok0+t) + 1))
  int n_heads;
  int S;        // splits
  int rows_per_block;  // wide kernels: query rows one workgroup owns (a multiple of 32, 256-channel rows of 16; at most 128)
  float* pm; float* pl; uint16_t* pacc16;
  // k16/v16 != nullptr: fused quantize-on-append - the workgroups whose tiles hold the new rows quantize and store them
  // before reading them.  Narrow kernel (M <= 2): rows [0, M) of the pass; wide kernel: k16/v16 point at row 0 of the
  // pass and the slice stores its own rows tok0 .. tok0 + M - 1.
  const uint16_t* k16; const uint16_t* v16;
  RowMap rows;  // narrow kernel only: multi-stream pass, one token per workgroup column, no depth table; k16 / v16 with at most 64 rows
  // narrow kernel only: tickets != nullptr folds the split combine into the launch - every workgroup of a (kv head, row
  // tile) column takes a ticket from tickets[kv head * gridDim.z + row tile] once its partials are out, and the one that
  // draws the last ticket merges the column's partials into out16 and puts the counter back to zero
  int* tickets = nullptr; uint16_t* out16 = nullptr; int out_bf16 = 0;
  int in_bf16 = 0;   // q16 / k16 / v16 are bf16 rows (rows16_to_f16)
  // wide kernel, slice of a prefill chunk (launch_attend_chunk): adapt != 0 (chunk_tile_cap) lets the device choose how many of the
  // S launched splits the slice uses (chunk_splits_used); out16 != nullptr: a slice that uses one writes its output rows itself
  // multi-stream pass: adapt != 0 shares the S * M workgroups of a kv head out by the streams' lengths (ms_share) and leaves the
  // shares in plan[M] for the combiner
  int adapt = 0;
  int2* plan = nullptr;
  int ms_short = 0;  // workgroups of a kv head a pass over short streams uses (0: all S * M)
};
// unrot != 0: the output row gets the inverse signed Hadamard rotation (7 butterfly stages, x 1/16, signs) before it is
// rounded to fp16 - the counterpart of rotating V rows on their way into the cache (src/q35_kernels.cu:1421)
struct CombineArgs { const float* pm; const float* pl; const uint16_t* pacc16; int S; int M; int n_heads; uint16_t* out16; int unrot;
                     int out_bf16 = 0;      // outputs leave as bf16 (rounded once from the fp32 result) instead of fp16
  // adapt != 0: partials of launch_attend_chunk - the splits in use follow from *d_pos as they did there, and with direct != 0 a
  // slice that used one split has written its output already
  int adapt = 0; int direct = 0; const int* d_pos = nullptr; int tok0 = 0; int n_kv = 0; int max_ctx = 0;
  const int2* plan = nullptr;   // partials of a multi-stream pass shared out by ms_share: first split and splits of every row
  int s_short = 0; };    // trellis decode: as in TbAttnArgs (d_pos is set then)
// Decode, its combiner and the trellis kernels of decode name what their first loads need as leading arguments of their own
// and are compiled with -amdgpu-kernarg-preload-count: those arrive in scalar registers with the wave, and the position
// (the combiner's partials) is asked for at once instead of 0.3 us later, behind the load of the argument block.  us per 16
// layers without / with: one token at 32,741 tokens 172.5 / 166.5, one 5-bit trellis row at 16,001 382 / 371, 8 rows at
// 12,037 (the combiner alone) 226 / 220, one token at 1,003 115.4 / 113.8, 16 streams 27.1 / 26.7 a pass.  The combiner
// of 256-channel rows takes its arguments as one block: split, it measured the same.
// In the int4 decode kernel and the combiners such a pointer travels as an integer, and the combiners' arguments are split
// into head and tail, not repeated: a pointer among a launch's arguments costs the host 0.2 us, and the 136 bytes of a
// repeated block 0.45 us more than these 96.  A call issued outside a graph is as long as the host takes; 16 layers of one
// token at 1,622 tokens, us: 177 without preloaded arguments, 192 with pointers and the block repeated, 185 with integers,
// 178 with the split.  The trellis kernels keep pointers and repeat what they preload: over such rows the device takes
// longer than the host on any context (one token at 600 tokens 13.8 us a layer against 11.8).
typedef uint32_t CombineHead __attribute__((ext_vector_type(8)));     // pm, pl, pacc16 (two words each), S, n_heads
struct CombineTail { uint16_t* out16; const int* d_pos; const int2* plan; int M, unrot, out_bf16, adapt, direct, tok0, n_kv, max_ctx, s_short; };
inline CombineHead combine_head(const CombineArgs& A) {
  const uint64_t pm = (uint64_t)(uintptr_t)A.pm, pl = (uint64_t)(uintptr_t)A.pl, acc = (uint64_t)(uintptr_t)A.pacc16;
  return CombineHead{(uint32_t)pm, (uint32_t)(pm >> 32), (uint32_t)pl, (uint32_t)(pl >> 32), (uint32_t)acc, (uint32_t)(acc >> 32), (uint32_t)A.S, (uint32_t)A.n_heads};
}
inline CombineTail combine_tail(const CombineArgs& A) {
  return CombineTail{A.out16, A.d_pos, A.plan, A.M, A.unrot, A.out_bf16, A.adapt, A.direct, A.tok0, A.n_kv, A.max_ctx, A.s_short};
}
// such an integer, or two words of a head, as a pointer into global memory; without the address space the loads behind it
// are flat ones
template <typename T> __device__ __forceinline__ T* head_ptr(uint64_t word) { return (T*)(__attribute__((address_space(1))) T*)word; }
template <typename T> __device__ __forceinline__ T* head_ptr(uint32_t lo, uint32_t hi) { return head_ptr<T>((uint64_t)lo | ((uint64_t)hi << 32)); }
__device__ __forceinline__ CombineArgs combine_args(CombineHead H, const CombineTail& T) {
  CombineArgs A{head_ptr<const float>(H[0], H[1]), head_ptr<const float>(H[2], H[3]), head_ptr<const uint16_t>(H[4], H[5]), (int)H[6], T.M, (int)H[7],
                T.out16, T.unrot, T.out_bf16, T.adapt, T.direct, T.d_pos, T.tok0, T.n_kv, T.max_ctx, T.plan, T.s_short};
  return A;
}
// The same for the mid and the wide kernel: head, sizes and tail together are AttnArgs without what only the other kernels use (the
// whole block with a repeated head cost the host 0.3 us more a launch: 8 rows at 2,000 tokens outside a graph 177.5 / 182.5 us per 16 layers).
// us per 16 layers without / with: 8 tree rows at 12,037 tokens 201.0 / 197.8, 64 rows at 32,768 686.7 / 681.7, 24 tree rows at 9,000
// 283.5 / 280.9, 40 rows at 2,000 outside a graph 236.1 / 233.7.
typedef uint32_t WindowHead __attribute__((ext_vector_type(8)));       // kv.base, kv.table, q16, d_pos (two words each)
typedef uint32_t WindowSizes __attribute__((ext_vector_type(4)));      // M | rows_per_block << 16, n_kv, S, max_ctx
struct WindowTail { const uint8_t* depth; float* pm; float* pl; uint16_t* pacc16; const uint16_t* k16; const uint16_t* v16; uint16_t* out16; int tok0, out_bf16, in_bf16, adapt; };
inline WindowHead window_head(const AttnArgs& A) {
  const uint64_t b = (uint64_t)(uintptr_t)A.kv.base, t = (uint64_t)(uintptr_t)A.kv.table, q = (uint64_t)(uintptr_t)A.q16, d = (uint64_t)(uintptr_t)A.d_pos;
  return WindowHead{(uint32_t)b, (uint32_t)(b >> 32), (uint32_t)t, (uint32_t)(t >> 32), (uint32_t)q, (uint32_t)(q >> 32), (uint32_t)d, (uint32_t)(d >> 32)};
}
inline WindowSizes window_sizes(const AttnArgs& A) {
  return WindowSizes{(uint32_t)A.M | (uint32_t)A.rows_per_block << 16, (uint32_t)A.kv.n_kv, (uint32_t)A.S, (uint32_t)A.kv.max_ctx};
}
inline WindowTail window_tail(const AttnArgs& A) {
  return WindowTail{A.depth, A.pm, A.pl, A.pacc16, A.k16, A.v16, A.out16, A.tok0, A.out_bf16, A.in_bf16, A.adapt};
}
__device__ __forceinline__ AttnArgs window_args(WindowHead H, WindowSizes N, const WindowTail& T) {
  AttnArgs A{KvView{head_ptr<uint8_t>(H[0], H[1]), head_ptr<const int32_t>(H[2], H[3]), (int)N[1], (int)N[3]},
             head_ptr<const uint16_t>(H[4], H[5]), head_ptr<const int>(H[6], H[7]), T.depth, (int)(N[0] & 0xffffu), T.tok0, kG * (int)N[1], (int)N[2],
             (int)(N[0] >> 16), T.pm, T.pl, T.pacc16, T.k16, T.v16};
  A.out16 = T.out16; A.out_bf16 = T.out_bf16; A.in_bf16 = T.in_bf16; A.adapt = T.adapt;
  return A;
}
// projection outputs xq [M][n_heads][128], xk / xv [M][n_kv][128] fp32 -> q16 and the cache rows at *d_pos + t
struct PostArgs {
  KvView kv; const float* xq; const float* xk; const float* xv; int M; int n_heads; const int* d_pos;
  const uint16_t* qn_w16; const uint16_t* kn_w16; float eps;
  const float* rope; int rd; int rope_rows;      // rope [rope_rows][rd/2] (cos, sin) pairs; rd = 0: no rotary step
  int rot; uint16_t* q16;
  // 256-channel heads only: if set, the finished K / V rows are written here as fp32 [M][n_kv][256] instead of being
  // quantized into kv (a handle with trellis-coded rows runs its encoder on them afterwards)
  float* k32_out = nullptr; float* v32_out = nullptr;
  // the gate half of the Q projection [M][n_heads][head_dim] fp32 -> gate16 (same shape, 16-bit), or nullptr
  const float* xgate = nullptr; uint16_t* gate16 = nullptr;
  int io_bf16 = 0;   // 16-bit rows that leave (q16, gate16) are bf16 instead of fp16
};

// Trellis-coded rows on their way into the cache (trellis.hip).  Row rj of the launch is (token rj / (2 n_kv), K | V, kv
// head) of the pass, read from k32 / v32 [M][n_kv][256]; its payload goes to pay0 (K) / pay1 (V) + (kvh * max_ctx + pos) *
// stride and its scale to scl0 / scl1 [kvh * max_ctx + pos].  Every group is trellis-coded with kb bits, without guard
// positions and directions.
struct TbEncArgs {
  const float* k32; const float* v32; const uint16_t* k16; const uint16_t* v16;   // fp32 rows, or 16-bit rows if k32 == nullptr
  const int* d_pos; int layer, tok0, n_kv, max_ctx, rot;
  int nrow, nm;                       // rows of the launch, scale multipliers of the profile: nrow * nm searches
  uint8_t* scr; size_t scr_w_ofs, scr_s_ofs;   // scratch: states [nrow * nm][256] bytes, at scr_w_ofs error sums [nrow * nm][8] fp32, at scr_s_ofs the scales tried [nrow * nm] fp32
  // pair tables and mean rows by group (TbAttnArgs), table gains by group, multipliers
  int kb; const uint32_t* pairs; const float* mu; const float* gains; const float* mults;
  uint8_t* pay0; uint8_t* pay1; float* scl0; float* scl1; int stride;
  int pos_limit;                      // rows at positions >= pos_limit are not stored (0: no limit besides max_ctx)
  RowMap rows;                        // multi-stream pass: token t sits at rows.pos[t] of container rows.slot[t] (pay / scl = container 0)
  int in_bf16;                        // k16 / v16 are bf16 rows
};
// The codec alone (reference TbFastArgs, src/kvq_fast.hpp:16-37): rows row0 .. row0 + nrow - 1 of yin with their own group
// and position, any profile; results indexed by row.
struct TbProbeArgs {
  const uint8_t* blob; int nm; int has_trellis;
  // what the host looked up in the blob (see tb_descriptors in abi.hip): [ngrp][8] words
  //   { mode | bits << 8 | table << 16 | guard << 24, directions | has_mean << 8, byte offset of the mean row, of the
  //     first direction, index (in int16 units, from desc) of the group's table as aligned int16, gain bits, 0, 0 }
  // followed by the tables; mult_off: byte offset of the scale multipliers in the blob
  const uint32_t* desc; int ngrp; unsigned mult_off;
  const float* yin; const int* grp; const int* pos; int row0, nrow;
  float* yout; uint32_t* side; uint8_t* pay; int stride;
  uint8_t* scr; size_t scr_w_ofs;     // states and error sums, as above
};
// what the searches of a launch have left in the scratch (TbEncArgs): nm jobs per row
struct TbJobs { const uint8_t* scr; size_t w_ofs, s_ofs; int nm; };
__host__ __device__ inline TbJobs tb_jobs(const TbEncArgs& A) { return TbJobs{A.scr, A.scr_w_ofs, A.scr_s_ofs, A.nm}; }
// attention over trellis-coded rows (attend_tb.hip).  pairs [groups][2^(8 + kb)]: entry i = the table's integers, as two
// fp16 values, of the states (i >> kb) & 255 and i & 255 (two consecutive elements from 8 + kb stream bits); gfac [groups]:
// gain / 256; mu [groups][256] fp32 mean rows (zero rows where a group has none) or nullptr if no group has one
// At a multiple of 64 bytes among a kernel's arguments: what a decode workgroup asks of it first does not straddle two
// cache lines, whatever stands in front (4 layers of one token of 4 bits at 16,000 tokens 65.2 us with the rows' pointers
// across two lines, 64.3 so).
struct alignas(64) TbAttnArgs {
  const uint8_t* kpay; const uint8_t* vpay; const float* kscl; const float* vscl; int max_ctx, n_kv, stride;
  const uint32_t* pairs; const float* gfac; const float* mu; int layer;
  const uint16_t* q16; const int* d_pos; const uint8_t* depth; int M, tok0, n_heads, S;
  float* pm; float* pl; uint16_t* pacc16;
  RowMap rows;  // narrow kernel only: multi-stream pass (one token per workgroup column; kpay .. vscl = container 0, `layer` = the profile's layer)
  int in_bf16 = 0;   // q16 is bf16 rows
  int adapt = 0;     // multi-stream pass: workgroups shared out by ms_share, the shares left in plan
  int2* plan = nullptr;
  int rows_per_block = 128;   // wide kernel only
  TbJobs jobs{};     // wide kernel: searches of the rows of the pass (at most kTbFuseRows), which its workgroups then store; scr == nullptr: they are stored
  int s_short = 0;   // decode: splits in use at a position up to kShortPos, S beyond; 0: always S (splits_at)
};
void launch_attend_tb(const TbAttnArgs&, int kb, hipStream_t);        // row tiles of 2 tokens x 6 heads (decode; any width)
void launch_attend_tb_wide(const TbAttnArgs&, int kb, hipStream_t);   // 3..64 rows: 128 query rows per workgroup, tiles decoded once into LDS
// decode workgroup b -> split and kv head.  With s_short the splits that are always in use come first: the workgroups that
// may exit then do not take the CUs the others would have had to themselves
__device__ __forceinline__ void tb_split_of(const TbAttnArgs& A, int b, int& split, int& kvh) {
  if (A.s_short) { split = b / A.n_kv; kvh = b % A.n_kv; } else { split = b % A.S; kvh = b / A.S; }
}
void launch_tb_encode(const TbEncArgs&, hipStream_t);
void launch_tb_search(const TbEncArgs&, hipStream_t);     // the searches alone: TbAttnArgs::jobs has their results stored
void launch_tb_probe(const TbProbeArgs&, hipStream_t);
// one or two tokens: searches of the encoder and attention over the keys in front of *d_pos; the combiner has to store the
// new rows and add them
void launch_tb_encode_attend(const TbEncArgs&, const TbAttnArgs&, int kb, hipStream_t);
void launch_tb_unpack(const uint8_t* blob, const int* grp, const int* pos, const uint8_t* pay, const uint32_t* side, int stride, const float* yin,
                      float* y, int rows, hipStream_t);

// Trellis windows of at most so many rows are coded and stored by the attention launch, the others by a launch of their
// own: the workgroup that holds the window codes 2 rows per token, 8 at a time, which costs about two tiles of its share
// (its range is shorter by so much) and saves the launch between.  us per 16 layers, launch / here: 16 rows of 5 bits at
// 16,384 tokens 743 / 687; per 4 layers at 500 tokens 3 rows 87.9 / 81.8, 10 rows 107.9 / 103.8, 16 rows 138.2 / 138.9, 16
// rows of 4 bits at 3,000 156.2 / 145.3.  16 is the widest window that loses nothing on short contexts, where nothing hides
// the coding.  Of wider ones (4 layers, 5 bits; 6 rows a wave for 17 and 21 rows, 12 for 32 and 48) 17, 21, 32 and 48 rows
// take 143 / 147, 158 / 162, 175 / 185 and 223 / 236 at 500 tokens, 152 / 142, 167 / 156, 193 / 183 and 244 / 234 at 3,000,
// and 184 / 169, 193 / 181, 256 / 242 and 346 / 336 at 16,000: what long contexts would gain short ones would pay, and the
// host does not know which it has.
constexpr int kTbFuseRows = 16;

// launchers (each checks nothing: the C layer validates shapes first)
void launch_append(const AppendArgs&, hipStream_t);
void launch_attend_narrow(const AttnArgs&, hipStream_t);   // 16-row tiles: 2 tokens x 6 heads per workgroup column
void launch_attend_wide(const AttnArgs&, hipStream_t);     // 3..64 tokens, and prefill slices
void launch_attend_chunk(const AttnArgs&, hipStream_t);    // slices of a prefill chunk (rows already in the cache) on the wide kernel
void launch_attend_mid(const AttnArgs&, hipStream_t);      // 3..16 tokens: a wave owns whole tiles, row tiles of 16 rows (wider: blocks of 16 tokens)
void launch_combine(const CombineArgs&, hipStream_t);
void launch_attn_post(const PostArgs&, hipStream_t);
void launch_attn_post256(const PostArgs&, hipStream_t);    // the same step for 256-channel heads (attend256.hip)
// the reference's own rows, head_dim 256 (attend256.hip): same argument structs, 67584-byte pages
void launch_append256(const AppendArgs&, hipStream_t);
void launch_rotate_q256(const float* x32, int rows, uint16_t* q16, hipStream_t);   // rotated query rows, rounded to fp16
void launch_attend256(const AttnArgs&, hipStream_t);       // row tiles of 2 tokens x 6 heads (decode; any width)
void launch_attend256_wide(const AttnArgs&, hipStream_t);  // 3..64 rows: 128 query rows per workgroup, tiles dequantized once into LDS
void launch_combine256(const CombineArgs&, hipStream_t);
void launch_combine256_new(const CombineArgs&, const TbAttnArgs&, const TbJobs&, int kb, hipStream_t);   // the partials of launch_tb_encode_attend and the new rows
void launch_export_rows256(const KvView&, int pos0, int n, uint32_t* kw, float* ks, uint32_t* vw, float* vs, hipStream_t);
void launch_import_rows256(const KvView&, int pos0, int n, const uint32_t* kw, const float* ks, const uint32_t* vw, const float* vs, hipStream_t);
// canonical <-> physical
void launch_export_rows(const KvView&, int pos0, int n, uint8_t* kc, uint16_t* ks, uint8_t* vc, uint16_t* vs, hipStream_t);
void launch_import_rows(const KvView&, int pos0, int n, const uint8_t* kc, const uint16_t* ks, const uint8_t* vc, const uint16_t* vs, hipStream_t);
void launch_dequant_rows(const KvView&, int pos0, int n, float* k, float* v, hipStream_t);
void launch_codec_probe(const uint16_t* x16, int rows, uint8_t* codes, uint16_t* scales, float* y, hipStream_t);
void launch_set_int(int* p, int v, hipStream_t);
void launch_zero_ints(int* p, int n, hipStream_t);   // a fill kernel (safe inside a captured graph, unlike a memset node)
// the reference's own 256-channel row format (row256.hip): mode 0 = int8 rows, 1 = flat int4 (32 MSB-first words per row)
void launch_row256_encode(const float* x, int rows, int mode, int rot, int8_t* q8, uint32_t* words, float* scales, hipStream_t);
void launch_row256_decode(int rows, int mode, int rot, const int8_t* q8, const uint32_t* words, const float* scales, float* y, hipStream_t);
// the step after attention for 256-channel heads: gate, signs, 512-point Hadamard transform, int8 groups of 512 (n_heads even)
void launch_attn_out256(const uint16_t* y16, const uint16_t* gate16, const int8_t* signs, int M, int n_heads, int lo, int8_t* qx, float* alpha, hipStream_t);

// machine probe (probe.hip): fixed instruction mixes that time themselves; rec gets (shader cycles, wall ticks) per wave
void launch_probe_mix(int nv, bool mfma, float* sink, unsigned long long* rec, int iters, int iters_b, int split, int blocks, int threads, hipStream_t);
void launch_probe_mfma16(float* sink, unsigned long long* rec, int iters, int blocks, hipStream_t);
void launch_probe_valu(int op, float* sink, unsigned long long* rec, int iters, int blocks, int threads, hipStream_t);
void launch_probe_cross(int op, float* sink, unsigned long long* rec, int iters, int iters_b, int blocks, hipStream_t);
void launch_probe_read(bool nt, const void* src, size_t bytes, float* sink, int blocks, hipStream_t);

// fp32 -> bf16 bit pattern, round to nearest even (finite inputs)
__device__ __forceinline__ uint16_t f2bf_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float bf_bits2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
// Rows a caller hands over in bf16 (option key 11) become fp16 where they are read: every kernel that takes 16-bit rows
// calls these on the registers it has loaded.  The fp32 value of a bf16 is rounded to fp16 (nearest even; exact for
// magnitudes between 2^-14 and 65504).  The flag is a kernel argument, i.e. a scalar.  One branch serves all
// registers of a thread (a branch per register makes every load wait for the one before it: 4 us of the 36 us of a
// 1,024-row prefill slice); kernels whose fp16 form a branch would slow down have a form of their own for bf16 rows.
// A launch of its own that converted the rows first cost 1.5 .. 4 us of every call (a third of a decode call at 1,000
// tokens: 9.8 us with it, 7.0 without).
__device__ __forceinline__ uint32_t bf_pair_to_f16(uint32_t w) {
  const uint16_t lo = __half_as_ushort(__float2half_rn(__uint_as_float(w << 16))), hi = __half_as_ushort(__float2half_rn(__uint_as_float(w & 0xffff0000u)));
  return (uint32_t)lo | ((uint32_t)hi << 16);
}
template <int N>
__device__ __forceinline__ void rows16_to_f16(uint4 (&r)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) { r[k].x = bf_pair_to_f16(r[k].x); r[k].y = bf_pair_to_f16(r[k].y); r[k].z = bf_pair_to_f16(r[k].z); r[k].w = bf_pair_to_f16(r[k].w); }
}
template <int N>
__device__ __forceinline__ void rows16_to_f16(uint4 (&r)[N], int bf16) { if (bf16) rows16_to_f16(r); }
// one value: both readings and a select, no branch
__device__ __forceinline__ float row16_value(uint16_t b, int bf16) {
  const float as_f16 = __half2float(__ushort_as_half(b)), as_bf16 = __half2float(__float2half_rn(bf_bits2f(b)));
  return bf16 ? as_bf16 : as_f16;
}
// 8 fp32 results -> 16 bytes of fp16 or bf16
__device__ __forceinline__ uint4 pack_out8(const float* y, int bf16) {
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint16_t lo = bf16 ? f2bf_bits(y[2 * k]) : __half_as_ushort(__float2half_rn(y[2 * k]));
    const uint16_t hi = bf16 ? f2bf_bits(y[2 * k + 1]) : __half_as_ushort(__float2half_rn(y[2 * k + 1]));
    w[k] = (uint32_t)lo | ((uint32_t)hi << 16);
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// 16 bytes of a partial row, written through the XCD's L2 (agent scope) as it leaves the workgroup.  The combiner runs on
// other XCDs, so what lies dirty in an L2 when the launch ends is written back then, with nothing else running: 9.6 MB of
// partials of 24 rows in 32 splits kept the combiner waiting 5 us behind the last workgroup, where 1.4 us are usual.
// Written through, the rows of the workgroups that end early are out before the last one ends.  us per 16 layers, ordinary
// / nontemporal / written through: 24 rows of 256 channels at 9,001 tokens 396 / 370 / 363, 64 rows of 128 at 32,768 741 /
// 733 / 730, 8 rows at 12,037 229 / 225 / 225.  Decode and the smallest windows leave little, which nobody waits for, and
// such stores are in the way of their end: one token at 32,741 tokens 173 / 173 / 176, 16 streams 27.2 / 27.8 / 28.0 a
// pass, 4 rows at 32,768 259 ordinary and 263; they keep ordinary stores.
__device__ __forceinline__ void store_partial16(uint16_t* p, uint4 v) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) u32x4*)p, u32x4{v.x, v.y, v.z, v.w}, "agent");
}

// least and greatest depth of tokens tok_lo .. tok_hi - 1 (at most 64), a token per lane: one trip to memory (a loop over
// them was one each: 4 layers of 16 rows with a depth table at 9,000 tokens 68.9 us, 63.7 so, of 24 rows of 256
// channels 88.8 and 85.8, of 16 trellis rows 177 and 172)
__device__ __forceinline__ void depth_range(const uint8_t* depth, int tok_lo, int tok_hi, int& least, int& most) {
  const int t = tok_lo + (int)(threadIdx.x & 63), last = max(tok_lo, tok_hi - 1);
  const int dp = depth[min(t, last)];
  least = __builtin_amdgcn_readfirstlane(lane_rows(lane_row16(dp, LaneMin{}), LaneMin{}));
  most = __builtin_amdgcn_readfirstlane(lane_rows(lane_row16(dp, LaneMax{}), LaneMax{}));
}

// Sums and maxima of the plans below run through lane-crossing moves (a shift inside rows of 16 lanes, then two row
// broadcasts), not through LDS: a plan stands in front of everything else a workgroup does (multi-stream passes, 5 trellis
// streams of up to 3,000 tokens: 28.4 us a pass before, 27.5 since; 30 int4 streams of 128 channels 14.9 and 13.9).
template <class Op>
__device__ __forceinline__ int wave_scan(int v, Op op) {            // inclusive over the lanes; 0 is the neutral value
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));        // row_shr:1, 2, 4, 8
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));        // row_bcast:15 into rows 1 and 3
  return op(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));     // row_bcast:31 into rows 2 and 3
}
__device__ __forceinline__ int wave_scan_add(int v) { return wave_scan(v, [](int a, int b) { return a + b; }); }

// Splits a slice of a prefill chunk uses, of the `S` its launch provides for.  The host sizes the grid without knowing the
// position, so the choice is made on the device, by every wave of the attention launch and again by the combiner: lane s -
// 1 prices s splits, the cheapest wins (ties: the fewest).  Whole numbers only, so that two compilations cannot disagree.
// Times are in sixteenths of the time a workgroup takes for one 32-key tile (0.56 us): a workgroup costs kChunkOverhead
// tiles before and after its loop (about 10 us: launch, query, first tile, merge, stores), one workgroup runs per CU, the
// longest start first, and more than one split costs a combiner pass over M * s partial rows.
// 1,500 rows on an empty cache in containers of 8,192 tokens, us per layer call: 105 with slices of 1,024 tokens in 4 and 8
// splits (39 + 39 in the attention, 23 in the combiners), 46 with one split (42 in the attention, which then waits for its
// longest workgroup: 47 tiles; 48 and 44 while the choice went through LDS).  2,048 rows behind 131,072: the same with 2
// splits of one slice as with 4 of two.
constexpr int kChunkOverhead = 18, kChunkMaxSplits = 64;
// Price of s splits in those units, for a slice whose first and last row blocks walk so many tiles.  Workgroups times tiles
// would pass 2^31 with 2,048 rows on 4 KV heads at 11 M tokens, and the two readers of a choice have to agree on it: the
// caller cuts the tiles at chunk_tile_cap (which changes no choice: beyond it the overhead is nothing).  That limit comes
// from the host, in `adapt`; 64-bit products or a unit chosen here cost 1 % of a prompt's first slice, as instructions
// fetched cold in front of everything else.
__host__ __device__ constexpr unsigned chunk_price(int first, int last, int base, int M, int s) {
  const unsigned lo = first * 16 / s + 16 * kChunkOverhead, hi = last * 16 / s + 16 * kChunkOverhead;
  const unsigned n = (unsigned)base * s, idle = (256 - (n & 255)) & 255;        // workgroups, and CUs without one in the last round
  const unsigned rounds = (n >> 1) * (lo + hi) / 256 + lo * idle / 256, t = hi > rounds ? hi : rounds;
  return s > 1 ? t + 96 + (unsigned)(M * s) / 13 : t;
}
constexpr int chunk_tile_cap(int base) { return base < 64 ? 1 << 20 : (1 << 26) / base; }
static_assert(chunk_price(chunk_tile_cap(384), chunk_tile_cap(384), 384, 2048, 2) * 10u < chunk_price(chunk_tile_cap(384), chunk_tile_cap(384), 384, 2048, 1) * 9u,
              "two splits fill 768 of 768 places, one 384 of 512, also on the longest contexts");
static_assert(chunk_price(chunk_tile_cap(4), chunk_tile_cap(4), 4, 22, 1) < 0x1fffffeu, "a price and a split count share 31 bits");
__device__ __forceinline__ int chunk_splits_used(int pos, int tok0, int M, int n_kv, int max_ctx, int S, int tile_cap) {
  const int base = n_kv * ((kG * M + 127) / 128), s = (int)(threadIdx.x & 63) + 1;
  const int first = max(0, min(pos + tok0 + min(M, 128 / kG + 1), max_ctx)), last = max(0, min(pos + tok0 + M, max_ctx));
  const unsigned t = chunk_price(min((first + 31) >> 5, tile_cap), min((last + 31) >> 5, tile_cap), base, M, s);
  // lowest price, then fewest splits: the largest key (lane 0 always has one)
  const int key = s <= S ? 0x7fffffff - (int)((min(t, 0x1fffffeu) << 6) | (unsigned)(s - 1)) : 0;
  const int top = __builtin_amdgcn_readlane(wave_scan(key, [](int a, int b) { return max(a, b); }), 63);
  return ((0x7fffffff - top) & 63) + 1;
}

// Trellis decode in containers that may hold more than kShortPos tokens: the grid provides two workgroups per CU and the
// position, found on the device, says whether both are used.  A workgroup alone on its CU makes the combiner cheaper; on a long
// context its waves wait for memory and LDS gathers that a second one fills.  us per layer call, one row of 5 bits, 64 / 128
// splits: 23.8 / 27.8 at 16,000 tokens, 41.3 / 42.7 at 70,000, 58.7 / 56.5 at 130,000, 81.7 / 74.1 at 200,000; 4 bits 39.5 /
// 41.6 at 70,000, 57.1 / 55.6 at 130,000.  (int4 rows of 256 channels gain nothing: 42.7 / 43.9 at 200,000.)
// The workgroups that exit cost 1 us below kShortPos (23.4 -> 24.5 us at 16,000 tokens in a container of 262,144).
constexpr int kShortPos = 98304;
__device__ __forceinline__ int splits_at(int S, int s_short, int pos) { return s_short && pos <= kShortPos ? s_short : S; }

// Multi-stream pass: how the W workgroups of one kv head are shared out over the pass's M <= 64 rows.  Streams differ in
// length, and with the same number of splits for each the workgroups of the longest set the pace: every split is given
// about the same number of 32-key tiles instead: row t gets ceil(tiles / c) splits, c >= 4 (one per wave) and no row more
// than 256.  c = (tiles of all rows) / (W - M) always fits, since every row may round up by one; four halvings look for a
// smaller one.
// 16 streams of 2,000 to 32,000 tokens: 36.7 us a pass with 16 splits each (the longest stream's workgroups walk 62 tiles,
// the shortest's 4), 32.5 shared out over two workgroups per CU (four: 34.5), 30.6 with the new rows stored here as well.
// Row t's splits are workgroups base .. base + n - 1 of the kv head, which is also where its partials lie.  Computed by
// every wave from the row map (lane t looks at row t); the first wave of the launch leaves the shares in memory for the
// combiner, whose workgroups have nothing to hide the computation under (48 streams of 300 tokens, 5 bits: its launch 6.0
// us when it computed the shares, 4.6 since).
struct MsShare { int row, split, n, pos, slot; size_t base; };
// ceil(a / b) for quotients up to 2^16 and a below 2^27: the float quotient is off by one at most
__device__ __forceinline__ int ms_tiles_per(int a, int b) {
  const int n = a + b - 1;
  int q = (int)((float)n * __builtin_amdgcn_rcpf((float)b));
  const int r = n - q * b;
  return q + (r >= b) - (r < 0);
}
// workgroup b of the kv head; row = -1: nothing left for it.  leave: this wave stores the plan.  W_short: of the W launched
// workgroups only so many are used while each of them would get fewer than kMsLong tiles (0: always all)
constexpr unsigned kMsLong = 48;
__device__ __forceinline__ MsShare ms_share(const RowMap& R, int M, int max_ctx, int W, int W_short, int b, int2* plan, bool leave) {
  const int lane = threadIdx.x & 63, pos = lane < M ? R.pos[lane] : -1, slot = lane < M ? R.slot[lane] : -1;
  // 0 tiles: a row that names no container or position
  const int tiles = pos >= 0 && pos < max_ctx && slot >= 0 && slot < R.n_slots ? (pos + 32) >> 5 : 0;
  // unsigned: 64 rows of the longest container are just under 2^32 tiles
  const unsigned total = max(1u, (unsigned)__builtin_amdgcn_readlane(wave_scan_add(tiles), 63));
  const int most = __builtin_amdgcn_readlane(wave_scan(tiles, [](int a, int b) { return max(a, b); }), 63);
  if (W_short && total < kMsLong * (unsigned)W_short) W = W_short;
  int lo = max(4, max((most + 255) >> 8, (int)((total - 1) / (unsigned)W + 1))), c = max(lo, (int)((total - 1) / (unsigned)(W - M) + 1));
  int mine = ms_tiles_per(tiles, c), incl = wave_scan_add(mine);
  for (int it = 0; it < 4 && lo < c; ++it) {       // c always fits; a smaller one may
    const int mid = (lo + c) >> 1, want = ms_tiles_per(tiles, mid), sum = wave_scan_add(want);
    if (__builtin_amdgcn_readlane(sum, 63) <= W) { c = mid; mine = want; incl = sum; } else lo = mid + 1;
  }
  if (leave && lane < M) plan[lane] = make_int2(incl - mine, mine);
  const int row = __popcll(__ballot(incl <= b));
  if (row >= M) return {-1, 0, 0, 0, 0, 0};
  const int n = __builtin_amdgcn_readlane(mine, row), base = __builtin_amdgcn_readlane(incl, row) - n;
  return {row, b - base, n, __builtin_amdgcn_readlane(pos, row), __builtin_amdgcn_readlane(slot, row), (size_t)base};
}

// Multi-stream pass of at most 64 rows whose attention launch stores the new rows itself: the rows of the pass (bit t = row
// t) that a workgroup of a row at `pos` in container `slot` has to store before it reads tiles [tile0, tile1) - rows of the
// same stream it can see.  Rows of one stream that follow each other are stored by every workgroup that reads them, the same
// bytes each time, so that no workgroup depends on another.
__device__ __forceinline__ uint64_t ms_new_rows(const RowMap& R, int M, int slot, int pos, int tile0, int tile1, int& lane_pos) {
  const int lane = threadIdx.x & 63;
  lane_pos = lane < M ? R.pos[lane] : -1;
  const bool mine = lane < M && R.slot[lane] == slot && lane_pos >= 0 && lane_pos <= pos && (lane_pos >> 5) >= tile0 && (lane_pos >> 5) < tile1;
  return __ballot(mine);
}

// A 16-bit value of a new row, requested before the position is known: whether the workgroup has to store the row is decided by
// the position, and a load that waited for that decision would be a trip to memory of its own.  Atomic (relaxed, workgroup
// scope: a plain load instruction) so that the compiler leaves the request where it stands instead of moving it to its use.
__device__ __forceinline__ uint2 request64(const uint64_t* p) {
  const uint64_t v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
}
__device__ __forceinline__ uint16_t request16(const uint16_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// start of the (page, kv head) block that holds token t
__device__ __forceinline__ uint8_t* kv_page(const KvView& kv, int kvh, int t) {
  const int lp = t / kPageTok;
  const int pp = kv.table ? kv.table[lp] : lp;
  return kv.base + (size_t)(pp * kv.n_kv + kvh) * kPageBytes;
}

// table[index] through the scalar data path; pointer and index are forced into scalar registers (they are uniform over
// the wave by contract, but the compiler cannot always prove it, e.g. inside a branch on a wave-uniform condition)
__device__ __forceinline__ int table_entry_scalar(const int32_t* table, int index) {
  const uint64_t a = (uint64_t)(uintptr_t)table;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  const uint64_t base = ((uint64_t)hi << 32) | lo;
  const int off = __builtin_amdgcn_readfirstlane(index * 4);
  int v;
  asm volatile("s_load_dword %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(base), "s"(off) : "memory");
  return v;
}

// The same for a token index that is uniform over the wave (the attention kernels' tile loops).  The page-table entry is
// fetched through the scalar data path: a vector load would share its completion counter with the tile loads a wave
// keeps in flight, so waiting for the entry would wait for all of them.  (Read only; the table is written by the host.)
__device__ __forceinline__ uint8_t* kv_page_uniform(const KvView& kv, int kvh, int t) {
  const int lp = t / kPageTok;
  int pp = lp;
  if (kv.table) pp = table_entry_scalar(kv.table, lp);
  return kv.base + (size_t)(pp * kv.n_kv + kvh) * kPageBytes;
}

}  // namespace yka
