// C ABI of libyka.so: handle, validation, launch sequencing, host-pointer hooks.
// Error convention of the reference's C layer (src/c_api.cpp:17,33,49): catch everything, keep a thread-local
// message, return -1.
#include "../../include/yka_abi.h"
#include "yka_internal.h"
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

using namespace yka;

static thread_local std::string g_err;

#define HIPCHK(expr)                                                                                  \
  do {                                                                                                \
    hipError_t rc_ = (expr);                                                                          \
    if (rc_ != hipSuccess) throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(rc_)); \
  } while (0)

struct yka_kv {
  yka_kv_config cfg{};
  int n_pages = 0;
  size_t layer_bytes = 0;
  uint8_t* pool = nullptr;
  int32_t* tables = nullptr;       // [n_layers][n_pages], paged mode only
  float *pm = nullptr, *pl = nullptr; uint16_t* pacc16 = nullptr;
  int* tickets = nullptr;     // [n_kv_heads][64] split tickets of the decode kernel, all zero between launches
  size_t ws_rows = 0;              // capacity of the partial workspace in (token, split) pairs
  int2* ms_plan = nullptr;         // [64] shares of a multi-stream pass, attention launch -> combiner
  int* d_pos = nullptr;            // position used by the host-pointer hooks
  hipStream_t stream = nullptr;    // stream of the host-pointer hooks
  int opt_splits_narrow = 0, opt_splits_wide = 0, opt_force_narrow = 0, opt_unrot = 0, opt_ctx_hint = 0, opt_profile_layer = 0, opt_merge_in_launch = 0;
  int opt_chunk_slice = 0;                     // tokens per prefill slice (0: kChunkSlice)
  int opt_io_bf16 = 0;                         // 16-bit rows at the boundary (Q, new K / V, gate, outputs) are bf16, not fp16
  // widest window the mid kernel takes (0: none), its split count (0: automatic).  Nine rows are a fourth row tile to it, and two waves
  // of rows beside two that decode to the wide kernel.  us per 16 layers, mid / wide: 8 rows at 1,000 tokens 172 / 190, at 12,000 198 / 202, at
  // 30,000 243.5 / 257.5; 9 rows at 1,000 202 / 190.4, at 9,000 242.5 / 198.4, 10 rows at 30,000 318 / 265; 4 layers at 100,000 8 rows 113.5 /
  // 115, 10 rows 158.7 / 116
  int opt_mid_rows = 8, opt_splits_mid = 0;
  // trellis-coded rows (set by yka_kv_set_profile; head_dim 256 only): rows as the reference lays them out, per layer
  // [K payload n_kv * max_ctx * stride][V payload][K scales n_kv * max_ctx fp32][V scales]
  struct Tb {
    int kb = 0, stride = 0, nm = 0, layers = 0; bool has_mu = false;   // layers: layers the profile has groups for
    uint32_t* pairs = nullptr; float* gfac = nullptr; float* mu = nullptr;
    uint8_t* pool = nullptr; size_t layer_bytes = 0, pay_bytes = 0, scl_bytes = 0;
    uint8_t* scr = nullptr; size_t scr_w_ofs = 0, scr_s_ofs = 0;
    const float* mults = nullptr; const float* gains = nullptr;    // scale multipliers and the groups' table gains, behind gfac
    float* stage = nullptr;          // fp32 K rows then V rows of one pass ([max_rows][n_kv][256] each): yka_attn_post -> encoder
    // 256 bytes in front of the first row: windows of the attention kernels begin in the word before a chunk
    uint8_t* kpay(int layer) const { return pool + 256 + (size_t)layer * layer_bytes; }
    uint8_t* vpay(int layer) const { return kpay(layer) + pay_bytes; }
    float* kscl(int layer) const { return reinterpret_cast<float*>(kpay(layer) + 2 * pay_bytes); }
    float* vscl(int layer) const { return reinterpret_cast<float*>(kpay(layer) + 2 * pay_bytes + scl_bytes); }
  };
  Tb* tb = nullptr;
  bool r256() const { return cfg.head_dim == 256; }   // the reference's own rows (attend256.hip); otherwise the 128-channel format
  int D() const { return cfg.head_dim; }
  KvView view(int layer) const {
    return KvView{pool + (size_t)layer * layer_bytes, tables ? tables + (size_t)layer * n_pages : nullptr, cfg.n_kv_heads, cfg.max_ctx};
  }
};

// Workspace of the allocation-free entry point: the split partials of one slice, in device memory the library's code
// object carries itself (every GPU that loads the library holds its own copy until the process ends).  The name is a
// host-side stand-in, not a device address: the address of a device's copy is looked up once per device with that
// device current, and only that address is ever handed to a kernel.
constexpr size_t kStaticPairs = 1536;                              // (token, split) pairs: 64 rows x 21 splits, or 16 rows x 64, ...
constexpr size_t kStaticHeads = 24;                                // query heads the array is sized for
constexpr size_t kStaticPmBytes = kStaticPairs * kStaticHeads * 4;  // a multiple of 256
constexpr size_t kStaticTicketBytes = 1024;                         // 4 kv heads x 64 row tiles; zero when the library is loaded, zero after every launch
constexpr size_t kStaticWsBytes = 2 * kStaticPmBytes + kStaticPairs * kStaticHeads * kD * 2 + kStaticTicketBytes;   // 9,733,120 bytes
static __device__ __align__(256) unsigned char scratch[kStaticWsBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_static_mu;
unsigned char* g_static_ptr[kMaxDevices] = {};                      // device address of `scratch` on each device, once looked up
// must be called with `device` current
unsigned char* static_workspace(int device) {
  if (device < 0 || device >= kMaxDevices) throw std::runtime_error("device ordinal beyond the static workspace table");
  std::lock_guard<std::mutex> lock(g_static_mu);
  if (!g_static_ptr[device]) {
    void* p = nullptr;
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw std::runtime_error("hipGetSymbolAddress returned no address for the static workspace");
    g_static_ptr[device] = static_cast<unsigned char*>(p);
  }
  return g_static_ptr[device];
}

struct DevBuf {  // device buffer that frees itself (hooks only; the launch path never allocates)
  void* p = nullptr;
  explicit DevBuf(size_t n) { HIPCHK(hipMalloc(&p, n ? n : 1)); }
  ~DevBuf() { if (p) (void)hipFree(p); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  template <class T> T* as() const { return static_cast<T*>(p); }
};

void on_device(const yka_kv* kv) {
  if (!kv) throw std::runtime_error("null handle");
  HIPCHK(hipSetDevice(kv->cfg.device));
}

constexpr int kMaxSplits = 256;
// (token, split) pairs of the partial workspace, n_heads * (2 * head_dim + 8) bytes each.  Windows and streams stay below
// kWsPairs (24 heads: 26 MB with 128 channels, 51 with 256); a slice of a prefill chunk may ask for more, kChunkPairs at
// most (ws_pairs_of)
constexpr size_t kWsPairs = 4096, kChunkPairs = 12288;

// splits for the narrow kernel: one workgroup per CU (256 of them) while a workgroup then walks at most 48 tiles - its
// waves keep the next tile in flight, and half as many partial rows make the combiner cheaper (measured: 12.2 against
// 13.1 us per layer call at 32k, 16.0 / 16.9 at 65k) - and two per CU beyond that (35.4 against 41.8 us at 262k)
int narrow_splits(const yka_kv* kv, int M, size_t ws_pairs = kWsPairs) {
  if (kv->opt_splits_narrow > 0) return std::min(kv->opt_splits_narrow, (int)(ws_pairs / (size_t)M));
  const int tiles = (M + 1) / 2;
  // launching a split costs more than letting it exit: the grid is sized for the context the caller expects (option
  // key 5; by default the capacity of the handle), two 32-key tiles per workgroup at least
  const int ctx = kv->opt_ctx_hint > 0 ? std::min(kv->opt_ctx_hint, kv->cfg.max_ctx) : kv->cfg.max_ctx;
  const int ctx_tiles = (ctx + 31) / 32;
  const int wgs = ctx_tiles > 48 * 64 ? 512 : 256;
  int S = std::min(wgs / (kv->cfg.n_kv_heads * tiles), ctx_tiles / 2);
  S = std::max(2, std::min(kMaxSplits, S));
  return std::min(S, (int)(ws_pairs / (size_t)M));
}

// Wide kernel geometry: a workgroup of 8 waves owns up to 128 query rows and one split (its two wave groups take alternate
// tiles of the split and merge on chip), one workgroup per compute unit.  Splits: one workgroup per CU (256 of them), at
// least four 32-key tiles (two steps of either group) per workgroup, sized like the decode grid by the expected context.
// At 64 rows (three row blocks) that is 21 splits: 64 x 21 x 24 partial rows of 264 bytes, 8.5 MB.
// The blocks of a window are cut at the even share of its rows rounded up to whole waves of 32: no block has more waves of rows than that, the last
// may have fewer (144 rows are 96 + 48 and not 128 + 16, 132 are 96 + 36; figures at the roles in attend_wide.hip).
int wide_rows_per_block(int M) {
  const int rows = kG * M, rb = (rows + 127) / 128;
  return M > kMaxSlice ? 128 : ((rows + rb - 1) / rb + 31) / 32 * 32;
}
int wide_splits(const yka_kv* kv, int M, size_t ws_pairs = kWsPairs) {
  const int rows = kG * M, rpb = wide_rows_per_block(M), rb = (rows + rpb - 1) / rpb;
  const int ctx = kv->opt_ctx_hint > 0 ? std::min(kv->opt_ctx_hint, kv->cfg.max_ctx) : kv->cfg.max_ctx;
  int S = kv->opt_splits_wide > 0 ? kv->opt_splits_wide : std::min(256 / (kv->cfg.n_kv_heads * rb), ((ctx + 31) / 32) / 4);
  S = std::max(1, std::min(kMaxSplits, S));
  return std::min(S, std::max(1, (int)(ws_pairs / (size_t)M)));
}

// Mid kernel (windows of 3..16 tokens; wider ones as blocks of 16 tokens): one workgroup of 4 waves per CU, every wave
// at least one tile.
int mid_splits(const yka_kv* kv, int M, size_t ws_pairs = kWsPairs) {
  const int nb = (M + 15) / 16, wgs = 256;
  const int ctx = kv->opt_ctx_hint > 0 ? std::min(kv->opt_ctx_hint, kv->cfg.max_ctx) : kv->cfg.max_ctx;
  int S = kv->opt_splits_mid > 0 ? kv->opt_splits_mid : std::min(wgs / (kv->cfg.n_kv_heads * nb), ((ctx + 31) / 32) / 4);
  S = std::max(1, std::min(kMaxSplits, S));
  return std::min(S, std::max(1, (int)(ws_pairs / (size_t)M)));
}

// Prefill chunks: slices of up to 2048 tokens, 128 rows per workgroup.  How many splits a slice uses is decided on the
// device (chunk_splits_used: a chunk early in its context needs none); the grid provides the number between 1 and
// kChunkMaxSplits that fills the rounds of 256 workgroups best on a long context - each split at least eight tiles of the
// expected context, at most 2,048 workgroups and the partial workspace.
constexpr int kChunkSlice = 2048, kMaxChunkSlice = 4096, kChunkSlice256 = 1024;
int chunk_splits(const yka_kv* kv, int Ms, size_t ws_pairs) {
  if (kv->opt_splits_wide > 0) return std::max(1, std::min(kv->opt_splits_wide, (int)(ws_pairs / (size_t)Ms)));
  const int rb = (kG * Ms + 127) / 128, base = kv->cfg.n_kv_heads * rb;
  const int ctx = kv->opt_ctx_hint > 0 ? std::min(kv->opt_ctx_hint, kv->cfg.max_ctx) : kv->cfg.max_ctx;
  const int top = std::min({kChunkMaxSplits, (int)(ws_pairs / (size_t)Ms), ((ctx + 31) / 32) / 8, 2048 / base});
  int best = 1;
  double best_fill = 0;
  for (int s = 1; s <= top; ++s) {
    const int n = base * s, rounds = (n + 255) / 256;
    const double fill = n / (256.0 * rounds) - 0.005 * s;
    if (fill > best_fill) { best_fill = fill; best = s; }
  }
  return best;
}

// 256-channel rows, both formats: how a pass is cut.  Passes of more than 64 rows (prompt chunks) go through the wide
// kernels in slices of up to 1,024 tokens: in slices of 64 a chunk on a short context is mostly launches (1,500 first rows,
// int4: 533 us per layer call in 24 slices, 146 in two).
// Row blocks of one slice get the same number of rows, in whole waves: the fragment reads of the waves that have rows set
// the pace of a tile, so 144 rows are 80 + 64 and not 128 + 16 (24 rows at 9,001 tokens: 25.0 us per layer call against
// 26.1).
// Splits of the decode kernels: one workgroup per CU (the waves keep the next tile in flight and the combiner has half the
// rows to read: 205 against 225 us for 16 layers at 20,011 tokens, 167 / 204 at 3,000, 97 / 101 for 2 layers at 200,000).
// Windows forced through them (option key 3): two, where one would leave whole splits of the row tiles too long.  us per
// layer call with 256 / 512 workgroups, 5 bits: 4 rows 26.3 / 28.6 at 1,000 tokens, 36.7 / 36.1 at 16,000, 8 rows 28.8 /
// 30.7 and 47.9 / 45.4, 48 rows 64.2 / 62.3 and 187 / 145; int4: 16 rows 14.6 / 17.1 and 32.8 / 33.1, 48 rows 19.8 / 20.3
// and 86.3 / 69.1.
// Of the wide ones: one workgroup per CU, at least 2 * row blocks tiles each; of a chunk the fewest that fill the last of
// at most four rounds of 256 workgroups best.
struct Part256 { int Ms, S, rows_per_block; bool narrow; int s_short; };
int slice256(const yka_kv* kv, int M) { return M > kMaxSlice && !kv->opt_force_narrow ? kChunkSlice256 : kMaxSlice; }
Part256 part256(const yka_kv* kv, int M, int s0, int slice) {
  const int ctx = kv->opt_ctx_hint > 0 ? std::min(kv->opt_ctx_hint, kv->cfg.max_ctx) : kv->cfg.max_ctx, ctx_tiles = (ctx + 31) / 32;
  const int Ms = std::min(slice, M - s0), rows = kG * Ms, rb = (rows + 127) / 128, base = kv->cfg.n_kv_heads * rb;
  const bool narrow = Ms <= 2 || kv->opt_force_narrow;
  // trellis decode in containers longer than kShortPos: a second workgroup per CU, used from there on (splits_at)
  const bool two = kv->tb && Ms <= 2 && !kv->opt_splits_narrow && ctx_tiles > kShortPos / 32;
  const int wgs = two || Ms > (kv->tb ? 4 : 16) ? 512 : 256;
  int S;
  if (narrow) S = kv->opt_splits_narrow > 0 ? kv->opt_splits_narrow : std::max(2, std::min(wgs / (kv->cfg.n_kv_heads * ((Ms + 1) / 2)), ctx_tiles / 2));
  else if (kv->opt_splits_wide > 0) S = kv->opt_splits_wide;
  else if (Ms <= kMaxSlice) S = std::min(256 / base, ctx_tiles / (2 * rb));
  else {
    S = 1;
    double best = 0;
    for (int s = 1; s <= std::min(1024 / base, ctx_tiles / 8); ++s) {
      const double fill = base * s / (256.0 * ((base * s + 255) / 256)) - 0.01 * s;
      if (fill > best) { best = fill; S = s; }
    }
  }
  const size_t pairs = Ms > kMaxSlice ? kv->ws_rows : kWsPairs;
  S = std::min(std::max(narrow ? 2 : 1, std::min(kMaxSplits, S)), (int)(pairs / (size_t)Ms));
  return {Ms, S, ((rows + rb - 1) / rb + 15) / 16 * 16, narrow, two ? std::min(S, std::max(2, 256 / kv->cfg.n_kv_heads)) : 0};
}

// Pairs a handle reserves: what the longest demand among the slices its max_rows allows comes to (a context hint only lowers it, a
// split count set by the caller is cut to what is there).  4 KV heads: 4,096 up to 341 rows, then up to 10,899 (1,557 rows x 7
// splits, 69 MB at 128 channels), with 256 channels 5,376 (67 MB).  1,500 rows behind 131,072 tokens take 3.26 ms with the 7 splits
// that fill their rounds and 4.33 with the 2 that 4,096 pairs hold.
size_t ws_pairs_of(const yka_kv* kv) {
  size_t need = kWsPairs;
  const int longest = std::min(kv->cfg.max_rows, kv->r256() ? kChunkSlice256 : kMaxChunkSlice);
  for (int Ms = kMaxSlice + 1; Ms <= longest; ++Ms)
    need = std::max(need, (size_t)Ms * (kv->r256() ? part256(kv, Ms, 0, kChunkSlice256).S : chunk_splits(kv, Ms, kChunkPairs)));
  return need;
}

void check_layer(const yka_kv* kv, int layer) {
  if (layer < 0 || layer >= kv->cfg.n_layers) throw std::runtime_error("layer out of range");
}
void check_rows(const yka_kv* kv, int M) {
  if (M < 1 || M > kv->cfg.max_rows) throw std::runtime_error("M must be in [1, max_rows]");
}

void check_tb_layer(const yka_kv* kv, int layer) {
  if (kv->tb && layer >= kv->tb->layers) throw std::runtime_error("the profile has no groups for this layer");
}
constexpr int kTbTileTok = 128;     // tokens per launch of the trellis encoder (its scratch holds that many)
TbEncArgs tb_encoder_args(const yka_kv* kv, int layer, int container, const uint16_t* k16, const uint16_t* v16, int t0, int M, const int* d_pos) {
  const yka_kv::Tb& T = *kv->tb;
  TbEncArgs A{};
  A.nm = T.nm;
  A.k16 = k16; A.v16 = v16; A.in_bf16 = kv->opt_io_bf16; A.d_pos = d_pos; A.layer = layer; A.tok0 = t0; A.n_kv = kv->cfg.n_kv_heads;
  A.max_ctx = kv->cfg.max_ctx;
  A.nrow = std::min(kTbTileTok, M - t0) * 2 * kv->cfg.n_kv_heads;
  A.scr = T.scr; A.scr_w_ofs = T.scr_w_ofs; A.scr_s_ofs = T.scr_s_ofs;
  A.kb = T.kb; A.pairs = T.pairs; A.mu = T.has_mu ? T.mu : nullptr; A.gains = T.gains; A.mults = T.mults;
  A.pay0 = T.kpay(container); A.pay1 = T.vpay(container); A.scl0 = T.kscl(container); A.scl1 = T.vscl(container); A.stride = T.stride;
  return A;
}
// trellis encoder over the rows of a pass: fp32 rows, or fp16 rows if k32 == nullptr
void tb_append(yka_kv* kv, int layer, const float* k32, const float* v32, const uint16_t* k16, const uint16_t* v16, int M, const int* d_pos,
               int rot, hipStream_t st, int pos_limit = 0, const RowMap* rows = nullptr) {
  const int container = rows ? 0 : layer;            // multi-stream pass: containers are streams, `layer` only names the groups
  check_tb_layer(kv, layer);
  for (int t0 = 0; t0 < M; t0 += kTbTileTok) {
    TbEncArgs A = tb_encoder_args(kv, layer, container, k16, v16, t0, M, d_pos);
    A.k32 = k32; A.v32 = v32; A.rot = rot; A.pos_limit = pos_limit;
    if (rows) A.rows = *rows;
    launch_tb_encode(A, st);
  }
}
// the step between the projection and the cache.  On trellis-coded rows the finished K / V rows go to a staging buffer
// as fp32 and the encoder runs on them (the reference: launch_q35_attn_post, then launch_tb_requant, q35_kernels.cu:1084-1092)
void post_launch(yka_kv* kv, int layer, PostArgs& A, hipStream_t st) {
  if (kv->tb) {
    A.k32_out = kv->tb->stage;
    A.v32_out = kv->tb->stage + (size_t)kv->cfg.max_rows * kv->cfg.n_kv_heads * 256;
    launch_attn_post256(A, st);
    // rows the post kernel drops (beyond the rotary table) are not stored by the encoder either
    tb_append(kv, layer, A.k32_out, A.v32_out, nullptr, nullptr, A.M, A.d_pos, 0, st, A.rd > 0 ? A.rope_rows : 0);
  } else if (kv->r256()) launch_attn_post256(A, st);
  else launch_attn_post(A, st);
}
void no_trellis(const yka_kv* kv) {
  if (kv->tb) throw std::runtime_error("this entry point does not work on trellis-coded rows");
}

void do_append(yka_kv* kv, int layer, const uint16_t* k16, const uint16_t* v16, int M, const int* d_pos, hipStream_t st) {
  if (kv->tb) tb_append(kv, layer, nullptr, nullptr, k16, v16, M, d_pos, 0, st);
  else {
    AppendArgs A{kv->view(layer), k16, v16, d_pos, M};
    A.in_bf16 = kv->opt_io_bf16;
    if (kv->r256()) launch_append256(A, st); else launch_append(A, st);
  }
}
void need_128(const yka_kv* kv) {
  if (kv->r256()) throw std::runtime_error("this entry point exists for head_dim 128 only");
}

// mode 0: attention + combine; 2: attention kernel alone.  k16/v16 != nullptr asks for quantize-on-append as well, which
// rides in the attention launch wherever a kernel stores its own rows (see the branches below).
struct Workspace { float* pm; float* pl; uint16_t* pacc16; size_t pairs; int* tickets; };
void do_attend(yka_kv* kv, int layer, const uint16_t* q16, int M, const int* d_pos, const uint8_t* depth, uint16_t* out16,
               hipStream_t st, int mode = 0, const uint16_t* k16 = nullptr, const uint16_t* v16 = nullptr, const Workspace* ws = nullptr) {
  const int NH = kv->cfg.n_heads;
  const Workspace W = ws ? *ws : Workspace{kv->pm, kv->pl, kv->pacc16, kWsPairs, kv->tickets};
  const int bf16 = kv->opt_io_bf16;                // type of the 16-bit rows that come in and of the outputs
  if (kv->tb) {
    // trellis-coded rows: the encoder runs first, in two launches (search, store); windows of up to kTbFuseRows rows launch
    // the search alone and the attention stores, decode launches nothing in front (see below).  Rows of at most 2 tokens
    // (or option key 3) run on row tiles of 2 tokens x 6 heads, wider slices on 128-row workgroups that decode every tile
    // once into LDS
    const yka_kv::Tb& T = *kv->tb;
    check_tb_layer(kv, layer);
    // decode without a depth table: the encoder's search rides in the attention launch, which leaves the new rows to the combiner
    const bool fuse = k16 && M <= 2 && !depth && mode == 0 && !kv->opt_force_narrow;
    const bool stores = k16 && M > 2 && M <= kTbFuseRows && !kv->opt_force_narrow;    // the wide kernel codes and stores the rows
    TbEncArgs E{};
    if (stores) launch_tb_search(E = tb_encoder_args(kv, layer, layer, k16, v16, 0, M, d_pos), st);
    else if (k16 && !fuse) do_append(kv, layer, k16, v16, M, d_pos, st);
    const int slice = slice256(kv, M);
    for (int s0 = 0; s0 < M; s0 += slice) {
      const Part256 P = part256(kv, M, s0, slice);
      TbAttnArgs A{T.kpay(layer), T.vpay(layer), T.kscl(layer), T.vscl(layer), kv->cfg.max_ctx, kv->cfg.n_kv_heads, T.stride,
                   T.pairs, T.gfac, T.has_mu ? T.mu : nullptr, layer, q16 + (size_t)s0 * NH * 256, d_pos, depth, P.Ms, s0, NH, P.S,
                   kv->pm, kv->pl, kv->pacc16, RowMap{}, bf16};
      A.rows_per_block = P.rows_per_block;
      CombineArgs C{kv->pm, kv->pl, kv->pacc16, P.S, P.Ms, NH, out16 + (size_t)s0 * NH * 256, kv->opt_unrot, bf16};
      A.s_short = C.s_short = P.s_short; C.d_pos = d_pos;
      if (stores) A.jobs = tb_jobs(E);
      if (fuse) {
        const TbEncArgs E = tb_encoder_args(kv, layer, layer, k16, v16, 0, M, d_pos);
        launch_tb_encode_attend(E, A, T.kb, st);
        launch_combine256_new(C, A, tb_jobs(E), T.kb, st);
        return;
      }
      if (P.narrow) launch_attend_tb(A, T.kb, st); else launch_attend_tb_wide(A, T.kb, st);
      if (mode != 2) launch_combine256(C, st);
    }
    return;
  }
  if (kv->r256()) {
    // 256-channel rows: rows of at most 2 tokens (or option key 3) run on row tiles of 2 tokens x 6 heads, one workgroup
    // per CU; wider slices on workgroups of 8 waves and up to 128 rows, one per CU.  Both kernels store the rows of a pass of
    // one slice themselves; a wide pass forced through the decode kernel and a pass of several slices launch the append first.
    const bool fuse256 = k16 && (M <= 2 || (M <= kMaxSlice && !kv->opt_force_narrow));
    if (k16 && !fuse256) do_append(kv, layer, k16, v16, M, d_pos, st);
    const int slice = slice256(kv, M);
    for (int s0 = 0; s0 < M; s0 += slice) {
      const Part256 P = part256(kv, M, s0, slice);
      AttnArgs A{kv->view(layer), q16 + (size_t)s0 * NH * 256, d_pos, depth, P.Ms, s0, NH, P.S, P.rows_per_block, kv->pm, kv->pl, kv->pacc16,
                 fuse256 ? k16 : nullptr, fuse256 ? v16 : nullptr};
      A.in_bf16 = bf16;
      if (P.narrow) launch_attend256(A, st); else launch_attend256_wide(A, st);
      if (mode != 2) launch_combine256(CombineArgs{kv->pm, kv->pl, kv->pacc16, P.S, P.Ms, NH, out16 + (size_t)s0 * NH * 256, kv->opt_unrot, bf16}, st);
    }
    return;
  }
  // quantize-on-append rides in the attention launch: in the decode kernel for rows of at most 2 tokens, in the wide
  // kernel for every 64-row slice (each slice stores its own rows); only a wide pass forced through the narrow kernel
  // launches the append kernel first
  // A pass of more than 64 rows is a prefill chunk (the reference cuts it into 64-row slices, engine35.cpp:935-947, one
  // attention launch each).  Here its rows are appended by one launch, then slices of up to 2048 tokens go through the
  // wide kernel - 128 rows per workgroup whatever the slice, the key range cut evenly into as many splits as the length
  // found on the device justifies - and one combiner launch per slice merges them.
  const bool chunk = M > kMaxSlice && !kv->opt_force_narrow && !ws;
  const bool fuse_append = k16 && !chunk && (M <= 2 || !kv->opt_force_narrow);
  if (k16 && !fuse_append) do_append(kv, layer, k16, v16, M, d_pos, st);
  const int slice = chunk ? (kv->opt_chunk_slice > 0 ? kv->opt_chunk_slice : kChunkSlice) : kMaxSlice;
  for (int s0 = 0; s0 < M; s0 += slice) {
    const int Ms = std::min(slice, M - s0);
    const bool narrow = !chunk && (Ms <= 2 || kv->opt_force_narrow);
    const bool mid = !chunk && !narrow && Ms <= kv->opt_mid_rows;
    const int S = narrow ? narrow_splits(kv, Ms, W.pairs) : mid ? mid_splits(kv, Ms, W.pairs) : (chunk ? chunk_splits(kv, Ms, kv->ws_rows) : wide_splits(kv, Ms, W.pairs));
    AttnArgs A{kv->view(layer), q16 + (size_t)s0 * NH * kD, d_pos, depth, Ms, s0, NH, S, wide_rows_per_block(Ms), W.pm, W.pl, W.pacc16,
               fuse_append ? k16 : nullptr, fuse_append ? v16 : nullptr};
    A.in_bf16 = bf16;
    CombineArgs C{W.pm, W.pl, W.pacc16, S, Ms, NH, out16 + (size_t)s0 * NH * kD, kv->opt_unrot, bf16};
    if (chunk && !kv->opt_splits_wide) {
      A.adapt = C.adapt = chunk_tile_cap(kv->cfg.n_kv_heads * ((kG * Ms + 127) / 128)); C.d_pos = d_pos; C.tok0 = s0; C.n_kv = kv->cfg.n_kv_heads; C.max_ctx = kv->cfg.max_ctx;
      if (!kv->opt_unrot && mode != 2) { A.out16 = C.out16; C.direct = 1; }
    }
    // option key 7, rows of at most 2 tokens: the last workgroup of each column merges the splits inside the attention launch
    const bool one_launch = narrow && mode == 0 && !kv->opt_unrot && kv->opt_merge_in_launch;
    if (one_launch) {
      // the counters are put back to zero by a fill kernel in front of every such launch: a launch that ended half way
      // (or anything else that left one non-zero) cannot make a later call skip its merge
      launch_zero_ints(W.tickets, kv->cfg.n_kv_heads * kMaxSlice, st);
      A.tickets = W.tickets; A.out16 = out16 + (size_t)s0 * NH * kD; A.out_bf16 = bf16;
    }
    if (narrow) launch_attend_narrow(A, st); else if (mid) launch_attend_mid(A, st); else if (chunk) launch_attend_chunk(A, st); else launch_attend_wide(A, st);
    if (mode != 2 && !one_launch && !(C.direct && S == 1)) launch_combine(C, st);
  }
}

// Multi-stream pass, 128-channel rows: splits per row the launch provides for.  Two workgroups per CU, one round, as long as
// whole splits of M rows fill it: streams of equal length get M times a whole number of workgroups, whatever the sharing-out.
// Where one and a half or two rounds are filled a seventh better the grid is launched for those, and the device decides by
// the streams' lengths which of the two it uses (ms_share; kMsLong).  us a pass, 512 / 768 / 1,024 workgroups provided:
//   48 streams of equal length  8,000 tokens 56.9 / 50.7 / 52.7   16,000 102 / 89.4 / 91.8   2,000 24.6 / 24.8 / 26.1
//   48 streams, a sixteenth up to 16,000 tokens 50.8 / 40.8 / 42.4   8,000 32.9 / 29.2 / 29.8   4,000 21.5 / 21.5 / 22.8
//   33 streams of equal length 16,000 tokens 71.5 / 70.5 / 66.9   4,000 27.4 / 27.7 / 28.8
// (before the sharing-out, 1,024 workgroups: 90.8 us for the 48 of 16,000, 65.7 for the 33)
struct MsGrid { int S, in_short; };
MsGrid ms_grid(const yka_kv* kv, int M) {
  const int per = kv->cfg.n_kv_heads * M, S = std::max(2, std::min(kMaxSplits, 512 / per));
  int best = S;
  double fill = 1.15 * std::min(1.0, S * per / 512.0);
  for (const int wgs : {768, 1024}) {
    const int s = wgs / per;
    if (s > S && s * per / (double)wgs >= fill) { fill = s * per / (double)wgs; best = s; }
  }
  const int fits = (int)(kWsPairs / (size_t)M);
  return {std::min({best, kMaxSplits, fits}), best > S ? std::min(S, fits) * M : 0};
}

// Multi-stream pass: rows are appended (several rows of one stream may follow each other and read each other's keys) by the
// attention launch or, beyond 64 rows and with a split count set by the caller, by a launch in front of it; every row
// attends to keys [0, pos[t]] of its own container.  One token per workgroup column.
void do_attend_ms(yka_kv* kv, const uint16_t* q16, const uint16_t* k16, const uint16_t* v16, int M, const int* row_pos,
                  const int* row_slot, uint16_t* out16, hipStream_t st) {
  const int NH = kv->cfg.n_heads, D = kv->D();
  const int share = !kv->opt_splits_narrow;        // the splits follow the streams' lengths (ms_share) unless the caller set their number
  const bool r256 = kv->r256();
  const int bf16 = kv->opt_io_bf16;
  if (kv->tb) {
    // trellis-coded rows: every container is a stream of the layer option key 6 names; its groups code and decode the rows
    const yka_kv::Tb& T = *kv->tb;
    const int pl = kv->opt_profile_layer;
    check_tb_layer(kv, pl);
    const RowMap R{row_pos, row_slot, kv->cfg.n_layers, T.layer_bytes, 0};
    if (k16) tb_append(kv, pl, nullptr, nullptr, k16, v16, M, nullptr, 0, st, 0, &R);
    for (int s0 = 0; s0 < M; s0 += kMaxSlice) {
      const int Ms = std::min(kMaxSlice, M - s0);
      int S = kv->opt_splits_narrow > 0 ? kv->opt_splits_narrow : 512 / (kv->cfg.n_kv_heads * Ms);
      S = std::min(std::max(2, std::min(kMaxSplits, S)), (int)(kWsPairs / (size_t)Ms));
      RowMap Rs = R; Rs.pos += s0; Rs.slot += s0;
      const TbAttnArgs A{T.kpay(0), T.vpay(0), T.kscl(0), T.vscl(0), kv->cfg.max_ctx, kv->cfg.n_kv_heads, T.stride,
                         T.pairs, T.gfac, T.has_mu ? T.mu : nullptr, pl, q16 + (size_t)s0 * NH * 256, nullptr, nullptr, Ms, s0, NH, S,
                         kv->pm, kv->pl, kv->pacc16, Rs, bf16, share, kv->ms_plan};
      launch_attend_tb(A, T.kb, st);
      CombineArgs C{kv->pm, kv->pl, kv->pacc16, S, Ms, NH, out16 + (size_t)s0 * NH * 256, kv->opt_unrot, bf16};
      if (share) C.plan = kv->ms_plan;
      launch_combine256(C, st);
    }
    return;
  }
  const RowMap R{row_pos, row_slot, kv->cfg.n_layers, kv->layer_bytes, kv->n_pages};
  // passes of at most 64 rows store their rows inside the attention launch (ms_new_rows)
  const bool one_launch = !r256 && !kv->opt_unrot && kv->opt_merge_in_launch;
  const bool fuse = k16 && share && !one_launch && M <= kMaxSlice;
  if (k16 && !fuse) { AppendArgs P{kv->view(0), k16, v16, nullptr, M, R}; P.in_bf16 = bf16; if (r256) launch_append256(P, st); else launch_append(P, st); }
  for (int s0 = 0; s0 < M; s0 += kMaxSlice) {
    const int Ms = std::min(kMaxSlice, M - s0);
    int S = kv->opt_splits_narrow > 0 ? kv->opt_splits_narrow : 512 / (kv->cfg.n_kv_heads * Ms);   // two workgroups per CU: one round
    S = std::min(std::max(2, std::min(kMaxSplits, S)), (int)(kWsPairs / (size_t)Ms));
    const MsGrid G = share && !one_launch && !r256 ? ms_grid(kv, Ms) : MsGrid{S, 0};
    S = G.S;
    RowMap Rs = R; Rs.pos += s0; Rs.slot += s0;
    AttnArgs A{kv->view(0), q16 + (size_t)s0 * NH * D, nullptr, nullptr, Ms, s0, NH, S, 128, kv->pm, kv->pl, kv->pacc16, nullptr, nullptr, Rs};
    A.in_bf16 = bf16;
    CombineArgs C{kv->pm, kv->pl, kv->pacc16, S, Ms, NH, out16 + (size_t)s0 * NH * D, kv->opt_unrot, bf16};
    if (share && !one_launch) { A.adapt = 1; A.ms_short = G.in_short; A.plan = kv->ms_plan; C.plan = kv->ms_plan; }
    if (fuse) { A.k16 = k16; A.v16 = v16; }
    if (r256) { launch_attend256(A, st); launch_combine256(C, st); }
    else if (one_launch) {
      launch_zero_ints(kv->tickets, kv->cfg.n_kv_heads * kMaxSlice, st);
      A.tickets = kv->tickets; A.out16 = C.out16; A.out_bf16 = bf16; launch_attend_narrow(A, st);
    }
    else { launch_attend_narrow(A, st); launch_combine(C, st); }
  }
}

}  // namespace

#define YKA_TRY try {
#define YKA_CATCH_INT                                                   \
  return 0; }                                                           \
  catch (const std::exception& e) { g_err = e.what(); return -1; }      \
  catch (...) { g_err = "unknown error"; return -1; }

extern "C" {

const char* yka_last_error(void) { return g_err.c_str(); }

const char* yka_build_info(void) {
  static const std::string s = [] {
    char b[128];
    snprintf(b, sizeof b, "hip=%d;arch=gfx950;page_bytes=%d;page_tokens=%d", HIP_VERSION, kPageBytes, kPageTok);
    return std::string(b);
  }();
  return s.c_str();
}

yka_kv* yka_kv_open(const yka_kv_config* cfg) {
  yka_kv* kv = nullptr;
  try {
    if (!cfg) throw std::runtime_error("null config");
    if (cfg->head_dim != kD && cfg->head_dim != 256) throw std::runtime_error("head_dim must be 128 (int4 in 32-channel groups) or 256 (the reference's own rows)");
    if (cfg->n_kv_heads < 1 || cfg->n_heads != cfg->n_kv_heads * kG) throw std::runtime_error("n_heads must be 6 * n_kv_heads");
    if (cfg->n_layers < 1) throw std::runtime_error("n_layers must be >= 1");
    if (cfg->max_ctx < kPageTok || cfg->max_ctx % kPageTok) throw std::runtime_error("max_ctx must be a positive multiple of 256");
    if (cfg->max_rows < 1 || cfg->max_rows > 8192) throw std::runtime_error("max_rows must be in [1, 8192]");
    {
      // sizes are 64-bit products of four caller-given ints: refuse what cannot exist before one of them wraps around
      if (cfg->n_kv_heads > 1024) throw std::runtime_error("n_kv_heads must be at most 1024");
      const unsigned __int128 per_token = cfg->head_dim == 256 ? (unsigned __int128)kPage256Bytes / kPageTok * cfg->n_kv_heads
                                                                 : (unsigned __int128)kv_page_bytes(cfg->n_kv_heads) / kPageTok;
      if (per_token * (unsigned __int128)cfg->max_ctx * (unsigned __int128)cfg->n_layers > ((unsigned __int128)1 << 40))
        throw std::runtime_error("n_layers x max_ctx x n_kv_heads describes a cache of more than 1 TiB");
    }
    int ndev = 0;
    HIPCHK(hipGetDeviceCount(&ndev));
    if (cfg->device < 0 || cfg->device >= ndev) throw std::runtime_error("device out of range");
    HIPCHK(hipSetDevice(cfg->device));
    if (cfg->device < kMaxDevices) (void)static_workspace(cfg->device);   // address of this device's static workspace, looked up once per device
    kv = new yka_kv();
    kv->cfg = *cfg;
    kv->n_pages = cfg->max_ctx / kPageTok;
    kv->layer_bytes = cfg->head_dim == 256 ? (size_t)kv->n_pages * cfg->n_kv_heads * kPage256Bytes : (size_t)kv->n_pages * kv_page_bytes(cfg->n_kv_heads);
    HIPCHK(hipMalloc((void**)&kv->pool, kv->layer_bytes * cfg->n_layers));
    HIPCHK(hipMemset(kv->pool, 0, kv->layer_bytes * cfg->n_layers));   // zero scales: unwritten rows decode to finite values
    if (cfg->paged) {
      std::vector<int32_t> ident((size_t)cfg->n_layers * kv->n_pages);
      for (size_t i = 0; i < ident.size(); ++i) ident[i] = (int32_t)(i % kv->n_pages);
      HIPCHK(hipMalloc((void**)&kv->tables, ident.size() * 4));
      HIPCHK(hipMemcpy(kv->tables, ident.data(), ident.size() * 4, hipMemcpyHostToDevice));
    }
    kv->ws_rows = kChunkPairs;                     // the bound the demand is taken under
    kv->ws_rows = ws_pairs_of(kv);
    const size_t np = kv->ws_rows * cfg->n_heads;
    HIPCHK(hipMalloc((void**)&kv->pm, np * 4));
    HIPCHK(hipMalloc((void**)&kv->pl, np * 4));
    HIPCHK(hipMalloc((void**)&kv->pacc16, np * cfg->head_dim * 2));
    HIPCHK(hipMalloc((void**)&kv->tickets, (size_t)cfg->n_kv_heads * kMaxSlice * 4));   // one counter per (kv head, row tile); zero between launches
    HIPCHK(hipMemset(kv->tickets, 0, (size_t)cfg->n_kv_heads * kMaxSlice * 4));
    HIPCHK(hipMalloc((void**)&kv->ms_plan, kMaxSlice * sizeof(int2)));
    HIPCHK(hipMalloc((void**)&kv->d_pos, 4));
    HIPCHK(hipMemset(kv->d_pos, 0, 4));
    HIPCHK(hipStreamCreateWithFlags(&kv->stream, hipStreamNonBlocking));
    HIPCHK(hipDeviceSynchronize());
    return kv;
  } catch (const std::exception& e) {
    g_err = e.what();
  } catch (...) { g_err = "unknown error"; }
  if (kv) yka_kv_close(kv);
  return nullptr;
}

void yka_kv_close(yka_kv* kv) {
  if (!kv) return;
  (void)hipSetDevice(kv->cfg.device);
  (void)hipDeviceSynchronize();
  if (kv->stream) (void)hipStreamDestroy(kv->stream);
  if (kv->tb) {
    (void)hipFree(kv->tb->pairs); (void)hipFree(kv->tb->gfac); (void)hipFree(kv->tb->mu); (void)hipFree(kv->tb->pool);
    (void)hipFree(kv->tb->scr); (void)hipFree(kv->tb->stage);
    delete kv->tb;
  }
  (void)hipFree(kv->pool); (void)hipFree(kv->tables); (void)hipFree(kv->pm); (void)hipFree(kv->pl); (void)hipFree(kv->pacc16); (void)hipFree(kv->d_pos); (void)hipFree(kv->tickets); (void)hipFree(kv->ms_plan);
  delete kv;
}

int yka_set_opt(yka_kv* kv, int key, int value) {
  YKA_TRY
  if (!kv) throw std::runtime_error("null handle");
  switch (key) {
    case 1: if (value < 0 || value > kMaxSplits) throw std::runtime_error("splits must be in [0, 256]"); kv->opt_splits_narrow = value; break;
    case 2: if (value < 0 || value > kMaxSplits) throw std::runtime_error("splits must be in [0, 256]"); kv->opt_splits_wide = value; break;
    case 3: kv->opt_force_narrow = value != 0; break;
    case 4: kv->opt_unrot = value != 0; break;
    case 5: if (value < 0) throw std::runtime_error("context hint must be >= 0"); kv->opt_ctx_hint = value; break;
    case 6: if (value < 0) throw std::runtime_error("profile layer must be >= 0"); kv->opt_profile_layer = value; break;
    case 7: kv->opt_merge_in_launch = value != 0; break;
    case 8: if (value < 0 || value > kMaxSlice) throw std::runtime_error("widest window of the mid kernel must be in [0, 64]"); kv->opt_mid_rows = value; break;
    case 9: if (value < 0 || value > kMaxSplits) throw std::runtime_error("splits must be in [0, 256]"); kv->opt_splits_mid = value; break;
    case 11: if (value != 0 && value != 1) throw std::runtime_error("row type must be 0 (fp16) or 1 (bf16)"); kv->opt_io_bf16 = value; break;
    case 10: if (value != 0 && (value < 128 || value > kMaxChunkSlice)) throw std::runtime_error("prefill slice must be 0 or in [128, 4096] tokens"); kv->opt_chunk_slice = value; break;
    default: throw std::runtime_error("unknown option key");
  }
  YKA_CATCH_INT
}

int yka_kv_set_page_table(yka_kv* kv, int layer, const int32_t* h_table, int n_pages) {
  YKA_TRY
  on_device(kv);
  if (!kv->cfg.paged) throw std::runtime_error("handle was opened in contiguous mode");
  if (!h_table || n_pages != kv->n_pages) throw std::runtime_error("page table must have max_ctx/256 entries");
  if (layer < -1 || layer >= kv->cfg.n_layers) throw std::runtime_error("layer out of range");
  std::vector<char> seen((size_t)n_pages, 0);
  for (int p = 0; p < n_pages; ++p) {
    if (h_table[p] < 0 || h_table[p] >= n_pages || seen[(size_t)h_table[p]]) throw std::runtime_error("page table is not a permutation");
    seen[(size_t)h_table[p]] = 1;
  }
  HIPCHK(hipDeviceSynchronize());
  for (int l = 0; l < kv->cfg.n_layers; ++l)
    if (layer < 0 || l == layer) HIPCHK(hipMemcpy(kv->tables + (size_t)l * n_pages, h_table, (size_t)n_pages * 4, hipMemcpyHostToDevice));
  YKA_CATCH_INT
}

int yka_append(yka_kv* kv, int layer, const uint16_t* d_k16, const uint16_t* d_v16, int M, const int* d_pos, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!d_k16 || !d_v16 || !d_pos) throw std::runtime_error("null pointer");
  do_append(kv, layer, d_k16, d_v16, M, d_pos, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_attend(yka_kv* kv, int layer, const uint16_t* d_q16, int M, const int* d_pos, const uint8_t* d_depth,
               uint16_t* d_out16, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!d_q16 || !d_pos || !d_out16) throw std::runtime_error("null pointer");
  do_attend(kv, layer, d_q16, M, d_pos, d_depth, d_out16, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_append_attend(yka_kv* kv, int layer, const uint16_t* d_q16, const uint16_t* d_k16, const uint16_t* d_v16, int M,
                      const int* d_pos, const uint8_t* d_depth, uint16_t* d_out16, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!d_q16 || !d_k16 || !d_v16 || !d_pos || !d_out16) throw std::runtime_error("null pointer");
  do_attend(kv, layer, d_q16, M, d_pos, d_depth, d_out16, (hipStream_t)hip_stream, 0, d_k16, d_v16);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_append_attend_static(yka_kv* kv, int layer, const uint16_t* d_q16, const uint16_t* d_k16, const uint16_t* d_v16, int M,
                             const int* d_pos, const uint8_t* d_depth, uint16_t* d_out16, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); need_128(kv);
  if (!d_q16 || !d_k16 || !d_v16 || !d_pos || !d_out16) throw std::runtime_error("null pointer");
  if (M < 1 || M > kMaxSlice || M > kv->cfg.max_rows) throw std::runtime_error("the static workspace serves passes of 1 to 64 rows");
  if ((size_t)kv->cfg.n_heads > kStaticHeads) throw std::runtime_error("the static workspace is sized for at most 24 query heads");
  unsigned char* base = kv->cfg.device < kMaxDevices ? g_static_ptr[kv->cfg.device] : nullptr;   // looked up when the handle was opened on this device
  if (!base) throw std::runtime_error("the static workspace of this device has no address");
  const Workspace W{reinterpret_cast<float*>(base), reinterpret_cast<float*>(base + kStaticPmBytes),
                    reinterpret_cast<uint16_t*>(base + 2 * kStaticPmBytes), kStaticPairs * kStaticHeads / (size_t)kv->cfg.n_heads,
                    reinterpret_cast<int*>(base + kStaticWsBytes - kStaticTicketBytes)};   // 24 heads = 4 kv heads x 64 row tiles of tickets at most
  do_attend(kv, layer, d_q16, M, d_pos, d_depth, d_out16, (hipStream_t)hip_stream, 0, d_k16, d_v16, &W);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_kv_poison_workspace(yka_kv* kv) {
  YKA_TRY
  on_device(kv);
  HIPCHK(hipDeviceSynchronize());
  const size_t rows = kv->ws_rows * (size_t)kv->cfg.n_heads;
  HIPCHK(hipMemset(kv->pm, 0xff, rows * 4));
  HIPCHK(hipMemset(kv->pl, 0xff, rows * 4));
  HIPCHK(hipMemset(kv->pacc16, 0xff, rows * (size_t)kv->D() * 2));
  HIPCHK(hipMemset(kv->ms_plan, 0xff, kMaxSlice * sizeof(int2)));
  HIPCHK(hipDeviceSynchronize());
  YKA_CATCH_INT
}

int yka_append_attend_ms(yka_kv* kv, const uint16_t* d_q16, const uint16_t* d_k16, const uint16_t* d_v16, int M,
                         const int* d_row_pos, const int* d_row_slot, uint16_t* d_out16, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_rows(kv, M);
  if (!d_q16 || !d_row_pos || !d_row_slot || !d_out16) throw std::runtime_error("null pointer");
  if ((d_k16 == nullptr) != (d_v16 == nullptr)) throw std::runtime_error("new K and V rows come together or not at all");
  do_attend_ms(kv, d_q16, d_k16, d_v16, M, d_row_pos, d_row_slot, d_out16, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_ms_call_host(yka_kv* kv, const uint16_t* q16, const uint16_t* k16, const uint16_t* v16, int M, const int32_t* row_pos,
                     const int32_t* row_slot, uint16_t* out16) {
  YKA_TRY
  on_device(kv); check_rows(kv, M);
  if (!q16 || !row_pos || !row_slot || !out16) throw std::runtime_error("null pointer");
  if ((k16 == nullptr) != (v16 == nullptr)) throw std::runtime_error("new K and V rows come together or not at all");
  const size_t nq = (size_t)M * kv->cfg.n_heads * kv->D(), nk = (size_t)M * kv->cfg.n_kv_heads * kv->D();
  DevBuf dq(nq * 2), dk(nk * 2), dv(nk * 2), dout(nq * 2), dp((size_t)M * 4), dsl((size_t)M * 4);
  HIPCHK(hipMemcpy(dq.p, q16, nq * 2, hipMemcpyHostToDevice));
  if (k16) { HIPCHK(hipMemcpy(dk.p, k16, nk * 2, hipMemcpyHostToDevice)); HIPCHK(hipMemcpy(dv.p, v16, nk * 2, hipMemcpyHostToDevice)); }
  HIPCHK(hipMemcpy(dp.p, row_pos, (size_t)M * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dsl.p, row_slot, (size_t)M * 4, hipMemcpyHostToDevice));
  do_attend_ms(kv, dq.as<uint16_t>(), k16 ? dk.as<uint16_t>() : nullptr, k16 ? dv.as<uint16_t>() : nullptr, M, dp.as<int>(), dsl.as<int>(),
               dout.as<uint16_t>(), kv->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(kv->stream));
  HIPCHK(hipMemcpy(out16, dout.p, nq * 2, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_codec_probe(const uint16_t* x16, int rows, uint8_t* codes, uint16_t* scales, float* y) {
  YKA_TRY
  if (!x16 || !codes || !scales || !y || rows < 1) throw std::runtime_error("bad argument");
  const size_t n = (size_t)rows * kD;
  DevBuf dx(n * 2), dc(n / 2), ds((size_t)rows * kNG * 2), dy(n * 4);
  HIPCHK(hipMemcpy(dx.p, x16, n * 2, hipMemcpyHostToDevice));
  launch_codec_probe(dx.as<uint16_t>(), rows, dc.as<uint8_t>(), ds.as<uint16_t>(), dy.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(codes, dc.p, n / 2, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(scales, ds.p, (size_t)rows * kNG * 2, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(y, dy.p, n * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

static void check_post(const yka_kv* kv, const yka_post_params* P) {
  if (!P) throw std::runtime_error("null parameter block");
  if (!P->d_qn_w16 || !P->d_kn_w16) throw std::runtime_error("null norm weights");
  if (P->rope_dims < 0 || P->rope_dims > kv->D() || (P->rope_dims & 1)) throw std::runtime_error("rope_dims must be even and in [0, head_dim]");
  if (P->rope_dims > 0 && (!P->d_rope || P->rope_rows < 1)) throw std::runtime_error("rotary table missing");
}

int yka_attn_post(yka_kv* kv, int layer, const float* d_xq, const float* d_xk, const float* d_xv, int M, const int* d_pos,
                  const yka_post_params* P, uint16_t* d_q16, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M); check_post(kv, P);
  if (!d_xq || !d_xk || !d_xv || !d_pos || !d_q16) throw std::runtime_error("null pointer");
  if ((P->d_xgate == nullptr) != (P->d_gate16 == nullptr)) throw std::runtime_error("the gate projection and its output come together or not at all");
  PostArgs A{kv->view(layer), d_xq, d_xk, d_xv, M, kv->cfg.n_heads, d_pos, P->d_qn_w16, P->d_kn_w16, P->eps,
             P->d_rope, P->rope_dims, P->rope_rows, P->rotate != 0, d_q16};
  A.xgate = P->d_xgate; A.gate16 = P->d_gate16; A.io_bf16 = kv->opt_io_bf16;
  post_launch(kv, layer, A, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_attn_post_host(yka_kv* kv, int layer, const float* xq, const float* xk, const float* xv, int M, int pos,
                       const uint16_t* qn_w16, const uint16_t* kn_w16, float eps, const float* rope, int rope_dims,
                       int rope_rows, int rotate, uint16_t* q16, const float* xgate, uint16_t* gate16) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!xq || !xk || !xv || !qn_w16 || !kn_w16 || !q16) throw std::runtime_error("null pointer");
  if (pos < 0 || (long long)pos + M > kv->cfg.max_ctx) throw std::runtime_error("rows outside the container");
  const int kD = kv->D();                          // 128 or 256 channels per head
  if (rope_dims < 0 || rope_dims > kD || (rope_dims & 1)) throw std::runtime_error("rope_dims must be even and in [0, head_dim]");
  if (rope_dims > 0 && (!rope || rope_rows < pos + M)) throw std::runtime_error("rotary table shorter than pos + M");
  const size_t nq = (size_t)M * kv->cfg.n_heads * kD, nk = (size_t)M * kv->cfg.n_kv_heads * kD;
  const size_t nr = rope_dims > 0 ? (size_t)rope_rows * rope_dims : 1;
  if ((xgate == nullptr) != (gate16 == nullptr)) throw std::runtime_error("the gate projection and its output come together or not at all");
  DevBuf dq(nq * 4), dk(nk * 4), dv(nk * 4), dqw((size_t)kD * 2), dkw((size_t)kD * 2), dr(nr * 4), dq16(nq * 2), dg(xgate ? nq * 4 : 4), dg16(xgate ? nq * 2 : 4);
  if (xgate) HIPCHK(hipMemcpy(dg.p, xgate, nq * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dq.p, xq, nq * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dk.p, xk, nk * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dv.p, xv, nk * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dqw.p, qn_w16, kD * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dkw.p, kn_w16, kD * 2, hipMemcpyHostToDevice));
  if (rope_dims > 0) HIPCHK(hipMemcpy(dr.p, rope, nr * 4, hipMemcpyHostToDevice));
  yka_post_params P{dqw.as<uint16_t>(), dkw.as<uint16_t>(), eps, dr.as<float>(), rope_dims, rope_rows, rotate, nullptr, nullptr};
  check_post(kv, &P);
  launch_set_int(kv->d_pos, pos, kv->stream);
  PostArgs A{kv->view(layer), dq.as<float>(), dk.as<float>(), dv.as<float>(), M, kv->cfg.n_heads, kv->d_pos,
             P.d_qn_w16, P.d_kn_w16, eps, P.d_rope, rope_dims, rope_rows, rotate != 0, dq16.as<uint16_t>()};
  if (xgate) { A.xgate = dg.as<float>(); A.gate16 = dg16.as<uint16_t>(); }
  A.io_bf16 = kv->opt_io_bf16;
  post_launch(kv, layer, A, kv->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(kv->stream));
  HIPCHK(hipMemcpy(q16, dq16.p, nq * 2, hipMemcpyDeviceToHost));
  if (xgate) HIPCHK(hipMemcpy(gate16, dg16.p, nq * 2, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_kvx256_probe(const float* x, int rows, int mode, int rot, int8_t* q8, uint32_t* words, float* scales, float* y) {
  YKA_TRY
  if (!x || !scales || !y || rows < 1 || (mode != 0 && mode != 1)) throw std::runtime_error("bad argument");
  if ((mode == 0 && !q8) || (mode == 1 && !words)) throw std::runtime_error("the output array of the selected mode is null");
  const size_t n = (size_t)rows * 256;
  DevBuf dx(n * 4), dq(mode == 0 ? n : 4), dw(mode == 1 ? (size_t)rows * 128 : 4), ds((size_t)rows * 4), dy(n * 4);
  HIPCHK(hipMemcpy(dx.p, x, n * 4, hipMemcpyHostToDevice));
  launch_row256_encode(dx.as<float>(), rows, mode, rot != 0, dq.as<int8_t>(), dw.as<uint32_t>(), ds.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  launch_row256_decode(rows, mode, rot != 0, dq.as<int8_t>(), dw.as<uint32_t>(), ds.as<float>(), dy.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  if (mode == 0) HIPCHK(hipMemcpy(q8, dq.p, n, hipMemcpyDeviceToHost));
  else HIPCHK(hipMemcpy(words, dw.p, (size_t)rows * 128, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(scales, ds.p, (size_t)rows * 4, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(y, dy.p, n * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

// ---- trellis-coded rows ----
}  // extern "C"
namespace {
struct TbInfo { int nm = 0, ngrp = 0, layers = 0, kv_heads = 0, tables = 0; bool has_trellis = false; };
// the checks of the reference's loaders (src/engine35.cpp:48-52, src/kvq_fast.hpp:52-76) plus bounds on every record
// Little-endian view of a profile blob: a 100-byte header, then three offset arrays (multipliers, tables, groups).
struct BlobView {
  const uint8_t* p; size_t n;
  unsigned half(size_t at) const { return (unsigned)p[at] + 256u * (unsigned)p[at + 1]; }
  uint32_t word(size_t at) const { return (uint32_t)half(at) + 65536u * (uint32_t)half(at + 2); }
  int table_int(size_t rec, int state) const { return (int)(int16_t)half(rec + 12 + 2 * (size_t)state); }
  size_t multipliers() const { return word(32); }
  size_t table_record(unsigned t) const { return word((size_t)word(36) + 4 * (size_t)t); }
  size_t group_record(int g) const { return word((size_t)word(40) + 4 * (size_t)g); }
};
TbInfo tb_check_blob(const uint8_t* b, size_t n) {
  auto bad = [](const char* what) { throw std::runtime_error(what); };
  if (!b || n < 100 || std::memcmp(b, "KVQP", 4) != 0) bad("not a KVQP v1 profile blob");
  const BlobView V{b, n};
  if (V.half(4) != 1 || V.word(8) != n) bad("not a KVQP v1 profile blob");
  if (V.half(16) != 256) bad("profile blob: rows must have 256 elements");
  TbInfo I;
  I.layers = (int)V.half(18); I.kv_heads = (int)V.half(20); I.nm = (int)V.half(24);
  const size_t n_grp = V.word(28);                       // checked as an unsigned count before it becomes an int
  const unsigned n_tab = V.half(22);
  I.tables = (int)n_tab;
  if (I.nm < 1 || I.nm > 16) bad("profile blob: bad scale-multiplier count");
  if (V.multipliers() + 4 * (size_t)I.nm > n || (size_t)V.word(36) + 4 * (size_t)n_tab > n || (size_t)V.word(40) + 4 * n_grp > n)
    bad("profile blob: offsets outside the blob");
  I.ngrp = (int)n_grp;                                   // < n / 4 <= 2^30
  for (unsigned t = 0; t < n_tab; ++t) {
    const size_t rec = V.table_record(t);
    if (rec + 12 + 512 > n || b[rec] != 8 || b[rec + 2] != 64 || b[rec + 3] != 8) bad("profile blob: tables must have 8 state bits, chunks of 64");
    for (int st = 0; st < 256; ++st)
      if (std::abs(V.table_int(rec, st)) > 1100) bad("profile blob: table value out of range");
  }
  for (int g = 0; g < I.ngrp; ++g) {
    const size_t rec = V.group_record(g);
    if (rec + 8 > n) bad("profile blob: group record outside the blob");
    const unsigned mode = b[rec], bits = b[rec + 1], table = b[rec + 2], ndir = b[rec + 4];
    const size_t tail = (b[rec + 5] ? 512u : 0u) + 512u * (size_t)ndir;
    if (mode > 1 || ndir > 2 || rec + 8 + tail > n) bad("profile blob: bad group record");
    if (mode != 0) continue;
    if (bits < 3 || bits > 5 || table >= n_tab) bad("profile blob: trellis groups need 3..5 bits and a table");
    I.has_trellis = true;
  }
  return I;
}
// What the encoder kernels would otherwise look up in the blob by four dependent loads (layout: TbProbeArgs::desc): a
// record per group, then every table as aligned int16.  The blob has passed tb_check_blob.
std::vector<uint32_t> tb_descriptors(const uint8_t* b, size_t n, const TbInfo& I) {
  const BlobView V{b, n};
  const size_t rec_words = 8 * (size_t)I.ngrp;
  std::vector<uint32_t> D(rec_words + 128 * (size_t)I.tables, 0u);
  for (int t = 0; t < I.tables; ++t) {
    const size_t rec = V.table_record((unsigned)t);
    for (int st = 0; st < 256; st += 2)
      D[rec_words + 128 * (size_t)t + st / 2] = (uint32_t)(uint16_t)V.table_int(rec, st) | ((uint32_t)(uint16_t)V.table_int(rec, st + 1) << 16);
  }
  for (int g = 0; g < I.ngrp; ++g) {
    const size_t rec = V.group_record(g);
    uint32_t* d = &D[8 * (size_t)g];
    const bool has_mean = b[rec + 5] != 0, trellis = b[rec] == 0;
    d[0] = (uint32_t)b[rec] | ((uint32_t)b[rec + 1] << 8) | ((uint32_t)b[rec + 2] << 16) | ((uint32_t)b[rec + 3] << 24);
    d[1] = (uint32_t)b[rec + 4] | ((uint32_t)has_mean << 8);
    d[2] = (uint32_t)(rec + 8);
    d[3] = (uint32_t)(rec + 8 + (has_mean ? 512 : 0));
    if (trellis) {
      d[4] = (uint32_t)(2 * (rec_words + 128 * (size_t)b[rec + 2]));            // in int16 units from the start of D
      std::memcpy(&d[5], b + V.table_record(b[rec + 2]) + 4, 4);                 // gain
    }
  }
  return D;
}
}  // namespace
extern "C" {

int yka_tb_pack_unpack(const uint8_t* blob, size_t blob_len, const float* x, const int* grp, const int* pos, int rows, int stride,
                       float* y_fq, uint8_t* pay, uint32_t* side, float* y_dec, float* ms_out) {
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
  struct EvGuard { hipEvent_t* e; ~EvGuard() { for (int i = 0; i < 3; ++i) if (e[i]) (void)hipEventDestroy(e[i]); } } ev_guard{ev};
  YKA_TRY
  if (!x || !grp || !pos || rows < 1 || !y_fq || !pay || !side || !y_dec) throw std::runtime_error("bad argument");
  if (stride < 160 || stride > 1024 || stride % 4) throw std::runtime_error("stride must be a multiple of 4 in [160, 1024]");
  const TbInfo I = tb_check_blob(blob, blob_len);
  const std::vector<uint32_t> desc = tb_descriptors(blob, blob_len, I);   // host work first: nothing is allocated for a bad blob
  constexpr int kTile = 1024;                        // rows per launch
  const size_t nx = (size_t)rows * 256, w_ofs = (size_t)kTile * I.nm * 256;
  DevBuf db(blob_len), dx(nx * 4), dg((size_t)rows * 4), dp((size_t)rows * 4), dy(nx * 4), dpay((size_t)rows * stride), dside((size_t)rows * 8),
         dd(nx * 4), scr(w_ofs + (size_t)kTile * I.nm * 32);
  HIPCHK(hipMemcpy(db.p, blob, blob_len, hipMemcpyHostToDevice));
  DevBuf dd_desc(desc.size() * 4);
  HIPCHK(hipMemcpy(dd_desc.p, desc.data(), desc.size() * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dx.p, x, nx * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dg.p, grp, (size_t)rows * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dp.p, pos, (size_t)rows * 4, hipMemcpyHostToDevice));
  for (int i = 0; i < 3; ++i) HIPCHK(hipEventCreate(&ev[i]));
  HIPCHK(hipEventRecord(ev[0], nullptr));
  for (int r0 = 0; r0 < rows; r0 += kTile) {
    TbProbeArgs A{};
    A.blob = db.as<uint8_t>(); A.nm = I.nm; A.has_trellis = I.has_trellis;
    A.desc = dd_desc.as<uint32_t>(); A.ngrp = I.ngrp; A.mult_off = BlobView{blob, blob_len}.word(32);
    A.yin = dx.as<float>(); A.grp = dg.as<int>(); A.pos = dp.as<int>(); A.row0 = r0; A.nrow = std::min(kTile, rows - r0);
    A.yout = dy.as<float>(); A.side = dside.as<uint32_t>(); A.scr = scr.as<uint8_t>(); A.scr_w_ofs = w_ofs;
    A.pay = dpay.as<uint8_t>(); A.stride = stride;
    launch_tb_probe(A, nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());                  // the scratch block is reused by the next tile
  }
  HIPCHK(hipEventRecord(ev[1], nullptr));
  launch_tb_unpack(db.as<uint8_t>(), dg.as<int>(), dp.as<int>(), dpay.as<uint8_t>(), dside.as<uint32_t>(), stride, dx.as<float>(), dd.as<float>(), rows, nullptr);
  HIPCHK(hipEventRecord(ev[2], nullptr));
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  if (ms_out) {                                        // encode and unpack times, as the reference's hook reports them (kvx_probe.cu:160)
    HIPCHK(hipEventElapsedTime(&ms_out[0], ev[0], ev[1]));
    HIPCHK(hipEventElapsedTime(&ms_out[1], ev[1], ev[2]));
  }
  HIPCHK(hipMemcpy(y_fq, dy.p, nx * 4, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(pay, dpay.p, (size_t)rows * stride, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(side, dside.p, (size_t)rows * 8, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(y_dec, dd.p, nx * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

static uint16_t int_to_f16_bits(int v) {               // |v| <= 2048: exact
  if (v == 0) return 0;
  const unsigned a = (unsigned)(v < 0 ? -v : v);
  int e = 31 - __builtin_clz(a);                       // a = 1.xxx * 2^e, e <= 11
  const unsigned mant = (a << (10 - e)) & 0x3ffu;      // e <= 10 for a < 2048; a == 2048: e = 11, mant 0
  return (uint16_t)((v < 0 ? 0x8000u : 0u) | ((unsigned)(e + 15) << 10) | (e <= 10 ? mant : 0u));
}

int yka_kv_set_profile(yka_kv* kv, const uint8_t* blob, size_t blob_len) {
  YKA_TRY
  on_device(kv);
  if (!kv->r256()) throw std::runtime_error("trellis-coded rows need a handle opened with head_dim 256");
  if (kv->cfg.paged) throw std::runtime_error("trellis-coded rows are not available in paged mode");
  if (kv->tb) throw std::runtime_error("the handle already has a profile");
  const TbInfo I = tb_check_blob(blob, blob_len);
  // The profile's layers are model layers.  A handle's containers are model layers too in single-stream use (a call then
  // names a layer the profile must have) or the streams of ONE layer in multi-stream passes (option key 6 names it).
  const int n_kv = kv->cfg.n_kv_heads;
  if (I.kv_heads != n_kv || I.ngrp < n_kv * 2) throw std::runtime_error("the profile does not cover the kv heads of the handle");
  const int need = (I.ngrp / (n_kv * 2)) * n_kv * 2;
  const BlobView V{blob, blob_len};
  // what the reference asks of a layer before it keeps packed rows for it (kvqaxpk_packable, src/kvq_atxpk.hpp:61-72)
  int kb = 0; bool has_mu = false;
  std::vector<uint16_t> tabs((size_t)need * 256); std::vector<float> gfac(need), gains(need), mu((size_t)need * 256, 0.f);
  std::vector<uint32_t> pairs;
  for (int g = 0; g < need; ++g) {
    const size_t rec = V.group_record(g);
    const int bits = blob[rec + 1];
    const bool plain_trellis = blob[rec] == 0 && blob[rec + 3] == 0 && blob[rec + 4] == 0;   // mode, guard, directions
    if (!plain_trellis || (bits != 4 && bits != 5))
      throw std::runtime_error("packed rows need every group trellis-coded with 4 or 5 bits, no guard position and no projected directions");
    if (kb != 0 && bits != kb) throw std::runtime_error("packed rows need the same bits per element in every group");
    kb = bits;
    const size_t trec = V.table_record(blob[rec + 2]);
    float gain; std::memcpy(&gain, blob + trec + 4, 4);
    if (!(gain > 0.f) || gain > 1e6f) throw std::runtime_error("profile blob: table gain must be positive and finite");
    gfac[g] = 0.00390625f * gain; gains[g] = gain;
    uint16_t* row = &tabs[(size_t)g * 256];
    for (int st = 0; st < 256; ++st) row[st] = int_to_f16_bits(V.table_int(trec, st));
    if (blob[rec + 5] == 0) continue;
    has_mu = true;
    for (int d = 0; d < 256; ++d) {                    // fp16 mean row, widened by hand (host code, no half type needed)
      const unsigned h = V.half(rec + 8 + 2 * (size_t)d), expo = (h >> 10) & 31u, frac = h & 1023u;
      if (expo == 31) throw std::runtime_error("profile blob: mean row is not finite");
      const float mag = expo == 0 ? std::ldexp((float)frac, -24) : std::ldexp((float)(frac + 1024u), (int)expo - 25);
      mu[(size_t)g * 256 + d] = (h & 0x8000u) ? -mag : mag;
    }
  }
  // pair tables: entry i decodes two consecutive elements from the 8 + kb stream bits that end with the second one
  const size_t npair = (size_t)1 << (8 + kb);
  pairs.resize((size_t)need * npair);
  for (int g = 0; g < need; ++g)
    for (size_t i = 0; i < npair; ++i)
      pairs[(size_t)g * npair + i] = (uint32_t)tabs[(size_t)g * 256 + ((i >> kb) & 255)] | ((uint32_t)tabs[(size_t)g * 256 + (i & 255)] << 16);
  struct TbGuard {                                     // a profile that could not be set up completely leaves the handle as it was
    yka_kv* kv; bool done = false;
    ~TbGuard() {
      if (done || !kv->tb) return;
      yka_kv::Tb* t = kv->tb;
      (void)hipFree(t->pairs); (void)hipFree(t->gfac); (void)hipFree(t->mu); (void)hipFree(t->pool); (void)hipFree(t->scr); (void)hipFree(t->stage);
      delete t; kv->tb = nullptr;
    }
  } guard{kv};
  yka_kv::Tb* T = new yka_kv::Tb();
  kv->tb = T;
  T->kb = kb; T->stride = 32 * kb; T->nm = I.nm; T->has_mu = has_mu; T->layers = need / (n_kv * 2);
  const size_t rows = (size_t)n_kv * kv->cfg.max_ctx;
  T->pay_bytes = rows * T->stride; T->scl_bytes = rows * 4; T->layer_bytes = 2 * T->pay_bytes + 2 * T->scl_bytes;
  const size_t jobs = (size_t)kTbTileTok * 2 * n_kv * I.nm;
  T->scr_w_ofs = jobs * 256; T->scr_s_ofs = T->scr_w_ofs + jobs * 32;
  HIPCHK(hipMalloc((void**)&T->pairs, pairs.size() * 4)); HIPCHK(hipMemcpy(T->pairs, pairs.data(), pairs.size() * 4, hipMemcpyHostToDevice));
  gfac.resize((size_t)need + I.nm);
  std::memcpy(gfac.data() + need, blob + V.multipliers(), (size_t)I.nm * 4);
  gfac.insert(gfac.end(), gains.begin(), gains.end());
  HIPCHK(hipMalloc((void**)&T->gfac, gfac.size() * 4)); T->mults = T->gfac + need; T->gains = T->mults + I.nm; HIPCHK(hipMemcpy(T->gfac, gfac.data(), gfac.size() * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMalloc((void**)&T->mu, mu.size() * 4)); HIPCHK(hipMemcpy(T->mu, mu.data(), mu.size() * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMalloc((void**)&T->pool, 256 + T->layer_bytes * kv->cfg.n_layers + 256));
  HIPCHK(hipMemset(T->pool, 0, 256 + T->layer_bytes * kv->cfg.n_layers + 256));     // unwritten rows: state 0 everywhere, scale 0
  HIPCHK(hipMalloc((void**)&T->scr, T->scr_s_ofs + jobs * 4));
  HIPCHK(hipMalloc((void**)&T->stage, (size_t)2 * kv->cfg.max_rows * n_kv * 256 * sizeof(float)));
  HIPCHK(hipDeviceSynchronize());
  guard.done = true;
  YKA_CATCH_INT
}

int yka_kv_profile_bits(const yka_kv* kv) { return kv && kv->tb ? kv->tb->kb : 0; }

int yka_kv_export_rows_tb(yka_kv* kv, int layer, int pos0, int n, uint32_t* kw, float* ks, uint32_t* vw, float* vs) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer);
  if (!kv->tb) throw std::runtime_error("the handle has no profile");
  if (pos0 < 0 || n < 1 || (long long)pos0 + n > kv->cfg.max_ctx) throw std::runtime_error("row range outside the container");
  if (!kw || !ks || !vw || !vs) throw std::runtime_error("null pointer");
  const yka_kv::Tb& T = *kv->tb;
  HIPCHK(hipDeviceSynchronize());
  for (int h = 0; h < kv->cfg.n_kv_heads; ++h) {
    const size_t row = (size_t)h * kv->cfg.max_ctx + pos0, nb = (size_t)n * T.stride;
    HIPCHK(hipMemcpy(reinterpret_cast<uint8_t*>(kw) + (size_t)h * nb, T.kpay(layer) + row * T.stride, nb, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(reinterpret_cast<uint8_t*>(vw) + (size_t)h * nb, T.vpay(layer) + row * T.stride, nb, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(ks + (size_t)h * n, T.kscl(layer) + row, (size_t)n * 4, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(vs + (size_t)h * n, T.vscl(layer) + row, (size_t)n * 4, hipMemcpyDeviceToHost));
  }
  YKA_CATCH_INT
}

static void check_range(const yka_kv* kv, int pos0, int n) {
  if (pos0 < 0 || n < 1 || (long long)pos0 + n > kv->cfg.max_ctx) throw std::runtime_error("row range outside the container");
}

int yka_kv_export_rows(yka_kv* kv, int layer, int pos0, int n, uint8_t* kc, uint16_t* ks, uint8_t* vc, uint16_t* vs) {
  YKA_TRY
  on_device(kv); need_128(kv); check_layer(kv, layer); check_range(kv, pos0, n);
  if (!kc || !ks || !vc || !vs) throw std::runtime_error("null pointer");
  const size_t rows = (size_t)kv->cfg.n_kv_heads * n;
  DevBuf dkc(rows * 64), dvc(rows * 64), dks(rows * kNG * 2), dvs(rows * kNG * 2);
  HIPCHK(hipDeviceSynchronize());
  launch_export_rows(kv->view(layer), pos0, n, dkc.as<uint8_t>(), dks.as<uint16_t>(), dvc.as<uint8_t>(), dvs.as<uint16_t>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(kc, dkc.p, rows * 64, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(vc, dvc.p, rows * 64, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(ks, dks.p, rows * kNG * 2, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(vs, dvs.p, rows * kNG * 2, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_kv_import_rows(yka_kv* kv, int layer, int pos0, int n, const uint8_t* kc, const uint16_t* ks, const uint8_t* vc, const uint16_t* vs) {
  YKA_TRY
  on_device(kv); need_128(kv); check_layer(kv, layer); check_range(kv, pos0, n);
  if (!kc || !ks || !vc || !vs) throw std::runtime_error("null pointer");
  const size_t rows = (size_t)kv->cfg.n_kv_heads * n;
  DevBuf dkc(rows * 64), dvc(rows * 64), dks(rows * kNG * 2), dvs(rows * kNG * 2);
  HIPCHK(hipMemcpy(dkc.p, kc, rows * 64, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dvc.p, vc, rows * 64, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dks.p, ks, rows * kNG * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dvs.p, vs, rows * kNG * 2, hipMemcpyHostToDevice));
  HIPCHK(hipDeviceSynchronize());
  launch_import_rows(kv->view(layer), pos0, n, dkc.as<uint8_t>(), dks.as<uint16_t>(), dvc.as<uint8_t>(), dvs.as<uint16_t>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  YKA_CATCH_INT
}

int yka_append256_f32(yka_kv* kv, int layer, const float* d_k32, const float* d_v32, int M, const int* d_pos, int rotate, void* hip_stream) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!kv->r256()) throw std::runtime_error("this entry point exists for head_dim 256 only");
  if (!d_k32 || !d_v32 || !d_pos) throw std::runtime_error("null pointer");
  AppendArgs A{kv->view(layer), nullptr, nullptr, d_pos, M};
  A.k32 = d_k32; A.v32 = d_v32; A.rot = rotate != 0;
  if (kv->tb) tb_append(kv, layer, d_k32, d_v32, nullptr, nullptr, M, d_pos, rotate != 0, (hipStream_t)hip_stream);
  else launch_append256(A, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_rotate_q256(const float* d_x32, int rows, uint16_t* d_q16, void* hip_stream) {
  YKA_TRY
  if (!d_x32 || !d_q16 || rows < 1) throw std::runtime_error("bad argument");
  launch_rotate_q256(d_x32, rows, d_q16, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_append256_f32_host(yka_kv* kv, int layer, const float* k32, const float* v32, int M, int pos, int rotate) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!kv->r256()) throw std::runtime_error("this entry point exists for head_dim 256 only");
  if (!k32 || !v32) throw std::runtime_error("null pointer");
  if (pos < 0 || (long long)pos + M > kv->cfg.max_ctx) throw std::runtime_error("pos + M exceeds max_ctx");
  const size_t nk = (size_t)M * kv->cfg.n_kv_heads * 256;
  DevBuf dk(nk * 4), dv(nk * 4);
  HIPCHK(hipMemcpy(dk.p, k32, nk * 4, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dv.p, v32, nk * 4, hipMemcpyHostToDevice));
  HIPCHK(hipDeviceSynchronize());
  launch_set_int(kv->d_pos, pos, kv->stream);
  AppendArgs A{kv->view(layer), nullptr, nullptr, kv->d_pos, M};
  A.k32 = dk.as<float>(); A.v32 = dv.as<float>(); A.rot = rotate != 0;
  if (kv->tb) tb_append(kv, layer, dk.as<float>(), dv.as<float>(), nullptr, nullptr, M, kv->d_pos, rotate != 0, kv->stream);
  else launch_append256(A, kv->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(kv->stream));
  YKA_CATCH_INT
}

int yka_rotate_q256_host(const float* x32, int rows, uint16_t* q16) {
  YKA_TRY
  if (!x32 || !q16 || rows < 1) throw std::runtime_error("bad argument");
  const size_t n = (size_t)rows * 256;
  DevBuf dx(n * 4), dq(n * 2);
  HIPCHK(hipMemcpy(dx.p, x32, n * 4, hipMemcpyHostToDevice));
  launch_rotate_q256(dx.as<float>(), rows, dq.as<uint16_t>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(q16, dq.p, n * 2, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_attn_out256(const uint16_t* d_y16, const uint16_t* d_gate16, const int8_t* d_signs, int M, int n_heads, int8_t* d_qx,
                    float* d_alpha, void* hip_stream) {
  YKA_TRY
  if (!d_y16 || !d_gate16 || !d_signs || !d_qx || !d_alpha) throw std::runtime_error("null pointer");
  if (M < 1 || n_heads < 2 || (n_heads & 1)) throw std::runtime_error("M must be positive and n_heads even");
  launch_attn_out256(d_y16, d_gate16, d_signs, M, n_heads, 0, d_qx, d_alpha, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_attn_out256_lo(const uint16_t* d_y16, const uint16_t* d_gate16, const int8_t* d_signs, int M, int n_heads, int8_t* d_qx,
                       float* d_alpha, void* hip_stream) {
  YKA_TRY
  if (!d_y16 || !d_gate16 || !d_signs || !d_qx || !d_alpha) throw std::runtime_error("null pointer");
  if (M < 1 || M > 8 || n_heads < 2 || (n_heads & 1)) throw std::runtime_error("the interleaved layout holds 1 to 8 tokens; n_heads must be even");
  launch_attn_out256(d_y16, d_gate16, d_signs, M, n_heads, 1, d_qx, d_alpha, (hipStream_t)hip_stream);
  HIPCHK(hipGetLastError());
  YKA_CATCH_INT
}

int yka_attn_out256_lo_host(const uint16_t* y16, const uint16_t* gate16, const int8_t* signs, int M, int n_heads, int8_t* qx, float* alpha) {
  YKA_TRY
  if (!y16 || !gate16 || !signs || !qx || !alpha) throw std::runtime_error("null pointer");
  if (M < 1 || M > 8 || n_heads < 2 || (n_heads & 1)) throw std::runtime_error("the interleaved layout holds 1 to 8 tokens; n_heads must be even");
  const size_t n = (size_t)M * n_heads * 256, ng = n / 512, nqx = (size_t)(n_heads / 2) * 4096;
  DevBuf dy(n * 2), dg(n * 2), ds((size_t)n_heads * 256), dq(nqx), da(ng * 4);
  HIPCHK(hipMemcpy(dy.p, y16, n * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dg.p, gate16, n * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(ds.p, signs, (size_t)n_heads * 256, hipMemcpyHostToDevice));
  HIPCHK(hipMemset(dq.p, 0, nqx));
  launch_attn_out256(dy.as<uint16_t>(), dg.as<uint16_t>(), ds.as<int8_t>(), M, n_heads, 1, dq.as<int8_t>(), da.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(qx, dq.p, nqx, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(alpha, da.p, ng * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_attn_out256_host(const uint16_t* y16, const uint16_t* gate16, const int8_t* signs, int M, int n_heads, int8_t* qx, float* alpha) {
  YKA_TRY
  if (!y16 || !gate16 || !signs || !qx || !alpha) throw std::runtime_error("null pointer");
  if (M < 1 || n_heads < 2 || (n_heads & 1)) throw std::runtime_error("M must be positive and n_heads even");
  const size_t n = (size_t)M * n_heads * 256, ng = n / 512;
  DevBuf dy(n * 2), dg(n * 2), ds((size_t)n_heads * 256), dq(n), da(ng * 4);
  HIPCHK(hipMemcpy(dy.p, y16, n * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dg.p, gate16, n * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(ds.p, signs, (size_t)n_heads * 256, hipMemcpyHostToDevice));
  launch_attn_out256(dy.as<uint16_t>(), dg.as<uint16_t>(), ds.as<int8_t>(), M, n_heads, 0, dq.as<int8_t>(), da.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(qx, dq.p, n, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(alpha, da.p, ng * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_kv_export_rows256(yka_kv* kv, int layer, int pos0, int n, uint32_t* kw, float* ks, uint32_t* vw, float* vs) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_range(kv, pos0, n);
  no_trellis(kv);
  if (!kv->r256()) throw std::runtime_error("this entry point exists for head_dim 256 only");
  if (!kw || !ks || !vw || !vs) throw std::runtime_error("null pointer");
  const size_t rows = (size_t)kv->cfg.n_kv_heads * n;
  DevBuf dkw(rows * 128), dvw(rows * 128), dks(rows * 4), dvs(rows * 4);
  HIPCHK(hipDeviceSynchronize());
  launch_export_rows256(kv->view(layer), pos0, n, dkw.as<uint32_t>(), dks.as<float>(), dvw.as<uint32_t>(), dvs.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(kw, dkw.p, rows * 128, hipMemcpyDeviceToHost)); HIPCHK(hipMemcpy(vw, dvw.p, rows * 128, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(ks, dks.p, rows * 4, hipMemcpyDeviceToHost)); HIPCHK(hipMemcpy(vs, dvs.p, rows * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_kv_import_rows256(yka_kv* kv, int layer, int pos0, int n, const uint32_t* kw, const float* ks, const uint32_t* vw, const float* vs) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_range(kv, pos0, n);
  no_trellis(kv);
  if (!kv->r256()) throw std::runtime_error("this entry point exists for head_dim 256 only");
  if (!kw || !ks || !vw || !vs) throw std::runtime_error("null pointer");
  const size_t rows = (size_t)kv->cfg.n_kv_heads * n;
  DevBuf dkw(rows * 128), dvw(rows * 128), dks(rows * 4), dvs(rows * 4);
  HIPCHK(hipMemcpy(dkw.p, kw, rows * 128, hipMemcpyHostToDevice)); HIPCHK(hipMemcpy(dvw.p, vw, rows * 128, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dks.p, ks, rows * 4, hipMemcpyHostToDevice)); HIPCHK(hipMemcpy(dvs.p, vs, rows * 4, hipMemcpyHostToDevice));
  HIPCHK(hipDeviceSynchronize());
  launch_import_rows256(kv->view(layer), pos0, n, dkw.as<uint32_t>(), dks.as<float>(), dvw.as<uint32_t>(), dvs.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  YKA_CATCH_INT
}

int yka_kv_dequant_rows(yka_kv* kv, int layer, int pos0, int n, float* k, float* v) {
  YKA_TRY
  on_device(kv); need_128(kv); check_layer(kv, layer); check_range(kv, pos0, n);
  if (!k || !v) throw std::runtime_error("null pointer");
  const size_t ne = (size_t)kv->cfg.n_kv_heads * n * kD;
  DevBuf dk(ne * 4), dv(ne * 4);
  HIPCHK(hipDeviceSynchronize());
  launch_dequant_rows(kv->view(layer), pos0, n, dk.as<float>(), dv.as<float>(), nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(k, dk.p, ne * 4, hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(v, dv.p, ne * 4, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_kv_replicate_layer(yka_kv* kv, int src) {
  YKA_TRY
  on_device(kv); check_layer(kv, src);
  HIPCHK(hipDeviceSynchronize());
  for (int l = 0; l < kv->cfg.n_layers; ++l) {
    if (l == src) continue;
    HIPCHK(hipMemcpy(kv->pool + (size_t)l * kv->layer_bytes, kv->pool + (size_t)src * kv->layer_bytes, kv->layer_bytes, hipMemcpyDeviceToDevice));
    if (kv->tables) HIPCHK(hipMemcpy(kv->tables + (size_t)l * kv->n_pages, kv->tables + (size_t)src * kv->n_pages, (size_t)kv->n_pages * 4, hipMemcpyDeviceToDevice));
    // trellis-coded rows are copied as they are: meaningful only if both layers' groups share tables and mean rows
    if (kv->tb) HIPCHK(hipMemcpy(kv->tb->kpay(l), kv->tb->kpay(src), kv->tb->layer_bytes, hipMemcpyDeviceToDevice));
  }
  HIPCHK(hipDeviceSynchronize());
  YKA_CATCH_INT
}

int yka_layer_call_host(yka_kv* kv, int layer, const uint16_t* q16, const uint16_t* k16, const uint16_t* v16, int M, int pos,
                        const uint8_t* depth, uint16_t* out16) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer); check_rows(kv, M);
  if (!q16 || !out16 || ((k16 == nullptr) != (v16 == nullptr))) throw std::runtime_error("bad pointer arguments");
  if (pos < 0 || (long long)pos + M > kv->cfg.max_ctx) throw std::runtime_error("pos + M exceeds max_ctx");
  const size_t nq = (size_t)M * kv->cfg.n_heads * kv->D(), nk = (size_t)M * kv->cfg.n_kv_heads * kv->D();
  DevBuf dq(nq * 2), dk(nk * 2), dv(nk * 2), dout(nq * 2), dd((size_t)M);
  hipStream_t st = kv->stream;
  HIPCHK(hipMemcpy(dq.p, q16, nq * 2, hipMemcpyHostToDevice));
  if (k16) { HIPCHK(hipMemcpy(dk.p, k16, nk * 2, hipMemcpyHostToDevice)); HIPCHK(hipMemcpy(dv.p, v16, nk * 2, hipMemcpyHostToDevice)); }
  if (depth) HIPCHK(hipMemcpy(dd.p, depth, (size_t)M, hipMemcpyHostToDevice));
  HIPCHK(hipDeviceSynchronize());
  launch_set_int(kv->d_pos, pos, st);
  do_attend(kv, layer, dq.as<uint16_t>(), M, kv->d_pos, depth ? dd.as<uint8_t>() : nullptr, dout.as<uint16_t>(), st, 0,
            k16 ? dk.as<uint16_t>() : nullptr, k16 ? dv.as<uint16_t>() : nullptr);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(st));
  HIPCHK(hipMemcpy(out16, dout.p, nq * 2, hipMemcpyDeviceToHost));
  YKA_CATCH_INT
}

int yka_append_host(yka_kv* kv, int layer, const uint16_t* k16, const uint16_t* v16, int M, int pos) {
  YKA_TRY
  on_device(kv); check_layer(kv, layer);
  if (!k16 || !v16 || M < 1) throw std::runtime_error("bad argument");
  if (pos < 0 || (long long)pos + M > kv->cfg.max_ctx) throw std::runtime_error("pos + M exceeds max_ctx");
  const size_t nk = (size_t)M * kv->cfg.n_kv_heads * kv->D();
  DevBuf dk(nk * 2), dv(nk * 2);
  HIPCHK(hipMemcpy(dk.p, k16, nk * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dv.p, v16, nk * 2, hipMemcpyHostToDevice));
  HIPCHK(hipDeviceSynchronize());
  launch_set_int(kv->d_pos, pos, kv->stream);
  do_append(kv, layer, dk.as<uint16_t>(), dv.as<uint16_t>(), M, kv->d_pos, kv->stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(kv->stream));
  YKA_CATCH_INT
}

int yka_machine_probe(int kind, int p0, int iters, int blocks, int threads, double* out) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = 0;
  try {
    if (!out || kind < 0 || kind > 5 || iters < 1 || blocks < 1 || blocks > 65536) throw std::runtime_error("bad argument");
    if (threads != 256 && threads != 512) throw std::runtime_error("threads must be 256 or 512");
    if (kind == 0 && (p0 < 0 || p0 > 8 || (p0 & 1))) throw std::runtime_error("kind 0: p0 = vector FMAs per MFMA, one of 0 2 4 6 8");
    if (kind == 2 && (p0 < 0 || p0 > 8)) throw std::runtime_error("kind 2: p0 = opcode 0..8");
    if (kind == 3 && (p0 < 1 || threads != 512)) throw std::runtime_error("kind 3: p0 = iterations of the vector waves, 512 threads");
    if (kind == 5 && (p0 < 0 || p0 > 7)) throw std::runtime_error("kind 5: p0 = opcode 0..7");
    if (kind == 5) threads = 512;
    if (kind == 4 && iters > 4096) throw std::runtime_error("kind 4: iters = MiB to read, at most 4096");
    // a probe loop cannot be stopped once launched: a million iterations (about a second) is the most a call may ask for
    if (iters > 1000000 || (kind == 3 && p0 > 1000000)) throw std::runtime_error("iters (and p0 of kind 3) must be at most 1000000");
    if (kind == 1) threads = 256;
    const int waves = blocks * (threads / 64);
    const size_t nbytes = kind == 4 ? (size_t)iters << 20 : 16;
    DevBuf sink((size_t)blocks * 512 * 4), rec((size_t)waves * 16), src(nbytes);
    HIPCHK(hipMemset(rec.p, 0, (size_t)waves * 16));
    if (kind == 4) HIPCHK(hipMemset(src.p, 1, nbytes));
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipDeviceSynchronize());
    auto run = [&]() {
      unsigned long long* r = rec.as<unsigned long long>();
      switch (kind) {
        case 0: launch_probe_mix(p0, true, sink.as<float>(), r, iters, 0, 0, blocks, threads, nullptr); break;
        case 1: launch_probe_mfma16(sink.as<float>(), r, iters, blocks, nullptr); break;
        case 2: if (p0 == 8) launch_probe_mix(0, false, sink.as<float>(), r, iters, 0, 0, blocks, threads, nullptr);
                else launch_probe_valu(p0, sink.as<float>(), r, iters, blocks, threads, nullptr);
                break;
        case 3: launch_probe_mix(0, true, sink.as<float>(), r, iters, p0, 1, blocks, 512, nullptr); break;
        case 5: launch_probe_cross(p0, sink.as<float>(), r, iters, std::max(1, iters * 2 / 3), blocks, nullptr); break;
        default: launch_probe_read(p0 != 0, src.p, nbytes, sink.as<float>(), blocks, nullptr); break;
      }
    };
    run();                                        // warm
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    HIPCHK(hipEventRecord(e0, nullptr));
    run();
    HIPCHK(hipEventRecord(e1, nullptr));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    HIPCHK(hipGetLastError());
    std::vector<unsigned long long> h((size_t)waves * 2);
    HIPCHK(hipMemcpy(h.data(), rec.p, h.size() * 8, hipMemcpyDeviceToHost));
    // class A: waves 0..3 of a workgroup (or all waves), class B: waves 4..7 when the workgroup is split into two roles
    double sum[4] = {0, 0, 0, 0}; size_t cnt[2] = {0, 0};
    const int wpb = threads / 64;
    for (int w = 0; w < waves; ++w) {
      const int cls = ((kind == 3 || kind == 5) && (w % wpb) >= 4) ? 1 : 0;
      sum[2 * cls] += (double)h[2 * (size_t)w]; sum[2 * cls + 1] += (double)h[2 * (size_t)w + 1]; ++cnt[cls];
    }
    int wall_khz = 0;
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    HIPCHK(hipDeviceGetAttribute(&wall_khz, hipDeviceAttributeWallClockRate, dev));
    out[0] = ms;
    out[1] = cnt[0] ? sum[0] / cnt[0] : 0; out[2] = cnt[0] ? sum[1] / cnt[0] : 0;
    out[3] = cnt[1] ? sum[2] / cnt[1] : 0; out[4] = cnt[1] ? sum[3] / cnt[1] : 0;
    out[5] = wall_khz;
  } catch (const std::exception& e) { g_err = e.what(); rc = -1; }
  catch (...) { g_err = "unknown error"; rc = -1; }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  return rc;
}

struct yka_pass { hipGraph_t graph = nullptr; hipGraphExec_t exec = nullptr; int device = 0; };

yka_pass* yka_pass_capture(yka_kv* kv, const int32_t* layers, int n, const uint16_t* d_q16, const uint16_t* d_k16,
                           const uint16_t* d_v16, int M, const int* d_pos, const uint8_t* d_depth, uint16_t* d_out16, int mode) {
  yka_pass* p = nullptr;
  bool capturing = false;
  try {
    on_device(kv); check_rows(kv, M);
    if (!layers || n < 1 || !d_q16 || !d_pos || !d_out16 || mode < 0 || mode > 2) throw std::runtime_error("bad argument");
    if (mode == 0 && (!d_k16 || !d_v16)) throw std::runtime_error("mode 0 needs d_k16 and d_v16");
    for (int i = 0; i < n; ++i) check_layer(kv, layers[i]);
    p = new yka_pass(); p->device = kv->cfg.device;
    hipStream_t st = kv->stream;
    HIPCHK(hipStreamSynchronize(st));
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    capturing = true;
    for (int i = 0; i < n; ++i) {
      do_attend(kv, layers[i], d_q16, M, d_pos, d_depth, d_out16, st, mode == 2 ? 2 : 0, mode == 0 ? d_k16 : nullptr, mode == 0 ? d_v16 : nullptr);
    }
    capturing = false;
    HIPCHK(hipStreamEndCapture(st, &p->graph));
    HIPCHK(hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0));
    return p;
  } catch (const std::exception& e) { g_err = e.what(); }
  catch (...) { g_err = "unknown error"; }
  if (capturing) { hipGraph_t g = nullptr; (void)hipStreamEndCapture(kv->stream, &g); if (g) (void)hipGraphDestroy(g); }
  yka_pass_destroy(p);
  return nullptr;
}

int yka_pass_launch(yka_pass* p, void* hip_stream) {
  YKA_TRY
  if (!p || !p->exec) throw std::runtime_error("null pass");
  HIPCHK(hipSetDevice(p->device));
  HIPCHK(hipGraphLaunch(p->exec, (hipStream_t)hip_stream));
  YKA_CATCH_INT
}

void yka_pass_destroy(yka_pass* p) {
  if (!p) return;
  if (p->exec) (void)hipGraphExecDestroy(p->exec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  delete p;
}

static int f16_order(uint16_t b) { return (b & 0x8000u) ? -(int)(b & 0x7fffu) : (int)(b & 0x7fffu); }   // bit pattern -> position on the fp16 number line

int yka_attn_bench(yka_kv* kv, const uint16_t* q16, const uint16_t* k16, const uint16_t* v16, int M, int pos, int mode,
                   int use_graph, int reps, float* ms, uint16_t* out16_last, int* inv) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipGraph_t graph = nullptr; hipGraphExec_t gexec = nullptr;
  int rc = 0;
  bool capturing = false;
  try {
    on_device(kv); check_rows(kv, M);
    if (!q16 || !ms || reps < 1 || mode < 0 || mode > 2) throw std::runtime_error("bad argument");
    if (mode == 0 && (!k16 || !v16)) throw std::runtime_error("mode 0 needs k16 and v16");
    if (pos < 0 || (long long)pos + M > kv->cfg.max_ctx) throw std::runtime_error("pos + M exceeds max_ctx");
    const size_t nq = (size_t)M * kv->cfg.n_heads * kv->D(), nk = (size_t)M * kv->cfg.n_kv_heads * kv->D();
    DevBuf dq(nq * 2), dk(nk * 2), dv(nk * 2), dout(nq * 2);
    hipStream_t st = kv->stream;
    HIPCHK(hipMemcpy(dq.p, q16, nq * 2, hipMemcpyHostToDevice));
    if (k16) { HIPCHK(hipMemcpy(dk.p, k16, nk * 2, hipMemcpyHostToDevice)); HIPCHK(hipMemcpy(dv.p, v16, nk * 2, hipMemcpyHostToDevice)); }
    HIPCHK(hipMemset(dout.p, 0, nq * 2));
    HIPCHK(hipDeviceSynchronize());
    launch_set_int(kv->d_pos, pos, st);
    auto sweep = [&]() {
      for (int l = 0; l < kv->cfg.n_layers; ++l) {
        do_attend(kv, l, dq.as<uint16_t>(), M, kv->d_pos, nullptr, dout.as<uint16_t>(), st, mode == 2 ? 2 : 0,
                  mode == 0 ? dk.as<uint16_t>() : nullptr, mode == 0 ? dv.as<uint16_t>() : nullptr);
      }
    };
    for (int l = 0; l < kv->cfg.n_layers; ++l) check_tb_layer(kv, l);   // what a sweep would refuse is refused before the capture begins
    if (use_graph) {
      HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      capturing = true;
      sweep();
      capturing = false;
      HIPCHK(hipStreamEndCapture(st, &graph));
      HIPCHK(hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0));
    }
    auto run = [&]() { if (use_graph) HIPCHK(hipGraphLaunch(gexec, st)); else sweep(); };
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    run();                                       // warm sweep
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    for (int r = 0; r < reps; ++r) {
      HIPCHK(hipEventRecord(e0, st));
      run();
      HIPCHK(hipEventRecord(e1, st));
      HIPCHK(hipEventSynchronize(e1));
      HIPCHK(hipEventElapsedTime(&ms[r], e0, e1));
    }
    HIPCHK(hipGetLastError());
    if (out16_last) HIPCHK(hipMemcpy(out16_last, dout.p, nq * 2, hipMemcpyDeviceToHost));
    if (inv) {
      // the reference's built-in check (kvx_probe.cu:419-441): the M-row pass against M one-row passes over the same
      // container.  inv[0] = rows whose outputs differ in any bit, inv[1] = rows compared, inv[2] = output values that
      // differ, inv[3] = the largest distance between two such values in units of fp16 spacing.
      const size_t row = (size_t)kv->cfg.n_heads * kv->D();
      std::vector<uint16_t> full(nq), one(row);
      launch_set_int(kv->d_pos, pos, st);
      do_attend(kv, 0, dq.as<uint16_t>(), M, kv->d_pos, nullptr, dout.as<uint16_t>(), st);
      HIPCHK(hipGetLastError());
      HIPCHK(hipStreamSynchronize(st));
      HIPCHK(hipMemcpy(full.data(), dout.p, nq * 2, hipMemcpyDeviceToHost));
      int bad_rows = 0, bad_vals = 0, max_ulp = 0;
      for (int t = 0; t < M; ++t) {
        launch_set_int(kv->d_pos, pos + t, st);
        do_attend(kv, 0, dq.as<uint16_t>() + (size_t)t * row, 1, kv->d_pos, nullptr, dout.as<uint16_t>(), st);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(st));
        HIPCHK(hipMemcpy(one.data(), dout.p, row * 2, hipMemcpyDeviceToHost));
        bool differs = false;
        for (size_t i = 0; i < row; ++i) {
          const uint16_t a = full[(size_t)t * row + i], b = one[i];
          if (a == b) continue;
          differs = true; ++bad_vals;
          max_ulp = std::max(max_ulp, std::abs(f16_order(a) - f16_order(b)));
        }
        bad_rows += differs;
      }
      inv[0] = bad_rows; inv[1] = M; inv[2] = bad_vals; inv[3] = max_ulp;
      launch_set_int(kv->d_pos, pos, st);
      HIPCHK(hipStreamSynchronize(st));
    }
  } catch (const std::exception& e) { g_err = e.what(); rc = -1; }
  catch (...) { g_err = "unknown error"; rc = -1; }
  if (capturing) { hipGraph_t g = nullptr; (void)hipStreamEndCapture(kv->stream, &g); if (g) (void)hipGraphDestroy(g); }   // leave the stream out of capture mode
  if (gexec) (void)hipGraphExecDestroy(gexec);
  if (graph) (void)hipGraphDestroy(graph);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  return rc;
}

}  // extern "C"
