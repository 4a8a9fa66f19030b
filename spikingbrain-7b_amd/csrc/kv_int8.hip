// Per-row symmetric INT8 for cached K/V: every (token, kv head) row of 128 values is stored as
// 128 signed bytes and one fp32 scale,
//   scale = clamp(max|x| / 127, 1e-5, 1e4),  code = clamp(round_half_even(x / scale), -128, 127),
// the arithmetic of quantize_sym (W8ASpike/window_attention.py:227-237), done once when the row
// enters the cache instead of on the whole window at every step (a row's codes depend on that
// row only, so the values attention sees are the same).
//
// One wavefront quantises the rows of one (token, K|V) for up to 4 heads: 16 lanes per head, 8
// values per lane; max|x| of a head is four xor-exchanges inside its 16 lanes.
#include "kv_codes.h"

namespace {

using namespace sb;

template <int DT>
__device__ __forceinline__ void load8(const char *p, float (&x)[8]) {
  if constexpr (DT == SB_F32) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
  } else {
    unpack8<DT>(*reinterpret_cast<const uint4 *>(p), x);
  }
}

template <int DT>
__device__ __forceinline__ void store8(char *p, const float (&x)[8]) {
  if constexpr (DT == SB_F32) {
    reinterpret_cast<float4 *>(p)[0] = make_float4(x[0], x[1], x[2], x[3]);
    reinterpret_cast<float4 *>(p)[1] = make_float4(x[4], x[5], x[6], x[7]);
  } else {
    *reinterpret_cast<uint4 *>(p) = pack8<DT>(x);
  }
}

// scale of the 128-value row this lane's 16-lane group holds, and this lane's 8 codes (as floats)
__device__ __forceinline__ float quantise_row(const float (&x)[8], float (&code)[8]) {
  float amax = max_abs8(x, 0.f);
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) amax = fmaxf(amax, __shfl_xor(amax, d));
  const float scale = int8_scale(amax);
  int8_codes(x, scale, code);
  return scale;
}

// ROUND: the first round_tokens tokens, a prompt that attends to its rows as the cache will hold them, also leave code * scale in the
// tensor's type, [tokens, heads, 128] each, what quantize_sym_kernel writes in two more launches: us of a layer call, 64 / 1517 tokens
// 34.8 / 45.7 -> 29.9 / 40.4, 8 x 2000 230 -> 222, 16 x 8192 level. Latency for small prompts, bytes (read once instead of twice) for large.
template <int DT, bool ROUND>
__global__ __launch_bounds__(256) void kv_append_int8_kernel(
    const char *__restrict__ key, const char *__restrict__ value, char *__restrict__ k_cache,
    char *__restrict__ v_cache, float *__restrict__ k_scale, float *__restrict__ v_scale,
    const int64_t *__restrict__ slot_mapping, int64_t num_tokens, int num_kv_heads, int block_size,
    int64_t key_tok_b, int64_t key_head_b, int64_t val_tok_b, int64_t val_head_b, int64_t blk_b, int64_t row_b,
    int64_t head_b, char *__restrict__ k_round, char *__restrict__ v_round, int64_t round_tokens) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t tok = wave >> 1;
  const int which = (int)(wave & 1);
  if (tok >= num_tokens) return;
  const int64_t slot = slot_mapping[tok];
  const bool rounds = ROUND && tok < round_tokens;
  if (slot < 0 && !rounds) return;  // padded lane / token older than the window
  const int64_t blk = slot / block_size;
  const int off = (int)(slot - blk * block_size);
  const int h = blockIdx.y * 4 + (lane >> 4);
  const int piece = lane & 15;
  // lanes of a head beyond num_kv_heads still take part in the exchanges (on zeros)
  const bool live = h < num_kv_heads;
  constexpr int kEsz = DT == SB_F32 ? 4 : 2;
  float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, code[8];
  if (live) {
    const char *src = which ? value + tok * val_tok_b + h * val_head_b : key + tok * key_tok_b + h * key_head_b;
    load8<DT>(src + piece * 8 * kEsz, x);
  }
  const float scale = quantise_row(x, code);
  if (!live) return;
  if (rounds) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = code[i] * scale;
    store8<DT>((which ? v_round : k_round) + ((tok * num_kv_heads + h) * 128 + piece * 8) * kEsz, y);
    if (slot < 0) return;
  }
  char *dst = (which ? v_cache : k_cache) + blk * blk_b + off * row_b + h * head_b + piece * 8;
  *reinterpret_cast<uint2 *>(dst) = int8_bytes(code);
  if (piece == 0) (which ? v_scale : k_scale)[(blk * num_kv_heads + h) * block_size + off] = scale;
}

// y = (code * scale) rounded to the tensor's dtype, row by row: what quantize_sym returns.
template <int DT>
__global__ __launch_bounds__(256) void quantize_sym_kernel(const char *__restrict__ in, char *__restrict__ out,
                                                           int64_t rows, int heads, int64_t in_row_b,
                                                           int64_t in_head_b, int64_t out_row_b, int64_t out_head_b) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (wave >= rows) return;
  const int h = blockIdx.y * 4 + (lane >> 4);
  const int piece = lane & 15;
  const bool live = h < heads;
  constexpr int kEsz = DT == SB_F32 ? 4 : 2;
  float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, code[8];
  if (live) load8<DT>(in + wave * in_row_b + h * in_head_b + piece * 8 * kEsz, x);
  const float scale = quantise_row(x, code);
  if (!live) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) code[i] *= scale;
  store8<DT>(out + wave * out_row_b + h * out_head_b + piece * 8 * kEsz, code);
}

struct Fp8Append {
  const char *key, *value;
  char *k_cache, *v_cache;
  const int64_t *slot_mapping;
  int64_t num_tokens;
  int num_kv_heads, block_size;
  int64_t key_tok_b, key_head_b, val_tok_b, val_head_b, blk_b, row_b, head_b;
  float k_scale, v_scale;
};

// one wavefront: four heads (16 lanes each) of one token's K (which = 0) or V row
template <int DT>
__device__ __forceinline__ void append_fp8(const Fp8Append &p, int64_t tok, int which, int head0, int lane) {
  const int64_t slot = p.slot_mapping[tok];
  if (slot < 0) return;
  const int64_t blk = slot / p.block_size;
  const int off = (int)(slot - blk * p.block_size);
  const int h = head0 + (lane >> 4);
  const int piece = lane & 15;
  if (h >= p.num_kv_heads) return;
  constexpr int kEsz = DT == SB_F32 ? 4 : 2;
  float x[8];
  const char *src = which ? p.value + tok * p.val_tok_b + h * p.val_head_b : p.key + tok * p.key_tok_b + h * p.key_head_b;
  load8<DT>(src + piece * 8 * kEsz, x);
  const float sc = which ? p.v_scale : p.k_scale;
  char *dst = (which ? p.v_cache : p.k_cache) + blk * p.blk_b + off * p.row_b + h * p.head_b + piece * 8;
  *reinterpret_cast<uint2 *>(dst) = fp8_bytes(x, sc);
}

// The append alone (28 of them in a captured step: through the kernel below, with its 300 bytes of arguments, the step took 319 instead
// of 315 us).
template <int DT>
__global__ __launch_bounds__(256) void kv_append_fp8_kernel(const Fp8Append p) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if ((wave >> 1) >= p.num_tokens) return;
  append_fp8<DT>(p, wave >> 1, (int)(wave & 1), blockIdx.y * 4, threadIdx.x & 63);
}

// y = e4m3fn(clamp(x / scale)) * scale rounded to the tensor's dtype: what a tensor looks like after a
// round trip through the fp8 cache (or through scaled_fp8_quant, meta_attention.py:806-811, :853-869).
struct Fp8Round {
  const char *in;
  char *out;
  int64_t rows, in_row_b, out_row_b;
  int row_vecs;
  float scale;
};
template <int DT>
__device__ __forceinline__ void round_fp8(const Fp8Round &p, int64_t t) {  // t: 8-element vector of the tensor
  const int64_t r = t / p.row_vecs;
  if (r >= p.rows) return;
  const int vec = (int)(t - r * p.row_vecs);
  constexpr int kEsz = DT == SB_F32 ? 4 : 2;
  const float scale = p.scale;
  float x[8];
  load8<DT>(p.in + r * p.in_row_b + vec * 8 * kEsz, x);
  float y[8];
  fp8_values(fp8_bytes(x, scale), scale, y);
  store8<DT>(p.out + r * p.out_row_b + vec * 8 * kEsz, y);
}

// What a step over an fp8 cache does in front of its attention, in one launch: the append and the round trips of the
// queries and (prompts) of the keys and values attended to in flight. Workgroups [0, first[0]) append, those
// from first[j] on round tensor j. The pieces touch different memory. As launches of their own they cost 4 to 5 us each.
constexpr int kMaxRounds = 3;
struct Fp8Step {
  Fp8Append append;
  Fp8Round round[kMaxRounds];
  int64_t first[kMaxRounds];
};
template <int DT>
__global__ __launch_bounds__(256) void fp8_step_kernel(const Fp8Step p) {
  const int64_t b = blockIdx.x;
  if (b < p.first[0]) {
    const int64_t wave = b * 4 + (threadIdx.x >> 6);
    const int groups = (p.append.num_kv_heads + 3) >> 2;
    const int64_t tok = (wave >> 1) / groups;
    if (tok >= p.append.num_tokens) return;
    append_fp8<DT>(p.append, tok, (int)(wave & 1), 4 * (int)((wave >> 1) - tok * groups), threadIdx.x & 63);
  } else if (b < p.first[1]) {
    round_fp8<DT>(p.round[0], (b - p.first[0]) * 256 + threadIdx.x);
  } else if (b < p.first[2]) {
    round_fp8<DT>(p.round[1], (b - p.first[1]) * 256 + threadIdx.x);
  } else {
    round_fp8<DT>(p.round[2], (b - p.first[2]) * 256 + threadIdx.x);
  }
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int elem_size(int dtype) {
  switch (dtype) {
    case SB_BF16:
    case SB_F16: return 2;
    case SB_F32: return 4;
    default: return 0;
  }
}

}  // namespace

static int append_int8(const sb_kv_append_int8_args *a, void *k_round, void *v_round, int64_t round_tokens) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_kv_append_int8: null args");
  if (a->num_tokens < 0) return fail(SB_ERR_INVALID, "sb_kv_append_int8: negative num_tokens");
  if (a->num_tokens == 0) return SB_OK;
  if (!a->key || !a->value || !a->k_cache || !a->v_cache || !a->k_scale || !a->v_scale || !a->slot_mapping)
    return fail(SB_ERR_INVALID, "sb_kv_append_int8: null tensor pointer");
  const int esz = elem_size(a->dtype);
  if (!esz) return fail(SB_ERR_UNSUPPORTED, "sb_kv_append_int8: unknown dtype %d", a->dtype);
  if (a->head_size != 128)
    return fail(SB_ERR_UNSUPPORTED, "sb_kv_append_int8: head_size %d (only 128 is built)", a->head_size);
  if (a->num_kv_heads <= 0 || a->block_size <= 0) return fail(SB_ERR_INVALID, "sb_kv_append_int8: non-positive shape");
  const int64_t in_strides[] = {a->key_stride_token, a->key_stride_head, a->value_stride_token, a->value_stride_head};
  for (int64_t s : in_strides)
    if ((s * esz) % 16 != 0)
      return fail(SB_ERR_INVALID, "sb_kv_append_int8: stride %lld elements is not 16-byte aligned", (long long)s);
  const int64_t c_strides[] = {a->cache_stride_block, a->cache_stride_row, a->cache_stride_head};
  for (int64_t s : c_strides)
    if (s % 8 != 0) return fail(SB_ERR_INVALID, "sb_kv_append_int8: cache stride %lld is not 8-byte aligned", (long long)s);
  if (!aligned16(a->key) || !aligned16(a->value) || !aligned16(a->k_cache) || !aligned16(a->v_cache))
    return fail(SB_ERR_INVALID, "sb_kv_append_int8: tensor base not 16-byte aligned");
  const int64_t waves = a->num_tokens * 2;
  const int64_t blocks = (waves + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_kv_append_int8: too many tokens");
  const dim3 grid((unsigned)blocks, (unsigned)((a->num_kv_heads + 3) / 4));
#define SB_ARGS                                                                                              \
  (const char *)a->key, (const char *)a->value, (char *)a->k_cache, (char *)a->v_cache, a->k_scale, a->v_scale, \
      a->slot_mapping, a->num_tokens, a->num_kv_heads, a->block_size, a->key_stride_token *esz,              \
      a->key_stride_head *esz, a->value_stride_token *esz, a->value_stride_head *esz, a->cache_stride_block,  \
      a->cache_stride_row, a->cache_stride_head, (char *)k_round, (char *)v_round, round_tokens
  hipStream_t st = (hipStream_t)a->stream;
#define SB_APPEND(DT)                                                                                          \
  do {                                                                                                         \
    if (round_tokens > 0) hipLaunchKernelGGL((kv_append_int8_kernel<DT, true>), grid, dim3(256), 0, st, SB_ARGS); \
    else hipLaunchKernelGGL((kv_append_int8_kernel<DT, false>), grid, dim3(256), 0, st, SB_ARGS);              \
  } while (0)
  if (a->dtype == SB_BF16) SB_APPEND(SB_BF16);
  else if (a->dtype == SB_F16) SB_APPEND(SB_F16);
  else SB_APPEND(SB_F32);
#undef SB_APPEND
#undef SB_ARGS
  return check_launch("kv_append_int8_kernel");
}

extern "C" int sb_kv_append_int8(const sb_kv_append_int8_args *a) { return append_int8(a, nullptr, nullptr, 0); }

extern "C" int sb_kv_append_int8_round(const sb_kv_append_int8_args *a, void *key_out, void *value_out, int64_t round_tokens) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_kv_append_int8_round: null args");
  if (round_tokens < 0 || round_tokens > a->num_tokens || (round_tokens > 0 && (!key_out || !value_out || !aligned16(key_out) || !aligned16(value_out))))
    return fail(SB_ERR_INVALID, "sb_kv_append_int8_round: 0 to num_tokens rounded tokens, outputs 16-byte aligned");
  return append_int8(a, key_out, value_out, round_tokens);
}

extern "C" int sb_quantize_sym(const sb_quantize_sym_args *a) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_quantize_sym: null args");
  if (a->rows < 0 || a->heads < 0) return fail(SB_ERR_INVALID, "sb_quantize_sym: negative size");
  if (a->rows == 0 || a->heads == 0) return SB_OK;
  if (!a->in || !a->out) return fail(SB_ERR_INVALID, "sb_quantize_sym: null tensor pointer");
  const int esz = elem_size(a->dtype);
  if (!esz) return fail(SB_ERR_UNSUPPORTED, "sb_quantize_sym: unknown dtype %d", a->dtype);
  if (a->head_size != 128)
    return fail(SB_ERR_UNSUPPORTED, "sb_quantize_sym: head_size %d (only 128 is built)", a->head_size);
  const int64_t strides[] = {a->in_stride_row, a->in_stride_head, a->out_stride_row, a->out_stride_head};
  for (int64_t s : strides)
    if ((s * esz) % 16 != 0)
      return fail(SB_ERR_INVALID, "sb_quantize_sym: stride %lld elements is not 16-byte aligned", (long long)s);
  if (!aligned16(a->in) || !aligned16(a->out)) return fail(SB_ERR_INVALID, "sb_quantize_sym: tensor base not 16-byte aligned");
  const int64_t blocks = (a->rows + 3) / 4;
  if (blocks > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_quantize_sym: too many rows");
  const dim3 grid((unsigned)blocks, (unsigned)((a->heads + 3) / 4));
#define SB_ARGS                                                                                         \
  (const char *)a->in, (char *)a->out, a->rows, a->heads, a->in_stride_row *esz, a->in_stride_head *esz, \
      a->out_stride_row *esz, a->out_stride_head *esz
  hipStream_t st = (hipStream_t)a->stream;
  if (a->dtype == SB_BF16) hipLaunchKernelGGL(quantize_sym_kernel<SB_BF16>, grid, dim3(256), 0, st, SB_ARGS);
  else if (a->dtype == SB_F16) hipLaunchKernelGGL(quantize_sym_kernel<SB_F16>, grid, dim3(256), 0, st, SB_ARGS);
  else hipLaunchKernelGGL(quantize_sym_kernel<SB_F32>, grid, dim3(256), 0, st, SB_ARGS);
#undef SB_ARGS
  return check_launch("quantize_sym_kernel");
}

namespace {

int check_append(const sb_kv_append_fp8_args *a) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_kv_append_fp8: null args");
  if (a->num_tokens < 0) return fail(SB_ERR_INVALID, "sb_kv_append_fp8: negative num_tokens");
  if (a->num_tokens == 0) return SB_OK;
  if (!a->key || !a->value || !a->k_cache || !a->v_cache || !a->slot_mapping)
    return fail(SB_ERR_INVALID, "sb_kv_append_fp8: null tensor pointer");
  const int esz = elem_size(a->dtype);
  if (!esz) return fail(SB_ERR_UNSUPPORTED, "sb_kv_append_fp8: unknown dtype %d", a->dtype);
  if (a->head_size != 128)
    return fail(SB_ERR_UNSUPPORTED, "sb_kv_append_fp8: head_size %d (only 128 is built)", a->head_size);
  if (a->num_kv_heads <= 0 || a->block_size <= 0) return fail(SB_ERR_INVALID, "sb_kv_append_fp8: non-positive shape");
  if (!(a->k_scale > 0.f) || !(a->v_scale > 0.f)) return fail(SB_ERR_INVALID, "sb_kv_append_fp8: scales must be positive");
  const int64_t in_strides[] = {a->key_stride_token, a->key_stride_head, a->value_stride_token, a->value_stride_head};
  for (int64_t s : in_strides)
    if ((s * esz) % 16 != 0)
      return fail(SB_ERR_INVALID, "sb_kv_append_fp8: stride %lld elements is not 16-byte aligned", (long long)s);
  const int64_t c_strides[] = {a->cache_stride_block, a->cache_stride_row, a->cache_stride_head};
  for (int64_t s : c_strides)
    if (s % 8 != 0) return fail(SB_ERR_INVALID, "sb_kv_append_fp8: cache stride %lld is not 8-byte aligned", (long long)s);
  if (!aligned16(a->key) || !aligned16(a->value) || !aligned16(a->k_cache) || !aligned16(a->v_cache))
    return fail(SB_ERR_INVALID, "sb_kv_append_fp8: tensor base not 16-byte aligned");
  if (a->num_tokens > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_kv_append_fp8: too many tokens");
  return SB_OK;
}

int check_round(const sb_fp8_round_args *a) {
  using namespace sb_host;
  if (a->rows < 0 || a->row_elems < 0) return fail(SB_ERR_INVALID, "sb_fp8_round: negative size");
  if (a->rows == 0 || a->row_elems == 0) return SB_OK;
  if (!a->in || !a->out) return fail(SB_ERR_INVALID, "sb_fp8_round: null tensor pointer");
  const int esz = elem_size(a->dtype);
  if (!esz) return fail(SB_ERR_UNSUPPORTED, "sb_fp8_round: unknown dtype %d", a->dtype);
  if (a->row_elems % 8 != 0 || (a->in_stride_row * esz) % 16 != 0 || (a->out_stride_row * esz) % 16 != 0 ||
      !aligned16(a->in) || !aligned16(a->out))
    return fail(SB_ERR_INVALID, "sb_fp8_round: rows must be whole 8-element vectors at 16-byte aligned addresses");
  if (!(a->scale > 0.f)) return fail(SB_ERR_INVALID, "sb_fp8_round: scale must be positive");
  return SB_OK;
}

// (a: checked, or null; r: n checked tensors, all of `dtype`)
int launch_fp8_step(const sb_kv_append_fp8_args *a, const sb_fp8_round_args *r, int n, int dtype, hipStream_t st) {
  using namespace sb_host;
  const int esz = elem_size(dtype);
  Fp8Step p = {};
  int64_t blocks = 0;
  if (a && a->num_tokens > 0) {
    p.append = Fp8Append{(const char *)a->key, (const char *)a->value, (char *)a->k_cache, (char *)a->v_cache, a->slot_mapping,
                         a->num_tokens, a->num_kv_heads, a->block_size, a->key_stride_token * esz, a->key_stride_head * esz,
                         a->value_stride_token * esz, a->value_stride_head * esz, a->cache_stride_block, a->cache_stride_row,
                         a->cache_stride_head, a->k_scale, a->v_scale};
    blocks = (a->num_tokens * 2 * ((a->num_kv_heads + 3) / 4) + 3) / 4;
    if (n == 0) {
      const dim3 agrid((unsigned)((a->num_tokens * 2 + 3) / 4), (unsigned)((a->num_kv_heads + 3) / 4));
      if (dtype == SB_BF16) hipLaunchKernelGGL(kv_append_fp8_kernel<SB_BF16>, agrid, dim3(256), 0, st, p.append);
      else if (dtype == SB_F16) hipLaunchKernelGGL(kv_append_fp8_kernel<SB_F16>, agrid, dim3(256), 0, st, p.append);
      else hipLaunchKernelGGL(kv_append_fp8_kernel<SB_F32>, agrid, dim3(256), 0, st, p.append);
      return check_launch("kv_append_fp8_kernel");
    }
  }
  for (int j = 0; j < kMaxRounds; ++j) {
    p.first[j] = blocks;
    if (j >= n || r[j].rows == 0 || r[j].row_elems == 0) continue;
    p.round[j] = Fp8Round{(const char *)r[j].in, (char *)r[j].out, r[j].rows, r[j].in_stride_row * esz, r[j].out_stride_row * esz,
                          (int)(r[j].row_elems / 8), r[j].scale};
    blocks += (r[j].rows * (r[j].row_elems / 8) + 255) / 256;
  }
  if (blocks == 0) return SB_OK;
  if (blocks > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_fp8_step: too many rows");
  const dim3 grid((unsigned)blocks);
  if (dtype == SB_BF16) hipLaunchKernelGGL(fp8_step_kernel<SB_BF16>, grid, dim3(256), 0, st, p);
  else if (dtype == SB_F16) hipLaunchKernelGGL(fp8_step_kernel<SB_F16>, grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL(fp8_step_kernel<SB_F32>, grid, dim3(256), 0, st, p);
  return check_launch("fp8_step_kernel");
}

}  // namespace

extern "C" int sb_kv_append_fp8(const sb_kv_append_fp8_args *a) {
  const int rc = check_append(a);
  return rc != SB_OK ? rc : launch_fp8_step(a, nullptr, 0, a->dtype, (hipStream_t)a->stream);
}

extern "C" int sb_fp8_round(const void *in, void *out, int64_t rows, int64_t row_elems, int64_t in_stride_row,
                            int64_t out_stride_row, int32_t dtype, float scale, void *stream) {
  const sb_fp8_round_args r = {in, out, rows, row_elems, in_stride_row, out_stride_row, dtype, scale};
  const int rc = check_round(&r);
  return rc != SB_OK ? rc : launch_fp8_step(nullptr, &r, 1, dtype, (hipStream_t)stream);
}

extern "C" int sb_fp8_step(const sb_kv_append_fp8_args *append, const sb_fp8_round_args *rounds, int32_t n_rounds,
                           void *stream) {
  using namespace sb_host;
  if (n_rounds < 0 || n_rounds > kMaxRounds || (n_rounds > 0 && !rounds))
    return fail(SB_ERR_INVALID, "sb_fp8_step: 0 to %d tensors to round", kMaxRounds);
  if (!append && n_rounds == 0) return SB_OK;
  if (append)
    if (int rc = check_append(append)) return rc;
  const int dtype = append ? append->dtype : rounds[0].dtype;
  bool same = true;
  for (int j = 0; j < n_rounds; ++j) {
    if (int rc = check_round(&rounds[j])) return rc;
    same = same && rounds[j].dtype == dtype;
  }
  if (!same) {  // tensors of several types: a launch each
    for (int j = 0; j < n_rounds; ++j)
      if (int rc = launch_fp8_step(nullptr, &rounds[j], 1, rounds[j].dtype, (hipStream_t)stream)) return rc;
    return append ? launch_fp8_step(append, nullptr, 0, dtype, (hipStream_t)stream) : SB_OK;
  }
  return launch_fp8_step(append, rounds, n_rounds, dtype, (hipStream_t)stream);
}
