// Byte-moving kernels of the cache path: slot-mapped KV append, block copy, and the
// dense-window shift used by the HuggingFace-style cache. All are pure copies in 16-byte
// lanes (one wavefront moves 1 KiB per instruction), so results are bit-exact.
#include "common.h"

namespace {

// One wavefront per (token, K|V). A row of num_kv_heads*head_size elements is moved as
// 16-byte chunks; chunk c belongs to head c / chunks_per_head.
__global__ __launch_bounds__(256) void kv_append_kernel(
    const char *__restrict__ key, const char *__restrict__ value, char *__restrict__ k_cache,
    char *__restrict__ v_cache, const int64_t *__restrict__ slot_mapping, int64_t num_tokens,
    int chunks_per_head, int n_chunks, int block_size, int64_t key_tok_b, int64_t key_head_b,
    int64_t val_tok_b, int64_t val_head_b, int64_t blk_b, int64_t row_b, int64_t head_b) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t tok = wave >> 1;
  const int which = (int)(wave & 1);
  if (tok >= num_tokens) return;
  const int64_t slot = slot_mapping[tok];
  if (slot < 0) return;  // padded lane / token older than the window
  const int64_t blk = slot / block_size;
  const int64_t off = slot - blk * block_size;
  const char *src = which ? value + tok * val_tok_b : key + tok * key_tok_b;
  const int64_t src_head_b = which ? val_head_b : key_head_b;
  char *dst = (which ? v_cache : k_cache) + blk * blk_b + off * row_b;
  for (int c = lane; c < n_chunks; c += 64) {
    const int h = c / chunks_per_head;
    const int w = c - h * chunks_per_head;
    const uint4 x = *reinterpret_cast<const uint4 *>(src + h * src_head_b + (int64_t)w * 16);
    *reinterpret_cast<uint4 *>(dst + h * head_b + (int64_t)w * 16) = x;
  }
}

// One workgroup per (pair, 4 KiB segment of the block).
__global__ __launch_bounds__(256) void copy_blocks_kernel(char *__restrict__ cache,
                                                          const int64_t *__restrict__ pairs,
                                                          int64_t block_bytes,
                                                          int64_t stride_block_bytes) {
  const int64_t pair = blockIdx.y;
  const int64_t src = pairs[2 * pair], dst = pairs[2 * pair + 1];
  const int64_t byte0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 16;
  if (byte0 >= block_bytes || src == dst) return;
  const uint4 x = *reinterpret_cast<const uint4 *>(cache + src * stride_block_bytes + byte0);
  *reinterpret_cast<uint4 *>(cache + dst * stride_block_bytes + byte0) = x;
}

// Dense window shift: per plane, dst rows [dst_row0, dst_row0+keep) <- src rows
// [src_row0, src_row0+keep), then n_new fresh rows behind them.
// grid: (ceil(rows*chunks / 256), planes, tensors): K and V of a layer move the same rows and are one launch (a token's
// append is a few KiB: what it costs is the launch; 4 x one token into a window of 4096: 2.2 us per launch)
struct ShiftTensors {
  const char *src[2];
  char *dst[2];
  const char *fresh[2];
};
__global__ __launch_bounds__(256) void window_shift_kernel(
    const ShiftTensors t, int64_t keep_rows, int64_t src_row0, int64_t dst_row0, int64_t n_new, int64_t row_bytes,
    int64_t src_plane_b, int64_t dst_plane_b, int64_t fresh_plane_b, int64_t fresh_row_b) {
  const char *__restrict__ const src = t.src[blockIdx.z];
  const char *__restrict__ const fresh = t.fresh[blockIdx.z];
  char *__restrict__ const dst = t.dst[blockIdx.z];
  const int64_t plane = blockIdx.y;
  const int64_t chunks_per_row = row_bytes >> 4;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = idx / chunks_per_row;
  const int64_t c = idx - row * chunks_per_row;
  if (row >= keep_rows + n_new) return;
  uint4 x;
  if (row < keep_rows) {
    x = *reinterpret_cast<const uint4 *>(src + plane * src_plane_b + (src_row0 + row) * row_bytes +
                                         c * 16);
  } else {
    x = *reinterpret_cast<const uint4 *>(fresh + plane * fresh_plane_b +
                                         (row - keep_rows) * fresh_row_b + c * 16);
  }
  *reinterpret_cast<uint4 *>(dst + plane * dst_plane_b + (dst_row0 + row) * row_bytes + c * 16) = x;
}

// Lengths and bounds of a dense left-padded batch: one workgroup per sequence counts its mask row (the only memory
// it reads: latency-bound, so 1024 threads of four independent loads each cover 4096 keys in one round trip) and
// writes the sequence's rows. Replaces a dozen elementwise launches and a reduction per layer call (four left-padded
// sequences, one token against 4096 keys: 159.6 -> 67.0 us a call, together with the paired shift above).
struct DenseRows {
  const void *mask;
  int64_t mask_cols, mask_sr, mask_sc, num_queries, num_keys, kv_step;
  int32_t *seq_lens, *row_seq, *key_lo;
  int64_t *kv_start;
};
template <typename M>
__device__ __forceinline__ void dense_rows(const DenseRows &p, int64_t b) {
  __shared__ int part[16];
  const int tid = threadIdx.x;
  int pad = 0;
  if (p.mask) {  // (uniform)
    const M *row = static_cast<const M *>(p.mask) + b * p.mask_sr;
    int n = 0;
    int64_t i = tid;
    for (; i + 3072 < p.mask_cols; i += 4096) {
      const M a0 = row[i * p.mask_sc], a1 = row[(i + 1024) * p.mask_sc], a2 = row[(i + 2048) * p.mask_sc],
              a3 = row[(i + 3072) * p.mask_sc];
      n += (a0 != 0) + (a1 != 0) + (a2 != 0) + (a3 != 0);
    }
    for (; i < p.mask_cols; i += 1024) n += row[i * p.mask_sc] != 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) n += __shfl_xor(n, d);
    if ((tid & 63) == 0) part[tid >> 6] = n;
    __syncthreads();
    n = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) n += part[w];
    pad = (int)(p.num_keys - n);
  }
  if (p.kv_start && tid == 0) p.kv_start[b] = b * p.kv_step;
  for (int64_t j = tid; j < p.num_queries; j += 1024) {
    const int64_t r = b * p.num_queries + j;
    if (p.seq_lens) p.seq_lens[r] = (int32_t)(p.num_keys - p.num_queries + 1 + j);
    if (p.row_seq) p.row_seq[r] = (int32_t)b;
    if (p.key_lo) p.key_lo[r] = pad;
  }
}
template <typename M>
__global__ __launch_bounds__(1024) void dense_rows_kernel(const DenseRows p) { dense_rows<M>(p, blockIdx.x); }

// The above and, by the workgroups behind, the rows a decode step adds to a layer's K and V windows (the two need nothing of
// each other): one launch less in front of the attention, 2 to 4 us of a layer call (4 sequences of 4096 keys 22.8 -> 20.7,
// 16 of 2000 24.8 -> 22.6, one of 128 22.7 -> 19.0).
struct NewRows {
  char *dst[2];
  const char *fresh[2];
  int64_t planes, n_new, chunks, dst_plane_b, dst_off, row_bytes, fresh_plane_b, fresh_row_b;
};
template <typename M>
__global__ __launch_bounds__(1024) void dense_step_kernel(const DenseRows p, const NewRows s, const unsigned batch) {
  if (blockIdx.x < batch) {
    dense_rows<M>(p, blockIdx.x);
    return;
  }
  int64_t i = (int64_t)(blockIdx.x - batch) * 1024 + threadIdx.x;   // [tensor][plane][row][16-byte chunk]
  const int64_t rows = i / s.chunks, c = (i - rows * s.chunks) * 16;
  const int64_t planes = rows / s.n_new, row = rows - planes * s.n_new;
  if (planes >= 2 * s.planes) return;
  const int which = planes >= s.planes;
  const int64_t plane = which ? planes - s.planes : planes;
  *reinterpret_cast<uint4 *>((which ? s.dst[1] : s.dst[0]) + plane * s.dst_plane_b + s.dst_off + row * s.row_bytes + c) =
      *reinterpret_cast<const uint4 *>((which ? s.fresh[1] : s.fresh[0]) + plane * s.fresh_plane_b + row * s.fresh_row_b + c);
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

namespace sb_host {

// Refuses what the append kernels do not take (num_tokens > 0 from here on; the prefill kernel's append goes by it too).
int check_kv_append(const sb_kv_append_args *a) {
  if (!a) return fail(SB_ERR_INVALID, "sb_kv_append: null args");
  if (a->num_tokens < 0) return fail(SB_ERR_INVALID, "sb_kv_append: negative num_tokens");
  if (a->num_tokens == 0) return SB_OK;
  if (!a->key || !a->value || !a->k_cache || !a->v_cache || !a->slot_mapping)
    return fail(SB_ERR_INVALID, "sb_kv_append: null tensor pointer");
  int esz;
  switch (a->dtype) {
    case SB_BF16:
    case SB_F16: esz = 2; break;
    case SB_F32: esz = 4; break;
    default: return fail(SB_ERR_UNSUPPORTED, "sb_kv_append: unknown dtype %d", a->dtype);
  }
  if (a->num_kv_heads <= 0 || a->head_size <= 0 || a->block_size <= 0)
    return fail(SB_ERR_INVALID, "sb_kv_append: non-positive shape");
  const int64_t head_bytes = (int64_t)a->head_size * esz;
  if (head_bytes % 16 != 0)
    return fail(SB_ERR_UNSUPPORTED, "sb_kv_append: head_size*elem (%lld B) not a multiple of 16",
                (long long)head_bytes);
  const int64_t strides[] = {a->key_stride_token,   a->key_stride_head,  a->value_stride_token,
                             a->value_stride_head,  a->cache_stride_block, a->cache_stride_row,
                             a->cache_stride_head};
  for (int64_t s : strides)
    if ((s * esz) % 16 != 0)
      return fail(SB_ERR_INVALID, "sb_kv_append: stride %lld elements is not 16-byte aligned",
                  (long long)s);
  if (!aligned16(a->key) || !aligned16(a->value) || !aligned16(a->k_cache) || !aligned16(a->v_cache))
    return fail(SB_ERR_INVALID, "sb_kv_append: tensor base not 16-byte aligned");
  if ((a->num_tokens * 2 + 3) / 4 > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_kv_append: too many tokens");
  return SB_OK;
}

}  // namespace sb_host

extern "C" int sb_kv_append(const sb_kv_append_args *a) {
  using namespace sb_host;
  if (const int rc = check_kv_append(a)) return rc;
  if (a->num_tokens == 0) return SB_OK;
  const int esz = a->dtype == SB_F32 ? 4 : 2;
  const int chunks_per_head = a->head_size * esz / 16;
  const int n_chunks = chunks_per_head * a->num_kv_heads;
  const int64_t blocks = (a->num_tokens * 2 + 3) / 4;
  hipLaunchKernelGGL(kv_append_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)a->stream,
                     (const char *)a->key, (const char *)a->value, (char *)a->k_cache,
                     (char *)a->v_cache, a->slot_mapping, a->num_tokens, chunks_per_head, n_chunks,
                     a->block_size, a->key_stride_token * esz, a->key_stride_head * esz,
                     a->value_stride_token * esz, a->value_stride_head * esz,
                     a->cache_stride_block * esz, a->cache_stride_row * esz,
                     a->cache_stride_head * esz);
  return check_launch("kv_append_kernel");
}

extern "C" int sb_copy_blocks(void *cache, const int64_t *pairs, int64_t num_pairs,
                              int64_t block_bytes, int64_t stride_block_bytes, void *stream) {
  using namespace sb_host;
  if (num_pairs < 0) return fail(SB_ERR_INVALID, "sb_copy_blocks: negative num_pairs");
  if (num_pairs == 0) return SB_OK;
  if (!cache || !pairs) return fail(SB_ERR_INVALID, "sb_copy_blocks: null pointer");
  if (block_bytes <= 0 || block_bytes % 16 != 0 || stride_block_bytes % 16 != 0 || !aligned16(cache))
    return fail(SB_ERR_INVALID, "sb_copy_blocks: sizes must be positive multiples of 16 bytes");
  if (num_pairs > 65535) return fail(SB_ERR_UNSUPPORTED, "sb_copy_blocks: more than 65535 pairs");
  const unsigned gx = (unsigned)((block_bytes / 16 + 255) / 256);
  hipLaunchKernelGGL(copy_blocks_kernel, dim3(gx, (unsigned)num_pairs), dim3(256), 0,
                     (hipStream_t)stream, (char *)cache, pairs, block_bytes, stride_block_bytes);
  return check_launch("copy_blocks_kernel");
}

namespace {

int check_window_shift(const sb_window_shift_args *a) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_window_shift: null args");
  if (a->planes < 0 || a->keep_rows < 0 || a->n_new < 0)
    return fail(SB_ERR_INVALID, "sb_window_shift: negative size");
  const int64_t rows = a->keep_rows + a->n_new;
  if (a->planes == 0 || rows == 0) return SB_OK;
  if (!a->dst || (a->keep_rows > 0 && !a->src) || (a->n_new > 0 && !a->fresh))
    return fail(SB_ERR_INVALID, "sb_window_shift: null pointer");
  if (a->row_bytes <= 0 || a->row_bytes % 16 != 0 || a->src_stride_plane_bytes % 16 != 0 ||
      a->dst_stride_plane_bytes % 16 != 0 || a->fresh_stride_plane_bytes % 16 != 0 ||
      a->fresh_stride_row_bytes % 16 != 0 || !aligned16(a->dst) || !aligned16(a->src) ||
      !aligned16(a->fresh))
    return fail(SB_ERR_INVALID, "sb_window_shift: rows and strides must be 16-byte multiples");
  if (a->planes > 65535) return fail(SB_ERR_UNSUPPORTED, "sb_window_shift: more than 65535 planes");
  const int64_t gx = (rows * (a->row_bytes / 16) + 255) / 256;
  if (gx > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_window_shift: too many rows");
  return SB_OK;
}

bool same_rows(const sb_window_shift_args *k, const sb_window_shift_args *v) {
  return k->planes == v->planes && k->keep_rows == v->keep_rows && k->src_row0 == v->src_row0 &&
         k->dst_row0 == v->dst_row0 && k->n_new == v->n_new && k->row_bytes == v->row_bytes &&
         k->src_stride_plane_bytes == v->src_stride_plane_bytes &&
         k->dst_stride_plane_bytes == v->dst_stride_plane_bytes &&
         k->fresh_stride_plane_bytes == v->fresh_stride_plane_bytes &&
         k->fresh_stride_row_bytes == v->fresh_stride_row_bytes && k->stream == v->stream;
}

// one launch for a, and for b too when given (same rows and strides as a)
int launch_window_shift(const sb_window_shift_args *a, const sb_window_shift_args *b) {
  const int64_t rows = a->keep_rows + a->n_new;
  if (a->planes == 0 || rows == 0) return SB_OK;
  const int64_t gx = (rows * (a->row_bytes / 16) + 255) / 256;
  ShiftTensors t;
  const sb_window_shift_args *const half[2] = {a, b ? b : a};
  for (int i = 0; i < 2; ++i) {
    t.src[i] = (const char *)half[i]->src;
    t.dst[i] = (char *)half[i]->dst;
    t.fresh[i] = (const char *)half[i]->fresh;
  }
  hipLaunchKernelGGL(window_shift_kernel, dim3((unsigned)gx, (unsigned)a->planes, b ? 2u : 1u), dim3(256), 0,
                     (hipStream_t)a->stream, t, a->keep_rows, a->src_row0, a->dst_row0, a->n_new, a->row_bytes,
                     a->src_stride_plane_bytes, a->dst_stride_plane_bytes, a->fresh_stride_plane_bytes,
                     a->fresh_stride_row_bytes);
  return sb_host::check_launch("window_shift_kernel");
}

}  // namespace

extern "C" int sb_window_shift(const sb_window_shift_args *a) {
  const int rc = check_window_shift(a);
  return rc != SB_OK ? rc : launch_window_shift(a, nullptr);
}

extern "C" int sb_window_shift_pair(const sb_window_shift_args *k, const sb_window_shift_args *v) {
  int rc = check_window_shift(k);
  if (rc == SB_OK) rc = check_window_shift(v);
  if (rc != SB_OK) return rc;
  if (same_rows(k, v)) return launch_window_shift(k, v);
  rc = launch_window_shift(k, nullptr);
  return rc != SB_OK ? rc : launch_window_shift(v, nullptr);
}

namespace {

int check_dense_rows(const sb_dense_rows_args *a) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_dense_rows: null args");
  if (a->batch < 0 || a->num_queries < 0 || a->num_keys < 0 || a->mask_cols < 0)
    return fail(SB_ERR_INVALID, "sb_dense_rows: negative size");
  if (a->batch == 0) return SB_OK;
  if (a->batch > 0x7fffffffLL || a->num_keys > 0x7fffffffLL || a->mask_cols > 0x7fffffffLL)
    return fail(SB_ERR_UNSUPPORTED, "sb_dense_rows: sizes beyond 2^31 - 1");
  const int m = a->mask ? a->mask_elem_bytes : 1;
  if (m != 1 && m != 2 && m != 4 && m != 8) return fail(SB_ERR_UNSUPPORTED, "sb_dense_rows: mask elements of %d bytes", m);
  return SB_OK;
}

template <typename M>
int launch_dense_rows(const sb_dense_rows_args *a, const NewRows *s) {
  const DenseRows p = {a->mask, a->mask_cols, a->mask_stride_row, a->mask_stride_col, a->num_queries, a->num_keys, a->kv_step,
                       a->seq_lens, a->row_seq, a->key_lo, a->kv_start};
  if (s) {
    const int64_t blocks = (2 * s->planes * s->n_new * s->chunks + 1023) / 1024;
    hipLaunchKernelGGL(dense_step_kernel<M>, dim3((unsigned)(a->batch + blocks)), dim3(1024), 0, (hipStream_t)a->stream, p, *s, (unsigned)a->batch);
    return sb_host::check_launch("dense_step_kernel");
  }
  hipLaunchKernelGGL(dense_rows_kernel<M>, dim3((unsigned)a->batch), dim3(1024), 0, (hipStream_t)a->stream, p);
  return sb_host::check_launch("dense_rows_kernel");
}
int launch_dense_rows(const sb_dense_rows_args *a, const NewRows *s) {
  switch (a->mask ? a->mask_elem_bytes : 1) {
    case 1: return launch_dense_rows<uint8_t>(a, s);
    case 2: return launch_dense_rows<uint16_t>(a, s);
    case 4: return launch_dense_rows<uint32_t>(a, s);
    default: return launch_dense_rows<uint64_t>(a, s);
  }
}

}  // namespace

extern "C" int sb_dense_rows(const sb_dense_rows_args *a) {
  const int rc = check_dense_rows(a);
  return rc != SB_OK || a->batch == 0 ? rc : launch_dense_rows(a, nullptr);
}

extern "C" int sb_dense_step(const sb_window_shift_args *k, const sb_window_shift_args *v, const sb_dense_rows_args *rows) {
  int rc = check_window_shift(k);
  if (rc == SB_OK) rc = check_window_shift(v);
  if (rc == SB_OK) rc = check_dense_rows(rows);
  if (rc != SB_OK) return rc;
  const int64_t chunks = k->row_bytes / 16, blocks = (2 * k->planes * k->n_new * chunks + 1023) / 1024;
  if (same_rows(k, v) && k->keep_rows == 0 && k->planes > 0 && k->n_new > 0 && rows->batch > 0 && k->stream == rows->stream &&
      rows->batch + blocks <= 0x7fffffffLL) {
    const NewRows s = {{(char *)k->dst, (char *)v->dst}, {(const char *)k->fresh, (const char *)v->fresh}, k->planes, k->n_new, chunks,
                       k->dst_stride_plane_bytes, k->dst_row0 * k->row_bytes, k->row_bytes, k->fresh_stride_plane_bytes,
                       k->fresh_stride_row_bytes};
    return launch_dense_rows(rows, &s);
  }
  rc = sb_window_shift_pair(k, v);
  return rc != SB_OK ? rc : sb_dense_rows(rows);
}

// ---- plain streaming copy: the bandwidth yardstick bench.py reports next to the kernels and the
// known-size launch that hardware byte counters are calibrated against --------------------------
namespace {
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void stream_copy_kernel(const u32x4_t *__restrict__ src,
                                                          u32x4_t *__restrict__ dst, int64_t n16) {
  int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * 1024;
  for (; i + 768 < n16; i += stride) {
    u32x4_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = __builtin_nontemporal_load(src + i + 256 * u);
#pragma unroll
    for (int u = 0; u < 4; ++u) __builtin_nontemporal_store(v[u], dst + i + 256 * u);
  }
}
}  // namespace

extern "C" int sb_stream_copy(void *dst, const void *src, int64_t bytes, void *stream) {
  using namespace sb_host;
  if (bytes < 0 || bytes % 16384 != 0) return fail(SB_ERR_INVALID, "sb_stream_copy: bytes must be a multiple of 16384");
  if (bytes == 0) return SB_OK;
  if (!dst || !src || !aligned16(dst) || !aligned16(src))
    return fail(SB_ERR_INVALID, "sb_stream_copy: null or misaligned pointer");
  const int64_t n16 = bytes / 16;
  int64_t blocks = n16 / 1024;
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(stream_copy_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const u32x4_t *)src, (u32x4_t *)dst, n16);
  return check_launch("stream_copy_kernel");
}
