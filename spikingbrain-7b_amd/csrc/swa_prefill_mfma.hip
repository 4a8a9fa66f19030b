// Causal sliding-window attention for many query tokens per sequence (prefill, chunked prefill,
// multi-token decode), bf16/fp16, on the matrix cores. Keys/values come either from the step's own
// key/value tensors (plain prompt) or from the paged cache through the block table (chunked prefill,
// prefix reuse). Replaces the varlen flash-attention call of
// vllm_hymeta/attention/fa_kernel_metatoken.py:235-253 (window_size=(window_left, 0), causal aligned to
// the end of the key sequence).
//
// Work decomposition
//   grid = (query tiles of 64 tokens, kv heads, groups of 4 or 3 query heads of the kv head, or of 2 and 1 in small
//   calls; parts of the tile's keys); a workgroup covers one of those groups (7 = 4 + 3 = 2 + 2 + 2 + 1; behind groups of
//   four a last group of 1 or 2 heads takes a launch of its own). A wavefront owns "column blocks" of 16 tokens x 1
//   head (no padding): a pair of heads is served by 4 wavefronts (one per 16-token sub-tile, a block of each head),
//   an odd last head by 4 wavefronts of one block each - 8 wavefronts for 4 heads and for 3. At 256 registers per
//   wavefront two of them share a SIMD.
//   The workgroup walks the union of its tokens' windows in chunks of 32 keys. Each chunk of K and V
//   (32 rows x 256 B each) is fetched from global memory ONCE per workgroup (every wavefront of an
//   8-wavefront workgroup fetches 4 rows with whole-row 16-byte lanes, else the first four fetch 8) into a
//   ring of three LDS chunks whose rows are padded to 288 B; all wavefronts then read their MFMA operands
//   from LDS. Global loads run three chunks ahead of the arithmetic (two register sets used alternately, the
//   loop written out for both). They are ordinary cached loads: the neighbouring query tiles, which run at
//   the same time on the same XCD, read the same rows. The arithmetic is staggered over two chunks: an
//   iteration issues the scores of chunk x+1 ahead of the numerators of chunk x, and the P V product of
//   chunk x ahead of the masking and maxima of chunk x+1, so that a wavefront's matrix instructions have
//   vector work of another chunk behind them.
//   A wavefront issues about one instruction per 5 cycles whatever its kind, and a scalar branch costs 15-25
//   cycles, so the loop is kept short: everything that does not depend on the lane lives in scalar registers
//   (a chunk's address is one block-table entry, read one iteration ahead, times the block stride, plus the
//   K and V bases; a lane adds a 32-bit offset), the range of chunks that need no masking is computed once,
//   and the rare paths (masking, raising the reference point) sit behind one branch each.
//   Meta rows, when given, are taken in a loop of their own in front of the walk.
//   Per chunk and column block: S^T = K Q^T (8 MFMA 16x16x32, tokens on the N axis), softmax numerators
//   per lane for token lane%16 in log2 units, O^T += V^T P^T (8 MFMA). P stays in the lane that produced
//   it; V^T operands come out of the [key][dim] stage through the transposing LDS load, shared by the two
//   blocks.
//   Workgroups are numbered so that each XCD (own L2) works through one contiguous run of tiles.
//
// Softmax reference point
//   The numerators are exp2(s - m_ref) with a per-row reference m_ref that is only raised when some
//   row of the wavefront scores more than kRaise (log2 units) above it, so they stay below 2^kRaise
//   (exact in fp32 sums, inside fp16 range). The check uses each lane's own 8 keys, so the common case
//   has no cross-lane traffic; raising m_ref (rare after the first chunks) takes the row maximum over
//   the four lanes of a token and rescales the output accumulators.
#include <algorithm>
#include <cmath>
#include <functional>

#include "common.h"
#include "mfma_util.h"

namespace sb_host {
int check_kv_append(const sb_kv_append_args *a);   // cache_ops.hip
}

namespace {

using namespace sb;

// An append of this call's keys and values that rides in the launch (see append_rides): workgroups from `first` on copy rows.
struct Append {
  const char *key, *value;
  char *k_cache, *v_cache;
  const int64_t *slots;
  int64_t tokens;
  unsigned first;
  int n_chunks, block_size;    // 16-byte chunks of a row (16 per head)
  int64_t key_st, key_sh, val_st, val_sh, blk, row, head;   // bytes
};
constexpr int kAppendTokens = 4;   // of a wavefront: eight rows in flight

struct PrefillParams {
  const char *q;
  const char *k;
  const char *v;
  char *out;
  float *lse;                 // [total_q, Hq] natural-log log-sum-exp, or null
  // byte-code caches (paged): per-row INT8 scales [nb, Hkv, bs], or one fp8 scale per tensor
  const float *k_scale;
  const float *v_scale;
  float k_scale_tensor, v_scale_tensor;
  int Hkv;
  const int32_t *block_table;
  const int64_t *kv_start;
  const int32_t *kv_start32;
  const int32_t *key_lo;      // [S] first visible key of each sequence, or null
  const int32_t *cu_q;        // [S+1] first q/out row of each sequence
  const int32_t *seq_lens_k;  // [S] keys of each sequence (context + new tokens)
  const int32_t *tile_seq;    // [tiles] sequence of each 64-token query tile
  const int32_t *tile_q0;     // [tiles] first query (index inside its sequence) of the tile
  int G, head_begin;          // query heads per kv head; first of them handled by this launch
  int Hq;
  int num_tiles;
  int bucket, head_groups;    // order of an XCD's workgroups (see the kernel); bucket 0: not by XCD
  int block_size, window_left;
  int tiles_per_block;        // block_size / 16
  TileDivision tile_div;      // by tiles_per_block
  float scale_log2;
  int64_t q_sr, q_sh, o_sr, o_sh;  // elements
  int64_t kv_sb, kv_sr, kv_sh;     // bytes
  int64_t bt_stride;
  // Meta tokens: meta_len rows [meta_len, Hkv, 128] of the query's type every query also attends to,
  // unmasked, in the same softmax: they are walked as the chunks in front of the window's. 0 = none.
  const char *meta_k;
  const char *meta_v;
  int meta_len;
  int64_t meta_sr, meta_sh;  // bytes
  ScoreOptions opt;          // soft cap / ALiBi slopes, applied to every raw score in front of the mask
  // ALiBi term of meta row j for packed query row t: -slope * |meta_bias_off + t - j|, meta_bias_off = row0 + meta_len - rows
  int meta_bias_off;
  // Key split: a tile's walk is cut into up to n_parts parts of part_chunks chunks (the last part takes what is left),
  // a workgroup each; a tile that fits one part stores its output itself, the others fp32 partials: numerators
  // [query row, query head, n_parts, 128] and (reference point, denominator) [query row, query head, n_parts, 2].
  int n_parts, part_chunks;
  float *ws_acc;
  float *ws_ml;
  Append append;              // tokens 0: none
};

// The walk of a tile in 32-key chunks: every chunk that holds a key some token of the tile can see.
struct Walk {
  int lo, hi;  // keys [lo, hi)
  int ch_begin, ch_end;
};
__device__ __forceinline__ Walk tile_walk(const PrefillParams &p, int seq, int q0, int Lq, int Lk) {
  Walk w;
  const int shift = Lk - Lq;  // query j sits at key index shift + j
  const int klo = p.key_lo ? max(p.key_lo[seq], 0) : 0;
  w.hi = shift + min(q0 + 63, Lq - 1) + 1;
  // (kept inside the sequence even when padding hides every key: such rows end up fully masked)
  w.lo = min(max(p.window_left >= 0 ? shift + q0 - p.window_left : 0, klo), w.hi - 1);
  w.ch_begin = w.lo >> 5;
  w.ch_end = ((w.hi - 1) >> 5) + 1;
  return w;
}
__device__ __forceinline__ int tile_parts(const PrefillParams &p, const Walk &w) {
  return min(p.n_parts, (w.ch_end - w.ch_begin + p.part_chunks - 1) / p.part_chunks);
}

constexpr int kRowPad = 288;   // LDS row stride of a K chunk: 256 B of data + 32 B (16-byte operand loads of 16 rows: measured 1.6 x the rate of a 272 B stride)
constexpr int kRowPadV = 288;  // of a V chunk: 256 B + 32 B (transposing loads: 4 rows x 32 B at a time)
constexpr int kStageK = 32 * kRowPad, kStageV = 32 * kRowPadV;
constexpr int kStage = kStageK + kStageV;  // one chunk of K and V

// ds_read_b64_tr_b16: in every group of 16 lanes, lane i names 8 bytes (4 elements) of LDS, "row i"; lane l
// receives element l % 4 of rows l / 4, l / 4 + 4, l / 4 + 8, l / 4 + 12. With row i = (key k0 + i / 4, dims
// d0 + 4 (i % 4) .. + 3), lane l gets dim d0 + l of keys k0 .. k0 + 3: V^T straight out of a [key][dim] stage.
__device__ __forceinline__ uint2 load_transposed(const char *row) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)row);
  return __builtin_bit_cast(uint2, v);
}
constexpr int kHandOver = 2048 * 4 + 1024;   // bytes of one wavefront's block between the halves of a walk: sums, reference points and denominators
static_assert(8 * kHandOver <= 6 * kStage, "hand-over of two sets of four wavefronts");
constexpr float kNegInf = kNegInfF;
constexpr float kRaise = 8.f;

// NHEADS query heads of one kv head per workgroup: head pairs are served by 4 wavefronts of two column blocks (one
// 16-token sub-tile, both heads of the pair), an odd last head by 4 of one. NHEADS = 4 also serves 3 heads and NHEADS = 2
// one, so that all groups of a GQA group of 7 are one launch either way.
// HALVES: the workgroup holds that set of wavefronts twice, and each takes half of the walk through a ring of its own; at the
// end they put their sums together in LDS.
template <int NHEADS, bool HALVES>
struct Shape {
  static constexpr int kSetWaves = 4 * (NHEADS / 2) + 4 * (NHEADS % 2);
  static constexpr int kWaves = kSetWaves * (HALVES ? 2 : 1);
  static constexpr int kFetchWaves = kSetWaves == 8 ? 8 : 4;    // wavefronts (of a set) that move K/V into LDS
  static constexpr int kLoads = 8 / kFetchWaves;                // 4-row loads per fetching lane, per K and per V
};

// The registers a fetching lane carries a chunk in: 16-byte pieces of K and V rows, or, for a byte-code
// cache (KVQ = SB_KV_INT8 / SB_KV_FP8), the 8 codes that become such a piece plus (INT8) their row's scales.
template <int KVQ, int N>
struct StageSet {
  uint4 k[N], v[N];
};
template <int N>
struct StageSet<SB_KV_INT8, N> {
  uint2 k[N], v[N];
  float ks[N], vs[N];
};
template <int N>
struct StageSet<SB_KV_FP8, N> {
  uint2 k[N], v[N];
};

template <int Q, int B>
__device__ __forceinline__ float code_value(uint32_t w) {
  if constexpr (Q == SB_KV_INT8) return (float)(int)(int8_t)(w >> (8 * B));
  else return __builtin_amdgcn_cvt_f32_fp8((int)w, B);
}
// 8 codes times their scale, rounded to E: the values the reference attends to after its own
// quantise-dequantise (code * scale cast back to the tensor's dtype)
template <typename E, int Q>
__device__ __forceinline__ uint4 dequant8(uint2 w, float s) {
  return make_uint4(Mma<E>::pack(code_value<Q, 0>(w.x) * s, code_value<Q, 1>(w.x) * s),
                    Mma<E>::pack(code_value<Q, 2>(w.x) * s, code_value<Q, 3>(w.x) * s),
                    Mma<E>::pack(code_value<Q, 0>(w.y) * s, code_value<Q, 1>(w.y) * s),
                    Mma<E>::pack(code_value<Q, 2>(w.y) * s, code_value<Q, 3>(w.y) * s));
}

__device__ __forceinline__ void append_rows(const PrefillParams &p, int64_t wave, int lane) {
  const int64_t tok0 = wave * kAppendTokens, last = p.append.tokens - 1;
  if (tok0 > last) return;
  for (int c = lane; c < p.append.n_chunks; c += 64) {
    const int64_t h = c >> 4, w = (int64_t)(c & 15) * 16;
    const char *const key = p.append.key + h * p.append.key_sh + w, *const value = p.append.value + h * p.append.val_sh + w;
    u32x4_t k[kAppendTokens], v[kAppendTokens];
#pragma unroll
    for (int u = 0; u < kAppendTokens; ++u) {
      const int64_t tok = min(tok0 + u, last);
      k[u] = *reinterpret_cast<const u32x4_t *>(key + tok * p.append.key_st);
      v[u] = *reinterpret_cast<const u32x4_t *>(value + tok * p.append.val_st);
    }
#pragma unroll
    for (int u = 0; u < kAppendTokens; ++u) {
      if (tok0 + u > last) continue;
      const int64_t slot = p.append.slots[tok0 + u];
      if (slot < 0) continue;   // (padded lane / token older than the window)
      const int64_t blk = slot / p.append.block_size;
      const int64_t at = blk * p.append.blk + (slot - blk * p.append.block_size) * p.append.row + h * p.append.head + w;
      *reinterpret_cast<u32x4_t *>(p.append.k_cache + at) = k[u];
      *reinterpret_cast<u32x4_t *>(p.append.v_cache + at) = v[u];
    }
  }
}

// ODD: the last group of heads may have one less (3 of 4, 1 of 2): a build of its own, because the second path costs
// the kernel of two heads 5 % (16 : 8 heads, 2000 tokens behind 3000 95 -> 100 us).
// APPEND: with the append that rides along (in-flight elements): builds of their own, because its code and arguments in front cost
// the calls without one 0.5 us (64 tokens, 28 : 4 heads 8.3 -> 8.8, behind 2000 18.7 -> 19.3; 8 : 8 5.4 -> 6.0).
template <typename E, int NHEADS, int KVQ, bool PAGED, bool ODD, bool HALVES, bool APPEND>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * Shape<NHEADS, HALVES>::kWaves, 64 * Shape<NHEADS, HALVES>::kWaves),
                          amdgpu_waves_per_eu(2, 2)))
void swa_prefill_kernel(const PrefillParams p) {
  using S = Shape<NHEADS, HALVES>;
  __shared__ __attribute__((aligned(16))) char smem_all[(HALVES ? 6 : 3) * kStage];  // ring(s) of three chunks, each [K|V]

  if constexpr (APPEND) {
    if (blockIdx.x >= p.append.first) {   // (the whole workgroup, ahead of every barrier)
      if (blockIdx.y == 0)
        append_rows(p, (int64_t)(blockIdx.x - p.append.first) * S::kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                    threadIdx.x & 63);
      return;
    }
  }
  // Workgroups are handed to the 8 XCDs round-robin by index, and each XCD has its own L2. Give XCD x
  // the x-th contiguous eighth of the tiles, so that the workgroups resident on one XCD at a time are
  // neighbouring tiles of one sequence and kv head, whose key windows overlap almost entirely.
  // Inside an XCD's list the order is: buckets of p.bucket tiles, in a bucket the head groups, in those the kv heads,
  // in those the tiles.
  const int per_xcd = (p.num_tiles + 7) >> 3;
  const int per_tile = p.Hkv * p.head_groups;
  int tile, pair;
  if (HALVES && p.bucket == 0) {
    // lists dealt longest walk first, walked in that order over all XCDs: no XCD has to itself what starts last (where all
    // workgroups start together the order of tile_order shares keys in an XCD's L2: 12 : 4, 2048 behind 10000 75.6 us, this way 81.7)
    const int rank = blockIdx.x / per_tile;
    tile = (rank & 7) * per_xcd + (rank >> 3);
    pair = blockIdx.x - rank * per_tile;
  } else {
    const int at = blockIdx.x >> 3;
    const int bucket = at / (p.bucket * per_tile);
    const int width = min(p.bucket, per_xcd - bucket * p.bucket);   // tiles of this bucket
    const int in_bucket = at - bucket * p.bucket * per_tile;
    pair = in_bucket / width;
    // (the parts of a tile go to XCDs one after the other: a call of one tile would otherwise run on one of them)
    tile = ((blockIdx.x + blockIdx.y) & 7) * per_xcd + bucket * p.bucket + (in_bucket - pair * width);
  }
  if (tile >= p.num_tiles) return;
  const int head_group = pair / p.Hkv, kvh = pair - head_group * p.Hkv;
  const int head_begin = p.head_begin + NHEADS * head_group;
  const int nheads = ODD ? min(NHEADS, p.G - head_begin) : NHEADS;
  const int tid = threadIdx.x;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = HALVES ? wave_all / S::kSetWaves : 0, wave = HALVES ? wave_all % S::kSetWaves : wave_all;
  char *const smem = smem_all + half * 3 * kStage;
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int c = lane & 15;

  const int seq = p.tile_seq[tile];
  const int q0 = p.tile_q0[tile];
  const int qrow0 = p.cu_q[seq];
  const int Lq = p.cu_q[seq + 1] - qrow0;
  const int Lk = p.seq_lens_k[seq];
  const int shift = Lk - Lq;  // query j sits at key index shift + j
  const int wl = p.window_left;

  // keys any token of this workgroup can see: [wg_lo, wg_hi)
  const Walk walk = tile_walk(p, seq, q0, Lq, Lk);
  const int wg_lo = walk.lo, wg_hi = walk.hi;
  const int klo = p.key_lo ? max(p.key_lo[seq], 0) : 0;
  const int first_tile = wg_lo >> 4, last_tile = (wg_hi - 1) >> 4;
  // this workgroup's part of the walk
  const int part = blockIdx.y, parts = tile_parts(p, walk);
  if (part >= parts) return;  // (the whole workgroup, ahead of every barrier)
  const int part_begin = walk.ch_begin + part * p.part_chunks;
  const int part_end = part + 1 == parts ? walk.ch_end : part_begin + p.part_chunks;
  // (halves are of one length: where the second has a chunk less, its last lies past every token and is masked)
  const int n_walk = HALVES ? (part_end - part_begin + 1) >> 1 : part_end - part_begin;
  const int ch_begin = part_begin + half * n_walk;  // the walk: index x is window chunk ch_begin + x
  const int meta_chunks = !HALVES && part == 0 ? (p.meta_len + 31) >> 5 : 0;   // (calls with meta rows do not take halves)

  // Everything from here on is written for NB column blocks per wavefront: two for the wavefronts of a head
  // pair, one for those of an odd last head (four wavefronts, one per 16-token sub-tile).
  auto run = [&](auto nb_tag) __attribute__((always_inline)) {
    constexpr int NB = decltype(nb_tag)::value;
    // this wavefront's NB column blocks: 16-token sub-tile ts[b] of head hd[b]
    int ts[NB], hd[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      ts[b] = wave & 3;
      hd[b] = NB == 2 ? 2 * (wave >> 2) + b : nheads - 1;
    }
    const int head0 = kvh * p.G + head_begin;
    // (rows past the end of the sequence repeat its last token; they are never stored)
    const int jw0 = min(q0 + 16 * ts[0], Lq - 1);            // first and last token of the wavefront
    const int jw_last = min(q0 + 16 * ts[NB - 1] + 15, Lq - 1);
    int my_pos[NB], my_lo[NB];
    uint4 qb[NB][4];  // Q^T operands: token lane%16 of the block, dims of 16-byte piece 4s+g
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int j_mine = min(q0 + 16 * ts[b] + c, Lq - 1);
      my_pos[b] = shift + j_mine;
      my_lo[b] = max(wl >= 0 ? my_pos[b] - wl : 0, klo);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        qb[b][s] = *reinterpret_cast<const uint4 *>(
            p.q + ((int64_t)(qrow0 + j_mine) * p.q_sr + (int64_t)(head0 + hd[b]) * p.q_sh + (4 * s + g) * 8) * 2);
    }
    // Chunks wholly visible to every token of the wavefront (at or above every token's lower bound, at or below
    // the first token) need no masking: walk indices [full_lo, full_lo + full_cnt).
    const int vis_lo = max(wl >= 0 ? shift + jw_last - wl : 0, klo);
    const int full_lo = ((vis_lo + 31) >> 5) - ch_begin;
    const unsigned full_cnt = (unsigned)max(((shift + jw0 + 1) >> 5) - ch_begin - full_lo, 0);

    f32x4_t acc[NB][8];
    float m[NB], l[NB];  // m: reference point of the numerators (log2 units), l: this lane's share of the sum
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      m[b] = kNegInf;
      l[b] = 0.f;
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) acc[b][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // ---- global -> registers -> LDS: the first kFetchWaves wavefronts move the chunk (32 K rows and
    // 32 V rows of 256 B); each of their loads covers 4 rows, all inside one 16-key tile of the table.
    // Rows outside [wg_lo, wg_hi) are clamped onto the nearest visible key (masked for every token).
    // Everything that does not depend on the lane is kept in scalar registers: per chunk, the tile's byte offset
    // (one block-table entry, looked up one call ahead of its use) added to the K and V bases; a lane adds its
    // row and column as a 32-bit offset.
    constexpr bool kFetchAll = S::kFetchWaves == S::kSetWaves;
    const bool fetcher = kFetchAll || wave < S::kFetchWaves;
    constexpr int rows_per_wave = 32 / S::kFetchWaves;                     // 4, 8 or 16
    const int tsel = (wave * rows_per_wave) >> 4;                          // which 16-key tile of a chunk this wavefront's rows are in
    const int lrow = (wave * rows_per_wave) % 16 + (lane >> 4);            // row inside the tile, +4 per load
    const uint32_t row_bytes = (uint32_t)p.kv_sr;                          // < 2^24 (host check)
    const uint32_t lane_col = c * (KVQ == SB_KV_NONE ? 16 : 8);
    const int64_t wg_off = (int64_t)kvh * p.kv_sh + (PAGED ? 0 : p.kv_start ? p.kv_start[seq] * p.kv_sr : p.kv_start32 ? p.kv_start32[seq] * p.kv_sr : 0);
    const char *const kbase = p.k + wg_off, *const vbase = p.v + wg_off;
    const int32_t *const table_row = PAGED ? p.block_table + (int64_t)seq * p.bt_stride : nullptr;
    auto walk_tile = [&](int x) __attribute__((always_inline)) {  // (past the end of the walk: the last tile again)
      return min(max(2 * (ch_begin + x) + tsel, first_tile), last_tile);
    };
    auto block_of = [&](int t) __attribute__((always_inline)) { return tile_block(t, p.tile_div); };
    int next_blk = 0;  // table entry of the tile the next fetch takes
    if constexpr (PAGED) next_blk = table_row[block_of(walk_tile(0))];
    int fx = 0;        // walk index the next fetch takes
    using Set = StageSet<KVQ, S::kLoads>;
    Set stage[2];  // walk index x travels in set x & 1
    auto fetch = [&](Set &st) __attribute__((always_inline)) {
      const int t = walk_tile(fx);
      ++fx;
      int64_t off;  // of the tile's first row from kbase / vbase
      [[maybe_unused]] int64_t scale_row = 0;  // INT8: index of that row in the scale tensors
      if constexpr (PAGED) {
        const int bi = block_of(t);
        const int64_t blk = next_blk;
        next_blk = table_row[block_of(walk_tile(fx))];
        const int in_block = (t - bi * p.tiles_per_block) << 4;
        off = blk * p.kv_sb + (int64_t)((uint32_t)in_block * row_bytes);
        if constexpr (KVQ == SB_KV_INT8) scale_row = (blk * p.Hkv + kvh) * p.block_size + in_block;
      } else {
        off = (int64_t)(t << 4) * p.kv_sr;
      }
      const char *const kp = kbase + off, *const vp = vbase + off;
      const int lo = wg_lo - (t << 4), hi = wg_hi - 1 - (t << 4);
#pragma unroll
      for (int u = 0; u < S::kLoads; ++u) {
        const int row = min(max(lrow + 4 * u, lo), hi);  // inside the tile: 0 .. 15
        const uint32_t vo = __umul24((uint32_t)row, row_bytes) + lane_col;
        if constexpr (KVQ == SB_KV_NONE) {
          st.k[u] = *reinterpret_cast<const uint4 *>(kp + vo);  // (cached: the neighbouring query tiles read the same rows)
          st.v[u] = *reinterpret_cast<const uint4 *>(vp + vo);
        } else {  // a row is 128 code bytes: 8 per lane
          const unsigned long long wk = *reinterpret_cast<const unsigned long long *>(kp + vo);
          const unsigned long long wv = *reinterpret_cast<const unsigned long long *>(vp + vo);
          st.k[u] = make_uint2((uint32_t)wk, (uint32_t)(wk >> 32));
          st.v[u] = make_uint2((uint32_t)wv, (uint32_t)(wv >> 32));
          if constexpr (KVQ == SB_KV_INT8) {
            st.ks[u] = (p.k_scale + scale_row)[(uint32_t)row];
            st.vs[u] = (p.v_scale + scale_row)[(uint32_t)row];
          }
        }
      }
    };
    const int stash_off = (wave * rows_per_wave + (lane >> 4)) * kRowPad + c * 16;   // of this lane's first row in a K chunk;
    const int stash_off_v = (wave * rows_per_wave + (lane >> 4)) * kRowPadV + c * 16 + kStageK;  // in the V chunk behind it
    auto stash = [&](int slot, const Set &st) __attribute__((always_inline)) {  // slot = byte offset of a ring slot
      char *sk = smem + slot + stash_off, *sv = smem + slot + stash_off_v;
#pragma unroll
      for (int u = 0; u < S::kLoads; ++u) {
        uint4 kq, vq;
        if constexpr (KVQ == SB_KV_NONE) {
          kq = st.k[u];
          vq = st.v[u];
        } else if constexpr (KVQ == SB_KV_INT8) {
          kq = dequant8<E, KVQ>(st.k[u], st.ks[u]);
          vq = dequant8<E, KVQ>(st.v[u], st.vs[u]);
        } else {
          kq = dequant8<E, KVQ>(st.k[u], p.k_scale_tensor);
          vq = dequant8<E, KVQ>(st.v[u], p.v_scale_tensor);
        }
        *reinterpret_cast<uint4 *>(sk + 4 * u * kRowPad) = kq;
        *reinterpret_cast<uint4 *>(sv + 4 * u * kRowPadV) = vq;
      }
    };

    // Scores live in two register sets used alternately: while the numerators of one chunk are formed in one set,
    // the matrix instructions write the next chunk's scores into the other. s[b][t][i]: block b, key 16 t + 4 g + i
    // of the chunk (raw dot products; -inf where masked).
    using Scores = f32x4_t[NB][2];
    Scores sa, sb2;
    float mx[NB];    // row maxima of the scores whose softmax comes next, in log2 units
    uint4 pb[NB];    // probabilities of the chunk whose P V product comes next

    // The two halves of an iteration. Each runs 16 matrix instructions next to the vector work of another chunk
    // that does not depend on them.
    //
    // first half: S^T = K Q^T of the next chunk (kNext; K from ring slot `slot`) into `sn`, next to the
    // numerators of the chunk in `sc` against the current reference points (kCur) -> pb, l.
    auto first_half = [&](int slot, Scores &sn, Scores &sc, auto next_tag, auto cur_tag) __attribute__((always_inline)) {
      constexpr bool kNext = decltype(next_tag)::value, kCur = decltype(cur_tag)::value;
      const char *sk0 = smem + slot + c * kRowPad + g * 16, *sk1 = sk0 + 16 * kRowPad;
      uint4 k0[4], k1[4];  // operand loads run one step ahead of their use (two pairs live)
      if constexpr (kNext) {
        k0[0] = *reinterpret_cast<const uint4 *>(sk0);
        k1[0] = *reinterpret_cast<const uint4 *>(sk1);
#pragma unroll
        for (int b = 0; b < NB; ++b) sn[b][0] = sn[b][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      float m_safe[NB], psum[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) m_safe[b] = (m[b] == kNegInf) ? 0.f : m[b];
      if constexpr (kNext) {  // 2 NB chains (block, tile), each four instructions deep, taken in turn
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (s + 1 < 4) {
            k0[s + 1] = *reinterpret_cast<const uint4 *>(sk0 + (s + 1) * 64);
            k1[s + 1] = *reinterpret_cast<const uint4 *>(sk1 + (s + 1) * 64);
          }
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            sn[b][0] = Mma<E>::run(k0[s], qb[b][s], sn[b][0]);
            sn[b][1] = Mma<E>::run(k1[s], qb[b][s], sn[b][1]);
          }
        }
      }
      if constexpr (kCur) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          psum[b] = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float e = fast_exp2(fmaf(sc[b][j >> 2][j & 3], p.scale_log2, -m_safe[b]));
            sc[b][j >> 2][j & 3] = e;
            psum[b] += e;
          }
        }
      }
      if constexpr (kCur) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          l[b] += psum[b];
          pb[b] = make_uint4(Mma<E>::pack(sc[b][0][0], sc[b][0][1]), Mma<E>::pack(sc[b][0][2], sc[b][0][3]),
                             Mma<E>::pack(sc[b][1][0], sc[b][1][1]), Mma<E>::pack(sc[b][1][2], sc[b][1][3]));
        }
      }
    };

    // second half: O^T += V^T P^T (kPV; probabilities pb), next to the row maxima of the (masked) scores `sn` of
    // the next chunk (kPost). True when some row of that chunk needs a higher reference point.
    // V^T operands of a chunk, dims 16 mt + c: this lane's 8 keys (4g .. 4g+3 of either 16-key tile, the order of
    // its probabilities) by two transposing loads per mt; built once, used by both blocks. They are requested at
    // the top of an iteration and arrive while the first half runs.
    uint2 vlo[8], vhi[8];
    auto load_v = [&](int slot) __attribute__((always_inline)) {
      const char *v0 = smem + slot + kStageK + (4 * g + (c >> 2)) * kRowPadV + (c & 3) * 8, *v1 = v0 + 16 * kRowPadV;
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) {
        vlo[mt] = load_transposed(v0 + mt * 32);
        vhi[mt] = load_transposed(v1 + mt * 32);
      }
    };
    auto second_half = [&](const Scores &sn, auto pv_tag, auto post_tag) __attribute__((always_inline)) -> bool {
      constexpr bool kPV = decltype(pv_tag)::value, kPost = decltype(post_tag)::value;
      float t[NB];
      if constexpr (kPV) {
#pragma unroll
        for (int mt = 0; mt < 8; ++mt)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            acc[b][mt] = Mma<E>::run(make_uint4(vlo[mt].x, vlo[mt].y, vhi[mt].x, vhi[mt].y), pb[b], acc[b][mt]);
      }
      if constexpr (kPost) {  // each lane checks its own 8 keys: no cross-lane traffic unless the reference point must move
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          t[b] = kNegInf;
#pragma unroll
          for (int j = 0; j < 8; ++j) t[b] = fmaxf(t[b], sn[b][j >> 2][j & 3]);
        }
      }
      bool raise = false;
      if constexpr (kPost) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          mx[b] = t[b] * p.scale_log2;
          raise |= mx[b] > m[b] + kRaise;  // also true for the first finite score of a row (m = -inf)
        }
      }
      return __builtin_amdgcn_ballot_w64(raise) != 0;
    };
    // Soft cap / ALiBi on the scores of walk index xn, in place (only when asked for: one uniform branch).
    float my_slope[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) my_slope[b] = p.opt.slopes ? p.opt.slopes[head0 + hd[b]] : 0.f;
    auto adjust_scores = [&](int xn, Scores &sn) __attribute__((always_inline)) {
      if (!p.opt.on) return;
      const int c0 = (ch_begin + xn) << 5;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          sn[b][j >> 2][j & 3] = adjust_score(p.opt, sn[b][j >> 2][j & 3], my_slope[b],
                                              (float)(c0 + ((j >> 2) << 4) + 4 * g + (j & 3) - my_pos[b]));
    };
    // Masking of the scores of walk index xn, in place (selects, not branches: the comparison results are
    // combined as bits). Skipped for the chunks every token of the wavefront sees whole.
    auto mask_scores = [&](int xn, Scores &sn) __attribute__((always_inline)) {
      if ((unsigned)(xn - full_lo) < full_cnt) return;
      const int c0 = (ch_begin + xn) << 5;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int key = c0 + ((j >> 2) << 4) + 4 * g + (j & 3);
          sn[b][j >> 2][j & 3] = bool((key > my_pos[b]) | (key < my_lo[b])) ? kNegInf : sn[b][j >> 2][j & 3];
        }
    };
    const std::true_type kYes{};
    const std::false_type kNo{};

    // lift the reference points to the running maxima and rescale what has been accumulated
    auto rescale = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float t = mx[b];  // row maximum over the four lanes that share a token
        t = fmaxf(t, __shfl_xor(t, 16));
        t = fmaxf(t, __shfl_xor(t, 32));
        const float m_new = fmaxf(m[b], t);
        const float m_safe = (m_new == kNegInf) ? 0.f : m_new;
        const float alpha = fast_exp2(m[b] - m_safe);
        m[b] = m_new;
        l[b] *= alpha;
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) acc[b][mt] *= alpha;
      }
    };

    if (fetcher) {
      fetch(stage[0]);
      fetch(stage[1]);
    }
    // ---- meta rows: global -> ring slot 0 -> scores, one chunk at a time, while the first two chunks of the
    // window are on their way (every row that exists is visible to every token)
    for (int mc = 0; mc < meta_chunks; ++mc) {
      if (fetcher) {
        const char *mk = p.meta_k + (int64_t)kvh * p.meta_sh + c * 16, *mv = p.meta_v + (int64_t)kvh * p.meta_sh + c * 16;
#pragma unroll
        for (int u = 0; u < S::kLoads; ++u) {
          const int kk = wave * rows_per_wave + (lane >> 4) + 4 * u;
          const int64_t row = min((mc << 5) + kk, p.meta_len - 1);
          *reinterpret_cast<uint4 *>(smem + kk * kRowPad + c * 16) = *reinterpret_cast<const uint4 *>(mk + row * p.meta_sr);
          *reinterpret_cast<uint4 *>(smem + kStageK + kk * kRowPadV + c * 16) =
              *reinterpret_cast<const uint4 *>(mv + row * p.meta_sr);
        }
      }
      __syncthreads();
      first_half(0, sa, sa, kYes, kNo);
      if (p.opt.on) {  // soft cap / ALiBi on the meta rows: the distance of the reference's stacked second attention
        const int c0 = mc << 5;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int me = p.meta_bias_off + qrow0 + min(q0 + 16 * ts[b] + c, Lq - 1);
#pragma unroll
          for (int j = 0; j < 8; ++j)
            sa[b][j >> 2][j & 3] = adjust_score(p.opt, sa[b][j >> 2][j & 3], my_slope[b],
                                                -fabsf((float)(me - (c0 + ((j >> 2) << 4) + 4 * g + (j & 3)))));
        }
      }
      {
        const int c0 = mc << 5;
        float t[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          t[b] = kNegInf;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int key = c0 + ((j >> 2) << 4) + 4 * g + (j & 3);
            sa[b][j >> 2][j & 3] = key >= p.meta_len ? kNegInf : sa[b][j >> 2][j & 3];
            t[b] = fmaxf(t[b], sa[b][j >> 2][j & 3]);
          }
        }
        bool raise = false;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          mx[b] = t[b] * p.scale_log2;
          raise |= mx[b] > m[b] + kRaise;
        }
        if (__builtin_amdgcn_ballot_w64(raise) != 0) rescale();
      }
      first_half(0, sa, sa, kNo, kYes);
      load_v(0);
      second_half(sa, kYes, kNo);
      __syncthreads();
    }

    // ---- chunk loop: one barrier per chunk, every wavefront visits every chunk -------------------
    // (chunks outside a wavefront's own band come out fully masked and add zero)
    // Iteration x: scores of chunk x+1 while the numerators of chunk x are formed, then P V of chunk x while the
    // scores of chunk x+1 are masked and searched for their maxima; chunk x+2 goes from registers into the ring
    // slot that chunk x-1 has left, and chunk x+3 is requested from global memory into the registers chunk x+1
    // has left (two register sets and two score sets used alternately; the loop is written out for both so that
    // every register index is static). Loads are issued unconditionally (past the end they re-read the last
    // rows), so the wait in front of each LDS store counts exactly the loads that may still be in flight.
    int r0 = 0, r1 = kStage, r2 = 2 * kStage;  // ring slots of chunks x, x+1, x+2
    auto body = [&](int x, Scores &sc, Scores &sn, Set &arriving, Set &leaving) __attribute__((always_inline)) {
      load_v(r0);
      if (fetcher) fetch(arriving);  // chunk x + 3
      first_half(r1, sn, sc, kYes, kYes);
      adjust_scores(x + 1, sn);
      mask_scores(x + 1, sn);
      if (second_half(sn, kYes, kYes)) rescale();
      if (fetcher) stash(r2, leaving);  // chunk x + 2
      __syncthreads();
      const int t = r0;
      r0 = r1;
      r1 = r2;
      r2 = t;
    };
    if (fetcher) {
      stash(r0, stage[0]);
      fetch(stage[0]);  // chunk 2
      stash(r1, stage[1]);
    }
    __syncthreads();
    first_half(r0, sa, sa, kYes, kNo);
    adjust_scores(0, sa);
    mask_scores(0, sa);
    if (second_half(sa, kNo, kYes)) rescale();
    int x = 0;
    for (; x + 2 < n_walk; x += 2) {
      body(x, sa, sb2, stage[1], stage[0]);
      body(x + 1, sb2, sa, stage[0], stage[1]);
    }
    if (x + 1 < n_walk) {
      body(x, sa, sb2, stage[1], stage[0]);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        sa[b][0] = sb2[b][0];
        sa[b][1] = sb2[b][1];
      }
    }
    // the last chunk: its numerators and its P V product
    load_v(r0);
    first_half(r1, sa, sa, kNo, kYes);
    second_half(sa, kYes, kNo);

    // ---- epilogue: lane (g, c) owns token c of each block, dims 16 mt + 4g + i --------------------------
    if constexpr (HALVES) {
      // Each set puts one of two blocks together (the first set the only one): the other set's sums come through LDS. What is handed
      // over lies across both sets' rings, whose last slots any wavefront of either set may still be reading: the first barrier is
      // what frees them, the second what makes the sums readable.
      float *const out_acc = reinterpret_cast<float *>(smem_all + (half * S::kSetWaves + wave) * kHandOver) + lane * 4;
      const float *const in_acc = reinterpret_cast<const float *>(smem_all + ((half ^ 1) * S::kSetWaves + wave) * kHandOver) + lane * 4;
      auto hand_over = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) *reinterpret_cast<f32x4_t *>(out_acc + mt * 256) = acc[b][mt];
        *reinterpret_cast<float2 *>(out_acc + 2048) = make_float2(m[b], l[b]);
      };
      auto put_together = [&](int b) __attribute__((always_inline)) {
        const float2 ml = *reinterpret_cast<const float2 *>(in_acc + 2048);
        const float m_new = fmaxf(m[b], ml.x), m_safe = m_new == kNegInf ? 0.f : m_new;
        const float mine = fast_exp2(m[b] - m_safe), other = fast_exp2(ml.x - m_safe);
        m[b] = m_new;
        l[b] = fmaf(ml.y, other, l[b] * mine);
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) {
          const f32x4_t x = *reinterpret_cast<const f32x4_t *>(in_acc + mt * 256);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[b][mt][i] = fmaf(x[i], other, acc[b][mt][i] * mine);
        }
      };
      __syncthreads();
      if (half) hand_over(0);
      else if (NB == 2) hand_over(NB - 1);
      __syncthreads();
      if (half) { if (NB == 2) put_together(NB - 1); }
      else put_together(0);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (HALVES && b != half) continue;   // (wave-uniform)
      float lt = l[b];
      lt += __shfl_xor(lt, 16);
      lt += __shfl_xor(lt, 32);
      if (q0 + 16 * ts[b] + c < Lq && parts > 1) {
        const int64_t rec = ((int64_t)(qrow0 + q0 + 16 * ts[b] + c) * p.Hq + head0 + hd[b]) * p.n_parts + part;
        float *dst = p.ws_acc + rec * 128 + 4 * g;
#pragma unroll
        for (int mt = 0; mt < 8; ++mt)
          *reinterpret_cast<float4 *>(dst + 16 * mt) = make_float4(acc[b][mt][0], acc[b][mt][1], acc[b][mt][2], acc[b][mt][3]);
        if (g == 0) *reinterpret_cast<float2 *>(p.ws_ml + rec * 2) = make_float2(m[b], lt);
      } else if (q0 + 16 * ts[b] + c < Lq) {
        const float inv = lt > 0.f ? 1.f / lt : 0.f;
        char *dst = p.out + ((int64_t)(qrow0 + q0 + 16 * ts[b] + c) * p.o_sr + (int64_t)(head0 + hd[b]) * p.o_sh +
                             4 * g) * 2;
#pragma unroll
        for (int mt = 0; mt < 8; ++mt)
          *reinterpret_cast<uint2 *>(dst + 32 * mt) = make_uint2(E::pack(acc[b][mt][0] * inv, acc[b][mt][1] * inv),
                                                                 E::pack(acc[b][mt][2] * inv, acc[b][mt][3] * inv));
        if (p.lse && g == 0)
          p.lse[(int64_t)(qrow0 + q0 + 16 * ts[b] + c) * p.Hq + head0 + hd[b]] =
              lt > 0.f ? (m[b] + log2f(lt)) * kLn2 : kNegInf;
      }
    }
  };
  if constexpr (NHEADS == 1) {
    run(std::integral_constant<int, 1>{});
  } else if constexpr (!ODD) {
    run(std::integral_constant<int, 2>{});
  } else if constexpr (NHEADS == 2) {
    if (nheads == 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  } else {
    if ((nheads & 1) && wave >= 4) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  }
}

// Puts the parts of a tile together: a workgroup per 8 query rows of a tile and query head, 32 lanes of four dims per
// row. A tile of one part has its output already. Latency and bytes (parts x 520 per row and head, once): with the 64
// rows of a tile in one workgroup, eight after the other, 24 parts took 60 us instead of 9.
template <typename E>
__global__ __launch_bounds__(256) void swa_prefill_merge_kernel(const PrefillParams p) {
  const int tile = blockIdx.x, head = blockIdx.y;
  const int seq = p.tile_seq[tile], q0 = p.tile_q0[tile];
  const int qrow0 = p.cu_q[seq], Lq = p.cu_q[seq + 1] - qrow0;
  const int parts = tile_parts(p, tile_walk(p, seq, q0, Lq, p.seq_lens_k[seq]));
  const int j = q0 + 8 * blockIdx.z + (threadIdx.x >> 5), d4 = threadIdx.x & 31;
  if (parts < 2 || j >= Lq) return;
  const int64_t rh = (int64_t)(qrow0 + j) * p.Hq + head;
  // from the first of the workgroup's rows on; past the last part an offset out of range, which gives zeros: that part again, times 0,
  // would be a NaN where it holds an infinity
  const int64_t rec0 = ((int64_t)(qrow0 + q0 + 8 * blockIdx.z) * p.Hq + head) * p.n_parts;
  const int rec = (int)(threadIdx.x >> 5) * p.Hq * p.n_parts;
  const __amdgpu_buffer_rsrc_t ml = __builtin_amdgcn_make_buffer_rsrc(p.ws_ml + rec0 * 2, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t acc = __builtin_amdgcn_make_buffer_rsrc(p.ws_acc + rec0 * 128, 0, 0x7fffffff, 0x00020000);
  float4 tot = make_float4(0.f, 0.f, 0.f, 0.f);
  float L = 0.f, M = kNegInf;
  for (int s0 = 0; s0 < parts; s0 += 4) {  // four parts per trip to memory
    float2 x[4];
    float4 a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool there = s0 + u < parts;
      x[u] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(ml, there ? (rec + s0 + u) * 8 : -16, 0, 0));
      a[u] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(acc, there ? (rec + s0 + u) * 512 + 16 * d4 : -16, 0, 0));
    }
    float Mn = M;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s0 + u >= parts) x[u].x = kNegInf;
      Mn = fmaxf(Mn, x[u].x);
    }
    const float ref = Mn == kNegInf ? 0.f : Mn;  // (nothing visible so far: every factor is 0, and a NaN stays one)
    const float keep = fast_exp2(M - ref);
    tot.x *= keep; tot.y *= keep; tot.z *= keep; tot.w *= keep;
    L *= keep;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float f = fast_exp2(x[u].x - ref);
      tot.x = fmaf(a[u].x, f, tot.x);
      tot.y = fmaf(a[u].y, f, tot.y);
      tot.z = fmaf(a[u].z, f, tot.z);
      tot.w = fmaf(a[u].w, f, tot.w);
      L = fmaf(x[u].y, f, L);
    }
    M = Mn;
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  char *dst = p.out + ((int64_t)(qrow0 + j) * p.o_sr + (int64_t)head * p.o_sh + 4 * d4) * 2;
  *reinterpret_cast<uint2 *>(dst) = make_uint2(E::pack(tot.x * inv, tot.y * inv), E::pack(tot.z * inv, tot.w * inv));
  if (p.lse && d4 == 0) p.lse[rh] = L > 0.f ? (M + log2f(L)) * kLn2 : kNegInf;
}

template <typename E, int KVQ, bool PAGED, bool APPEND = false>
void launch_prefill_q(int nh, bool odd, bool halves, dim3 grid, hipStream_t st, const PrefillParams &p) {
  const dim3 b4(256), b8(512);
  if (halves && nh == 1) hipLaunchKernelGGL((swa_prefill_kernel<E, 1, KVQ, PAGED, false, true, APPEND>), grid, b8, 0, st, p);
  else if (halves && odd) hipLaunchKernelGGL((swa_prefill_kernel<E, 2, KVQ, PAGED, true, true, APPEND>), grid, b8, 0, st, p);
  else if (halves) hipLaunchKernelGGL((swa_prefill_kernel<E, 2, KVQ, PAGED, false, true, APPEND>), grid, b8, 0, st, p);
  else if (nh == 1) hipLaunchKernelGGL((swa_prefill_kernel<E, 1, KVQ, PAGED, false, false, APPEND>), grid, b4, 0, st, p);
  else if (nh == 2 && odd) hipLaunchKernelGGL((swa_prefill_kernel<E, 2, KVQ, PAGED, true, false, APPEND>), grid, b4, 0, st, p);
  else if (nh == 2) hipLaunchKernelGGL((swa_prefill_kernel<E, 2, KVQ, PAGED, false, false, APPEND>), grid, b4, 0, st, p);
  else if (odd) hipLaunchKernelGGL((swa_prefill_kernel<E, 4, KVQ, PAGED, true, false, APPEND>), grid, b8, 0, st, p);
  else hipLaunchKernelGGL((swa_prefill_kernel<E, 4, KVQ, PAGED, false, false, APPEND>), grid, b8, 0, st, p);
}
}  // namespace

// The launches over INT8 caches, whose kernels swa_prefill_int8.hip compiles from this file; params: a PrefillParams.
namespace sb_host {
void launch_prefill_int8(int dtype, int nh, bool odd, bool halves, dim3 grid, hipStream_t st, const void *params)
#ifndef SB_PREFILL_INT8
    ;
#else
{
  const PrefillParams &p = *static_cast<const PrefillParams *>(params);
  if (dtype == SB_BF16) launch_prefill_q<BF16, SB_KV_INT8, true>(nh, odd, halves, grid, st, p);
  else launch_prefill_q<F16, SB_KV_INT8, true>(nh, odd, halves, grid, st, p);
}
#endif
}  // namespace sb_host

#ifndef SB_PREFILL_INT8
namespace {

template <typename E>
void launch_prefill(int kv_quant, int nh, bool odd, bool halves, dim3 grid, hipStream_t st, const PrefillParams &p) {
  if (kv_quant == SB_KV_FP8) launch_prefill_q<E, SB_KV_FP8, true>(nh, odd, halves, grid, st, p);
  else if (p.block_table) launch_prefill_q<E, SB_KV_NONE, true>(nh, odd, halves, grid, st, p);
  else if (p.append.tokens > 0) launch_prefill_q<E, SB_KV_NONE, false, true>(nh, odd, halves, grid, st, p);
  else launch_prefill_q<E, SB_KV_NONE, false>(nh, odd, halves, grid, st, p);
}

constexpr int64_t kDealtTiles = 1024;   // shorter tile lists come dealt to the XCDs, see sb_swa_prefill_plan

// Most 32-key chunks a tile of 64 queries walks when no sequence has more than max_keys keys.
int64_t most_chunks(const sb_swa_prefill_args *a, int64_t max_keys) {
  int64_t span = max_keys;
  if (a->window_left >= 0 && span > (int64_t)a->window_left + 64) span = (int64_t)a->window_left + 64;
  return (span + 30) / 32 + 1;
}

// How a call is spread over the GPU: with groups of four heads a workgroup of eight wavefronts fills a CU, and a call
// of `wgs` of them takes as long as its longest walk while wgs <= 256. Two ways to shorten that:
//  * pairs: workgroups of two heads and four wavefronts, two to a CU. Measured, with L the longest walk in chunks and L' the
//    walk of the longest workgroup that has to share its CU (in whole prompts a long walk shares with a short one; behind a
//    context all are as long): groups of four 8.4 + 0.94 L us, pairs 6.3 + 0.72 L + 0.35 L'. So they always pay while every
//    CU gets one, and up to 256 workgroups of four where L' < 6 + 0.63 L (28 : 4 heads, us of groups of four -> pairs):
//      whole prompts, window 4096   300 / 700 / 1000 / 1517 / 2560 tokens 16.6 / 28.3 / 35.8 / 50.7 / 80.7 -> 13.1 / 21.9 / 28.2 / 42.3 / 69
//      behind 4200                  window 512: 1075 / 2035 28.8 / 29.9 -> 29.2 / 30.1, 1024: 42.4 / 43.7 -> 44.5 / 45.3, 4096: 124 / 129 -> 136 / 142
//      between                      1200 behind 300 49.6 -> 41.7, 2000 behind 800 85.5 -> 74.7; 2035, window 512 28.1 -> 28.7 (not taken)
//    From 256 to 384 workgroups of four (a second round that leaves most CUs idle) they pay unless the walks are many chunks
//    long: 3059 tokens, window 4096 92.8 -> 88.8; behind 4200, windows 512 / 1024 / 2048 / 4096 52.4 / 77.1 / 127 / 228 -> 47 / 72.9 / 124 /
//    230; beyond that they lose (1 x 6000: 256 -> 271).
//  * halves: workgroups of two heads that hold their four wavefronts twice, each set walking half of the keys (see halves_us).
//  * parts: the keys of a walk cut into parts of 8 chunks or more side by side, at the price of fp32 partials and
//    a merge (64 / 200 / 512 / 1024 tokens behind 4200: 100 with pairs, 123 with groups of four -> 27.5 (12 parts) / 37 (8) /
//    54 (4) / 85 (2) us; 64 tokens in 8 parts 25.7, which the estimate below does not find).
struct Spread {
  int parts;
  bool pairs;
};
int64_t quad_workgroups(const sb_swa_prefill_args *a) {
  return a->num_tiles * a->num_kv_heads * ((a->num_q_heads / a->num_kv_heads + 3) / 4);
}
bool pairs_pay(const sb_swa_prefill_args *a, int64_t chunks, int64_t parts, int64_t cus) {
  const int64_t wgs = quad_workgroups(a) * parts;
  if (2 * wgs <= cus) return true;
  if (parts > 1 || 2 * wgs > 3 * cus) return false;
  if (wgs > cus) return chunks <= 2 * a->num_tiles + 2;
  if (!a->tile_keys) return false;   // (unknown: as if all walks were equal)
  const int64_t pairs_per_tile = (int64_t)a->num_kv_heads * ((a->num_q_heads / a->num_kv_heads + 1) / 2);
  const int64_t sharing = cus / pairs_per_tile;   // tiles in front of the first one that shares
  return sharing >= a->num_tiles || (double)most_chunks(a, a->tile_keys[sharing]) < 6.0 + 0.63 * (double)chunks;
}
// Halves: us such a call takes, or infinity where it is better without. A workgroup fills a CU and takes 8.9 + 0.487 L us for a walk of L
// chunks, a pair 9 + 0.69 L, so they pay wherever every workgroup has a CU, from walks of 9 chunks on (28 : 4 heads, us of pairs -> halves:
// whole prompts of 200 / 300 / 700 / 1000 tokens 12.3 / 14.3 / 23.5 / 30.2 -> 12.5 / 13.4 / 20.7 / 25.5, 1024 tokens behind 10000 with a
// window of 512 / 4096 24.2 / 102 -> 22 / 77; 16 : 8, 3000 whole 73.6 -> 54.8). A second round pays where it is short walks that are left for
// the CUs that come free first: with the lists walked longest first over all XCDs, 1300 / 1517 / 2000 whole 38.6 / 43.3 / 54.9 -> 32.1 / 35.3 /
// 50.0 (38 / 40 / 54.6 with an XCD's tiles to itself), 2048 behind 800 79.7 -> 77, 18 : 6, 1517 behind 2000 93 -> 81; not 2 x 1000
// 33.6 -> 34, 4 x 500 23 -> 26.7, 2048 behind 10000 (groups of four: 132) -> 149 and, in three rounds, 2560 69.7 -> 78, nor against groups of
// three heads, whose chunks are shorter (12 : 4, 3000 behind 2000 105 -> 111.6; 24 : 8, 1517 behind 2000 88 -> 96). One head per kv head,
// second round: 16 : 16, 4 x 500 17 -> 19.9 (not taken).
double halves_us(const sb_swa_prefill_args *a, int64_t max_keys, int64_t chunks, int64_t cus) {
  const int64_t G = a->num_q_heads / a->num_kv_heads, per_tile = a->num_kv_heads * ((G + 1) / 2), wgs = a->num_tiles * per_tile;
  if (a->meta_len > 0 || max_keys >= INT32_MAX || chunks < 9) return HUGE_VAL;   // (of calls without a bound the walks are unknown)
  const double l0 = (double)chunks, alone = 8.9 + 0.487 * l0;
  if (wgs <= cus) return alone;
  if (G == 1 || wgs > 2 * cus || !a->tile_keys) return HUGE_VAL;
  const double next = (double)most_chunks(a, a->tile_keys[cus / per_tile]), first_done = (double)most_chunks(a, a->tile_keys[(cus - 1) / per_tile]);
  const double halves = std::max(alone, 13.0 + 0.51 * (first_done + next));
  double others = 6.3 + 0.72 * l0 + 0.35 * next;   // pairs
  if (quad_workgroups(a) <= cus) others = std::min(others, 8.4 + (G == 3 ? 0.75 : 0.94) * l0);   // groups of three or four heads
  return halves < 0.93 * others ? halves : HUGE_VAL;
}
// Whether a call in halves has more workgroups than an XCD's eighth of the tiles leaves CUs for: they are then walked over all XCDs
// (24 : 4 heads, 800 and 300 behind 1000, 216 workgroups of which an XCD would get 36 for its 32 CUs: 55.3 -> 49.9 us).
bool halves_in_rounds(const sb_swa_prefill_args *a, int64_t cus) {
  return (a->num_tiles + 7) / 8 * 8 * a->num_kv_heads * ((a->num_q_heads / a->num_kv_heads + 1) / 2) > cus;
}
// Order of a short list's tiles. Dealt to the XCDs longest walk first, in tile-major order, evens out the work of walks of
// different lengths; in sequence order, kv heads outermost, the tiles that run on an XCD at a time are neighbours of one head and
// share its keys in the L2. Where the walks are as good as equal there is nothing to even out, and the fewer query heads share
// a kv head (the less a workgroup does per byte), the more the L2 counts. us, dealt -> in sequence order (mean walk / longest walk):
//   28 : 4   6000 / 20000 behind 12000 381 / 1246 -> 359 / 1162 (1.0); 2500 x 4 behind 3000 574 -> 589 (0.94); 6000 whole 253 -> 348 (0.66)
//   12 : 4   6000 behind 3000 231 -> 205 (0.98), 2500 x 4 behind 3000 284 -> 311 (0.94)
//   16 : 8   6000 with a window of 1024 79.7 -> 72.6 (0.92), 800 x 6 behind 3000 183 -> 196 (0.90)
//   16 : 16  6000 / 20000 behind 12000 461 / 1489 -> 287 / 908 (1.0), 20000 whole 1300 -> 870 (0.90), 800 x 6 behind 800 115 -> 96 (0.77);
//            below, dealt with kv heads outermost where that is many workgroups for how uneven the walks are (tiles * kv heads per
//            CU): 6000 whole 268 -> 243 (0.66, 5.9), 40 : 40, 2500 x 4 behind 800 915 -> 650 (0.63, 25), but 3000 whole 71 -> 101 (0.52,
//            2.9), 2500 x 4 whole 163 -> 192 (0.52, 10) and 40 : 40, 2000 whole 108 -> 118 (0.52, 5)
//   20 : 4, 24 : 4 and 16 : 8  20000 whole 967 -> 863, 1018 -> 978, 695 -> 657 (0.90)
enum class Order { kDealt, kDealtByHead, kSequence };
Order tile_order(const sb_swa_prefill_args *a, int64_t max_keys, int64_t chunks, int64_t cus) {
  if (a->num_tiles >= kDealtTiles || !a->tile_keys || !a->ordered_tile_seq || !a->ordered_tile_q0) return Order::kDealt;
  int64_t total = 0;
  for (int64_t t = 0; t < a->num_tiles; ++t) total += most_chunks(a, a->tile_keys[t] < max_keys ? a->tile_keys[t] : max_keys);
  const int G = a->num_q_heads / a->num_kv_heads;
  const double even = (double)total / (double)(a->num_tiles * chunks);
  // (a last launch of one or two heads reads as much per head as G <= 2 does; over many rounds it decides)
  const bool thin = G <= 3 || G % 4 == 1 || G % 4 == 2, rounds6 = quad_workgroups(a) >= 6 * cus;
  if (even >= (G == 1 ? 0.75 : thin && rounds6 ? 0.88 : G == 2 ? 0.92 : 0.97)) return Order::kSequence;
  return G == 1 && 2 * a->num_tiles * a->num_kv_heads >= (even >= 0.65 ? 7 : 22) * cus ? Order::kDealtByHead : Order::kDealt;
}

// What a call in parts takes, for the choice between them and halves: it goes by the heads the workgroups of the parts hold (two, and one,
// run four wavefronts; three run eight, of which four hold one head's scores; four run eight of two). us by least squares over 1500 calls of
// 20 head counts (G = 2 / 3 / 4 / 7 and pairs: 0.70 / 0.75 / 0.90 / 0.89 and 0.69 to 0.73 a chunk; +- 1.5 to 3.4). Parts -> halves, not
// taken: 8 : 4, 700 behind 2000, window 1024 20.5 -> 26.4, 2048 behind 2000 59.8 -> 69.4; 16 : 8, 400 behind 800 21.1 -> 27.5; 12 : 4, 2048
// behind 2000 66 -> 71.5; 24 : 8, 400 behind 800 26.4 -> 28.1; taken: 28 : 4, 1024 behind 10000 79.7 -> 74.1. Where few tiles leave XCDs
// without any it is too low (30 : 10, 576 behind 2000, nine tiles on five XCDs: estimated 50, 71.5; in halves 48.9, not taken).
double parts_us(const sb_swa_prefill_args *a, const Spread &s, int64_t chunks, int64_t cus) {
  const int64_t G = a->num_q_heads / a->num_kv_heads;
  const double n = (double)s.parts, fill = n * (double)quad_workgroups(a) / (double)cus, walk = (double)((chunks + s.parts - 1) / s.parts);
  if (s.pairs || G == 2) return 9.1 + 0.11 * n + (G == 2 ? 7.0 : 15.0) * fill + 0.7 * walk;
  return 14.0 + 0.33 * n + 6.0 * fill + (G == 3 ? 0.75 : 0.9) * walk;
}

Spread spread_of(const sb_swa_prefill_args *a, int64_t max_keys) {
  const int64_t chunks = most_chunks(a, max_keys), wgs = quad_workgroups(a), cus = sb_host::device_cu_count(), G = a->num_q_heads / a->num_kv_heads;
  const Spread whole{1, pairs_pay(a, chunks, 1, cus)};
  Spread best = whole;
  double best_us = 5.0 + (whole.pairs ? 0.69 : 0.9) * (double)chunks;
  for (int64_t n = 2; n * wgs <= cus && 8 * n <= chunks; ++n) {
    const bool pairs = pairs_pay(a, chunks, n, cus);
    const double us = 13.5 + 0.28 * (double)n + 8.0 * (double)(n * wgs) / (double)cus +
                      (pairs ? 0.69 : 0.86) * (double)((chunks + n - 1) / n);
    if (us < best_us) {
      best = Spread{(int)n, pairs};
      best_us = us;
    }
  }
  if (best.parts > 1 && G > 1 && halves_us(a, max_keys, chunks, cus) < 0.95 * parts_us(a, best, chunks, cus)) best = whole;
  return best;
}

// The append of a call whose keys are in flight rides along as workgroups behind those of the attention: they copy on CUs that have
// none or whose own are done, and a launch less is made. us of the layer call, append in front -> in it (28 : 4 heads): 64 / 300 / 700 / 1517 /
// 2500 / 4000 tokens 17.8 / 18.4 / 22.2 / 36.5 / 73.0 / 143.0 -> 14.2 / 14.7 / 19.4 / 34.4 / 70.0 / 139.8, 4 x 700 30.6 -> 28.1, 8 x 2000
// 210 -> 204. From 8000 tokens on they wait for the attention's CUs and it is level (1 x 8000 373.5 -> 373; 16 x 8192: 5925 + 62 -> 5985 by
// the trace), the extra workgroups moving 4 to 5 TB/s as the kernel of its own did.
bool append_rides(const sb_swa_prefill_args *a, const sb_kv_append_args *ap) {
  return !a->block_table && ap->head_size == 128 && ap->dtype != SB_F32 && ap->stream == a->stream && a->num_tiles > 0;
}

int prefill(const sb_swa_prefill_args *a, int64_t max_keys, int n_parts, float *ws_acc, float *ws_ml, const sb_kv_append_args *ap = nullptr) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_swa_prefill: null args");
  if (a->num_tiles < 0) return fail(SB_ERR_INVALID, "sb_swa_prefill: negative num_tiles");
  if (a->num_tiles == 0) return SB_OK;
  if (!a->q || !a->k || !a->v || !a->out || !a->cu_seqlens_q || !a->seq_lens_k || !a->tile_seq || !a->tile_q0)
    return fail(SB_ERR_INVALID, "sb_swa_prefill: null tensor pointer");
  if (a->head_size != 128)
    return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: head_size %d (only 128 is built)", a->head_size);
  if (a->dtype != SB_BF16 && a->dtype != SB_F16)
    return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: dtype must be bf16 or fp16");
  if (a->num_q_heads <= 0 || a->num_kv_heads <= 0 || a->num_q_heads % a->num_kv_heads != 0)
    return fail(SB_ERR_INVALID, "sb_swa_prefill: num_q_heads must be a positive multiple of num_kv_heads");
  if (!(a->scale > 0.f)) return fail(SB_ERR_INVALID, "sb_swa_prefill: scale must be positive");
  if (a->block_table && (a->block_size < 16 || a->block_size % 16 != 0))
    return fail(SB_ERR_INVALID, "sb_swa_prefill: block_size %d must be a multiple of 16", a->block_size);
  if (a->num_tiles > 0x7ffffff0LL || a->num_kv_heads > 65535)
    return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: grid too large");
  const bool codes = a->kv_quant == SB_KV_INT8 || a->kv_quant == SB_KV_FP8;
  if (a->kv_quant != SB_KV_NONE && !codes)
    return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: unknown kv_quant %d", a->kv_quant);
  if (codes && !a->block_table) return fail(SB_ERR_INVALID, "sb_swa_prefill: a byte-code cache needs paged mode");
  if (a->kv_quant == SB_KV_INT8 && (!a->k_scale || !a->v_scale))
    return fail(SB_ERR_INVALID, "sb_swa_prefill: the INT8 cache needs both scale tensors");
  if (a->kv_quant == SB_KV_FP8 && (!(a->k_scale_tensor > 0.f) || !(a->v_scale_tensor > 0.f)))
    return fail(SB_ERR_INVALID, "sb_swa_prefill: the fp8 cache needs positive k_scale_tensor and v_scale_tensor");
  const int kv_esz = codes ? 1 : 2;
  const int64_t es[] = {a->q_stride_row, a->q_stride_head, a->out_stride_row, a->out_stride_head};
  for (int64_t s : es)
    if ((s * 2) % 16 != 0)
      return fail(SB_ERR_INVALID, "sb_swa_prefill: stride %lld elements is not 16-byte aligned", (long long)s);
  const int64_t kes[] = {a->kv_stride_block, a->kv_stride_row, a->kv_stride_head};
  for (int64_t s : kes)
    if ((s * kv_esz) % 16 != 0)
      return fail(SB_ERR_INVALID, "sb_swa_prefill: cache stride %lld elements is not 16-byte aligned", (long long)s);
  if (a->kv_stride_row <= 0 || a->kv_stride_row * kv_esz >= (1 << 24))
    return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: cache row stride %lld elements (must be positive and below 16 MiB)",
                (long long)a->kv_stride_row);
  if ((reinterpret_cast<uintptr_t>(a->q) | reinterpret_cast<uintptr_t>(a->k) | reinterpret_cast<uintptr_t>(a->v) |
       reinterpret_cast<uintptr_t>(a->out)) & 15u)
    return fail(SB_ERR_INVALID, "sb_swa_prefill: q/k/v/out base not 16-byte aligned");

  PrefillParams p;
  p.q = (const char *)a->q; p.k = (const char *)a->k; p.v = (const char *)a->v; p.out = (char *)a->out;
  p.lse = a->lse; p.Hq = a->num_q_heads;
  p.block_table = a->block_table; p.kv_start = a->kv_start; p.kv_start32 = a->kv_start32; p.key_lo = a->key_lo;
  p.cu_q = a->cu_seqlens_q; p.seq_lens_k = a->seq_lens_k; p.tile_seq = a->tile_seq; p.tile_q0 = a->tile_q0;
  p.G = a->num_q_heads / a->num_kv_heads; p.head_begin = 0;
  p.block_size = a->block_size > 0 ? a->block_size : 16; p.window_left = a->window_left;
  p.tiles_per_block = p.block_size / 16;
  p.tile_div = tile_division((uint32_t)p.tiles_per_block);
  p.scale_log2 = a->scale * sb::kLog2e;
  p.q_sr = a->q_stride_row; p.q_sh = a->q_stride_head; p.o_sr = a->out_stride_row; p.o_sh = a->out_stride_head;
  p.kv_sb = a->kv_stride_block * kv_esz; p.kv_sr = a->kv_stride_row * kv_esz; p.kv_sh = a->kv_stride_head * kv_esz;
  p.k_scale = a->k_scale; p.v_scale = a->v_scale;
  p.k_scale_tensor = a->k_scale_tensor; p.v_scale_tensor = a->v_scale_tensor; p.Hkv = a->num_kv_heads;
  p.bt_stride = a->block_table_stride;
  p.num_tiles = (int)a->num_tiles;
  const int64_t chunks = most_chunks(a, max_keys);
  const int64_t cus = sb_host::device_cu_count();
  const bool halves = n_parts == 1 && halves_us(a, max_keys, chunks, cus) < HUGE_VAL;
  const bool rounds = halves && halves_in_rounds(a, cus);
  const Order order = n_parts == 1 && !rounds ? tile_order(a, max_keys, chunks, cus) : Order::kDealt;
  if (order == Order::kSequence) {
    p.tile_seq = a->ordered_tile_seq;
    p.tile_q0 = a->ordered_tile_q0;
  }
  p.n_parts = n_parts; p.part_chunks = (int)((chunks + n_parts - 1) / n_parts);
  p.ws_acc = ws_acc; p.ws_ml = ws_ml;
  p.meta_k = p.meta_v = nullptr;
  p.meta_len = 0;
  p.meta_sr = p.meta_sh = 0;
  p.opt.on = 0;
  p.opt.slopes = nullptr;
  p.opt.cap = p.opt.inv_cap2_log2e = 0.f;
  p.opt.mult = a->scale;  // (byte-code rows are dequantised on their way into LDS: the scores are those of elements)
  p.opt.inv_mult = 1.f / p.opt.mult;
  if (a->softcap < 0.f || a->softcap != a->softcap) return fail(SB_ERR_INVALID, "sb_swa_prefill: softcap must be >= 0");
  p.meta_bias_off = 0;
  if (a->softcap > 0.f || a->alibi_slopes) {
    if (a->meta_len > 0) {
      if (a->meta_bias_row0 < 0 || a->meta_bias_rows <= 0 || a->meta_bias_rows > 0x3fffffffLL ||
          a->meta_bias_row0 > a->meta_bias_rows)
        return fail(SB_ERR_INVALID, "sb_swa_prefill: soft cap / ALiBi with meta tokens need meta_bias_rows (the query rows "
                                    "of the reference's stacked second attention) and meta_bias_row0 inside it");
      p.meta_bias_off = (int)(a->meta_bias_row0 + a->meta_len - a->meta_bias_rows);
    }
    p.opt.on = 1;
    p.opt.slopes = a->alibi_slopes;
    if (a->softcap > 0.f) {
      p.opt.cap = a->softcap;
      p.opt.inv_cap2_log2e = 2.f * sb::kLog2e / a->softcap;
    }
  }
  if (a->meta_len < 0) return fail(SB_ERR_INVALID, "sb_swa_prefill: negative meta_len");
  if (a->meta_len > 0) {
    if (!a->meta_k || !a->meta_v) return fail(SB_ERR_INVALID, "sb_swa_prefill: meta_len without meta_k / meta_v");
    if (((reinterpret_cast<uintptr_t>(a->meta_k) | reinterpret_cast<uintptr_t>(a->meta_v)) & 15u) ||
        (a->meta_stride_row * 2) % 16 || (a->meta_stride_head * 2) % 16)
      return fail(SB_ERR_INVALID, "sb_swa_prefill: meta rows must be 16-byte aligned");
    p.meta_k = (const char *)a->meta_k; p.meta_v = (const char *)a->meta_v;
    p.meta_len = a->meta_len;
    p.meta_sr = a->meta_stride_row * 2; p.meta_sh = a->meta_stride_head * 2;
  }

  // Groups of four heads, and a last one of three, are one launch (workgroups of eight wavefronts each); a last group
  // of one or two heads runs workgroups of four and is a launch of its own.
  const int64_t per_xcd = (a->num_tiles + 7) / 8;
  // Tiles per bucket of an XCD's order, 1 / 2 / 4 / 8 / all, measured: 1 x 3000 tokens 97 / 98 / 116 / 134 / 134 us and
  // 1 x 8192 388 / 398 / 411 / 458 / 448 us (tile lists sorted longest first: what starts last should be short whatever
  // its heads); 16 x 8192 in sequence order 6.34 ms at 1 against 6.04 at 4, 6.08 at 16 and 6.13 at all (four tiles and one
  // kv head at a time keep their keys in the XCD's L2).
  // Up to four query heads per kv head that is 1 to 10 % slower than all (16 : 16 3194 / 2951 us, 16 : 8 2270 / 2222, 32 : 8 4407 / 4356
  // for 10 x 8192). Shorter lists: see tile_order.
  p.bucket = rounds ? 0 : a->num_tiles >= kDealtTiles ? (p.G <= 4 ? (int)per_xcd : 4) : order == Order::kDealt ? 1 : (int)per_xcd;
  const bool pairs = p.G > 1 && (halves || pairs_pay(a, chunks, n_parts, cus));
  if (per_xcd * 8 * a->num_kv_heads * p.G > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: grid too large");
  for (int h0 = 0; h0 < p.G;) {
    const int left = p.G - h0;
    const int groups = pairs ? (left + 1) / 2 : (left >= 3 ? left / 4 + (left % 4 == 3) : 1);
    const int nh = pairs ? 2 : (left >= 3 ? 4 : left);
    const bool odd = nh * groups > left;   // (the last group has one head less)
    p.head_begin = h0;
    h0 += nh * groups;
    p.head_groups = groups;
    dim3 grid((unsigned)(per_xcd * 8 * a->num_kv_heads * groups), (unsigned)n_parts);
    p.append = Append{};
    if (ap && p.head_begin == 0) {   // (the first launch takes it along)
      const int waves = nh == 4 || halves ? 8 : 4;
      const int64_t esz = 2;
      p.append = Append{(const char *)ap->key, (const char *)ap->value, (char *)ap->k_cache, (char *)ap->v_cache, ap->slot_mapping,
                        ap->num_tokens, grid.x, ap->num_kv_heads * 16, ap->block_size, ap->key_stride_token * esz,
                        ap->key_stride_head * esz, ap->value_stride_token * esz, ap->value_stride_head * esz,
                        ap->cache_stride_block * esz, ap->cache_stride_row * esz, ap->cache_stride_head * esz};
      const int64_t more = (ap->num_tokens + kAppendTokens * waves - 1) / (kAppendTokens * waves);
      if (grid.x + more > 0x7fffffffLL) return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill: grid too large");
      grid.x += (unsigned)more;
    }
    if (a->kv_quant == SB_KV_INT8) launch_prefill_int8(a->dtype, nh, odd, halves, grid, (hipStream_t)a->stream, &p);
    else if (a->dtype == SB_BF16) launch_prefill<BF16>(a->kv_quant, nh, odd, halves, grid, (hipStream_t)a->stream, p);
    else launch_prefill<F16>(a->kv_quant, nh, odd, halves, grid, (hipStream_t)a->stream, p);
    const int rc = check_launch("swa_prefill_kernel");
    if (rc != SB_OK) return rc;
  }
  if (n_parts > 1) {
    const dim3 mgrid((unsigned)a->num_tiles, (unsigned)a->num_q_heads, 8);
    if (a->dtype == SB_BF16) hipLaunchKernelGGL(swa_prefill_merge_kernel<BF16>, mgrid, dim3(256), 0, (hipStream_t)a->stream, p);
    else hipLaunchKernelGGL(swa_prefill_merge_kernel<F16>, mgrid, dim3(256), 0, (hipStream_t)a->stream, p);
    return check_launch("swa_prefill_merge_kernel");
  }
  return SB_OK;
}

}  // namespace

// The kernel gives XCD x the x-th contiguous eighth of the tile list. In lists of less than this many tiles those late in a
// long sequence, which see the most keys, are dealt out in turn, latest first, so that the XCDs get equal shares and the longest
// workgroups start first (unless the call finds sequence order better, tile_order above). Longer lists stay in sequence
// order: an XCD's neighbouring tiles then share their keys in its L2, and there are enough of them to even out.
constexpr int kTileTokens = 64;

// Native because every new prompt pays it in front of its first layer: the whole plan of 64 / 1517 / 8192 / 16 x 8192 tokens in
// numpy took 39 / 39 / 43 / 37 us of host time, in Python loops without the dealing 13 / 17 / 35 / 370; here 13 / 13 / 14 / 21.
extern "C" int sb_swa_prefill_plan(const int32_t *query_lens, const int32_t *seq_lens_k, int64_t num_seqs, int64_t num_tiles,
                                   int32_t *plan, int32_t *tile_keys) {
  using namespace sb_host;
  if (num_seqs < 0 || num_tiles < 0 || !plan || (num_seqs > 0 && (!query_lens || !seq_lens_k)))
    return fail(SB_ERR_INVALID, "sb_swa_prefill_plan: negative size or null pointer");
  const bool dealt = num_tiles < kDealtTiles;
  // (in sequence order: behind the dealt lists, or in their place)
  int32_t *const cu = plan, *const keys = plan + num_seqs + 1, *const dealt_seq = keys + num_seqs, *const dealt_q0 = dealt_seq + num_tiles;
  int32_t *const seq = dealt ? dealt_q0 + num_tiles : dealt_seq, *const q0 = seq + num_tiles;
  int64_t order[kDealtTiles];   // dealt: (position of the tile in the keys, earlier tiles of the list first) of every tile
  int64_t total = 0, tiles = 0;
  for (int64_t s = 0; s < num_seqs; ++s) {
    if (query_lens[s] < 0 || seq_lens_k[s] < query_lens[s])
      return fail(SB_ERR_INVALID, "sb_swa_prefill_plan: sequence %lld: %d queries need at least as many keys, got %d", (long long)s,
                  query_lens[s], seq_lens_k[s]);
    cu[s] = (int32_t)total;
    keys[s] = seq_lens_k[s];
    total += query_lens[s];
    if (total > INT32_MAX) return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill_plan: more than 2^31 - 1 packed query rows");
    for (int64_t at = 0; at < query_lens[s]; at += kTileTokens, ++tiles) {
      if (tiles >= num_tiles) return fail(SB_ERR_INVALID, "sb_swa_prefill_plan: the sequences hold more than %lld tiles", (long long)num_tiles);
      seq[tiles] = (int32_t)s;
      q0[tiles] = (int32_t)at;
      if (dealt) order[tiles] = ((at + seq_lens_k[s] - query_lens[s]) << 12) | (kDealtTiles - 1 - tiles);
    }
  }
  cu[num_seqs] = (int32_t)total;
  if (tiles != num_tiles)
    return fail(SB_ERR_INVALID, "sb_swa_prefill_plan: the sequences hold %lld tiles, not %lld", (long long)tiles, (long long)num_tiles);
  if (!dealt) return SB_OK;
  std::sort(order, order + tiles, std::greater<int64_t>());
  const int64_t per_xcd = (tiles + 7) / 8;
  int64_t next = 0;
  for (int64_t k = 0; k < 8 * per_xcd; ++k) {
    const int64_t slot = (k % 8) * per_xcd + k / 8;
    if (slot >= tiles) continue;
    if (tile_keys) tile_keys[next] = (int32_t)std::min<int64_t>((order[next] >> 12) + kTileTokens, INT32_MAX);
    const int64_t t = kDealtTiles - 1 - (order[next++] & 0xfff);
    dealt_seq[slot] = seq[t];
    dealt_q0[slot] = q0[t];
  }
  return SB_OK;
}

extern "C" int sb_swa_prefill(const sb_swa_prefill_args *a) { return prefill(a, INT32_MAX, 1, nullptr, nullptr); }

extern "C" int32_t sb_swa_prefill_parts(const sb_swa_prefill_args *a, int64_t max_keys) {
  if (!a || a->num_tiles <= 0 || a->num_kv_heads <= 0 || a->num_q_heads < a->num_kv_heads || max_keys <= 0) return 1;
  return spread_of(a, max_keys < INT32_MAX ? max_keys : INT32_MAX).parts;
}

extern "C" int32_t sb_swa_prefill_halves(const sb_swa_prefill_args *a, int64_t max_keys, int32_t n_parts) {
  if (!a || a->num_tiles <= 0 || a->num_kv_heads <= 0 || a->num_q_heads < a->num_kv_heads || max_keys <= 0 || n_parts > 1) return 0;
  if (max_keys > INT32_MAX) max_keys = INT32_MAX;
  return halves_us(a, max_keys, most_chunks(a, max_keys), sb_host::device_cu_count()) < HUGE_VAL;
}

extern "C" int32_t sb_swa_prefill_group_heads(const sb_swa_prefill_args *a, int64_t max_keys, int32_t n_parts) {
  if (!a || a->num_tiles <= 0 || a->num_kv_heads <= 0 || a->num_q_heads < a->num_kv_heads || max_keys <= 0) return 4;
  if (max_keys > INT32_MAX) max_keys = INT32_MAX;
  return sb_swa_prefill_halves(a, max_keys, n_parts) ||
         pairs_pay(a, most_chunks(a, max_keys), n_parts < 1 ? 1 : n_parts, sb_host::device_cu_count()) ? 2 : 4;
}

extern "C" size_t sb_swa_prefill_workspace_bytes(const sb_swa_prefill_args *a, int64_t total_q, int32_t n_parts) {
  if (!a || n_parts < 2 || total_q <= 0 || a->num_q_heads <= 0) return 0;
  return (size_t)total_q * (size_t)a->num_q_heads * (size_t)n_parts * (128 + 2) * sizeof(float);
}

static int prefill_parted(const sb_swa_prefill_args *a, int64_t total_q, int64_t max_keys, int32_t n_parts, void *workspace,
                          size_t workspace_bytes, const sb_kv_append_args *ap) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_swa_prefill_parted: null args");
  if (a->num_tiles <= 0) return sb_swa_prefill(a);
  if (total_q <= 0 || max_keys <= 0) return fail(SB_ERR_INVALID, "sb_swa_prefill_parted: total_q and max_keys must be positive");
  if (max_keys > INT32_MAX) max_keys = INT32_MAX;
  if (n_parts < 2) return prefill(a, max_keys, 1, nullptr, nullptr, ap);
  if (n_parts > 1024 || a->num_q_heads > 65535) return fail(SB_ERR_UNSUPPORTED, "sb_swa_prefill_parted: too many parts or heads");
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 15u) ||
      workspace_bytes < sb_swa_prefill_workspace_bytes(a, total_q, n_parts))
    return fail(SB_ERR_WORKSPACE, "sb_swa_prefill_parted: workspace of %zu bytes (16-byte aligned) needed, got %zu",
                sb_swa_prefill_workspace_bytes(a, total_q, n_parts), workspace ? workspace_bytes : (size_t)0);
  // (the merge addresses eight rows of a head with 32 bits; fewer parts are always right)
  if (a->num_q_heads > 0)
    n_parts = (int32_t)std::max<int64_t>(1, std::min<int64_t>(n_parts, INT32_MAX / ((int64_t)8 * 512 * a->num_q_heads)));
  float *acc = static_cast<float *>(workspace);
  return prefill(a, max_keys, n_parts, acc, acc + total_q * a->num_q_heads * n_parts * 128, ap);
}

extern "C" int sb_swa_prefill_parted(const sb_swa_prefill_args *a, int64_t total_q, int64_t max_keys, int32_t n_parts, void *workspace,
                                     size_t workspace_bytes) {
  return prefill_parted(a, total_q, max_keys, n_parts, workspace, workspace_bytes, nullptr);
}

extern "C" int sb_swa_prefill_append(const sb_swa_prefill_args *a, const sb_kv_append_args *append, int64_t total_q, int64_t max_keys,
                                     int32_t n_parts, void *workspace, size_t workspace_bytes) {
  using namespace sb_host;
  if (!a) return fail(SB_ERR_INVALID, "sb_swa_prefill_append: null args");
  if (const int rc = check_kv_append(append)) return rc;
  if (append->num_tokens == 0 || append_rides(a, append))
    return prefill_parted(a, total_q, max_keys, n_parts, workspace, workspace_bytes, append->num_tokens ? append : nullptr);
  const int rc = sb_kv_append(append);
  return rc ? rc : prefill_parted(a, total_q, max_keys, n_parts, workspace, workspace_bytes, nullptr);
}
#endif  // SB_PREFILL_INT8
