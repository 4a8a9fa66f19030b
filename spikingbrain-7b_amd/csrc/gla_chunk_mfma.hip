// GLA over prompts on the matrix cores: the recurrence S <- diag(exp g) S + k^T v, o = (q*scale) S
// advanced 32 tokens at a time in its exact block form. With B_t = g_1 + .. + g_t (per key dim,
// inside the block) and S_0 the state before the block,
//   o_t  = (q_t * exp(B_t)) S_0 + sum_{s<=t} [(q_t * exp(B_t)) . (k_s * exp(-B_s))] v_s
//   S_32 = diag(exp(B_32)) (S_0 + sum_s (k_s * exp(-B_s))^T v_s)
// i.e. per block three [16x16] score products (the fourth lies above the diagonal), two products into o and a
// rank-32 update of the state, all v_mfma_f32_16x16x32_bf16 with fp32 accumulation; k * exp(-B_s) serves both as the
// score operand and, transposed, as the state-update operand. The reference computes prompts with fla's
// fused_chunk_gla (vllm_hymeta/model_for_7B/gla_attention.py:207-208), the same block mathematics.
//
// One workgroup per (sequence, head), four wavefronts; wavefront w keeps the state columns
// [32w, 32w+32) as 16 accumulator tiles (64 registers) for the whole prompt: the state crosses HBM
// once each way. Per block a thread turns 8 dims of two neighbouring tokens of q, k, v and gate into LDS operands, and each
// wavefront runs 66 matrix instructions on them. A block has two stretches of code between barriers:
//   1. the gates of block n + 1 are summed over the tokens (see scan_gates), next to the outputs of block n;
//   2. the operands of block n + 1 are formed, next to the state's update with block n.
// k and v operands are double-buffered, q's (read in the first stretch, written in the second) are not.
//
// What bounds it is memory, and there the pattern: heads of a token lie side by side, so a workgroup reads pieces of 256
// bytes (512 of the fp32 gates) and a wavefront's share of a row is what one of its loads finds together. A loop of the
// same loads and stores that computes nothing (profiles/gla_prompt_copy.hip) takes, for 16 x 8192 tokens x 28 heads (5.64 GB), 1243 us
// where a wavefront's load covers 64 bytes of 16 rows and its store 32, 1207 with 64 bytes per store, 1164 with 128 bytes of 8 rows
// per load as here, 1166 with whole rows (which would cut the sum over the tokens into four wavefronts).
// Measured (us per call, blocks of 16 tokens read in 64-byte pieces -> this form): 16 x 8192 tokens 1400 -> 1240 (4.5 TB/s),
// 8 x 4096 368 -> 283, 16 x 500 82 -> 66, 4 x 900 75 -> 68; shared states 16 x 8192 777 -> 659.
//
// Precision: the state update uses k * exp(-B_s) as hi + lo, two bf16 terms, so the state keeps fp32-level
// accuracy (decay and accumulation are fp32; v is bf16 as given), and the scores enter o = A v as
// hi + lo as well (their signed products per row do not average out a 2^-9 rounding). The rest of
// the output path rounds its operands (q*exp(B), k*exp(-B), S_0) to bf16 like any bf16 GEMM.
// exp(-B_s) grows with the gates of one block: 32 * max|g| stays far below the fp32/bf16
// exponent range for any log-sigmoid gate (|g| up to 2.5 per token, sustained); the exponent is clamped at
// 80 as a guard. Gates that reach the clamp in a block (results then under-weight near-diagonal terms) are counted, per 32
// key dims, in a device counter that sb_gla_gate_range_hits reads.
//
// Tile row order: accumulator tile rt of the state holds rows 32*(rt/2) + 8*(m/4) + 4*(rt%2) + m%4
// (m = tile row), so that the 8 consecutive rows a lane needs as the B operand of q S_0 are exactly
// the rows it already holds in tiles 2*st and 2*st+1: no cross-lane movement between the update
// and the next block's read of the state.
//
// Token order of a contraction over tokens: a lane's k index 8g + j stands for token 4g + j for j < 4 and
// token 16 + 4g + j - 4 above, which is where the accumulator tiles of the two 16-token halves leave the scores.
#include <mutex>

#include "common.h"
#include "mfma_util.h"

// Events of gla_chunk_kernel meeting gates beyond the block form's range (one per 32 key dims and block
// concerned) since the counter was last cleared; one copy per GPU (the name is only the host's handle for
// hipGetSymbolAddress).
static __device__ unsigned int gla_range_hits;

namespace {

using namespace sb;

struct GlaChunkParams {
  const uint16_t *q, *k, *v;  // bf16
  const void *g;
  void *state;
  uint16_t *out;
  const int32_t *slot_idx;
  const int32_t *cu;
  int H, T;
  float scale;
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, g_sb, g_sh, g_st, o_sb, o_sh, o_st;
  int64_t s_slot, s_head;
  // Shared states: G query heads per head of k, v, g and state; head index hh of this launch (H of them)
  // stands for state head hh / jn and query head (hh / jn) * G + j0 + hh % jn; write_state: store the
  // final state. One state per head: G = jn = 1, j0 = 0, write_state = 1.
  int G, jn, j0, write_state;
  unsigned int *range_hits;  // device counter of (32 key dims, block) events whose gates reached the exponent clamp
  // Prompts cut into segments (0: not cut): seg_tokens tokens each, n_seg of them for the longest prompt. ws holds
  // per (row, state head) n_seg states in register order, 16384 floats each, and behind all of those (chains of them) the decays of
  // the segments, 128 factors each. State 0 is the one the prompt starts from, state 1 the one behind its first segment, state i > 1
  // what segment i - 1 adds; scanned: gla_segment_scan_kernel has turned them into the states that the segments start from.
  int seg_tokens, n_seg, scanned;
  int64_t chains;
  float *ws;
};

constexpr int kCB = 32;      // tokens per block
constexpr float kMaxExp = 80.f;

// All operands are stored token-major, one 16-byte store per thread each. The state update and the output
// product contract over tokens and need [dim][token] operands: those are read with the transposing LDS load
// (ds_read_b64_tr_b16), no transposed copy is ever written.
typedef uint16_t Operand[kCB * 128];   // [token][dim], the 16-byte pieces of a row permuted: see piece_at

struct KvStage {
  Operand ks;      // k * exp(-B_t) rounded to bf16: score operand, and high part of the state-update operand
  Operand kl;      // what the rounding left: low part of the state-update operand
  Operand vs;      // v as loaded
  float dec[128];  // exp(B_32)
};
// Gate sums of the block's first 16 tokens, for the wavefronts that hold the second 16; those of the first half read zeros.
// Stores that are not wanted go to `spare`: no branches in that code.
struct Carry {
  float first[128], zero[128], spare[4];
};

// Rows are 256 bytes = all 64 banks, so piece p of row t lies at place p ^ f(t), with f such that the 16-byte accesses of 8
// consecutive rows (matrix operands), of rows 0, 2, 4, 6 and two pieces (the stores) and the transposing loads of four rows
// by four pieces all spread over the banks: the low two bits of t in front (a transposing load takes pieces 4 P .. 4 P + 3 of
// rows 4 j .. 4 j + 3), bits 2 and 3 behind them. (Rows padded to 304 bytes instead spent half of the LDS cycles on conflicts; the counter
// still gives 0.43, 809 of a block's 1899 cycles, and where those come from is open.)
__device__ __forceinline__ int piece_at(int t, int piece) {
  return t * 128 + ((piece ^ ((t & 3) << 2 | (t >> 1 & 2) | (t >> 3 & 1))) << 3);
}

// ds_read_b64_tr_b16: in every group of 16 lanes, lane i names 8 bytes (4 elements) of LDS, "row i"; lane l
// receives element l % 4 of rows l / 4, l / 4 + 4, l / 4 + 8, l / 4 + 12 (checked on the GPU). With row
// i = (token t0 + i / 4, dims f(i % 4) .. + 3), lane l gets dim f(l / 4) + l % 4 of tokens t0 .. t0 + 3.
__device__ __forceinline__ uint2 load_transposed(const uint16_t *row) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)row);
  return __builtin_bit_cast(uint2, v);
}

// Loads through buffer descriptors: the descriptor holds a block's first row (wave-uniform, scalar registers),
// the thread's token row and column are a 32-bit vector offset that is the same for every block: no vector
// arithmetic per load.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_from(const char *first_row) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(first_row), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}
// x of the lane `shift` places down the row of 16 lanes, 0 where the row has no such lane
template <int kShift>
__device__ __forceinline__ float row_shr(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x110 + kShift, 0xf, 0xf, true));
}

__device__ __forceinline__ float bf16_to_f32(uint16_t x) { return __uint_as_float((uint32_t)x << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }  // v_cvt_pk_bf16_f32

// ---- pieces of a block that the kernels below share (same operations in the same order in all of them, so their
// states and outputs are the same bits) ----------------------------------------------------------------------------
template <int GDT>
constexpr int kGateBytes = GDT == SB_F32 ? 4 : 2;

// What thread `lane` of wavefront w loads and prepares: dims 8 piece .. 8 piece + 7 of tokens tok and tok + 1. A wavefront has
// half of the dims of half of the tokens, so that its loads find 128 bytes of a row together; two pieces by eight token pairs
// sit in the 16 lanes of a DPP row, the pairs two lanes apart.
struct Share {
  int piece, tok;
  bool last_pair;   // of its half of the block
  __device__ __forceinline__ Share(int w, int lane)
      : piece(8 * (w & 1) + 2 * (lane >> 4) + (lane & 1)), tok(16 * (w >> 1) + (lane & 14)), last_pair((lane & 14) == 14) {}
};
template <int GDT>
struct GateIn {
  uint4 g[2][kGateBytes<GDT> / 2];  // fp32: dims 0..3, 4..7 of the piece; 16-bit: all 8
};
struct KvIn {
  uint4 k[2], v[2];
};

// Where a thread's two rows lie behind a block's first row, in bytes. Tokens past the end of the prompt lie outside the
// descriptors: such a load gives zeros, and a token with g = 0, q = k = v = 0 changes nothing.
struct RowOffsets {
  uint32_t at[2];
  __device__ __forceinline__ RowOffsets(const Share &me, int piece_bytes, int64_t row_bytes) {
    at[0] = me.tok * (int)row_bytes + me.piece * piece_bytes;
    at[1] = at[0] + (int)row_bytes;
  }
  __device__ __forceinline__ void cut(const Share &me, int valid) {   // only tokens 0 .. valid - 1 of the block exist
    if (me.tok >= valid) at[0] = 0x80000000u;
    if (me.tok + 1 >= valid) at[1] = 0x80000000u;
  }
};

template <int GDT>
__device__ __forceinline__ float gate_at(const uint4 *g, int i) {
  if constexpr (GDT == SB_F32) return __uint_as_float(word(g[i >> 2], i & 3));
  else if constexpr (GDT == SB_BF16) return (i & 1) ? bf16_hi(word(g[0], i >> 1)) : bf16_lo(word(g[0], i >> 1));
  else return (i & 1) ? f16_hi(word(g[0], i >> 1)) : f16_lo(word(g[0], i >> 1));
}

// Gates of the thread's two tokens summed from the start of its half of the block on, per dim, in log2 units (bare v_exp
// afterwards); the first half's totals go to LDS. One add inside the pair, three row-shift adds over the pairs, one more for
// the first token (two separate tokens would take eight).
template <int GDT>
__device__ __forceinline__ void scan_gates(const GateIn<GDT> &in, const Share &me, int w, Carry &carry, float (&b0)[8], float (&b1)[8]) {
#pragma clang fp contract(off)   // (the last sum as a multiply-add would need its shifted operand moved first)
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x0 = gate_at<GDT>(in.g[0], i) * kLog2e;
    float x = x0 + gate_at<GDT>(in.g[1], i) * kLog2e;
    x += row_shr<2>(x);
    x += row_shr<4>(x);
    x += row_shr<8>(x);
    b1[i] = x;
    b0[i] = x0 + row_shr<2>(x);
  }
  const bool keep = w < 2 && me.last_pair;
  float *d = keep ? &carry.first[8 * me.piece] : carry.spare;
  *reinterpret_cast<float4 *>(d) = make_float4(b1[0], b1[1], b1[2], b1[3]);
  *reinterpret_cast<float4 *>(keep ? d + 4 : d) = make_float4(b1[4], b1[5], b1[6], b1[7]);
}
// ... and from the start of the block on, behind the barrier that follows
__device__ __forceinline__ void add_carry(const Carry &carry, const Share &me, int w, float (&b0)[8], float (&b1)[8]) {
  const float *first = (w < 2 ? carry.zero : carry.first) + 8 * me.piece;
  const f32x4_t x[2] = {*reinterpret_cast<const f32x4_t *>(first), *reinterpret_cast<const f32x4_t *>(first + 4)};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    b0[i] += x[i >> 2][i & 3];
    b1[i] += x[i >> 2][i & 3];
  }
}

// k-hat of the thread's two tokens as hi + lo, and v, into their rows
__device__ __forceinline__ void store_kv(KvStage &st, const Share &me, const KvIn &in, const float (&b0)[8], const float (&b1)[8]) {
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float(&b)[8] = u ? b1 : b0;
    uint32_t ks[4], kl[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x0 = bf16_lo(word(in.k[u], i)) * fast_exp2(fminf(-b[2 * i], kMaxExp * kLog2e));
      const float x1 = bf16_hi(word(in.k[u], i)) * fast_exp2(fminf(-b[2 * i + 1], kMaxExp * kLog2e));
      // the rounded value is the score operand and the high part of the state-update operand
      ks[i] = Mma<BF16>::pack(x0, x1);
      kl[i] = Mma<BF16>::pack(x0 - __uint_as_float(ks[i] << 16), x1 - __uint_as_float(ks[i] & 0xffff0000u));
    }
    const int at = piece_at(me.tok + u, me.piece);
    *reinterpret_cast<uint4 *>(&st.ks[at]) = make_uint4(ks[0], ks[1], ks[2], ks[3]);
    *reinterpret_cast<uint4 *>(&st.kl[at]) = make_uint4(kl[0], kl[1], kl[2], kl[3]);
    *reinterpret_cast<uint4 *>(&st.vs[at]) = in.v[u];
  }
}
// q * scale * exp(B) of the two tokens; e: exp(B)
__device__ __forceinline__ void store_q(Operand &qs, const Share &me, const uint4 (&q)[2], const float (&e0)[8], const float (&e1)[8],
                                        float scale) {
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float(&e)[8] = u ? e1 : e0;
    uint32_t x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      x[i] = Mma<BF16>::pack(bf16_lo(word(q[u], i)) * scale * e[2 * i], bf16_hi(word(q[u], i)) * scale * e[2 * i + 1]);
    *reinterpret_cast<uint4 *>(&qs[piece_at(me.tok + u, me.piece)]) = make_uint4(x[0], x[1], x[2], x[3]);
  }
}
// The block's decay: exp(B_32) of the last token
__device__ __forceinline__ void store_decay(KvStage &st, Carry &carry, const Share &me, int w, const float (&e1)[8]) {
  const bool keep = w >= 2 && me.last_pair;
  float *d = keep ? &st.dec[8 * me.piece] : carry.spare;
  *reinterpret_cast<float4 *>(d) = make_float4(e1[0], e1[1], e1[2], e1[3]);
  *reinterpret_cast<float4 *>(keep ? d + 4 : d) = make_float4(e1[4], e1[5], e1[6], e1[7]);
}

// The lane's place in a matrix tile, for code behind the block loop: worked out again there, or the addresses that the loop
// keeps for its operands would have copies of their own live across it (34 spilled registers).
struct TileLane {
  int g, c;
  __device__ __forceinline__ explicit TileLane(int lane) {
    asm volatile("" : "+v"(lane));
    g = lane >> 4;
    c = lane & 15;
  }
};

// 16-byte matrix operand: dims 32 s4 + 8g .. + 7 of token c of a half
__device__ __forceinline__ uint4 row_operand(const Operand &x, int half, int g, int c, int s4) {
  return *reinterpret_cast<const uint4 *>(&x[piece_at(c, 4 * s4 + g) + half * 16 * 128]);
}
// Operand of a product that contracts over the block's tokens: dims f(j) = 32 block + 8 j + 4 part, j = c / 4, element c % 4
__device__ __forceinline__ uint4 column_operand(const Operand &x, int g, int c, int block, int part) {
  const int at = piece_at(4 * g + (c >> 2), 4 * block + (c & 3)) + 4 * part;
  const uint2 lo = load_transposed(&x[at]), hi = load_transposed(&x[at + 16 * 128]);
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// The state of one (slot, head): 16 tiles of this wavefront's 32 columns; column n = c of tile nt is column
// 32w + 8 (c / 4) + 4 nt + c % 4, so that a lane has 8 neighbouring columns of its tokens' outputs in its two tiles (one
// 16-byte store). A lane's elements lie at one offset of its own
// plus constants (scalar offsets of the buffer loads: no address registers per element).
typedef f32x4_t StateTiles[8][2];
__device__ __forceinline__ int state_offset(int rt, int nt, int i) { return (32 * (rt >> 1) + 4 * (rt & 1) + i) * 128 + 4 * nt; }
template <bool kF32>
__device__ __forceinline__ void load_state(StateTiles &S, const char *base, int g, int c, int w) {
  const __amdgpu_buffer_rsrc_t rows = rows_from(base);
  const int at = (8 * g * 128 + 32 * w + 8 * (c >> 2) + (c & 3)) * (kF32 ? 4 : 2);
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        S[rt][nt][i] = kF32 ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, at, state_offset(rt, nt, i) * 4, 0))
                            : bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rows, at, state_offset(rt, nt, i) * 2, 0));
}
template <bool kF32>
__device__ __forceinline__ void store_state(const StateTiles &S, char *base, int g, int c, int w) {
  const __amdgpu_buffer_rsrc_t rows = rows_from(base);
  const int at = (8 * g * 128 + 32 * w + 8 * (c >> 2) + (c & 3)) * (kF32 ? 4 : 2);
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (kF32) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[rt][nt][i]), rows, at, state_offset(rt, nt, i) * 4, 0);
        else __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(S[rt][nt][i]), rows, at, state_offset(rt, nt, i) * 2, 0);
      }
}

// Scores x (rows s = 4g + i of a half, column t = c) as two bf16 terms
__device__ __forceinline__ void split_scores(const f32x4_t &x, uint2 &hi, uint2 &lo) {
  hi.x = Mma<BF16>::pack(x[0], x[1]);
  hi.y = Mma<BF16>::pack(x[2], x[3]);
  lo.x = Mma<BF16>::pack(x[0] - __uint_as_float(hi.x << 16), x[1] - __uint_as_float(hi.x & 0xffff0000u));
  lo.y = Mma<BF16>::pack(x[2] - __uint_as_float(hi.y << 16), x[3] - __uint_as_float(hi.y & 0xffff0000u));
}
__device__ __forceinline__ void mask_diagonal(f32x4_t &x, int g, int c) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * g + i > c) x[i] = 0.f;
}

// Rows 32 s4 + 8g .. + 7 of the state, rounded, as operand of q S_0
__device__ __forceinline__ uint4 state_operand(const StateTiles &S, int s4, int nt) {
  const f32x4_t &a = S[2 * s4][nt], &b = S[2 * s4 + 1][nt];
  return make_uint4(Mma<BF16>::pack(a[0], a[1]), Mma<BF16>::pack(a[2], a[3]), Mma<BF16>::pack(b[0], b[1]), Mma<BF16>::pack(b[2], b[3]));
}

// Scores of one head and block, and what they contribute to its outputs, o[half][tile]: o^T = v^T A^T, lane (g, c) has token c
// of a half and 4 of the tile's columns (the operand registers are the same either way round: a lane holds
// index c of the tile's outer dimension and 8g..8g+7 of the contraction in both operands).
__device__ __forceinline__ void output_scores(const uint4 (&ka)[2][4], const uint4 (&qa)[2][4], const uint4 (&vb)[2], int g, int c,
                                              f32x4_t (&o)[2][2]) {
  // (transposed) a[s half][t half], element i = A[t = c][s = 4g + i], zero above the diagonal
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t a00 = zero, a01 = zero, a11 = zero;
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) {
    a00 = Mma<BF16>::run(ka[0][s4], qa[0][s4], a00);
    a01 = Mma<BF16>::run(ka[0][s4], qa[1][s4], a01);
    a11 = Mma<BF16>::run(ka[1][s4], qa[1][s4], a11);
  }
  mask_diagonal(a00, g, c);
  mask_diagonal(a11, g, c);
  uint2 h00, l00, h01, l01, h11, l11;
  split_scores(a00, h00, l00);
  split_scores(a01, h01, l01);
  split_scores(a11, h11, l11);
  // the first half's scores fill half of the contraction: their low terms take the other, against v repeated
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    o[0][nt] = Mma<BF16>::run(make_uint4(vb[nt].x, vb[nt].y, vb[nt].x, vb[nt].y), make_uint4(h00.x, h00.y, l00.x, l00.y), zero);
    o[1][nt] = Mma<BF16>::run(vb[nt], make_uint4(l01.x, l01.y, l11.x, l11.y), zero);
    o[1][nt] = Mma<BF16>::run(vb[nt], make_uint4(h01.x, h01.y, h11.x, h11.y), o[1][nt]);
  }
}

// S <- diag(dec) (S + k-hat^T v); a tile pair is decayed behind the matrix instructions of the next one
__device__ __forceinline__ void update_state(StateTiles &S, const KvStage &st, int g, int c, const uint4 (&vb)[2]) {
  auto decay = [&](int rt) {
    const float4 dc = *reinterpret_cast<const float4 *>(&st.dec[32 * (rt >> 1) + 8 * g + 4 * (rt & 1)]);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      S[rt][nt][0] *= dc.x; S[rt][nt][1] *= dc.y; S[rt][nt][2] *= dc.z; S[rt][nt][3] *= dc.w;
    }
  };
#pragma unroll
  for (int rt = 0; rt < 8; ++rt) {
    // this lane's operand row is state row 32 (rt / 2) + 8 (c / 4) + 4 (rt % 2) + c % 4
    const uint4 kh = column_operand(st.ks, g, c, rt >> 1, rt & 1), kl = column_operand(st.kl, g, c, rt >> 1, rt & 1);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) S[rt][nt] = Mma<BF16>::run(kh, vb[nt], S[rt][nt]);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) S[rt][nt] = Mma<BF16>::run(kl, vb[nt], S[rt][nt]);
    if (rt > 0) decay(rt - 1);
  }
  decay(7);
}

// 8 columns of one token's output; rows past the end of the prompt fall outside the descriptor and are dropped
__device__ __forceinline__ void store_out(__amdgpu_buffer_rsrc_t rows, uint32_t off, const f32x4_t &a, const f32x4_t &b) {
  u32x4_t val;
  val.x = Mma<BF16>::pack(a[0], a[1]);
  val.y = Mma<BF16>::pack(a[2], a[3]);
  val.z = Mma<BF16>::pack(b[0], b[1]);
  val.w = Mma<BF16>::pack(b[2], b[3]);
  __builtin_amdgcn_raw_buffer_store_b128(val, rows, off, 0, 0);
}

// The state that segment `seg` of a prompt starts from: that behind the first segment, decayed and added to by those in between, or
// the one the scan left. A few additions are requested together. lds: room for kFoldMax segments' decays.
// Up to this many segments each one adds up what the segments before it hand on; from there on a scan over them, a launch of its own, is
// faster (us per call, added up / scanned: a workgroup per head, 2 x 2048 tokens in 9 72.1 / 77.8, 4 x 2048 in 4 120.5 / 127.7,
// 1 x 1024 in 9 40.1 / 40.2 and in 16 47.9 / 46.7, 16 heads 1 x 1000 in 16 37.5 / 33.8; a workgroup per group, 16 x 200 in 4
// 39.2 / 43.8, 4 x 200 in 6 31.6 / 32.2, 4 x 512 in 8 39.9 / 38.5).
constexpr int kFoldMax = 9, kFoldMaxGroup = 6;
__device__ __forceinline__ void segment_start(StateTiles &S, const GlaChunkParams &p, int64_t chain, int seg, int tid, int g, float *lds) {
  const int first = p.scanned ? seg : min(seg, 1), steps = seg - first;
  const f32x4_t *const entry = reinterpret_cast<const f32x4_t *>(p.ws + (chain * p.n_seg + first) * 16384) + tid;
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) S[rt][nt] = entry[(2 * rt + nt) * 256];
  if (steps == 0) return;
  const f32x4_t *const decay = reinterpret_cast<const f32x4_t *>(p.ws + ((p.chains * 128 + chain) * p.n_seg + 1) * 128);
  for (int i = tid; i < steps * 32; i += 256) reinterpret_cast<f32x4_t *>(lds)[i] = decay[i];
  __syncthreads();
  constexpr int kAhead = 3;
#pragma unroll
  for (int half = 0; half < 2; ++half)
    for (int i0 = 0; i0 < steps; i0 += kAhead) {
      f32x4_t add[kAhead][4][2];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int x = 0; x < 8; ++x) add[j][x >> 1][x & 1] = entry[(int64_t)(min(i0 + j, steps - 1) + 1) * 4096 + (8 * half + x) * 256];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
        if (i0 + j < steps)
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            const int rt = 4 * half + r4;
            const f32x4_t d = *reinterpret_cast<const f32x4_t *>(lds + (i0 + j) * 128 + 32 * (rt >> 1) + 8 * g + 4 * (rt & 1));
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
              for (int i = 0; i < 4; ++i) S[rt][nt][i] = fmaf(d[i], S[rt][nt][i], add[j][r4][nt][i]);
          }
    }
}

// kCheck: report gates beyond the block form's range (SB_GLA_CHECK_GATES); a build of its own, because even this
// little extra work shifts the register allocation of a kernel that runs at the edge of its budget (0-4 % slower).
// kSeg: the workgroup runs one segment of its prompt, from the state that segment_start finds in the workspace
// for it; the workgroup of a prompt's last segment stores the final state.
template <bool kStateF32, int GDT, bool kCheck, bool kSeg>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gla_chunk_kernel(const GlaChunkParams p) {
  const int seg = kSeg ? (int)blockIdx.y : 0;
  const int b = blockIdx.x / p.H;
  const int hh = blockIdx.x - b * p.H;
  const int hk = hh / p.jn;
  const int h = hk * p.G + p.j0 + (hh - hk * p.jn);
  const int64_t slot = p.slot_idx ? (int64_t)p.slot_idx[b] : (int64_t)b;
  if (slot < 0) return;
  int T = p.T;
  int64_t qo, ko, vo, go, oo;
  if (p.cu) {
    const int64_t t0 = p.cu[b];
    T = p.cu[b + 1] - (int)t0;
    qo = t0 * p.q_st; ko = t0 * p.k_st; vo = t0 * p.v_st; go = t0 * p.g_st; oo = t0 * p.o_st;
  } else {
    qo = b * p.q_sb; ko = b * p.k_sb; vo = b * p.v_sb; go = b * p.g_sb; oo = b * p.o_sb;
  }
  bool last_segment = true;
  if constexpr (kSeg) {
    const int64_t t0 = (int64_t)seg * p.seg_tokens;
    // (the last segment there is takes what is left, also of a prompt longer than the call's bound said)
    last_segment = seg + 1 == p.n_seg || T <= t0 + p.seg_tokens;
    T = last_segment ? (int)(T - t0) : p.seg_tokens;
    qo += t0 * p.q_st; ko += t0 * p.k_st; vo += t0 * p.v_st; go += t0 * p.g_st; oo += t0 * p.o_st;
  }
  if (T <= 0) return;
  qo += h * p.q_sh; ko += hk * p.k_sh; vo += hk * p.v_sh; go += hk * p.g_sh; oo += h * p.o_sh;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const Share me(w, lane);

  __shared__ __attribute__((aligned(16))) KvStage stage[2];
  __shared__ __attribute__((aligned(16))) Operand qs;   // q * exp(B_t) * scale
  __shared__ __attribute__((aligned(16))) Carry carry;

  // ---- state: 8 row tiles x 2 column tiles of this wavefront's 32 columns -------------------------
  char *sbase = reinterpret_cast<char *>(p.state) + (slot * p.s_slot + (int64_t)hk * p.s_head) * (kStateF32 ? 4 : 2);
  StateTiles S;

  // ---- block inputs in registers -------------------------------------------------------------------------
  constexpr int GB = kGateBytes<GDT>;
  const char *gb = reinterpret_cast<const char *>(p.g) + go * GB;
  const char *qb = reinterpret_cast<const char *>(p.q + qo), *kb = reinterpret_cast<const char *>(p.k + ko),
             *vb_ = reinterpret_cast<const char *>(p.v + vo);
  const int64_t g_row = p.g_st * GB, q_row = p.q_st * 2, k_row = p.k_st * 2, v_row = p.v_st * 2, o_row = p.o_st * 2;
  RowOffsets q_at(me, 16, q_row), k_at(me, 16, k_row), v_at(me, 16, v_row), g_at(me, 8 * GB, g_row);
  const int last = (T - 1) / kCB;   // (only this block can have rows past the end, and it is fetched last)
  GateIn<GDT> gates;
  KvIn kv;
  uint4 q[2];
  auto fetch_gates = [&](int n) {
    if ((n + 1) * kCB > T) g_at.cut(me, T - n * kCB);
    const __amdgpu_buffer_rsrc_t gr = rows_from(gb + n * kCB * g_row);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < GB / 2; ++j) gates.g[u][j] = load16(gr, g_at.at[u] + 16 * j);
  };
  auto fetch = [&](int n) {
    if ((n + 1) * kCB > T) { q_at.cut(me, T - n * kCB); k_at.cut(me, T - n * kCB); v_at.cut(me, T - n * kCB); }
    const __amdgpu_buffer_rsrc_t qr = rows_from(qb + n * kCB * q_row), kr = rows_from(kb + n * kCB * k_row),
                                 vr = rows_from(vb_ + n * kCB * v_row);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      kv.k[u] = load16(kr, k_at.at[u]);
      q[u] = load16(qr, q_at.at[u]);
      kv.v[u] = load16(vr, v_at.at[u]);
    }
  };

  // ---- the LDS operands of one block -----------------------------------------------------------------------
  float b0[8], b1[8];   // gate sums of the thread's two tokens
  auto prepare = [&](KvStage &st, [[maybe_unused]] bool real) {
    add_carry(carry, me, w, b0, b1);
    // Gate range: the largest exponent formed in a block is minus its total log-decay; one event per 32 dims = half of the
    // wavefronts that hold the last token, reported on the spot
    if constexpr (kCheck) {
      const float worst = fminf(fminf(fminf(b1[0], b1[1]), fminf(b1[2], b1[3])), fminf(fminf(b1[4], b1[5]), fminf(b1[6], b1[7])));
      const uint64_t hit = __builtin_amdgcn_ballot_w64(real && w >= 2 && me.last_pair && worst < -kMaxExp * kLog2e);
      if (hit != 0 && lane == 0) atomicAdd(p.range_hits, ((uint32_t)hit != 0) + ((uint32_t)(hit >> 32) != 0));
    }
    store_kv(st, me, kv, b0, b1);
#pragma unroll
    for (int i = 0; i < 8; ++i) { b0[i] = fast_exp2(b0[i]); b1[i] = fast_exp2(b1[i]); }
    store_q(qs, me, q, b0, b1, p.scale);
    store_decay(st, carry, me, w, b1);
  };

  // ---- the outputs of one block on this wavefront's 32 state columns ----------------------------------------
  uint4 vb[2];
  auto outputs = [&](int n, const KvStage &st) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) vb[nt] = column_operand(st.vs, g, c, w, nt);
    uint4 qa[2][4], ka[2][4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int u = 0; u < 2; ++u) { ka[u][s4] = row_operand(st.ks, u, g, c, s4); qa[u][s4] = row_operand(qs, u, g, c, s4); }
    f32x4_t o[2][2];
    output_scores(ka, qa, vb, g, c, o);
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const uint4 sb16 = state_operand(S, s4, nt);
#pragma unroll
        for (int u = 0; u < 2; ++u) o[u][nt] = Mma<BF16>::run(sb16, qa[u][s4], o[u][nt]);
      }
    const __amdgpu_buffer_rsrc_t orows = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<char *>(p.out + oo) + n * kCB * o_row, 0, min(kCB, T - n * kCB) * (int)o_row, 0x00020000);
#pragma unroll
    for (int u = 0; u < 2; ++u) store_out(orows, (16 * u + c) * (int)o_row + (32 * w + 8 * g) * 2, o[u][0], o[u][1]);
  };

  // ---- block loop. Loads are issued as soon as their registers are free: the gates of block n + 2 in the first stretch of
  // block n, its q, k and v in the second.
  if (tid < 128) carry.zero[tid] = 0.f;
  fetch_gates(0);
  fetch(0);
  if constexpr (kSeg) segment_start(S, p, b * (int64_t)(p.H / p.jn) + hk, seg, tid, g, reinterpret_cast<float *>(&stage[1]));
  else load_state<kStateF32>(S, sbase, g, c, w);   // (behind the first block's loads, which are waited for first)
  scan_gates<GDT>(gates, me, w, carry, b0, b1);
  fetch_gates(min(1, last));
  __syncthreads();
  prepare(stage[0], true);
  fetch(min(1, last));
  // (one body for all blocks: the last one forms operands that nothing multiplies, 0.5 us; a copy of the body without them
  // behind the loop costs registers that the loop needs, 8 x 4096 tokens 283 -> 288-328 us)
  for (int n = 0; n <= last; ++n) {
    const KvStage &now = stage[n & 1];
    __syncthreads();
    scan_gates<GDT>(gates, me, w, carry, b0, b1);
    fetch_gates(min(n + 2, last));
    outputs(n, now);
    __syncthreads();   // the first half's gate sums are there, and every wavefront has read this block's q
    prepare(stage[(n & 1) ^ 1], n < last);
    fetch(min(n + 2, last));
    update_state(S, now, g, c, vb);
  }

  if (kSeg ? (!last_segment || hh % p.jn != 0) : !p.write_state) return;
  store_state<kStateF32>(S, sbase, g, c, w);
}

// ---- prompts cut into segments -----------------------------------------------------------------------------------
// Few chains (one prompt: 28 of them) leave most CUs idle, so long prompts are cut: the segments' own contributions
// to the state (from a zero start) and total decays are formed side by side (gla_segment_state_kernel), and the prompt kernels
// then run all segments at once, each from the state that the segments before it add up to (segment_start; with many segments
// a scan, gla_segment_scan_kernel, adds up once for all). Segments are whole blocks, so the operands of a block are those of the
// uncut prompt. k, v and the gate are read twice; what is bought is n_seg times as many workgroups.

// One workgroup per (row, state head, segment but the last): S_loc = sum over the segment's tokens of
// (k_s exp(B_end - B_s))^T v_s (the first one starts from the prompt's state instead of zero), with the operand arithmetic and the tiles of gla_chunk_kernel but
// without its outputs (32 matrix instructions per wavefront and block instead of 66, no q).

template <bool kStateF32, int GDT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gla_segment_state_kernel(const GlaChunkParams p) {
  const int seg = blockIdx.y;
  const int Hk = p.H;   // state heads here
  const int b = blockIdx.x / Hk;
  const int hk = blockIdx.x - b * Hk;
  const int64_t slot = p.slot_idx ? (int64_t)p.slot_idx[b] : (int64_t)b;
  if (slot < 0) return;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const int64_t chain = blockIdx.x;
  StateTiles S;
  auto hand_on = [&](int entry) __attribute__((always_inline)) {
    f32x4_t *dst = reinterpret_cast<f32x4_t *>(p.ws + (chain * p.n_seg + entry) * 16384) + tid;
#pragma unroll
    for (int rt = 0; rt < 8; ++rt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) dst[(2 * rt + nt) * 256] = S[rt][nt];
  };
  int T = p.T;
  int64_t ko, vo, go;
  if (p.cu) {
    const int64_t t0 = p.cu[b];
    T = p.cu[b + 1] - (int)t0;
    ko = t0 * p.k_st; vo = t0 * p.v_st; go = t0 * p.g_st;
  } else {
    ko = b * p.k_sb; vo = b * p.v_sb; go = b * p.g_sb;
  }
  const int64_t s0 = (int64_t)seg * p.seg_tokens;
  const char *const sbase = reinterpret_cast<const char *>(p.state) + (slot * p.s_slot + (int64_t)hk * p.s_head) * (kStateF32 ? 4 : 2);
  if (T <= s0 + p.seg_tokens) {   // a prompt's last segment hands nothing on
    if (seg == 0) {
      load_state<kStateF32>(S, sbase, g, c, w);
      hand_on(0);
    }
    return;
  }
  ko += s0 * p.k_st + hk * p.k_sh; vo += s0 * p.v_st + hk * p.v_sh; go += s0 * p.g_st + hk * p.g_sh;

  const Share me(w, lane);

  __shared__ __attribute__((aligned(16))) KvStage stage[2];
  __shared__ __attribute__((aligned(16))) Carry carry;

  constexpr int GB = kGateBytes<GDT>;
  const char *gb = reinterpret_cast<const char *>(p.g) + go * GB;
  const char *kb = reinterpret_cast<const char *>(p.k + ko), *vb_ = reinterpret_cast<const char *>(p.v + vo);
  const int64_t g_row = p.g_st * GB, k_row = p.k_st * 2, v_row = p.v_st * 2;
  const RowOffsets k_at(me, 16, k_row), v_at(me, 16, v_row), g_at(me, 8 * GB, g_row);   // (every block of such a segment is whole)
  const int last = p.seg_tokens / kCB - 1;
  GateIn<GDT> gates;
  KvIn kv;
  auto fetch_gates = [&](int n) {
    const __amdgpu_buffer_rsrc_t gr = rows_from(gb + n * kCB * g_row);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < GB / 2; ++j) gates.g[u][j] = load16(gr, g_at.at[u] + 16 * j);
  };
  auto fetch = [&](int n) {
    const __amdgpu_buffer_rsrc_t kr = rows_from(kb + n * kCB * k_row), vr = rows_from(vb_ + n * kCB * v_row);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      kv.k[u] = load16(kr, k_at.at[u]);
      kv.v[u] = load16(vr, v_at.at[u]);
    }
  };
  float b0[8], b1[8], total[8];   // total: of the segment, in the lanes that hold the last token of a block
#pragma unroll
  for (int i = 0; i < 8; ++i) total[i] = 0.f;
  auto prepare = [&](KvStage &st) {
    add_carry(carry, me, w, b0, b1);
    store_kv(st, me, kv, b0, b1);
#pragma unroll
    for (int i = 0; i < 8; ++i) { total[i] += b1[i]; b1[i] = fast_exp2(b1[i]); }
    store_decay(st, carry, me, w, b1);
  };

  if (tid < 128) carry.zero[tid] = 0.f;
  fetch_gates(0);
  fetch(0);
  if (seg == 0) load_state<kStateF32>(S, sbase, g, c, w);
  else
#pragma unroll
    for (int rt = 0; rt < 8; ++rt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) S[rt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  scan_gates<GDT>(gates, me, w, carry, b0, b1);
  fetch_gates(min(1, last));
  __syncthreads();
  prepare(stage[0]);
  // the prompt's state is also passed on as it is: the segments of the next launch read it while the last of them stores the final
  // one into the cache
  if (seg == 0) hand_on(0);
  fetch(min(1, last));
  int n = 0;
  uint4 vb[2];
  auto v_operands = [&](const KvStage &st, int g, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) vb[nt] = column_operand(st.vs, g, c, w, nt);
  };
  for (; n < last; ++n) {
    const KvStage &now = stage[n & 1];
    __syncthreads();
    scan_gates<GDT>(gates, me, w, carry, b0, b1);
    fetch_gates(min(n + 2, last));
    v_operands(now, g, c);
    __syncthreads();
    prepare(stage[(n & 1) ^ 1]);
    fetch(min(n + 2, last));
    update_state(S, now, g, c, vb);
  }
  __syncthreads();
  const TileLane end(lane);
  v_operands(stage[n & 1], end.g, end.c);
  update_state(S, stage[n & 1], end.g, end.c, vb);
  hand_on(seg + 1);
  if (w >= 2 && me.last_pair) {
    float4 *d = reinterpret_cast<float4 *>(p.ws + ((p.chains * 128 + chain) * p.n_seg + seg) * 128 + 8 * me.piece);
#pragma unroll
    for (int i = 0; i < 8; ++i) total[i] = fast_exp2(total[i]);
    d[0] = make_float4(total[0], total[1], total[2], total[3]);
    d[1] = make_float4(total[4], total[5], total[6], total[7]);
  }
}

// Grid (rows x state heads, 16 accumulator tiles): thread tid of workgroup (., tile) owns the four state elements
// that thread tid of the other kernels holds in that tile. In place: what segment i - 1 adds becomes the state that segment i
// starts from, with the operations of segment_start. A few segments' contributions are requested together, ahead of the
// chain over them.
__global__ __launch_bounds__(256) void gla_segment_scan_kernel(const GlaChunkParams p) {
  const int b = blockIdx.x / p.H;
  if (p.slot_idx && p.slot_idx[b] < 0) return;
  const int T = p.cu ? p.cu[b + 1] - p.cu[b] : p.T;
  const int n = min((T + p.seg_tokens - 1) / p.seg_tokens, p.n_seg);   // segments of this prompt
  const int tid = threadIdx.x, g = (tid & 63) >> 4;
  const int rt = blockIdx.y >> 1;
  const int64_t chain = blockIdx.x;
  f32x4_t *const ws = reinterpret_cast<f32x4_t *>(p.ws + chain * p.n_seg * 16384) + blockIdx.y * 256 + tid;
  const float *const decay = p.ws + (p.chains * 128 + chain) * p.n_seg * 128 + 32 * (rt >> 1) + 8 * g + 4 * (rt & 1);
  if (n < 3) return;
  f32x4_t S = ws[4096];
  constexpr int kAhead = 4;
  for (int s0 = 2; s0 < n; s0 += kAhead) {
    f32x4_t add[kAhead], d[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int s = min(s0 + j, n - 1);
      add[j] = ws[(int64_t)s * 4096];
      d[j] = *reinterpret_cast<const f32x4_t *>(decay + (s - 1) * 128);
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (s0 + j < n) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S[i] = fmaf(d[j][i], S[i], add[j][i]);
        ws[(int64_t)(s0 + j) * 4096] = S;
      }
  }
}

// ---- one pass for a whole GQA group (shared states) -----------------------------------------------------------
// One workgroup per (sequence, state head): the state is advanced ONCE per block and the outputs of all G query
// heads of the group are formed against it, instead of one workgroup per query head each carrying the whole
// recurrence (G - 1 of them only for their outputs). Per head the arithmetic and its order are those of
// gla_chunk_kernel (same operands, same matrix instructions in the same sequence), so the results are the same
// bits. The q operands of the G heads sit side by side in LDS; k-hat, v and the decays are prepared once.
constexpr int kMaxGroup = 8;

struct GroupStage {
  KvStage kv[2];
  Operand qs[kMaxGroup];
  Carry carry;
};

template <bool kStateF32, int GDT, bool kSeg>
__global__ __launch_bounds__(256) void gla_chunk_group_kernel(const GlaChunkParams p) {
  const int seg = kSeg ? (int)blockIdx.y : 0;
  const int b = blockIdx.x / p.H;   // p.H: state heads here
  const int hk = blockIdx.x - b * p.H;
  const int G = p.G;
  const int64_t slot = p.slot_idx ? (int64_t)p.slot_idx[b] : (int64_t)b;
  if (slot < 0) return;
  int T = p.T;
  int64_t qo, ko, vo, go, oo;
  if (p.cu) {
    const int64_t t0 = p.cu[b];
    T = p.cu[b + 1] - (int)t0;
    qo = t0 * p.q_st; ko = t0 * p.k_st; vo = t0 * p.v_st; go = t0 * p.g_st; oo = t0 * p.o_st;
  } else {
    qo = b * p.q_sb; ko = b * p.k_sb; vo = b * p.v_sb; go = b * p.g_sb; oo = b * p.o_sb;
  }
  bool last_segment = true;
  if constexpr (kSeg) {
    const int64_t t0 = (int64_t)seg * p.seg_tokens;
    // (the last segment there is takes what is left, also of a prompt longer than the call's bound said)
    last_segment = seg + 1 == p.n_seg || T <= t0 + p.seg_tokens;
    T = last_segment ? (int)(T - t0) : p.seg_tokens;
    qo += t0 * p.q_st; ko += t0 * p.k_st; vo += t0 * p.v_st; go += t0 * p.g_st; oo += t0 * p.o_st;
  }
  if (T <= 0) return;
  qo += (int64_t)hk * G * p.q_sh; ko += hk * p.k_sh; vo += hk * p.v_sh; go += hk * p.g_sh; oo += (int64_t)hk * G * p.o_sh;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const Share me(w, lane);

  extern __shared__ __attribute__((aligned(16))) char group_smem[];
  GroupStage &stage = *reinterpret_cast<GroupStage *>(group_smem);

  char *sbase = reinterpret_cast<char *>(p.state) + (slot * p.s_slot + (int64_t)hk * p.s_head) * (kStateF32 ? 4 : 2);
  StateTiles S;
  constexpr int GB = kGateBytes<GDT>;
  const char *gb = reinterpret_cast<const char *>(p.g) + go * GB;
  const char *qb = reinterpret_cast<const char *>(p.q + qo), *kb = reinterpret_cast<const char *>(p.k + ko),
             *vb_ = reinterpret_cast<const char *>(p.v + vo);
  const int64_t g_row = p.g_st * GB, q_row = p.q_st * 2, k_row = p.k_st * 2, v_row = p.v_st * 2, o_row = p.o_st * 2;
  const int64_t q_head = p.q_sh * 2, o_head = p.o_sh * 2;  // bytes between the group's heads
  RowOffsets q_at(me, 16, q_row), k_at(me, 16, k_row), v_at(me, 16, v_row), g_at(me, 8 * GB, g_row);
  const int last = (T - 1) / kCB;   // (only this block can have rows past the end, and it is fetched last)
  GateIn<GDT> gates;
  KvIn kv;
  uint4 q[kMaxGroup][2];
  auto fetch_gates = [&](int n) {
    if ((n + 1) * kCB > T) g_at.cut(me, T - n * kCB);
    const __amdgpu_buffer_rsrc_t gr = rows_from(gb + n * kCB * g_row);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < GB / 2; ++j) gates.g[u][j] = load16(gr, g_at.at[u] + 16 * j);
  };
  auto fetch = [&](int n) {
    if ((n + 1) * kCB > T) { q_at.cut(me, T - n * kCB); k_at.cut(me, T - n * kCB); v_at.cut(me, T - n * kCB); }
    const __amdgpu_buffer_rsrc_t kr = rows_from(kb + n * kCB * k_row), vr = rows_from(vb_ + n * kCB * v_row);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      kv.k[u] = load16(kr, k_at.at[u]);
      kv.v[u] = load16(vr, v_at.at[u]);
    }
#pragma unroll
    for (int h = 0; h < kMaxGroup; ++h)
      if (h < G) {
        const __amdgpu_buffer_rsrc_t qr = rows_from(qb + n * kCB * q_row + h * q_head);
        q[h][0] = load16(qr, q_at.at[0]);
        q[h][1] = load16(qr, q_at.at[1]);
      }
  };
  float b0[8], b1[8];   // gate sums of the thread's two tokens
  auto prepare = [&](KvStage &st) {
    add_carry(stage.carry, me, w, b0, b1);
    store_kv(st, me, kv, b0, b1);
#pragma unroll
    for (int i = 0; i < 8; ++i) { b0[i] = fast_exp2(b0[i]); b1[i] = fast_exp2(b1[i]); }
#pragma unroll
    for (int h = 0; h < kMaxGroup; ++h)
      if (h < G) store_q(stage.qs[h], me, q[h], b0, b1, p.scale);
    store_decay(st, stage.carry, me, w, b1);
  };

  uint4 vb[2];
  auto outputs = [&](int n, const KvStage &st, int g, int c) __attribute__((always_inline)) {
    // what every head of the group shares: k-hat as the score operand, v, and the state before the block as
    // the operand of q S_0
    uint4 ka[2][4], sb16[4][2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) vb[nt] = column_operand(st.vs, g, c, w, nt);
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int u = 0; u < 2; ++u) { ka[u][s4] = row_operand(st.ks, u, g, c, s4); sb16[s4][u] = state_operand(S, s4, u); }
    for (int h = 0; h < G; ++h) {
      uint4 qa[2][4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int u = 0; u < 2; ++u) qa[u][s4] = row_operand(stage.qs[h], u, g, c, s4);
      f32x4_t o[2][2];
      output_scores(ka, qa, vb, g, c, o);
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int u = 0; u < 2; ++u) o[u][nt] = Mma<BF16>::run(sb16[s4][nt], qa[u][s4], o[u][nt]);
      // (a descriptor per head: its bound drops the rows past the end of the prompt, whatever the head stride)
      const __amdgpu_buffer_rsrc_t orows = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char *>(p.out + oo) + n * kCB * o_row + h * o_head, 0, min(kCB, T - n * kCB) * (int)o_row, 0x00020000);
#pragma unroll
      for (int u = 0; u < 2; ++u) store_out(orows, (16 * u + c) * (int)o_row + (32 * w + 8 * g) * 2, o[u][0], o[u][1]);
    }
  };

  if (tid < 128) stage.carry.zero[tid] = 0.f;
  fetch_gates(0);
  fetch(0);
  if constexpr (kSeg) segment_start(S, p, blockIdx.x, seg, tid, g, reinterpret_cast<float *>(&stage.kv[1]));
  else load_state<kStateF32>(S, sbase, g, c, w);
  scan_gates<GDT>(gates, me, w, stage.carry, b0, b1);
  fetch_gates(min(1, last));
  __syncthreads();
  prepare(stage.kv[0]);
  fetch(min(1, last));
  auto finish = [&](int n) __attribute__((always_inline)) {
    const TileLane end(lane);
    __syncthreads();
    outputs(n, stage.kv[n & 1], end.g, end.c);
    if (!last_segment) return;
    update_state(S, stage.kv[n & 1], end.g, end.c, vb);
    store_state<kStateF32>(S, sbase, end.g, end.c, w);
  };
  if (last == 0) {
    finish(0);
    return;
  }
  int n = 0;
  do {
    const KvStage &now = stage.kv[n & 1];
    __syncthreads();
    scan_gates<GDT>(gates, me, w, stage.carry, b0, b1);
    fetch_gates(min(n + 2, last));
    outputs(n, now, g, c);
    __syncthreads();
    prepare(stage.kv[(n & 1) ^ 1]);
    fetch(min(n + 2, last));
    update_state(S, now, g, c, vb);
  } while (++n < last);
  finish(n);
}

}  // namespace

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_hits_mu;
unsigned int *g_hits_ptr[kMaxDevices];  // per device: address of that device's copy of gla_range_hits

// Address of the current device's counter (looked up once per device), or null with the error set.
unsigned int *range_hits_ptr() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    sb_host::set_error("gla_chunk: hipGetDevice: %s (device %d)", hipGetErrorString(e), dev);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_hits_mu);
  if (!g_hits_ptr[dev]) {
    void *ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(gla_range_hits));
    if (e != hipSuccess || !ptr) {
      sb_host::set_error("gla_chunk: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return nullptr;
    }
    g_hits_ptr[dev] = (unsigned int *)ptr;
  }
  return g_hits_ptr[dev];
}
}  // namespace

extern "C" int sb_gla_gate_range_hits(int64_t *hits, int32_t reset) {
  using namespace sb_host;
  if (!hits) return fail(SB_ERR_INVALID, "sb_gla_gate_range_hits: null pointer");
  unsigned int *ptr = range_hits_ptr();
  if (!ptr) return SB_ERR_INVALID;
  unsigned int h = 0;
  hipError_t e = hipMemcpy(&h, ptr, sizeof(h), hipMemcpyDeviceToHost);  // waits for the work queued before it
  if (e != hipSuccess) return fail((int)e, "sb_gla_gate_range_hits: hipMemcpy: %s", hipGetErrorString(e));
  if (reset) {
    e = hipMemset(ptr, 0, sizeof(h));
    if (e != hipSuccess) return fail((int)e, "sb_gla_gate_range_hits: hipMemset: %s", hipGetErrorString(e));
  }
  *hits = (int64_t)h;
  return SB_OK;
}

namespace sb_host {

static GlaChunkParams fill(const sb_gla_recurrent_args *a, int heads, int G, int jn, int j0, int write_state) {
  GlaChunkParams p;
  p.q = (const uint16_t *)a->q; p.k = (const uint16_t *)a->k; p.v = (const uint16_t *)a->v; p.g = a->g;
  p.state = a->state; p.out = (uint16_t *)a->out; p.slot_idx = a->slot_idx; p.cu = a->cu_seqlens;
  p.H = heads; p.T = a->seq_len; p.scale = a->scale;
  p.G = G; p.jn = jn; p.j0 = j0; p.write_state = write_state;
  p.q_sb = a->q_stride_b; p.q_sh = a->q_stride_h; p.q_st = a->q_stride_t;
  p.k_sb = a->k_stride_b; p.k_sh = a->k_stride_h; p.k_st = a->k_stride_t;
  p.v_sb = a->v_stride_b; p.v_sh = a->v_stride_h; p.v_st = a->v_stride_t;
  p.g_sb = a->g_stride_b; p.g_sh = a->g_stride_h; p.g_st = a->g_stride_t;
  p.o_sb = a->out_stride_b; p.o_sh = a->out_stride_h; p.o_st = a->out_stride_t;
  p.s_slot = a->state_stride_slot; p.s_head = a->state_stride_head;
  p.range_hits = nullptr;
  p.seg_tokens = p.n_seg = p.scanned = 0;
  p.chains = 0;
  p.ws = nullptr;
  return p;
}

// Launch for bf16 q/k/v/out; g of any built type. Grid: one workgroup per (row, head).
// Returns SB_OK, or an error when the device's hit counter cannot be located (nothing is launched then).
int launch_gla_chunk(const sb_gla_recurrent_args *a, int64_t groups, int heads, int G, int jn, int j0, int write_state) {
  GlaChunkParams p = fill(a, heads, G, jn, j0, write_state);
  const bool check = (a->flags & SB_GLA_CHECK_GATES) != 0;
  p.range_hits = check ? range_hits_ptr() : nullptr;
  if (check && !p.range_hits) return SB_ERR_INVALID;
  const dim3 grid((unsigned)groups), block(256);
  hipStream_t st = (hipStream_t)a->stream;
#define SB_LAUNCH(F32S, GDT)                                                                     \
  do {                                                                                           \
    if (check) hipLaunchKernelGGL((gla_chunk_kernel<F32S, GDT, true, false>), grid, block, 0, st, p);   \
    else hipLaunchKernelGGL((gla_chunk_kernel<F32S, GDT, false, false>), grid, block, 0, st, p);        \
  } while (0)
  if (a->state_dtype == SB_F32) {
    if (a->g_dtype == SB_F32) SB_LAUNCH(true, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(true, SB_BF16);
    else SB_LAUNCH(true, SB_F16);
  } else {
    if (a->g_dtype == SB_F32) SB_LAUNCH(false, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(false, SB_BF16);
    else SB_LAUNCH(false, SB_F16);
  }
#undef SB_LAUNCH
  return SB_OK;
}

static bool group_fits(const sb_gla_recurrent_args *a, int G) {
  return G >= 2 && G <= kMaxGroup && a->q_stride_h >= 0 && a->out_stride_h >= 0 && (int64_t)G * a->q_stride_h * 2 < (1LL << 30) &&
         (int64_t)G * a->out_stride_h * 2 < (1LL << 30);
}

template <bool kSeg>
static int launch_group_kernel(const sb_gla_recurrent_args *a, const GlaChunkParams &p, dim3 grid) {
  const dim3 block(256);
  hipStream_t st = (hipStream_t)a->stream;
  constexpr int kLds = (int)sizeof(GroupStage);
#define SB_LAUNCH(F32S, GDT)                                                                                     \
  do {                                                                                                           \
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gla_chunk_group_kernel<F32S, GDT, kSeg>), \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);                        \
    if (e != hipSuccess) return fail((int)e, "gla_chunk_group_kernel: %s", hipGetErrorString(e));                \
    hipLaunchKernelGGL((gla_chunk_group_kernel<F32S, GDT, kSeg>), grid, block, kLds, st, p);                     \
  } while (0)
  if (a->state_dtype == SB_F32) {
    if (a->g_dtype == SB_F32) SB_LAUNCH(true, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(true, SB_BF16);
    else SB_LAUNCH(true, SB_F16);
  } else {
    if (a->g_dtype == SB_F32) SB_LAUNCH(false, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(false, SB_BF16);
    else SB_LAUNCH(false, SB_F16);
  }
#undef SB_LAUNCH
  return SB_OK;
}

// Prompts cut into n_seg segments of seg_tokens tokens (whole blocks); ws: see GlaChunkParams. With shared
// states the segments fill the machine, so the one-pass kernel per group runs them (it does 0.4 x the work; per query
// head where its strides do not fit, again in one launch: no head reads the state cache the last segments store into).
int launch_gla_chunk_segments(const sb_gla_recurrent_args *a, int G, int n_seg, int seg_tokens, float *ws) {
  const int Hk = a->num_heads / G;
  GlaChunkParams p = fill(a, Hk, G, G, 0, 1);
  p.seg_tokens = seg_tokens; p.n_seg = n_seg; p.ws = ws;
  p.chains = a->batch * (int64_t)Hk;
  const bool grouped = group_fits(a, G) && !(a->flags & SB_GLA_PER_HEAD);
  p.scanned = n_seg > (grouped ? kFoldMaxGroup : kFoldMax);
  const dim3 block(256);
  const unsigned chains = (unsigned)p.chains;
  hipStream_t st = (hipStream_t)a->stream;
  const dim3 sgrid(chains, (unsigned)(n_seg - 1));
#define SB_LAUNCH(F32S, GDT) hipLaunchKernelGGL((gla_segment_state_kernel<F32S, GDT>), sgrid, block, 0, st, p)
  if (a->state_dtype == SB_F32) {
    if (a->g_dtype == SB_F32) SB_LAUNCH(true, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(true, SB_BF16);
    else SB_LAUNCH(true, SB_F16);
  } else {
    if (a->g_dtype == SB_F32) SB_LAUNCH(false, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(false, SB_BF16);
    else SB_LAUNCH(false, SB_F16);
  }
#undef SB_LAUNCH
  if (int rc = check_launch("gla_segment_state_kernel")) return rc;
  if (p.scanned) {
    hipLaunchKernelGGL(gla_segment_scan_kernel, dim3(chains, 16), block, 0, st, p);
    if (int rc = check_launch("gla_segment_scan_kernel")) return rc;
  }
  if (grouped) {
    const int rc = launch_group_kernel<true>(a, p, dim3(chains, (unsigned)n_seg));
    return rc ? rc : check_launch("gla_chunk_group_kernel");
  }
  p.H = a->num_heads;
  const dim3 grid((unsigned)(a->batch * (int64_t)a->num_heads), (unsigned)n_seg);
#define SB_LAUNCH(F32S, GDT) hipLaunchKernelGGL((gla_chunk_kernel<F32S, GDT, false, true>), grid, block, 0, st, p)
  if (a->state_dtype == SB_F32) {
    if (a->g_dtype == SB_F32) SB_LAUNCH(true, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(true, SB_BF16);
    else SB_LAUNCH(true, SB_F16);
  } else {
    if (a->g_dtype == SB_F32) SB_LAUNCH(false, SB_F32);
    else if (a->g_dtype == SB_BF16) SB_LAUNCH(false, SB_BF16);
    else SB_LAUNCH(false, SB_F16);
  }
#undef SB_LAUNCH
  return check_launch("gla_chunk_kernel");
}

// Shared states, one pass: grid = one workgroup per (row, state head), each forming the outputs of its G query
// heads. SB_ERR_UNSUPPORTED (nothing launched) where the group's head offsets do not fit the kernel's 32-bit
// in-block offsets; the caller then takes the launches per query head.
int launch_gla_chunk_group(const sb_gla_recurrent_args *a, int state_heads, int G) {
  if (!group_fits(a, G)) return SB_ERR_UNSUPPORTED;
  return launch_group_kernel<false>(a, fill(a, state_heads, G, 1, 0, 1), dim3((unsigned)(a->batch * (int64_t)state_heads)));
}

}  // namespace sb_host
