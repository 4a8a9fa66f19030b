// Window-bounded single-query attention over a per-row INT8 K/V cache (codes int8
// [nb, bs, Hkv, 128], scales fp32 [nb, Hkv, bs]), split-K, matrix cores. Half the HBM bytes of
// the bf16 cache per visible key (2 x 128 B codes + 8 B scales per kv head).
//
// Same decomposition and lane layouts as the bf16 kernel (one wavefront per kv head, chunks of
// 32 keys, S^T = K Q^T then O^T += V^T P^T with P staying in-lane); what differs:
//   * codes are widened to the query's 16-bit type on the way into the matrix cores (small integers
//     are exact there); a key's K scale multiplies its score, its V scale multiplies its
//     probability, both in fp32, so nothing is rounded that the reference does not round;
//   * the contraction over head dims is order-free, so lane (g, c) takes the 32 contiguous bytes
//     [32g, 32g+32) of key c (two 16-byte loads; the query operand uses the same dim order);
//   * V codes are loaded as 8-byte row pieces (lane (g,c): its 8 keys, dims 8c..8c+7); picking byte
//     mt of each while widening IS the 8x8 transpose the bf16 kernel does with v_perm;
//   * no byte pattern of a code is a NaN, so edge chunks only clamp their TILES into the resident
//     range (rows of a resident block are always addressable) and mask by key index; scales of
//     masked keys may be stale, so masked probabilities are selected to zero, never multiplied;
//   * a fused append (APPEND) quantises the newest row first: the wavefront whose run ends a row works its codes out while its
//     last chunk's loads are on their way, puts them in the place of what it reads there and stores them (nothing is read
//     back from memory; the bits are those of an append kernel in front). It saves that kernel's launch, and over fp8 the queries' round
//     trip, of which every decode layer had one: us per call, INT8 / fp8, 1 x 6000 keys 22.1 / 21.7 -> 13.0 / 13.3, 8 x 4000 22.1 / 21.7 ->
//     14.1 / 14.6, 256 x 400 24.5 / 25.2 -> 23.4 / 23.0, 100 uneven rows of a full window 80.5 / 77.2 -> 78.2 / 74.5; a captured step of 28
//     layers, 8 sequences, 345 / 337 -> 313 / 312. A build of its own, as it takes 28 to 36 registers;
//   * meta tokens (rows every query also attends to) are not part of the cache: they stay elements of the
//     query's type and are taken, ahead of the window, in chunks of 32 dealt round robin to the splits.
#include "common.h"
#include "kv_codes.h"
#include "mfma_util.h"
#include "swa_decode_params.h"

namespace {

using namespace sb;

constexpr float kNegInf = kNegInfF;

struct ChunkI8 {
  uint4 k[2][2];     // tile, half: bytes [32g + 16*half, +16) of key c
  uint2 v[8];        // key kk = 8g..8g+7 of the chunk: dims 8c..8c+7
  float4 ks[2], vs[2];  // scales of keys 4g..4g+3 of tile 0 / tile 1
};

// byte B of w as a float: a signed INT8 code, or an fp8 (OCP e4m3fn) code
template <int Q, int B>
__device__ __forceinline__ float code_to_float(uint32_t w) {
  if constexpr (Q == SB_KV_INT8) return (float)(int)(int8_t)(w >> (8 * B));
  else return __builtin_amdgcn_cvt_f32_fp8((int)w, B);
}

// 8 codes (two dwords) -> 8 elements of type E
template <typename E, int Q>
__device__ __forceinline__ uint4 widen8(uint32_t lo, uint32_t hi) {
  return make_uint4(Mma<E>::pack(code_to_float<Q, 0>(lo), code_to_float<Q, 1>(lo)),
                    Mma<E>::pack(code_to_float<Q, 2>(lo), code_to_float<Q, 3>(lo)),
                    Mma<E>::pack(code_to_float<Q, 0>(hi), code_to_float<Q, 1>(hi)),
                    Mma<E>::pack(code_to_float<Q, 2>(hi), code_to_float<Q, 3>(hi)));
}

__device__ __forceinline__ uint32_t word2(const uint2 &v, int i) { return i == 0 ? v.x : v.y; }

template <typename E, int Q, int B>
__device__ __forceinline__ uint4 v_column(const uint2 (&v)[8], int w) {
  return make_uint4(Mma<E>::pack(code_to_float<Q, B>(word2(v[0], w)), code_to_float<Q, B>(word2(v[1], w))),
                    Mma<E>::pack(code_to_float<Q, B>(word2(v[2], w)), code_to_float<Q, B>(word2(v[3], w))),
                    Mma<E>::pack(code_to_float<Q, B>(word2(v[4], w)), code_to_float<Q, B>(word2(v[5], w))),
                    Mma<E>::pack(code_to_float<Q, B>(word2(v[6], w)), code_to_float<Q, B>(word2(v[7], w))));
}

// 256 registers per wavefront (two per SIMD): the matrix-core results then live in ordinary registers
// and the rescale inside the loop costs no accumulator-register traffic.
// Q = SB_KV_FP8: the codes are fp8 with one scale per tensor: the K scale is folded into the softmax
// scale and the V scale into the result on the host side of the launch, nothing per key; an fp8 byte
// CAN be a NaN, so the V codes of masked keys are zeroed before they meet their zero probability.
template <typename E, int Q, bool APPEND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void swa_decode_split_i8_kernel(const DecodeParams p, const int G, const int Hkv) {
  const int64_t r = blockIdx.x;
  const int split = blockIdx.z;
  const int tid = threadIdx.x;
  const int kvh = blockIdx.y * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(tid >> 6);
  if (kvh >= Hkv) return;  // whole wavefront; there is no barrier in this kernel
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int c = lane & 15;

  const int64_t seq = p.row_seq ? (int64_t)p.row_seq[r] : r;
  const int hi = p.seq_lens[r];
  int lo = p.window_left >= 0 ? max(0, hi - 1 - p.window_left) : 0;
  if (p.key_lo) lo = max(lo, p.key_lo[r]);
  const bool any = hi > lo;
  const int first_tile = lo >> 4;
  const int last_tile = any ? (hi - 1) >> 4 : first_tile;
  const int first_chunk = lo >> 5;
  const int n_chunks = any ? ((hi - 1) >> 5) - first_chunk + 1 : 0;
  const int cps = (n_chunks + p.n_split - 1) / p.n_split;
  const int cb = first_chunk + split * cps;
  const int ce = min(cb + cps, first_chunk + n_chunks);

  // Q^T operands: head c of the group, dims 32g + 8s .. +7 for step s; zero rows pad the group
  uint4 qb[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    qb[s] = make_uint4(0u, 0u, 0u, 0u);
    if (c < G)
      qb[s] = *reinterpret_cast<const uint4 *>(
          p.q + (r * p.q_sr + (int64_t)(kvh * G + c) * p.q_sh + 32 * g + 8 * s) * 2);
  }

  // ---- the newest row: its elements now, its codes (in the layout of a chunk: K bytes [32g, +32), V bytes [8c, +8), both
  // scales) when the last chunk's loads are on their way, its stores at the end. 40 divisions a lane in front of the first
  // loads would be a microsecond of every owner, and a store ahead of the table lookups makes vector loads of them ----
  constexpr int kType = std::is_same_v<E, BF16> ? SB_BF16 : SB_F16;
  [[maybe_unused]] uint4 raw_k[4], raw_v;
  [[maybe_unused]] uint2 nk[4], nv;
  [[maybe_unused]] float nks = 1.f, nvs = 1.f;
  [[maybe_unused]] bool fresh = false;   // (uniform) this wavefront has it
  [[maybe_unused]] int64_t slot = -1;
  if constexpr (APPEND) {
    slot = p.slot_mapping[r];
    fresh = slot >= 0 && (any ? cb < ce && ce == first_chunk + n_chunks : split == 0);
    if (fresh) {
      const char *newk = p.new_k + r * p.nk_st + (int64_t)kvh * p.nk_sh, *newv = p.new_v + r * p.nv_st + (int64_t)kvh * p.nv_sh;
#pragma unroll
      for (int s = 0; s < 4; ++s) raw_k[s] = *reinterpret_cast<const uint4 *>(newk + 64 * g + 16 * s);
      raw_v = *reinterpret_cast<const uint4 *>(newv + 16 * c);
    }
  }
  auto round_queries = [&]() __attribute__((always_inline)) {   // their round trip through fp8
    if (APPEND && Q == SB_KV_FP8 && p.q_round > 0.f) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float x[8], y[8];
        unpack8<kType>(qb[s], x);
        fp8_values(fp8_bytes(x, p.q_round), p.q_round, y);
        qb[s] = pack8<kType>(y);
      }
    }
  };
  auto quantise_fresh = [&]() __attribute__((always_inline)) {
    if constexpr (APPEND) {
      if (!fresh) return;
      float x[4][8], vx[8], code[8];
#pragma unroll
      for (int s = 0; s < 4; ++s) unpack8<kType>(raw_k[s], x[s]);
      unpack8<kType>(raw_v, vx);
      if constexpr (Q == SB_KV_INT8) {
        float ka = 0.f, va = max_abs8(vx, 0.f);
#pragma unroll
        for (int s = 0; s < 4; ++s) ka = max_abs8(x[s], ka);
        ka = fmaxf(ka, __shfl_xor(ka, 16));
        ka = fmaxf(ka, __shfl_xor(ka, 32));
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) va = fmaxf(va, __shfl_xor(va, d));
        nks = int8_scale(ka);
        nvs = int8_scale(va);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          int8_codes(x[s], nks, code);
          nk[s] = int8_bytes(code);
        }
        int8_codes(vx, nvs, code);
        nv = int8_bytes(code);
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) nk[s] = fp8_bytes(x[s], p.nk_scale);
        nv = fp8_bytes(vx, p.nv_scale);
      }
    }
  };

  const float my_slope = (p.opt.slopes && c < G) ? p.opt.slopes[kvh * G + c] : 0.f;  // ALiBi slope of this lane's head

  f32x4_t acc[8];
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) acc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = kNegInf, l = 0.f;

  const uint32_t kv_sr32 = (uint32_t)p.kv_sr;
  const uint32_t koff = c * kv_sr32 + g * 32;
  uint32_t voff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) voff[j] = (4 * g + j) * kv_sr32 + c * 8;

  // Where a chunk's two tiles are: block-table entry and first row inside the block. Looked up one chunk ahead of its
  // loads (the lookup inside them kept every chunk's loads waiting for a table entry, and its block a division; with
  // the edge tests out of the interior chunks and nothing read twice at a run's end: 100 ragged rows 83.5 -> 81.0 us a call;
  // the code grew by 1100 instructions for it, which shows in the shortest fp8 runs: 100 rows of 200 keys 12.4 -> 13.0 us, of
  // 6000 80.0 -> 77.8; INT8 14.8 -> 13.5, 82.7 -> 80.4).
  const int tiles_per_block = p.block_size >> 4;
  const int32_t *const table_row = p.block_table + seq * p.bt_stride;
  struct Where {
    int blk[2], row[2];
  };
  auto locate = [&](int cc, Where &at) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int tile = min(max(2 * cc + t, first_tile), last_tile);  // resident, uniform over the wavefront
      const int bi = tile_block(tile, p.tile_div);
      at.row[t] = (tile - bi * tiles_per_block) << 4;
      at.blk[t] = table_row[bi];
    }
  };
  auto load_chunk = [&](const Where &at, ChunkI8 &ck) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int row = at.row[t];
      const int64_t blk = at.blk[t];
      const int64_t base = blk * p.kv_sb + (int64_t)row * p.kv_sr + (int64_t)kvh * p.kv_sh;
      const char *kp = p.k + base, *vp = p.v + base;
      ck.k[t][0] = load_stream16(kp + koff);
      ck.k[t][1] = load_stream16(kp + koff + 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned long long w = __builtin_nontemporal_load(reinterpret_cast<const unsigned long long *>(vp + voff[j]));
        ck.v[4 * t + j] = make_uint2((uint32_t)w, (uint32_t)(w >> 32));
      }
      if constexpr (Q == SB_KV_INT8) {
        const int64_t sbase = (blk * Hkv + kvh) * p.block_size + row + 4 * g;
        ck.ks[t] = *reinterpret_cast<const float4 *>(p.k_scale + sbase);
        ck.vs[t] = *reinterpret_cast<const float4 *>(p.v_scale + sbase);
      }
    }
  };

  // LAST: may be the last chunk of the run
  auto compute_chunk = [&](int ch, ChunkI8 &ck, auto last_tag) __attribute__((always_inline)) {
    [[maybe_unused]] constexpr bool LAST = APPEND && decltype(last_tag)::value;
    if constexpr (LAST) {
      if (fresh && ch == (hi - 1) >> 5) {
        const int key = (hi - 1) & 31;
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (key >> 4 == t && c == (key & 15)) {
            ck.k[t][0] = make_uint4(nk[0].x, nk[0].y, nk[1].x, nk[1].y);
            ck.k[t][1] = make_uint4(nk[2].x, nk[2].y, nk[3].x, nk[3].y);
          }
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (key == ((j >> 2) << 4) + 4 * g + (j & 3)) {
            ck.v[j] = nv;
            if constexpr (Q == SB_KV_INT8) {
              (&ck.ks[j >> 2].x)[j & 3] = nks;
              (&ck.vs[j >> 2].x)[j & 3] = nvs;
            }
          }
      }
    }
    f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint4 &a = ck.k[0][s >> 1], &b = ck.k[1][s >> 1];
      s0 = Mma<E>::run((s & 1) ? widen8<E, Q>(a.z, a.w) : widen8<E, Q>(a.x, a.y), qb[s], s0);
      s1 = Mma<E>::run((s & 1) ? widen8<E, Q>(b.z, b.w) : widen8<E, Q>(b.x, b.y), qb[s], s1);
    }
    float sc[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
    float vsc[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
    if constexpr (Q == SB_KV_INT8) {
      const float ksc[8] = {ck.ks[0].x, ck.ks[0].y, ck.ks[0].z, ck.ks[0].w, ck.ks[1].x, ck.ks[1].y, ck.ks[1].z, ck.ks[1].w};
      const float vs8[8] = {ck.vs[0].x, ck.vs[0].y, ck.vs[0].z, ck.vs[0].w, ck.vs[1].x, ck.vs[1].y, ck.vs[1].z, ck.vs[1].w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sc[j] *= ksc[j];
        vsc[j] = vs8[j];
      }
    }
    const int i0 = ch << 5;
    if (p.opt.on) {  // soft cap / ALiBi (wave-uniform; the query sits at key index hi - 1)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        sc[j] = adjust_score(p.opt, sc[j], my_slope, (float)(i0 + ((j >> 2) << 4) + 4 * g + (j & 3) - (hi - 1)));
    }
    if (i0 < lo || i0 + 32 > hi) {  // (first and last chunk of a window only) masked keys: no score, no scale, no fp8 byte
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int i = i0 + ((j >> 2) << 4) + 4 * g + (j & 3);
        if (i < lo || i >= hi) {
          sc[j] = kNegInf;
          vsc[j] = 0.f;
          if constexpr (Q == SB_KV_FP8) ck.v[j] = make_uint2(0u, 0u);
        }
      }
    }
    float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m, mx * p.scale_log2);
    const float m_safe = (m_new == kNegInf) ? 0.f : m_new;
    const float alpha = fast_exp2(m - m_safe);
    const bool grew = m_new > m;
    m = m_new;
    float psum = 0.f, pv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = fast_exp2(fmaf(sc[j], p.scale_log2, -m_safe));
      psum += e;
      pv[j] = e * vsc[j];
    }
    l = fmaf(l, alpha, psum);
    if (__builtin_amdgcn_ballot_w64(grew) != 0) {
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) acc[mt] *= alpha;
    }
    const uint4 pb = make_uint4(Mma<E>::pack(pv[0], pv[1]), Mma<E>::pack(pv[2], pv[3]),
                                Mma<E>::pack(pv[4], pv[5]), Mma<E>::pack(pv[6], pv[7]));
    acc[0] = Mma<E>::run(v_column<E, Q, 0>(ck.v, 0), pb, acc[0]);
    acc[1] = Mma<E>::run(v_column<E, Q, 1>(ck.v, 0), pb, acc[1]);
    acc[2] = Mma<E>::run(v_column<E, Q, 2>(ck.v, 0), pb, acc[2]);
    acc[3] = Mma<E>::run(v_column<E, Q, 3>(ck.v, 0), pb, acc[3]);
    acc[4] = Mma<E>::run(v_column<E, Q, 0>(ck.v, 1), pb, acc[4]);
    acc[5] = Mma<E>::run(v_column<E, Q, 1>(ck.v, 1), pb, acc[5]);
    acc[6] = Mma<E>::run(v_column<E, Q, 2>(ck.v, 1), pb, acc[6]);
    acc[7] = Mma<E>::run(v_column<E, Q, 3>(ck.v, 1), pb, acc[7]);
  };

  // ---- meta rows: dense element tensors [meta_len, Hkv, 128], chunk cc = rows 32cc .. 32cc+31 clamped to the
  // last row (masked by their true index). K operand in this kernel's dim order (lane (g, c): bytes
  // [64g, 64g+64) of row c), V rows as the element kernel takes them (lane (g, c): bytes [16c, 16c+16) of its
  // 8 keys, transposed in registers). The rows have no scales: meta_k_mult / meta_v_mult undo the tensor
  // scales an fp8 cache folds into scale_log2 and kv_out_scale.
  auto meta_chunk = [&](int cc) {
    const char *mk = p.meta_k + (int64_t)kvh * p.meta_sh, *mv = p.meta_v + (int64_t)kvh * p.meta_sh;
    const int last = p.meta_len - 1, i0 = cc << 5;
    const char *pk0 = mk + (int64_t)min(i0 + c, last) * p.meta_sr + g * 64;
    const char *pk1 = mk + (int64_t)min(i0 + 16 + c, last) * p.meta_sr + g * 64;
    uint4 v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = *reinterpret_cast<const uint4 *>(mv + (int64_t)min(i0 + 4 * g + j, last) * p.meta_sr + c * 16);
      v[4 + j] = *reinterpret_cast<const uint4 *>(mv + (int64_t)min(i0 + 16 + 4 * g + j, last) * p.meta_sr + c * 16);
    }
    f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      s0 = Mma<E>::run(*reinterpret_cast<const uint4 *>(pk0 + s * 16), qb[s], s0);
      s1 = Mma<E>::run(*reinterpret_cast<const uint4 *>(pk1 + s * 16), qb[s], s1);
    }
    float sc[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
    bool vis[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int key = i0 + ((j >> 2) << 4) + 4 * g + (j & 3);
      vis[j] = key < p.meta_len;
      float x = sc[j] * p.meta_k_mult;
      // soft cap / ALiBi: the meta rows' distance is that of the stacked second attention of the reference
      if (p.opt.on) x = adjust_score(p.opt, x, my_slope, -fabsf((float)(p.meta_bias_off + (int)r - key)));
      sc[j] = vis[j] ? x : kNegInf;
    }
    float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m, mx * p.scale_log2);
    const float m_safe = (m_new == kNegInf) ? 0.f : m_new;
    const float alpha = fast_exp2(m - m_safe);
    m = m_new;
    float psum = 0.f, pv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = fast_exp2(fmaf(sc[j], p.scale_log2, -m_safe));
      psum += e;
      pv[j] = vis[j] ? e * p.meta_v_mult : 0.f;
    }
    l = fmaf(l, alpha, psum);
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) acc[mt] *= alpha;
    const uint4 pb = make_uint4(Mma<E>::pack(pv[0], pv[1]), Mma<E>::pack(pv[2], pv[3]),
                                Mma<E>::pack(pv[4], pv[5]), Mma<E>::pack(pv[6], pv[7]));
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) acc[mt] = Mma<E>::run(v_transposed(v, mt), pb, acc[mt]);
  };
  if (p.meta_len > 0)
    for (int cc = split; cc < (p.meta_len + 31) >> 5; cc += p.n_split) meta_chunk(cc);

  // one chunk of loads in flight behind the one being computed and the next one's blocks being looked up; two
  // register sets, the loop written out for both so that neither is ever copied, and its end written out so that
  // nothing is read twice (the last chunk was, one of 26 at 100 rows in 5 splits)
  if (cb < ce) {
    ChunkI8 a, b;
    Where at_a, at_b;
    int ch = cb;
    locate(ch, at_a);
    locate(ch + 1, at_b);
    load_chunk(at_a, a);
    round_queries();
    constexpr std::false_type inner{};
    for (; ch + 2 < ce; ch += 2) {
      load_chunk(at_b, b);
      locate(ch + 2, at_a);
      compute_chunk(ch, a, inner);
      load_chunk(at_a, a);
      locate(ch + 3, at_b);
      compute_chunk(ch + 1, b, inner);
    }
    if (ch + 1 < ce) {
      load_chunk(at_b, b);
      quantise_fresh();
      compute_chunk(ch, a, inner);
      compute_chunk(ch + 1, b, std::true_type{});
    } else {
      quantise_fresh();
      compute_chunk(ch, a, std::true_type{});
    }
  } else {
    quantise_fresh();
  }

  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  // ---- this wavefront's result: lane (g, c < G) owns head c, dims 32g + 8i + mt --------------
  if (c < G) {
    const int hq = kvh * G + c;
    if (p.n_split == 1) {
      const float inv = l > 0.f ? p.kv_out_scale / l : 0.f;
      char *dst = p.out + (r * p.o_sr + (int64_t)hq * p.o_sh + 32 * g) * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint4 o;
        o.x = E::pack(acc[0][i] * inv, acc[1][i] * inv);
        o.y = E::pack(acc[2][i] * inv, acc[3][i] * inv);
        o.z = E::pack(acc[4][i] * inv, acc[5][i] * inv);
        o.w = E::pack(acc[6][i] * inv, acc[7][i] * inv);
        *reinterpret_cast<uint4 *>(dst + 16 * i) = o;
      }
      if (g == 0 && p.lse) p.lse[r * p.Hq + hq] = l > 0.f ? (m + log2f(l)) * kLn2 : kNegInf;
    } else {
      const int64_t part = (r * p.Hq + hq) * p.n_split + split;
      float *dst = p.ws_acc + part * 128 + 32 * g;
      const float os = p.kv_out_scale;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        reinterpret_cast<float4 *>(dst + 8 * i)[0] = make_float4(acc[0][i] * os, acc[1][i] * os, acc[2][i] * os, acc[3][i] * os);
        reinterpret_cast<float4 *>(dst + 8 * i)[1] = make_float4(acc[4][i] * os, acc[5][i] * os, acc[6][i] * os, acc[7][i] * os);
      }
      if (g == 0) {
        p.ws_ml[part * 2] = m;
        p.ws_ml[part * 2 + 1] = l;
      }
    }
  }
  if constexpr (APPEND) {
    if (fresh) {
      const int64_t blk = slot / p.block_size;
      const int off = (int)(slot - blk * p.block_size);
      const int64_t base = blk * p.kv_sb + (int64_t)off * p.kv_sr + (int64_t)kvh * p.kv_sh;
      if (c == 0) {
        uint4 *dst = reinterpret_cast<uint4 *>(const_cast<char *>(p.k) + base + 32 * g);
        dst[0] = make_uint4(nk[0].x, nk[0].y, nk[1].x, nk[1].y);
        dst[1] = make_uint4(nk[2].x, nk[2].y, nk[3].x, nk[3].y);
      }
      if (g == 0) *reinterpret_cast<uint2 *>(const_cast<char *>(p.v) + base + 8 * c) = nv;
      if (Q == SB_KV_INT8 && lane == 0) {
        const int64_t at = (blk * Hkv + kvh) * p.block_size + off;
        const_cast<float *>(p.k_scale)[at] = nks;
        const_cast<float *>(p.v_scale)[at] = nvs;
      }
    }
  }
}

}  // namespace

namespace sb_host {

// Launches the split kernel over an INT8 or fp8 cache (query dtype bf16 or fp16, group size <= 16, paged mode).
void launch_swa_decode_split_i8(int dtype, int kv_quant, int G, int Hkv, unsigned rows, unsigned n_split, hipStream_t st,
                                const sb::DecodeParams &p) {
  const int waves = Hkv < 4 ? Hkv : 4;
  const dim3 grid(rows, (unsigned)((Hkv + waves - 1) / waves), n_split), block(64 * waves);
  const bool append = p.new_k != nullptr;
#define SB_I8(E, Q)                                                                                                  \
  do {                                                                                                               \
    if (append) hipLaunchKernelGGL((swa_decode_split_i8_kernel<E, Q, true>), grid, block, 0, st, p, G, Hkv);         \
    else hipLaunchKernelGGL((swa_decode_split_i8_kernel<E, Q, false>), grid, block, 0, st, p, G, Hkv);               \
  } while (0)
  if (kv_quant == SB_KV_INT8) {
    if (dtype == SB_BF16) SB_I8(sb::BF16, SB_KV_INT8);
    else SB_I8(sb::F16, SB_KV_INT8);
  } else {
    if (dtype == SB_BF16) SB_I8(sb::BF16, SB_KV_FP8);
    else SB_I8(sb::F16, SB_KV_FP8);
  }
#undef SB_I8
}

}  // namespace sb_host
