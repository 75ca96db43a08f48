// pkv_append.hip -- append-and-quantize, reference-format gather and page copy.
//
// append: one wave per (sequence, new token, KV head) quantizes the K and V
// rows group-wise with the reference quantizer's arithmetic
// (src/mlx_one/engine/paged.py:30-40, restated):
//   bias  = f16(min(group))                         f32 -> f16, round to nearest even
//   scale = f16(max(f32(max - f32(bias)) / (2^b - 1), 1e-6))
//   code  = clamp(rint((x - f32(bias)) / f32(scale)), 0, 2^b - 1)
// with IEEE-correct f32 division and half-to-even rint, then scatters the
// codes and the (scale, bias) word into the MFMA-ordered page format of
// pkv_format.h.  Float pages store the input bits unchanged.
#include "pkv_launch.h"
#include "pkv_token.h"

namespace pkv {


template <int DP, int BITS>
__global__ __launch_bounds__(256) void append_kernel(const AppendArgs a) {
  constexpr int EPL = DP / 64;
  __shared__ uint8_t s_codes[4][2][DP];
  __shared__ uint32_t s_meta[4][2][8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const Geo &g = a.g;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  const int64_t items = (int64_t)a.batch * a.tokens * g.hk;
  if (item >= items) return;
  const int kh = (int)(item % g.hk);
  const int t = (int)((item / g.hk) % a.tokens);
  const int b = (int)(item / ((int64_t)g.hk * a.tokens));
  // The new rows first: every (sequence, token, KV head) row of the inputs
  // exists, and they do not depend on the position and page lookups below,
  // so both requests are in flight together.
  const int64_t row = (((int64_t)b * g.hk + kh) * a.tokens + t) * g.dim;
  const uint16_t *src[2] = {a.keys + row, a.values + row};
  uint16_t raw[2][EPL];
#pragma unroll
  for (int side = 0; side < 2; ++side)
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int d = lane * EPL + i;
      raw[side][i] = d < g.dim ? src[side][d] : (uint16_t)0;
    }
  const int width = a.widths ? a.widths[b] : a.tokens;
  // start position: given, or the sequence's length after the append less the new tokens
  const int start = a.start_pos ? a.start_pos[b] : a.lens_after[b] - a.tokens;
  if (a.new_lens && t == 0 && kh == 0 && lane == 0) a.new_lens[b] = start + width;
  if (t >= width) return;
  const int pos = start + t;
  if (pos < 0 || pos / g.page >= a.max_pages) return;
  const int page = a.table[(int64_t)b * a.max_pages + pos / g.page];
  if (page < 0 || page >= a.num_pages) return;
  const int slot = pos % g.page, tt = slot % PKV_TILE;
  uint8_t *head = a.pool + (int64_t)page * g.page_bytes + (int64_t)kh * g.head_bytes;
  const int64_t tile = (int64_t)(slot / PKV_TILE) * g.tile_bytes;
  uint8_t *ktile = head + tile, *vtile = head + g.v_offset + tile;

  if (BITS == 16) {
    // float pages: scatter the input bits
    for (int side = 0; side < 2; ++side) {
#pragma unroll
      for (int i = 0; i < EPL; ++i) {
        const int d = lane * EPL + i;
        const uint16_t v = raw[side][i];
        int64_t off;
        if (side == 0) {
          const int kb = d / 32, jj = (d % 32) / 8, e = d % 8;
          off = payload_offset(tt + 16 * jj, 2 * (8 * kb + e), g.chunk);
          *(uint16_t *)(ktile + off) = v;
        } else {
          const int n = d / 16, col = d % 16, jj = tt / 4, r = tt % 4;
          off = payload_offset(col + 16 * jj, 2 * (4 * n + r), g.chunk);
          *(uint16_t *)(vtile + off) = v;
        }
      }
    }
    return;
  }

  for (int side = 0; side < 2; ++side) {
    float x[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int d = lane * EPL + i;
      x[i] = d < g.dim ? bits_to_float(raw[side][i], g.float_kind) : 0.0f;  // zero pad
    }
    quantize_row<EPL>(x, lane, g.group, BITS, s_codes[wave][side], s_meta[wave][side]);
  }
  wave_lds_sync();
  const uint8_t *kc = s_codes[wave][0], *vc = s_codes[wave][1];

  store_token<DP, BITS>(g, head, slot, kc, vc, s_meta[wave][0], s_meta[wave][1], lane);
}

// ---- append of several tokens per sequence: one wave per 16-token tile side -----
//
// The row kernel above scatters a token's codes byte by byte into the tile
// payloads (64 separate lines per V row) and spends a wave, and two row reads,
// on every padding row of a ragged batch.  With several tokens per sequence
// the unit here is one side (K or V) of a page tile of one (sequence, KV
// head): lane (t, jj) holds the elements d = 32*kb + 8*jj + e of token t --
// 16-byte loads, and, once quantized, exactly the lane's share of the K
// payload (16-byte stores).  V is quantized the same way and turned to its
// column order through LDS.  HBM-bound for long chunks: 16 sequences x 1,024
// tokens x 8 heads x 128 to int8 (103 MB) 106 -> 25.5 us (4.0 TB/s), 4-bit
// 101 -> 23 us, f16 pages 94 -> 29 us; 36 sequences padded to 512 tokens, 32
// of them one token wide, 48 -> 12.6 us.
// The codes are the row kernel's bit for bit (codes8, pkv_token.h); a wave that
// meets infinities, NaN or a range past f16 does the row kernel's operations.

// Quantize the lane's share of its token's row: meta words of every storage
// group and the codes, 8 per kb, as two words of four bytes.  The whole wave
// calls.
template <int DP, int G, int BITS, int FK>
__device__ __forceinline__ void quantize_share(const u4 (&raw)[DP / 32], uint32_t (&meta)[DP / G],
                                               uint32_t (&codes)[DP / 16]) {
  constexpr int NG = DP / G, KPG = G / 32;
  const float levels = (float)((1 << BITS) - 1);
  float lo[NG], hi[NG], bias[NG], scale[NG];
  auto affine = [&](int gi) __attribute__((always_inline)) {
    const uint16_t b16 = f32_to_f16_bits(lo[gi]);
    bias[gi] = f16_bits_to_f32(b16);
    const uint16_t s16 = f32_to_f16_bits(fmaxf(__fdiv_rn(hi[gi] - bias[gi], levels), 1e-6f));
    scale[gi] = f16_bits_to_f32(s16);
    meta[gi] = (uint32_t)s16 | ((uint32_t)b16 << 16);
  };
  // min and max by the NaN-propagating three-input forms (half the operations
  // of fminf / fmaxf, and no canonicalisation)
  bool odd = false;
#pragma unroll
  for (int gi = 0; gi < NG; ++gi) {
    float l = 0.0f, h = 0.0f;
#pragma unroll
    for (int k = 0; k < KPG; ++k) {
      float x[8];
      unpack8<FK>(raw[gi * KPG + k], x);
      if (k == 0) l = h = x[0];
      minmax8(x, l, h);
    }
    l = __builtin_elementwise_minimum(l, __shfl_xor(l, 16, 64));
    h = __builtin_elementwise_maximum(h, __shfl_xor(h, 16, 64));
    lo[gi] = __builtin_elementwise_minimum(l, __shfl_xor(l, 32, 64));
    hi[gi] = __builtin_elementwise_maximum(h, __shfl_xor(h, 32, 64));
    affine(gi);
    odd |= !(fabsf(bias[gi]) < INFINITY && scale[gi] < INFINITY && hi[gi] - lo[gi] < INFINITY);
  }
  if (__any(odd)) {  // rare: infinities, NaN, or a range past f16: the row kernel's operations
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
      float l = 0.0f, h = 0.0f;
#pragma unroll
      for (int k = 0; k < KPG; ++k) {
        float x[8];
        unpack8<FK>(raw[gi * KPG + k], x);
        if (k == 0) l = h = x[0];
#pragma unroll
        for (int e = 0; e < 8; ++e) { l = fminf(l, x[e]); h = fmaxf(h, x[e]); }
      }
      lo[gi] = xor32_min(xor16_min(l));
      hi[gi] = xor32_max(xor16_max(h));
      affine(gi);
    }
#pragma unroll
    for (int kb = 0; kb < DP / 32; ++kb) {
      float x[8];
      unpack8<FK>(raw[kb], x);
      codes8_div(x, bias[kb / KPG], scale[kb / KPG], levels, codes[2 * kb], codes[2 * kb + 1]);
    }
    return;
  }
  float rcp[NG];
#pragma unroll
  for (int gi = 0; gi < NG; ++gi) rcp[gi] = __fdiv_rn(1.0f, scale[gi]);
#pragma unroll
  for (int kb = 0; kb < DP / 32; ++kb) {
    const int gi = kb / KPG;
    float x[8];
    unpack8<FK>(raw[kb], x);
    codes8(x, bias[gi], scale[gi], rcp[gi], levels, codes[2 * kb], codes[2 * kb + 1]);
  }
}

template <int DP, int G, int BITS>
__global__ __launch_bounds__(256) void append_tiles_kernel(const AppendArgs a, int tiles, bool vec) {
  constexpr int KB = DP / 32, NB = DP / 16;
  constexpr int ROWW = BITS == 16 ? DP / 2 + 4 : DP / 4 + 4;  // V rows in LDS, words
  __shared__ __attribute__((aligned(16))) uint32_t s_v[4][16 * ROWW];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Geo &g = a.g;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  if (item >= (int64_t)a.batch * g.hk * tiles * 2) return;
  // neighbouring waves take neighbouring tiles of one side
  const int ti = (int)(item % tiles);
  const int side = (int)((item / tiles) & 1);
  const int kh = (int)((item / tiles / 2) % g.hk);
  const int b = (int)(item / ((int64_t)tiles * 2 * g.hk));
  const int width = min(a.widths ? a.widths[b] : a.tokens, a.tokens);
  const int start = a.start_pos ? a.start_pos[b] : a.lens_after[b] - a.tokens;
  if (a.new_lens && ti == 0 && kh == 0 && side == 0 && lane == 0)
    a.new_lens[b] = start + (a.widths ? a.widths[b] : a.tokens);
  // the ti-th tile the new positions [max(start, 0), start + width) touch
  const int tile = max(start, 0) / PKV_TILE + ti;
  const int pos0 = tile * PKV_TILE;
  if (width <= 0 || pos0 >= start + width || pos0 / g.page >= a.max_pages) return;
  const int page = a.table[(int64_t)b * a.max_pages + pos0 / g.page];  // read beside the rows
  const int t = lane & 15, jj = lane >> 4;
  const int tok = pos0 + t - start;  // the lane's token among the new ones
  const bool mine = tok >= 0 && tok < width;
  const int64_t row = (((int64_t)b * g.hk + kh) * a.tokens + (mine ? tok : 0)) * g.dim;
  const uint16_t *src = (side ? a.values : a.keys) + row;
  u4 raw[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int d0 = 32 * kb + 8 * jj;
    u4 v = {0, 0, 0, 0};  // zero pad past the head dim
    if (vec) {
      if (mine && d0 < g.dim) v = *(const u4 *)(src + d0);
    } else if (mine) {
      uint32_t e8[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) e8[e] = d0 + e < g.dim ? src[d0 + e] : (uint16_t)0;
      v = u4{e8[0] | (e8[1] << 16), e8[2] | (e8[3] << 16), e8[4] | (e8[5] << 16), e8[6] | (e8[7] << 16)};
    }
    raw[kb] = v;
  }
  if (page < 0 || page >= a.num_pages) return;
  uint8_t *head = a.pool + (int64_t)page * g.page_bytes + (int64_t)kh * g.head_bytes;
  const int slot0 = pos0 % g.page;
  const int64_t toff = (int64_t)(slot0 / PKV_TILE) * g.tile_bytes;
  uint8_t *ktile = head + toff, *vtile = head + g.v_offset + toff;
  uint32_t *vrow = s_v[wave] + t * ROWW;
  if constexpr (BITS == 16) {
    if (side == 0) {
      if (mine) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) *(u4 *)(ktile + kb * 1024 + lane * 16) = raw[kb];
      }
      return;
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) *(u4 *)(vrow + 16 * kb + 4 * jj) = raw[kb];
  } else {
    constexpr int NG = DP / G;
    uint32_t meta[NG], codes[2 * KB];
    if (g.float_kind == 0) quantize_share<DP, G, BITS, 0>(raw, meta, codes);
    else quantize_share<DP, G, BITS, 1>(raw, meta, codes);
    if (mine) {
      // the token's (scale, bias) words: group gi by lane jj = gi % 4
      uint32_t *m = (uint32_t *)(head + (side ? g.vmeta_offset : g.kmeta_offset)) + (slot0 + t) * NG;
#pragma unroll
      for (int gi = 0; gi < NG; ++gi)
        if (gi % 4 == jj) m[gi] = meta[gi];
    }
    if (side == 0) {
      // K: the lane's payload, 16-byte chunks (8 bytes where it holds no more)
      constexpr int LW = DP * BITS / 128;
      uint32_t w[LW];
#pragma unroll
      for (int i = 0; i < LW; ++i) {
        if constexpr (BITS == 8) {
          w[i] = codes[i];
        } else {
          // nibble (e odd ? 4 : 0) + e / 2 holds element e
          const uint32_t c0 = codes[2 * i], c1 = codes[2 * i + 1];
          const uint32_t ev = (c0 & 15u) | ((c0 >> 12) & 0xF0u) | ((c1 & 15u) << 8) | ((c1 >> 4) & 0xF000u);
          const uint32_t od = ((c0 >> 8) & 15u) | ((c0 >> 20) & 0xF0u) | (c1 & 0xF00u) | ((c1 >> 12) & 0xF000u);
          w[i] = ev | (od << 16);
        }
      }
      if (mine) {
        if constexpr (LW >= 4) {
#pragma unroll
          for (int c = 0; c < LW / 4; ++c)
            *(u4 *)(ktile + c * 1024 + lane * 16) = u4{w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]};
        } else {
          *(u2 *)(ktile + lane * 8) = u2{w[0], w[1]};
        }
      }
      return;
    }
    // codes of d = 32*kb + 8*jj + 0..7: words 8*kb + 2*jj, + 1 of the row
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) *(u2 *)(vrow + 8 * kb + 2 * jj) = u2{codes[2 * kb], codes[2 * kb + 1]};
  }
  wave_lds_sync();
  // V: lane (col, jj) takes column d = 16*n + col of tokens 4*jj .. 4*jj + 3
  const int col = t;
  const int first = pos0 + 4 * jj - start;  // token 4*jj of the tile, among the new ones
  const bool all4 = first >= 0 && first + 3 < width;
  const uint32_t *vcol = s_v[wave] + 4 * jj * ROWW;
  if constexpr (BITS == 16) {
    const uint32_t sel = (col & 1) ? 0x07060302u : 0x05040100u;
    uint32_t w[2 * NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      uint32_t r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = vcol[i * ROWW + 8 * n + (col >> 1)];
      w[2 * n] = __builtin_amdgcn_perm(r[1], r[0], sel);
      w[2 * n + 1] = __builtin_amdgcn_perm(r[3], r[2], sel);
    }
    if (all4) {
#pragma unroll
      for (int c = 0; c < NB / 2; ++c)
        *(u4 *)(vtile + c * 1024 + lane * 16) = u4{w[4 * c], w[4 * c + 1], w[4 * c + 2], w[4 * c + 3]};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (first + i < 0 || first + i >= width) continue;
#pragma unroll
        for (int n = 0; n < NB; ++n)
          *(uint16_t *)(vtile + (n / 2) * 1024 + lane * 16 + 8 * (n & 1) + 2 * i) =
              (uint16_t)(w[2 * n + i / 2] >> (16 * (i & 1)));
      }
    }
  } else {
    // a word's bytes: tokens 0..3 of a column (8-bit), or 0, 2, 1, 3 with the
    // odd block's codes in the high nibbles (4-bit)
    const uint32_t cb = col & 3;
    const uint32_t sel = cb | ((4 + cb) << 8) | 0x0C0C0000u;  // bytes cb of both sources
    uint32_t w[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      uint32_t r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = vcol[i * ROWW + 4 * n + (col >> 2)];
      const uint32_t p01 = __builtin_amdgcn_perm(r[BITS == 8 ? 1 : 2], r[0], sel);
      const uint32_t p23 = __builtin_amdgcn_perm(r[3], r[BITS == 8 ? 2 : 1], sel);
      w[n] = p01 | (p23 << 16);
    }
    constexpr int LW = DP * BITS / 128;
    uint32_t o[LW];
#pragma unroll
    for (int i = 0; i < LW; ++i) o[i] = BITS == 8 ? w[i] : w[2 * i] | (w[2 * i + 1] << 4);
    if (all4) {
      if constexpr (LW >= 4) {
#pragma unroll
        for (int c = 0; c < LW / 4; ++c)
          *(u4 *)(vtile + c * 1024 + lane * 16) = u4{o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]};
      } else {
        *(u2 *)(vtile + lane * 8) = u2{o[0], o[1]};
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (first + i < 0 || first + i >= width) continue;
        const int byte = BITS == 8 ? i : v4_byte(i);
#pragma unroll
        for (int x = 0; x < LW; ++x)
          vtile[payload_offset(lane, 4 * x + byte, LW >= 4 ? 16 : 8)] = (uint8_t)(o[x] >> (8 * byte));
      }
    }
  }
}

// ---- gather to the reference format ---------------------------------------


__device__ __forceinline__ int read_code(const uint8_t *tile, int side, int bits, int tt, int d,
                                         int chunk) {
  if (side == 0) {
    const int kb = d / 32, jj = (d % 32) / 8, e = d % 8, lane = tt + 16 * jj;
    if (bits == 8) return tile[payload_offset(lane, 8 * kb + e, chunk)];
    const int nib = k4_nibble(e);
    return (tile[payload_offset(lane, 4 * kb + nib / 2, chunk)] >> (4 * (nib & 1))) & 15;
  }
  const int n = d / 16, col = d % 16, jj = tt / 4, r = tt % 4, lane = col + 16 * jj;
  if (bits == 8) return tile[payload_offset(lane, 4 * n + r, chunk)];
  return (tile[payload_offset(lane, 4 * (n / 2) + v4_byte(r), chunk)] >> (4 * (n % 2))) & 15;
}

// One thread per (page, head, token, output byte); grid-stride.
__global__ __launch_bounds__(256) void gather_kernel(const GatherArgs a) {
  const Geo &g = a.g;
  const bool quant = g.bits != 16;
  const int per_row = quant ? a.dq : g.dim;  // codes bytes or float elements per row
  const int64_t rows = (int64_t)a.count * g.hk * g.page;
  const int64_t total = rows * per_row;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % per_row);
    const int64_t rowi = i / per_row;
    const int tok = (int)(rowi % g.page);
    const int kh = (int)((rowi / g.page) % g.hk);
    const int pi = (int)(rowi / ((int64_t)g.page * g.hk));
    const int page = a.ids[pi];
    if (page < 0 || page >= a.num_pages) continue;
    const uint8_t *head = a.pool + (int64_t)page * g.page_bytes + (int64_t)kh * g.head_bytes;
    const int64_t tile = (int64_t)(tok / PKV_TILE) * g.tile_bytes;
    const int tt = tok % PKV_TILE;
    for (int side = 0; side < 2; ++side) {
      const uint8_t *payload = head + (side ? g.v_offset : 0) + tile;
      if (!quant) {
        const int d = x;
        int64_t off;
        if (side == 0) {
          off = payload_offset(tt + 16 * ((d % 32) / 8), 2 * (8 * (d / 32) + d % 8), g.chunk);
        } else {
          off = payload_offset(d % 16 + 16 * (tt / 4), 2 * (4 * (d / 16) + tt % 4), g.chunk);
        }
        uint16_t *dst = (uint16_t *)(side ? a.vc : a.kc);
        dst[rowi * g.dim + d] = *(const uint16_t *)(payload + off);
        continue;
      }
      uint8_t out;
      if (g.bits == 8) {
        out = (uint8_t)read_code(payload, side, 8, tt, x, g.chunk);
      } else {
        out = (uint8_t)(read_code(payload, side, 4, tt, 2 * x, g.chunk) |
                        (read_code(payload, side, 4, tt, 2 * x + 1, g.chunk) << 4));
      }
      (side ? a.vc : a.kc)[rowi * a.dq + x] = out;
      if (x < a.ngr) {
        const uint32_t word = *(const uint32_t *)(head + (side ? g.vmeta_offset : g.kmeta_offset) +
                                                  ((int64_t)tok * g.ng + x) * 4);
        (side ? a.vs : a.ks)[rowi * a.ngr + x] = (uint16_t)(word & 0xFFFFu);
        (side ? a.vb : a.kb)[rowi * a.ngr + x] = (uint16_t)(word >> 16);
      }
    }
  }
}

// Rows of whole 16-byte units at aligned addresses: one wave per side (K or V) of
// a tile.  The tile payload is read as the attention reads it (16-byte chunks),
// turned to token rows through LDS (V by byte exchanges within quads of lanes
// first), and its 16 output rows, which are contiguous, leave as 1 KiB stores.
// HBM-bound: 1,024 pages of 16 tokens x 8 heads x 128 int8 (71 MB moved)
// 122 -> 13.6 us (5.2 TB/s; the general kernel moves single bytes behind 64-bit
// divisions).
template <int DP, int BITS>
__global__ __launch_bounds__(256) void gather_tiles_kernel(const GatherArgs a, int row_bytes, int64_t items) {
  constexpr int LB = DP * BITS / 32, LW = LB / 4, NB = DP / 16, KB = DP / 32;
  constexpr int ROWB = DP * BITS / 8;  // stored bytes per row
  __shared__ __attribute__((aligned(16))) uint8_t s_rows[4][16 * (ROWB + 16)];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Geo &g = a.g;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  if (item >= items) return;
  const int side = (int)(item & 1);
  const int tpp = g.page / PKV_TILE;
  const int64_t tile = item >> 1;  // (page index, KV head, tile in the page)
  const int ti = (int)(tile % tpp);
  const int kh = (int)((tile / tpp) % g.hk);
  const int pi = (int)(tile / ((int64_t)tpp * g.hk));
  const int page = a.ids[pi];
  if (page < 0 || page >= a.num_pages) return;
  const uint8_t *head = a.pool + (int64_t)page * g.page_bytes + (int64_t)kh * g.head_bytes;
  const uint8_t *src = head + (side ? g.v_offset : 0) + (int64_t)ti * g.tile_bytes;
  uint32_t w[LW];
  if constexpr (LW >= 4) {
#pragma unroll
    for (int c = 0; c < LW / 4; ++c) {
      const u4 v = *(const u4 *)(src + c * 1024 + lane * 16);
      w[4 * c] = v.x; w[4 * c + 1] = v.y; w[4 * c + 2] = v.z; w[4 * c + 3] = v.w;
    }
  } else {
    const u2 v = *(const u2 *)(src + lane * 8);
    w[0] = v.x; w[1] = v.y;
  }
  const int t = lane & 15, jj = lane >> 4;
  uint8_t *rows = s_rows[wave];
  const int64_t row0 = (((int64_t)pi * g.hk + kh) * tpp + ti) * PKV_TILE;  // output row of token 0
  if constexpr (BITS != 16) {
    // the tile's (scale, bias) words, token-major
    const uint32_t *m = (const uint32_t *)(head + (side ? g.vmeta_offset : g.kmeta_offset)) + ti * PKV_TILE * g.ng;
    for (int i = lane; i < PKV_TILE * g.ng; i += 64) {
      const int tok = i / g.ng, gi = i % g.ng;
      const uint32_t word = m[i];
      if (gi < a.ngr) {
        (side ? a.vs : a.ks)[(row0 + tok) * a.ngr + gi] = (uint16_t)(word & 0xFFFFu);
        (side ? a.vb : a.kb)[(row0 + tok) * a.ngr + gi] = (uint16_t)(word >> 16);
      }
    }
  }
  constexpr int STRIDE = ROWB + 16;
  if (side == 0) {
    // lane (t, jj): elements 32*kb + 8*jj + 0..7 of token t
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      uint8_t *dst = rows + t * STRIDE + (32 * kb + 8 * jj) * BITS / 8;
      if constexpr (BITS == 8) {
        *(u2 *)dst = u2{w[2 * kb], w[2 * kb + 1]};
      } else if constexpr (BITS == 4) {
        // low half: nibbles of elements 0, 2, 4, 6; high half: 1, 3, 5, 7
        auto spread = [](uint32_t x) __attribute__((always_inline)) {
          x = (x | (x << 8)) & 0x00FF00FFu;
          return (x | (x << 4)) & 0x0F0F0F0Fu;
        };
        *(uint32_t *)dst = spread(w[kb] & 0xFFFFu) | (spread(w[kb] >> 16) << 4);
      } else {
        *(u4 *)dst = u4{w[4 * kb], w[4 * kb + 1], w[4 * kb + 2], w[4 * kb + 3]};
      }
    }
  } else if constexpr (BITS == 16) {
    // lane (col, jj): tokens 4*jj .. 4*jj + 3 of columns 16*n + col
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *(uint16_t *)(rows + (4 * jj + r) * STRIDE + 2 * (16 * n + t)) = (uint16_t)(w[2 * n + r / 2] >> (16 * (r & 1)));
  } else {
    // 4x4 byte exchange in each quad of lanes: lane i of the quad takes byte i of
    // all four, the codes of token 4*jj + i (4-bit: byte v4_byte(i)) in four
    // neighbouring columns
    const uint32_t i = lane & 3;
    const uint32_t by = BITS == 8 ? i : (uint32_t)v4_byte((int)i);
    const uint32_t sel = by | ((4 + by) << 8) | 0x0C0C0000u;
#pragma unroll
    for (int x = 0; x < LW; ++x) {
      const int q = (int)w[x];
      const uint32_t q0 = (uint32_t)__builtin_amdgcn_mov_dpp(q, 0x00, 0xF, 0xF, false);
      const uint32_t q1 = (uint32_t)__builtin_amdgcn_mov_dpp(q, 0x55, 0xF, 0xF, false);
      const uint32_t q2 = (uint32_t)__builtin_amdgcn_mov_dpp(q, 0xAA, 0xF, 0xF, false);
      const uint32_t q3 = (uint32_t)__builtin_amdgcn_mov_dpp(q, 0xFF, 0xF, 0xF, false);
      const uint32_t v = __builtin_amdgcn_perm(q1, q0, sel) | (__builtin_amdgcn_perm(q3, q2, sel) << 16);
      uint8_t *dst = rows + (4 * jj + i) * STRIDE;
      const int c4 = t & ~3;  // the quad's first column
      if constexpr (BITS == 8) {
        *(uint32_t *)(dst + 16 * x + c4) = v;
      } else {
        // low nibbles: block 2x, high: block 2x + 1; two columns to a byte
        auto pairs = [](uint32_t y) __attribute__((always_inline)) {
          y = (y | (y >> 4)) & 0x00FF00FFu;
          return (uint16_t)(y | (y >> 8));
        };
        *(uint16_t *)(dst + (32 * x + c4) / 2) = pairs(v & 0x0F0F0F0Fu);
        *(uint16_t *)(dst + (32 * x + 16 + c4) / 2) = pairs((v >> 4) & 0x0F0F0F0Fu);
      }
    }
  }
  wave_lds_sync();
  uint8_t *out = (side ? a.vc : a.kc) + row0 * row_bytes;
  const int upr = row_bytes / 16;  // 16-byte units per output row
  for (int u = lane; u < 16 * upr; u += 64) {
    const int tok = u / upr, c = u % upr;
    *((u4 *)out + u) = *(const u4 *)(rows + tok * STRIDE + 16 * c);
  }
}

// ---- page copy ---------------------------------------------------------------

// A workgroup copies up to kCopyUnits 16-byte units of one page, four in flight
// per thread (the page and its ids once per workgroup).
constexpr int kCopyUnits = 1024;

__global__ __launch_bounds__(256) void copy_pages_kernel(uint8_t *pool, int64_t num_pages, int64_t page_bytes,
                                                         const int32_t *src, const int32_t *dst, int chunks) {
  const int pi = (int)(blockIdx.x / chunks);
  const int64_t vec = page_bytes / 16;
  const int64_t u0 = (int64_t)(blockIdx.x % chunks) * kCopyUnits + threadIdx.x;
  const int s = src[pi], d = dst[pi];
  if (s < 0 || s >= num_pages || d < 0 || d >= num_pages) return;
  const u4 *from = (const u4 *)(pool + (int64_t)s * page_bytes);
  u4 *to = (u4 *)(pool + (int64_t)d * page_bytes);
  u4 v[kCopyUnits / 256];
#pragma unroll
  for (int i = 0; i < kCopyUnits / 256; ++i)
    if (u0 + 256 * i < vec) v[i] = from[u0 + 256 * i];
#pragma unroll
  for (int i = 0; i < kCopyUnits / 256; ++i)
    if (u0 + 256 * i < vec) to[u0 + 256 * i] = v[i];
}

// ---- host launchers (called from pkv_abi.hip) ------------------------------

hipError_t launch_append(hipStream_t stream, const AppendArgs &a) {
  const int64_t items = (int64_t)a.batch * a.tokens * a.g.hk;
  if (items == 0) return hipSuccess;
  // Tiles past half a tile of new tokens: below, a wave's 32 elements per lane
  // are a longer chain than the row kernel's two (a 5-token verify step of 16
  // sequences: 32.4 us by rows, 33.7 by tiles; 16 x 12 tokens alone: 4.5 us by
  // rows, 3.8 by tiles).
  if (a.tokens > PKV_TILE / 2) {
    // tiles the new tokens of one sequence can touch (the first may be begun)
    const int tiles = (a.tokens + 2 * PKV_TILE - 2) / PKV_TILE;
    const int64_t blocks = ((int64_t)a.batch * a.g.hk * tiles * 2 + 3) / 4;
    if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
    // 16-byte row loads need rows and tensors at 16-byte addresses
    const bool vec = a.g.dim % 8 == 0 && ((uintptr_t)a.keys & 15) == 0 && ((uintptr_t)a.values & 15) == 0;
    dim3 grid((unsigned)blocks), block(256);
#define PKV_TILES(DP_, G_, BITS_)                                                                     \
  if (a.g.dp == DP_ && a.g.bits == BITS_ && (BITS_ == 16 || a.g.group == G_)) {                       \
    hipLaunchKernelGGL((append_tiles_kernel<DP_, G_, BITS_>), grid, block, 0, stream, a, tiles, vec); \
    return hipGetLastError();                                                                         \
  }
#define PKV_TILES_Q(DP_, G_) PKV_TILES(DP_, G_, 4) PKV_TILES(DP_, G_, 8)
    PKV_TILES(64, 32, 16) PKV_TILES(128, 32, 16) PKV_TILES(256, 32, 16)
    PKV_TILES_Q(64, 32) PKV_TILES_Q(64, 64)
    PKV_TILES_Q(128, 32) PKV_TILES_Q(128, 64) PKV_TILES_Q(128, 128)
    PKV_TILES_Q(256, 32) PKV_TILES_Q(256, 64) PKV_TILES_Q(256, 128)
#undef PKV_TILES_Q
#undef PKV_TILES
    return hipErrorInvalidValue;
  }
  dim3 grid((unsigned)((items + 3) / 4)), block(256);
#define PKV_APPEND(DP_, BITS_)                                                       \
  if (a.g.dp == DP_ && a.g.bits == BITS_) {                                          \
    hipLaunchKernelGGL((append_kernel<DP_, BITS_>), grid, block, 0, stream, a);      \
    return hipGetLastError();                                                        \
  }
  PKV_APPEND(64, 4) PKV_APPEND(64, 8) PKV_APPEND(64, 16)
  PKV_APPEND(128, 4) PKV_APPEND(128, 8) PKV_APPEND(128, 16)
  PKV_APPEND(256, 4) PKV_APPEND(256, 8) PKV_APPEND(256, 16)
#undef PKV_APPEND
  return hipErrorInvalidValue;
}

hipError_t launch_gather(hipStream_t stream, const GatherArgs &a) {
  const int per_row = a.g.bits != 16 ? a.dq : a.g.dim;
  const int64_t total = (int64_t)a.count * a.g.hk * a.g.page * per_row;
  if (total == 0) return hipSuccess;
  // by tiles where an output row is whole 16-byte units at aligned addresses
  const int row_bytes = a.g.bits != 16 ? a.dq : 2 * a.g.dim;
  const int64_t items = (int64_t)a.count * a.g.hk * (a.g.page / PKV_TILE) * 2;
  if (row_bytes % 16 == 0 && (((uintptr_t)a.kc | (uintptr_t)a.vc) & 15) == 0 && (items + 3) / 4 <= 0x7FFFFFFF) {
    const dim3 grid((unsigned)((items + 3) / 4)), block(256);
#define PKV_GATHER(DP_, BITS_)                                                                             \
  if (a.g.dp == DP_ && a.g.bits == BITS_) {                                                                \
    hipLaunchKernelGGL((gather_tiles_kernel<DP_, BITS_>), grid, block, 0, stream, a, row_bytes, items);    \
    return hipGetLastError();                                                                              \
  }
    PKV_GATHER(64, 4) PKV_GATHER(64, 8) PKV_GATHER(64, 16)
    PKV_GATHER(128, 4) PKV_GATHER(128, 8) PKV_GATHER(128, 16)
    PKV_GATHER(256, 4) PKV_GATHER(256, 8) PKV_GATHER(256, 16)
#undef PKV_GATHER
  }
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(gather_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_copy(hipStream_t stream, uint8_t *pool, int64_t num_pages, int64_t page_bytes,
                       const int32_t *src, const int32_t *dst, int count) {
  const int64_t vec = page_bytes / 16;
  const int64_t chunks = (vec + kCopyUnits - 1) / kCopyUnits;
  if (vec == 0 || count <= 0) return hipSuccess;
  if (chunks * count > 0x7FFFFFFF) return hipErrorInvalidValue;
  hipLaunchKernelGGL(copy_pages_kernel, dim3((unsigned)(chunks * count)), dim3(256), 0, stream, pool,
                     num_pages, page_bytes, src, dst, (int)chunks);
  return hipGetLastError();
}

}  // namespace pkv
