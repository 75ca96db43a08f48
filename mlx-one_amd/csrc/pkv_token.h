// pkv_token.h -- quantize one token's K/V rows and store them into a page
// (device functions shared by the append kernel and the fused append +
// attention kernel).
//
// The reference quantizer's arithmetic (src/mlx_one/engine/paged.py:30-40,
// restated):
//   bias  = f16(min(group))                         f32 -> f16, round to nearest even
//   scale = f16(max(f32(max - f32(bias)) / (2^b - 1), 1e-6))
//   code  = clamp(rint((x - f32(bias)) / f32(scale)), 0, 2^b - 1)
// with IEEE-correct f32 division and half-to-even rint.  The codes are then
// scattered into the MFMA-ordered page format of pkv_format.h.
#pragma once
#include "pkv_device.h"

namespace pkv {

// Quantize the wave's row (EPL elements per lane, natural order d = lane*EPL + i)
// and leave the codes in `codes[d]` (LDS) and the meta word per group in `meta`.
template <int EPL>
__device__ __forceinline__ void quantize_row(const float (&x)[EPL], int lane, int group, int bits,
                                             uint8_t *codes, uint32_t *meta) {
  float lo = x[0], hi = x[0];
#pragma unroll
  for (int i = 1; i < EPL; ++i) { lo = fminf(lo, x[i]); hi = fmaxf(hi, x[i]); }
  const int lanes_per_group = group / EPL;  // 8..128
  for (int o = 1; o < lanes_per_group && o < 64; o <<= 1) {
    lo = fminf(lo, __shfl_xor(lo, o, 64));
    hi = fmaxf(hi, __shfl_xor(hi, o, 64));
  }
  const float levels = (float)((1 << bits) - 1);
  uint16_t b16 = f32_to_f16_bits(lo);
  float b = f16_bits_to_f32(b16);
  float s = __fdiv_rn(hi - b, levels);
  s = fmaxf(s, 1e-6f);
  uint16_t s16 = f32_to_f16_bits(s);
  float sf = f16_bits_to_f32(s16);
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    float c = rintf(__fdiv_rn(x[i] - b, sf));
    c = fminf(fmaxf(c, 0.0f), levels);
    codes[lane * EPL + i] = (uint8_t)c;
  }
  if ((lane * EPL) % group == 0) meta[(lane * EPL) / group] = (uint32_t)s16 | ((uint32_t)b16 << 16);
}

// 8 float_kind elements in 16 bytes -> f32
template <int FK>
__device__ __forceinline__ void unpack8(const u4 &v, float (&x)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = bits_to_float((uint16_t)(w[i] & 0xFFFFu), FK);
    x[2 * i + 1] = bits_to_float((uint16_t)(w[i] >> 16), FK);
  }
}

// Running min and max with 8 more values, by the NaN-propagating three-input
// forms (half the operations of fminf / fmaxf, and no canonicalisation).
__device__ __forceinline__ void minmax8(const float (&x)[8], float &lo, float &hi) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    lo = __builtin_elementwise_minimum(__builtin_elementwise_minimum(x[e], x[e + 1]), lo);
    hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(x[e], x[e + 1]), hi);
  }
}

// Codes of 8 elements of one group, one byte each, as the division by the
// scale gives them.
__device__ __forceinline__ void codes8_div(const float (&x)[8], float bias, float scale, float levels,
                                           uint32_t &w0, uint32_t &w1) {
  uint32_t w[2] = {0, 0};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float c = rintf(__fdiv_rn(x[e] - bias, scale));
    c = fminf(fmaxf(c, 0.0f), levels);
    w[e / 4] |= (uint32_t)c << (8 * (e % 4));
  }
  w0 = w[0];
  w1 = w[1];
}

// The same codes where bias, scale and every x are finite, with rcp = 1 / scale
// (rounded once): the correctly rounded quotient takes three operations per
// element (Markstein: with y = RN(1/s) and q = RN(n*y), RN(q + y*(n - q*s)) is
// RN(n/s)).
__device__ __forceinline__ void codes8(const float (&x)[8], float bias, float scale, float rcp, float levels,
                                       uint32_t &w0, uint32_t &w1) {
  uint32_t c[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float n = x[e] - bias;
    float q = n * rcp;
    q = __builtin_fmaf(__builtin_fmaf(-q, scale, n), rcp, q);
    // clamped, then rounded half to even into the low bits of 1.5 * 2^23 + c
    // (the bounds are integers: rounding first gives the same code)
    c[e] = __float_as_uint(__builtin_amdgcn_fmed3f(q, 0.0f, levels) + 12582912.0f);
  }
  w0 = __builtin_amdgcn_perm(c[1], c[0], 0x0C0C0400u) | __builtin_amdgcn_perm(c[3], c[2], 0x04000C0Cu);
  w1 = __builtin_amdgcn_perm(c[5], c[4], 0x0C0C0400u) | __builtin_amdgcn_perm(c[7], c[6], 0x04000C0Cu);
}

// Make one wave's LDS writes visible to its other lanes.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Store a quantized token (codes kc/vc in natural order, meta words km/vm per
// group, all in LDS) at page slot `slot` of head block `head`: the K payload
// (lane' = tt + 16*jj owns elements d = 32*kb + 8*jj + e), the V payload
// (lane' = col + 16*jj holds V[4*jj + r][16*n + col]) and the (scale, bias)
// words.  One wave; lanes split the work.
template <int DP, int BITS>
__device__ __forceinline__ void store_token(const Geo &g, uint8_t *head, int slot, const uint8_t *kc,
                                            const uint8_t *vc, const uint32_t *km, const uint32_t *vm,
                                            int lane) {
  constexpr int EPL = DP / 64;
  const int tt = slot % PKV_TILE;
  const int64_t tile = (int64_t)(slot / PKV_TILE) * g.tile_bytes;
  uint8_t *ktile = head + tile, *vtile = head + g.v_offset + tile;
  if constexpr (BITS == 8) {
    constexpr int WPJ = DP / 16;  // dwords per jj
    if (lane < 4 * WPJ) {
      const int jj = lane / WPJ, w = lane % WPJ;
      const int d0 = 32 * (w / 2) + 8 * jj + 4 * (w % 2);
      const uint32_t word = (uint32_t)kc[d0] | ((uint32_t)kc[d0 + 1] << 8) |
                            ((uint32_t)kc[d0 + 2] << 16) | ((uint32_t)kc[d0 + 3] << 24);
      *(uint32_t *)(ktile + payload_offset(tt + 16 * jj, 4 * w, g.chunk)) = word;
    }
  } else {
    constexpr int WPJ = DP / 32;
    if (lane < 4 * WPJ) {
      const int jj = lane / WPJ, kb = lane % WPJ;
      uint32_t word = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        word |= (uint32_t)(kc[32 * kb + 8 * jj + e] & 15) << (4 * k4_nibble(e));
      *(uint32_t *)(ktile + payload_offset(tt + 16 * jj, 4 * kb, g.chunk)) = word;
    }
  }
  const int vjj = tt / 4, r = tt % 4;
  if constexpr (BITS == 8) {
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int d = lane * EPL + i, n = d / 16, col = d % 16;
      vtile[payload_offset(col + 16 * vjj, 4 * n + r, g.chunk)] = vc[d];
    }
  } else {
    // one byte per (block pair m, col): low nibble block 2m, high nibble 2m+1
    for (int idx = lane; idx < DP / 2; idx += 64) {
      const int m = idx / 16, col = idx % 16;
      const uint8_t byte = (uint8_t)((vc[32 * m + col] & 15) | ((vc[32 * m + 16 + col] & 15) << 4));
      vtile[payload_offset(col + 16 * vjj, 4 * m + v4_byte(r), g.chunk)] = byte;
    }
  }
  if (lane < g.ng) {
    *(uint32_t *)(head + g.kmeta_offset + ((int64_t)slot * g.ng + lane) * 4) = km[lane];
    *(uint32_t *)(head + g.vmeta_offset + ((int64_t)slot * g.ng + lane) * 4) = vm[lane];
  }
}

}  // namespace pkv
