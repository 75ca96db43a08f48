// pkv_quant.hip -- row quantizer / dequantizer in the reference's page format.
//
// quantize: one wave per row of `dim` values, groups of `group` along the row
// (zero padded to whole groups), the quantize_page arithmetic of
// src/mlx_one/engine/paged.py:30-40 (see pkv_append.hip); 4-bit output packs
// code[2i] | code[2i+1] << 4 (paged.py:39-40).
// dequantize: x = f32(code) * f32(scale) + f32(bias) (paged.py:44-54), float32 out.
#include "pkv_launch.h"
#include "pkv_token.h"

namespace pkv {

// Rows of a multiple of 8 elements at 16-byte addresses: a lane takes 8
// consecutive elements (one 16-byte load, one 8- or 4-byte store), G/8
// neighbouring lanes a group, so a wave covers 512 elements whatever the row
// length and reduces with DPP exchanges; each thread keeps kUnits loads in
// flight.  HBM-bound: 33.5M bf16 values to int8, G64 (103 MB) 119 -> 22 us
// (4.7 TB/s; the wave-per-row kernel below reads 2 bytes and stores 1 per
// lane).  Codes as there (codes8 and codes8_div, pkv_token.h).
template <int G, int BITS, int FK>
__global__ __launch_bounds__(256) void quantize_vec_kernel(const QuantRowsArgs a, uint32_t units_per_row,
                                                           uint32_t live_per_row) {
  constexpr int kUnits = 4;
  constexpr int LPG = G / 8;  // lanes per group
  const float levels = (float)((1 << BITS) - 1);
  const int64_t units = a.rows * units_per_row;
  const int64_t base = (int64_t)blockIdx.x * (256 * kUnits) + threadIdx.x;
  u4 raw[kUnits];
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int64_t u = base + 256 * i;
    raw[i] = u4{0, 0, 0, 0};  // zero pad past the row
    if (units_per_row == live_per_row) {
      if (u < units) raw[i] = *((const u4 *)a.values + u);
    } else if (u < units) {
      const int64_t row = u / units_per_row;
      const uint32_t c = (uint32_t)(u - row * units_per_row);
      if (c < live_per_row) raw[i] = *((const u4 *)a.values + row * live_per_row + c);
    }
  }
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int64_t u = base + 256 * i;
    float x[8];
    unpack8<FK>(raw[i], x);
    float lo = x[0], hi = x[0];
    minmax8(x, lo, hi);
    auto reduce = [&](auto mn, auto mx) __attribute__((always_inline)) {
      lo = mn(lo, row_xchg<0xB1>(lo)); hi = mx(hi, row_xchg<0xB1>(hi));
      lo = mn(lo, row_xchg<0x4E>(lo)); hi = mx(hi, row_xchg<0x4E>(hi));
      if (LPG >= 8) { lo = mn(lo, row_xchg<0x141>(lo)); hi = mx(hi, row_xchg<0x141>(hi)); }
      if (LPG >= 16) { lo = mn(lo, row_xchg<0x140>(lo)); hi = mx(hi, row_xchg<0x140>(hi)); }
    };
    float bias, scale;
    uint16_t b16, s16;
    auto affine = [&]() __attribute__((always_inline)) {
      b16 = f32_to_f16_bits(lo);
      bias = f16_bits_to_f32(b16);
      s16 = f32_to_f16_bits(fmaxf(__fdiv_rn(hi - bias, levels), 1e-6f));
      scale = f16_bits_to_f32(s16);
    };
    reduce([](float p, float q) { return __builtin_elementwise_minimum(p, q); },
           [](float p, float q) { return __builtin_elementwise_maximum(p, q); });
    affine();
    uint32_t w0, w1;
    if (__any(!(fabsf(bias) < INFINITY && scale < INFINITY && hi - lo < INFINITY))) {
      lo = INFINITY;
      hi = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) { lo = fminf(lo, x[e]); hi = fmaxf(hi, x[e]); }
      reduce([](float p, float q) { return fminf(p, q); }, [](float p, float q) { return fmaxf(p, q); });
      affine();
      codes8_div(x, bias, scale, levels, w0, w1);
    } else {
      codes8(x, bias, scale, __fdiv_rn(1.0f, scale), levels, w0, w1);
    }
    if (u >= units) continue;  // (after the exchanges: whole waves reach them)
    if constexpr (BITS == 8) {
      *((u2 *)a.codes + u) = u2{w0, w1};
    } else {
      // bytes code[2i] | code[2i+1] << 4
      w0 |= w0 >> 4;
      w1 |= w1 >> 4;
      *((uint32_t *)a.codes + u) = __builtin_amdgcn_perm(w1, w0, 0x06040200u);
    }
    if ((threadIdx.x & (LPG - 1)) == 0) {
      a.scale[u / LPG] = s16;
      a.bias[u / LPG] = b16;
    }
  }
}

__global__ __launch_bounds__(256) void quantize_rows_kernel(const QuantRowsArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= a.rows) return;
  const int padded = (a.dim + a.group - 1) / a.group * a.group;
  const int ngroups = padded / a.group;
  const int qbytes = a.bits == 4 ? padded / 2 : padded;
  const float levels = (float)((1 << a.bits) - 1);
  const uint16_t *src = a.values + row * a.dim;
  for (int gi = 0; gi < ngroups; ++gi) {
    // group elements: lane handles d = gi*group + lane + 64*i
    const int per = (a.group + 63) / 64;
    float x[2];
    float lo = INFINITY, hi = -INFINITY;
    for (int i = 0; i < per; ++i) {
      const int k = lane + 64 * i;
      const int d = gi * a.group + k;
      float v = 0.0f;
      if (k < a.group) {
        v = d < a.dim ? bits_to_float(src[d], a.float_kind) : 0.0f;
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
      }
      x[i] = v;
    }
    for (int o = 1; o < 64; o <<= 1) {
      lo = fminf(lo, __shfl_xor(lo, o, 64));
      hi = fmaxf(hi, __shfl_xor(hi, o, 64));
    }
    const uint16_t b16 = f32_to_f16_bits(lo);
    const float b = f16_bits_to_f32(b16);
    const float s = fmaxf(__fdiv_rn(hi - b, levels), 1e-6f);
    const uint16_t s16 = f32_to_f16_bits(s);
    const float sf = f16_bits_to_f32(s16);
    if (lane == 0) {
      a.scale[row * ngroups + gi] = s16;
      a.bias[row * ngroups + gi] = b16;
    }
    for (int i = 0; i < per; ++i) {
      const int k = lane + 64 * i;
      float c = rintf(__fdiv_rn(x[i] - b, sf));
      c = fminf(fmaxf(c, 0.0f), levels);
      const int code = (int)c;
      const int d = gi * a.group + k;
      if (a.bits == 8) {
        if (k < a.group) a.codes[row * qbytes + d] = (uint8_t)code;
      } else {
        const int high = __shfl_down(code, 1, 64);
        if (k < a.group && (k & 1) == 0)
          a.codes[row * qbytes + d / 2] = (uint8_t)((code & 15) | ((high & 15) << 4));
      }
    }
  }
}

__global__ __launch_bounds__(256) void dequantize_rows_kernel(const DequantRowsArgs a) {
  const int padded = (a.dim + a.group - 1) / a.group * a.group;
  const int ngroups = padded / a.group;
  const int qbytes = a.bits == 4 ? padded / 2 : padded;
  const int64_t total = a.rows * a.dim;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = i / a.dim;
    const int d = (int)(i % a.dim);
    int code;
    if (a.bits == 8) {
      code = a.codes[row * qbytes + d];
    } else {
      code = (a.codes[row * qbytes + d / 2] >> (4 * (d & 1))) & 15;
    }
    const int gi = d / a.group;
    const float s = f16_bits_to_f32(a.scale[row * ngroups + gi]);
    const float b = f16_bits_to_f32(a.bias[row * ngroups + gi]);
    a.out[i] = (float)code * s + b;
  }
}

// Rows of a multiple of 4 elements: a lane takes 4 consecutive ones (one group),
// so a wave stores 1 KiB runs; each thread keeps kUnits code loads in flight.
// HBM-bound on its float32 output: 33.5M values (170 MB) 74 -> 27 us (6.4 TB/s;
// the kernel above stores 4 bytes per lane behind two 64-bit divisions).
template <int BITS>
__global__ __launch_bounds__(256) void dequantize_vec_kernel(const DequantRowsArgs a, uint32_t units_per_row,
                                                             uint32_t units) {
  constexpr int kUnits = 4;
  const uint32_t padded = (a.dim + a.group - 1) / a.group * a.group;
  const uint32_t ngroups = padded / a.group;
  const uint32_t upg = a.group / 4;  // units per group
  const uint32_t base = blockIdx.x * (256 * kUnits) + threadIdx.x;
  uint32_t code[kUnits];
  float s[kUnits], b[kUnits];
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const uint32_t u = base + 256 * i;
    code[i] = 0;
    s[i] = b[i] = 0.0f;
    if (u < units) {
      const uint32_t row = u / units_per_row, c = u - row * units_per_row;
      const int64_t gi = (int64_t)row * ngroups + c / upg;
      if constexpr (BITS == 8) {
        code[i] = *(const uint32_t *)(a.codes + (int64_t)row * padded + 4 * c);
      } else {
        const uint32_t h = *(const uint16_t *)(a.codes + (int64_t)row * (padded / 2) + 2 * c);
        code[i] = (h & 0xFu) | ((h & 0xF0u) << 4) | ((h & 0xF00u) << 8) | ((h & 0xF000u) << 12);
      }
      s[i] = f16_bits_to_f32(a.scale[gi]);
      b[i] = f16_bits_to_f32(a.bias[gi]);
    }
  }
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const uint32_t u = base + 256 * i;
    if (u >= units) continue;
    f4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = (float)((code[i] >> (8 * e)) & 0xFFu) * s[i] + b[i];
    *((f4 *)a.out + u) = x;
  }
}

hipError_t launch_quantize_rows(hipStream_t stream, const QuantRowsArgs &a) {
  if (a.rows == 0) return hipSuccess;
  // the vector kernel's loads and stores need whole 16-byte units at aligned addresses
  const int64_t padded = ((int64_t)a.dim + a.group - 1) / a.group * a.group;
  const int64_t blocks = (a.rows * (padded / 8) + 1023) / 1024;
  if (a.dim % 8 == 0 && (((uintptr_t)a.values & 15) | ((uintptr_t)a.codes & 7)) == 0 && blocks <= 0x7FFFFFFF) {
    const uint32_t per = (uint32_t)(padded / 8), live = (uint32_t)(a.dim / 8);
#define PKV_QV(G_, BITS_, FK_)                                                                        \
  if (a.group == G_ && a.bits == BITS_ && a.float_kind == FK_) {                                      \
    hipLaunchKernelGGL((quantize_vec_kernel<G_, BITS_, FK_>), dim3((unsigned)blocks), dim3(256), 0,   \
                       stream, a, per, live);                                                         \
    return hipGetLastError();                                                                         \
  }
#define PKV_QV4(G_) PKV_QV(G_, 8, 0) PKV_QV(G_, 8, 1) PKV_QV(G_, 4, 0) PKV_QV(G_, 4, 1)
    PKV_QV4(32) PKV_QV4(64) PKV_QV4(128)
#undef PKV_QV4
#undef PKV_QV
  }
  hipLaunchKernelGGL(quantize_rows_kernel, dim3((unsigned)((a.rows + 3) / 4)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_dequantize_rows(hipStream_t stream, const DequantRowsArgs &a) {
  const int64_t total = a.rows * a.dim;
  if (total == 0) return hipSuccess;
  // four elements per lane: rows of whole units at aligned addresses, in 32-bit indices
  if (a.dim % 4 == 0 && (((uintptr_t)a.out & 15) | ((uintptr_t)a.codes & 3)) == 0 && total < (int64_t)1 << 32) {
    const uint32_t units = (uint32_t)(total / 4);
    const dim3 grid((units + 1023) / 1024), block(256);
    if (a.bits == 8)
      hipLaunchKernelGGL(dequantize_vec_kernel<8>, grid, block, 0, stream, a, (uint32_t)(a.dim / 4), units);
    else
      hipLaunchKernelGGL(dequantize_vec_kernel<4>, grid, block, 0, stream, a, (uint32_t)(a.dim / 4), units);
    return hipGetLastError();
  }
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(dequantize_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace pkv
