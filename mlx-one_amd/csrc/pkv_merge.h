// pkv_merge.h -- the decode kernels' work split, and the log-sum-exp merge of
// the partials it leaves (device functions shared by the kernels that split
// and the kernels that merge).
#pragma once
#include "pkv_mfma.h"

namespace pkv {

// Tiles of a sequence: at least one, so that an empty sequence still owns a
// piece that writes its zero output.
__device__ __forceinline__ int seq_tiles(int len) {
  return len <= 0 ? 1 : (len + PKV_TILE - 1) / PKV_TILE;
}

// Work split.  Split tiles are numbered over (sequence b, KV head kh) in that
// order, T in all: each (b, kh) segment spans `lead` tiles with no data, then
// its own tiles.  Wave w of W (W <= T) owns the run [start(w), start(w+1)):
// equal runs whatever the lengths, so no wave waits on a ragged tail and each
// pays its start-up once.  A run is cut into pieces at segment boundaries; a
// run that holds lead tiles only has no piece.
struct Split {
  int T, W, q, r;  // T tiles over W waves: the first r runs have q + 1 tiles, the rest q
  __device__ __forceinline__ void init(int t, int w) {
    T = t; W = w; q = t / w; r = t - q * w;
  }
  __device__ __forceinline__ int start(int w) const { return w * q + min(w, r); }
  // the wave whose run holds tile g
  __device__ __forceinline__ int wave_of(int g) const {
    const int big = r * (q + 1);
    return g < big ? g / (q + 1) : r + (g - big) / q;
  }
};

// Partial slots: the first piece of wave w's run goes to slot 2w, a later
// (its last) one to 2w+1; pieces in between cover whole segments and write
// the output directly.  A segment starting at split tile sv has its tiles at
// [s0, s1) (s0 = sv + lead); its pieces are those of waves wa .. wa+n-1, and
// wave wa's piece is its first one unless its run started before sv.
struct SegPieces {
  int n, wa, slot0;
  __device__ __forceinline__ int slot(int i) const { return i == 0 ? slot0 : 2 * (wa + i); }
};

__device__ __forceinline__ SegPieces seg_pieces(const Split &sp, int sv, int s0, int s1) {
  SegPieces p;
  p.wa = sp.wave_of(s0);
  p.n = sp.wave_of(s1 - 1) - p.wa + 1;
  p.slot0 = sp.start(p.wa) < sv ? 2 * p.wa + 1 : 2 * p.wa;
  return p;
}

// Tiles the split gives sequence idx (< batch): seq_tiles, or none for a
// sequence of a mixed batch that the prefill kernel serves (its width is past
// narrow_q, the query rows this launch covers).  Served sequences have at
// least one tile, so "served" is "tiles > 0", and only they are charged lead
// tiles.
__device__ __forceinline__ int split_tiles(const int32_t *lens, const int32_t *widths, int narrow_lo,
                                           int narrow_q, int idx) {
  if (narrow_q > 0 && (widths[idx] > narrow_q || widths[idx] <= narrow_lo)) return 0;
  return seq_tiles(lens[idx]);
}

// Runs of a launch over T split tiles: `runs`, or as few as leave each 2^least tiles.
__device__ __forceinline__ int split_runs(int runs, int least, int T) {
  return min(runs, ((T - 1) >> least) + 1);
}

// The lead tiles a launch's split charges ahead of each segment: `lead`, or
// none when the lead-free split's equal runs already end on segment
// boundaries (every sequence's tile count a multiple of the run length), so
// that no run crosses one.  nt0: the lane's tile count in the first
// 64-sequence chunk; t0: the lead-free tile total over all segments.
__device__ __forceinline__ int charged_lead(const int32_t *lens, const int32_t *widths, int narrow_lo,
                                            int narrow_q, int batch, int waves, int least, int lead, int nt0,
                                            int t0, int lane) {
  if (lead == 0 || t0 == 0) return 0;
  const int w0 = split_runs(waves, least, t0);
  if (t0 % w0) return lead;
  const int q0 = t0 / w0;
  bool off = lane < batch && nt0 % q0 != 0;
  for (int c0 = 64; c0 < batch; c0 += 64) {
    const int idx = c0 + lane;
    off |= idx < batch && split_tiles(lens, widths, narrow_lo, narrow_q, idx) % q0 != 0;
  }
  return __any(off) ? lead : 0;
}

// Log-sum-exp merge of partition partials (paged_attention.py:191-204, in
// the exp2 domain): one NW-wave workgroup (1, 2 or 4 waves, as many as a
// segment's pieces need at 16 per wave) per (segment, query
// row) of a segment split over several waves' runs; whole segments were
// written by the attention kernel.  Every wave finds M = max m and
// S = sum l 2^(m - M) over the pieces (lanes stride the pieces); wave w
// weighs pieces w, w+NW, ..., whose partial rows (lanes stride the DP
// columns, up to 16 in flight) it requests before that pass, and the NW sums
// meet in LDS.  Up to 16*NW pieces the merge is one memory round trip.
template <int DP, int NW>
__device__ __forceinline__ void merge_unit(const MergeArgs &a, int unit) {
  constexpr int PER = DP / 64 > 0 ? DP / 64 : 1;  // output columns per lane
  constexpr int KW = 16;                          // pieces per wave in flight
  __shared__ float s_acc[NW > 1 ? NW - 1 : 1][64 * PER];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = unit % a.rows, seg = unit / a.rows;
  const int b = seg / a.hk, kh = seg % a.hk;
  // (a mixed batch's launch holds units of sequences its part does not serve)
  if (a.narrow_q > 0 && split_tiles(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, b) == 0) return;
  // tiles (and served sequences) before sequence b, and the launch's split
  // (as the attention kernel made it)
  int pre = 0, spre = 0, tiles = 0, served = 0, nt0 = 0;
  for (int c0 = 0; c0 < a.batch; c0 += 64) {
    const int idx = c0 + lane;
    const int nt = idx < a.batch ? split_tiles(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, idx) : 0;
    if (c0 == 0) nt0 = nt;
    tiles += wave_sum(nt);
    served += wave_sum(nt > 0 ? 1 : 0);
    pre += wave_sum(idx < b ? nt : 0);
    spre += wave_sum(idx < b && nt > 0 ? 1 : 0);
  }
  const int ntb = split_tiles(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, b);
  const int t0 = __builtin_amdgcn_readfirstlane(tiles) * a.hk;
  const int lead = charged_lead(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, a.batch, a.waves, a.least, a.lead, nt0,
                                t0, lane);
  const int T = t0 + __builtin_amdgcn_readfirstlane(served) * a.hk * lead;
  const int sv = (__builtin_amdgcn_readfirstlane(pre) + __builtin_amdgcn_readfirstlane(spre) * lead) *
                     a.hk + kh * (ntb + lead);
  Split sp;
  sp.init(T, split_runs(a.waves, a.least, T));
  const SegPieces pc = seg_pieces(sp, sv, sv + lead, sv + lead + ntb);
  if (pc.n < 2) return;  // the same for every wave of the workgroup

  // this wave's partial rows of pieces k0 + wv + NW*i, all requested at once
  float x[KW][PER];
  auto request = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KW; ++i) {
      const int k = k0 + wv + NW * i;
#pragma unroll
      for (int e = 0; e < PER; ++e) x[i][e] = 0.0f;
      if (k < pc.n) {
        const float *src = a.part_acc + ((int64_t)pc.slot(k) * a.rows + row) * DP + lane * PER;
        if constexpr (PER == 4) {
          const f4 v = *(const f4 *)src;
          x[i][0] = v[0]; x[i][1] = v[1]; x[i][2] = v[2]; x[i][3] = v[3];
        } else if constexpr (PER == 2) {
          const float2 v = *(const float2 *)src;
          x[i][0] = v.x; x[i][1] = v.y;
        } else {
          x[i][0] = src[0];
        }
      }
    }
  };
  // The first rows go out before the (m, l) pass: both in one memory round trip.
  request(0);

  // M = max m, S = sum l 2^(m - M) over the pieces (lanes stride the pieces);
  // lane l keeps piece l's (m, l)
  float mx = -INFINITY, sm = 0.0f;
  float2 mine = make_float2(-INFINITY, 0.0f);
  for (int k0 = 0; k0 < pc.n; k0 += 64) {
    const int k = k0 + lane;
    if (k < pc.n) {
      const float2 ml = *(const float2 *)(a.part_ml + ((int64_t)pc.slot(k) * a.rows + row) * 2);
      if (k0 == 0) mine = ml;
      if (ml.y > 0.0f) {  // a piece with no visible token holds l = 0
        const float nm = fmaxf(mx, ml.x);
        sm = sm * __builtin_amdgcn_exp2f(mx - nm) + ml.y * __builtin_amdgcn_exp2f(ml.x - nm);
        mx = nm;
      }
    }
  }
  // combine across lanes: within 16-lane rows by DPP exchanges (the
  // combination is symmetric, so both lanes of a pair hold the same bits),
  // then the four rows' results, read as uniform values, in row order
  auto combine = [&](float om, float os) __attribute__((always_inline)) {
    const float nm = fmaxf(mx, om);
    sm = nm == -INFINITY ? 0.0f
                         : sm * __builtin_amdgcn_exp2f(mx - nm) + os * __builtin_amdgcn_exp2f(om - nm);
    mx = nm;
  };
  combine(row_xchg<0xB1>(mx), row_xchg<0xB1>(sm));
  combine(row_xchg<0x4E>(mx), row_xchg<0x4E>(sm));
  combine(row_xchg<0x141>(mx), row_xchg<0x141>(sm));
  combine(row_xchg<0x140>(mx), row_xchg<0x140>(sm));
  {
    float rm[4], rs[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      rm[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx), 16 * r));
      rs[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sm), 16 * r));
    }
    mx = rm[0];
    sm = rs[0];
#pragma unroll
    for (int r = 1; r < 4; ++r) combine(rm[r], rs[r]);
  }
  const float inv = 1.0f / fmaxf(sm, 1e-20f);
  // lane l: weight 2^(m - M) / S of piece l
  const float w_first = mine.y > 0.0f ? __builtin_amdgcn_exp2f(mine.x - mx) * inv : 0.0f;
  float acc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) acc[i] = 0.0f;
  for (int k0 = 0; k0 < pc.n; k0 += NW * KW) {
    if (k0 > 0) request(k0);
    // lane l: weight of piece k0 + l (pieces below 64 from the pass above)
    const bool held = k0 + NW * KW <= 64;
    float wl = w_first;
    if (!held) {
      wl = 0.0f;
      const int k = k0 + lane;
      if (k < pc.n) {
        const float2 ml = *(const float2 *)(a.part_ml + ((int64_t)pc.slot(k) * a.rows + row) * 2);
        wl = ml.y > 0.0f ? __builtin_amdgcn_exp2f(ml.x - mx) * inv : 0.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < KW; ++i) {
      const int src_lane = held ? k0 + wv + NW * i : wv + NW * i;
      const float wk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl), src_lane));
#pragma unroll
      for (int e = 0; e < PER; ++e) acc[e] += wk * x[i][e];
    }
  }
  if (wv > 0) {
#pragma unroll
    for (int e = 0; e < PER; ++e) s_acc[wv - 1][lane * PER + e] = acc[e];
  }
  __syncthreads();
  if (wv != 0) return;
  const int qi = row / a.gqa, h = kh * a.gqa + row % a.gqa;
  uint16_t *o = a.out + (((int64_t)b * a.heads + h) * a.nq_stride + qi) * a.dim;
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int d = lane * PER + e;
    float v = acc[e];
#pragma unroll
    for (int k = 0; k < NW - 1; ++k) v += s_acc[k][d];
    if (d < a.dim) o[d] = float_to_bits(v, a.float_kind);
  }
}

}  // namespace pkv
