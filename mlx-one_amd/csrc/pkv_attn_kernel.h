// pkv_attn_kernel.h -- paged decode / verify attention for gfx950.
//
// Semantics are the reference's (src/mlx_one/engine/paged_attention.py:62-113
// kernel, :127-206 dispatch and merge): query row (q, h) attends tokens
// t <= q_pos[q] of its sequence, KV head kh = h / (H/HK), softmax(q.k*scale).v,
// normaliser floored at 1e-20, rows q >= width give 0.
//
// Work split (stream-K).  The 16-token tiles of every (sequence, KV head)
// segment, in that order, are shared out as equal contiguous runs over a grid
// of resident waves (one 64-thread workgroup each): no wave waits on a ragged
// tail and each pays its start-up latency once.  The split counts `lead`
// extra tiles ahead of each segment for the cost of starting a piece, so a
// run that crosses into another segment holds fewer real tiles.  A wave
// processes the pieces of the segments its run crosses; all R = Q*(H/HK)
// query rows of the KV head share each K/V tile load (GQA reuse).
//
// Column slots.  The 16 columns of a 16x16 MFMA tile hold SLOTS = 16/RPS
// groups of RPS query rows; slot j of an iteration works on tile (SLOTS*it +
// j).  The slot-j query operand is zero outside its columns, so the score
// MFMAs of SLOTS tiles accumulate into one dense 16x16 tile, and every lane's
// softmax work is useful (decode at GQA 4 would otherwise leave 12 of 16
// columns empty).  Each column keeps its own online-softmax state, so the
// SLOTS columns of a row are independent sub-partitions (interleaved tiles)
// merged by log-sum-exp once per unit.
//
// Per iteration (SLOTS tiles of 16 tokens):
//   S^T[t][col] = K.Q^T   v_mfma_f32_16x16x32_f16 over the codes as f16
//                         (1024 + c, one v_perm per two codes); one
//                         accumulator per quantization group, then
//                         s = sum_g scale_g*acc_g + qsum_g*(bias_g - 1024*scale_g)
//   softmax               exp2 domain, online with lazy rescaling: a column's
//                         running max moves only when a score exceeds it by > 8
//   O^T[d][col] += V^T.P' v_mfma_f32_16x16x16_f16 with P'_g = p*scale_v[g]
//                         (V is never dequantized); bias_v enters as
//                         sum p*bias_v, the 1024 offset as 1024*sum P'.
// O is kept transposed (d in rows, columns in lanes): rescaling a column
// touches only the lane's own registers.
//
// Loads.  The page format stores a lane's share of a tile where its MFMA
// operand registers want it (16-byte chunks at tile + c*1024 + lane*16), so K
// and V stream from HBM straight into VGPRs (global_load_dwordx4, no LDS
// staging).  The next iteration's K and score metadata are requested as soon
// as the score MFMAs have consumed the current ones, its V and value metadata
// after the PV MFMAs; the other waves of the CU (one wave per workgroup, no
// LDS, bounded VGPRs) cover the rest of the latency.
// Float (bf16/f16) pages use the same schedule without the affine terms.
// A piece that covers its whole segment writes the normalised output; other
// pieces write (acc, m, l) partials that merge_kernel, launched next on the
// same stream, combines by log-sum-exp (the kernel boundary makes them
// visible across the XCDs' L2s without any cache maintenance in the loop).
#pragma once
#include <type_traits>

#include "pkv_merge.h"
#include "pkv_mfma.h"
#include "pkv_token.h"

namespace pkv {

// Column slots for a layout: the count the rows allow, halved while the
// per-lane register estimate (payload of SLOTS tiles, metadata, O^T, Q) stays
// above what leaves room for three waves per SIMD.
constexpr int fit_slots(int bits, int dp, int g, int slots) {
  const int lw = dp * bits / 128;
  const int mw = bits != 16 ? 4 * (dp / g) : 0;
  while (slots > 1 && slots * 2 * lw + 2 * mw + dp / 4 + dp / 8 + 40 > 176) slots /= 2;
  return slots;
}

// Shapes whose register needs sit just above 256 VGPRs: asking for two waves
// per SIMD costs them at most a few spills outside the tile loop and doubles
// their occupancy.  Others keep the compiler's choice (heavier shapes would
// spill inside the loop: int8 D256 G128 forced to two waves spilled 98 VGPRs
// and ran 5.6% slower than at one wave per SIMD).
constexpr int min_waves_per_simd(int bits, int dp, int g, int rb, int slots) {
  return (bits == 8 && dp == 128 && g == 64 && rb == 1 && slots == 4) ||
                 (bits == 4 && dp == 128 && g == 32 && rb == 1 && slots == 4) ||
                 (bits == 4 && dp == 128 && g == 64 && rb == 2) ||
                 (bits == 8 && dp == 128 && g == 64 && rb == 2)
             ? 2
             : 1;
}

// Two-row-block kernels dequantize quantized V tiles in registers (see attn_kernel).
constexpr bool kDequantRows = true;

// Waves per run: the kernels for 5-8 rows (two column slots) and 17-32 rows
// (two row blocks) per KV head give each run of the split to a workgroup of
// this many waves, which share its iterations round robin and combine their
// states in LDS at each piece's end; the others run one wave per run.  The fused
// single-token append runs as its shape does without it: the wave that takes a
// piece's last iteration appends (8 sequences of 32K 4-bit tokens, 8 rows per KV
// head: 50.5 us at one wave per run, 38.4 grouped).
constexpr int kGroup = 4;
constexpr int run_waves(int rb, int slots) { return rb == 2 || slots == 2 ? kGroup : 1; }

template <int BITS, int DP, int G, int RB, int FK, int SLOTS, bool APPEND, int GW>
__global__ __launch_bounds__(64 * GW)
__attribute__((amdgpu_waves_per_eu(min_waves_per_simd(BITS, DP, G, RB, SLOTS)))) void attn_kernel(
    const AttnArgs a) {
  using C = Cfg<BITS, DP, G, RB, FK, SLOTS>;
  constexpr bool QUANT = C::QUANT;
  static_assert(!APPEND || RB == 1, "fused append: one row block");
  // Tiles stream in with non-temporal loads for one row block (decode rows:
  // C2 67.7 -> 59.9 us per fused launch); two row blocks (verify) keep plain
  // loads, which let the sequences of a shared prefix meet its pages in L2
  // (C4: 32.8 against 33.8 us with non-temporal loads).
  constexpr bool NT = RB == 1;
  // Quantized V tiles for two row blocks (17-32 query rows per KV head) are
  // dequantized once per tile in registers -- per lane its four tokens,
  // (c - 1024)*scale + bias in f16 as the prefill kernel does -- and the PV
  // contraction takes P itself: with 20 rows the per-group P' operands and
  // bias sums of the undequantized form (AFF) cost more VALU than the
  // elements' conversion.  K stays undequantized at every shape (codes exact
  // in the MFMA, scales applied to the f32 scores), which keeps queries far
  // past unit scale within the bar.
  constexpr bool DEQ = QUANT && RB == 2 && kDequantRows;
  constexpr bool AFF = QUANT && !DEQ;
  constexpr int NG = C::NG, KB = C::KB, NB = C::NB, RPS = C::RPS;
  // MFMA operand types: quantized pages run in f16 (codes as 1024 + c).
  using FO = FloatOps<QUANT ? 1 : FK>;
  using KT = typename FO::KT;
  using VT = typename FO::VT;
  // bf16 pages: P enters the PV MFMA as a bf16 pair hi + lo (16 significant
  // bits).  One bf16 alone is 2^-9 relative, which values of outlier channels
  // (|v| ~ 30) turn into more than the output tolerance on short sequences.
  constexpr bool SPLITP = !QUANT && FK == 0;

  // Lane-derived values are refreshed at every piece through an opaque copy
  // of the lane id, so the compiler recomputes per-lane addresses inside the
  // piece loop instead of hoisting them all and pinning them in registers.
  // Runs of GW waves (GW > 1): wave wk of the workgroup takes iterations wk,
  // wk + GW, ... of each piece of the run.
  const int wk = GW > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  int lane = threadIdx.x & 63;
  int col, jj, slot_l, rowc;  // slot_l: this lane's column slot; rowc: its row within the slot
  auto refresh_lane = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(lane));
    col = lane & 15;
    jj = lane >> 4;
    slot_l = col / RPS;
    rowc = col % RPS;
  };
  refresh_lane();
  const int w = blockIdx.x;
  const Geo &g = a.g;
  const int hk = g.hk;
  const int tpp_shift = __builtin_ctz(g.page / PKV_TILE);
  const int tpp_mask = (1 << tpp_shift) - 1;

  // ---- sequences: lanes hold one 64-sequence chunk (length, tiles, inclusive
  // tile prefix over all sequences); chunk_pre / chunk_end bound its prefix
  int cbase = 0, len_l = 0, nt_l = 0, incl_l = 0, chunk_pre = 0, chunk_end = 0, lead = 0;
  auto scan_chunk = [&](int base, int pre) __attribute__((always_inline)) {
    cbase = base;
    chunk_pre = pre;
    incl_l = wave_scan_incl(base + lane < a.batch && nt_l > 0 ? nt_l + lead : 0, lane) + pre;
    chunk_end = __builtin_amdgcn_readlane(incl_l, 63);
  };
  auto load_chunk = [&](int base, int pre) __attribute__((always_inline)) {
    const int idx = base + lane;
    len_l = idx < a.batch ? a.seq_lens[idx] : 0;
    nt_l = idx < a.batch ? split_tiles(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, idx) : 0;
    scan_chunk(base, pre);
  };
  Split sp;
  if (!a.seg_runs) {
    len_l = lane < a.batch ? a.seq_lens[lane] : 0;
    nt_l = lane < a.batch ? split_tiles(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, lane) : 0;
    int all_tiles = wave_sum(nt_l), served = wave_sum(nt_l > 0 ? 1 : 0);
    for (int c0 = 64; c0 < a.batch; c0 += 64) {
      const int idx = c0 + lane;
      const int nt = idx < a.batch ? split_tiles(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, idx) : 0;
      all_tiles += wave_sum(nt);
      served += wave_sum(nt > 0 ? 1 : 0);
    }
    // tile counts fit in int32: the host bounds batch * (max_pages * pages' tiles + 16) * HK
    const int t0 = __builtin_amdgcn_readfirstlane(all_tiles) * hk;
    if (t0 == 0) return;  // every sequence is served by the prefill kernel
    lead = charged_lead(a.seq_lens, a.widths, a.narrow_lo, a.narrow_q, a.batch, a.waves, a.least, a.lead, nt_l, t0,
                        lane);
    scan_chunk(0, 0);
    const int T = t0 + __builtin_amdgcn_readfirstlane(served) * hk * lead;
    const int W = split_runs(a.waves, a.least, T);
    if (w >= W) return;
    sp.init(T, W);
  }

  // the segment holding split tile g (uniform): sequence, KV head, length,
  // tiles, and its first split tile (its own tiles start `lead` split tiles later)
  auto locate = [&](int gt, int &pb, int &pkh, int &pL, int &pnt, int &pseg0)
      __attribute__((always_inline)) {
    if (gt < chunk_pre * hk) load_chunk(0, 0);
    while (gt >= chunk_end * hk && cbase + 64 < a.batch) load_chunk(cbase + 64, chunk_end);
    const unsigned long long hit = __ballot(cbase + lane < a.batch && incl_l * hk > gt);
    const int f = hit ? __ffsll((long long)hit) - 1 : 0;
    pb = cbase + f;
    pnt = __builtin_amdgcn_readlane(nt_l, f);
    pL = __builtin_amdgcn_readlane(len_l, f);
    const int span = pnt + lead;
    const int pre = (__builtin_amdgcn_readlane(incl_l, f) - span) * hk;
    pkh = (gt - pre) / span;
    pseg0 = pre + pkh * span;
  };

  // ---- per-piece metadata, requested a piece ahead: page-id window (page
  // win + lane), raw query words and query positions
  auto fetch_window = [&](int pb, int win, int t1) __attribute__((always_inline)) -> int {
    const int p = win + lane;
    int id = -1;
    if (p < a.max_pages && (int64_t)p * g.page < t1) id = a.table[(int64_t)pb * a.max_pages + p];
    return id < a.num_pages ? id : -1;
  };
  auto fetch_q = [&](int pb, int pkh, u4 (&raw)[RB][KB], int (&qp)[RB]) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int row = SLOTS > 1 ? rowc : rb * 16 + col;
      const int rowv = row < a.rows ? row : 0;  // rows past the block load row 0, zeroed later
      const int qi = rowv / a.gqa, h = pkh * a.gqa + rowv % a.gqa;
      const uint16_t *qrow = a.q + (((int64_t)pb * a.heads + h) * a.nq_stride + qi) * g.dim;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int d0 = 32 * kb + 8 * jj;
        if ((g.dim & 7) == 0) {
          raw[rb][kb] = *(const u4 *)(qrow + (d0 < g.dim ? d0 : 0));
        } else {
          uint16_t e8[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) e8[e] = qrow[d0 + e < g.dim ? d0 + e : 0];
          raw[rb][kb] = u4{(uint32_t)e8[0] | ((uint32_t)e8[1] << 16), (uint32_t)e8[2] | ((uint32_t)e8[3] << 16),
                           (uint32_t)e8[4] | ((uint32_t)e8[5] << 16), (uint32_t)e8[6] | ((uint32_t)e8[7] << 16)};
        }
      }
      qp[rb] = a.q_pos ? a.q_pos[(int64_t)pb * a.nq_stride + qi] : 0;
    }
  };

  // query operands, row limits and per-row score scales of the current piece
  int lim[RB];
  float rsc[RB];
  KT qv[RB][KB];
  KT qsl[SLOTS > 1 ? SLOTS : 1][KB];  // per slot: the lane's query operand in that slot's columns
  float qs[RB][NG];
  // Grouped runs over quantized pages: the GW waves convert a piece's query
  // operands together -- (row block, kb) pair i by wave i % GW -- and share
  // them, with their f16 sums, through LDS (the same values and sums each
  // wave would form); a row whose group sum overflows f16 takes the per-wave
  // scaled conversion below.
  constexpr bool QSHARE = QUANT && GW > 1;
  constexpr int QPAIRS = RB * KB;
  __shared__ u4 s_qop[QSHARE ? QPAIRS : 1][QSHARE ? 64 : 1];
  __shared__ float s_qsum[QSHARE ? QPAIRS : 1][QSHARE ? 64 : 1];
  auto set_queries = [&](int pL, int pwidth, int t1, const u4 (&raw)[RB][KB], const int (&qp)[RB])
      __attribute__((always_inline)) {
    if constexpr (QSHARE) {
#pragma unroll
      for (int i = 0; i < QPAIRS; ++i) {
        if (i % GW != wk) continue;
        const int rb = i / KB, kb = i % KB;
        const int row = SLOTS > 1 ? rowc : rb * 16 + col;
        const bool valid = row < a.rows;
        const int d0 = 32 * kb + 8 * jj;
        const u4 x = raw[rb][kb];
        uint16_t e8[8] = {(uint16_t)(x.x & 0xFFFF), (uint16_t)(x.x >> 16), (uint16_t)(x.y & 0xFFFF),
                          (uint16_t)(x.y >> 16), (uint16_t)(x.z & 0xFFFF), (uint16_t)(x.z >> 16),
                          (uint16_t)(x.w & 0xFFFF), (uint16_t)(x.w >> 16)};
        h8 v;
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const _Float16 hv = (_Float16)(bits_to_float(!valid || d0 + e >= g.dim ? (uint16_t)0 : e8[e],
                                                       g.float_kind) * 1.0f);
          v[e] = hv;
          sum += (float)hv;
        }
        s_qop[i][lane] = __builtin_bit_cast(u4, v);
        s_qsum[i][lane] = sum;
      }
      __syncthreads();
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int row = SLOTS > 1 ? rowc : rb * 16 + col;
      const bool valid = row < a.rows;
      const int qi = row / a.gqa;
      const bool live = valid && qi < pwidth;
      const int pos = a.q_pos ? qp[rb] : pL - pwidth + qi;
      lim[rb] = live ? min(pos, t1 - 1) : -1;
#pragma unroll
      for (int gi = 0; gi < NG; ++gi) qs[rb][gi] = 0.0f;
      // f16 operands hold at most 65504: a row of bf16 queries with a larger
      // element (seen as a non-finite group sum) is converted again, scaled by
      // a power of two sc that brings its largest element into [2^14, 2^15)
      // (exact), and the inverse is folded into its softmax scale
      float sc = 1.0f;
      auto convert = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int d0 = 32 * kb + 8 * jj;
        u4 x = raw[rb][kb];
        uint16_t e8[8] = {(uint16_t)(x.x & 0xFFFF), (uint16_t)(x.x >> 16), (uint16_t)(x.y & 0xFFFF),
                          (uint16_t)(x.y >> 16), (uint16_t)(x.z & 0xFFFF), (uint16_t)(x.z >> 16),
                          (uint16_t)(x.w & 0xFFFF), (uint16_t)(x.w >> 16)};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (!valid || d0 + e >= g.dim) e8[e] = 0;
        if constexpr (QUANT || FK == 1) {
          h8 v;
          float sum = 0.0f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const _Float16 hv = (_Float16)(bits_to_float(e8[e], g.float_kind) * sc);
            v[e] = hv;
            sum += (float)hv;
          }
          if constexpr (QUANT) qs[rb][(32 * kb) / G] += sum;
          qv[rb][kb] = __builtin_bit_cast(KT, v);
        } else {
          u4 packed = {(uint32_t)e8[0] | ((uint32_t)e8[1] << 16), (uint32_t)e8[2] | ((uint32_t)e8[3] << 16),
                       (uint32_t)e8[4] | ((uint32_t)e8[5] << 16), (uint32_t)e8[6] | ((uint32_t)e8[7] << 16)};
          qv[rb][kb] = __builtin_bit_cast(KT, packed);
        }
      }
      };
      if constexpr (QSHARE) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          qv[rb][kb] = __builtin_bit_cast(KT, s_qop[rb * KB + kb][lane]);
          qs[rb][(32 * kb) / G] += s_qsum[rb * KB + kb][lane];
        }
      } else {
        convert();
      }
      if constexpr (QUANT) {
        bool bad = false;
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) bad |= !__builtin_isfinite(qs[rb][gi]);
        if (__any(bad)) {  // rare: bf16 queries past the f16 range
          float mx = 0.0f;
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            const int d0 = 32 * kb + 8 * jj;
            const u4 x = raw[rb][kb];
            const uint32_t w4[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const uint16_t bits = (uint16_t)(w4[e >> 1] >> (16 * (e & 1)));
              if (valid && d0 + e < g.dim) mx = fmaxf(mx, fabsf(bits_to_float(bits, g.float_kind)));
            }
          }
          mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
          mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
          if (mx >= 32768.0f && mx < INFINITY) {
            int ex;
            frexpf(mx, &ex);  // mx in [2^(ex-1), 2^ex)
            sc = ldexpf(1.0f, 15 - ex);
          }
#pragma unroll
          for (int gi = 0; gi < NG; ++gi) qs[rb][gi] = 0.0f;
          convert();
        }
      }
      rsc[rb] = a.scale_log2 / sc;
      if constexpr (QUANT) {
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
          qs[rb][gi] = xor32_add(xor16_add(qs[rb][gi]));
        }
      }
    }
    if constexpr (SLOTS > 1) {
      // slot j's operands, masked once per piece (column slots need one row block)
      const u4 zero = {0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < SLOTS; ++j)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) qsl[j][kb] = slot_l == j ? qv[0][kb] : __builtin_bit_cast(KT, zero);
    }
  };
  // slot j's query operand: the lane's rows in slot j's columns, zero elsewhere
  auto qop = [&](int j, int rb, int kb) __attribute__((always_inline)) -> KT {
    if constexpr (SLOTS == 1) return qv[rb][kb];
    else return qsl[j][kb];
  };

  // Tiles of iteration `it` of a piece (first tile pta, ntl tiles, page window
  // pwin held in ppid): per slot, the byte offset of its head block in the pool
  // and its tile within the page (uniform); bit j of the returned mask is set
  // when slot j's tile exists.  Loads of absent tiles (past the piece, unmapped
  // pages) read head block kh of page 0; their results are never used.
  auto plan = [&](int pta, int ntl, int pwin, int ppid, int it, int (&pg)[SLOTS], int (&tp)[SLOTS])
      __attribute__((always_inline)) {
    int mask = 0;
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      const int tile = it * SLOTS + j;
      int id = 0, t = 0;
      if (tile < ntl) {
        const int st = pta + tile;
        const int pid_j = __builtin_amdgcn_readlane(ppid, (st >> tpp_shift) - pwin);
        if (pid_j >= 0) {
          id = pid_j;
          t = st & tpp_mask;
          mask |= 1 << j;
        }
      }
      pg[j] = id;
      tp[j] = t;
    }
    return mask;
  };
  // a tile's K payload in the pool (V is g.v_offset further)
  auto tile_at = [&](int pkh, int id, int t) __attribute__((always_inline)) {
    return a.pool + (int64_t)id * g.page_bytes + (int64_t)pkh * g.head_bytes + (int64_t)t * g.tile_bytes;
  };
  // the lane's metadata words: its slot's tile of an iteration as plan()
  // placed it (absent tiles: page 0, tile 0), tokens 4*jj..4*jj+3; the page
  // id comes from plan's uniform values by selects (no lane permute)
  auto meta_at = [&](int pkh, const int (&pg)[SLOTS], const int (&tp)[SLOTS], int64_t side)
      __attribute__((always_inline)) {
    int id = pg[0], t = tp[0];
#pragma unroll
    for (int j = 1; j < SLOTS; ++j) {
      id = slot_l == j ? pg[j] : id;
      t = slot_l == j ? tp[j] : t;
    }
    const int64_t h = (int64_t)pkh * g.head_bytes + (int64_t)id * g.page_bytes;
    return a.pool + h + side + (int64_t)(t * PKV_TILE + 4 * jj) * (NG * 4);
  };

  uint32_t kw[SLOTS][C::LW], vw[SLOTS][C::LW];
  uint32_t km[C::MW], vm[C::MW];
  auto load_k = [&](int pkh, const int (&pg)[SLOTS], const int (&tp)[SLOTS], const uint8_t *mp)
      __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) load_payload<C, NT>(kw[j], tile_at(pkh, pg[j], tp[j]), lane);
    if constexpr (QUANT) load_meta<C, NT>(km, mp);
  };
  auto load_v = [&](int pkh, const int (&pg)[SLOTS], const int (&tp)[SLOTS], const uint8_t *mp)
      __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) load_payload<C, NT>(vw[j], tile_at(pkh, pg[j], tp[j]) + g.v_offset, lane);
    if constexpr (QUANT) load_meta<C, NT>(vm, mp);
  };

  // ---- pieces.  Current: tiles [cta, ctb) of segment (cb, ckh) starting at
  // tile cseg0; the run ends at run_end.  Next (n*): the rest of the run.
  int run_end, cb, ckh, cL, cnt, cseg0, cta, ctb;
  bool cfirst = true;
  if (a.seg_runs) {  // run w is segment w, whole
    cb = w / hk;
    ckh = w - cb * hk;
    cL = __builtin_amdgcn_readfirstlane(a.seq_lens[cb]);
    cnt = run_end = ctb = seq_tiles(cL);
    cseg0 = cta = 0;
  } else {
    run_end = sp.start(w + 1);
    locate(sp.start(w), cb, ckh, cL, cnt, cseg0);
    cta = max(sp.start(w) - cseg0 - lead, 0);
    ctb = min(cnt, run_end - cseg0 - lead);
    if (ctb <= 0) return;  // the run holds lead tiles only: no piece
  }
  int cpid = fetch_window(cb, cta >> tpp_shift, min(cL, ctb * PKV_TILE));

  bool has_next = false;
  int nb = 0, nkh = 0, nL = 0, nnt = 1, nta = 0, ntb = 0, npid = -1, nseg0 = 0;

  // next piece: the next segment's tiles up to the run's end, and its
  // page-id window (read at the next switch)
  auto set_next = [&](int gstart) __attribute__((always_inline)) {
    locate(gstart, nb, nkh, nL, nnt, nseg0);
    nta = max(gstart - nseg0 - lead, 0);
    ntb = min(nnt, run_end - nseg0 - lead);
    npid = fetch_window(nb, nta >> tpp_shift, min(nL, ntb * PKV_TILE));
  };

  int pg[SLOTS], npg[SLOTS], tp[SLOTS], ntp[SLOTS];

  // ---- fused single-token append (APPEND).  The wave whose piece holds a
  // segment's last tile quantizes the sequence's new K/V token (it sits at
  // seq_lens - 1) into LDS (float pages: copies its rows), stores it into its page slot, and patches its
  // codes and (scale, bias) words into the tile registers of the iteration
  // that holds it; no other wave reads that tile in this launch, so the
  // store needs no ordering against the tile loads.
  // (read by words in patch_k)
  __shared__ __attribute__((aligned(16))) uint8_t s_app_codes[2][APPEND && QUANT ? DP : 4];
  __shared__ __attribute__((aligned(16))) uint16_t s_app_raw[2][APPEND && !QUANT ? DP : 2];  // float pages: the rows
  __shared__ uint32_t s_app_meta[2][8];
  int app_it = -1, app_j = 0, app_tt = 0;
  // the new rows are requested with the piece's queries, ahead of its tiles
  // (loads return in order)
  constexpr int AEPL = DP / 64;
  uint16_t app_raw[APPEND ? 2 : 1][APPEND ? AEPL : 1];
  int app_pid = -1;
  auto append_fetch = [&](int pb, int pkh, int pos) __attribute__((always_inline)) {
    if constexpr (APPEND) {
      // (a position past the block table has no page: the token is dropped, as
      // the append kernels drop it)
      const int slot = pos / g.page;
      app_pid = slot < a.max_pages ? a.table[(int64_t)pb * a.max_pages + slot] : -1;
      const int64_t row = ((int64_t)pb * hk + pkh) * g.dim;
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        const uint16_t *src = (side ? a.new_v : a.new_k) + row;
#pragma unroll
        for (int i = 0; i < AEPL; ++i) {
          const int d = lane * AEPL + i;
          app_raw[side][i] = d < g.dim ? src[d] : (uint16_t)0;
        }
      }
    }
  };
  auto append_token = [&](int pkh, int pos, int pta) __attribute__((always_inline)) {
    if constexpr (APPEND) {
      if (app_pid < 0 || app_pid >= a.num_pages) return;  // an unmapped page holds no tile either
      const int tile = pos / PKV_TILE - pta;  // within the piece
      app_it = tile / SLOTS;
      app_j = tile % SLOTS;
      app_tt = pos % PKV_TILE;
      if constexpr (!QUANT) {
        uint8_t *head = a.wpool + (int64_t)app_pid * g.page_bytes + (int64_t)pkh * g.head_bytes +
                        (int64_t)(pos % g.page / PKV_TILE) * g.tile_bytes;
#pragma unroll
        for (int i = 0; i < AEPL; ++i) {
          const int d = lane * AEPL + i;
          s_app_raw[0][d] = app_raw[0][i];
          s_app_raw[1][d] = app_raw[1][i];
          *(uint16_t *)(head + payload_offset(app_tt + 16 * (d % 32 / 8), 2 * (8 * (d / 32) + d % 8), 16)) =
              app_raw[0][i];
          *(uint16_t *)(head + g.v_offset +
                        payload_offset(d % 16 + 16 * (app_tt / 4), 2 * (4 * (d / 16) + app_tt % 4), 16)) =
              app_raw[1][i];
        }
        wave_lds_sync();
        return;
      }
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        float x[AEPL];
#pragma unroll
        for (int i = 0; i < AEPL; ++i) {
          const int d = lane * AEPL + i;
          x[i] = d < g.dim ? bits_to_float(app_raw[side][i], g.float_kind) : 0.0f;  // zero pad
        }
        quantize_row<AEPL>(x, lane, G, BITS, s_app_codes[side], s_app_meta[side]);
      }
      wave_lds_sync();
      if constexpr (QUANT)
        store_token<DP, BITS>(g, a.wpool + (int64_t)app_pid * g.page_bytes + (int64_t)pkh * g.head_bytes,
                              pos % g.page, s_app_codes[0], s_app_codes[1], s_app_meta[0], s_app_meta[1],
                              lane);
    }
  };
  // the token's K payload (lanes col == tt hold its elements d = 32kb + 8jj + e)
  // and K meta word (lanes of its slot whose four tokens 4jj..4jj+3 hold it)
  auto patch_k = [&]() __attribute__((always_inline)) {
    if constexpr (APPEND) {
      const bool mine = col == app_tt;
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        if (j != app_j) continue;
#pragma unroll
        for (int x = 0; x < C::LW; ++x) {
          uint32_t word = 0;
          if constexpr (!QUANT) {
            word = *(const uint32_t *)&s_app_raw[0][32 * (x / 4) + 8 * jj + 2 * (x % 4)];
          } else if constexpr (BITS == 8) {
            word = *(const uint32_t *)&s_app_codes[0][32 * (x / 2) + 8 * jj + 4 * (x % 2)];
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              word |= (uint32_t)(s_app_codes[0][32 * x + 8 * jj + e] & 15) << (4 * k4_nibble(e));
          }
          kw[j][x] = mine ? word : kw[j][x];
        }
      }
      if constexpr (!QUANT) return;
      const bool mm = slot_l == app_j && jj == app_tt / 4;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
          if (r == app_tt % 4) km[r * NG + gi] = mm ? s_app_meta[0][gi] : km[r * NG + gi];
    }
  };
  // the token's V payload (lanes jj == tt/4, byte r = tt%4 of each block) and V meta word
  auto patch_v = [&]() __attribute__((always_inline)) {
    if constexpr (APPEND) {
      const int r = app_tt % 4;
      const bool mine = jj == app_tt / 4;
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        if (j != app_j) continue;
        if constexpr (!QUANT) {
#pragma unroll
          for (int n = 0; n < NB; ++n) {
            const uint32_t v = s_app_raw[1][16 * n + col];
#pragma unroll
            for (int h = 0; h < 2; ++h) {  // word h of the block: tokens 2h, 2h + 1
              const uint32_t old = vw[j][2 * n + h];
              const uint32_t word = (r & 1) ? (old & 0x0000FFFFu) | (v << 16) : (old & 0xFFFF0000u) | v;
              vw[j][2 * n + h] = mine && r / 2 == h ? word : old;
            }
          }
        } else if constexpr (BITS == 8) {
#pragma unroll
          for (int n = 0; n < NB; ++n) {
            const uint32_t sh = 8 * r;
            const uint32_t word = (vw[j][n] & ~(0xFFu << sh)) | ((uint32_t)s_app_codes[1][16 * n + col] << sh);
            vw[j][n] = mine ? word : vw[j][n];
          }
        } else {
#pragma unroll
          for (int m2 = 0; m2 < NB / 2; ++m2) {
            const uint32_t sh = 8 * v4_byte(r);
            const uint32_t byte = (uint32_t)(s_app_codes[1][32 * m2 + col] & 15) |
                                  ((uint32_t)(s_app_codes[1][32 * m2 + 16 + col] & 15) << 4);
            const uint32_t word = (vw[j][m2] & ~(0xFFu << sh)) | (byte << sh);
            vw[j][m2] = mine ? word : vw[j][m2];
          }
        }
      }
      if constexpr (!QUANT) return;
      const bool mm = slot_l == app_j && jj == app_tt / 4;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
          if (rr == r) vm[rr * NG + gi] = mm ? s_app_meta[1][gi] : vm[rr * NG + gi];
    }
  };

  // ---- grouped runs: the GW waves' states of a piece meet in LDS (64 KB at
  // head_dim 128, two row blocks).  At the piece's end every wave publishes
  // its rows' maxima, sums and O^T values as its epilogue leaves them (jj
  // lanes and column slots folded; writer lanes); then wave wk combines
  // output columns d in [16*NB/GW*wk, 16*NB/GW*(wk+1)) by log-sum-exp (a wave
  // without a visible token holds l = 0 and weighs nothing) and writes them,
  // normalised (whole segment) or as the run's partial.  (Deferring the
  // combine until the next piece's first loads were issued measured slower:
  // C4 29.6 against 29.1 us.)
  constexpr int GWL = GW > 1 ? GW : 1;
  constexpr int RBL = GW > 1 ? RB : 1;
  constexpr int NBL = GW > 1 ? NB : 1;
  __shared__ f4 s_gO[GWL][RBL][NBL][GW > 1 ? 64 : 1];
  __shared__ float s_gm[GWL][RBL][16], s_gl[GWL][RBL][16];
  auto group_combine = [&](bool whole, int slot, int pb, int pkh) __attribute__((always_inline)) {
    if constexpr (GW > 1) {
      constexpr int NPW = NB / GW;
      static_assert(NPW * GW == NB, "output column blocks per wave");
      __syncthreads();  // every wave's state is published
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        float M = -INFINITY, mk[GW], lk[GW], wt[GW];
#pragma unroll
        for (int k = 0; k < GW; ++k) {
          mk[k] = s_gm[k][rb][col];
          lk[k] = s_gl[k][rb][col];
          if (lk[k] > 0.0f) M = fmaxf(M, mk[k]);
        }
        float L = 0.0f;
#pragma unroll
        for (int k = 0; k < GW; ++k) {
          wt[k] = lk[k] > 0.0f ? __builtin_amdgcn_exp2f(mk[k] - M) : 0.0f;
          L += wt[k] * lk[k];
        }
        const int row = SLOTS > 1 ? rowc : rb * 16 + col;
        const bool writer = slot_l == 0 && row < a.rows;
        const int qi = row / a.gqa, h = pkh * a.gqa + row % a.gqa;
        const float inv = 1.0f / fmaxf(L, 1e-20f);
        uint16_t *o = a.out + (((int64_t)pb * a.heads + h) * a.nq_stride + qi) * g.dim;
        float *pa = a.part_acc + ((int64_t)slot * a.rows + row) * DP;
#pragma unroll
        for (int i = 0; i < NPW; ++i) {
          const int n = wk * NPW + i;
          f4 v = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int k = 0; k < GW; ++k) v += wt[k] * s_gO[k][rb][n][lane];
          const int d = 16 * n + 4 * jj;
          if (!writer) continue;
          if (whole) {
            if ((g.dim & 3) == 0 && d + 4 <= g.dim) {
              u2 packed = {(uint32_t)float_to_bits(v[0] * inv, g.float_kind) |
                               ((uint32_t)float_to_bits(v[1] * inv, g.float_kind) << 16),
                           (uint32_t)float_to_bits(v[2] * inv, g.float_kind) |
                               ((uint32_t)float_to_bits(v[3] * inv, g.float_kind) << 16)};
              *(u2 *)(o + d) = packed;
            } else {
#pragma unroll
              for (int r = 0; r < 4; ++r)
                if (d + r < g.dim) o[d + r] = float_to_bits(v[r] * inv, g.float_kind);
            }
          } else {
            *(f4 *)(pa + d) = v;
          }
        }
        if (wk == 0 && writer && !whole && jj == 0)
          *(float2 *)(a.part_ml + ((int64_t)slot * a.rows + row) * 2) = make_float2(M, L);
      }
      __syncthreads();  // the next piece's states are published over these
    }
  };
  for (;;) {
    refresh_lane();
    // ---- start the piece: query rows and its first tiles, in flight together
    const int width = a.widths ? a.widths[cb] : a.nq;
    const int t0 = cta * PKV_TILE;
    const int t1 = min(cL, ctb * PKV_TILE);
    const int ntl = t1 > t0 ? (t1 - t0 + PKV_TILE - 1) / PKV_TILE : 0;
    const int niters = max(1, (ntl + SLOTS - 1) / SLOTS);
    int cwin = cta >> tpp_shift;
    int cmask;
    // the piece holds the segment's last tile, this wave its last iteration
    const bool appends = APPEND && ctb == cnt && cL > 0 && (GW == 1 || (niters - 1) % GW == wk);
    {
      u4 raw[RB][KB];
      int qp[RB];
      if constexpr (APPEND) {
        if (appends) append_fetch(cb, ckh, cL - 1);
      }
      fetch_q(cb, ckh, raw, qp);
      cmask = plan(cta, ntl, cwin, cpid, wk, pg, tp);
      load_k(ckh, pg, tp, meta_at(ckh, pg, tp, g.kmeta_offset));
      load_v(ckh, pg, tp, meta_at(ckh, pg, tp, g.vmeta_offset));
      set_queries(cL, width, t1, raw, qp);
      // the new token: quantized and stored while the piece's first tiles
      // are in flight (it is patched into the registers of the piece's last
      // iteration)
      if constexpr (APPEND) {
        app_it = -1;
        if (appends) append_token(ckh, cL - 1, cta);
      }
      // the rest of the run is the next piece: its page-id window now
      has_next = ctb == cnt && cseg0 + cnt + 2 * lead < run_end;
      if (has_next) set_next(cseg0 + lead + cnt);
    }

    float m[RB], lsum[RB], corr[RB][NG], osum[RB][NG];
    // Two row blocks of quantized pages take the per-column sums over tokens
    // on the MFMA pipe instead of the VALU: csum = sum p * bias_v (the V bias
    // term) and osum4 = sum P' (the 1024 offset), as 16x16x16 products of the
    // tokens' f16 biases (or ones) with p (or P'); every row of the result
    // holds the column's sum.
    constexpr bool MSUM = RB == 2 && AFF;
    f4 csum[MSUM ? RB : 1][MSUM ? NG : 1], osum4[MSUM ? RB : 1][MSUM ? NG : 1];
    f4 O[RB][NB];  // O^T[d = 16n + 4jj + r][column]
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      m[rb] = -INFINITY;
      lsum[rb] = 0.0f;
#pragma unroll
      for (int n = 0; n < NB; ++n) O[rb][n] = f4{0, 0, 0, 0};
#pragma unroll
      for (int gi = 0; gi < NG; ++gi) { corr[rb][gi] = 0.0f; osum[rb][gi] = 0.0f; }
      if constexpr (MSUM) {
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) { csum[rb][gi] = f4{0, 0, 0, 0}; osum4[rb][gi] = f4{0, 0, 0, 0}; }
      }
    }

    // One iteration over SLOTS tiles; with `more`, the next iteration's tiles
    // are requested as soon as each half's registers are free (the last
    // iteration is peeled so nothing is in flight across the epilogue).
    auto iterate = [&](auto more, int it) __attribute__((always_inline)) {
      constexpr bool MORE = decltype(more)::value;
      refresh_lane();
      // the appended token sits in the piece's last tile, hence in its last
      // iteration (the peeled one): the loop body stays the plain kernel's
      if constexpr (APPEND && !MORE) {
        if (app_it >= 0) patch_k();
      }
      // Float pages: a page reused after another sequence may hold anything
      // past this piece's last token, and the column-slot products multiply
      // a slot's K rows by other slots' zero query columns (and every V row by
      // its P), so 0 * inf would spread.  Those rows are zeroed in registers
      // in the iteration that holds the piece's end.  (Codes are always finite.)
      const bool tail_it = t0 + (it + 1) * SLOTS * PKV_TILE > t1;
      if constexpr (!QUANT) {
        if (tail_it) {
#pragma unroll
          for (int j = 0; j < SLOTS; ++j) {
            const bool dead = t0 + (it * SLOTS + j) * PKV_TILE + col >= t1;
#pragma unroll
            for (int x = 0; x < C::LW; ++x) kw[j][x] = dead ? 0u : kw[j][x];
          }
        }
      }
      // S^T for the iteration's tiles (slot j -> columns of slot j).  Codes
      // are finite whatever a register holds, and an absent tile's columns
      // are masked by select (scores) or hold exact-zero P' operands, so
      // quantized pages with several slots run every slot's products
      // unguarded: straight-line code, no per-tile branches.
      constexpr bool UNGUARDED = QUANT && SLOTS > 1;
      // (unguarded chains start from zeros held in registers: an inline-zero
      // accumulator would let the compiler place a chain's first product over
      // part of its own operands)
      f4 zacc = f4{0, 0, 0, 0};
      if constexpr (UNGUARDED) asm volatile("" : "+v"(zacc));
      f4 acc[RB][NG];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) acc[rb][gi] = zacc;
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        if (UNGUARDED || (cmask & (1 << j))) {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            KT kop;
            if constexpr (QUANT) {
              kop = Conv<BITS>::template kop<C::LW>(kw[j], kb);
            } else {
              u4 r = {kw[j][4 * kb], kw[j][4 * kb + 1], kw[j][4 * kb + 2], kw[j][4 * kb + 3]};
              kop = __builtin_bit_cast(KT, r);
            }
            const int gi = QUANT ? (32 * kb) / G : 0;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) acc[rb][gi] = FO::qk(kop, qop(j, rb, kb), acc[rb][gi]);
          }
        }
      }
      // scores of the lane's tile (its slot's tile of this iteration)
      const bool my_ok = (cmask >> slot_l) & 1;
      const int tok0 = t0 + (it * SLOTS + slot_l) * PKV_TILE + 4 * jj;
      // One slot: the tile's presence (uniform) folded into the rows'
      // limits, opaque to the compiler, which otherwise branches around every
      // score's assembly (eight branches per tile at two row blocks; C4
      // launch -3.8%).  Several slots keep the per-lane flag (the fold
      // measured 2.5% slower at C3).
      int limv[RB];
      if constexpr (SLOTS == 1) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          limv[rb] = my_ok ? lim[rb] : -1;
          asm volatile("" : "+v"(limv[rb]));
        }
      }
      float s[RB][4];
      bool vis[RB][4];
      bool need = false;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v;
          if constexpr (QUANT) {
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
              const uint32_t word = km[r * NG + gi];
              const float ks = f16_bits_to_f32(word);
              const float kbias = f16_bits_to_f32(word >> 16) - 1024.0f * ks;
              const float term = ks * acc[rb][gi][r] + qs[rb][gi] * kbias;
              v = gi == 0 ? term : v + term;  // no 0.0f + term: the add would stay (signed zero)
            }
          } else {
            v = acc[rb][0][r];
          }
          if constexpr (SLOTS == 1) vis[rb][r] = tok0 + r <= limv[rb];
          else vis[rb][r] = my_ok && tok0 + r <= lim[rb];
          v = vis[rb][r] ? v * rsc[rb] : -INFINITY;
          s[rb][r] = v;
          need |= v > m[rb] + kTau;
        }
      // K registers and score metadata are free: request the next iteration's
      int nmask = 0;
      const uint8_t *nmv = nullptr;
      if constexpr (MORE) {
        __builtin_amdgcn_sched_barrier(0);
        const int first = cta + (it + GW) * SLOTS;
        const int last = cta + min((it + GW) * SLOTS + SLOTS, ntl) - 1;
        if ((last >> tpp_shift) - cwin > 63) {
          cwin = first >> tpp_shift;  // the iteration's tiles leave the window: slide it
          cpid = fetch_window(cb, cwin, t1);
        }
        nmask = plan(cta, ntl, cwin, cpid, it + GW, npg, ntp);
        load_k(ckh, npg, ntp, meta_at(ckh, npg, ntp, g.kmeta_offset));
        nmv = meta_at(ckh, npg, ntp, g.vmeta_offset);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (__any(need)) {
        // Until a column sees its first visible token its running max is
        // -inf and its sums and O^T are exact zeros: while that holds for
        // every column (a piece's first iteration), the max moves without
        // the rescale.
        bool fresh = true;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) fresh &= m[rb] == -INFINITY;
        const bool rescale = !__all(fresh);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          float tm = fmaxf(fmaxf(s[rb][0], s[rb][1]), fmaxf(s[rb][2], s[rb][3]));
          tm = xor32_max(xor16_max(tm));
          const float mn = fmaxf(m[rb], tm);
          if (!rescale) {
            m[rb] = mn;
            continue;
          }
          const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m[rb] - mn);
          m[rb] = mn;
          lsum[rb] *= alpha;
#pragma unroll
          for (int gi = 0; gi < NG; ++gi) {
            if constexpr (MSUM) {
              csum[rb][gi] *= alpha;
              osum4[rb][gi] *= alpha;
            } else if constexpr (AFF) {
              corr[rb][gi] *= alpha;
              osum[rb][gi] *= alpha;
            }
          }
#pragma unroll
          for (int n = 0; n < NB; ++n) O[rb][n] *= alpha;
        }
      }
      if constexpr (APPEND && !MORE) {
        if (app_it >= 0) patch_v();
      }
      // probabilities and the P operands (per group for quantized V).  Masked
      // tokens contribute exact zeros through selects, whatever their page
      // holds.  The column-sum products take the tokens' biases as an MFMA
      // operand, so for them the value metadata of tokens the piece does not
      // hold (past its end, absent tiles) is cleared as well.
      uint32_t vmw[MSUM ? C::MW : 1];
      if constexpr (MSUM) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool held = my_ok && tok0 + r < t1;
#pragma unroll
          for (int gi = 0; gi < NG; ++gi) vmw[r * NG + gi] = held ? vm[r * NG + gi] : 0u;
        }
      }
      VT pop[RB][NG];
      VT plo[SPLITP ? RB : 1];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = vis[rb][r] ? __builtin_amdgcn_exp2f(s[rb][r] - m[rb]) : 0.0f;
        lsum[rb] += (p[0] + p[1]) + (p[2] + p[3]);
        if constexpr (AFF) {
#pragma unroll
          for (int gi = 0; gi < NG; ++gi) {
            h4 pv;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const uint32_t word = vm[r * NG + gi];
              const _Float16 ps = (_Float16)(p[r] * f16_bits_to_f32(word));
              pv[r] = vis[rb][r] ? ps : (_Float16)0.0f;
              if constexpr (!MSUM) {
                corr[rb][gi] += vis[rb][r] ? p[r] * f16_bits_to_f32(word >> 16) : 0.0f;
                osum[rb][gi] += (float)pv[r];
              }
            }
            pop[rb][gi] = pv;
            if constexpr (MSUM) {
              // A: the lane's four tokens' biases (or ones) for every row; B: p (or P')
              const h4 bias4 = __builtin_bit_cast(
                  h4, u2{perm(vmw[NG + gi], vmw[gi], 0x07060302u), perm(vmw[3 * NG + gi], vmw[2 * NG + gi], 0x07060302u)});
              const h4 p16 = {(_Float16)p[0], (_Float16)p[1], (_Float16)p[2], (_Float16)p[3]};
              const h4 ones = {(_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f};
              csum[rb][gi] = FO::pv(bias4, p16, csum[rb][gi]);
              osum4[rb][gi] = FO::pv(ones, pv, osum4[rb][gi]);
            }
          }
        } else {
          pop[rb][0] = FO::pack_p(p[0], p[1], p[2], p[3]);
          if constexpr (SPLITP) plo[rb] = FO::pack_lo(p[0], p[1], p[2], p[3], pop[rb][0]);
        }
      }
      if constexpr (!QUANT) {
        if (tail_it) {  // V rows past the piece's end (see the K rows above)
#pragma unroll
          for (int j = 0; j < SLOTS; ++j) {
            const int tb = t0 + (it * SLOTS + j) * PKV_TILE + 4 * jj;
            const uint32_t keep01 = (tb < t1 ? 0x0000FFFFu : 0u) | (tb + 1 < t1 ? 0xFFFF0000u : 0u);
            const uint32_t keep23 = (tb + 2 < t1 ? 0x0000FFFFu : 0u) | (tb + 3 < t1 ? 0xFFFF0000u : 0u);
#pragma unroll
            for (int n = 0; n < NB; ++n) {
              vw[j][2 * n] &= keep01;
              vw[j][2 * n + 1] &= keep23;
            }
          }
        }
      }
      if constexpr (DEQ) {
        static_assert(SLOTS == 1, "dequantized V rows take one column slot");
        if (tail_it) {
          // the lane's tokens past the piece's end (stale page bytes): scale
          // and bias 0, so they dequantize to exact zeros (one select per
          // word here rather than a branch per column block below)
          const int tb = t0 + it * PKV_TILE + 4 * jj;
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) vm[r * NG + gi] = tb + r < t1 ? vm[r * NG + gi] : 0u;
        }
      }
      // O^T += V^T . P'^T for each tile
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        if (UNGUARDED || (cmask & (1 << j))) {
          VT bop[RB][NG], blo[SPLITP ? RB : 1];
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            const u2 zero = {0, 0};
#pragma unroll
            for (int gi = 0; gi < NG; ++gi)
              bop[rb][gi] = (SLOTS == 1 || slot_l == j) ? pop[rb][gi] : __builtin_bit_cast(VT, zero);
            if constexpr (SPLITP) blo[rb] = (SLOTS == 1 || slot_l == j) ? plo[rb] : __builtin_bit_cast(VT, zero);
          }
#pragma unroll
          for (int n = 0; n < NB; ++n) {
            VT vop;
            if constexpr (DEQ) {
              // the lane's four tokens 4jj..4jj+3 of column 16n + col,
              // dequantized (tokens past the piece's end: zero metadata)
              const int gi = (16 * n) / G;
              h4 sc, bi;
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const h2 sb = __builtin_bit_cast(h2, vm[r * NG + gi]);
                sc[r] = sb.x;
                bi[r] = sb.y;
              }
              const h4 c = Conv<BITS>::template vop<C::LW>(vw[j], n);
              vop = __builtin_bit_cast(VT, __builtin_elementwise_fma(c - (_Float16)1024.0f, sc, bi));
            } else if constexpr (QUANT) {
              vop = Conv<BITS>::template vop<C::LW>(vw[j], n);
            } else {
              u2 r = {vw[j][2 * n], vw[j][2 * n + 1]};
              vop = __builtin_bit_cast(VT, r);
            }
            const int gi = AFF ? (16 * n) / G : 0;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              O[rb][n] = FO::pv(vop, bop[rb][gi], O[rb][n]);
              if constexpr (SPLITP) O[rb][n] = FO::pv(vop, blo[rb], O[rb][n]);
            }
          }
        }
      }
      // V registers and value metadata are free: request the next iteration's
      if constexpr (MORE) {
        __builtin_amdgcn_sched_barrier(0);
        load_v(ckh, npg, ntp, nmv);
        __builtin_amdgcn_sched_barrier(0);
        cmask = nmask;
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) { pg[j] = npg[j]; tp[j] = ntp[j]; }
      }
    };
    if constexpr (GW == 1) {
      for (int it = 0; it + 1 < niters; ++it) iterate(std::true_type(), it);
      iterate(std::false_type(), niters - 1);
    } else if (wk < niters) {  // (uniform per wave) a wave past the piece's iterations holds nothing
      const int last = wk + GW * ((niters - 1 - wk) / GW);
      for (int it = wk; it < last; it += GW) iterate(std::true_type(), it);
      iterate(std::false_type(), last);
    }

    // ---- piece epilogue: fold the 4 jj lanes of a column, then the slots of a
    // row, and write the output (whole segment) or the partial
    const bool whole = cta == 0 && ctb == cnt;
    const int slot = cfirst ? 2 * w : 2 * w + 1;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      lsum[rb] = xor32_add(xor16_add(lsum[rb]));
#pragma unroll
      for (int gi = 0; gi < NG; ++gi) {
        if constexpr (MSUM) {  // already summed over the tokens of every lane
          corr[rb][gi] = csum[rb][gi][0];
          osum[rb][gi] = osum4[rb][gi][0];
        } else if constexpr (AFF) {
          corr[rb][gi] = xor32_add(xor16_add(corr[rb][gi]));
          osum[rb][gi] = xor32_add(xor16_add(osum[rb][gi]));
        }
      }
      float mrow = m[rb], lrow = lsum[rb], wgt = 1.0f;
      if constexpr (SLOTS > 1) {
        // the row's slot columns (lanes col, col +- RPS, ...) merge by log-sum-exp
#pragma unroll
        for (int o = RPS; o < 16; o <<= 1) mrow = fmaxf(mrow, __shfl_xor(mrow, o, 64));
        wgt = lsum[rb] > 0.0f ? __builtin_amdgcn_exp2f(m[rb] - mrow) : 0.0f;
        lrow = wgt * lsum[rb];
#pragma unroll
        for (int o = RPS; o < 16; o <<= 1) lrow += __shfl_xor(lrow, o, 64);
      }
      const int row = SLOTS > 1 ? rowc : rb * 16 + col;
      const bool writer = slot_l == 0 && row < a.rows;
      const int qi = row / a.gqa, h = ckh * a.gqa + row % a.gqa;
      const float inv = 1.0f / fmaxf(lrow, 1e-20f);
      uint16_t *o = a.out + (((int64_t)cb * a.heads + h) * a.nq_stride + qi) * g.dim;
      float *pa = a.part_acc + ((int64_t)slot * a.rows + row) * DP;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        float v4[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = O[rb][n][r];
          if constexpr (AFF) {
            const int gi = (16 * n) / G;
            v += corr[rb][gi] - 1024.0f * osum[rb][gi];
          }
          v *= wgt;
          if constexpr (SLOTS > 1) {
#pragma unroll
            for (int o2 = RPS; o2 < 16; o2 <<= 1) v += __shfl_xor(v, o2, 64);
          }
          v4[r] = v;
        }
        if constexpr (GW > 1) {  // published; the group's combine writes
          s_gO[wk][rb][n][lane] = f4{v4[0], v4[1], v4[2], v4[3]};
          continue;
        }
        if (!writer) continue;
        const int d = 16 * n + 4 * jj;
        if (whole) {
          if ((g.dim & 3) == 0 && d + 4 <= g.dim) {
            u2 packed = {(uint32_t)float_to_bits(v4[0] * inv, g.float_kind) |
                             ((uint32_t)float_to_bits(v4[1] * inv, g.float_kind) << 16),
                         (uint32_t)float_to_bits(v4[2] * inv, g.float_kind) |
                             ((uint32_t)float_to_bits(v4[3] * inv, g.float_kind) << 16)};
            *(u2 *)(o + d) = packed;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (d + r < g.dim) o[d + r] = float_to_bits(v4[r] * inv, g.float_kind);
          }
        } else {
          *(f4 *)(pa + d) = f4{v4[0], v4[1], v4[2], v4[3]};
        }
      }
      if constexpr (GW > 1) {
        if (jj == 0) {
          s_gm[wk][rb][col] = mrow;
          s_gl[wk][rb][col] = lrow;
        }
      } else if (writer && !whole && jj == 0) {
        *(float2 *)(a.part_ml + ((int64_t)slot * a.rows + row) * 2) = make_float2(mrow, lrow);
      }
    }
    if constexpr (GW > 1) group_combine(whole, slot, cb, ckh);

    // ---- switch to the next piece
    if (!has_next) break;
    cb = nb; ckh = nkh; cL = nL; cnt = nnt; cseg0 = nseg0; cta = nta; ctb = ntb;
    cfirst = false; cpid = npid;
  }

}

typedef void (*AttnKernel)(AttnArgs);

// GROUP: the form of kGroup waves per run (the only one where run_waves says so)
template <int BITS, int DP, int G, int RB, int FK, int SLOTS, bool APPEND, bool GROUP>
static AttnKernel kernel_of() {
  if constexpr (RB > 1 && DP > 128) {
    return nullptr;  // 17..32 rows at head_dim > 128 run on the prefill kernel
  } else if constexpr (APPEND && RB > 1) {
    return nullptr;  // the fused append serves one row block
  } else {
    constexpr int slots = fit_slots(BITS, DP, G, SLOTS);
    return attn_kernel<BITS, DP, G, RB, FK, slots, APPEND, GROUP ? kGroup : run_waves(RB, slots)>;
  }
}

template <int RB, int SLOTS, bool APPEND, bool GROUP>
static AttnKernel select_shape(const Geo &g) {
#define PKV_Q(BITS_, DP_, G_) \
  if (g.bits == BITS_ && g.dp == DP_ && g.group == G_) return kernel_of<BITS_, DP_, G_, RB, 1, SLOTS, APPEND, GROUP>();
  PKV_Q(8, 64, 32) PKV_Q(8, 64, 64)
  PKV_Q(8, 128, 32) PKV_Q(8, 128, 64) PKV_Q(8, 128, 128)
  PKV_Q(8, 256, 32) PKV_Q(8, 256, 64) PKV_Q(8, 256, 128)
  PKV_Q(4, 64, 32) PKV_Q(4, 64, 64)
  PKV_Q(4, 128, 32) PKV_Q(4, 128, 64) PKV_Q(4, 128, 128)
  PKV_Q(4, 256, 32) PKV_Q(4, 256, 64) PKV_Q(4, 256, 128)
#undef PKV_Q
#define PKV_F(DP_, FK_) \
  if (g.bits == 16 && g.dp == DP_ && g.float_kind == FK_) return kernel_of<16, DP_, 32, RB, FK_, SLOTS, APPEND, GROUP>();
  PKV_F(64, 0) PKV_F(64, 1) PKV_F(128, 0) PKV_F(128, 1) PKV_F(256, 0) PKV_F(256, 1)
#undef PKV_F
  return nullptr;
}

// The grouped form (kGroup waves per run) of every decode shape; `append`: the
// fused single-token append, up to 8 rows.  In a source of its own
// (pkv_attention_grouped.hip), so that the two sets of kernels compile side by side.
AttnKernel select_grouped(const Geo &g, int rows, bool append);

}  // namespace pkv
