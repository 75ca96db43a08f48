// pkv_launch.h -- kernel argument structs and host launchers of libpkv.
#pragma once
#include "pkv_device.h"

namespace pkv {

struct AppendArgs {
  Geo g;
  uint8_t *pool;
  int64_t num_pages;
  const uint16_t *keys, *values;  // [B][HK][T][D]
  int batch, tokens, max_pages;
  const int32_t *table, *start_pos, *widths;
  const int32_t *lens_after;  // start_pos NULL: start = lens_after[b] - tokens
  int32_t *new_lens;
};

struct GatherArgs {
  Geo g;
  const uint8_t *pool;
  int64_t num_pages;
  const int32_t *ids;
  int count;
  uint8_t *kc, *vc;        // codes, or float K/V (2 bytes per element)
  uint16_t *ks, *kb, *vs, *vb;
  int dq;                  // reference code bytes per row (quantized)
  int ngr;                 // reference groups per row
};

// Partial slots of the attention workspace per work wave: the first and the
// last piece of its run.
constexpr int kSlotsPerWave = 2;

struct AttnArgs {
  Geo g;
  const uint8_t *pool;
  int64_t num_pages;
  const uint16_t *q;  // [B][H][nq_stride][D]
  int batch, heads, nq, gqa, rows;
  // Q extent of queries, q_pos and out (= nq except for the decode part of a
  // mixed batch, which covers the first nq of nq_stride query rows)
  int nq_stride;
  // Mixed batches (narrow_q 0: off).  Decode kernel: serve only sequences
  // whose width w has narrow_lo < w <= narrow_q.  Prefill kernel: leave
  // sequences of width at most narrow_q to the decode kernel (their rows are
  // written as zeros first).
  int narrow_lo, narrow_q;
  const int32_t *table;
  int max_pages;
  const int32_t *seq_lens, *q_pos, *widths;
  float scale_log2;  // softmax scale * log2(e)
  int waves;         // runs (grid size)
  // Waves per run where the launch asks for the grouped form of a kernel that
  // otherwise runs one wave per run (else 0), and whether run w is segment w,
  // whole, instead of an equal share of the tiles (no partials, no merge).
  int group = 0, seg_runs = 0;
  int least = 0;     // a run holds 2^least tiles at least (fewer runs where there are too few tiles)
  int lead;          // tiles of start-up cost charged ahead of each segment in the split
  float *part_acc;   // [2*waves][rows][DP]
  float *part_ml;    // [2*waves][rows][2]
  uint16_t *out;     // [B][H][Q][D]
  // Fused single-token append (new_k non-NULL): each sequence's new K/V row
  // [B][HK][D] is quantized into slot seq_lens[b] - 1 of its pages (wpool is
  // the pool, writable) by the wave that attends the sequence's last tile.
  uint8_t *wpool = nullptr;
  const uint16_t *new_k = nullptr, *new_v = nullptr;
  // Prefill kernel: the CUs to fill (0: no span is cut), the units of the longest
  // span the block table can hold, and the partials of spans cut into pieces
  // (prefill_longest): pieces per row block, then per piece the rows' (m, l)
  // [block*S + piece][rows per block][2] and O^T as its lanes hold it.
  int pre_cus = 0, pre_units = 0;
  int32_t *pre_cnt = nullptr;
  float *pre_ml = nullptr, *pre_acc = nullptr;
};

struct MergeArgs {
  int batch, hk, heads, nq, gqa, rows, dim, dp, float_kind;
  int waves, lead, least = 0;  // as launched for the attention kernel
  int nq_stride, narrow_lo, narrow_q;
  const int32_t *seq_lens, *widths;
  const float *part_acc, *part_ml;
  uint16_t *out;
};

// A sequence of `units` units of 128 tokens in a prefill grid of `blocks` row
// blocks (one workgroup per CU each: LDS) that would leave CUs idle: the longest
// piece its row blocks' spans are cut into, in units (all of them: whole spans).
// A unit takes about 4.2 us (head_dim 128), a piece a step of the merge, which
// walks them in order, and its partials, so the best number of pieces grows as
// the root of the units: sqrt(2 * units) is within 4% of it for 8 to 32 blocks of
// 6 to 64 units at head_dim 64, 128 and 256, and past 32 blocks the CUs bound it
// (8 blocks of 64 units, 8-bit pages: 278 us whole, 89 in 4 pieces, 62 in 11, 77
// in 32).  Sequences of less than 4 units stay whole, and of a few more where
// many blocks would write partials (64 blocks of 4: 32.2 us, 35.0 in two pieces;
// 96 of 6: 41.0 and 37.9; 128 of 6: 41.5 and 40.7, of 8: 49.3 and 45.3).
// More pieces than CUs, in two rounds, where their shorter rounds save 6 units,
// the second start-up and its partials (160 blocks, three pieces: 12 units 67 us
// whole, 78 cut).
constexpr int kMaxPrefillSplit = 32;
constexpr int kPrefillUnit = 128;  // tokens: the largest page, one or two stages
struct PrefillRounds {
  int once, twice;  // pieces per span that fill the CUs once and twice (0: no span is cut)
  __host__ __device__ PrefillRounds(int64_t blocks, int units, int cus) {
    const bool whole = units < 4 || blocks < 1 || blocks > cus || blocks > 32 * ((int64_t)units - 3);
    once = whole ? 0 : cus / (int)blocks;
    twice = whole ? 0 : 2 * cus / (int)blocks;
    if (twice > kMaxPrefillSplit) twice = kMaxPrefillSplit;
    if ((int64_t)units * (twice - 2 * once) <= (int64_t)6 * once * twice) twice = 0;  // not worth it
    // the root of the units, at most once
    int p = 1;
    while (p < once && p < kMaxPrefillSplit && (p + 1) * (p + 1) <= 2 * units) ++p;
    once = p;
  }
};
__host__ __device__ inline int prefill_longest(int units, int64_t blocks, int cus) {
  const PrefillRounds r(blocks, units, cus);
  const int pieces = r.twice > 0 ? r.twice : r.once;
  return (units + pieces - 1) / pieces;
}

// The most pieces a span is cut into there, in sequences of up to `units` units;
// with `zeros` (a mixed batch's dead rows to be written by the grid as well) at
// least as many workgroups per row block as fill the CUs.
__host__ __device__ inline int prefill_split(int units, int64_t blocks, int cus, bool zeros) {
  const PrefillRounds r(blocks, units, cus);
  int p = r.twice > r.once ? r.twice : r.once;
  if (zeros && blocks > 0 && cus / (int)blocks > p) p = cus / (int)blocks;
  return p < kMaxPrefillSplit ? p : kMaxPrefillSplit;
}

// What a wide call's prefill grid may need where it has CUs to fill; with `share`
// (a mixed batch, whose live sequences only the device knows) over any number of
// live sequences.
struct PrefillCut {
  int64_t items = 0;   // most workgroups of a grid of more than its row blocks (0: none is)
  int64_t parts = 0;   // most of them in one that cuts spans: partials
  int64_t blocks = 0;  // most row blocks of such a grid
};
inline PrefillCut prefill_cut(int64_t per_seq, int64_t batch, bool share, int units, int cus) {
  PrefillCut c;
  for (int64_t n = share ? 1 : batch; n <= batch && n * per_seq <= cus; ++n) {
    const int split = prefill_split(units, n * per_seq, cus, share && n < batch);
    if (split < 2) continue;
    const int64_t items = n * per_seq * split;
    c.items = c.items > items ? c.items : items;
    if (prefill_split(units, n * per_seq, cus, false) < 2) continue;
    c.parts = c.parts > items ? c.parts : items;
    c.blocks = n * per_seq;
  }
  return c;
}

struct QuantRowsArgs {
  const uint16_t *values;  // [rows][dim], float_kind
  int64_t rows;
  int dim, bits, group, float_kind;
  uint8_t *codes;          // [rows][ceil(dim/group)*group * bits/8]
  uint16_t *scale, *bias;  // [rows][ceil(dim/group)] f16 bits
};

struct DequantRowsArgs {
  const uint8_t *codes;
  const uint16_t *scale, *bias;
  int64_t rows;
  int dim, bits, group;
  float *out;              // [rows][dim]
};

// Rotate-half RoPE of a fused projection [rows][heads + 2*kv_heads][dim]
// (rows = B*T) into head-major q [B][heads][T][dim], k and v [B][kv_heads][T][dim].
struct RopeArgs {
  const uint16_t *qkv;
  int64_t rows;
  int tokens, heads, kv_heads, dim, float_kind;
  const int32_t *positions;  // [rows]
  const float *inv_freq;     // [dim/2]
  uint16_t *q, *k, *v;
};

hipError_t launch_rope(hipStream_t stream, const RopeArgs &a);

// Device page allocator (pkv_arena.hip).  State words: [0] free pages,
// [1] error bits, header padded to kArenaHeaderWords, then the free stack
// [capacity] and the reference counts [capacity].
constexpr int kArenaHeaderWords = 16;
constexpr int kMaxArenaPools = 128;
constexpr int kArenaOutOfPages = 1, kArenaTableFull = 2, kArenaBadArgument = 4, kArenaCorrupt = 8;

enum class ArenaOp { Reserve, Release, Fork };

struct ArenaArgs {
  int32_t *state;
  int capacity, page_tokens;
  int32_t *table;   // [num_slots][max_pages]
  int max_pages, num_slots;
  int32_t *lens;    // [num_slots]
  const int32_t *slots, *arg;  // per item: slot, and width / kept tokens / fork destination
  int count;
  uint8_t *pools[kMaxArenaPools];  // reserve: copy-on-write in every layer's pool
  int num_pools;
  int64_t page_bytes;
  int32_t *batch_table, *batch_starts, *batch_lens;  // reserve outputs
};

hipError_t launch_arena_init(hipStream_t stream, int32_t *state, int capacity);
hipError_t launch_arena(hipStream_t stream, ArenaOp op, const ArenaArgs &a);
hipError_t launch_quantize_rows(hipStream_t stream, const QuantRowsArgs &a);
hipError_t launch_dequantize_rows(hipStream_t stream, const DequantRowsArgs &a);
hipError_t launch_append(hipStream_t stream, const AppendArgs &a);
hipError_t launch_gather(hipStream_t stream, const GatherArgs &a);
// Streaming read of the listed pages (all heads) by `waves` one-wave
// workgroups; out: waves * 64 words.
hipError_t launch_read_probe(hipStream_t stream, const uint8_t *pool, int64_t num_pages, int64_t page_bytes,
                             const int32_t *ids, int64_t count, int waves, uint32_t *out);
hipError_t launch_copy(hipStream_t stream, uint8_t *pool, int64_t num_pages, int64_t page_bytes,
                       const int32_t *src, const int32_t *dst, int count);
hipError_t launch_attention(hipStream_t stream, const AttnArgs &a);
hipError_t launch_merge(hipStream_t stream, const MergeArgs &a);
// Waves per merge workgroup.
int merge_waves(const MergeArgs &a);
// Query blocks wider than the decode kernel serves (chunked prefill).
hipError_t launch_prefill(hipStream_t stream, const AttnArgs &a);
// Row blocks per (sequence, KV head) and rows per block of the prefill kernel.
int prefill_blocks(const Geo &g, int rows);
int prefill_block_rows(const Geo &g);
// The merges of a wide call in one launch: the decode parts' (`tiers` of
// `tier`) and, with `prefill` (a.pre_cus > 0), the split prefill spans'.
hipError_t launch_tail_merge(hipStream_t stream, const MergeArgs *tier, int tiers, const AttnArgs &a, bool prefill);
int device_cus();
// Resident waves of the attention kernel for this layout and row count on the
// current device (CUs x workgroups per CU); <0 on error.
int attention_waves(const Geo &g, int rows);
// Waves per run of the split for `rows` query rows per KV head (`append`: the
// fused single-token form): a launch of W waves has
// max(1, W / attention_group(rows, append)) runs, each with its partials.
int attention_group(const Geo &g, int rows, bool append);
// Lead tiles the decode split charges per segment for `rows` query rows per KV
// head (more for a launch that fuses the single-token append).
int attention_lead(const Geo &g, int rows, bool append);
// Waves per run and lead tiles of the grouped form every decode shape also has.
int attention_group_waves();
// Column slots (tiles per iteration of a wave) of the shape's kernel.
int attention_slots(const Geo &g, int rows);
int attention_group_lead();
// Whether the split-K decode kernel serves this many rows per KV head (else
// launch_prefill does).
bool decode_serves(const Geo &g, int rows);
// Whether the decode kernel fuses the single-token append for this layout and
// row count (at most 8 rows per KV head).
bool append_fusable(const Geo &g, int rows);
// Decode kernel for <= 4 rows per KV head over quantized pages (head_dim <=
// 128): process-wide; select returns the previous choice.
constexpr int kDecodeMfma = 0, kDecodeValu = 1;
int select_decode_kernel(int kind);
const int32_t *decode_kernel_choice();  // where the choice stands
int decode_kernel();

}  // namespace pkv
