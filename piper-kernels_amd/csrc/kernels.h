// Kernel parameter blocks and launchers shared by the C ABI and the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace piper {

constexpr int kMeanLevels = 4;  // accumulator levels of torch's CPU cascade sum

// The K/V sequence means follow torch's CPU FP32 reduction order (the reference's
// torch.mean(dim=2), piper_attention/reference.py:50, sage/reference.py:89): rows are summed in
// blocks of L = cascade_block_rows(S) rows, L consecutive blocks form a level-1 sum over a
// chunk of L^2 rows, L consecutive level-1 sums form a level-2 sum, and the level-2 sums are
// added in order; trailing rows and unfinished levels are combined at the end as
// ((rows + level 1) + level 2) + level 3.  Every partial starts from +0.0 and every addition
// is one FP32 rounding; the mean is that sum divided by S in FP32.
__host__ __device__ inline int cascade_block_rows(int length) {
  const int ceil_log2 = length > 1 ? 32 - __builtin_clz(static_cast<unsigned>(length - 1)) : 0;
  const int power = ceil_log2 / kMeanLevels > 4 ? ceil_log2 / kMeanLevels : 4;
  return 1 << power;
}

__host__ __device__ inline int cascade_chunks(int length) {  // chunks of L^2 rows, the last may be short
  const long rows = static_cast<long>(cascade_block_rows(length)) * cascade_block_rows(length);
  return static_cast<int>((length + rows - 1) / rows);
}

// Workspace of piper_prepare: the mean partials ([2][batch_heads][chunks + 1][D] floats), then
// the single-pass prep's sync words (an arrival counter per batch-head tensor, a status word;
// the rest is spare, padding to 16 bytes).
inline long prep_partial_bytes(long batch_heads, int length, int head_dim) {
  return 2 * batch_heads * (cascade_chunks(length) + 1) * head_dim * 4;
}
inline long prep_sync_words(long batch_heads) { return 4 * batch_heads + 4; }
// Index of the status word among the sync words (after the 2 * batch_heads arrival counters):
// the number of chunks of the last call that gave up waiting and computed their mean themselves.
inline long prep_status_word(long batch_heads) { return 2 * batch_heads; }

// One 64-key tile record is byte for byte the attention kernel's LDS stage, so it is copied
// with direct global -> LDS loads in 1 KiB pieces: K codes [64][D] in rows of D + 16 bytes,
// V^T codes [D][64] in rows of 80 bytes (the 16 spare bytes per row spread LDS banks), 64
// log2 scales, 64 inverse multipliers, D biased corrections, padded to a KiB multiple.
// Bytes [D, D + 4) (padding of K row 0) hold the tile's K scale; other padding is unspecified.
constexpr int kv_k_stride(int head_dim) { return head_dim + 16; }
constexpr int kv_v_stride() { return 64 + 16; }
constexpr int kv_v_offset(int head_dim) { return 64 * kv_k_stride(head_dim); }
constexpr int kv_log_offset(int head_dim) { return kv_v_offset(head_dim) + head_dim * kv_v_stride(); }
constexpr int kv_inv_offset(int head_dim) { return kv_log_offset(head_dim) + 256; }
constexpr int kv_corr_offset(int head_dim) { return kv_inv_offset(head_dim) + 256; }
constexpr int kv_tile_bytes(int head_dim) { return (kv_corr_offset(head_dim) + 4 * head_dim + 1023) / 1024 * 1024; }

// SageAttention2++ tile record: the same K rows (and K scale in the padding of row 0),
// then FP8 E4M3 V^T codes [D][64] in rows of 80 bytes; no softmax metadata (the V scale is
// per channel and applied in the epilogue).  A whole number of KiB for D = 64 and 128.
constexpr int sage_v_offset(int head_dim) { return 64 * kv_k_stride(head_dim); }
constexpr int sage_tile_bytes(int head_dim) {
  return (sage_v_offset(head_dim) + head_dim * kv_v_stride() + 1023) / 1024 * 1024;
}

// Workgroups of four waves resident per CU, so waves per SIMD, under PIPER_PLAN_THREE_WORKGROUPS.
// D = 128: three (64 numerator registers of a wave leave room for 168 VGPRs per wave).  D = 64: four
// (32 numerator registers; every instantiation fits 128 VGPRs without a spill, five waves' 96 do not,
// and four two-stage rings take 88 KiB of LDS).  Measured at D = 64 against three: B1 H16 S8192
// (1024 query tiles, one round instead of 1.33) 350 -> 301 us, SageAttention2++ 284 -> 256 us; B2 H24
// S8192 (three rounds instead of four) 901 -> 884 us; B4 H16 S4096 causal 214 -> 208 us,
// SageAttention2++ 210 -> 197 us.
constexpr int waves_per_simd(int head_dim) { return head_dim == 64 ? 4 : 3; }

// Workgroups of attention_streams_kernel resident per CU: two double-buffered sets of KS tile records each
// (D = 128: 80 or 160 KiB of the CU's 160; D = 64: 44 or 88).  A key split of 2 or 4 parts takes that kernel
// when its grid then fits the GPU at once; beyond, the workgroups would queue and the parts' partial sums
// cost less than reading the records again for fewer queries.  Unsplit, parts, streams (us, 10-13 of them
// the launching loop's floor): B1 H8 S1024 D64 22.4, 17.7, 13.9 (4); B1 H24 S1024 D64 22.7, 25.8, 18.4
// (2); B1 H16 S1024 D128 30.2, 30.2, 20.4 (2); B1 H16 S2048 53.6, 52.5, 44.7 (2); B2 H12 Sq1000 Sk333 16.6,
// 27.1, 15.6 (2); B1 H4 Sq512 Sk2048 52.4, 23.5, 24.6 (4).
constexpr int stream_workgroups(int head_dim, int streams) {
  return streams == 4 ? 1 : head_dim == 64 ? 3 : 2;
}

// Key streams of a grid whose plan does not choose them (causal Piper Attention, SageAttention2++; both give the
// sequential kernels' bits), from its 128-row query tiles and 64-key tiles: four where that gives at most one
// workgroup per CU, two where that does, and two for causal grids of up to `quarters` quarters of a
// workgroup of 128 rows per CU, whose longest tile sets the time, if the keys are long enough to pay for the
// shorter query tiles' prologues.
// Measured, none against the choice (us without the host): Piper Attention causal B1 H8 S1024 D64 22, 11.6
// (4); B1 H9 S1024 D128 27.5, 21.1 (2); B2 H16 S1531 D128 42, 36.5 (2); B1 H12 S4096 98, 72 (2); B1 H8 S8192
// 198, 177 (2); B1 H2 S32768 734, 668 (2).  At the line, D = 128: S1024 (16 key tiles) 384 query tiles 30.8,
// 29.7, not taken 448 31.4, 33.7; S1536 432 tiles 41.9, 40.5, not 504 42.1, 46.8; S2048 448 tiles 53.1, 50.3,
// not 512 54.0, 55.8; S3072 not 504 75.7, 76.9; S4096 512 tiles 98.9, 95.4, not 768 114, 129.  D = 64: 512 tiles
// of S1024 23.1, 23.3, of S2048 40.7, 33.9.  SageAttention2++ B1 H8 S1024 D64 18.2, 11.9 (4); B1 H16 S1024 D128
// 24.3, 21.0 (2); B1 H24 Sq256 Sk16384 268, 166 (4); B1 H1 S8192 140, 87 (4); B1 H2 S6000 D64 84.6, 67.5 (2);
// causal B1 H16 S2048 43.1, 36.6 (2); B1 H32 S1024 D128 26.0, 22.5 (2); B1 H1 S16384 276, 230 (2); not taken: B1 H16 S2048
// 42.9, 45.1, causal B2 H16 S1531 36.8, 38.8.
inline int small_grid_streams(bool sage, bool causal, int head_dim, long tiles, int key_tiles, int cus) {
  if (key_tiles < 4) return 1;
  if (4 * tiles <= cus) return 4;
  if (2 * tiles <= cus) return 2;
  if (!causal || key_tiles < 16) return 1;
  const int quarters = sage ? 4 : head_dim == 64 || key_tiles >= 64 ? 8 : key_tiles >= 24 ? 7 : 6;
  return 4 * tiles <= static_cast<long>(quarters) * cus ? 2 : 1;
}

struct InputTensor {
  const void* data;  // 16-bit floats; the head_dim axis is contiguous
  long stride_batch;  // element strides
  long stride_head;
  long stride_seq;
};

struct MeanParams {
  InputTensor key;
  InputTensor value;
  // [tensors][batch_heads][chunks + 1][D]: the level-1 sum of each chunk of L^2 rows (for a
  // short last chunk, the sum of its complete L-row blocks), then the sum of the trailing
  // length % L rows; SageAttention2++'s V slots hold per-chunk max |v| instead
  float* partials;
  float* key_mean;   // [batch_heads][D]
  float* value_mean; // [batch_heads][D]
  int batch_heads;
  int heads;
  int length;  // key length
  int block_rows;  // L = cascade_block_rows(length)
  int chunks;      // cascade_chunks(length)
  int tensors; // 1 = K only (causal), 2 = K and V
  // 1: the V statistic is the per-column max of |v| (SageAttention2++), finalised into
  // value_scale = amax / 2.25 + 1e-7; 0: the V sum, finalised into value_mean
  int value_absmax;
  float* value_scale;  // [batch_heads][D] (value_absmax only)
  uint32_t* status;    // the prep's give-up count, cleared by the finalisation (NULL: none)
};

// Scales stored per quantisation block: one per thread group of the reference's per_thread
// granularity (8 per 32-row Q block, 4 per 64-row K block); per-block quantisation repeats its
// one scale in every slot, so the attention kernel reads both the same way.
constexpr int kQueryScaleSlots = 8;
constexpr int kKeyScaleSlots = 4;

// Both operators' prep quantisation.  SageAttention2++ has no query blocks and no value means: it
// quantises K (per 64-row block, after K smoothing) and V (FP8 per channel) into its own tile records.
struct QuantParams {
  InputTensor query;
  InputTensor key;
  InputTensor value;
  int batch_heads;
  int heads;
  int query_length;
  int key_length;
  int sq32;
  int sk64;
  int nqb;
  int nkb;
  int q_blocks_wg;  // workgroups (4 units each) per unit kind
  int k_blocks_wg;
  int v_blocks_wg;
  int center_value;
  int per_thread;  // 1: Q/K scales per thread group (per_thread); 0: one per block (per_warp)
  const float* key_mean;
  const float* value_mean;
  int8_t* query_code;
  float* query_scale;
  float* key_scale;
  float* value_scale;  // Piper Attention's per-key scales (SageAttention2++'s per channel: MeanParams)
  uint8_t* kv_tiles;  // [batch_heads][nkb][kv_tile_bytes(D) or sage_tile_bytes(D)] (layout in piper_mi355x.h)
};

// Order of a causal longest-first grid whose plan leaves it open: across heads while all K/V tile
// records fit the 256 MiB last-level cache, head by head beyond (then only a few heads' records are
// live at a time).  Measured, head by head against across heads, Piper Attention at D = 128: B2 H16
// S1531 48.4 -> 41.8 us, B1 H32 S4096 168 -> 126, B1 H24 S16384 (126 MB of records) 1409 -> 1302, B1 H42
// S20000 (269 MB) 3866 -> 3765, B1 H48 S24000 (369 MB) 5693 -> 5873, B1 H40 S32768 (419 MB) 8605 -> 9065;
// batch-heads not divisible by 8, B1 H12 S20000 1212 -> 1015; D = 64, B4 H40 S8192 (231 MB) 1709 ->
// 1501; SageAttention2++ B1 H24 S4096 143 -> 95, B1 H10 S16384 678 -> 467.
constexpr long kAcrossHeadsBytes = 256L << 20;
inline bool order_across_heads(long batch_heads, long key_tiles, int tile_bytes) {
  return batch_heads * key_tiles * tile_bytes <= kAcrossHeadsBytes;
}

struct AttnParams {
  const int8_t* query_code;
  const float* query_scale;
  const float* key_scale;
  const uint8_t* kv_tiles;
  const float* value_mean;
  void* output;
  int batch_heads;
  int query_length;
  int key_length;
  int sq32;
  int sk64;
  int nqb;
  int nkb;
  int query_tiles;  // workgroup query tiles per (batch, head)
  float scale_log2e;
  int causal_forward;  // causal grids: 1 = query tiles in forward order, 0 = longest first
  int xcd_remap;       // 1 = consecutive workgroups of a head share an XCD, 0 = hardware order
  int across_heads;    // causal, longest first: 1 = across heads, 0 = head by head
  // Fused query quantisation: each wave quantises its own 32-row query block from `query`
  // (query_code and query_scale are then unused).
  int fused_query;
  // Q/K scale granularity: 1 = per thread group (query scale slot n % 8 of the row's block, the
  // tile's four K group scales), 0 = per block (slot 0, one K scale)
  int per_thread;
  int query_bf16;
  int heads;
  InputTensor query;
  // Key-range split (non-causal, PIPER_PLAN_THREE_WORKGROUPS): query tiles [0, whole_tiles), whole
  // rounds of resident workgroups, run unsplit; the key tiles of each later query tile are cut into
  // key_parts ranges of part_tiles tiles, one workgroup per range, which writes its unnormalised
  // numerator (x 255), denominator and reference maximum to `partials` ([key_parts][split rows][D]
  // floats, then [key_parts][split rows] float2 (den, mref)); attention_merge_kernel combines them.
  // The split rows are the output's rows from split_row0 on (rows of [batch_heads * query_length]).
  // key_parts = 1: no split.
  int key_parts;
  int part_tiles;
  int whole_tiles;
  long split_row0;
  float* partials;
  // Key streams (attention_streams_kernel): 2 or 4 waves of a workgroup share its queries; 1: none.
  int key_streams;
  // Work-queue plan (three workgroups per CU, no key-range split): a persistent grid takes query
  // tiles from queue_xccs queues of consecutive logical ids, counters in `queue` (zero before the
  // launch).  queue_xccs = 0: the hardware dispatches one workgroup per query tile.
  int queue_xccs;
  int queue_workers;  // the persistent grid (at most waves_per_simd workgroups per CU)
  float score_multiplier;  // scale_log2e * 2^26 (kScoreUnit), exact: the logits' multiplier per query scale
  uint32_t* queue;
};

__host__ __device__ inline long split_rows(const AttnParams& p) {
  return static_cast<long>(p.batch_heads) * p.query_length - p.split_row0;
}

// How a plan of `parts` key parts runs a grid on a device of `cus` compute units: only the query tiles
// beyond whole rounds of resident workgroups are split, no part is empty, and two or four parts of a grid
// whose workgroups then all fit the GPU at once are key streams, which need no partial sums.  The launch
// and the workspace's size both come from here.
struct KeySplit {
  int parts;         // key ranges of a split query tile (1: nothing is split)
  int streams;       // key streams (1: none)
  int part_tiles;    // key tiles per range
  long whole_tiles;  // query tiles that run unsplit, before the split ones
  long row0;         // the first output row (of batch_heads * query_length) of the split tiles
  long bytes;        // workspace: the split rows' partial sums, D numerators and two floats per part
};

inline KeySplit key_split(long batch_heads, long query_length, int key_tiles, int head_dim, int parts, int cus) {
  constexpr int kRows = 128;  // query rows of a workgroup
  KeySplit k{1, 1, key_tiles, 0, 0, 0};
  if (parts <= 1) return k;
  const long per_head = (query_length + kRows - 1) / kRows;
  const long tiles = per_head * batch_heads;
  const long slots = static_cast<long>(waves_per_simd(head_dim)) * (cus > 1 ? cus : 1);
  k.part_tiles = (key_tiles + parts - 1) / parts;
  k.whole_tiles = tiles / slots * slots;
  k.row0 = k.whole_tiles / per_head * query_length + k.whole_tiles % per_head * kRows;
  if ((parts == 2 || parts == 4) && parts * tiles <= static_cast<long>(stream_workgroups(head_dim, parts)) * cus) {
    k.streams = parts;
  } else if (k.whole_tiles < tiles) {
    k.parts = (key_tiles + k.part_tiles - 1) / k.part_tiles;
    if (k.parts > 1) k.bytes = k.parts * (batch_heads * query_length - k.row0) * (head_dim + 2) * 4;
  }
  return k;
}

// The work-queue plan's counters: one per XCC, at most kQueueCounters.
constexpr int kQueueCounters = 64;
constexpr long kQueueBytes = kQueueCounters * 4;

struct SageParams {
  const uint8_t* kv_tiles;
  const float* value_scale;  // [batch_heads][D]
  void* output;
  InputTensor query;
  int query_bf16;
  int heads;
  int batch_heads;
  int query_length;
  int key_length;
  int nkb;
  int query_tiles;  // workgroup query tiles per (batch, head)
  float scale_log2e;
  int causal_forward;
  int xcd_remap;
  int across_heads;
  int per_thread;  // Q/K scales per thread group (the tile's four K slots, per-row-group Q scales)
  int key_streams;  // sage_streams_kernel: 2 or 4 waves of a workgroup share its queries; 1: none
  int fp16_partials;  // round each block's FP8 product to FP16 (the reference's arithmetic)
};

constexpr int kPrepSpinLimit = 1 << 20;  // polls of a waiting single-pass chunk (with s_sleep): about a second

// The GPU the prep runs on, and the single-pass prep's wait bound.
struct PrepDevice {
  int cus;         // compute units
  int xccs;        // XCCs (accelerator complex dies) the workgroups are dealt over, round-robin
  int spin_limit;  // polls of a waiting chunk before it computes the mean itself (0: at once)
};

// The single-pass prep keeps each chunk of a batch-head tensor resident until the tensor's last
// chunk has arrived, so all of a tensor's chunks must fit in one XCC at once: at least four
// workgroups per CU (the kernel's occupancy allows more) on cus / xccs CUs.
__host__ __device__ inline bool single_pass_resident(int chunks, int cus, int xccs) {
  return xccs > 0 && cus >= xccs && chunks <= 4 * (cus / xccs);
}

hipError_t launch_prep(bool bf16, int head_dim, const MeanParams& mp, const QuantParams& qp, const PrepDevice& dev,
                       hipStream_t stream);
hipError_t launch_sage_prep(bool bf16, int head_dim, const MeanParams& mp, const QuantParams& qp, const PrepDevice& dev,
                            hipStream_t stream);
hipError_t launch_sage_attention(int head_dim, bool causal, int out_dtype, int waves, const SageParams& sp,
                                 hipStream_t stream);

// out_dtype: 0 = fp16, 1 = bf16, 2 = fp32.  waves: 8 or 4 query waves per workgroup (two waves per
// SIMD), or 3 for three 4-wave workgroups per CU.
hipError_t launch_attention(int head_dim, bool causal, int out_dtype, int waves, const AttnParams& ap,
                            hipStream_t stream);

}  // namespace piper
