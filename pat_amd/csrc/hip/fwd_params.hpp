// Kernel-argument structures shared by the host launcher and the gfx950 kernels.
#pragma once
#include <cstdint>

#include "pat_amd.h"

namespace pat {

constexpr int kMaxBuckets = 12;    // the reference dispatches 12 tile shapes (static_switch.h:3-66)
constexpr int kWaves = 4;          // waves per split-kernel workgroup
constexpr int kThreads = kWaves * 64;
constexpr int kStepTokens = 32;    // KV tokens one wave consumes per loop iteration
constexpr int kGridX = 1 << 20;     // workgroups per grid.x slice (grid.y counts slices)
constexpr int kMaxTall32Tokens = 64 * 64; // tokens of a tall piece in the 32-row form (an address per lane and 64-token super-step)
constexpr int kMaxChunkPages = 128; // page ids of a chunk: two per lane of a wave
constexpr int kMaxTailTokens = PAT_MAX_TAIL_TOKENS;  // tokens of a tail (the planner's bound)
static_assert(32 * (kMaxTailTokens / 16) <= 2 * 64, "the pages, of 16 tokens and more, of the tails of a wave's 32 rows are two per lane");
// The merge kernel's forms by slots and rows. Launches of up to 8 slots per row: a wave per row, or a half-wave from so many rows.
// Launches of 9 slots and more: where rows are few a workgroup takes a row, a wave of which requests eight rows at once, as many as
// one of the other forms. Whole calls, us (the split kernel is the same in all), a wave per row / the form taken:
//  * 9..32 slots, four waves, every slot requested at once: up to so many slots over all rows. Empty slots are requested too,
//    which has to cost less than the two round trips it saves (merges: 32 rows x 32 slots 5.1 / 3.0, 592 x 10 4.5 / 4.0, 2048 x 14
//    5.6 / 5.0, but 4096 x 18 5.2 / 7.2).
//  * 33..64 slots, eight waves, the same, up to so many slots of 512 bytes (head_dim 64: 256): one request of 16384 tokens in 64
//    pieces 20.9 / 15.9, 96 rows x 41 slots 14.1 / 10.8, 512 x 48 18.6 / 16.2, 768 x 64 (head_dim 64) 16.0 / 14.1; 832 x 45
//    25.9 / 27.2, with the LSEs first 25.7, 1024 x 64 24.4 / 24.5, 23.0.
//  * more, and where that is too many: the LSEs first, then the filled slots only, with eight waves up to so many rows (64 x 72
//    15.6 / 11.2, 528 x 138 21.1 / 14.3), with four up to so many. A workgroup per row costs its launch also where most slots are
//    empty, and many rows keep the chip busy either way: pieces of 32 tokens, one request in 16 of all slots and the others of four
//    filled, head_dim 64, 1536 x 64 22.6 / 19.2, 2048 x 64 16.1 / 13.9, 3072 x 64 19.5 / 18.0, 3072 x 40 16.0 / 15.7, but 4096 x 40
//    18.7 / 19.9, 6144 x 40 24.5 / 27.9, 8192 x 160 40.7 / 45.0, head_dim 128 8192 x 40 43.0 / 48.4; half of the requests of all
//    slots 2048 x 40 27.1 / 25.8, 3072 x 40 36.4 / 36.3, 4096 x 40 45.5 / 46.8, 8192 x 40 88.1 / 93.1.
constexpr int64_t kMergePairsRows = 16384;
constexpr int kMergeWideBatch = 8;
constexpr int kMergeWideSlots = 4 * kMergeWideBatch;
constexpr int64_t kMergeWideMost = 32768;
constexpr int64_t kMergeWide8Most = 28672;
constexpr int64_t kMergeWide8Rows = 768;
constexpr int64_t kMergeWide4Rows = 3072;
enum MergeForm {
  kMergeNone = 0,       // the split kernel writes `out`
  kMergeWave = 1,       // a wave per row
  kMergeHalfWave = 2,
  kMergeWide4All = 3,   // a workgroup per row, four or eight waves: every slot requested at once ...
  kMergeWide8All = 4,
  kMergeWide4 = 5,      // ... the filled ones only
  kMergeWide8 = 6,
};
inline MergeForm merge_form(int64_t rows, int num_slots, int head_dim) {
  const int64_t slots = rows * num_slots;
  if (num_slots <= 8) return rows >= kMergePairsRows ? kMergeHalfWave : kMergeWave;
  if (num_slots <= kMergeWideSlots) return slots <= kMergeWideMost ? kMergeWide4All : kMergeWave;
  if (num_slots <= 2 * kMergeWideSlots && slots * head_dim <= kMergeWide8Most * 128) return kMergeWide8All;
  return rows <= kMergeWide8Rows ? kMergeWide8 : rows <= kMergeWide4Rows ? kMergeWide4 : kMergeWave;
}

// One workgroup's work: a launch record, written once per plan by the record kernel
// (capi_fwd.hip) and read by the split kernel in a single round trip. In memory:
//   RecordHead | int32 seq[max_seqs] | int32 slot[max_seqs] | int32 page[max_pages]
//   (tails: | int32 tail_tokens[max_seqs] | int32 tail_page[max_seqs][tail_pages])
// seq[j] / slot[j]: batch index of the box's j-th sequence and the partial-result slot its rows
// of this piece go to (-1 / -1: no such row); page[i]: physical KV block of the piece's i-th page,
// already clamped to the cache. tail_tokens[j]: tokens of the j-th sequence's tail that this workgroup walks (0: none), on pages
// tail_page[j][..]. Records are record_stride bytes apart (a multiple of 64).
struct RecordHead {
  int32_t tokens;      // KV tokens of this piece; 0: nothing to compute (the workgroup only marks slots empty)
  int32_t rows;        // rows of the box, or of the two boxes of an item (sequences x heads per kv head), <= 16 x tiles
  int32_t mode;        // bits 0-7: 16-row tiles (1 = KV steps split over waves on wave-private tiles,
                       // 2/4/8 = tiles shared through LDS); bit 8: a kv head per wave; bit 9: V read past the caches;
                       // bit 10: a list of `tokens` boxes of one sequence each, seq[i] / slot[i] of box i; page[] holds the boxes' tokens
                       // (list_boxes entries), then their pages (list_pages each)
  int32_t head;        // first kv head this workgroup serves
  int32_t fill_begin;  // slots slot[j] + fill_begin .. slot[j] + fill_end - 1 of every row stay empty:
  int32_t fill_end;    // this workgroup marks them (-inf)
  int32_t pad[2];
};
static_assert(sizeof(RecordHead) == 32, "RecordHead is read as two 16-byte pieces");
constexpr int kRecordModeHeadPerWave = 0x100;
constexpr int kRecordModeStreamV = 0x200;
constexpr int kRecordModeList = 0x400;      // several boxes of one sequence each: see RecordHead
constexpr int kMaxListBoxes = 8;            // (their tokens and pages, two at most for 32 tokens, fit the 64 page entries of a record's first trip)

struct SplitParams {
  const char* records;      // one per workgroup, in launch order
  int32_t record_stride;    // bytes
  int32_t record_max_seqs;  // seq[] / slot[] entries per record
  int32_t record_max_pages; // page[] entries per record
  const void* q;
  const void* k;
  const void* v;
  float* o_part;     // [batch, heads, num_slots, head_dim] fp32, normalised partial outputs
  float* lse_part;   // [batch, heads, num_slots] fp32, natural-log LSE of each partial (-inf = empty)
  int64_t q_stride_b, q_stride_h;              // elements
  int64_t k_stride_page, k_stride_slot, k_stride_h;
  int64_t v_stride_page, v_stride_slot, v_stride_h;
  int32_t heads, group;     // group = heads / kv_heads
  int32_t page_size;
  int32_t num_slots;        // partial-result slots per (sequence, head)
  int32_t total_items;      // workgroups of the launch
  float scale_log2;         // softmax_scale * log2(e)
  uint32_t hpp_magic;       // ceil(2^32 / (page_size / 16)): h / (page_size / 16) == umulhi(h, hpp_magic) for h < 2^16; unused when page_size / 16 is a power of two
  // single-slot launches (every row has one partial slot; no merge kernel follows): the rows go
  // to `out`.
  void* out;         // [batch, 1, heads, head_dim] in the element type
  float* lse_out;    // optional [batch, heads] fp32
  int64_t o_stride_b, o_stride_h;              // elements
  int32_t direct;    // 1: such a launch
  int32_t tall_apart;  // 32-row form: K and V tiles of a super-step handed over apart (see the kernel)
  int32_t stream_v;  // records may ask for V past the caches (host side: picks the kernel instance)
  int32_t waves;     // waves per workgroup (host side: picks the kernel instance)
  int32_t list_boxes; // most boxes of a list workgroup (kRecordModeList), 0: the launch has none
  int32_t list_pages; // ... and pages per box in its record
  int32_t tail_pages; // tails: pages per tail in the records, 0: the launch has none
  int32_t tall_rows; // rows per wave on boxes of 17..64 rows: 32 (32x32x16 tiles) or 16 (host side: picks the kernel instance)
};

// One tile bucket as the record kernel sees it.
struct RecordBucket {
  const int32_t* q_table;
  const int32_t* block_table;
  const int32_t* num_seqs;
  const int32_t* rank;
  const int32_t* kv;
  const int32_t* q_slot; // optional [num_boxes, q_stride]: ordinal of the box among its sequence's boxes
  int32_t q_stride;      // elements between q_table (and q_slot) rows
  int32_t bt_stride;     // elements between block_table rows
  int32_t num_boxes;
  int32_t max_seqs;      // valid q_table columns
  int32_t max_blocks;    // valid block_table columns
  int32_t chunk_tokens;  // KV tokens per workgroup (multiple of 32 and of page_size)
  int32_t chunks;        // workgroups along the KV axis reserved per box
  int32_t item_begin;    // first workgroup of this bucket in the launch
  int32_t row_tiles;     // 16-row tiles per box: 1, 2 or 4
  const int32_t* items;  // [num_items, 2]: boxes served together (-1: no second one), or null: every box by itself
  int32_t num_items;     // work items along the box axis: rows of `items`, or num_boxes
  int32_t heads_per_wg;  // 1, or kWaves: wave w serves kv head h0 + w alone
  int32_t list_boxes;    // 0, or: a workgroup serves so many boxes one after the other (num_items counts such lists)
  const int32_t* tails;  // [num_boxes, max_seqs]: launch bucket << 27 | row of each sequence's tail, or null
  int32_t tail_id;       // a bucket of tails: its place among the launch's buckets, as `tails` numbers them; else -1
};

struct RecordParams {
  char* records;
  int32_t record_stride, record_max_seqs, record_max_pages;
  int32_t num_buckets, total_items, grid_items;   // grid_items: total_items rounded up to the split kernel's grid
  int32_t batch, kv_heads, group, page_size, num_pages;
  int32_t chunks_per_rank;  // slots reserved per box ordinal
  int32_t max_split;
  int32_t list_boxes, list_pages;   // as in SplitParams
  int32_t tail_pages;       // pages per tail in a record; 0: no tails. Buckets of tails have no items, only tables.
  int32_t stream_tokens;    // V tiles of pieces that no other box reads go past the caches (kRecordModeStreamV) where the boxes of
                            // <= 16 rows hold so many tokens between them; negative: nowhere
  RecordBucket bucket[kMaxBuckets];
};

struct MergeParams {
  const float* o_part;
  const float* lse_part;
  const int32_t* num_split_per_seq;
  void* out;
  float* lse_out;           // may be null
  int64_t o_stride_b, o_stride_h;
  int32_t batch, heads, head_dim;
  int32_t chunks_per_rank, num_slots, max_split;
  int32_t kv_heads;
};

}  // namespace pat
