// Internal launch interface between the C-ABI host layer and the gfx950 kernels.
// Plain structs and pointers only; nothing here is exported from the library.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ringattn_jobs.h"

namespace ringattn {

constexpr int kWalkM = 256;   // query rows per workgroup of ring_walk_kernel (8 waves x 32 rows)
constexpr int kSplitM = 32;   // query rows per workgroup of ring_split_kernel
constexpr int kPairM = 128;  // query rows per workgroup of ring_pair_kernel
constexpr int kThinM = 128;  // query rows per workgroup of thin::ring_walk_kernel
constexpr int kDealtM = 32;  // query rows per workgroup of dealt::ring_walk_kernel
constexpr int kMaxParts = 64; // partial slots a merge can combine
constexpr int kComputeUnits = 256, kXcds = 8;

// One unit of block-attention work as the host layer lists it: the queries
// [q_start, q_start + q_len) of every head against the keys/values
// [kv_start, kv_start + kv_len) of the matching KV head -- the body of one ring step of one
// rank (csrc/ring_attention.cu:456-470,531-610: rank r at step s works on the KV chunk of rank
// (r + s) mod P).  Row numbers are local to a head's [S, D] slab and need not be multiples of
// any tile size.  The normalised partial O and the partial LSE of the item go to partial slot
// `slot`, at the rows of its queries.
struct WorkItem {
  int q_start, q_len;
  int kv_start, kv_len;
  int diag_off;  // < 0: every key is visible.  >= 0: key kl (local to the KV range) is visible
                 // to query ql (local to the query range) iff kl <= ql + diag_off; then
                 // diag_off + q_len <= kv_len
  int slot;
  int pad0, pad1;
};

// What the attention kernel runs: a SEGMENT is a range of query rows (of every head) together with
// ALL the key ranges it meets -- the ring steps of the reference's step loop
// (csrc/ring_attention.cu:456-620) for those rows.  One workgroup owns kWalkM rows of a segment,
// keeps their Q in registers and walks the segment's items, as the reference's CTA walks the
// ring steps (:439-443,456), emitting one (partial O, partial LSE) per item.
struct SegItem {
  int kv_start, kv_len;
  int diag_off;         // as in WorkItem, relative to the first row of the segment
  int part_bh_stride;   // rows between consecutive heads in this item's partial block
  int64_t part_base;    // row (in the partial buffers) of the segment's first row of head 0
  int slot;             // ring step: the entry of a row's run with row-major partials, else for inspection only
  int part_row_mul;     // 0: the partial of row r lives at row r of the buffers; n > 0: at entry n r + slot (a row's
                        // steps next to each other, n of them)
};
static_assert(sizeof(SegItem) == 32, "SegItem is read as two 16-byte scalar loads");

struct Segment {
  int q_start, q_len;
  int item_begin, item_count;  // slice of the SegItem table, in ascending ring-step order
  int last_item;               // index (within the slice) of the item to run last, -1: table order.
                               // A masked (diagonal) item runs last: its length differs per q tile,
                               // and the q tiles that share a KV chunk in L2 stay in step until then.
  int reverse_tiles;           // the q tiles with the most visible keys are scheduled first
  int pad0, pad1;
};
static_assert(sizeof(Segment) == 32, "Segment is read as two 16-byte scalar loads");

// What a workgroup does with the softmax state (max, sum, acc-O) of its rows between the KV chunks it walks.
enum BlockMode {
  kBlockPartials = 0,        // per chunk: emit the normalised partial (O, LSE), reset the state
  kBlockPartialsMerged = 1,  // per chunk: the same partial, merged into out / lse.  ring_walk_kernel merges it on the spot;
                             // ring_walk64_kernel emits it to o_part / lse_part and merges after the last chunk
  kBlockCarryState = 2,      // carry the state across the chunks, as the reference's CTA does across its ring
                             // steps (csrc/ring_attention.cu:439-443,597), and write out / lse once: no partials
};

struct BlockArgs {
  const void* q;       // [BH, S, D] storage dtype
  const void* k;       // [batch * heads / kv_group, S, D]
  const void* v;       // [batch * heads / kv_group, S, D]
  void* o_part;        // partial O rows (normalised), fp32 or fp16 (half_partials); indexed by SegItem::part_base
  float* lse_part;     // partial LSE rows (natural log), same row numbering; both unused with kBlockCarryState
  void* out;           // unless kBlockPartials: [BH, S, D] storage dtype
  float* lse;          // unless kBlockPartials: [BH, S]; may be NULL with kBlockCarryState
  const Segment* segs; // device arrays; both NULL: the launch has the one segment and the one item below, which then come
  const SegItem* items;  // with the kernel arguments and not from memory
  int64_t bh_stride;   // elements between heads of q and out (= S * D)
  int64_t kv_bh_stride;      // elements between heads of k and v
  int S;               // rows per head of q, out and lse
  int q_tiles_max;     // kWalkM-row q tiles of the longest segment (grid dimension)
  int n_segs;
  int BH;              // batch * heads
  Divisor by_group;    // query heads per KV head: head bh of all batch entries reads K and V of head bh / that
  float scale_log2;    // softmax_scale * log2(e)
  int half_partials;   // partial O stored as fp16 instead of fp32
  int mode;            // BlockMode
  int causal;          // some item is masked
  Divisor by_q_tiles;  // q_tiles_max, and the jobs: job_grid
  JobMap map;
  int few;             // see job_grid
  Divisor by_heads;    // BH
  int second_lap;      // see lap_order in ringattn_device.h
  Segment one_seg;
  SegItem one_item;
};

// Workgroups of a launch over n_segs segments of q_tiles_max q tiles each, for every head (decode_job in ringattn_device.h is the other
// half of this).
//
// A launch of no more workgroups than there are compute units has all of them running at once, so their order is no matter, and where
// heads and XCDs divide each other workgroup b can be tile b / BH of head b mod BH: heads lie on the XCDs as job_map lays them, and the
// place of a workgroup is one multiplication.  us a launch before and after, one behind the other: d = 64, 4 ranks x 128 tokens 5.25, 5.10, 4 heads x
// 64 4.30, 4.18; d = 128, 2 x 256 5.94, 5.81, 2048 causal 11.40, 11.28; a step of 4 x 512, d = 64, 6.01, 5.92; from 20 us on the same.
inline int64_t job_grid(BlockArgs& a, bool masked) {
  a.by_q_tiles = divisor(a.q_tiles_max > 0 ? a.q_tiles_max : 1);
  const int64_t jobs = (int64_t)a.BH * a.n_segs * a.q_tiles_max;
  a.few = jobs <= kComputeUnits && (a.BH % kXcds == 0 || kXcds % a.BH == 0);
  if (a.few) {
    a.by_heads = divisor(a.BH);
    return jobs;
  }
  return job_map(a.map, a.BH, (int64_t)a.n_segs * a.q_tiles_max, masked);
}

// Merge of (O, LSE) partials into the final O (storage dtype) and LSE, for row ranges of every
// head: a region covers rows [start, start + len) and reads the slots whose bit is set in `active`.
struct MergeRegion {
  int start, len;
  uint64_t active;
};
static_assert(sizeof(MergeRegion) == 16, "MergeRegion is read as one 16-byte scalar load");

struct MergeArgs {
  const void* o_parts;    // [slots, heads * S, D] fp32, or fp16 with half_partials
  const float* lse_parts; // [slots, heads * S]
  void* out;              // [heads * S, D] storage dtype
  float* lse;             // [heads * S]
  const MergeRegion* regions;  // device array of n_regions entries, one grid row each; NULL: `single`
  MergeRegion single;
  int n_regions;          // 1 with `single`
  int max_len;            // longest region (grid columns)
  int heads;              // batch * heads: every region is merged for each of them
  int S;                  // rows per head
  int64_t part_stride_rows;  // rows between consecutive slots (>= heads * S)
  int64_t part_rows;         // rows of partials the launch reads, all regions and slots together
  int half_partials;
  int slot0_last;         // 1: slot 0, the masked step of a causal plan, is merged after the others, as the attention kernels walk it
  int row_mul;            // 0: slot-major partials as above; n > 0: [heads * S, n, D] / [heads * S, n], a row's slots adjacent
};

// dtype: 0 = fp16, 1 = bf16.  Return hipSuccess or the launch error.
// The walks of a launch, for what ring_walk_kernel makes of their number and lengths.
struct Walks {
  int tiles = 0;        // 256-row q tiles of a head that there are (the grid has as many for every segment)
  int longest = 0;      // 32-key tiles of the longest
  bool uneven = false;  // they differ in length
  bool masked = false;  // ... by a causal diagonal, so that those of a segment come longest first
};
hipError_t launch_walk(BlockArgs a, const Walks& walks, int dtype, int dim, hipStream_t stream);  // ring_walk_kernel, any BlockMode
// its kBlockPartialsMerged, the grid laid out (ringattn_steps.hip)
hipError_t launch_steps(const BlockArgs& a, unsigned grid, int dtype, int dim, hipStream_t stream);
// the same at d = 64 for launches that leave compute units idle, the ring steps apart (a.q_tiles_max counts tiles of kThinM rows)
hipError_t launch_thin(BlockArgs a, int dtype, hipStream_t stream);
// the same, kBlockPartials only, for launches of a few row tiles (a.q_tiles_max counts tiles of kDealtM rows)
hipError_t launch_dealt(BlockArgs a, int dtype, hipStream_t stream);
// ring_walk64_kernel: the carried-state forward at d = 128 with 64 query rows per wave; only for tables that
// walk64_takes() accepts
hipError_t launch_walk64(BlockArgs a, int dtype, int dim, hipStream_t stream);
// ring_split_kernel: kSplitM query rows per workgroup (a.q_tiles_max counts tiles of that many rows), the keys split over
// its waves (eight; `many_waves`, d = 64 only: sixteen), `columns` of V and O (32, 64 or all) in a workgroup; kBlockCarryState
hipError_t launch_split(BlockArgs a, int dtype, int dim, bool many_waves, int columns, hipStream_t stream);
// the same with the ring steps apart, kBlockPartials and kBlockPartialsMerged (which has all columns); eight waves
hipError_t launch_split_steps(BlockArgs a, int dtype, int dim, int columns, hipStream_t stream);
// either with fewer columns than all, the grid laid out
hipError_t launch_split_columns(const BlockArgs& a, unsigned grid, int dtype, int dim, bool many_waves, int columns, hipStream_t stream);
// ring_pair_kernel: kPairM query rows per workgroup (a.q_tiles_max counts tiles of that many rows), the keys dealt to two
// pairs of waves; kBlockCarryState, tables that CarryCosts::add finds fit for it
hipError_t launch_pair(BlockArgs a, int dtype, int dim, hipStream_t stream);
hipError_t launch_merge(const MergeArgs& a, int dtype, int dim, hipStream_t stream);

}  // namespace ringattn
