// Host side of the C ABI declared in include/ringattn.h: parameter validation, plan and
// workspace lifetime, the ring step loop over P virtual ranks, optional hipGraph replay.
// It replaces the host functions of the reference -- set_params_fprop
// (csrc/ring_attention.cu:361-395), run_ring_fwd (:669-704) and ring_attention (:706-722).
#include "ringattn.h"
#include "ringattn_kernels.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <unordered_set>
#include <vector>

namespace {

// Live plan handles.  A handle is valid only while it is in this set, so a second
// destroy (or a garbage pointer) is reported instead of touching freed memory.
std::mutex g_plans_mu;
std::unordered_set<const void*> g_plans;

thread_local int g_last_hip_error = 0;

inline int hip_fail(hipError_t e) {
  g_last_hip_error = (int)e;
  return RINGATTN_ERR_HIP;
}
#define RA_HIP(expr)                          \
  do {                                        \
    hipError_t e__ = (expr);                  \
    if (e__ != hipSuccess) return hip_fail(e__); \
  } while (0)

constexpr float kLog2e = 1.4426950408889634f;

struct Derived {
  int start[RINGATTN_MAX_NPES + 1] = {};  // rank r owns rows [start[r], start[r+1]) of every head
  int max_len = 0;
  bool zigzag = false;  // causal ring over the zigzag layout (without the mask the layouts coincide)
  int64_t S = 0;
  int64_t BH = 0;
  int64_t kv_BH = 0;
  int64_t rows = 0;  // BH * S
  float scale = 0.f;
};

// All checks that need no GPU.  Mirrors what the reference leaves unchecked: its kernel
// has no tail predication (csrc/ring_attention.cu:143-145) and is instantiated for
// dim 64 only (:707-710); here unsupported shapes are refused instead of mis-computed.
int validate(const ringattn_params* p, Derived* d) {
  if (!p) return RINGATTN_ERR_NULL;
  if (p->npes < 1 || p->npes > RINGATTN_MAX_NPES) return RINGATTN_ERR_NPES;
  if (!p->h_seqlen) return RINGATTN_ERR_NULL;
  if (p->dim != 64 && p->dim != 128) return RINGATTN_ERR_DIM;
  if (p->dtype != RINGATTN_DTYPE_FP16 && p->dtype != RINGATTN_DTYPE_BF16) return RINGATTN_ERR_DTYPE;
  if (p->batch < 1 || p->heads < 1) return RINGATTN_ERR_SHAPE;
  if (p->kv_heads < 0 || (p->kv_heads > 0 && p->heads % p->kv_heads != 0)) return RINGATTN_ERR_SHAPE;
  if (p->layout != RINGATTN_LAYOUT_CONTIGUOUS && p->layout != RINGATTN_LAYOUT_ZIGZAG) return RINGATTN_ERR_SHAPE;
  // any positive length (the zigzag layout halves it, so even there); multiples of
  // RINGATTN_TILE waste no part of a tile
  const int granule = p->layout == RINGATTN_LAYOUT_ZIGZAG ? 2 : 1;
  int64_t S = 0;
  int max_len = 0;
  for (int r = 0; r < p->npes; ++r) {
    const int c = p->h_seqlen[r];
    if (c <= 0 || c % granule != 0) return RINGATTN_ERR_SEQLEN;
    S += c;
    if (c > max_len) max_len = c;
  }
  const int64_t BH = (int64_t)p->batch * p->heads;
  if (S > INT32_MAX / 2 || BH > INT32_MAX / 2) return RINGATTN_ERR_SHAPE;
  if (BH * p->npes * p->npes > (int64_t)INT32_MAX / 64) return RINGATTN_ERR_SHAPE;  // grid size
  if (BH * S > (int64_t)1 << 40) return RINGATTN_ERR_SHAPE;
  if (!std::isfinite(p->softmax_scale)) return RINGATTN_ERR_SHAPE;
  if (d) {
    d->start[0] = 0;
    for (int r = 0; r < p->npes; ++r) d->start[r + 1] = d->start[r] + p->h_seqlen[r];
    d->max_len = max_len;
    d->zigzag = p->layout == RINGATTN_LAYOUT_ZIGZAG && p->causal;
    d->S = S;
    d->BH = BH;
    d->kv_BH = p->kv_heads > 0 ? (int64_t)p->batch * p->kv_heads : BH;
    d->rows = BH * S;
    d->scale = p->softmax_scale > 0.f ? p->softmax_scale : 1.0f / std::sqrt((float)p->dim);
  }
  return RINGATTN_OK;
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

inline bool half_partials(const ringattn_params& p) { return (p.flags & RINGATTN_FLAG_HALF_PARTIALS) != 0; }
inline bool step_partials(const ringattn_params& p) { return (p.flags & RINGATTN_FLAG_STEP_PARTIALS) != 0; }
inline bool row_partials(const ringattn_params& p) { return (p.flags & RINGATTN_FLAG_ROW_PARTIALS) != 0; }

inline ringattn::WorkItem make_item(int q_start, int q_len, int kv_start, int kv_len, int diag_off, int slot) {
  ringattn::WorkItem w;
  w.q_start = q_start;
  w.q_len = q_len;
  w.kv_start = kv_start;
  w.kv_len = kv_len;
  w.diag_off = diag_off;
  w.slot = slot;
  w.pad0 = w.pad1 = 0;
  return w;
}

// The work of virtual rank r at ring step s: it visits the KV of rank j = (r + s) mod P
// (csrc/ring_attention.cu:463,531,615).  Partials go to slot s.
//   no mask            : all queries of r against all keys of j;
//   causal, contiguous : j > r nothing, j == r diagonal, j < r everything;
//   causal, zigzag     : rank r holds a low half (sequence position r) and a high half
//       (position 2P-1-r) back to back.  The low queries see the low keys of j <= r; the high
//       queries see every low half and the high halves of j >= r.  So: j < r, all queries of
//       r against the low half of j; j == r, the plain diagonal over the whole chunk (its
//       low half precedes its high half in the sequence too); j > r, the high queries of r
//       against the whole chunk of j.  Every rank does the same amount of work.
void append_items(std::vector<ringattn::WorkItem>& out, const Derived& d, int P, bool causal, int r, int s) {
  const int j = (r + s) % P;
  const int q0 = d.start[r], ql = d.start[r + 1] - q0;
  const int k0 = d.start[j], kl = d.start[j + 1] - k0;
  if (!causal) {
    out.push_back(make_item(q0, ql, k0, kl, -1, s));
  } else if (j == r) {
    out.push_back(make_item(q0, ql, k0, kl, 0, s));
  } else if (!d.zigzag) {
    if (j < r) out.push_back(make_item(q0, ql, k0, kl, -1, s));
  } else {
    if (j < r) out.push_back(make_item(q0, ql, k0, kl / 2, -1, s));
    else out.push_back(make_item(q0 + ql / 2, ql / 2, k0, kl, -1, s));
  }
}

// A SEGMENT: rows of one rank that meet the same ring steps, with those steps' key ranges in
// ascending step order -- what one workgroup of the attention kernel walks (the reference's CTA
// walks the steps of its rows the same way, csrc/ring_attention.cu:456-620).  Contiguous
// layouts have one segment per rank; a zigzag rank has two (its low half sees fewer steps).
struct HostSegment {
  int start = 0, len = 0;
  std::vector<ringattn::WorkItem> items;  // restricted to the segment: q_start = start, q_len = len
  uint64_t active = 0;                    // the steps (partial slots) of the items
  int64_t tile_work = 0;                  // keys the busiest q tile of the segment visits
};

void rank_segments(std::vector<HostSegment>& out, const Derived& d, int P, bool causal, int r) {
  std::vector<ringattn::WorkItem> all;
  for (int s = 0; s < P; ++s) append_items(all, d, P, causal, r, s);
  const int q0 = d.start[r], q1 = d.start[r + 1];
  std::vector<int> cut{q0, q1};
  if (d.zigzag) cut.push_back(q0 + (q1 - q0) / 2);
  for (const auto& w : all) {
    cut.push_back(w.q_start);
    cut.push_back(w.q_start + w.q_len);
  }
  std::sort(cut.begin(), cut.end());
  cut.erase(std::unique(cut.begin(), cut.end()), cut.end());
  for (size_t i = 0; i + 1 < cut.size(); ++i) {
    HostSegment sg;
    sg.start = cut[i];
    sg.len = cut[i + 1] - cut[i];
    for (const auto& w : all) {
      if (w.q_start > sg.start || sg.start + sg.len > w.q_start + w.q_len) continue;
      ringattn::WorkItem x = w;
      x.q_start = sg.start;
      x.q_len = sg.len;
      if (w.diag_off >= 0) x.diag_off = w.diag_off + (sg.start - w.q_start);
      sg.items.push_back(x);
      sg.active |= (uint64_t)1 << w.slot;
      sg.tile_work += x.diag_off >= 0 ? std::min<int64_t>(x.kv_len, (int64_t)x.diag_off + sg.len) : x.kv_len;
    }
    if (!sg.items.empty()) out.push_back(sg);
  }
}

// All segments of a forward, busiest first: the attention kernel's workgroups are dispatched in
// this order, so the launch ends on its shortest ones.
std::vector<HostSegment> forward_segments(const Derived& d, int P, bool causal) {
  std::vector<HostSegment> segs;
  for (int r = 0; r < P; ++r) rank_segments(segs, d, P, causal, r);
  std::stable_sort(segs.begin(), segs.end(),
                   [](const HostSegment& x, const HostSegment& y) { return x.tile_work > y.tile_work; });
  return segs;
}

// What the forward that carries the softmax state walks.  The state runs from one ring step to the next, so a step's
// boundary means nothing to it, and the key ranges that lie next to each other in memory are walked as one: without a
// mask every row sees every key (one segment of all rows, one range of all keys), a causal ring in the contiguous layout
// is causal attention over the whole sequence (one segment, one masked range), a zigzag rank's high half sees the
// chunks of the ranks after it as one range.  Fewer, longer ranges: no q tile ends at a rank's end (ranks of 128 rows
// filled half a tile), all q tiles of a head walk the keys in the same order and meet in L2, and ranks whose lengths
// are no multiples of a key tile no longer break the walk up.
std::vector<HostSegment> walk_segments(const Derived& d, int P, bool causal) {
  if (!causal || !d.zigzag) {
    HostSegment sg;
    sg.len = (int)d.S;
    sg.items.push_back(make_item(0, sg.len, 0, sg.len, causal ? 0 : -1, 0));
    sg.active = 1;
    sg.tile_work = d.S;
    return {sg};
  }
  std::vector<HostSegment> segs = forward_segments(d, P, causal);
  for (auto& sg : segs) {
    std::sort(sg.items.begin(), sg.items.end(),
              [](const ringattn::WorkItem& x, const ringattn::WorkItem& y) { return x.kv_start < y.kv_start; });
    std::vector<ringattn::WorkItem> joined;
    for (const auto& w : sg.items) {
      if (!joined.empty() && w.diag_off < 0 && joined.back().diag_off < 0 &&
          joined.back().kv_start + joined.back().kv_len == w.kv_start)
        joined.back().kv_len += w.kv_len;
      else
        joined.push_back(w);
    }
    sg.items = joined;
  }
  return segs;
}

// Workspace of a forward that keeps per-step partials (RINGATTN_FLAG_STEP_PARTIALS; none
// otherwise): one partial block [batch*heads, len] rows per (segment, item) -- only the
// (rank, step) pairs the mask leaves visible -- partial O of every block first (fp32, or fp16
// with RINGATTN_FLAG_HALF_PARTIALS), then the fp32 partial LSEs.
int64_t partial_rows_of(const std::vector<HostSegment>& segs, const Derived& d) {
  int64_t rows = 0;
  for (const auto& sg : segs) rows += (int64_t)sg.items.size() * d.BH * sg.len;
  return rows;
}

size_t workspace_bytes_of(const ringattn_params* p, const Derived& d) {
  if (!step_partials(*p)) return 0;
  const size_t o_elem = half_partials(*p) ? 2 : 4;
  const int64_t rows = partial_rows_of(forward_segments(d, p->npes, p->causal != 0), d);
  return (size_t)rows * ((size_t)p->dim * o_elem + sizeof(float));
}

}  // namespace

// ---- which kernel runs a launch that carries the softmax state ---------------------------------------------------------
// The keys an R-row q tile of `seg` visits, in 32-key tiles: what a launch costs is the longest of its tiles' walks while
// there are compute units to spare, and their sum over the compute units when there are not.
struct WalkCost {
  int64_t tiles = 0;   // of the longest walk
  int64_t total = 0;   // of all walks
  int64_t jobs = 0;    // walks
};
template <class ItemFn>
static void add_walks(WalkCost& c, const ringattn::Segment& seg, int rows, int64_t heads, ItemFn item) {
  const int q_tiles = (seg.q_len + rows - 1) / rows;
  int64_t fixed = 0, first = 0, last = 0;  // keys of the unmasked ranges; of the masked one for the first and the last q tile
  for (int i = 0; i < seg.item_count; ++i) {
    const ringattn::SegItem& it = item(i);
    if (it.diag_off < 0) fixed += (it.kv_len + 31) / 32;
    else {
      first += (std::min(it.kv_len, it.diag_off + rows) + 31) / 32;
      last += (std::min(it.kv_len, it.diag_off + seg.q_len) + 31) / 32;
    }
  }
  c.tiles = std::max(c.tiles, fixed + std::max(first, last));
  c.total += heads * q_tiles * (fixed + (first + last) / 2);
  c.jobs += heads * q_tiles;
}
// The generated loops (ring_walk64_kernel, ring_pair_kernel) keep the place of a key range -- and the place of its last
// tile, where that one is ragged -- as a byte offset within the head, in 32 bits: tile 1 of the range has to begin within 4 GiB.
// (A range may reach beyond that: the loops add whole tiles to 64-bit addresses.)
static bool begins_within_4g(const ringattn::SegItem& it, int dim) { return ((int64_t)it.kv_start + 32) * 2 * dim <= UINT32_MAX; }

using ringattn::kComputeUnits;
struct CarryCosts {
  WalkCost whole, halves, thin;  // with q tiles of kWalkM, kPairM and kSplitM rows
  bool pair = true;              // every segment suits ring_pair_kernel
  bool masked = false;           // the walks differ in length
  template <class ItemFn>
  void add(const ringattn::Segment& seg, int64_t heads, int dim, ItemFn item) {
    add_walks(whole, seg, ringattn::kWalkM, heads, item);
    add_walks(halves, seg, ringattn::kPairM, heads, item);
    add_walks(thin, seg, ringattn::kSplitM, heads, item);
    // ring_pair_kernel: what runs past the end of a walk goes round the first rows of a head, so a KV range holds at least
    // 128 keys; only the range walked last may end in a tile of fewer than 32 keys, whose place the kernel keeps in 32 bits
    const int last = seg.last_item >= 0 ? seg.last_item : seg.item_count - 1;
    for (int i = 0; i < seg.item_count; ++i) {
      const ringattn::SegItem& it = item(i);
      masked = masked || it.diag_off >= 0;
      pair = pair && begins_within_4g(it, dim) && it.kv_len >= 128 && (it.kv_len % 32 == 0 || (i == last && it.kv_start + it.kv_len <= 1 << 24));
    }
  }
};

// A slice of the device tables: what one block launch runs.
struct TableSlice {
  int seg_begin = 0, seg_count = 0;
  int q_len_max = 0;    // rows of the longest segment
  bool wide = false;    // every KV range of the slice suits ring_walk64_kernel
  int min_kv = 0;       // the shortest KV range of the slice
  ringattn::Walks walks;
  CarryCosts costs;     // pl->walk only
};

// ring_walk64_kernel walks whole 32-key tiles, and past the end of its sequence its load streams go round the first
// four tiles of a head: a KV range must be a multiple of 32 keys, hold at least 128 and begin within 4 GiB.
static bool walk64_takes(const ringattn::SegItem& it, int dim) {
  return it.kv_len % 32 == 0 && it.kv_len >= 128 && begins_within_4g(it, dim);
}
// RINGATTN_WIDE=0 in the environment keeps every forward on ring_walk_kernel (for comparisons)
static bool walk64_enabled() {
  const char* e = std::getenv("RINGATTN_WIDE");
  return !(e && e[0] == '0');
}
// RINGATTN_WIDE_PARTIALS in the environment: 0 keeps the launches that emit per-step partials on ring_walk_kernel,
// 1 puts them on ring_walk64_kernel whenever the shapes allow (tests); unset, the chunk length decides
// RINGATTN_WIDE_D64=0 keeps the d = 64 forwards (state carried) on ring_walk_kernel
static bool walk64_d64_enabled() {
  const char* e = std::getenv("RINGATTN_WIDE_D64");
  return !(e && e[0] == '0');
}
static int walk64_partials_choice() {
  const char* e = std::getenv("RINGATTN_WIDE_PARTIALS");
  return !e ? -1 : (e[0] == '0' ? 0 : 1);
}

// RINGATTN_SPLIT=0 and RINGATTN_PAIR=0 in the environment take ring_split_kernel and ring_pair_kernel out of the choice below,
// RINGATTN_PAIR=1 takes the latter whenever the shapes allow, RINGATTN_SPLIT=8 or 16 the former with that many waves (16 at
// d = 64 only); RINGATTN_WIDE=0, RINGATTN_WIDE_D64=0 (d = 64) and RINGATTN_WIDE_PARTIALS=1, which name one of the 256-row
// kernels, keep every launch on these (comparisons, tests).
static int split_choice() {  // -1: unset
  const char* e = std::getenv("RINGATTN_SPLIT");
  return e ? std::atoi(e) : -1;
}
// The columns of V and O that a workgroup of ring_split_kernel has.  A launch of few row tiles gains from fewer of them while their
// workgroups find compute units of their own; with all of these busy they share what L2 delivers, and every one of them asks for the
// whole of K.  us with all, 64 and 32 columns, d = 128: 16 row tiles x 16 key tiles 8.0, 7.1, 6.7, x 256 37.5, 29.7, 27.8; 32 x 32 10.1,
// 8.7, 8.4, x 256 37.8, 30.2, 29.3; 64 x 64 14.5, 12.3, 12.4, x 512 75.6, 59.6, 67.6; 96 x 96 18.8, 16.3, 28.1; 128 x 128 22.6, 21.6,
// 37.1; 256 x 64 17.3, 24.8.  d = 64, all and 32: 32 x 32 6.9, 6.4; 64 x 64 9.4, 9.1, x 512 40.7, 39.5; 75 x 25 6.5, 6.2; 96 x 96 12.0, 11.9;
// 128 x 128 14.4, 14.6, x 256 23.7, 25.3.
// A caller may have O, or fp16 partials, written over Q.  That is all right while one workgroup reads a row of Q and writes it; with the columns
// dealt out one of them could have stored its part before another has read the row, so such a launch keeps all columns.
// RINGATTN_SPLIT_COLUMNS in the environment: 32, 64 or 128, at most the head dimension (comparisons, tests).
static int split_columns(const ringattn::BlockArgs& a, int dim) {
  if ((a.mode == ringattn::kBlockCarryState ? a.out : a.o_part) == a.q) return dim;
  const int64_t row_tiles = (int64_t)a.n_segs * a.q_tiles_max * a.BH;
  const char* e = std::getenv("RINGATTN_SPLIT_COLUMNS");
  const int asked = e ? std::atoi(e) : 0;
  if (asked == 32 || asked == 64 || asked == 128) return std::min(asked, dim);
  if (dim == 64) return row_tiles <= 96 ? 32 : 64;
  return row_tiles <= 32 ? 32 : row_tiles <= 128 ? 64 : 128;
}
static int pair_choice() {
  const char* e = std::getenv("RINGATTN_PAIR");
  return !e ? -1 : (e[0] == '0' ? 0 : 1);
}

// A launch that carries the state has its choice of three kernels, with 256, 128 and 32 query rows per workgroup (kWalkM, kPairM,
// kSplitM) -- the first of them ring_walk64_kernel where the ranges suit it (walk64_takes) and ring_walk_kernel elsewhere, 5 to
// 11 % slower --, a workgroup per compute unit (at d = 64 two of ring_split_kernel and of ring_walk_kernel): the fewer the rows, the shorter the walks (the waves that do not own rows of their own share out the
// keys) and the more of them, but the more often a K/V tile is fetched from L2.  A launch of few q tiles takes as long as
// its longest walk, one of many as all of them over the compute units, at a lower clock.  Each kernel by three measured
// numbers: us per step of a walk (one, two and eight key tiles) with most compute units idle and with all of them busy,
// and us per workgroup besides (Q, first tiles, result).  When they were fitted they gave the time of 150 launches of whole tiles -- heads
// 1 to 64, sequences of 320 to 32768, with and without the causal mask, logits N(0, 1) -- to 2-4 % rms, from these and others; us
// measured on ring_walk64_kernel and the 128- and 32-row kernel at d = 128, and at d = 64:
//     1 head x 2048                         44, 28, 17        34, 22, 13
//     8 heads x 2048                        43, 29, 33        34, 22, 19
//     8 heads x 4096, causal                79, 50, 65        61, 38, 35
//     16 heads x 4096, causal               85, 69, 127       62, 46, 62
//     4 heads x 8192                       151, 117, 197     118, 77, 103
//     8 heads x 8192                       211, 230, 389     131, 145, 198
//     9 heads x 8192 (288 q tiles of 256)  355, 310, 437     244, 208, 223
//     16 heads x 8192, causal              221, 245, 424     142, 159, 209
// ring_split_kernel has since become 5 to 30 % faster where compute units idle (its file) and 5 % elsewhere, so the third row of either table
// below overstates it by that much and draws lines, but does not give its times.  (What the columns gain on top of that, split_columns, is no matter to the
// lines: of 56 000 drawn forwards of so few row tiles every one is on ring_split_kernel.)  It is left, because the lines
// are those between equals: with new numbers d = 64 launches moved to it that both kernels run alike (us on
// ring_split_kernel and ring_pair_kernel: causal 8 x 4928 47, 48; 12 x 3054 33, 34; 4 x 10816 97, 94; no mask 6 x 3394 39, 38; 1 x
// 20971 184, 164), and at d = 128 some whose second round of workgroups is mostly empty (4 x 3328 43.5, 40.6).
enum class CarryKernel { kWhole, kPair, kSplit, kSplit16 };
struct KernelRate {
  int tiles_per_step;
  double lone, busy, job;
  int per_cu = 1;      // workgroups that a compute unit holds at once
  double shared = 0;   // per_cu == 2: us per step of walks that have a compute unit to two, with others idle
};
constexpr KernelRate kRates128[3] = {{1, 0.55, 0.79, 5.3}, {2, 0.60, 0.84, 6.0}, {8, 1.15, 1.35, 4.9}};
constexpr KernelRate kRates64[3] = {{1, 0.42, 0.49, 3.2}, {2, 0.46, 0.53, 4.0}, {8, 0.96, 0.71, 1.9}};
// ring_walk_kernel on ragged lengths (4 % rms over 180 launches).  Its two waves per SIMD cover for each other when references move;
// the one wave of ring_pair_kernel waits for itself.  With logits N(0, 81) a launch takes 8 to 15 % longer there, and 30 to 50 % on
// ring_pair_kernel, which has to be ahead by 12 % on flat ones to be taken: at d = 64, where two workgroups of ring_walk_kernel
// share a compute unit, it led by 1 to 9 % and fell back by 9 to 36 %.  us on ring_walk_kernel and ring_pair_kernel, logits N(0, 1)
// and N(0, 81), d = 64: 24 heads x 3000 91, 90 and 103, 140; 16 x 6001 185, 174 and 204, 247; 12 x 6000 175, 165 and 193, 233; 8 x
// 12001 363, 332 and 389, 423.  Still taken: d = 128 causal, 16 x 4400 123, 95 and 120, 129; d = 64, 9 x 8191 239, 220 and 257, 296.
constexpr KernelRate kWalkRate128 = {1, 0.57, 0.85, 8.0}, kWalkRate64 = {1, 0.46, 0.515, 5.5, 2, 0.90};

static double carry_time(const WalkCost& w, const KernelRate& r, bool equal_walks) {
  const double longest = (double)w.tiles / r.tiles_per_step;
  if (equal_walks) {  // round after round, the last one on what compute units it needs
    const int64_t at_once = kComputeUnits * r.per_cu, rounds = w.jobs / at_once, rest = w.jobs % at_once;
    const double t = (double)(rounds * r.per_cu) * (r.busy * longest + r.job);
    const double slowest = rest > kComputeUnits ? r.shared : r.lone;
    return rest == 0 ? t : t + r.job + longest * std::max(slowest, r.busy * (double)rest / kComputeUnits);
  }
  // the longest walk and the even share of all of them; where these are alike, what is left at the end adds to both
  const double x = r.lone * longest + r.job;
  const double y = (r.busy * (double)w.total / r.tiles_per_step + r.job * (double)w.jobs) / kComputeUnits;
  return std::sqrt(std::sqrt(x * x * x * x + y * y * y * y));
}

// `wide`: the 256-row kernel of this launch is ring_walk64_kernel
static CarryKernel carry_kernel(const CarryCosts& c, int dim, bool wide) {
  if (!walk64_enabled() || (dim == 64 && !walk64_d64_enabled()) || walk64_partials_choice() == 1) return CarryKernel::kWhole;
  if (c.pair && pair_choice() == 1) return CarryKernel::kPair;
  const int split = split_choice();
  if (split == 8 || split == 16) return split == 16 && dim == 64 ? CarryKernel::kSplit16 : CarryKernel::kSplit;
  const KernelRate* r = dim == 128 ? kRates128 : kRates64;
  // the 256-row kernels unless another is ahead by more than these times are good for
  double best = carry_time(c.whole, r[0], !c.masked) * 0.95;
  if (!wide) best = std::min(best, carry_time(c.whole, dim == 128 ? kWalkRate128 : kWalkRate64, !c.masked) * 0.88);
  CarryKernel kernel = CarryKernel::kWhole;
  if (c.pair && pair_choice() != 0) {
    const double t = carry_time(c.halves, r[1], !c.masked);
    if (t < best) best = t, kernel = CarryKernel::kPair;
  }
  if (split != 0 && carry_time(c.thin, r[2], false) < best) kernel = CarryKernel::kSplit;
  // At d = 64 two workgroups of ring_split_kernel fit on a compute unit.  A launch of no more workgroups than there are compute
  // units fills the other half with waves of the same workgroup, sixteen of them instead of eight, where the walk has 96
  // tiles or more.  A row's keys then meet twice as many references, and its probabilities are rounded closer: relative error of
  // O against float64, eight and sixteen waves, 48 calls of 96 to 500 tiles, fp16 2.79e-4, 2.76e-4 (N(0, 1) logits) and 2.34e-4,
  // 2.24e-4 (N(0, 81)), bf16 2.23e-3, 2.21e-3 and 1.85e-3, 1.77e-3.  That is what draws the line, not the time, us: 4096 rows x
  // 4096 keys 15.0, 16.7; 8192 x 8192 28.4, 30.3, causal 24.3, 24.8; 8192 x 16384 53.3, 54.4; 4096 x 16384 43.5, 42.0; 2048 x 16384 42.6,
  // 41.3; the last three with N(0, 81) logits 56.2, 55.9; 48.0, 44.2; 47.1, 43.4.
  if (kernel == CarryKernel::kSplit && dim == 64 && c.thin.jobs <= kComputeUnits && c.thin.tiles >= 96)
    kernel = CarryKernel::kSplit16;
  return kernel;
}

struct ringattn_plan {
  ringattn_params p{};
  int seqlen[RINGATTN_MAX_NPES]{};
  Derived d{};
  void* ws = nullptr;
  size_t ws_bytes = 0;
  bool own_ws = false;
  bool small_steps = false;    // launches that keep the ring steps apart: steps::ring_split_kernel
  void* o_parts = nullptr;     // partial O rows, fp32 (fp16 with RINGATTN_FLAG_HALF_PARTIALS)
  float* lse_parts = nullptr;  // partial LSE rows
  // Segment / item tables (host copies; device copies made by ensure_tables).  Three
  // families of slices: the forward (all ring steps of every rank, one launch, partials in the
  // workspace), one ring step of every rank (ringattn_block_fwd, partials in the caller's
  // [batch*heads, S] slot), one step of one rank on rank-local rows (ringattn_rank_step_fwd).
  std::vector<ringattn::Segment> h_segs;
  std::vector<ringattn::SegItem> h_segitems;
  TableSlice fwd;                  // the ring steps of every row, one by one (RINGATTN_FLAG_STEP_PARTIALS)
  TableSlice walk;                 // the same rows and keys as the forward that carries the state walks them
  std::vector<TableSlice> step;    // [npes]
  std::vector<TableSlice> local;   // [npes * npes]
  // the same schedule as plain work items, for ringattn_plan_work_items
  std::vector<ringattn::WorkItem> h_items;
  int fwd_items = 0;               // h_items[0, fwd_items): the forward, in run order
  std::vector<int> step_begin;     // [npes + 1] slices of h_items, one per ring step
  // merge regions, rank by rank (global rows), then the same with rank-local rows
  std::vector<ringattn::MergeRegion> regions;
  int n_regions = 0;               // global ones; regions[n_regions + i] is regions[i] in local rows
  std::vector<int> region_rank;    // [n_regions]
  int region_max_len = 0;
  ringattn::Segment* d_segs = nullptr;
  ringattn::SegItem* d_segitems = nullptr;
  ringattn::MergeRegion* d_regions = nullptr;
  hipEvent_t ev_t0 = nullptr, ev_t1 = nullptr;  // RINGATTN_FLAG_TIMING: around the block launch
  bool timed_forward = false;                    // a forward has recorded them
  bool tables_ready = false;
  // hipGraph replay (RINGATTN_FLAG_GRAPH): one captured graph per pointer set
  hipStream_t cap_stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  const void *gq = nullptr, *gk = nullptr, *gv = nullptr;
  void* gout = nullptr;
  float* glse = nullptr;
};

namespace {

// fields of the launch arguments that depend only on the geometry
void fill_geometry(ringattn::BlockArgs& a, const ringattn_params& p, const Derived& d) {
  std::memset(&a, 0, sizeof(a));
  a.bh_stride = d.S * p.dim;
  a.kv_bh_stride = d.S * p.dim;
  a.S = (int)d.S;
  a.BH = (int)d.BH;
  a.by_group = ringattn::divisor(p.kv_heads > 0 ? p.heads / p.kv_heads : 1);
  a.scale_log2 = d.scale * kLog2e;
  a.half_partials = half_partials(p) ? 1 : 0;
  a.causal = p.causal != 0;
}

inline int q_tiles_of(int len, int tile = ringattn::kWalkM) { return (len + tile - 1) / tile; }

// Appends one segment with its items to the tables.  part_base(i) / stride: where item i's
// partial block lives.  A masked (diagonal) item runs last and the q tiles go busiest first.
template <class BaseFn>
void push_segment(ringattn_plan* pl, TableSlice& slice, int q_start, int q_len,
                  const std::vector<ringattn::WorkItem>& items, int kv_shift, BaseFn part_base, int part_bh_stride,
                  int part_row_mul = 0) {
  ringattn::Segment sg;
  std::memset(&sg, 0, sizeof(sg));
  sg.q_start = q_start;
  sg.q_len = q_len;
  sg.item_begin = (int)pl->h_segitems.size();
  sg.item_count = (int)items.size();
  sg.last_item = -1;
  for (size_t i = 0; i < items.size(); ++i) {
    const ringattn::WorkItem& w = items[i];
    ringattn::SegItem it;
    std::memset(&it, 0, sizeof(it));
    it.kv_start = w.kv_start - kv_shift;
    it.kv_len = w.kv_len;
    it.diag_off = w.diag_off;
    it.part_bh_stride = part_bh_stride;
    it.part_base = part_base((int)i);
    it.slot = w.slot;
    it.part_row_mul = part_row_mul;
    if (w.diag_off >= 0) {
      sg.last_item = (int)i;
      sg.reverse_tiles = 1;
    }
    pl->h_segitems.push_back(it);
  }
  if (sg.item_count == 1) sg.last_item = -1;
  pl->h_segs.push_back(sg);
  bool wide = true;
  for (size_t i = 0; i < items.size(); ++i) wide = wide && walk64_takes(pl->h_segitems[(size_t)sg.item_begin + i], pl->p.dim);
  slice.wide = slice.seg_count == 0 ? wide : (slice.wide && wide);
  int keys = 0;
  for (const auto& w : items) {
    keys += (w.kv_len + 31) / 32;
    if (w.diag_off >= 0) slice.walks.masked = slice.walks.uneven = true;
  }
  if (slice.seg_count > 0 && keys != slice.walks.longest) slice.walks.uneven = true;
  slice.walks.longest = std::max(slice.walks.longest, keys);
  slice.walks.tiles += q_tiles_of(q_len);
  for (size_t i = 0; i < items.size(); ++i) {
    const int kv = pl->h_segitems[(size_t)sg.item_begin + i].kv_len;
    slice.min_kv = (slice.seg_count == 0 && i == 0) ? kv : std::min(slice.min_kv, kv);
  }
  ++slice.seg_count;
  slice.q_len_max = std::max(slice.q_len_max, q_len);
}

// The tables of a plan (host side; nothing here touches the GPU).
void build_schedule(ringattn_plan* pl) {
  const int P = pl->p.npes;
  const Derived& d = pl->d;
  const bool causal = pl->p.causal != 0;

  // ---- the forward: every segment with all its steps; partial blocks packed in the workspace
  const std::vector<HostSegment> segs = forward_segments(d, P, causal);
  pl->fwd.seg_begin = 0;
  int64_t next_row = 0;
  for (const auto& sg : segs) {
    const int64_t block_rows = d.BH * sg.len;
    const int64_t base = next_row;
    push_segment(pl, pl->fwd, sg.start, sg.len, sg.items, 0,
                 [&](int i) { return base + (int64_t)i * block_rows; }, sg.len);
    next_row += (int64_t)sg.items.size() * block_rows;
    // the same items in run order (the masked one last), for inspection
    const ringattn::Segment& t = pl->h_segs.back();
    for (int i = 0; i < t.item_count; ++i) {
      int idx = i;
      if (t.last_item >= 0) idx = (i == t.item_count - 1) ? t.last_item : (i >= t.last_item ? i + 1 : i);
      pl->h_items.push_back(sg.items[(size_t)idx]);
    }
  }
  pl->fwd_items = (int)pl->h_items.size();
  // ---- the forward that carries the state: no partials, the ring steps joined where they can be
  pl->walk.seg_begin = (int)pl->h_segs.size();
  for (const auto& sg : walk_segments(d, P, causal))
    push_segment(pl, pl->walk, sg.start, sg.len, sg.items, 0, [](int) { return (int64_t)0; }, 0);
  for (int i = 0; i < pl->walk.seg_count; ++i) {
    const ringattn::Segment& sg = pl->h_segs[(size_t)(pl->walk.seg_begin + i)];
    pl->walk.costs.add(sg, d.BH, pl->p.dim, [&](int k) -> const ringattn::SegItem& { return pl->h_segitems[(size_t)(sg.item_begin + k)]; });
  }

  // ---- one ring step of every rank: partials at the rows of the queries in a [BH, S] slot
  for (int s = 0; s < P; ++s) {
    pl->step_begin.push_back((int)pl->h_items.size());
    TableSlice sl;
    sl.seg_begin = (int)pl->h_segs.size();
    std::vector<ringattn::WorkItem> one;
    for (int r = 0; r < P; ++r) {
      one.clear();
      append_items(one, d, P, causal, r, s);
      for (const auto& w : one) {
        pl->h_items.push_back(w);
        const std::vector<ringattn::WorkItem> v1{w};
        push_segment(pl, sl, w.q_start, w.q_len, v1, 0, [&](int) { return (int64_t)w.q_start; }, (int)d.S,
                     row_partials(pl->p) ? P : 0);
      }
    }
    pl->step.push_back(sl);
  }
  pl->step_begin.push_back((int)pl->h_items.size());

  // ---- one step of one rank in rank-local rows (queries from 0, keys from 0 of the visited chunk)
  for (int r = 0; r < P; ++r)
    for (int s = 0; s < P; ++s) {
      TableSlice sl;
      sl.seg_begin = (int)pl->h_segs.size();
      std::vector<ringattn::WorkItem> one;
      append_items(one, d, P, causal, r, s);
      const int q0 = d.start[r], rows = d.start[r + 1] - q0, k0 = d.start[(r + s) % P];
      for (const auto& w : one) {
        const std::vector<ringattn::WorkItem> v1{w};
        push_segment(pl, sl, w.q_start - q0, w.q_len, v1, k0, [&](int) { return (int64_t)(w.q_start - q0); }, rows,
                     row_partials(pl->p) ? P : 0);
      }
      pl->local.push_back(sl);
    }

  // ---- merge regions of caller-held per-step partials, rank by rank
  for (int r = 0; r < P; ++r) {
    std::vector<HostSegment> rs;
    rank_segments(rs, d, P, causal, r);
    for (const auto& sg : rs) {
      pl->regions.push_back(ringattn::MergeRegion{sg.start, sg.len, sg.active});
      pl->region_rank.push_back(r);
      pl->region_max_len = std::max(pl->region_max_len, sg.len);
    }
  }
  pl->n_regions = (int)pl->regions.size();
  for (int i = 0; i < pl->n_regions; ++i) {
    ringattn::MergeRegion m = pl->regions[(size_t)i];
    m.start -= d.start[pl->region_rank[(size_t)i]];
    pl->regions.push_back(m);
  }
}

// The copies of ensure_tables, by way of `copies`: NULL, or a stream of its own next to one that is being captured.
int upload_tables(ringattn_plan* pl, hipStream_t copies) {
  // a call that failed half way is resumed: nothing is created twice
  auto upload = [&](void** dst, const void* src, size_t bytes) -> int {
    if (!*dst) RA_HIP(hipMalloc(dst, bytes));
    if (copies) RA_HIP(hipMemcpyAsync(*dst, src, bytes, hipMemcpyHostToDevice, copies));
    else RA_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    return RINGATTN_OK;
  };
  int rc = upload((void**)&pl->d_segs, pl->h_segs.data(), pl->h_segs.size() * sizeof(ringattn::Segment));
  if (rc == RINGATTN_OK) rc = upload((void**)&pl->d_segitems, pl->h_segitems.data(), pl->h_segitems.size() * sizeof(ringattn::SegItem));
  if (rc == RINGATTN_OK) rc = upload((void**)&pl->d_regions, pl->regions.data(), pl->regions.size() * sizeof(ringattn::MergeRegion));
  return rc;
}

// Device copies of the tables and the timing events: made by the first call of a step or a merge, and by the first forward
// whose launch does not carry its only range in its arguments.  That call may sit in a capture of `stream` (the forwards
// that warmed the plan up needed no tables): the copies are then made beside the captured work, at once, on a stream of
// their own, in the capture mode that allows the thread to allocate.
int ensure_tables(ringattn_plan* pl, hipStream_t stream) {
  if (pl->tables_ready) return RINGATTN_OK;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (stream) RA_HIP(hipStreamIsCapturing(stream, &capture));
  if (capture == hipStreamCaptureStatusNone) {
    const int rc = upload_tables(pl, nullptr);
    if (rc != RINGATTN_OK) return rc;
  } else {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RA_HIP(hipThreadExchangeStreamCaptureMode(&mode));
    hipStream_t copies = nullptr;
    hipError_t e = hipStreamCreateWithFlags(&copies, hipStreamNonBlocking);
    int rc = e == hipSuccess ? upload_tables(pl, copies) : hip_fail(e);
    if (copies) {
      e = hipStreamSynchronize(copies);
      if (rc == RINGATTN_OK && e != hipSuccess) rc = hip_fail(e);
      (void)hipStreamDestroy(copies);
    }
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (rc != RINGATTN_OK) return rc;
  }
  if (pl->p.flags & RINGATTN_FLAG_TIMING) {
    if (!pl->ev_t0) RA_HIP(hipEventCreate(&pl->ev_t0));
    if (!pl->ev_t1) RA_HIP(hipEventCreate(&pl->ev_t1));
  }
  pl->tables_ready = true;
  return RINGATTN_OK;
}

// ring_walk64_kernel runs the launch of a slice when every KV range suits it and d = 128.  The launches that emit
// partials go by the forward's ranges, so that the forward and the steps run one by one keep giving the same bits.
// A chunk walked on its own costs ring_walk64_kernel a start and a drain of its pipeline, and it writes its partials to memory and
// reads them back where ring_walk_kernel merges them on the chip; its loop is the faster one, also because it skips masked
// tiles wave by wave.  Whichever is taken runs the forward and the single steps of a plan.  us on ring_walk_kernel and on
// ring_walk64_kernel, fp16, fp32 partials (in brackets fp16 partials), causal forwards of 4 ranks, 4 and 32 heads: chunks of 1024
// 89, 120 (90, 110) and 145, 186 (146, 164); of 2048 166, 193 (167, 184) and 541, 580 (544, 557); of 4096 349, 362 (353, 356) and 1992, 1978
// (1989, 1909); of 8192 981, 937 and 7702, 7317.  One step of a rank of them, masked, 8 and 32 heads: chunks of 1024 30, 29 and
// 32, 30; of 2048 50, 47 and 57, 52; of 4096 89, 84 and 144, 132; any other step 28, 29 and 31, 31; 47, 47 and 69, 66; 88, 85 and 253,
// 237.  So from 2048 keys on a ring run step by step gains up to 9 %, and the forward in one launch loses up to 14 % at 2048, 4 % at
// 4096 where heads are few, and gains beyond.  Without a mask ring_walk64_kernel lies 0 to 6 % ahead at 4096 keys and 3 to 8 % at 8192, and is
// not taken.
constexpr int kWidePartialsMinKeys = 2048;
bool slice_takes_walk64(const ringattn_plan* pl, const TableSlice& sl, int mode) {
  if (!sl.wide || !walk64_enabled()) return false;
  if (mode != ringattn::kBlockCarryState) {
    const int choice = walk64_partials_choice();
    if (pl->p.dim != 128 || choice == 0 || !pl->fwd.wide) return false;
    if (choice < 0 && !(pl->p.causal && pl->fwd.min_kv >= kWidePartialsMinKeys)) return false;
    return true;
  }
  return pl->p.dim == 128 || (pl->p.dim == 64 && walk64_d64_enabled());
}

// thin::ring_walk_kernel gives the bits of ring_walk_kernel with one wave per SIMD on half the rows, so a launch may have either.  It is the
// faster one, at d = 64, while there are compute units to spare (figures in ringattn_thin.hip); places within a
// range are 32-bit offsets there.  RINGATTN_THIN=0 and 1 in the environment: never, and whatever the size (comparisons, tests).
constexpr int64_t kThinMaxJobs = 128;  // 256-row q tiles
bool takes_thin(const ringattn_plan* pl, const TableSlice& sl) {
  if (pl->p.dim != 64 || pl->d.S * 2 * pl->p.dim > INT32_MAX) return false;
  const char* e = std::getenv("RINGATTN_THIN");
  if (e) return e[0] != '0';
  return (int64_t)sl.seg_count * q_tiles_of(sl.q_len_max) * pl->d.BH <= kThinMaxJobs;
}

// Of the launches that thin::ring_walk_kernel may have, dealt::ring_walk_kernel, which gives the same bits again, takes single steps of no more
// 32-row q tiles than there are compute units, each of which holds one of its workgroups; under the diagonal, where the short walks of
// a second round fill in behind the long ones, of twice as many.  us on thin and dealt: 8 heads x 1024 x 1024 15.6, 10.7 (256 workgroups), 6 x
// 1500 x 1500 21.1, 23.9 (282), 16 x 1024 x 1024 16.1, 19.2 (512); causal 8 x 2048 x 2048 27.1, 19.2 (512).
// With a second round the walks have to be the longer the more of it there is, or it costs more than dealing the tiles gains: time on dealt over
// that on thin, 257 to 512 workgroups, above the line of the rule, a tile to sixteen workgroups, 0.52 to 0.92 with N(0, 1) logits and up to 0.96 with
// N(0, 9), below it 0.91 to 1.40 and 0.92 to 1.42 (1100 drawn steps).  64 heads x 223 8.4, 12.2 (448), 35 x 342 10.7, 13.4 (385), 29 x 512 11.4, 12.2 (464).
// A walk that is over within a round has nothing to share out: 64 heads x 64 x 64 4.8, 5.4, 8 x 60 x 60 5.0, 5.2; 32 x 128 x 128 5.9, 5.3.
// A move of the references costs a round of short walks more than it gains.  With N(0, 81) logits the lines leave 0.57 to 1.10 of the time on thin
// without a mask, where twelve to sixteen tiles have 0.91 to 1.10, and 0.55 to 1.18 under the diagonal, where up to nine have 0.89 to 1.18; with N(0, 1) the
// same take 0.76 to 0.87 and 0.76 to 0.93, and N(0, 9) logits lose nowhere (1700 drawn steps within the lines).
// RINGATTN_DEALT=0 and 1 in the environment: never, and whatever the size (comparisons, tests); RINGATTN_THIN names the other two.
bool takes_dealt(const ringattn_plan* pl, const TableSlice& sl) {
  if (std::getenv("RINGATTN_THIN")) return false;
  const char* e = std::getenv("RINGATTN_DEALT");
  if (e) return e[0] != '0';
  const int64_t tiles = (int64_t)sl.seg_count * q_tiles_of(sl.q_len_max, ringattn::kDealtM) * pl->d.BH;
  if (tiles <= ringattn::kComputeUnits) return sl.walks.longest >= (sl.walks.masked ? 4 : 12);
  return sl.walks.masked && tiles <= 2 * ringattn::kComputeUnits && 16 * (int64_t)sl.walks.longest >= tiles;
}

// steps::ring_split_kernel runs the launches of a plan that keep the ring steps apart -- single steps of one rank and of all, and
// the forward with RINGATTN_FLAG_STEP_PARTIALS -- where even the largest of them are small.  Its partials have other bits than those of the
// 256-row kernels, and all launches of a plan give the same, so there is one choice for the three, whichever a program
// calls.  Those of one step stop gaining where there are more 32-row q tiles than a round of workgroups, but the longer their walks the later,
// the forward where the 256-row kernels fill the device.  2780 of 4100 drawn plans (P 1 to 32, 600 to 60 000 rows, logits N(0, 1) and N(0, 81), 2700 of
// them around the lines) are within the lines.  What these leave of the time on the kernels that had the launches before it (ring_walk_kernel, at d = 64
// thin::), geometric mean (the worst of fifty in brackets) of a rank's step, a step of all and the forward: d = 64 0.51 (0.93), 0.58 (0.98), 0.52 (0.88), under
// the mask 0.52 (0.93), 0.55 (1.01), 0.48 (0.82); d = 128 0.39 (0.86), 0.47 (0.94), 0.44 (0.84), under the mask 0.38 (0.89), 0.43 (0.99), 0.37 (0.65).
// A rank's step lost in none of them.  A step of all lost in 25, up to 16 %, nearly all of them with chunks of up to 128 keys, which are one wave's
// work (2 ranks x 41 heads x 128, zigzag, 5.5, 6.4), and in one, whose short segments leave holes in a grid larger than the device, 46 % (23 x 3
// heads x 76 on average, d = 128: 9.0, 13.1); their forwards take 0.33 to 1.01 of the time.  The forward lost in two, of one rank: d = 64, 38 heads x 256 7.4, 8.3, 35 x
// 256 8.8, 9.4.  us before and after: d = 64, 4 heads x 4 x 512 9.9, 10.1, 29.9 and 6.2, 6.9, 17.7, 2 x 4 x 2048 25.6, 27.6, 94 and 10.1, 19.1, 65;
// d = 128, 2 heads x 4 x 2048 46, 49, 163 and 15.3, 36, 123, causal 4 x 4 x 777 29.5, 29.7, 100 and 11.9, 11.8, 42.  Beyond them, d = 64, 8 heads x 8 x
// 1024: 15.6, 30.3, 181 and 8.4, 45, 296; d = 128, 8 x 8 x 256 12.9, 14.3, 56 and 7.0, 14.8, 47.
// RINGATTN_SPLIT_STEPS=0 and 1 in the environment: never, and always (comparisons, tests); the switches that name one of the
// other kernels for these launches, or all launches, take this one out.
bool small_steps(const ringattn_params& p, const Derived& d) {
  int64_t tiles = 0;
  for (int r = 0; r < p.npes; ++r) tiles += d.BH * ((d.start[r + 1] - d.start[r] + ringattn::kSplitM - 1) / ringattn::kSplitM);
  const double chunk = (double)d.S / p.npes;
  if (chunk < (p.npes == 1 ? 192 : 64)) return false;  // (a tile or two: one wave's work)
  const double more = p.dim == 64 ? 1.03 * std::pow(std::max(1.0, chunk / 128), 0.25) : std::min(2.5, std::max(1.0, std::sqrt(chunk / 512)));
  const double masked = p.causal && (p.dim == 64 || chunk >= 512) ? 1.4 : 1.0;
  return (double)tiles <= ringattn::kComputeUnits * more * masked;
}
bool takes_split_steps(const ringattn_plan* pl) {
  const char* e = std::getenv("RINGATTN_SPLIT_STEPS");
  if (e) return e[0] != '0';
  return pl->small_steps && walk64_enabled() && walk64_partials_choice() < 0 && split_choice() != 0 && !std::getenv("RINGATTN_THIN");
}

// the slice ringattn_fwd launches
const TableSlice& forward_slice(const ringattn_plan* pl) { return step_partials(pl->p) ? pl->fwd : pl->walk; }

// A launch of one segment with one key range carries both in its arguments: a forward without a mask or with the
// contiguous causal layout, one step of one rank.  No table to upload before the first launch, and none to read -- a chain
// of dependent memory round trips at the start of every workgroup.
bool in_arguments(const ringattn_plan* pl, const TableSlice& sl, int mode) {
  return mode != ringattn::kBlockPartialsMerged && sl.seg_count == 1 && pl->h_segs[(size_t)sl.seg_begin].item_count == 1;
}

// the launch of `kernel` over q tiles of its size; `wide`: kWhole is ring_walk64_kernel
hipError_t launch_q_tiles(ringattn::BlockArgs& a, CarryKernel kernel, bool wide, const ringattn::Walks& walks, int q_len, int dtype, int dim,
                          hipStream_t stream) {
  switch (kernel) {
    case CarryKernel::kPair:
      a.q_tiles_max = q_tiles_of(q_len, ringattn::kPairM);
      return ringattn::launch_pair(a, dtype, dim, stream);
    case CarryKernel::kSplit:
    case CarryKernel::kSplit16:
      a.q_tiles_max = q_tiles_of(q_len, ringattn::kSplitM);
      return ringattn::launch_split(a, dtype, dim, kernel == CarryKernel::kSplit16, split_columns(a, dim), stream);
    default:
      a.q_tiles_max = q_tiles_of(q_len);
      return wide ? ringattn::launch_walk64(a, dtype, dim, stream) : ringattn::launch_walk(a, walks, dtype, dim, stream);
  }
}

// A block launch over a slice of the tables.
int launch_slice(ringattn_plan* pl, const TableSlice& sl, ringattn::BlockArgs& a, hipStream_t stream) {
  if (sl.seg_count == 0) return RINGATTN_OK;
  if (in_arguments(pl, sl, a.mode)) {
    a.one_seg = pl->h_segs[(size_t)sl.seg_begin];
    a.one_item = pl->h_segitems[(size_t)a.one_seg.item_begin];
    a.one_seg.item_begin = 0;  // the item's place is with the arguments now
  } else {
    const int rc = ensure_tables(pl, stream);
    if (rc != RINGATTN_OK) return rc;
    a.segs = pl->d_segs + sl.seg_begin;
    a.items = pl->d_segitems;
  }
  a.n_segs = sl.seg_count;
  if (a.mode != ringattn::kBlockCarryState && takes_split_steps(pl)) {
    a.q_tiles_max = q_tiles_of(sl.q_len_max, ringattn::kSplitM);
    const int columns = a.mode == ringattn::kBlockPartials ? split_columns(a, pl->p.dim) : pl->p.dim;
    RA_HIP(ringattn::launch_split_steps(a, pl->p.dtype, pl->p.dim, columns, stream));
    return RINGATTN_OK;
  }
  const bool wide = slice_takes_walk64(pl, sl, a.mode);
  if (a.mode != ringattn::kBlockCarryState && !wide && takes_thin(pl, sl)) {
    if (a.mode == ringattn::kBlockPartials && takes_dealt(pl, sl)) {
      a.q_tiles_max = q_tiles_of(sl.q_len_max, ringattn::kDealtM);
      RA_HIP(ringattn::launch_dealt(a, pl->p.dtype, stream));
      return RINGATTN_OK;
    }
    a.q_tiles_max = q_tiles_of(sl.q_len_max, ringattn::kThinM);
    RA_HIP(ringattn::launch_thin(a, pl->p.dtype, stream));
    return RINGATTN_OK;
  }
  const CarryKernel kernel =
      a.mode == ringattn::kBlockCarryState ? carry_kernel(sl.costs, pl->p.dim, wide) : CarryKernel::kWhole;
  RA_HIP(launch_q_tiles(a, kernel, wide, sl.walks, sl.q_len_max, pl->p.dtype, pl->p.dim, stream));
  return RINGATTN_OK;
}

// The ring step loop (csrc/ring_attention.cu:456-620) and the epilogue (:621-664), ONE launch:
// every workgroup walks the ring steps of its 256 rows with the softmax state carried in
// registers, like the reference's CTA (:439-443,597).  With RINGATTN_FLAG_STEP_PARTIALS it
// makes a partial (O, LSE) per step instead: ring_walk_kernel merges each where it arises,
// ring_walk64_kernel writes them to the workspace and merges them at the end.
int run_forward(ringattn_plan* pl, const void* q, const void* k, const void* v, void* out,
                float* lse, hipStream_t stream) {
  const bool timing = (pl->p.flags & RINGATTN_FLAG_TIMING) && !(pl->p.flags & RINGATTN_FLAG_GRAPH);
  ringattn::BlockArgs a;
  fill_geometry(a, pl->p, pl->d);
  a.q = q;
  a.k = k;
  a.v = v;
  a.o_part = pl->o_parts;
  a.lse_part = pl->lse_parts;
  a.out = out;
  a.lse = lse;
  a.mode = step_partials(pl->p) ? ringattn::kBlockPartialsMerged : ringattn::kBlockCarryState;
  if (timing) RA_HIP(hipEventRecord(pl->ev_t0, stream));
  const int rc = launch_slice(pl, forward_slice(pl), a, stream);
  if (rc != RINGATTN_OK) return rc;
  if (timing) {
    RA_HIP(hipEventRecord(pl->ev_t1, stream));
    pl->timed_forward = true;
  }
  return RINGATTN_OK;
}

void drop_graph(ringattn_plan* pl) {
  if (pl->exec) (void)hipGraphExecDestroy(pl->exec);
  if (pl->graph) (void)hipGraphDestroy(pl->graph);
  pl->exec = nullptr;
  pl->graph = nullptr;
}

inline bool plan_ok(const ringattn_plan* pl) {
  if (!pl) return false;
  std::lock_guard<std::mutex> lk(g_plans_mu);
  return g_plans.count(pl) != 0;
}

// ---- the reference-shaped call for one rank (ringattn_ring_attention and its variant that
// allocates nothing) ------------------------------------------------------------------------
// One segment, one key range (the chunks a rank sees lie next to each other: all of them, or with the mask those up to
// its own): the launch carries both in its arguments, so the call needs no device memory of its own.
struct RankCall {
  ringattn_params p;
  Derived d;
  ringattn::Segment seg;
  ringattn::SegItem item;
};

int prepare_rank_call(RankCall* rc, const void* q, const void* k, const void* v, void* out, int npes, int mype,
                      const int* seqlen, int dim, int max_seq, int dtype, int causal, float softmax_scale) {
  ringattn_params& p = rc->p;
  std::memset(&p, 0, sizeof(p));
  p.npes = npes;
  p.h_seqlen = seqlen;
  p.dim = dim;
  p.softmax_scale = softmax_scale;
  p.batch = 1;
  p.heads = 1;
  p.dtype = dtype;
  p.causal = causal;
  int err = validate(&p, &rc->d);
  if (err != RINGATTN_OK) return err;
  const Derived& d = rc->d;
  if (mype < 0 || mype >= npes) return RINGATTN_ERR_RANK;
  if (max_seq < d.max_len) return RINGATTN_ERR_SEQLEN;
  if (!q || !k || !v || !out) return RINGATTN_ERR_NULL;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return RINGATTN_ERR_ALIGN;
  // the query rows are local to the caller's rank-sized q and out buffers
  const int c = d.start[mype + 1] - d.start[mype];
  std::memset(&rc->seg, 0, sizeof(rc->seg));
  rc->seg.q_len = c;
  rc->seg.item_count = 1;
  rc->seg.last_item = -1;
  rc->seg.reverse_tiles = causal ? 1 : 0;
  std::memset(&rc->item, 0, sizeof(rc->item));
  rc->item.kv_len = causal ? d.start[mype + 1] : (int)d.S;
  rc->item.diag_off = causal ? d.start[mype] : -1;
  return RINGATTN_OK;
}

// One launch on `stream`; nothing is allocated or copied from the host.
int run_rank_call(const RankCall& rc, const void* q, const void* k, const void* v, void* out, float* lse, hipStream_t stream) {
  const int dim = rc.p.dim, c = rc.seg.q_len;
  ringattn::BlockArgs a;
  fill_geometry(a, rc.p, rc.d);
  a.q = q;
  a.k = k;
  a.v = v;
  a.out = out;
  a.lse = lse;  // may be NULL
  a.mode = ringattn::kBlockCarryState;
  a.one_seg = rc.seg;
  a.one_item = rc.item;
  a.n_segs = 1;
  a.bh_stride = (int64_t)c * dim;  // q and out hold this rank's rows only; k and v the whole sequence
  a.S = c;
  const bool wide = (dim == 128 || (dim == 64 && walk64_d64_enabled())) && walk64_enabled() && walk64_takes(rc.item, dim);
  CarryCosts costs;
  costs.add(rc.seg, 1, dim, [&](int) -> const ringattn::SegItem& { return rc.item; });
  RA_HIP(launch_q_tiles(a, carry_kernel(costs, dim, wide), wide, {}, c, rc.p.dtype, dim, stream));
  return RINGATTN_OK;
}

// merge launch over `count` regions of the plan's device table starting at `first`
int launch_regions(const ringattn_plan* pl, int first, int count, int max_len, int rows_per_head, int64_t part_stride_rows,
                   const void* o_parts, const float* lse_parts, void* out, float* lse, hipStream_t stream) {
  ringattn::MergeArgs m;
  std::memset(&m, 0, sizeof(m));
  m.o_parts = o_parts;
  m.lse_parts = lse_parts;
  m.out = out;
  m.lse = lse;
  m.regions = pl->d_regions + first;
  m.n_regions = count;
  m.max_len = max_len;
  m.heads = (int)pl->d.BH;
  m.S = rows_per_head;
  m.part_stride_rows = part_stride_rows;
  for (int i = first; i < first + count; ++i) {
    const ringattn::MergeRegion& reg = pl->regions[(size_t)i];
    m.part_rows += (int64_t)m.heads * reg.len * __builtin_popcountll(reg.active);
  }
  m.half_partials = half_partials(pl->p) ? 1 : 0;
  m.slot0_last = pl->p.causal ? 1 : 0;
  m.row_mul = row_partials(pl->p) ? pl->p.npes : 0;
  RA_HIP(ringattn::launch_merge(m, pl->p.dtype, pl->p.dim, stream));
  return RINGATTN_OK;
}

}  // namespace

extern "C" {

size_t ringattn_workspace_bytes(const ringattn_params* params) {
  Derived d;
  if (validate(params, &d) != RINGATTN_OK) return 0;
  return workspace_bytes_of(params, d);
}

int ringattn_plan_create(const ringattn_params* params, void* workspace, size_t workspace_bytes,
                         ringattn_plan** plan_out) {
  if (!plan_out) return RINGATTN_ERR_NULL;
  *plan_out = nullptr;
  Derived d;
  int rc = validate(params, &d);
  if (rc != RINGATTN_OK) return rc;
  const size_t need = workspace_bytes_of(params, d);
  if (workspace) {
    if (workspace_bytes < need) return RINGATTN_ERR_WORKSPACE;
    if (!aligned16(workspace)) return RINGATTN_ERR_ALIGN;
  }
  ringattn_plan* pl = new (std::nothrow) ringattn_plan();
  if (!pl) return RINGATTN_ERR_ALLOC;
  pl->p = *params;
  std::memcpy(pl->seqlen, params->h_seqlen, sizeof(int) * (size_t)params->npes);
  pl->p.h_seqlen = pl->seqlen;
  pl->d = d;
  pl->ws_bytes = need;
  if (workspace) {
    pl->ws = workspace;
    pl->own_ws = false;
  } else if (need > 0) {
    hipError_t e = hipMalloc(&pl->ws, need);
    if (e != hipSuccess) {
      delete pl;
      g_last_hip_error = (int)e;
      return e == hipErrorOutOfMemory ? RINGATTN_ERR_ALLOC : RINGATTN_ERR_HIP;
    }
    pl->own_ws = true;
  }
  build_schedule(pl);
  pl->small_steps = small_steps(pl->p, d);
  const size_t part_rows = need / ((size_t)params->dim * (half_partials(*params) ? 2 : 4) + sizeof(float));
  pl->o_parts = pl->ws;
  pl->lse_parts = (float*)((char*)pl->ws + part_rows * params->dim * (half_partials(*params) ? 2 : 4));
  {
    std::lock_guard<std::mutex> lk(g_plans_mu);
    g_plans.insert(pl);
  }
  *plan_out = pl;
  return RINGATTN_OK;
}

int ringattn_plan_destroy(ringattn_plan* plan) {
  {
    std::lock_guard<std::mutex> lk(g_plans_mu);
    if (!plan || g_plans.erase(plan) == 0) return RINGATTN_ERR_PLAN;
  }
  int rc = RINGATTN_OK;
  drop_graph(plan);
  if (plan->cap_stream) (void)hipStreamDestroy(plan->cap_stream);
  // whatever ensure_tables() got to create, also after a failure half way
  if (plan->ev_t0) (void)hipEventDestroy(plan->ev_t0);
  if (plan->ev_t1) (void)hipEventDestroy(plan->ev_t1);
  if (plan->d_segs) (void)hipFree(plan->d_segs);
  if (plan->d_segitems) (void)hipFree(plan->d_segitems);
  if (plan->d_regions) (void)hipFree(plan->d_regions);
  if (plan->own_ws && plan->ws) {
    hipError_t e = hipFree(plan->ws);
    if (e != hipSuccess) rc = hip_fail(e);
  }
  delete plan;
  return rc;
}

int ringattn_fwd(ringattn_plan* plan, const void* q, const void* k, const void* v, void* out,
                 float* lse, void* stream_) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!q || !k || !v || !out || !lse) return RINGATTN_ERR_NULL;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || ((uintptr_t)lse & 3u)) return RINGATTN_ERR_ALIGN;
  hipStream_t stream = (hipStream_t)stream_;
  if ((plan->p.flags & (RINGATTN_FLAG_TIMING | RINGATTN_FLAG_GRAPH)) || step_partials(plan->p)) {
    const int rc0 = ensure_tables(plan, stream);  // the timing events too; and nothing may be allocated during the capture
    if (rc0 != RINGATTN_OK) return rc0;
  }
  if (!(plan->p.flags & RINGATTN_FLAG_GRAPH)) return run_forward(plan, q, k, v, out, lse, stream);

  // hipGraph replay: the launch of a forward is captured once per pointer set on a private
  // stream (kernel nodes only, no memset nodes) and replayed on the caller's stream.
  if (!plan->exec || plan->gq != q || plan->gk != k || plan->gv != v || plan->gout != out || plan->glse != lse) {
    drop_graph(plan);
    if (!plan->cap_stream) RA_HIP(hipStreamCreateWithFlags(&plan->cap_stream, hipStreamNonBlocking));
    RA_HIP(hipStreamBeginCapture(plan->cap_stream, hipStreamCaptureModeThreadLocal));
    int rc = run_forward(plan, q, k, v, out, lse, plan->cap_stream);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(plan->cap_stream, &g);
    if (rc != RINGATTN_OK) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return hip_fail(e);
    plan->graph = g;
    e = hipGraphInstantiate(&plan->exec, plan->graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
      drop_graph(plan);
      return hip_fail(e);
    }
    plan->gq = q;
    plan->gk = k;
    plan->gv = v;
    plan->gout = out;
    plan->glse = lse;
  }
  RA_HIP(hipGraphLaunch(plan->exec, stream));
  return RINGATTN_OK;
}

int ringattn_block_fwd(ringattn_plan* plan, int step, const void* q, const void* k, const void* v,
                       void* o_part, float* lse_part, void* stream) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!q || !k || !v || !o_part || !lse_part) return RINGATTN_ERR_NULL;
  if (step < 0 || step >= plan->p.npes) return RINGATTN_ERR_RANK;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o_part) || ((uintptr_t)lse_part & 3u)) return RINGATTN_ERR_ALIGN;
  const int rc = ensure_tables(plan, (hipStream_t)stream);  // whether or not this step reads them: the merge will
  if (rc != RINGATTN_OK) return rc;
  ringattn::BlockArgs a;
  fill_geometry(a, plan->p, plan->d);
  a.q = q;
  a.k = k;
  a.v = v;
  a.o_part = o_part;
  a.lse_part = lse_part;
  return launch_slice(plan, plan->step[(size_t)step], a, (hipStream_t)stream);
}

int ringattn_merge_ring(ringattn_plan* plan, const void* o_parts, const float* lse_parts, void* out,
                        float* lse, void* stream) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!o_parts || !lse_parts || !out || !lse) return RINGATTN_ERR_NULL;
  if (!aligned16(o_parts) || !aligned16(out) || ((uintptr_t)lse_parts & 3u) || ((uintptr_t)lse & 3u)) return RINGATTN_ERR_ALIGN;
  int rc = ensure_tables(plan, (hipStream_t)stream);
  if (rc != RINGATTN_OK) return rc;
  // ONE launch: a grid row per region
  return launch_regions(plan, 0, plan->n_regions, plan->region_max_len, (int)plan->d.S, plan->d.rows, o_parts, lse_parts,
                        out, lse, (hipStream_t)stream);
}

int ringattn_rank_step_fwd(ringattn_plan* plan, int rank, int step, const void* q, const void* k_chunk,
                           const void* v_chunk, void* o_part, float* lse_part, void* stream) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!q || !k_chunk || !v_chunk || !o_part || !lse_part) return RINGATTN_ERR_NULL;
  const int P = plan->p.npes;
  if (rank < 0 || rank >= P || step < 0 || step >= P) return RINGATTN_ERR_RANK;
  if (!aligned16(q) || !aligned16(k_chunk) || !aligned16(v_chunk) || !aligned16(o_part) || ((uintptr_t)lse_part & 3u)) return RINGATTN_ERR_ALIGN;
  const int rc = ensure_tables(plan, (hipStream_t)stream);  // whether or not this step reads them: the merge will
  if (rc != RINGATTN_OK) return rc;
  const Derived& d = plan->d;
  const int j = (rank + step) % P;
  const int64_t q_rows = d.start[rank + 1] - d.start[rank], kv_rows = d.start[j + 1] - d.start[j];
  ringattn::BlockArgs a;
  fill_geometry(a, plan->p, d);
  a.q = q;
  a.k = k_chunk;
  a.v = v_chunk;
  a.o_part = o_part;
  a.lse_part = lse_part;
  a.bh_stride = q_rows * plan->p.dim;      // every tensor holds one rank's rows only
  a.kv_bh_stride = kv_rows * plan->p.dim;
  a.S = (int)q_rows;
  // an empty slice: nothing of the visited chunk is visible to this rank
  return launch_slice(plan, plan->local[(size_t)rank * P + step], a, (hipStream_t)stream);
}

int ringattn_rank_merge(ringattn_plan* plan, int rank, const void* o_parts, const float* lse_parts, void* out,
                        float* lse, void* stream) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!o_parts || !lse_parts || !out || !lse) return RINGATTN_ERR_NULL;
  if (rank < 0 || rank >= plan->p.npes) return RINGATTN_ERR_RANK;
  if (!aligned16(o_parts) || !aligned16(out) || ((uintptr_t)lse_parts & 3u) || ((uintptr_t)lse & 3u)) return RINGATTN_ERR_ALIGN;
  int rc = ensure_tables(plan, (hipStream_t)stream);
  if (rc != RINGATTN_OK) return rc;
  const Derived& d = plan->d;
  const int rows = d.start[rank + 1] - d.start[rank];
  int first = -1, count = 0, max_len = 0;  // the regions of a rank are consecutive
  for (int i = 0; i < plan->n_regions; ++i)
    if (plan->region_rank[(size_t)i] == rank) {
      if (first < 0) first = i;
      ++count;
      max_len = std::max(max_len, plan->regions[(size_t)i].len);
    }
  if (count == 0) return RINGATTN_OK;
  return launch_regions(plan, plan->n_regions + first, count, max_len, rows, d.BH * (int64_t)rows, o_parts, lse_parts,
                        out, lse, (hipStream_t)stream);
}

int ringattn_plan_work_items(const ringattn_plan* plan, int step, ringattn_work_item* out, int capacity, int* n_out) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!n_out || (capacity > 0 && !out)) return RINGATTN_ERR_NULL;
  if (step < -1 || step >= plan->p.npes) return RINGATTN_ERR_RANK;
  const int begin = step < 0 ? 0 : plan->step_begin[(size_t)step];
  const int end = step < 0 ? plan->fwd_items : plan->step_begin[(size_t)step + 1];
  *n_out = end - begin;
  for (int i = begin; i < end && i - begin < capacity; ++i) {
    const ringattn::WorkItem& w = plan->h_items[(size_t)i];
    out[i - begin] = ringattn_work_item{w.q_start, w.q_len, w.kv_start, w.kv_len, w.diag_off, w.slot};
  }
  return RINGATTN_OK;
}

int ringattn_plan_launch_times(ringattn_plan* plan, float* ms, int capacity, int* n_out) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!n_out || (capacity > 0 && !ms)) return RINGATTN_ERR_NULL;
  if (!plan->timed_forward) return RINGATTN_ERR_PLAN;
  *n_out = 1;
  if (capacity > 0) {
    RA_HIP(hipEventSynchronize(plan->ev_t1));
    RA_HIP(hipEventElapsedTime(&ms[0], plan->ev_t0, plan->ev_t1));
  }
  return RINGATTN_OK;
}

const char* ringattn_plan_forward_kernel(const ringattn_plan* plan) {
  if (!plan_ok(plan)) return nullptr;
  const int mode = step_partials(plan->p) ? ringattn::kBlockPartialsMerged : ringattn::kBlockCarryState;
  if (mode != ringattn::kBlockCarryState && takes_split_steps(plan)) return "ring_split_kernel";
  const bool wide = slice_takes_walk64(plan, forward_slice(plan), mode);
  if (mode == ringattn::kBlockCarryState) {
    const CarryKernel kernel = carry_kernel(plan->walk.costs, plan->p.dim, wide);
    if (kernel != CarryKernel::kWhole) return kernel == CarryKernel::kPair ? "ring_pair_kernel" : "ring_split_kernel";
  }
  return wide ? "ring_walk64_kernel" : "ring_walk_kernel";
}

int ringattn_plan_merge_regions(const ringattn_plan* plan, int* start, int* len, uint64_t* active, int capacity, int* n_out) {
  if (!plan_ok(plan)) return RINGATTN_ERR_PLAN;
  if (!n_out || (capacity > 0 && (!start || !len || !active))) return RINGATTN_ERR_NULL;
  const int n = plan->n_regions;
  *n_out = n;
  for (int i = 0; i < n && i < capacity; ++i) {
    const ringattn::MergeRegion& m = plan->regions[(size_t)i];
    start[i] = m.start;
    len[i] = m.len;
    active[i] = m.active;
  }
  return RINGATTN_OK;
}

int ringattn_merge(const float* o_parts, const float* lse_parts, int n_parts, int64_t rows, int dim,
                   int dtype, void* out, float* lse, void* stream) {
  if (!o_parts || !lse_parts || !out || !lse) return RINGATTN_ERR_NULL;
  if (n_parts < 1 || n_parts > ringattn::kMaxParts) return RINGATTN_ERR_NPES;
  if (dim != 64 && dim != 128) return RINGATTN_ERR_DIM;
  if (dtype != RINGATTN_DTYPE_FP16 && dtype != RINGATTN_DTYPE_BF16) return RINGATTN_ERR_DTYPE;
  if (rows < 0 || rows > ((int64_t)1 << 40)) return RINGATTN_ERR_SHAPE;
  if (!aligned16(o_parts) || !aligned16(out)) return RINGATTN_ERR_ALIGN;
  // one launch per 2^30 rows (a launch's row count is an int)
  const int64_t kChunk = (int64_t)1 << 30;
  for (int64_t r0 = 0; r0 < rows; r0 += kChunk) {
    const int len = (int)std::min(kChunk, rows - r0);
    ringattn::MergeArgs m;
    std::memset(&m, 0, sizeof(m));
    m.o_parts = o_parts + r0 * dim;
    m.lse_parts = lse_parts + r0;
    m.out = (char*)out + r0 * dim * 2;
    m.lse = lse + r0;
    m.single = ringattn::MergeRegion{0, len, n_parts >= 64 ? ~(uint64_t)0 : (((uint64_t)1 << n_parts) - 1)};
    m.n_regions = 1;
    m.max_len = len;
    m.heads = 1;
    m.S = len;
    m.part_stride_rows = rows;
    m.part_rows = (int64_t)len * n_parts;
    RA_HIP(ringattn::launch_merge(m, dtype, dim, (hipStream_t)stream));
  }
  return RINGATTN_OK;
}

int ringattn_ring_attention(const void* q, const void* k, const void* v, void* out, float* lse,
                            int npes, int mype, const int* seqlen, int dim, int max_seq,
                            int dtype, int causal, float softmax_scale) {
  RankCall rc_;
  int rc = prepare_rank_call(&rc_, q, k, v, out, npes, mype, seqlen, dim, max_seq, dtype, causal, softmax_scale);
  if (rc != RINGATTN_OK) return rc;
  rc = run_rank_call(rc_, q, k, v, out, lse, nullptr);
  hipError_t e = hipDeviceSynchronize();  // blocking, as csrc/ring_attention.cu:721
  if (rc == RINGATTN_OK && e != hipSuccess) rc = hip_fail(e);
  return rc;
}

// (an upper bound since the launch carries its one range in its arguments: nothing of it is used)
size_t ringattn_noalloc_scratch_bytes(void) { return 4096; }

int ringattn_ring_attention_noalloc(const void* q, const void* k, const void* v, void* out, float* lse,
                                    int npes, int mype, const int* seqlen, int dim, int max_seq,
                                    int dtype, int causal, float softmax_scale, void* stream) {
  RankCall rc_;
  int rc = prepare_rank_call(&rc_, q, k, v, out, npes, mype, seqlen, dim, max_seq, dtype, causal, softmax_scale);
  if (rc != RINGATTN_OK) return rc;
  return run_rank_call(rc_, q, k, v, out, lse, (hipStream_t)stream);
}

const char* ringattn_strerror(int code) {
  switch (code) {
    case RINGATTN_OK: return "ok";
    case RINGATTN_ERR_NULL: return "a required pointer is NULL";
    case RINGATTN_ERR_NPES: return "npes out of range";
    case RINGATTN_ERR_DIM: return "dim must be 64 or 128";
    case RINGATTN_ERR_DTYPE: return "dtype must be fp16 (0) or bf16 (1)";
    case RINGATTN_ERR_SEQLEN: return "per-rank sequence lengths must be positive (even with the zigzag layout), and max_seq at least the longest";
    case RINGATTN_ERR_SHAPE: return "batch/heads/kv_heads/layout/scale invalid or sizes overflow";
    case RINGATTN_ERR_WORKSPACE: return "workspace too small";
    case RINGATTN_ERR_RANK: return "rank or step outside [0, npes)";
    case RINGATTN_ERR_PLAN: return "invalid or destroyed plan";
    case RINGATTN_ERR_HIP: return "HIP runtime error";
    case RINGATTN_ERR_ALLOC: return "allocation failed";
    case RINGATTN_ERR_ALIGN: return "pointer not sufficiently aligned";
    default: return "unknown ringattn error";
  }
}

int ringattn_last_hip_error(void) { return g_last_hip_error; }

}  // extern "C"
