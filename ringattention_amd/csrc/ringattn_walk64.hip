// gfx950 (CDNA4) kernel: block attention over the ring steps of 256 query rows, 64 rows per wave.
//
//   ring_walk64_kernel : the forward of ring_walk_kernel (ringattn_walk.hip; the reference's CTA
//       that walks its ring steps with max / sum / acc-O in registers,
//       csrc/ring_attention.cu:439-443,456-620, epilogue :621-664; or, chunk by chunk, with a partial
//       (O, LSE) per ring step and their merge at the end), laid out for ONE wave
//       per SIMD: a workgroup of FOUR waves owns the same 256 query rows, each wave two 32-query
//       blocks.  Every K fragment and every V^T fragment read from LDS then feeds two MFMAs (one per
//       block) instead of one: half the LDS fragment traffic per MFMA.  With 512 registers per wave
//       the tile pipeline is skewed by a tile on either side so that, within one iteration, the
//       matrix work and the vector work have no dependence on each other and interleave freely in
//       the single instruction stream:
//           iteration u :  S(u+1) = K(u+1) Q^T   |   P(u) = exp2(S(u) k2 - m k2), row sums   |   O += P(u-1) V(u-1)
//       The exponentials are taken against the reference max as it stands; out of line, and only when a sum of four of
//       them came out above 2^14, the reference moves (rescale of l and acc-O, :226-232) and they are taken again.
//       The KV chunks of a segment are walked as ONE sequence of 32-key tiles (the diagonal chunk
//       last): a chunk boundary is only a jump of the load address.
//       One wave per SIMD has nobody to wait behind, so nothing may be waited for: the K and V rings are eight
//       tiles deep (128 KB of LDS) and a tile is loaded four or more iterations before the barrier that hands it
//       over (s_waitcnt vmcnt(12): the loads of the last three iterations stay in flight).
//       Described for d = 128; at d = 64 (state carried only) a tile is 4 KB, an iteration has 16 MFMAs and the
//       rings take 64 KB.  Shapes it takes: every KV range a multiple of 32 keys and at least 128 (the host checks);
//       anything else runs ring_walk_kernel.
#include "ringattn_device.h"

#include <type_traits>

namespace ringattn {

// Merge of the workgroup's 256 rows over the partials the workgroup has written (the arithmetic and its order are
// MergeState's, so the bits are the merge kernel's).  With one wave
// per SIMD nobody covers for a wave that waits for memory, so the partial rows are not fetched into registers a
// batch at a time but streamed through LDS, which the rings have left free: every wave merges eight rows of each
// group of 32 and keeps six blocks (eight rows of one part: 4 KB, 2 KB as fp16) in flight in a ring of its own,
// with no barrier between the waves.  LDS: the partial LSEs [parts][256], the parts' first rows, the four rings.
constexpr int kStagedMergeMaxParts = 24;  // LSEs of at most this many parts fit below the rings
template <int DT, bool HP>
static __device__ __forceinline__ void merge_rows_staged(const BlockArgs& a, const Segment& seg, int bh, int qt,
                                                         unsigned char* smem, unsigned smem_base) {
  constexpr int D = 128, BM = kWalkM;
  constexpr int RB = HP ? D * 2 : D * 4;  // bytes per partial row
  constexpr int SLOT = 8 * RB;            // a block: eight rows of one part
  constexpr int LPB = SLOT / 1024;        // load instructions per block (1 KB per wave and instruction)
  constexpr int NS = 6;                   // blocks in flight per wave
  constexpr int PPR = RB / 16;            // 16-byte pieces per row
  constexpr int NK = PPR / 8;             // pieces per lane and row
  constexpr int CPP = HP ? 8 : 4;         // columns per piece
  constexpr int kBaseAt = kStagedMergeMaxParts * BM * 4;  // behind the LSEs: the parts' first rows (int64 each)
  constexpr int kRingAt = kBaseAt + 1024;  // (every 1 KB transfer stays inside a 1 KB block of LDS)
  static_assert(kStagedMergeMaxParts * 8 <= 1024, "the parts' first rows fit");
  static_assert(kRingAt + 4 * NS * SLOT <= 2 * 8 * 8192 + 8 * (kMaxParts + 4), "inside the kernel's LDS (rings and chunk list)");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_parts = seg.item_count;
  const SegItem* its = a.items + seg.item_begin;
  const int row0 = qt * BM;
  const int rows_here = min(BM, seg.q_len - row0);
  const int n_groups = (rows_here + 31) / 32;
  float* lse_s = (float*)smem;
  int64_t* base_s = (int64_t*)(smem + kBaseAt);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // the partial stores of all waves have completed and are visible to them; the LDS is idle
  for (int i0 = 0; i0 < n_parts; i0 += 8) {  // thread tid: the LSEs of row tid; parts in the order they were walked
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < n_parts) {
        const SegItem* it = its + run_order(seg, i0 + u);
        const int64_t prow = it->part_base + (int64_t)bh * it->part_bh_stride + row0;
        v[u] = tid < rows_here ? a.lse_part[prow + tid] : -INFINITY;
        if (tid == 0) base_s[i0 + u] = prow;
      }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < n_parts) lse_s[(i0 + u) * BM + tid] = v[u];
  }
  __syncthreads();

  // block t = (group, part) in that order; this wave's rows of a group: 32 group + 8 wave + [0, 8)
  const int total = n_groups * n_parts;
  const unsigned ring = smem_base + kRingAt + wave * (NS * SLOT);
  int ig = 0, ii = 0;  // group and part of the next block to issue
  auto issue_block = [&](int slot) {
    const int64_t prow = base_s[ii];
    const uint64_t addr = (uint64_t)(uintptr_t)a.o_part + (uint64_t)prow * RB;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)addr), hi = __builtin_amdgcn_readfirstlane((unsigned)(addr >> 32));
    const char* src = (const char*)(uintptr_t)(((uint64_t)hi << 32) | lo);  // row 0 of the job in part ii
    const int r_first = 32 * ig + 8 * wave;
#pragma unroll
    for (int k = 0; k < LPB; ++k) {
      const int pos = k * 64 + lane;  // 16-byte position within the block
      const int r = pos / PPR, piece = (pos % PPR) ^ (8 * (r & 1));
      const int rr = min(r_first + r, rows_here - 1);  // rows past the end of the segment: its last row again
      load_lds_16_settled(src, rr * RB + piece * 16, ring + slot * SLOT + k * 1024);
    }
    if (++ii == n_parts) {
      ii = 0;
      ++ig;
    }
  };
  for (int t = 0; t < NS && t < total; ++t) issue_block(t);

  const int r8 = lane >> 3, c = lane & 7;
  MergeState st;
  float acc[NK * CPP];
  int cg = 0, ci = 0;  // group and part of the block to consume
  int slot = 0;
  for (int t = 0; t < total; ++t) {
    if (t + NS <= total) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * LPB) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int row = 32 * cg + 8 * wave + r8;  // within the job
    f32x4 x[NK];
    const unsigned char* blk = smem + kRingAt + wave * (NS * SLOT) + slot * SLOT + r8 * RB;
#pragma unroll
    for (int k = 0; k < NK; ++k) x[k] = *(const f32x4*)(blk + (((c + 8 * k) ^ (8 * (r8 & 1))) << 4));
    if (ci == 0) {  // new rows
      st = MergeState();
#pragma unroll
      for (int e = 0; e < NK * CPP; ++e) acc[e] = 0.f;
    }
    const float L = lse_s[ci * BM + row];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the block is in registers: its slot takes the block NS further on
    if (t + NS < total) issue_block(slot);
    if (row < rows_here && L != -INFINITY) {  // (-inf: the identity element, its O may hold anything)
      float keep, w;
      st.weigh(L, keep, w);
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        if (HP) {
          const f16x8 hv = __builtin_bit_cast(f16x8, x[k]);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[8 * k + e] = merge_in_part(acc[8 * k + e], keep, w, (float)hv[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * k + e] = merge_in_part(acc[4 * k + e], keep, w, x[k][e]);
        }
      }
    }
    if (ci == n_parts - 1 && row < rows_here) {  // all parts in: normalise and store
      const float inv = st.inverse();
#pragma unroll
      for (int e = 0; e < NK * CPP; ++e) acc[e] *= inv;
      const int64_t out_row = (int64_t)bh * a.S + seg.q_start + row0 + row;
      typename Elem<DT>::type* orow = (typename Elem<DT>::type*)a.out + out_row * D;
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        if (HP) {
          Store8<DT>::st(orow + (c + 8 * k) * 8, &acc[8 * k]);
        } else {
          typename Elem<DT>::vec4 o4;
#pragma unroll
          for (int e = 0; e < 4; ++e) o4[e] = (typename Elem<DT>::type)acc[4 * k + e];
          *(typename Elem<DT>::vec4*)(orow + (c + 8 * k) * 4) = o4;
        }
      }
      if (c == 0) a.lse[out_row] = st.lse();
    }
    if (++ci == n_parts) {
      ci = 0;
      ++cg;
    }
    slot = slot + 1 == NS ? 0 : slot + 1;
  }
}

// The same merge where the LSEs of the parts leave no room for the staging rings: all of them are parked in LDS (lse_s:
// [items][256] floats), and the partial O rows move through registers in batches of 256 bytes per thread
// (two output rows x four or eight parts), three batches in flight at any time.
typedef __attribute__((address_space(3))) float lds_float;
template <int DT, bool HP>
static __device__ __forceinline__ void merge_job_rows(const void* o_part, const float* lse_part, void* out, float* lse,
                                                      const SegItem* items, const Segment& seg, int bh, int qt, int S,
                                                      lds_float* lse_s) {
  constexpr int D = 128, BM = kWalkM, WAVES = 4, THREADS = 64 * WAVES;
  constexpr int TPR = D / 8;  // threads per row, 8 columns each
  constexpr int ROWS = THREADS / TPR;
  constexpr int KMAX = kMaxParts / WAVES;  // parts per wave in the LSE sweep
  constexpr int LR = BM / 64;              // rows per lane in the LSE sweep
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_parts = seg.item_count;
  const int row0 = qt * BM;  // first row of the job within the segment
  const int last_row = min(BM, seg.q_len - row0) - 1;
  // lane i keeps where the job's rows begin in the partials of the i-th item walked
  int64_t first_row = 0;
  if (lane < n_parts) {
    const SegItem* w = items + seg.item_begin + run_order(seg, lane);
    first_row = w->part_base + (int64_t)bh * w->part_bh_stride + row0;
  }
  auto part_row = [&](int i) -> int64_t {
    return (int64_t)(((uint64_t)(unsigned)__builtin_amdgcn_readlane((int)(first_row >> 32), i) << 32) |
                     (unsigned)__builtin_amdgcn_readlane((int)first_row, i));
  };
  __syncthreads();  // the partial stores of all waves have completed and are visible to them; the LDS is idle
  {
    float v[KMAX][LR];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      const int i = wave + WAVES * k;
      if (i < n_parts) {
        const int64_t prow = part_row(i);
#pragma unroll
        for (int r = 0; r < LR; ++r) v[k][r] = (row0 + lane + 64 * r < seg.q_len) ? lse_part[prow + lane + 64 * r] : -INFINITY;
      }
    }
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      const int i = wave + WAVES * k;
      if (i < n_parts) {
#pragma unroll
        for (int r = 0; r < LR; ++r) lse_s[i * BM + lane + 64 * r] = v[k][r];
      }
    }
  }
  __syncthreads();
  const int c8 = tid % TPR, rsub = tid / TPR;
  // this thread's 8 columns of a partial row: 16 bytes as fp16, 32 as fp32
  constexpr int PB = HP ? 16 : 32;
  constexpr int NV = PB / 16;
  // R rows and G parts of a thread per batch: 64 registers
  constexpr int R = 2, G = HP ? 8 : 4;
  constexpr int RSTEP = R * ROWS;
  const int n_groups = (n_parts + G - 1) / G;
  const int n_batches = (BM / RSTEP) * n_groups;  // batch b: rows of b / n_groups, parts of b % n_groups
  struct Batch {
    f32x4 raw[R][G][NV];  // as loaded; fp16 partials are widened when they are used
  };
  auto row_of = [&](int b, int j) { return (b / n_groups) * RSTEP + j * ROWS + rsub; };  // within the job
  // Every load of a batch is made, those of parts and rows that do not exist from the last one that does: with loads under
  // conditions the compiler cannot count those in flight, and waits for the batches fetched ahead as well.  Where the parts
  // lie comes from a lane of first_row and not from the table, a scalar round trip for each.
  auto fetch = [&](int b, Batch& t) {
    const int i0 = (b % n_groups) * G;
    int at[R];
#pragma unroll
    for (int j = 0; j < R; ++j) at[j] = min(row_of(b, j), last_row) * (D * (PB / 8)) + c8 * PB;
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const char* base = (const char*)o_part + part_row(min(i0 + u, n_parts - 1)) * (D * (PB / 8));
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const f32x4* src = (const f32x4*)(base + at[j] + 16 * v);
          t.raw[j][u][v] = HP ? __builtin_nontemporal_load(src) : *src;
        }
    }
  };
  MergeState st[R];
  float acc[R][8];
  auto accumulate = [&](int b, const Batch& t) {
    const int g = b % n_groups, i0 = g * G;
    if (g == 0) {  // new rows
#pragma unroll
      for (int j = 0; j < R; ++j) {
        st[j] = MergeState();
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[j][e] = 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < G; ++u)
      if (i0 + u < n_parts) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const float L = lse_s[(i0 + u) * BM + row_of(b, j)];
          if (row0 + row_of(b, j) >= seg.q_len || L == -INFINITY) continue;  // identity element: its O may hold anything
          float keep, w;
          st[j].weigh(L, keep, w);
          float x[8];
          if (HP) {
            const f16x8 hv = __builtin_bit_cast(f16x8, t.raw[j][u][0]);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (float)hv[e];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[e] = t.raw[j][u][0][e];
              x[4 + e] = t.raw[j][u][NV - 1][e];
            }
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[j][e] = merge_in_part(acc[j][e], keep, w, x[e]);
        }
      }
    if (g == n_groups - 1) {  // all parts in: normalise and store
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (row0 + row_of(b, j) >= seg.q_len) continue;
        const float inv = st[j].inverse();
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[j][e] *= inv;
        const int64_t out_row = (int64_t)bh * S + seg.q_start + row0 + row_of(b, j);
        Store8<DT>::st((char*)out + (out_row * D + c8 * 8) * 2, acc[j]);
        if (c8 == 0) lse[out_row] = st[j].lse();
      }
    }
  };
  // three batches in flight
  Batch t0, t1, t2;
  fetch(0, t0);
  if (1 < n_batches) fetch(1, t1);
  int b = 0;
#pragma unroll 1
  for (; b + 4 < n_batches; b += 3) {
    fetch(b + 2, t2);
    accumulate(b, t0);
    fetch(b + 3, t0);
    accumulate(b + 1, t1);
    fetch(b + 4, t1);
    accumulate(b + 2, t2);
  }
#pragma unroll 1
  for (; b < n_batches; b += 3) {
    if (b + 2 < n_batches) fetch(b + 2, t2);
    accumulate(b, t0);
    if (b + 3 < n_batches) fetch(b + 3, t0);
    if (b + 1 < n_batches) accumulate(b + 1, t1);
    if (b + 4 < n_batches) fetch(b + 4, t1);
    if (b + 2 < n_batches) accumulate(b + 2, t2);
  }
}

// KEEP: max / sum / acc-O run through all chunks of the q tile and the rows' result is written once (kBlockCarryState).
// Otherwise the chunks are walked one by one, each as a sequence of its own -- prologue, loop, drain --, and each
// ends in its normalised partial (O, LSE) (kBlockPartials, kBlockPartialsMerged; HP: partial O as fp16).
// D = 64 (state carried only): half the MFMAs per tile for the same vector work, 4 KB tiles (one 1 KB piece per wave),
// 64 KB of rings.
template <int DT, int D, bool KEEP, bool HP>
__global__ __launch_bounds__(256, 1) void ring_walk64_kernel(const BlockArgs a) {
  using E = Elem<DT>;
  static_assert(D == 128 || (D == 64 && KEEP && !HP), "d = 64 is built with the state carried only");
  constexpr int WAVES = 4;
  constexpr int BM = kWalkM;       // query rows per workgroup: 4 waves x 64
  constexpr int BN = 32;           // keys per tile
  constexpr int NBUF = 8;          // ring depth of the K and of the V tiles: loads run seven to eight tiles ahead of the products
  constexpr int CPR = D / 8;       // 16-byte chunks per row
  constexpr int ROWB = D * 2;      // bytes per row
  constexpr int TILE = BN * ROWB;  // bytes per tile
  constexpr int PIECES = TILE / 4096;  // 1 KB pieces of a tile per wave
  constexpr int KS = D / 16;       // contraction slices of QK^T
  constexpr int DB = D / 32;       // 32-wide blocks of the head dim in PV
  static_assert(BM == 64 * WAVES, "two 32-row blocks per wave");
  constexpr int kListAt = 2 * NBUF * TILE;  // behind the rings: the chunks of this q tile in walking order, (byte offset, tiles) each
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kListAt + 8 * (kMaxParts + 4)];

  const unsigned smem_base = lds_offset(smem);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;

  Segment seg;
  int bh, qt;
  if (!decode_job<BM>(a, seg, bh, qt)) return;
  const int q_start = seg.q_start, q_len = seg.q_len;
  const int all_items = seg.item_count;
  const ItemPtr items = items_of(a);
  // items in run order: table order, except that item `last_item` (the diagonal one) is moved to the end
  auto item_in_order = [&](int i) -> ItemPtr { return items + seg.item_begin + run_order(seg, i); };
  const int64_t head_off = (int64_t)bh * a.bh_stride;
  const int kv_bh = quotient(bh, a.by_group);
  const int64_t kv_head_off = (int64_t)kv_bh * a.kv_bh_stride;
  const char* qbase = (const char*)a.q + (head_off + (int64_t)(q_start + qt * BM) * D) * 2;
  const char* k_head = (const char*)a.k + kv_head_off * 2;
  const char* v_head = (const char*)a.v + kv_head_off * 2;

  // Q of this lane's two rows (B operands for the whole launch); rows beyond the range read the last valid row
  s16x8 qf[2][KS];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int ql = min(qt * BM + 64 * wave + 32 * b + n, q_len - 1) - qt * BM;
    const char* qrow = qbase + (int64_t)ql * ROWB + h * 16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[b][ks] = *(const s16x8*)(qrow + ks * 32);
  }
  // the 1 KB pieces of a tile this wave loads (d = 128: pieces 2 wave and 2 wave + 1 of eight; d = 64: piece wave of four)
  int goff_k[PIECES], goff_v[PIECES];
#pragma unroll
  for (int j = 0; j < PIECES; ++j) {
    const int pk = (PIECES * wave + j) * 64 + lane;
    goff_k[j] = (pk / CPR) * ROWB + (((pk % CPR) ^ k_swizzle<D>(pk / CPR)) << 4);
    goff_v[j] = (pk / CPR) * ROWB + (((pk % CPR) ^ v_swizzle<D>(pk / CPR)) << 4);
  }
  int koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = n * ROWB + (((2 * ks + h) ^ k_swizzle<D>(n)) << 4);
  int voff[DB];
  {
    const int s = lane & 15, g1 = (lane >> 4) & 1;
    const int row8 = 4 * h + (s >> 2);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int c = 2 * (2 * db + g1) + ((s & 3) >> 1);
      voff[db] = row8 * ROWB + ((c ^ v_swizzle<D>(row8)) << 4) + ((s & 1) << 3);
    }
  }

  // ---- a pass walks n_items chunks from item `first` on as one sequence: all of them (KEEP), or one
  const int n_items = KEEP ? all_items : 1;
  for (int first = 0; first < all_items; first += n_items) {
  auto item_at = [&](int i) -> ItemPtr { return item_in_order(first + i); };
  // ---- the flattened tile sequence of the pass: item i contributes tiles_of(i) tiles
  const int diag_item = (n_items > 0 && item_at(n_items - 1)->diag_off >= 0) ? n_items - 1 : -1;
  auto tiles_of = [&](ItemPtr w) {
    const int kv_tiles = w->kv_len / BN;
    return w->diag_off >= 0 ? min(kv_tiles, (w->diag_off + qt * BM + BM - 1) / BN + 1) : kv_tiles;
  };
  int N = 0;
  for (int i = 0; i < n_items; ++i) N += tiles_of(item_at(i));
  // this wave's share of the diagonal chunk: tiles below Mw are visible to all its rows, tiles from Ew on to none
  int Mw = N, Ew = N, diag_base = 0, diag_rows = 0;
  if (diag_item >= 0) {
    const ItemPtr w = item_at(diag_item);
    const int n_last = tiles_of(w);
    diag_base = N - n_last;
    diag_rows = w->diag_off + qt * BM;  // keys below this local index are visible to the whole q tile
    Mw = diag_base + min(n_last, (diag_rows + 64 * wave + 1) / BN);
    Ew = diag_base + min(n_last, (diag_rows + 64 * wave + 63) / BN + 1);
  }

  // ---- load streams: K is loaded seven to eight tiles ahead of its product, V four to five.  A stream is a byte
  // offset from the head's first row; past the last chunk it goes round the first four tiles of the head (valid
  // memory: some KV range of 128 keys lies in every head; nobody reads these tiles from LDS), so that every
  // iteration issues the same number of loads.  At most nine tiles are loaded past the end: three such rounds.
  struct Stream {
    unsigned off;  // the next tile to load
    int left;      // tiles left in its chunk, that one included
    int idx;       // the chunk
  };
  auto chunk_of = [&](int i, unsigned& off, int& cnt) {
    if (i < n_items) {
      const ItemPtr w = item_at(i);
      off = (unsigned)w->kv_start * ROWB;
      cnt = tiles_of(w);
    } else {
      off = 0;
      cnt = 4;
    }
  };
  auto step = [&](Stream& s) {
    s.off += TILE;
    if (--s.left == 0) {
      s.idx += 1;
      chunk_of(s.idx, s.off, s.left);
    }
  };
  Stream kst, vst;
  kst.idx = vst.idx = 0;
  chunk_of(0, kst.off, kst.left);
  chunk_of(0, vst.off, vst.left);
  auto issue_k = [&](int slot) {
    const unsigned dst = __builtin_amdgcn_readfirstlane(smem_base + slot * TILE + PIECES * wave * 1024);
    const char* p = k_head + __builtin_amdgcn_readfirstlane(kst.off);
#pragma unroll
    for (int j = 0; j < PIECES; ++j) load_lds_16_settled(p, goff_k[j], dst + 1024 * j);
    step(kst);
  };
  auto issue_v = [&](int slot) {
    const unsigned dst = __builtin_amdgcn_readfirstlane(smem_base + (NBUF + slot) * TILE + PIECES * wave * 1024);
    const char* p = v_head + __builtin_amdgcn_readfirstlane(vst.off);
#pragma unroll
    for (int j = 0; j < PIECES; ++j) load_lds_16_settled(p, goff_v[j], dst + 1024 * j);
    step(vst);
  };

  // ---- softmax state of the two blocks
  float m[2] = {-INFINITY, -INFINITY};  // reference max (raw score units)
  float ms[2] = {0.f, 0.f};             // m * k2, kNoReference while m is -inf (guard of csrc/ring_attention.cu:183)
  float ls[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  f32x16 oacc[2][DB];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[b][db][e] = 0.f;
  f32x16 sacc[2];     // scores of tile u, consumed by the exponentials of iteration u
  s16x8 pprev[2][2];  // probabilities of tile u-1 (B operands), consumed by the PV product of iteration u
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int e = 0; e < 16; ++e) sacc[b][e] = 0.f;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int e = 0; e < 8; ++e) pprev[b][t2][e] = 0;
  }

  // S^T = K Q^T of one 32-key tile for both blocks (csrc/ring_attention.cu:565): each K fragment feeds two MFMAs
  auto qk = [&](int kbytes, f32x16 (&s)[2]) {
    const unsigned char* ks_lds = smem + kbytes;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[b][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const s16x8 kfr = *(const s16x8*)(ks_lds + koff[ks]);
      s[0] = E::mma(kfr, qf[0][ks], s[0]);
      s[1] = E::mma(kfr, qf[1][ks], s[1]);
    }
  };
  // max(m, row max of the tile): two chains of v_max3_f32, one exchange between the halves of the wave
  auto tile_max = [&](const f32x16& s, float mb) {
    float m0 = mb, m1 = mb;
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      m0 = fmaxf(fmaxf(m0, s[e]), s[e + 1]);
      m1 = fmaxf(fmaxf(m1, s[e + 2]), s[e + 3]);
    }
    return cross_half_max(fmaxf(m0, m1));
  };
  // causal mask of flattened tile t (a tile of the diagonal chunk): key visible iff key_local <= query_local + diag_off
  auto mask_tile = [&](f32x16 (&s)[2], int t) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int lim = diag_rows + 64 * wave + 32 * b + n - (t - diag_base) * BN - 4 * h;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = 8 * (e >> 2) + (e & 3);
        if (key > lim) s[b][e] = -INFINITY;
      }
    }
  };
  // ---- prologue: K(0) .. K(6) and V(0) .. V(4) next to the Q loads; the scores of tile 0.  V ring slot 7 -- "tile
  // -1", which the first iteration multiplies with all-zero probabilities -- is cleared.
  if (first > 0) __syncthreads();  // every wave is done with the rings and the chunk list of the pass before
  for (int t = 0; t < 7; ++t) issue_k(t);
  for (int t = 0; t < 5; ++t) issue_v(t);
  if (tid < n_items + 4) {  // the chunk list the hand-scheduled loop steps its load streams through
    unsigned o;
    int c;
    chunk_of(tid, o, c);
    *(int2*)(smem + kListAt + 8 * tid) = int2{(int)o, c};
  }
  {
    f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TILE / 4096; ++j) *(f32x4*)(smem + (NBUF + 7) * TILE + tid * (TILE / 256) + 16 * j) = zero;
  }
  __builtin_amdgcn_s_waitcnt(0);  // retire the Q loads with a wait the compiler can see (and the tiles)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // (every wave has a tile: the first key of the sequence is visible to all rows)
  qk(0, sacc);
  if (0 >= Mw) mask_tile(sacc, 0);
#pragma unroll
  for (int b = 0; b < 2; ++b) {  // the first reference: the row maxima of tile 0
    m[b] = tile_max(sacc[b], m[b]);
    ms[b] = (m[b] == -INFINITY) ? kNoReference : m[b] * a.scale_log2;
  }

  // LDS addresses for the hand-scheduled loop: fragment offsets from the start of LDS, and where this wave's two
  // tile pieces go in ring slot 0 of K and of V
  int koff_a[KS], voff_a[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff_a[ks] = koff[ks] + (int)smem_base;
#pragma unroll
  for (int db = 0; db < DB; ++db) voff_a[db] = voff[db] + (int)smem_base + NBUF * TILE;  // from the start of the V ring
  const unsigned lds_dst_k = __builtin_amdgcn_readfirstlane(smem_base + PIECES * wave * 1024);
  const unsigned lds_dst_v = lds_dst_k + NBUF * TILE;
  auto uni = [](unsigned x) { return (unsigned)__builtin_amdgcn_readfirstlane((int)x); };
  const unsigned kh_lo = uni((unsigned)(uintptr_t)k_head), kh_hi = uni((unsigned)((uintptr_t)k_head >> 32));
  const unsigned vh_lo = uni((unsigned)(uintptr_t)v_head), vh_hi = uni((unsigned)((uintptr_t)v_head >> 32));
  const unsigned k2_bits = uni(__builtin_bit_cast(unsigned, a.scale_log2));

  // The hand-scheduled loop (ringattn_walk64_loop.inc) runs all iterations of the workgroup, 0 to N: every iteration
  // whose score tile u+1 this wave computes -- masking the tiles of the diagonal chunk that need it --, the wave's last
  // two iterations, and then only the wave's share of the loads and the barriers.  Every wave goes through it: the
  // barriers and tile loads in it are the workgroup's.  (A wave has two tiles at least: a range is four, and of a diagonal
  // one the first 64 keys are visible to some row of every wave.  The loop would do with one.)
  {
    unsigned asm_u = 0, asm_far = 0;
    const unsigned asm_stop = uni((unsigned)(Ew - 1)), asm_mw1 = uni((unsigned)(Mw - 1));
    int vlim[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) vlim[b] = diag_rows + 64 * wave + 32 * b + n - 4 * h - (1 - diag_base) * BN;
    const uint64_t kp = (uint64_t)(uintptr_t)k_head + kst.off, vp = (uint64_t)(uintptr_t)v_head + vst.off;
    unsigned k_lo = uni((unsigned)kp), k_hi = uni((unsigned)(kp >> 32)), v_lo = uni((unsigned)vp), v_hi = uni((unsigned)(vp >> 32));
    unsigned k_left = uni((unsigned)kst.left), v_left = uni((unsigned)vst.left);
    unsigned k_next = uni(smem_base + kListAt + 8 * (kst.idx + 1)), v_next = uni(smem_base + kListAt + 8 * (vst.idx + 1));
    const unsigned asm_n = uni((unsigned)N);
    if constexpr (D == 128) {
#include "ringattn_walk64_loop.inc"
    } else {
#include "ringattn_walk64_loop_d64.inc"
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  if (KEEP) {
    // ---- the rows' result: the reference's epilogue (csrc/ring_attention.cu:621-664), O = acc / l in the storage
    // type, plus the LSE
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float l = cross_half_sum((ls[b][0] + ls[b][1]) + (ls[b][2] + ls[b][3]));
      const float inv = (l > 0.f) ? 1.f / l : 0.f;
      const int row0 = qt * BM + 64 * wave + 32 * b;
      const int64_t row = (int64_t)bh * a.S + q_start + row0;  // the block's first row
      store_block<DT, D>(oacc[b], inv, (char*)a.out + row * ROWB, ROWB, q_len - row0);
      if (h == 0 && row0 + n < q_len && a.lse)
        a.lse[row + n] = (l > 0.f) ? (ms[b] + __builtin_amdgcn_logf(l)) * 0.6931471805599453f : -INFINITY;
    }
  } else {
    // ---- the chunk's partial (csrc/ring_attention.cu:621-633): normalised O and LSE at the rows of the queries
    const ItemPtr w = item_at(0);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float l = cross_half_sum((ls[b][0] + ls[b][1]) + (ls[b][2] + ls[b][3]));
      const float inv = (l > 0.f) ? 1.f / l : 0.f;
      const int row0 = qt * BM + 64 * wave + 32 * b;
      int64_t prow = w->part_base + (int64_t)bh * w->part_bh_stride + row0;  // of the block's first row
      const int step = w->part_row_mul > 0 ? w->part_row_mul : 1;            // n: a row's steps next to each other
      if (w->part_row_mul > 0) prow = prow * step + w->slot;
      constexpr int PB = HP ? 2 : 4;  // fp16 partials: |O_part| <= max |V|, the caller vouches that this fits
      store_block<HP ? 0 : 2, D>(oacc[b], inv, (char*)a.o_part + prow * (D * PB), (int64_t)step * (D * PB), q_len - row0);
      if (h == 0 && row0 + n < q_len)
        a.lse_part[prow + (int64_t)n * step] = (l > 0.f) ? (ms[b] + __builtin_amdgcn_logf(l)) * 0.6931471805599453f : -INFINITY;
    }
  }
  }  // passes
  if constexpr (!KEEP) {
    if (a.mode == kBlockPartialsMerged) {  // this workgroup's rows over the partials it has just written
      if (all_items <= kStagedMergeMaxParts)
        merge_rows_staged<DT, HP>(a, seg, bh, qt, smem, smem_base);
      else
        merge_job_rows<DT, HP>(a.o_part, a.lse_part, a.out, a.lse, a.items, seg, bh, qt, a.S,
                               (lds_float*)(__attribute__((address_space(3))) void*)smem);
    }
  }
}

hipError_t launch_walk64(BlockArgs a, int dtype, int dim, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int q_tiles = a.q_tiles_max;
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (q_tiles <= 0 || blocks > INT32_MAX) return hipErrorInvalidValue;
  if (a.mode != kBlockCarryState && a.mode != kBlockPartials && a.mode != kBlockPartialsMerged) return hipErrorInvalidValue;
  if (dtype != 0 && dtype != 1) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  if (dim == 64) {  // state carried only
    if (a.mode != kBlockCarryState) return hipErrorInvalidValue;
    if (dtype == 0) ring_walk64_kernel<0, 64, true, false><<<grid, 256, 0, stream>>>(a);
    else ring_walk64_kernel<1, 64, true, false><<<grid, 256, 0, stream>>>(a);
    return hipGetLastError();
  }
  if (dim != 128) return hipErrorInvalidValue;
#define RA_LAUNCH_WALK64(DT_)                                                                            \
  do {                                                                                                  \
    if (a.mode == kBlockCarryState) ring_walk64_kernel<DT_, 128, true, false><<<grid, 256, 0, stream>>>(a);  \
    else if (a.half_partials) ring_walk64_kernel<DT_, 128, false, true><<<grid, 256, 0, stream>>>(a);        \
    else ring_walk64_kernel<DT_, 128, false, false><<<grid, 256, 0, stream>>>(a);                            \
  } while (0)
  if (dtype == 0) RA_LAUNCH_WALK64(0);
  else RA_LAUNCH_WALK64(1);
#undef RA_LAUNCH_WALK64
  return hipGetLastError();
}

}  // namespace ringattn
