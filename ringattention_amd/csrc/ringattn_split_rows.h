// gfx950 (CDNA4) kernel: block attention for launches with few query rows.  The workgroup's program; ringattn_split.hip,
// ringattn_split_steps.hip and ringattn_split_columns.hip wrap it into kernels.
//
//   ring_split_kernel : the forward of ring_walk_kernel and ring_walk64_kernel (the reference's CTA that walks its ring
//       steps with max / sum / acc-O in registers, csrc/ring_attention.cu:439-443,456-620, epilogue :621-664) with the
//       work split over the KEYS inside a workgroup: all WAVES (eight; sixteen at d = 64 where a compute unit
//       has only one workgroup) own the same 32 query rows, wave w takes the 32-key tiles w, w + WAVES, ...
//       of the rows' key ranges with a softmax state of its own, and the states are combined through LDS at the end (the rescale of
//       :226-232 once more, across waves instead of tiles).
//       A workgroup of the other kernels owns 256 rows, so a launch of 8192 rows has 32 workgroups on 256 compute units;
//       here it has 256, and the walk of a workgroup is an eighth as long.
//
//       Nothing is shared between the waves until the end, so there is no barrier in the loop: a wave loads its own
//       tiles (one K and one V tile of LDS per wave).  One buffer each is enough (with two, which leaves a compute unit at d = 64 one
//       workgroup, nothing got faster): the next K tile is fetched as soon as
//       the fragments of this one are in registers and has the products, the softmax and the PV product to arrive in, the next V tile
//       has the QK^T product and the softmax; two (d = 64: four) waves per SIMD overlap one another's matrix and vector
//       phases without any coordination.
//       What bounds it: a K/V tile fetched from L2 feeds 32 query rows instead of 256, and a compute unit takes in 46 (d = 64) to
//       50 (d = 128) of the 64 bytes per clock that its path to L2 carries (34 with all of them busy).  A full device reaches 730 TFLOP/s at d = 128 and
//       690 at d = 64 (ring_walk64_kernel 1260 and 940), so this kernel is for launches that leave it compute units idle: the
//       host weighs the kernels (carry_kernel in ringattn_api.hip).  A tile costs a wave 75 vector and 52 scalar instructions (93 and
//       100 before its place became a count that only the end of a range sends to the table, pieces within
//       4 KB shared M0 and address, and the first score of a row overflowed into the branch that moves its reference: 8192 rows x
//       16384 keys, d = 64, 60.2 -> 54.4 us, 8192 x 8192, d = 128, 57 -> 53).
//       A launch of two tiles a wave (4 ranks x 128 tokens, d = 64) took, of 6.0 us, 2.1 for any launch, 0.5 to find its place, 0.5 for Q and
//       the first tiles, 1.5 for the tiles and 1.4 for the combination, half of that in reads of one wave's state after the
//       other behind a branch on whether that wave had seen anything.  The reads of all waves are on their way together now, the
//       factor of a state comes with its reader, which spares a barrier, and the next K tile is asked for behind the first product of the
//       chain and not behind the last: 5.46 us; 256 rows x 256 keys 5.45 -> 4.84, 640 x 640 6.76 -> 6.15, 1280 x 8960 causal 24.9 -> 24.0;
//       d = 128, 4 heads x 256 7.18 -> 6.89, 512 x 2048 causal 13.8 -> 13.5.
//       Where a launch has so few row tiles that it leaves compute units idle, the COLUMNS of V and O are dealt to workgroups
//       as well: each takes all of K and 64 or 32 columns of V.  A compute unit then takes in three quarters (d = 128, half
//       the columns) of the bytes a tile, has half or a quarter of the products of P V to do, and as much less to put together at
//       the end; scores are computed once per workgroup.  The columns of a row do not meet, so the bits are the same.  us before and after:
//       d = 128, 512 rows x 2048 causal 13.5 -> 11.0, 512 x 512 8.0 -> 6.7, 1024 x 1024 10.1 -> 8.4, 512 x 8192 37.5 -> 27.8;
//       d = 64, 512 x 512 5.5 -> 5.2, 1024 x 1024 6.9 -> 6.4; how many columns: split_columns in ringattn_api.hip.
#pragma once
#include "ringattn_device.h"

namespace ringattn {

// LDS of a wave: its K tile and C columns of its V tile; at the end its acc-O.
template <int D, int C = D> constexpr int kSplitWaveLds = 64 * D + 64 * C;
// LDS of a workgroup that merges the steps of its rows: eight waves', the ranges, and ten numbers to eight columns of a row
template <int D> constexpr int kSplitStepsLds = 8 * kSplitWaveLds<D> + 16 * kMaxParts + 4 * 10 * kSplitM * (D / 8);

// The steps apart: the waves that share a key range of so many tiles, each with a run of up to four of them while there are waves; one,
// two, four or all eight, so that whole ranges fill the workgroup.  It goes by the range alone: its partial has the same bits
// in every launch.
static __device__ __forceinline__ int split_units(int tiles) { return tiles <= 4 ? 1 : tiles <= 8 ? 2 : tiles <= 16 ? 4 : 8; }

// MODE: one state of the rows through all of their keys (kBlockCarryState), or one per key range, whose partial is stored
// (kBlockPartials) or merged into the rows' result (kBlockPartialsMerged); HP: partial O rounded to fp16.
// C: the columns of V and O that a workgroup has, blockIdx.y the how many-th of them.
template <int DT, int D, int C, int WAVES, bool HP, int MODE>
static __device__ __forceinline__ void split_rows(const BlockArgs& a, unsigned char* smem, float2 (*stat)[kSplitM]) {
  using E = Elem<DT>;
  constexpr int BM = kSplitM;      // query rows per workgroup, all of them in every wave
  constexpr int BN = 32;           // keys per tile
  constexpr int CPR = D / 8;       // 16-byte chunks per row
  constexpr int ROWB = D * 2;      // bytes per row
  constexpr int TILE = BN * ROWB;  // bytes per K tile
  constexpr int ROWV = C * 2;      // bytes per row of a V tile
  constexpr int KS = D / 16;       // contraction slices of QK^T
  constexpr int DB = C / 32;       // 32-wide blocks of the head dim in PV
  constexpr int PIECES_K = TILE / 1024, PIECES_V = BN * ROWV / 1024;  // 1 KB wave-loads per tile
  static_assert(BM == 32, "one 32-row block");
  constexpr int WREG = kSplitWaveLds<D, C>;
  static_assert(WREG == TILE + BN * ROWV && WREG >= BM * C * 4, "acc-O of a wave as fp32 takes the place of its tiles");
  constexpr bool KEEP = MODE == kBlockCarryState, MERGE = MODE == kBlockPartialsMerged;
  static_assert(KEEP || WAVES == 8, "split_units");
  static_assert(C == D || !MERGE, "kSplitStepsLds");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;

  if (!KEEP) fetch_arguments(a);
  Segment seg;
  int bh, qt;
  if (!decode_job<BM>(a, seg, bh, qt)) return;
  const int n_items = MODE == kBlockPartials ? 1 : seg.item_count;
  const int q0 = qt * BM;  // first row of the tile within the segment
  const int q_last = min(q0 + BM, seg.q_len) - 1;
  const ItemPtr items = items_of(a) + seg.item_begin;  // the order they are walked in does not matter to a carried state

  const int64_t head_off = (int64_t)bh * a.bh_stride;
  // grouped-query attention: query head h of a batch entry reads KV head h / kv_group, and heads are whole groups
  const int kv_bh = quotient(bh, a.by_group);
  const char* k_head = (const char*)a.k + (int64_t)kv_bh * a.kv_bh_stride * 2;
  const int column = C == D ? 0 : blockIdx.y * C;  // this workgroup's first
  const char* v_head = (const char*)a.v + ((int64_t)kv_bh * a.kv_bh_stride + column) * 2;

  // Q of this lane's row (B operands for the whole launch); rows beyond the range read the last valid row
  s16x8 qf[KS];
  {
    const char* qrow = (const char*)a.q + (head_off + (int64_t)(seg.q_start + min(q0 + n, q_last)) * D) * 2 + h * 16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const s16x8*)(qrow + ks * 32);
  }

  // ---- LDS of this wave, fragment offsets, load offsets
  unsigned char* my = smem + wave * WREG;
  const unsigned my_lds = lds_offset(smem) + wave * WREG;
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
      voff[db] = TILE + row8 * ROWV + ((c ^ v_swizzle<C>(row8)) << 4) + ((s & 1) << 3);
    }
  }
  // Offsets of this lane's 16 bytes within a 1 KB piece of a tile; the swizzles repeat after a few pieces.  A load instruction's
  // own offset moves both ends, so pieces up to 4 KB apart share a base address and an M0 (d = 128 needs two of each).  With
  // some of the columns of V its pieces lie further apart in memory than in LDS: the difference is in the offsets.
  constexpr int NPK = D == 128 ? 4 : 2, NPV = C < D ? PIECES_V : D == 128 ? 2 : 1;
  int goff_k[NPK], goff_v[NPV];
#pragma unroll
  for (int j = 0; j < NPK; ++j) {
    const int row = lane / CPR;
    goff_k[j] = row * ROWB + (((lane % CPR) ^ k_swizzle<D>(1024 / ROWB * j + row)) << 4);
  }
#pragma unroll
  for (int j = 0; j < NPV; ++j) {
    const int row = lane / (C / 8);
    goff_v[j] = row * ROWB + (((lane % (C / 8)) ^ v_swizzle<C>(1024 / ROWV * j + row)) << 4);
    if (C < D) goff_v[j] += j * (1024 / ROWV * ROWB - 1024);
  }
  // the tile at `base` to `dst`, its rows of ROW bytes; `rows` of it exist (if fewer than 32, the others read the last one of them)
  auto load_tile = [&](const char* base, unsigned dst, int rows, const auto& goff, auto row_bytes) {
    constexpr int NP = sizeof(goff) / sizeof(int), ROW = decltype(row_bytes)::value, PIECES = BN * ROW / 1024;
    if (rows >= BN) {
      if constexpr (PIECES == 2) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024" ::"s"(
                         __builtin_amdgcn_readfirstlane(dst)),
                     "v"(goff[0]), "v"(goff[1 % NP]), "s"(base)
                     : "m0");
      } else {
#pragma unroll
        for (int j = 0; j < PIECES; j += 4)
          asm volatile(
              "s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %5\n\tglobal_load_lds_dwordx4 %2, %5 offset:1024\n\t"
              "global_load_lds_dwordx4 %3, %5 offset:2048\n\tglobal_load_lds_dwordx4 %4, %5 offset:3072" ::"s"(
                  __builtin_amdgcn_readfirstlane(dst + 1024 * j)),
              "v"(goff[j % NP]), "v"(goff[(j + 1) % NP]), "v"(goff[(j + 2) % NP]), "v"(goff[(j + 3) % NP]), "s"(base + 1024 * j)
              : "m0");
      }
    } else {
      int row = 16 * lane / ROW;
      asm volatile("" : "+v"(row));  // (keeps this seldom taken arithmetic from being done ahead of the loop, in registers)
#pragma unroll
      for (int j = 0; j < PIECES; ++j)
        load_lds_16_settled(base, goff[j % NP] + 1024 * j - max(0, 1024 / ROW * j + row - (rows - 1)) * ROWB,
                            __builtin_amdgcn_readfirstlane(dst + 1024 * j));
    }
  };

  // ---- the tiles of this wave.  KEEP: numbers wave, wave + WAVES, ... of the items' tiles laid end to end; the steps apart: a run of
  // tiles of one item
  int item = 0, t = wave, tiles = 0;   // the tile that is loaded next: tile t of `tiles` of item `item`
  int len = 0, diag = -1;
  int64_t start = 0;
  auto enter = [&]() {  // t may lie beyond the item: on to the one that holds it; false past the last
    for (; item < n_items; ++item) {
      const ItemPtr w = items + item;
      len = a.items ? w->kv_len : a.one_item.kv_len;
      diag = a.items ? w->diag_off : a.one_item.diag_off;
      start = a.items ? w->kv_start : a.one_item.kv_start;
      tiles = (len + BN - 1) / BN;
      if (diag >= 0) tiles = min(tiles, (diag + q_last) / BN + 1);
      if (t < tiles) return true;
      t -= tiles;
    }
    return false;
  };
  auto advance = [&]() {
    t += KEEP ? WAVES : 1;
    if (t < tiles) return true;
    if (!KEEP) return false;
    t -= tiles;
    ++item;
    return enter();
  };

  float m, ms, ls[4];  // reference max (raw score units); m * k2; row sums
  f32x16 oacc[DB];
  auto reset = [&]() {
    m = -INFINITY;
    ms = kNoReference;  // while m is -inf (guard of csrc/ring_attention.cu:183): a first finite score overflows
#pragma unroll
    for (int i = 0; i < 4; ++i) ls[i] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[db][e] = 0.f;
  };

  // a tile's place and mask, carried from its loads to its scores
  struct Tile {
    int64_t at;    // byte offset of its first row from the head's
    int rows;      // keys from its first on to the end of its item
    int visible;   // keys from its first on that the first row of the q tile sees (with `rows`, what the mask goes by)
  };
  auto tile_here = [&]() {
    Tile x;
    x.at = (start + (int64_t)t * BN) * ROWB;
    x.rows = len - t * BN;
    x.visible = diag >= 0 ? diag + q0 + 1 - t * BN : INT32_MAX - BM;
    return x;
  };
  auto issue_k = [&](const Tile& x) { load_tile(k_head + x.at, my_lds, x.rows, goff_k, std::integral_constant<int, ROWB>{}); };
  auto issue_v = [&](const Tile& x) { load_tile(v_head + x.at, my_lds + TILE, x.rows, goff_v, std::integral_constant<int, ROWV>{}); };
  // P = exp2(S k2 - m k2) and the sums of four: from the unrounded values (:242); rounded for the MFMA (:604)
  f32x16 sacc;
  s16x8 pf[2];
  float sums[4];
  auto exponentials = [&]() {
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      typename E::vec8 pv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[8 * t2 + e], a.scale_log2, -ms));
        sums[e & 3] = t2 == 0 && e < 4 ? p : sums[e & 3] + p;
        pv[e] = (typename E::type)p;
      }
      pf[t2] = __builtin_bit_cast(s16x8, pv);
    }
  };
  auto move_reference = [&](bool wanted) {  // rescale of l and acc-O as in :226-232
    float m0 = m, m1 = m;
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      m0 = fmaxf(fmaxf(m0, sacc[e]), sacc[e + 1]);
      m1 = fmaxf(fmaxf(m1, sacc[e + 2]), sacc[e + 3]);
    }
    m0 = cross_half_max(fmaxf(m0, m1));
    m = KEEP || wanted ? m0 : m;
    const float cs = (m == -INFINITY) ? kNoReference : m * a.scale_log2;
    const float alpha = __builtin_amdgcn_exp2f(ms - cs);
#pragma unroll
    for (int i = 0; i < 4; ++i) ls[i] *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
    ms = cs;
  };

  // this wave's tiles from t on, if there is one
  auto walk = [&](bool more) {
    Tile cur{}, nxt{};
    if (more) {
      cur = tile_here();
      issue_k(cur);
      issue_v(cur);
    }
    __builtin_amdgcn_s_waitcnt(0);  // retire the Q loads with a wait the compiler can see (and the first tiles)
    for (int pass = 1; more; pass = 0) {  // pass: 1 while there is no reference to take exponentials against
      more = advance();
      // ---- S^T = K Q^T (csrc/ring_attention.cu:565): K(t) is in, V(t) may still be on its way
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PIECES_V) : "memory");
      {
        s16x8 kfr[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kfr[ks] = *(const s16x8*)(my + koff[ks]);
        // the fragments are in registers: the K buffer takes the next tile, next to the chain of products
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 16; ++e) sacc[e] = 0.f;
        sacc = E::mma(kfr[0], qf[0], sacc);
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
          nxt = tile_here();
          issue_k(nxt);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 1; ks < KS; ++ks) sacc = E::mma(kfr[ks], qf[ks], sacc);
      }
      __builtin_amdgcn_sched_barrier(0);
      // key visible iff inside the KV range and key_local <= query_local + diag_off
      if (min(cur.rows, cur.visible) < BN) {
        const int lim = min(cur.rows, cur.visible + n) - 4 * h;
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (8 * (e >> 2) + (e & 3) >= lim) sacc[e] = -INFINITY;
      }
      // ---- softmax (:194-245): exponentials against the reference as it stands; the row maximum is only looked at when a
      // sum of four exponentials is above 2^14 (or not a number)
#pragma unroll 1
      for (bool mine = true;; pass = 1) {
        if (pass) move_reference(mine);
        exponentials();
        const bool large = !(fmaxf(fmaxf(sums[0], sums[1]), fmaxf(sums[2], sums[3])) <= 16384.f);
        const uint64_t which = __builtin_amdgcn_ballot_w64(large);
        if (pass || which == 0) break;
        // (the steps apart: what becomes of a row is its own affair, so that it does not matter which rows share its q tile)
        mine = KEEP || ((which >> n | which >> (n + 32)) & 1) != 0;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) ls[i] += sums[i];
      // ---- O^T += V^T P^T (:609): V(t) is in, K of the next tile may still be on its way
      if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PIECES_K) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      {
        constexpr int AHEAD = 2;  // fragments read ahead of the MFMA that consumes one
        s16x8 vfr[2 * DB];
        auto read_v = [&](int f) {
          if (f >= 2 * DB) return;
          const unsigned char* vrow = my + 16 * (f / DB) * ROWV + voff[f % DB];
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vrow));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vrow + 8 * ROWV));
          vfr[f] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
#pragma unroll
        for (int f = 0; f < AHEAD; ++f) read_v(f);
#pragma unroll
        for (int f = 0; f < 2 * DB; ++f) {
          read_v(f + AHEAD);
          __builtin_amdgcn_sched_barrier(0);
          oacc[f % DB] = E::mma(vfr[f], pf[f / DB], oacc[f % DB]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (more) issue_v(nxt);
      cur = nxt;
    }
  };

  // This wave's state where the workgroup can read it: acc-O as fp32 over its own tiles, 16-byte chunk c of row n at chunk c ^ n, so
  // that neither these writes (32 rows at once) nor the reads (a few whole rows at once) meet in a bank.
  // (`fresh`: what an address is worked out from.  Worked out ahead of the rounds these would be twenty registers through every tile.)
  auto fresh = [&](int x) {
    if (MERGE) asm volatile("" : "+v"(x));
    return x;
  };
  auto show_state = [&]() {
    const float l = cross_half_sum((ls[0] + ls[1]) + (ls[2] + ls[3]));
    const int n = fresh(lane) & 31, h = fresh(lane) >> 5;
    if (h == 0) stat[wave][n] = float2{l == 0.f ? -INFINITY : ms, l};  // (0: nothing seen; a NaN stays one)
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        f32x4 val;
#pragma unroll
        for (int e = 0; e < 4; ++e) val[e] = oacc[db][4 * q4 + e];
        const int c = 8 * db + 2 * q4 + h;
        *(f32x4*)(my + n * (C * 4) + ((c ^ (n & (C / 4 - 1))) << 4)) = val;
      }
  };
  // The states of `count` waves from `first` on put together, for eight columns of a row: their reference, row sum and acc-O.
  constexpr int TPR = C / 8;  // threads of a row (at 64 columns half the threads have none, with sixteen waves three quarters)
  auto owner = [&]() { return (MERGE ? fresh(tid) : tid) / TPR < min(BM, q_last + 1 - q0); };
  float top, l, o[8];
  auto combine = [&](int first, auto count) {
    const int row = fresh(tid) / TPR, c8 = fresh(tid) % TPR;
    top = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int w = 0; w < count; ++w) top = fmaxf(top, stat[first + w][row].x);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.f;
    // (no branch on what a wave has seen: the reads of all waves are on their way together)
#pragma unroll(WAVES > 8 || MERGE ? 4 : 8)  // (else they would not fit the registers)
    for (int w = 0; w < count; ++w) {
      const float2 st = stat[first + w][row];
      const unsigned char* src = smem + (first + w) * WREG + row * (C * 4);
      const f32x4 x0 = *(const f32x4*)(src + (((2 * c8) ^ (row & (C / 4 - 1))) << 4));
      const f32x4 x1 = *(const f32x4*)(src + (((2 * c8 + 1) ^ (row & (C / 4 - 1))) << 4));
      const float f = st.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(st.x - top);
      l = __builtin_fmaf(st.y, f, l);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = __builtin_fmaf(x0[e], f, o[e]);
        o[4 + e] = __builtin_fmaf(x1[e], f, o[4 + e]);
      }
    }
  };

  reset();
  if constexpr (KEEP) {
    walk(enter());
    show_state();
    __syncthreads();
    if (!owner()) return;
    combine(0, std::integral_constant<int, WAVES>{});
    const int row = tid / TPR, c8 = tid % TPR;
    const float inv = (l > 0.f) ? 1.f / l : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= inv;
    const int64_t orow = (int64_t)bh * a.S + seg.q_start + q0 + row;
    Store8<DT>::st((char*)a.out + (orow * D + column + c8 * 8) * 2, o);
    if (column + c8 == 0 && a.lse) a.lse[orow] = partial_lse(l, top);
    return;
  }

  // a run of tiles: run `unit` of `units` of a range that begins at row `start`
  auto enter_unit = [&](int unit, int units) {
    const int all = (len + BN - 1) / BN;
    t = unit * all / units;
    tiles = (unit + 1) * all / units;
    if (diag >= 0) tiles = min(tiles, (diag + q_last) / BN + 1);
    return t < tiles;
  };
  if constexpr (MODE == kBlockPartials) {  // one range
    start = items->kv_start;
    len = items->kv_len;
    diag = items->diag_off;
    const int units = split_units((len + BN - 1) / BN);
    const bool seen = wave < units && enter_unit(wave, units);
    walk(seen);
    show_state();
    __syncthreads();
    if (!owner()) return;
    combine(0, units);
    const int row = tid / TPR, c8 = tid % TPR;
    // its partial (:621-633)
    const float inv = (l > 0.f) ? 1.f / l : 0.f;
    int64_t prow = items->part_base + (int64_t)bh * items->part_bh_stride + q0 + row;
    if (items->part_row_mul > 0) prow = prow * items->part_row_mul + items->slot;  // a row's steps next to each other
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = partial_entry<HP>(o[e], inv);
    if constexpr (HP) {  // fp16 partials: |O_part| <= max |V|, the caller vouches that this fits
      Store8<0>::st((char*)a.o_part + (prow * D + column + c8 * 8) * 2, o);
    } else {
      float* to = (float*)a.o_part + prow * D + column + c8 * 8;
      *(f32x4*)to = f32x4{o[0], o[1], o[2], o[3]};
      *(f32x4*)(to + 4) = f32x4{o[4], o[5], o[6], o[7]};
    }
    if (column + c8 == 0) a.lse_part[prow] = partial_lse(l, top);
    return;
  }

  if constexpr (MERGE) {
    // rounds of as many whole ranges as there are waves for.  What lasts from round to round -- the ranges in the order of the walk, and
    // the rows' result so far -- waits in LDS: in registers it would be more than two workgroups on a compute unit can have at d = 64.
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    i32x4* its = (i32x4*)(smem + WAVES * WREG);  // first row, rows, diag_off, units
    constexpr int kStride = BM * TPR;
    auto kept = [&](int i) -> float& { return ((float*)(its + kMaxParts))[i * kStride + fresh(tid)]; };  // of owners
    static_assert(WAVES * WREG + 16 * kMaxParts + 4 * 10 * kStride == kSplitStepsLds<D>, "tiles, ranges, results");
    if (lane < n_items) {  // (every wave writes all of them, the same: it reads none but after its own)
      const ItemPtr w = items + run_order(seg, lane);
      its[lane] = i32x4{w->kv_start, w->kv_len, w->diag_off, split_units((w->kv_len + BN - 1) / BN)};
    }
    auto range = [&](int i) {
      i32x4 x = its[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_readfirstlane(x[e]);
      return x;
    };
    MergeState mst;  // the result of the row so far, and this thread's columns of it
    float macc[8];
    for (int round = 0; round < n_items;) {
      int end = round, used = 0;
      bool seen = false;
      for (; end < n_items; ++end) {
        const i32x4 x = range(end);
        if (used + x[3] > WAVES) break;
        if (wave >= used && wave < used + x[3]) {
          start = x[0];
          len = x[1];
          diag = x[2];
          seen = enter_unit(wave - used, x[3]);
        }
        used += x[3];
      }
      if (round > 0) {
        reset();
        __syncthreads();  // the states of the round before have been read
      }
      walk(seen);
      show_state();
      __syncthreads();
      if (owner()) {
        mst = MergeState();
#pragma unroll
        for (int e = 0; e < 8; ++e) macc[e] = 0.f;
        if (round > 0) {
          mst.top = kept(0);
          mst.sum = kept(1);
#pragma unroll
          for (int e = 0; e < 8; ++e) macc[e] = kept(2 + e);
        }
      }
      int first = 0;  // the wave that has the first run of a range
      for (int i = round; i < end; ++i) {
        const int g = range(i)[3];
        if (owner()) {
          combine(first, g);
          const float inv = (l > 0.f) ? 1.f / l : 0.f, L = partial_lse(l, top);
          if (L != -INFINITY) {  // (-inf: the identity)
            float keep, wt;
            mst.weigh(L, keep, wt);
#pragma unroll
            for (int e = 0; e < 8; ++e) macc[e] = merge_in_part(macc[e], keep, wt, partial_entry<HP>(o[e], inv));
          }
        }
        first += g;
      }
      round = end;
      if (owner() && round < n_items) {
        kept(0) = mst.top;
        kept(1) = mst.sum;
#pragma unroll
        for (int e = 0; e < 8; ++e) kept(2 + e) = macc[e];
      }
    }
    if (!owner()) return;
    const int row = fresh(tid) / TPR, c8 = fresh(tid) % TPR;
    const float inv = mst.inverse();
#pragma unroll
    for (int e = 0; e < 8; ++e) macc[e] *= inv;
    const int64_t orow = (int64_t)bh * a.S + seg.q_start + q0 + row;
    Store8<DT>::st((char*)a.out + (orow * D + c8 * 8) * 2, macc);
    if (c8 == 0) a.lse[orow] = mst.lse();
  }
}

}  // namespace ringattn
