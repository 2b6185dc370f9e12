// gfx950 (CDNA4) kernel: ring_walk_kernel's arithmetic for launches that leave compute units idle.
//
//   thin::ring_walk_kernel : the steps of ring_walk_kernel (ringattn_walk_rows.h) with FOUR waves of 32 rows in a workgroup, one per
//       SIMD, where that one has eight.  What happens to a row is the same, operation by operation and in the same order
//       -- scores, the choice to move its reference (a wave's 32 rows decide together in both), exponentials, sums, P V --,
//       so a partial has the same bits whichever of the two ran it, and the host may choose launch by launch.
//       With a compute unit to itself per 256 rows ring_walk_kernel is bound by the chain of a wave: products, softmax and products
//       take turns, and the second wave of a SIMD has the same chain.  Here a wave's iteration holds three things that do not depend on
//       each other, in one instruction stream in a fixed order:
//           iteration u :  S(u+1) = K(u+1) Q^T   |   P(u) = softmax of S(u)   |   O += P(u-1) V(u-1)
//       A move of the reference rescales acc-O at the end of the iteration, when the product of the tile before is in it.
//       The products of Q K^T are one chain, each issued only when the one before is done, so those of P V go in between: a
//       wave that waits for a product issues nothing else (0.40 -> 0.32 us an iteration).
//       K and V rings are eight tiles deep with a barrier per two iterations: in front of an even iteration u every wave has read K(u)
//       and V(u-2).  Even iterations load K(u+7) and K(u+8), odd ones V(u+4) and V(u+5); behind the barrier of u all of K up to
//       tile u+4 and of V up to tile u have landed, and the K fragments of an iteration are read at the end of the one before.
//       What bounds it: 750 cycles an iteration, of which some 450 issue an instruction -- one wave issues no more than one per four
//       cycles, v_exp_f32 one per sixteen.  us on ring_walk_kernel and on this: one step, 8 heads x 1024 rows x 1024 keys 21.5, 16.4; 4
//       x 2048 x 2048 36.5, 26.6; all steps of 4 heads x 8 x 777 tokens, merged, 118, 82, of 4 x 4 x 2048 138, 108.  With more
//       than 128 tiles of 256 rows that one's second wave pays: 8 heads x 8 x 1024 tokens 180, 191.  d = 64 only: at d = 128 the products
//       of a tile take twice as long for the same softmax (a step of 32 tiles 28.6, 25.5; its forwards 177, 190).
#include "ringattn_walk_rows.h"

#include <utility>

namespace ringattn {
namespace thin {

template <class F, int... I> static __device__ __forceinline__ void for_each_slot(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <int DT, bool HP, int MODE>
__global__ __launch_bounds__(256, 2) void ring_walk_kernel(const BlockArgs a) {
  using E = Elem<DT>;
  static_assert(MODE == kBlockPartials || MODE == kBlockPartialsMerged, "the ring steps apart");
  constexpr bool MERGE = MODE == kBlockPartialsMerged;
  constexpr int D = 64;
  constexpr int BM = kThinM;       // query rows per workgroup: 4 waves x 32
  constexpr int BN = 32;           // keys per tile
  constexpr int NBUF = 8;          // ring depth of the K and of the V tiles
  constexpr int CPR = D / 8;       // 16-byte chunks per row
  constexpr int ROWB = D * 2;      // bytes per row
  constexpr int TILE = BN * ROWB;  // bytes per tile
  constexpr int PIECES = TILE / 4096;  // 1 KB pieces of a tile per wave
  constexpr int KS = D / 16;       // contraction slices of QK^T
  constexpr int DB = D / 32;       // 32-wide blocks of the head dim in PV
  constexpr float kLazyLog2 = 8.f, kSpecLimit = 16384.f;  // as in ring_walk_kernel
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * NBUF * TILE];

  const unsigned smem_base = lds_offset(smem);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;

  Segment seg;
  int bh, qt;
  if (!decode_job<BM>(a, seg, bh, qt)) return;
  const int q_len = seg.q_len, n_items = seg.item_count;
  const int row0 = qt * BM + 32 * wave;  // the wave's first row within the segment
  const ItemPtr items = items_of(a);

  const int64_t head_off = (int64_t)bh * a.bh_stride;
  // grouped-query attention: query head h of a batch entry reads KV head h / kv_group, and heads are whole groups
  const int kv_bh = quotient(bh, a.by_group);
  const int64_t kv_head_off = (int64_t)kv_bh * a.kv_bh_stride;

  // this lane's query row; rows beyond the range read the last valid row
  s16x8 qf[KS];
  {
    const char* qrow = (const char*)a.q + (head_off + (int64_t)(seg.q_start + min(row0 + n, q_len - 1)) * D) * 2 + h * 16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const s16x8*)(qrow + ks * 32);
  }
  int prow[PIECES], chunk_k[PIECES], chunk_v[PIECES];  // this wave's pieces of a tile: this lane's row, and 16 bytes of it
#pragma unroll
  for (int j = 0; j < PIECES; ++j) {
    const int pk = (PIECES * wave + j) * 64 + lane;
    prow[j] = pk / CPR;
    chunk_k[j] = ((pk % CPR) ^ k_swizzle<D>(prow[j])) << 4;
    chunk_v[j] = ((pk % CPR) ^ v_swizzle<D>(prow[j])) << 4;
  }
  const unsigned lds_mine = __builtin_amdgcn_readfirstlane(smem_base + PIECES * wave * 1024);  // where they go in K ring slot 0
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
      voff[db] = NBUF * TILE + row8 * ROWB + ((c ^ v_swizzle<D>(row8)) << 4) + ((s & 1) << 3);
    }
  }

  float m = -INFINITY;  // reference max (raw score units)
  float ms = 0.f;       // m * k2, 0 while m is -inf (guard of csrc/ring_attention.cu:183)
  float ls[4];
  f32x16 oacc[DB], sacc[2];  // scores of tile u in sacc[u & 1]
  s16x8 pf[2][2];            // its probabilities in pf[u & 1]

  MergeState mst;  // MERGE: the result of this lane's row so far (merge_partial in ringattn_walk_rows.h)
  f32x16 macc[MERGE ? DB : 1];
  if (MERGE) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) macc[db][e] = 0.f;
  }

  for (int it = 0; it < n_items; ++it) {
    const ItemPtr w = items + seg.item_begin + run_order(seg, it);
    const int kv_len = w->kv_len;
    const bool diag = w->diag_off >= 0;
    const int diag_rows = w->diag_off + qt * BM;  // keys below this local index are visible to the whole q tile
    const int kv_tiles = (kv_len + BN - 1) / BN;
    const int n_tiles = diag ? min(kv_tiles, (diag_rows + BM + BN - 1) / BN) : kv_tiles;
    const int kv_tail = (kv_len % BN) ? kv_len / BN : -1;  // the tile with surplus keys, if any
    // tiles from here on need a mask (causal diagonal or surplus keys)
    const int first_masked = min(diag ? diag_rows / BN : n_tiles, kv_tail >= 0 ? kv_tail : n_tiles);
    const char* kbase = (const char*)a.k + (kv_head_off + (int64_t)w->kv_start * D) * 2;
    const char* vbase = (const char*)a.v + (kv_head_off + (int64_t)w->kv_start * D) * 2;
    // Tile t to ring slot `slot`, every wave its pieces.  Rows beyond the KV range, those of tiles past its end (which nobody
    // reads from LDS) among them, read the last valid row: a minimum per lane, and no branch and no 64-bit address per load.
    auto issue = [&](const char* base, const int (&chunk)[PIECES], unsigned ring, int t, int slot) {
#pragma unroll
      for (int j = 0; j < PIECES; ++j)
        load_lds_16(base, (unsigned)min(t * BN + prow[j], kv_len - 1) * ROWB + chunk[j], lds_mine + ring + slot * TILE + 1024 * j);
    };
    auto issue_k = [&](int t, int slot) { issue(kbase, chunk_k, 0, t, slot); };
    auto issue_v = [&](int t, int slot) { issue(vbase, chunk_v, NBUF * TILE, t, slot); };
    // key visible iff inside the KV range and key_local <= query_local + diag_off
    auto mask_tile = [&](f32x16& s, int t) {
      int lim = kv_len - 1 - t * BN - 4 * h;
      if (diag) lim = min(lim, diag_rows + 32 * wave + n - t * BN - 4 * h);
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (8 * (e >> 2) + (e & 3) > lim) s[e] = -INFINITY;
    };
    auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };

    // ---- prologue
    if (it > 0) __syncthreads();  // every wave is done with the rings of the chunk before
#pragma unroll
    for (int t = 0; t < 7; ++t)
      if (t < n_tiles) issue_k(t, t);
#pragma unroll
    for (int t = 0; t < 5; ++t)
      if (t < n_tiles) issue_v(t, t);
    ms = 0.f;
    m = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) ls[i] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[db][e] = 0.f;
    __builtin_amdgcn_s_waitcnt(0);  // retire the Q loads with a wait the compiler can see (and the tiles)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 16; ++e) sacc[0][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) sacc[0] = E::mma(*(const s16x8*)(smem + koff[ks]), qf[ks], sacc[0]);
    if (first_masked <= 0) mask_tile(sacc[0], 0);
    s16x8 kfr[KS];  // the K fragments of tile u+1
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kfr[ks] = *(const s16x8*)(smem + TILE + koff[ks]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // tile 0 is in registers: its place is given away behind the first barrier

    auto iteration = [&](auto slot_c, auto first_c, int u) {
      constexpr int SLOT = decltype(slot_c)::value;      // u mod NBUF
      constexpr bool FIRST = decltype(first_c)::value;   // u == 0: no tile before
      constexpr int NMFMA = KS + (FIRST ? 0 : 2 * DB);
      f32x16 &cur = sacc[SLOT & 1], &nxt = sacc[(SLOT & 1) ^ 1];
      s16x8(&p_cur)[2] = pf[SLOT & 1];
      const s16x8(&p_prev)[2] = pf[(SLOT & 1) ^ 1];
      if (SLOT % 2 == 0) {  // the loads of the last three iterations may be in flight
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(6 * PIECES) : "memory");
        issue_k(u + 7, (SLOT + 7) % NBUF);
        issue_k(u + 8, SLOT);
      } else {
        issue_v(u + 4, (SLOT + 4) % NBUF);
        issue_v(u + 5, (SLOT + 5) % NBUF);
      }
      // ---- the MFMAs: those of QK^T are one chain, and the next of a chain is issued when the last is done, so P V goes in between.
      // Places 0 and 1 are Q K^T, then they alternate.  kfr, K of tile u+1, was read in the iteration before; V^T of tile u-1 is read
      // kAhead fragments ahead.
      constexpr int kAhead = 4;
      s16x8 vfr[2 * DB];
      auto read_v = [&](int f) {
        if (f >= 2 * DB || FIRST) return;
        const unsigned char* src = smem + (SLOT + NBUF - 1) % NBUF * TILE + 16 * (f / DB) * ROWB + voff[f % DB];
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src + 8 * ROWB));
        vfr[f] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      };
      auto read_k = [&](int k) { kfr[k] = *(const s16x8*)(smem + (SLOT + 2) % NBUF * TILE + koff[k]); };  // of the next iteration
      auto mfma = [&](int i) {
        static_assert(KS == 2 * DB, "as many of either product");
        const bool q = FIRST || i < 2 || (i < 2 * KS - 1 && (i & 1) != 0);
        if (q) {
          const int k = FIRST || i < 2 ? i : (i + 1) / 2;
          if (k == 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) nxt[e] = 0.f;
          }
          nxt = E::mma(kfr[k], qf[k], nxt);
          read_k(k);
        } else {
          const int f = i == 2 * KS - 1 ? 2 * DB - 1 : (i - 2) / 2;
          oacc[f % DB] = E::mma(vfr[f], p_prev[f / DB], oacc[f % DB]);
          read_v(f + kAhead);
        }
        fence();
      };
      // ---- softmax of tile u: the exponentials in steps that are kExpAhead values apart
      float x[16], sums[4] = {0.f, 0.f, 0.f, 0.f};
      typename E::vec8 pv[2];
      constexpr int kExpAhead = 4, kSteps = 16 + 2 * kExpAhead;
      auto exp_step = [&](int k) {
        if (k < 16) x[k & 15] = __builtin_fmaf(cur[k & 15], a.scale_log2, -ms);
        if (k >= kExpAhead && k < 16 + kExpAhead) x[(k - kExpAhead) & 15] = __builtin_amdgcn_exp2f(x[(k - kExpAhead) & 15]);
        if (k >= 2 * kExpAhead && k < kSteps) {
          const int e = (k - 2 * kExpAhead) & 15;
          sums[e & 3] += x[e];
          if (e & 1) {
            pv[e >> 3][(e & 7) - 1] = (typename E::type)x[e - 1];
            pv[e >> 3][e & 7] = (typename E::type)x[e];
          }
        }
        fence();
      };
#pragma unroll
      for (int f = 0; f < kAhead; ++f) read_v(f);
      fence();
      constexpr int kHead = 4;  // steps in front of the first product
#pragma unroll
      for (int k = 0; k < kHead; ++k) exp_step(k);
#pragma unroll
      for (int i = 0; i < NMFMA; ++i) {
        mfma(i);
#pragma unroll
        for (int k = kHead + (kSteps - kHead) * i / NMFMA; k < kHead + (kSteps - kHead) * (i + 1) / NMFMA; ++k) exp_step(k);
      }
      // exponentials too large for the reference as it stands, or none yet: it moves where some row's maximum lies far above it
      float alpha = 1.f;
      bool moved = false;
      const float largest = fmaxf(fmaxf(sums[0], sums[1]), fmaxf(sums[2], sums[3]));
      const bool again = !(largest <= kSpecLimit) || m == -INFINITY;
      if (__builtin_amdgcn_ballot_w64(again) != 0) {
        float m0 = m, m1 = m;
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
          m0 = fmaxf(fmaxf(m0, cur[e]), cur[e + 1]);
          m1 = fmaxf(fmaxf(m1, cur[e + 2]), cur[e + 3]);
        }
        const float cand = cross_half_max(fmaxf(m0, m1));
        const bool far = (cand - m) * a.scale_log2 > kLazyLog2;
        if (__builtin_amdgcn_ballot_w64(far) != 0) {
          const float cs = (cand == -INFINITY) ? 0.f : cand * a.scale_log2;
          alpha = __builtin_amdgcn_exp2f(m * a.scale_log2 - cs);
          moved = true;
#pragma unroll
          for (int i = 0; i < 4; ++i) ls[i] *= alpha;
          m = cand;
          ms = cs;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[i] = 0.f;
#pragma unroll
        for (int k = 0; k < kSteps; ++k) exp_step(k);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) ls[i] += sums[i];
      if (moved) {
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
      }
      p_cur[0] = __builtin_bit_cast(s16x8, pv[0]);
      p_cur[1] = __builtin_bit_cast(s16x8, pv[1]);
      if (u + 1 >= first_masked) mask_tile(nxt, u + 1);
    };

    // (one way out of the loop: with an exit behind every iteration the compiler moves the accumulators about)
    iteration(std::integral_constant<int, 0>{}, std::true_type{}, 0);
    for (int u = 1; u < n_tiles; u += NBUF)
      for_each_slot(
          [&](auto i) {
            constexpr int I = decltype(i)::value;
            if (I == 0 || u + I < n_tiles) iteration(std::integral_constant<int, (I + 1) % NBUF>{}, std::false_type{}, u + I);
          },
          std::make_integer_sequence<int, NBUF>{});
    // O += P V of the last tile
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if ((n_tiles & 1) == 0) {
      pf[0][0] = pf[1][0];
      pf[0][1] = pf[1][1];
    }
#pragma unroll
    for (int f = 0; f < 2 * DB; ++f) {
      const unsigned char* src = smem + (n_tiles - 1) % NBUF * TILE + 16 * (f / DB) * ROWB + voff[f % DB];
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src + 8 * ROWB));
      oacc[f % DB] = E::mma(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pf[0][f / DB], oacc[f % DB]);
    }

    const float l = cross_half_sum((ls[0] + ls[1]) + (ls[2] + ls[3]));
    if (!MERGE) {
      store_partial<D, HP>(a, w, oacc, l, ms, bh, row0, q_len);
    } else {
      const float inv = (l > 0.f) ? 1.f / l : 0.f, L = partial_lse(l, ms);
      if (L != -INFINITY) {  // (-inf: the identity)
        float keep, wt;
        mst.weigh(L, keep, wt);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int e = 0; e < 16; ++e) macc[db][e] = merge_in_part(macc[db][e], keep, wt, partial_entry<HP>(oacc[db][e], inv));
      }
    }
  }
  if constexpr (MERGE) {
    const int64_t row = (int64_t)bh * a.S + seg.q_start + row0;  // the wave's first row
    store_block<DT, D>(macc, mst.inverse(), (char*)a.out + row * ROWB, ROWB, q_len - row0);
    if (h == 0 && row0 + n < q_len) a.lse[row + n] = mst.lse();
  }
}

}  // namespace thin

hipError_t launch_thin(BlockArgs a, int dtype, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (a.q_tiles_max <= 0 || blocks > INT32_MAX || a.mode == kBlockCarryState) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
#define RA_LAUNCH_THIN(DT_, HP_)                                                                                     \
  do {                                                                                                              \
    if (a.mode == kBlockPartials) thin::ring_walk_kernel<DT_, HP_, kBlockPartials><<<grid, 256, 0, stream>>>(a);    \
    else thin::ring_walk_kernel<DT_, HP_, kBlockPartialsMerged><<<grid, 256, 0, stream>>>(a);                       \
  } while (0)
  if (dtype == 0 && a.half_partials) RA_LAUNCH_THIN(0, true);
  else if (dtype == 0) RA_LAUNCH_THIN(0, false);
  else if (dtype == 1 && a.half_partials) RA_LAUNCH_THIN(1, true);
  else if (dtype == 1) RA_LAUNCH_THIN(1, false);
#undef RA_LAUNCH_THIN
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
