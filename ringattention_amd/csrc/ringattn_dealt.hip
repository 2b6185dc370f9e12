// gfx950 (CDNA4) kernel: ring_walk_kernel's arithmetic for launches of a few row tiles, the key tiles dealt to waves.
//
//   dealt::ring_walk_kernel : a step of a ring (one key range, its partial stored) with 32 query rows in a workgroup and the work on a
//       key tile spread over waves: four waves compute scores and probabilities, of four tiles at once, and two waves sum up P V, 32
//       of the 64 columns each.  What happens to a row is what ring_walk_kernel (ringattn_walk_rows.h) does to it, operation by
//       operation and in the same order, so a partial has the same bits whichever of the two, or thin::ring_walk_kernel, ran it, and the
//       host may choose launch by launch.  (ring_split_kernel shares out the keys as well, but gives each wave a state of its own, and
//       putting those together rounds differently.)
//       What orders the tiles of a row is the sums -- acc-O, the row sum -- and the reference of the exponentials.  The sums are done
//       by the waves of P V, tile after tile.  The reference seldom moves: all four tiles of a round take their exponentials against
//       it as it stands, each says whether it wants a move, and if one does, the tiles from the first such one on are gone through
//       again, it by itself and those behind it together.  So a round without a move has one barrier:
//           waves 0-3, round r :  S(r+1) = K Q^T  |  P(r), its sums, the wish   -> LDS, barrier, whose wish?
//           waves 4-5, round r :  barrier, whose wish?  O += P(r) V(r), read V(r+1)
//       probs, row_sums, factors and news are double-buffered by round: those of round r are read before the barrier of round r+1, and
//       those of a round without a move are written again behind it.  In a round with one the tile that moves writes its probs, row_sums and
//       news again, and the tiles behind it theirs a barrier later, while others may still be reading what stood there: of the first two
//       they then have something of each, and read again behind the last barrier of the round; the news say the same to who
//       reads early and who reads late (ringattn_news.h).  K tiles belong to the wave that loads them; V tiles are loaded half by one, half by the other wave of P V: a
//       wave passes the barrier of round r with its part of V(r+1) landed, and with V(r) in its registers.
//       A step of 8 heads x 1024 rows is 64 workgroups of thin::ring_walk_kernel whose waves walk 32 tiles each; here it is 256, with eight
//       rounds.  us on thin::ring_walk_kernel and here: 8 heads x 1024 rows x 1024 keys 15.6, 10.7; 4 x 2048 x 2048 26.3, 16.0; 2 x 4096
//       x 4096 47.4, 26.3; 8 x 512 x 512 9.8, 7.7; 8 x 256 x 256 7.1, 6.0; 1024 x 8192 89, 43; causal 8 x 1024 16.4, 10.3; with N(0, 81) logits,
//       whose references move in many rounds, 8 x 1024 19.6, 16.3, 4 x 512 12.1, 11.9.
//       What bounds it: 1540 cycles a round at 2.4 GHz, of which a wave of scores issues some 850 (93 vector instructions, sixteen of them
//       exponentials at 16 cycles, and 54 scalar ones) and spends the rest on the way through LDS: P out, barrier, wishes in.  Eight tiles a
//       round with eight waves, and V loaded column by column, took as long a tile.
#include "ringattn_walk_rows.h"
#include "ringattn_news.h"

#include <utility>

namespace ringattn {
namespace dealt {

constexpr int kScoreWaves = 4;   // key tiles of a round, one to each
constexpr int kAhead = 4;        // rounds of K and of V that are loaded ahead

template <int DT, bool HP>
__global__ __launch_bounds__(64 * (kScoreWaves + 2), 2) void ring_walk_kernel(const BlockArgs a) {
  using E = Elem<DT>;
  constexpr int D = 64;
  constexpr int BM = kDealtM, BN = 32, W = kScoreWaves;
  constexpr int ROWB = D * 2;          // bytes per row
  constexpr int TILE = BN * ROWB;      // bytes per K tile
  constexpr int KS = D / 16, DB = D / 32;
  constexpr int PIECES = TILE / 1024;  // 1 KB loads of a tile
  constexpr float kLazyLog2 = 8.f, kSpecLimit = 16384.f;  // as in ring_walk_kernel
  __shared__ __attribute__((aligned(1024))) unsigned char k_ring[W][kAhead][TILE];
  __shared__ __attribute__((aligned(1024))) unsigned char v_ring[kAhead][W][TILE];
  __shared__ s16x8 probs[2][W][2][64];   // the probabilities of a round, as the lanes hold them
  __shared__ f32x4 row_sums[2][W][64];   // their sums of four
  __shared__ float factors[2][W][BM];    // where a tile moved the references: what the sums so far are multiplied by
  __shared__ __attribute__((aligned(16))) int news[2][W];  // kNewsWish, kNewsMoved or neither
  __shared__ float reference[BM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;

  fetch_arguments(a);
  Segment seg;
  int bh, qt;
  if (!decode_job<BM>(a, seg, bh, qt)) return;
  const int q_len = seg.q_len, row0 = qt * BM;
  const ItemPtr w = items_of(a) + seg.item_begin;  // one key range
  const int kv_len = w->kv_len;
  const bool diag = w->diag_off >= 0;
  const int diag_rows = w->diag_off + row0;  // keys below this local index are visible to the whole q tile
  const int kv_tiles = (kv_len + BN - 1) / BN;
  const int n_tiles = diag ? min(kv_tiles, (diag_rows + BM + BN - 1) / BN) : kv_tiles;
  const int rounds = (n_tiles + W - 1) / W;
  const int kv_tail = (kv_len % BN) ? kv_len / BN : -1;  // the tile with surplus keys, if any
  const int first_masked = min(diag ? diag_rows / BN : n_tiles, kv_tail >= 0 ? kv_tail : n_tiles);
  // grouped-query attention: query head h of a batch entry reads KV head h / kv_group, and heads are whole groups
  const int kv_bh = quotient(bh, a.by_group);
  const int64_t kv_off = ((int64_t)kv_bh * a.kv_bh_stride + (int64_t)w->kv_start * D) * 2;

  auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  auto read_news = [&](int r) { return *(const i32x4*)news[r & 1]; };
  static_assert(W == kNewsTiles, "news_of_round");
  auto bits_of = [&](const i32x4& x) { return __builtin_amdgcn_readfirstlane(news_of_round(x[0], x[1], x[2], x[3])); };

  if (wave < W) {
    // ---- a wave of scores
    s16x8 qf[KS];
    {
      const char* qrow = (const char*)a.q + ((int64_t)bh * a.bh_stride + (int64_t)(seg.q_start + min(row0 + n, q_len - 1)) * D) * 2 + h * 16;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const s16x8*)(qrow + ks * 32);
    }
    const char* kbase = (const char*)a.k + kv_off;
    // Offsets of this lane's 16 bytes within a 1 KB piece of a tile (the swizzle repeats after two pieces); a load instruction's own
    // offset moves both ends, so the pieces share address and M0.
    int goff[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) goff[j] = lane / 8 * ROWB + (((lane % 8) ^ k_swizzle<D>(8 * j + lane / 8)) << 4);
    static_assert(PIECES == 4, "one block of loads");
    const unsigned ring = __builtin_amdgcn_readfirstlane(lds_offset(k_ring[wave][0]));
    // this wave's tile of round r; rows beyond the KV range, those of tiles past its end among them, read the last valid row
    auto issue = [&](int r) {
      const int first = (r * W + wave) * BN;
      const unsigned dst = ring + (r % kAhead) * TILE;
      if (first + BN <= kv_len) {
        asm volatile(
            "s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024\n\t"
            "global_load_lds_dwordx4 %1, %3 offset:2048\n\tglobal_load_lds_dwordx4 %2, %3 offset:3072" ::"s"(dst),
            "v"(goff[0]), "v"(goff[1]), "s"(kbase + (int64_t)first * ROWB)
            : "m0");
      } else {
        int row = lane / 8;
        asm volatile("" : "+v"(row));  // (keeps this seldom taken arithmetic from being done ahead of the loop, in registers)
#pragma unroll
        for (int j = 0; j < PIECES; ++j)
          load_lds_16_settled(kbase, (unsigned)min(first + 8 * j + row, kv_len - 1) * ROWB + (((lane % 8) ^ k_swizzle<D>(8 * j + row)) << 4), dst + 1024 * j);
      }
    };
    int koff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) koff[ks] = n * ROWB + (((2 * ks + h) ^ k_swizzle<D>(n)) << 4);
    s16x8 kfr[KS];
    auto read_k = [&](int r, int ks) { kfr[ks] = *(const s16x8*)(k_ring[wave][r % kAhead] + koff[ks]); };
    // key visible iff inside the KV range and key_local <= query_local + diag_off
    auto mask_tile = [&](f32x16& s, int t) {
      int lim = kv_len - 1 - t * BN - 4 * h;
      if (diag) lim = min(lim, diag_rows + n - t * BN - 4 * h);
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (8 * (e >> 2) + (e & 3) > lim) s[e] = -INFINITY;
    };
    auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };

#pragma unroll
    for (int r = 0; r < kAhead; ++r) issue(r);
    __builtin_amdgcn_s_waitcnt(0);  // retire the Q loads with a wait the compiler can see (and the tiles)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    f32x16 sacc[2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) read_k(0, ks);
#pragma unroll
    for (int e = 0; e < 16; ++e) sacc[0][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) sacc[0] = E::mma(kfr[ks], qf[ks], sacc[0]);
    if (wave >= first_masked) mask_tile(sacc[0], wave);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) read_k(1, ks);
    float m = -INFINITY;  // reference max (raw score units)
    float ms = 0.f;       // m * k2, 0 while m is -inf
    auto row_max = [&](const f32x16& s) {
      float m0 = m, m1 = m;
#pragma unroll
      for (int e = 0; e < 16; e += 4) {
        m0 = fmaxf(fmaxf(m0, s[e]), s[e + 1]);
        m1 = fmaxf(fmaxf(m1, s[e + 2]), s[e + 3]);
      }
      return cross_half_max(fmaxf(m0, m1));
    };
    auto set_reference = [&](float x) {
      m = x;
      ms = (m == -INFINITY) ? 0.f : m * a.scale_log2;
    };
    // The first tile sets the references: everybody's exponentials wait for these.  (There is nothing to rescale yet.)
    if (wave == 0) {
      const float top = row_max(sacc[0]);
      if (h == 0) reference[n] = top;
    }
    barrier();
    set_reference(reference[n]);

    auto round = [&](auto odd, int r) {
      constexpr int ODD = decltype(odd)::value;
      f32x16 &cur = sacc[ODD], &nxt = sacc[ODD ^ 1];
      const int u = r * W + wave;
      issue(r + kAhead);  // over the tile of this round, whose fragments were read in the round before the last
      float x[16], sums[4];
      typename E::vec8 pv[2];
      constexpr int kApart = 4, kSteps = 16 + 2 * kApart;
      auto exp_step = [&](int k) {
        if (k < 16) x[k & 15] = __builtin_fmaf(cur[k & 15], a.scale_log2, -ms);
        if (k >= kApart && k < 16 + kApart) x[(k - kApart) & 15] = __builtin_amdgcn_exp2f(x[(k - kApart) & 15]);
        if (k >= 2 * kApart && k < kSteps) {
          const int e = (k - 2 * kApart) & 15;
          sums[e & 3] += x[e];
          if (e & 1) {
            pv[e >> 3][(e & 7) - 1] = (typename E::type)x[e - 1];
            pv[e >> 3][e & 7] = (typename E::type)x[e];
          }
        }
        fence();
      };
      auto exponentials = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[i] = 0.f;
#pragma unroll
        for (int k = 0; k < kSteps; ++k) exp_step(k);
      };
      // exponentials too large for the reference as it stands, or none yet: it moves where some row's maximum lies far above it
      auto wish = [&]() {
        const float largest = fmaxf(fmaxf(sums[0], sums[1]), fmaxf(sums[2], sums[3]));
        const bool again = !(largest <= kSpecLimit) || m == -INFINITY;
        if (__builtin_amdgcn_ballot_w64(again) == 0) return false;
        return __builtin_amdgcn_ballot_w64((row_max(cur) - m) * a.scale_log2 > kLazyLog2) != 0;
      };
      auto hand_over = [&](int what) {
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) probs[r & 1][wave][t2][lane] = __builtin_bit_cast(s16x8, pv[t2]);
        row_sums[r & 1][wave][lane] = f32x4{sums[0], sums[1], sums[2], sums[3]};
        if (lane == 0) news[r & 1][wave] = what;
      };
      // S of the next round's tile next to the exponentials of this one's
#pragma unroll
      for (int i = 0; i < 4; ++i) sums[i] = 0.f;
      constexpr int kHead = 4;  // steps in front of the first product
#pragma unroll
      for (int k = 0; k < kHead; ++k) exp_step(k);
#pragma unroll
      for (int e = 0; e < 16; ++e) nxt[e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        nxt = E::mma(kfr[ks], qf[ks], nxt);
        fence();
#pragma unroll
        for (int k = kHead + (kSteps - kHead) * ks / KS; k < kHead + (kSteps - kHead) * (ks + 1) / KS; ++k) exp_step(k);
      }
      hand_over(u < n_tiles && wish() ? kNewsWish : 0);
      // K of the round after the next one: two rounds' loads may be in flight
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kAhead - 2) * PIECES) : "memory");
      barrier();
      i32x4 said = read_news(r);
      fence();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) read_k(r + 2, ks);
      int from = 0;
      for (int first; (first = first_wish(bits_of(said), from)) < W; said = read_news(r)) {  // in the order of the tiles, from the first that moves
        if (wave == first) {
          const float cand = row_max(cur);
          const float cs = (cand == -INFINITY) ? 0.f : cand * a.scale_log2;
          const float alpha = __builtin_amdgcn_exp2f(m * a.scale_log2 - cs);
          set_reference(cand);
          exponentials();
          hand_over(kNewsMoved);
          if (h == 0) {
            factors[r & 1][wave][n] = alpha;
            reference[n] = m;
          }
        }
        barrier();
        if (wave != first) set_reference(reference[n]);
        from = first + 1;
        if (from == W) break;
        if (wave >= from) {
          exponentials();
          hand_over(u < n_tiles && wish() ? kNewsWish : 0);
        }
        barrier();
      }
      if (u + W >= first_masked) mask_tile(nxt, u + W);
    };
    for (int r = 0; r < rounds; r += 2) {
      round(std::integral_constant<int, 0>{}, r);
      if (r + 1 < rounds) round(std::integral_constant<int, 1>{}, r + 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS that is no longer this workgroup's
    return;
  }

  // ---- a wave of 32 columns of P V; it loads half of the V tiles, for both
  const int db = wave - W;
  const char* vbase = (const char*)a.v + kv_off;
  const unsigned ring = __builtin_amdgcn_readfirstlane(lds_offset(v_ring[0][W / DB * db]));
  const int goff = lane / 8 * ROWB + (((lane % 8) ^ v_swizzle<D>(lane / 8)) << 4);  // of this lane's 16 bytes within a 1 KB piece
  auto issue = [&](int r) {
    const int first = (r * W + W / DB * db) * BN;
    const unsigned dst = ring + (r % kAhead) * W * TILE;
#pragma unroll
    for (int i = 0; i < W / DB; ++i) {
      if (first + (i + 1) * BN <= kv_len) {
        asm volatile(
            "s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024\n\t"
            "global_load_lds_dwordx4 %1, %2 offset:2048\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072" ::"s"(dst + i * TILE),
            "v"(goff), "s"(vbase + (int64_t)(first + i * BN) * ROWB)
            : "m0");
      } else {
        int row = lane / 8;
        asm volatile("" : "+v"(row));
#pragma unroll
        for (int j = 0; j < PIECES; ++j)
          load_lds_16_settled(vbase, (unsigned)min(first + i * BN + 8 * j + row, kv_len - 1) * ROWB + (((lane % 8) ^ v_swizzle<D>(row)) << 4),
                              dst + i * TILE + 1024 * j);
      }
    }
  };
#pragma unroll
  for (int r = 0; r < kAhead; ++r) issue(r);
  int voff;
  {
    const int s = lane & 15, g1 = (lane >> 4) & 1;
    const int row8 = 4 * h + (s >> 2), c = 2 * (2 * db + g1) + ((s & 3) >> 1);
    voff = row8 * ROWB + ((c ^ v_swizzle<D>(row8)) << 4) + ((s & 1) << 3);
  }
  float ls[4] = {0.f, 0.f, 0.f, 0.f};
  f32x16 oacc[1];
#pragma unroll
  for (int e = 0; e < 16; ++e) oacc[0][e] = 0.f;
  s16x8 vfr[2][W][2];  // V^T of this round and of the next one
  auto read_v = [&](int r, s16x8 (&to)[W][2]) {
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const unsigned char* src = v_ring[r % kAhead][i] + 16 * t2 * ROWB + voff;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src + 8 * ROWB));
        to[i][t2] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
  };
  constexpr int kLoads = W / DB * PIECES;  // of a round
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kAhead - 1) * kLoads) : "memory");
  barrier();
  read_v(0, vfr[0]);
  auto round = [&](auto odd, int r) {
    constexpr int ODD = decltype(odd)::value;
    s16x8 pf[W][2];
    f32x4 sums[W];
    auto read_p = [&]() {
#pragma unroll
      for (int i = 0; i < W; ++i) {
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) pf[i][t2] = probs[r & 1][i][t2][lane];
        sums[i] = row_sums[r & 1][i][lane];
      }
    };
    // two rounds' loads may be in flight; at the barrier V of the next round is in, and V of this round in everybody's registers, so that
    // its place is given away behind it
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kAhead - 2) * kLoads) : "memory");
    barrier();
    i32x4 said = read_news(r);
    read_p();
    issue(r + kAhead);
    int from = 0;
    for (int first; (first = first_wish(bits_of(said), from)) < W;) {
      barrier();
      from = first + 1;
      if (from < W) barrier();
      said = read_news(r);
      read_p();
      if (from == W) break;
    }
    const int moves = bits_of(said >> kNewsMovedBit);
    read_v(r + 1, vfr[ODD ^ 1]);
#pragma unroll
    for (int i = 0; i < W; ++i) {
      if (r * W + i >= n_tiles) break;
      if (moves >> i & 1) {  // rescale of l and acc-O as in csrc/ring_attention.cu:226-232
        const float alpha = factors[r & 1][i][n];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ls[e] *= alpha;
          asm volatile("" : "+v"(ls[e]));  // (a product of its own, as in ring_walk_kernel)
        }
        oacc[0] *= alpha;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) ls[e] += sums[i][e];
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) oacc[0] = E::mma(vfr[ODD][i][t2], pf[i][t2], oacc[0]);
    }
  };
  for (int r = 0; r < rounds; r += 2) {
    round(std::integral_constant<int, 0>{}, r);
    if (r + 1 < rounds) round(std::integral_constant<int, 1>{}, r + 1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // the partial of the range (csrc/ring_attention.cu:621-633), store_partial's for these columns
  const float l = cross_half_sum((ls[0] + ls[1]) + (ls[2] + ls[3]));
  const float inv = (l > 0.f) ? 1.f / l : 0.f;
  const float m = reference[n];
  const float ms = (m == -INFINITY) ? 0.f : m * a.scale_log2;
  const int step = w->part_row_mul > 0 ? w->part_row_mul : 1;  // n: a row's steps next to each other
  const int64_t prow = (w->part_base + (int64_t)bh * w->part_bh_stride + row0) * step + (w->part_row_mul > 0 ? w->slot : 0);
  if constexpr (HP) {  // fp16 partials: |O_part| <= max |V|, the caller vouches that this fits
    store_block<0, 32>(oacc, inv, (char*)a.o_part + prow * (D * 2) + 64 * db, (int64_t)step * (D * 2), q_len - row0);
  } else if (row0 + n < q_len) {
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      f32x4 val;
#pragma unroll
      for (int e = 0; e < 4; ++e) val[e] = oacc[0][4 * q4 + e] * inv;
      *(f32x4*)((float*)a.o_part + (prow + (int64_t)n * step) * D + 32 * db + 8 * q4 + 4 * h) = val;
    }
  }
  if (db == 0 && h == 0 && row0 + n < q_len) a.lse_part[prow + (int64_t)n * step] = partial_lse(l, ms);
}

}  // namespace dealt

hipError_t launch_dealt(BlockArgs a, int dtype, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (a.q_tiles_max <= 0 || blocks > INT32_MAX || a.mode != kBlockPartials) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  constexpr int kThreads = 64 * (dealt::kScoreWaves + 2);
  if (dtype == 0 && a.half_partials) dealt::ring_walk_kernel<0, true><<<grid, kThreads, 0, stream>>>(a);
  else if (dtype == 0) dealt::ring_walk_kernel<0, false><<<grid, kThreads, 0, stream>>>(a);
  else if (dtype == 1 && a.half_partials) dealt::ring_walk_kernel<1, true><<<grid, kThreads, 0, stream>>>(a);
  else if (dtype == 1) dealt::ring_walk_kernel<1, false><<<grid, kThreads, 0, stream>>>(a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
