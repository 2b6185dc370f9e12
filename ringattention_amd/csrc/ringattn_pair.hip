// gfx950 (CDNA4) kernel: block attention for launches of some tens to some hundreds of 256-row q tiles.
//
//   ring_pair_kernel : the forward of ring_walk64_kernel (ringattn_walk64.hip; the reference's CTA that walks its ring
//       steps with max / sum / acc-O in registers, csrc/ring_attention.cu:439-443,456-620, epilogue :621-664) with a
//       workgroup of 128 query rows: waves 0 and 1 own 64 rows each, waves 2 and 3 the same rows again, and the two GROUPS
//       (waves 0-1, waves 2-3) take the 32-key tiles of the rows' walk in turn -- group 0 tiles 0, 2, 4, ..., group 1
//       tiles 1, 3, 5, ....  Each group has K and V rings and a softmax state of its own; the two states are combined at
//       the end (the rescale of :226-232 once more, between groups instead of tiles).
//       The wave's program is that of ring_walk64_kernel -- one wave per SIMD, the same hand-scheduled iteration --, so
//       it runs at nearly its rate; what differs is that a tile fetched from L2 feeds 128 rows instead of 256 (an iteration
//       loads twice the bytes, 32 KB a compute unit at d = 128), that the rings are four tiles deep instead of eight (the
//       same LDS for twice the streams), and that there is a barrier per iteration instead of one per two.
//       What it is for: twice the workgroups with walks half as long.  The time of a launch of few q tiles is that of its
//       longest walk, and under the causal mask the longest walk is twice the average one.
//       What bounds it: as ring_walk64_kernel the one instruction stream of a wave, plus the barrier and the loads: with every
//       compute unit busy a workgroup of 128 rows takes 0.84 us per two tiles at d = 128 and 0.53 at d = 64, ring_walk64_kernel
//       0.79 and 0.49 per tile of 256 rows.  us a pass, that kernel (or ring_split_kernel) before and this one after: d = 128,
//       causal, 8 heads x 4096 65 -> 50, 8 heads x 8192 161 -> 124; no mask, 4 heads x 8192 151 -> 117, 9 heads x 8192 355 -> 310;
//       16 heads x 4400, causal (not a multiple of 32: ring_walk_kernel) 100 -> 88.  carry_kernel in ringattn_api.hip chooses.
//       Moves of the references (peaked logits) have no second wave to hide behind: that launch takes 129 us with N(0, 81) logits,
//       ring_walk_kernel 120.
//       Shapes it takes: every key range at least 128 keys, every one but the last walked a multiple of 32 keys, and none that
//       begins beyond 4 GiB of its head.
#include "ringattn_device.h"

namespace ringattn {

template <int DT, int D>
__global__ __launch_bounds__(256, 1) void ring_pair_kernel(const BlockArgs a) {
  using E = Elem<DT>;
  constexpr int GROUPS = 2;        // groups of two waves the keys are dealt to
  constexpr int BM = kPairM;       // query rows per workgroup: 64 per wave, the same in both groups
  constexpr int BN = 32;           // keys per tile
  constexpr int NBUF = 4;          // ring depth of the K and of the V tiles of a group
  constexpr int CPR = D / 8;       // 16-byte chunks per row
  constexpr int ROWB = D * 2;      // bytes per row
  constexpr int TILE = BN * ROWB;  // bytes per tile
  constexpr int PIECES = TILE / 2048;  // 1 KB pieces of a tile per wave
  constexpr int KS = D / 16;       // contraction slices of QK^T
  constexpr int DB = D / 32;       // 32-wide blocks of the head dim in PV
  static_assert(BM == 128, "two waves of two 32-row blocks");
  constexpr int kGroupBytes = 2 * NBUF * TILE;         // K ring, V ring
  constexpr int kListAt = GROUPS * kGroupBytes;        // per group: its chunks in walking order, (byte offset, tiles) each
  constexpr int kListLen = kMaxParts + 5;              // the ranges, the ragged last tile, four rounds of spare tiles
  constexpr int kStatAt = kListAt + GROUPS * 8 * kListLen;  // (reference max * k2, row sum) of every row in both groups
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kStatAt + GROUPS * BM * 8];

  const unsigned smem_base = lds_offset(smem);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 1, half = wave & 1;  // (half: which 64 rows, and which half of a tile the wave loads)
  const int n = lane & 31, h = lane >> 5;

  Segment seg;
  int bh, qt;
  if (!decode_job<BM>(a, seg, bh, qt)) return;
  const int q_start = seg.q_start, q_len = seg.q_len;
  const int n_items = seg.item_count;
  const ItemPtr items = items_of(a);
  // items in run order: table order, except that item `last_item` (the diagonal one) is moved to the end
  auto item_at = [&](int i) -> ItemPtr {
    int idx = i;
    if (seg.last_item >= 0) idx = (i == n_items - 1) ? seg.last_item : (i >= seg.last_item ? i + 1 : i);
    return items + seg.item_begin + idx;
  };
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
    const int ql = min(qt * BM + 64 * half + 32 * b + n, q_len - 1) - qt * BM;
    const char* qrow = qbase + (int64_t)ql * ROWB + h * 16;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[b][ks] = *(const s16x8*)(qrow + ks * 32);
  }

  // ---- the walk: the tiles of all ranges laid end to end, dealt to the groups in turn.  This group's share of a range that
  // starts at tile `before` of the sequence: its tiles `first`, `first` + 2, ...
  auto tiles_of = [&](ItemPtr w) {
    const int kv_tiles = (w->kv_len + BN - 1) / BN;
    return w->diag_off >= 0 ? min(kv_tiles, (w->diag_off + qt * BM + BM - 1) / BN + 1) : kv_tiles;
  };
  int before_last = 0;  // tiles in front of the last range
  for (int i = 0; i + 1 < n_items; ++i) before_last += tiles_of(item_at(i));
  const ItemPtr last = item_at(n_items - 1);
  const int n_last = tiles_of(last);
  const int total = before_last + n_last;
  const int N = (total + 1) / 2;                       // iterations of the workgroup: tiles of the busier group
  const int base = (before_last + 1 - grp) / 2;        // this group's tiles in front of the last range
  const int first = (grp + before_last) & 1;           // its first tile within the last range
  // the last tile of the last range has fewer than 32 keys: which group loads it, and how many there are
  const int tail_rows = n_last * BN > last->kv_len ? last->kv_len % BN : 0;
  const bool tail = tail_rows > 0 && ((n_last - 1) & 1) == first;
  // Tiles of the last range below `clear` are visible to all rows of this wave, tiles from `end` on to none (the causal
  // mask, which hides the keys past a ragged end as well; or only those keys); `limit`: the last key a lane's row sees.
  const bool diag = last->diag_off >= 0;
  const int diag_rows = last->diag_off + qt * BM;  // keys below this one are visible to the whole q tile
  const int clear = diag ? min(n_last, (diag_rows + 64 * half + 1) / BN) : (tail_rows > 0 ? n_last - 1 : n_last);
  const int end = diag ? min(n_last, (diag_rows + 64 * half + 63) / BN + 1) : n_last;
  // in tiles of this group's sequence.  Ew >= 1: a range has four tiles or the q tile sees two of it
  const int Mw = base + (max(clear - first, 0) + 1) / 2, Ew = base + (max(end - first, 0) + 1) / 2;
  int limit[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) limit[b] = (diag ? diag_rows + 64 * half + 32 * b + n : last->kv_len - 1) - 4 * h;

  // this wave's 1 KB pieces of a tile, and what they step back by when only tail_rows rows of it exist
  int goff_k[PIECES], goff_v[PIECES], back[PIECES];
#pragma unroll
  for (int j = 0; j < PIECES; ++j) {
    const int pk = (PIECES * half + j) * 64 + lane, row = pk / CPR;
    goff_k[j] = row * ROWB + (((pk % CPR) ^ k_swizzle<D>(row)) << 4);
    goff_v[j] = row * ROWB + (((pk % CPR) ^ v_swizzle<D>(row)) << 4);
    back[j] = max(0, row - (tail_rows - 1)) * ROWB;
  }
  // fragment offsets from the start of LDS, in this group's rings
  const unsigned rings = smem_base + grp * kGroupBytes;
  int koff_a[KS], voff_a[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff_a[ks] = (int)rings + n * ROWB + (((2 * ks + h) ^ k_swizzle<D>(n)) << 4);
  {
    const int s = lane & 15, g1 = (lane >> 4) & 1;
    const int row8 = 4 * h + (s >> 2);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int c = 2 * (2 * db + g1) + ((s & 3) >> 1);
      voff_a[db] = (int)rings + NBUF * TILE + row8 * ROWB + ((c ^ v_swizzle<D>(row8)) << 4) + ((s & 1) << 3);
    }
  }

  // ---- load streams.  Entries of the list: the ranges, the ragged tile (bit 0 of its offset set), then rounds of tiles 0
  // and 2 of the head (valid memory: a range has 128 keys; nobody reads them from LDS), so that every iteration issues the
  // same number of loads.  The loop loads K(u + 4) in iteration u <= N and the group has N - 1 tiles at least: at most six
  // tiles past the end, three rounds and the entry after them.
  const int n_entries = n_items + (tail ? 1 : 0);
  auto chunk_of = [&](int i, unsigned& off, int& cnt) {
    if (i < n_items) {
      int before = 0;
      for (int j = 0; j < i; ++j) before += tiles_of(item_at(j));
      const ItemPtr w = item_at(i);
      const int t0 = (grp + before) & 1;
      off = (unsigned)w->kv_start * ROWB + t0 * TILE;
      cnt = (tiles_of(w) - t0 + 1) / 2 - (tail && i == n_items - 1 ? 1 : 0);
    } else if (i < n_entries) {
      off = ((unsigned)last->kv_start + (n_last - 1) * BN) * ROWB | 1u;
      cnt = 1;
    } else {
      off = 0;
      cnt = 2;
    }
  };
  struct Stream {
    unsigned off;  // the next tile to load
    int left;      // tiles left in its chunk, that one included
    int idx;       // the chunk
  };
  Stream kst, vst;
  kst.idx = vst.idx = 0;
  chunk_of(0, kst.off, kst.left);
  vst = kst;
  auto issue = [&](Stream& s, const char* head, int (&goff)[PIECES], unsigned dst) {
    const char* p = head + __builtin_amdgcn_readfirstlane(s.off);
#pragma unroll
    for (int j = 0; j < PIECES; ++j)
      load_lds_16_settled(p, goff[j], __builtin_amdgcn_readfirstlane(dst + 1024 * (PIECES * half + j)));
    s.off += GROUPS * TILE;
    if (--s.left == 0) {
      s.idx += 1;
      chunk_of(s.idx, s.off, s.left);
      if (s.off & 1) {
        s.off &= ~1u;
#pragma unroll
        for (int j = 0; j < PIECES; ++j) goff[j] -= back[j];
      }
    }
  };

  // ---- prologue: K(0) .. K(3), V(0) and V(1) next to the Q loads; V ring slot 3 -- "tile -1", which the first iteration
  // multiplies with all-zero probabilities -- is cleared; the chunk list the loop steps its load streams through
#pragma unroll 1
  for (int t = 0; t < 4; ++t) issue(kst, k_head, goff_k, rings + t * TILE);
#pragma unroll 1
  for (int t = 0; t < 2; ++t) issue(vst, v_head, goff_v, rings + (NBUF + t) * TILE);
  const int list_at = kListAt + grp * 8 * kListLen;
  for (int i = tid & 127; i < n_entries + 4; i += 128) {
    unsigned o;
    int c;
    chunk_of(i, o, c);
    *(int2*)(smem + list_at + 8 * i) = int2{(int)o, c};
  }
  {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TILE / 2048; ++j)
      *(f32x4*)(smem + grp * kGroupBytes + (NBUF + 3) * TILE + ((tid & 127) + 128 * j) * 16) = zero;
  }
  __builtin_amdgcn_s_waitcnt(0);  // retire the Q loads with a wait the compiler can see (and the tiles)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- softmax state of the two blocks
  float m[2], ms[2];  // reference max (raw score units); m * k2, kNoReference while m is -inf (guard of csrc/ring_attention.cu:183)
  float ls[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  f32x16 oacc[2][DB];
  f32x16 sacc[2];     // scores of tile u, consumed by the exponentials of iteration u
  s16x8 pprev[2][2];  // probabilities of tile u-1 (B operands), consumed by the PV product of iteration u
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[b][db][e] = 0.f;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int e = 0; e < 8; ++e) pprev[b][t2][e] = 0;
  }
  // scores of the first tile of group g, `t` being its place within the last range (if it lies there): key visible iff not
  // past this lane's limit
  auto scores = [&](int g, int t, bool masked) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) sacc[b][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const s16x8 kfr = *(const s16x8*)(smem + (koff_a[ks] - (int)smem_base) + (g - grp) * kGroupBytes);
      sacc[0] = E::mma(kfr, qf[0][ks], sacc[0]);
      sacc[1] = E::mma(kfr, qf[1][ks], sacc[1]);
    }
    if (masked) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (8 * (e >> 2) + (e & 3) > limit[b] - t * BN) sacc[b][e] = -INFINITY;
    }
  };
  // The first reference of BOTH groups: the row maxima of tile 0 of the whole walk, whose first key every row sees.  (A row may
  // see nothing of the second group's first tile, and a reference that has nothing to do with its scores would not do.)  Group
  // 0 loads over that tile behind the loop's first barrier.
  scores(0, 0, before_last == 0 && clear <= 0);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float m0 = -INFINITY, m1 = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      m0 = fmaxf(fmaxf(m0, sacc[b][e]), sacc[b][e + 1]);
      m1 = fmaxf(fmaxf(m1, sacc[b][e + 2]), sacc[b][e + 3]);
    }
    m[b] = cross_half_max(fmaxf(m0, m1));
    ms[b] = (m[b] == -INFINITY) ? kNoReference : m[b] * a.scale_log2;
  }
  if (grp == 1) scores(1, 1, before_last == 0 && clear <= 1);

  // The hand-scheduled loop runs all iterations of the workgroup, 0 to N: every iteration whose score tile u+1 this wave
  // computes -- masking those that need it --, the wave's last two iterations, and then only the wave's share of the loads
  // and the barriers.
  {
    const unsigned smem_list = smem_base + list_at;
    auto uni = [](unsigned x) { return (unsigned)__builtin_amdgcn_readfirstlane((int)x); };
    const unsigned lds_dst_k = uni(rings + 1024 * PIECES * half);
    const unsigned lds_dst_v = lds_dst_k + NBUF * TILE;
    const unsigned kh_lo = uni((unsigned)(uintptr_t)k_head), kh_hi = uni((unsigned)((uintptr_t)k_head >> 32));
    const unsigned vh_lo = uni((unsigned)(uintptr_t)v_head), vh_hi = uni((unsigned)((uintptr_t)v_head >> 32));
    const unsigned k2_bits = uni(__builtin_bit_cast(unsigned, a.scale_log2));
    unsigned asm_u = 0, asm_far = 0;
    const unsigned asm_stop = uni((unsigned)(Ew - 1)), asm_mw1 = uni((unsigned)(Mw - 1));
    const unsigned asm_n = uni((unsigned)N);
    int vlim[2];  // the limits within tile 1 of this group's sequence
#pragma unroll
    for (int b = 0; b < 2; ++b) vlim[b] = limit[b] - (first + GROUPS * (1 - base)) * BN;
    const uint64_t kp = (uint64_t)(uintptr_t)k_head + kst.off, vp = (uint64_t)(uintptr_t)v_head + vst.off;
    unsigned k_lo = uni((unsigned)kp), k_hi = uni((unsigned)(kp >> 32)), v_lo = uni((unsigned)vp), v_hi = uni((unsigned)(vp >> 32));
    unsigned k_left = uni((unsigned)kst.left), v_left = uni((unsigned)vst.left);
    unsigned k_next = uni(smem_list + 8 * (kst.idx + 1)), v_next = uni(smem_list + 8 * (vst.idx + 1));
    if constexpr (D == 128) {
#include "ringattn_pair_loop.inc"
    } else {
#include "ringattn_pair_loop_d64.inc"
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- combine the two states.  A wave finishes block `grp` of its 64 rows and hands the other block, scaled to the common
  // reference, to the wave that owns the same rows in the other group; lanes of the two waves hold the same places.
  float l[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    l[b] = cross_half_sum((ls[b][0] + ls[b][1]) + (ls[b][2] + ls[b][3]));
    // (a sum of exactly 0: nothing seen.  A NaN stays one)
    if (h == 0) *(float2*)(smem + kStatAt + 8 * (grp * BM + 64 * half + 32 * b + n)) = float2{l[b] == 0.f ? -INFINITY : ms[b], l[b]};
  }
  __syncthreads();  // (and the rings are idle: every wave's loads have landed)
  float top[2], f[2], sum = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const float2 other = *(const float2*)(smem + kStatAt + 8 * ((1 - grp) * BM + 64 * half + 32 * b + n));
    const float own = l[b] == 0.f ? -INFINITY : ms[b];
    top[b] = fmaxf(own, other.x);
    f[b] = own == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(own - top[b]);
    const float fo = other.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(other.x - top[b]);
    if (b == grp) sum = l[b] * f[b] + other.y * fo;
  }
  unsigned char* give = smem + wave * (32 * D * 4) + lane * 16;
  const unsigned char* take = smem + (wave ^ 2) * (32 * D * 4) + lane * 16;
  static_assert(4 * 32 * D * 4 <= kListAt, "in the place of the rings");
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = grp ? oacc[0][db][4 * q4 + e] * f[0] : oacc[1][db][4 * q4 + e] * f[1];
      *(f32x4*)(give + (4 * db + q4) * 1024) = x;
    }
  __syncthreads();
  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const f32x4 x = *(const f32x4*)(take + (4 * db + q4) * 1024);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[db][4 * q4 + e] = (grp ? oacc[1][db][4 * q4 + e] * f[1] : oacc[0][db][4 * q4 + e] * f[0]) + x[e];
    }
  const float inv = (sum > 0.f) ? 1.f / sum : 0.f;
  const int row0 = qt * BM + 64 * half + 32 * grp;
  const int64_t row = (int64_t)bh * a.S + q_start + row0;  // the block's first row
  store_block<DT, D>(acc, inv, (char*)a.out + row * ROWB, ROWB, q_len - row0);
  if (h == 0 && row0 + n < q_len && a.lse)
    a.lse[row + n] = (sum > 0.f) ? (top[grp] + __builtin_amdgcn_logf(sum)) * 0.6931471805599453f : -INFINITY;
}

hipError_t launch_pair(BlockArgs a, int dtype, int dim, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (a.q_tiles_max <= 0 || blocks > INT32_MAX || a.mode != kBlockCarryState) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  if (dtype == 0 && dim == 64) ring_pair_kernel<0, 64><<<grid, 256, 0, stream>>>(a);
  else if (dtype == 1 && dim == 64) ring_pair_kernel<1, 64><<<grid, 256, 0, stream>>>(a);
  else if (dtype == 0 && dim == 128) ring_pair_kernel<0, 128><<<grid, 256, 0, stream>>>(a);
  else if (dtype == 1 && dim == 128) ring_pair_kernel<1, 128><<<grid, 256, 0, stream>>>(a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
