// Device-side helpers shared by the gfx950 kernels of this library (vector types, direct-to-LDS
// loads, MFMA wrappers, cross-half exchanges, LDS swizzles, the workgroup -> job mapping).
#pragma once
#include "ringattn_kernels.h"

#include <cstddef>
#include <type_traits>

namespace ringattn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// 16 bytes per lane HBM -> LDS without passing through registers: lane i's data lands
// at lds_addr + 16 i (lds_addr is wave-uniform and travels in M0).  Written as inline
// asm so the compiler does not serialise later LDS reads behind the transfer; the
// kernel waits for it explicitly (s_waitcnt vmcnt(0)) before the tile barrier.
// No "memory" clobber: a transfer only ever targets a ring slot that no LDS read between
// the surrounding barriers touches, so the compiler may move LDS reads across it.
// M0 is declared clobbered, and the s_nop is the wait state the hardware needs between a
// scalar write of M0 and the LDS-DMA instruction that reads it (the assembler inserts none
// inside inline asm).
static __device__ __forceinline__ void load_lds_16(const void* base, int voff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(base) : "m0");
}
// The same transfer for call sites whose base address may have just come out of a v_readfirstlane: a vector
// instruction that wrote a scalar register must be five wait states ahead of the memory instruction that reads it,
// and the compiler does not see into inline asm to provide them.
static __device__ __forceinline__ void load_lds_16_settled(const void* base, int voff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(base) : "m0");
}
static __device__ __forceinline__ unsigned lds_offset(const void* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

template <int DT> struct Elem;
template <> struct Elem<0> {
  using type = _Float16;
  using vec8 = f16x8;
  using vec4 = f16x4;
  static __device__ __forceinline__ f32x16 mma(s16x8 a, s16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(vec8, a), __builtin_bit_cast(vec8, b), c, 0, 0, 0);
  }
};
template <> struct Elem<1> {
  using type = __bf16;
  using vec8 = bf16x8;
  using vec4 = bf16x4;
  static __device__ __forceinline__ f32x16 mma(s16x8 a, s16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(vec8, a), __builtin_bit_cast(vec8, b), c, 0, 0, 0);
  }
};

// max / sum across the two 32-lane halves of a wave.  v_permlane32_swap exchanges the
// upper half of its first operand with the lower half of its second, so with both
// operands holding x every lane ends up with its own x and the x of the lane 32 away.
// Inline asm on purpose: the compiler builtin, given the same value for both operands,
// merges the two results into one register and drops the exchanged half.  The s_nop
// covers the VALU-write -> permlane-read hazard the assembler does not see inside asm.
static __device__ __forceinline__ void swap_halves(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
static __device__ __forceinline__ float cross_half_max(float x) {
  float a = x, b = x, r;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %1, %2\n\ts_nop 1\n\tv_max_f32 %0, %1, %2" : "=v"(r), "+v"(a), "+v"(b));
  return r;
}
static __device__ __forceinline__ float cross_half_sum(float x) {
  float a = x, b = x;
  swap_halves(a, b);
  return a + b;
}

// XOR swizzles on 16-byte chunk indices within a tile row (row = key, 2*D bytes).
// K is read with ds_read_b128 by 32 lanes on 32 consecutive rows; V is read with
// ds_read_b64_tr_b16 by groups of 16 lanes covering 4 rows x 32 bytes.
template <int D> static __device__ __forceinline__ int k_swizzle(int row) {
  return D == 128 ? (row & 15) : ((row >> 1) & 7);
}
template <int D> static __device__ __forceinline__ int v_swizzle(int row) {
  return D == 128 ? (((row & 3) << 2) | (((row >> 2) & 1) << 1))
                  : ((((row >> 1) & 1) << 2) | (((row >> 2) & 1) << 1));
}

// m * k2 of a row in the generated loops while its scores so far are all -inf (keys that a coordinate of -inf hides: left
// padding): the exponential of such a score against it is 0, and that of the first finite one infinite, which is what makes the
// loops look at the row maximum (redo_routine in gen_walk64_loop.py).
constexpr float kNoReference = -3.402823466e38f;

// The segments and items of a launch: the tables in memory, or the one of each that came with the kernel arguments (the
// single parameter of every kernel of this library sits at the start of the argument segment).  Pointers to constant
// memory either way: a table is not written while a kernel runs, and the loads are then scalar ones.
typedef const __attribute__((address_space(4))) SegItem* ItemPtr;
typedef const __attribute__((address_space(4))) Segment* SegPtr;
static __device__ __forceinline__ ItemPtr items_of(const BlockArgs& a) {
  const auto* args = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
  return a.items ? (ItemPtr)(uintptr_t)a.items : (ItemPtr)(args + offsetof(BlockArgs, one_item));
}
static __device__ __forceinline__ SegPtr segs_of(const BlockArgs& a) {
  const auto* args = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
  return a.items ? (SegPtr)(uintptr_t)a.segs : (SegPtr)(args + offsetof(BlockArgs, one_seg));
}

// workgroup -> job (segment, head, q tile); false for the holes of the grid.  blockIdx mod 8 is the XCD.  Heads are dealt
// to the XCDs round-robin, and an XCD runs the segments of a head one after the other (busiest first), the q tiles of a
// segment as consecutive workgroups: everything that reads a head's K and V follows each other through that XCD's L2.
// The batch * heads mod 8 heads that do not deal out evenly are shared: with rem of them, gcd(8, rem) sets of XCDs take
// rem / gcd heads each and split their tiles round-robin, so that one head (or any number) still fills all XCDs.  The last
// a.tail_heads heads of an XCD and its part of the shared ones are interleaved (job_grid says why).
template <int TILE_ROWS>
static __device__ __forceinline__ bool decode_job(const BlockArgs& a, Segment& seg, int& bh, int& qt) {
  const int q_tiles = a.q_tiles_max;
  const int per_head = a.n_segs * q_tiles;
  const int xcd = blockIdx.x & 7, w = blockIdx.x >> 3;
  const int full = a.BH >> 3, rem = a.BH & 7;
  const int lead = (full - a.tail_heads) * per_head;
  int job;  // its number among those of its head
  if (w < lead) {
    bh = (w / per_head) * 8 + xcd;
    job = w % per_head;
  } else {
    int p = w - lead;
    const int own = a.tail_heads * per_head;  // jobs of whole heads
    const int sets = rem & -rem;
    const int share = rem ? 8 / sets : 1, sub = rem ? xcd / sets : 0, heads = rem ? rem / sets : 0;
    const int shared = (heads * per_head - sub + share - 1) / share;  // this XCD's jobs of the shared heads
    if (p >= own + shared) return false;
    // p-th of both lists merged in proportion
    const int from_shared = rem ? (int)((int64_t)p * shared / (own + shared)) : 0;
    const int with_this = rem ? (int)((int64_t)(p + 1) * shared / (own + shared)) : 0;
    if (with_this > from_shared) {
      const int j = from_shared * share + sub;
      job = a.causal ? j / heads : j % per_head;
      bh = (a.BH & ~7) + (xcd & (sets - 1)) + sets * (a.causal ? j % heads : j / per_head);
    } else {
      p -= from_shared;
      job = p / a.tail_heads;
      bh = (full - a.tail_heads + p % a.tail_heads) * 8 + xcd;
    }
  }
  const SegPtr sp = segs_of(a) + job / q_tiles;
  seg.q_start = sp->q_start;
  seg.q_len = sp->q_len;
  seg.item_begin = sp->item_begin;
  seg.item_count = sp->item_count;
  seg.last_item = sp->last_item;
  seg.reverse_tiles = sp->reverse_tiles;
  qt = job % q_tiles;
  if (qt * TILE_ROWS >= seg.q_len) return false;  // segments shorter than the longest one
  if (seg.reverse_tiles) qt = (seg.q_len + TILE_ROWS - 1) / TILE_ROWS - 1 - qt;  // most keys first
  return true;
}

// ---- conversions of 8 columns of a row, shared by the merge kernel and the merge at the end of a workgroup
template <int DT> struct Store8;
template <> struct Store8<0> {
  static __device__ __forceinline__ void st(void* p, const float* x) {
    f16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (_Float16)x[e];
    *(f16x8*)p = v;
  }
};
template <> struct Store8<1> {
  static __device__ __forceinline__ void st(void* p, const float* x) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (__bf16)x[e];
    *(bf16x8*)p = v;
  }
};

// 8 consecutive columns of one partial row as floats
template <bool HP> struct PartRow;
template <> struct PartRow<false> {
  using ptr = const float*;
  static __device__ __forceinline__ void ld(ptr p, f32x4& x0, f32x4& x1) {
    x0 = *(const f32x4*)p;
    x1 = *(const f32x4*)(p + 4);
  }
};
template <> struct PartRow<true> {
  using ptr = const _Float16*;
  static __device__ __forceinline__ void ld(ptr p, f32x4& x0, f32x4& x1) {
    const f16x8 v = *(const f16x8*)p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x0[e] = (float)v[e];
      x1[e] = (float)v[4 + e];
    }
  }
};

// A 32-row block of a wave's accumulators times `scale` (of the lane's own row), to rows `first + r * stride` in memory, those
// with r < rows.  OT: 0 fp16, 1 bf16, 2 fp32.  The accumulators hold O^T: lane (n, h) has four columns of every eight of
// row n, and a store straight from them touches 32 rows with 16 or 32 bytes each -- as many cache lines per instruction
// as rows.  Halves of the wave (and, for 16-bit rows first, the four-column pieces of a lane) are exchanged in registers so
// that a store writes 64 contiguous bytes of 16 rows.  (Forward with fp16 per-step partials, 64 heads x 32 x 512 tokens, d = 128:
// 12.5 -> 12.0 ms; one rank's steps of the 8 x 4096 causal zigzag ring with fp32 partials 1106 -> 1093 us.)
template <int OT, int D>
static __device__ __forceinline__ void store_block(const f32x16 (&acc)[D / 32], float scale, char* first, int64_t stride, int rows) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, c = 2 * ((lane >> 4) & 1) + (lane >> 5);  // row (and row + 16), 16-byte piece of the 64
  char* p0 = first + r * stride + 16 * c;
  char* p1 = p0 + 16 * stride;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  auto swap16 = [](unsigned& x, unsigned& y) {
    const auto s = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = s[0];
    y = s[1];
  };
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int j = 0; j < (OT == 2 ? 2 : 1); ++j) {
      u32x4 x, y;  // fp32: columns 16 j + [0, 4) + 4 h and those eight further on; 16 bits: [0, 8) + 8 h and 16 further on
      if (OT == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = __builtin_bit_cast(unsigned, acc[db][8 * j + e] * scale);
          y[e] = __builtin_bit_cast(unsigned, acc[db][8 * j + 4 + e] * scale);
        }
      } else {
        auto pack = [&](int e) {
          typedef typename Elem<OT == 2 ? 0 : OT>::type T;
          typedef T T2 __attribute__((ext_vector_type(2)));
          const T2 v = {(T)(acc[db][e] * scale), (T)(acc[db][e + 1] * scale)};
          return __builtin_bit_cast(unsigned, v);
        };
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          u32x4& t = k == 0 ? x : y;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const auto s = __builtin_amdgcn_permlane32_swap(pack(8 * k + 2 * i), pack(8 * k + 4 + 2 * i), false, false);
            t[i] = s[0];
            t[2 + i] = s[1];
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        unsigned a = x[e], b = y[e];
        swap16(a, b);
        x[e] = a;
        y[e] = b;
      }
      const int at = (OT == 2 ? 128 * db + 64 * j : 64 * db);
      if (r < rows) *(u32x4*)(p0 + at) = x;
      if (r + 16 < rows) *(u32x4*)(p1 + at) = y;
    }
}

// ---- merge of one job's rows (BM rows of a segment, one head) over the partials of the
// segment's items.  The same arithmetic, in the same order, as merge_row; only the loads are
// arranged differently: the attention kernel, which runs this at the end of a workgroup, has just two
// waves per SIMD to hide memory latency with, and every round trip it waits for is time its
// compute unit runs half empty.  So all partial LSEs are fetched in one sweep and parked in LDS
// (lse_s: [items][BM] floats), and the partial O rows move in batches of 256 bytes per thread
// (two output rows x four or eight parts), three batches in flight at any time.
typedef __attribute__((address_space(3))) float lds_float;
template <int DT, int D, bool HP, int BM, int THREADS>
static __device__ __forceinline__ void merge_job_rows(const void* o_part, const float* lse_part, void* out, float* lse,
                                                      const SegItem* items, const Segment& seg, int bh, int qt, int S,
                                                      lds_float* lse_s) {
  constexpr int WAVES = THREADS / 64;
  constexpr int TPR = D / 8;  // threads per row, 8 columns each
  constexpr int ROWS = THREADS / TPR;
  constexpr int KMAX = kMaxParts / WAVES;  // parts per wave in the LSE sweep
  constexpr int LR = BM / 64;              // rows per lane in the LSE sweep
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_parts = seg.item_count;
  const int row0 = qt * BM;  // first row of the job within the segment
  const int last_row = min(BM, seg.q_len - row0) - 1;
  // lane i keeps where the job's rows begin in the partials of item i
  int64_t first_row = 0;
  if (lane < n_parts) {
    const SegItem* w = items + seg.item_begin + lane;
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
  // R rows and G parts of a thread per batch
  auto merge_in = [&](auto rows_c, auto parts_c) {
    constexpr int R = decltype(rows_c)::value, G = decltype(parts_c)::value;
    constexpr int RSTEP = R * ROWS;
    const int n_groups = (n_parts + G - 1) / G;
    const int n_batches = (BM / RSTEP) * n_groups;  // batch b: rows of b / n_groups, parts of b % n_groups
    struct Batch {
      f32x4 raw[R][G][NV];  // as loaded; fp16 partials are widened when they are used
    };
    auto row_of = [&](int b, int j) { return (b / n_groups) * RSTEP + j * ROWS + rsub; };  // within the job
    // Every load of a batch is made, those of parts and rows that do not exist from the last one that does: with loads under
    // conditions the compiler cannot count those in flight, and waits for the batches fetched ahead as well.  Where the parts
    // lie comes from a lane of first_row and not from the table, a scalar round trip for each.  Together, and past the
    // cache's retention (fp16; fp32 rows measured 1.6 % slower that way): forward with fp16 partials, 64 heads x 32 x 512, d = 128
    // 11.74 -> 10.70 ms, of which the merge was 2.4 ms; fp32 partials, 16 heads 3.74 -> 3.64 ms.
    auto fetch = [&](int b, Batch& t) {
      const int i0 = (b % n_groups) * G;
      int at[R];
#pragma unroll
      for (int j = 0; j < R; ++j) at[j] = min(row_of(b, j), last_row) * (D * (PB / 8)) + c8 * PB;
#pragma unroll
      for (int u = 0; u < G; ++u) {
        if (G == 2 && u == 1 && n_parts == 1) break;  // (nothing is fetched ahead of it that a wait could include)
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
    float mx[R], wsum[R], acc[R][8];
    auto accumulate = [&](int b, const Batch& t) {
      const int g = b % n_groups, i0 = g * G;
      if (g == 0) {  // new rows: L = max over the parts first
#pragma unroll
        for (int j = 0; j < R; ++j) {
          mx[j] = -INFINITY;
          wsum[j] = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[j][e] = 0.f;
        }
        for (int i = 0; i < n_parts; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j) mx[j] = fmaxf(mx[j], lse_s[i * BM + row_of(b, j)]);
      }
#pragma unroll
      for (int u = 0; u < G; ++u)
        if (i0 + u < n_parts) {
#pragma unroll
          for (int j = 0; j < R; ++j) {
            const float L = lse_s[(i0 + u) * BM + row_of(b, j)];
            if (row0 + row_of(b, j) >= seg.q_len || L == -INFINITY) continue;  // identity element: its O may hold anything
            const float w = __expf(L - mx[j]);
            wsum[j] += w;
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
            for (int e = 0; e < 8; ++e) acc[j][e] = __builtin_fmaf(w, x[e], acc[j][e]);
          }
        }
      if (g == n_groups - 1) {  // all parts in: normalise and store
#pragma unroll
        for (int j = 0; j < R; ++j) {
          if (row0 + row_of(b, j) >= seg.q_len) continue;
          if (mx[j] != -INFINITY) {
            const float inv = 1.f / wsum[j];
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[j][e] *= inv;
          }
          const int64_t out_row = (int64_t)bh * S + seg.q_start + row0 + row_of(b, j);
          Store8<DT>::st((char*)out + (out_row * D + c8 * 8) * 2, acc[j]);
          if (c8 == 0) lse[out_row] = (mx[j] == -INFINITY) ? -INFINITY : mx[j] + __logf(wsum[j]);
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
  };
  // 64 registers a batch.  Of a segment with one part or two most of such a batch would be loads of rows that are there
  // already, so these take twice the rows of two parts instead.  Forward with the steps apart, d = 128, us, one shape of batch ->
  // two: 256 heads x 256 tokens, one part 36.8 -> 31.0, with fp16 partials 39.9 -> 25.2 (34.7 and 30.7 with loads under
  // conditions); 2 x 256 tokens 108 -> 95 and 99 -> 73; causal 128 heads x 5 x 256 201 -> 187 and 163 -> 143.
  if (n_parts <= 2) merge_in(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
  else merge_in(std::integral_constant<int, 2>{}, std::integral_constant<int, HP ? 8 : 4>{});
}

}  // namespace ringattn
