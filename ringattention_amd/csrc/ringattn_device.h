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
  if (D == 32) return 0;  // (four rows of 64 bytes are all banks)
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

// Asks for the arguments that the start of a workgroup goes by, all at once: left to itself the compiler asks for each where it needs it, six
// round trips one after the other in front of the first tile load.  us a step before and after: 4 heads x 512 rows, d = 64 5.91, 5.77, 8 x 1024 10.35, 10.19;
// 8 x 256, d = 128 7.22, 7.11.  (ring_split_kernel with the state carried: no difference, and none made.)
static __device__ __forceinline__ void fetch_arguments(const BlockArgs& a) {
  asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.segs), "s"(a.items), "s"(a.bh_stride), "s"(a.kv_bh_stride), "s"(a.q_tiles_max), "s"(a.BH),
               "s"(a.by_group.mul), "s"(a.by_group.shift), "s"(a.scale_log2), "s"(a.by_q_tiles.mul), "s"(a.by_q_tiles.shift), "s"(a.few),
               "s"(a.by_heads.mul), "s"(a.by_heads.shift), "s"(a.one_seg.q_start), "s"(a.one_seg.q_len), "s"(a.one_seg.item_begin), "s"(a.one_seg.item_count),
               "s"(a.one_seg.reverse_tiles), "s"(a.one_item.kv_start), "s"(a.one_item.kv_len), "s"(a.one_item.diag_off));
}

// An XCD hands its workgroups to its 32 compute units in turn.  Where a compute unit holds two, the first 32 jobs, longest walk first,
// are the first ones of the compute units and the next 32 the second ones: those run shortest first (a.second_lap: how many
// of the XCD's first 64 there are; 0: as they come), so that long walks share a compute unit with short ones.
static __device__ __forceinline__ int lap_order(const BlockArgs& a, int w) {
  constexpr int lap = kComputeUnits / kXcds;
  return w >= lap && w < a.second_lap ? a.second_lap + lap - 1 - w : w;
}

// workgroup -> job (segment, head, q tile); false for the holes of the grid.  blockIdx mod 8 is the XCD.  Heads are dealt
// to the XCDs round-robin, and an XCD runs the segments of a head one after the other (busiest first), the q tiles of a
// segment as consecutive workgroups: everything that reads a head's K and V follows each other through that XCD's L2
// (job_map in ringattn_jobs.h).
// LAPS: compute units hold two workgroups (lap_order).
// Launches of few workgroups do without that table (job_grid).
template <int TILE_ROWS, bool LAPS = false>
static __device__ __forceinline__ bool decode_job(const BlockArgs& a, Segment& seg, int& bh, int& qt) {
  const int place = blockIdx.x >> 3;
  int job;  // its number among those of its head
  if (a.few) {
    job = quotient(blockIdx.x, a.by_heads);
    bh = blockIdx.x - job * a.BH;
  } else if (!job_of(a.map, a.causal, blockIdx.x & 7, LAPS ? lap_order(a, place) : place, bh, job)) return false;
  const int nth = quotient(job, a.by_q_tiles);
  if (!a.items) {
    seg = a.one_seg;
  } else {
    const SegPtr sp = segs_of(a) + nth;
    seg.q_start = sp->q_start;
    seg.q_len = sp->q_len;
    seg.item_begin = sp->item_begin;
    seg.item_count = sp->item_count;
    seg.last_item = sp->last_item;
    seg.reverse_tiles = sp->reverse_tiles;
  }
  qt = job - nth * a.q_tiles_max;
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

// Place in a segment's slice of the item table of the i-th item its workgroups walk: table order, except that item
// `last_item` (the masked one) is moved to the end.
static __device__ __forceinline__ int run_order(const Segment& seg, int i) {
  if (seg.last_item < 0) return i;
  return i == seg.item_count - 1 ? seg.last_item : (i >= seg.last_item ? i + 1 : i);
}

static __device__ __forceinline__ float partial_lse(float l, float ms) {
  return (l > 0.f) ? (ms + __builtin_amdgcn_logf(l)) * 0.6931471805599453f : -INFINITY;
}
// An entry of a normalised partial row as it is stored: as fp16 rounded twice, not by a fused multiply-and-convert.
template <bool HP> static __device__ __forceinline__ float partial_entry(float x, float inv) {
  float p = x * inv;
  if (HP) {
    asm("" : "+v"(p));
    p = (float)(_Float16)p;
  }
  return p;
}

// ---- the merge of per-step partials of a row: L = logsumexp_s L_s, O = sum_s exp(L_s - L) O_s, one part after the other.  The
// reference of the weights is the largest L_s so far; when it moves, the sums so far are scaled down to it (the rescale of
// csrc/ring_attention.cu:226-232).  So a merge needs no look at all the L_s ahead of the first O_s, and a workgroup that
// walks the steps of its rows merges each partial where it arises.  Every merge of a plan's steps (the merge kernel and
// those in the attention kernels) is these operations on the same operands in the same order -- ring steps ascending, the
// masked one last (a causal plan's step 0), as the attention kernels walk them --, so they give the same bits.  ringattn_merge knows
// no plan and takes its parts as they come.  A part with L_s = -inf is the identity: callers pass it by, whatever its O may hold.
struct MergeState {
  float top = -INFINITY, sum = 0.f;  // the reference; the weights' sum against it
  // the weight of a part, and what the sums so far keep
  __device__ __forceinline__ void weigh(float L, float& keep, float& w) {
    constexpr float kLog2e = 1.4426950408889634f;
    const float t = fmaxf(top, L);
    keep = __builtin_amdgcn_exp2f((top - t) * kLog2e);  // 1 while the reference stays, 0 for the first part
    w = __builtin_amdgcn_exp2f((L - t) * kLog2e);
    sum = __builtin_fmaf(sum, keep, w);
    top = t;
  }
  __device__ __forceinline__ float inverse() const { return top == -INFINITY ? 0.f : 1.f / sum; }
  __device__ __forceinline__ float lse() const {
    return top == -INFINITY ? -INFINITY : __builtin_fmaf(__builtin_amdgcn_logf(sum), 0.6931471805599453f, top);
  }
};
static __device__ __forceinline__ float merge_in_part(float acc, float keep, float w, float x) {
  return __builtin_fmaf(w, x, acc * keep);
}

}  // namespace ringattn
