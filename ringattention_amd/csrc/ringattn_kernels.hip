// gfx950 (CDNA4) kernels around the attention kernel (ring_walk_kernel, ringattn_walk.hip).
//
//   merge_kernel : P-way merge of per-step (O, LSE) partials over row ranges.  The reference
//       has no such function: it carries (max, sum, acc-O) in registers across ring steps
//       (csrc/ring_attention.cu:439-443,597).  The merge is the algebraic equivalent on
//       (O, LSE) pairs (:207-245,621-633).
#include "ringattn_device.h"

#include <type_traits>


namespace ringattn {

// ---- merge of one row (MergeState in ringattn_device.h) ---------------------------------------------------------------
// The parts of one row: the set bits of a mask over equally spaced slots, ascending from slot `first` on, round to the slots before it.
struct SlotParts {
  uint64_t rest;  // bit i: slot (first + i) mod 64
  int first;
  int64_t row, stride;  // the row in slot 0, rows between slots
  __device__ __forceinline__ int left() const { return __builtin_popcountll(rest); }
  __device__ __forceinline__ int64_t take() {
    const int64_t r = row + (int64_t)((__builtin_ctzll(rest) + first) & 63) * stride;
    rest &= rest - 1;
    return r;
  }
};
// This thread owns columns [8 c8, 8 c8 + 8) of the row.
template <int DT, int D, bool HP, bool AHEAD, class Parts>
static __device__ __forceinline__ void merge_row(Parts p, const void* o_parts, const float* lse_parts,
                                                 void* out, float* lse, int64_t out_row, int c8) {
  const typename PartRow<HP>::ptr o_base = (typename PartRow<HP>::ptr)o_parts + c8 * 8;
  MergeState st;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  auto merge_in = [&](float L, const f32x4& x0, const f32x4& x1) {
    if (L == -INFINITY) return;  // identity element: its O may hold anything
    float keep, w;
    st.weigh(L, keep, w);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[e] = merge_in_part(acc[e], keep, w, x0[e]);
      acc[4 + e] = merge_in_part(acc[4 + e], keep, w, x1[e]);
    }
  };
  // Batches of four parts.  AHEAD: one on its way while another is merged, in 98 to 107 registers, for launches whose parts come from HBM;
  // without it 60, and twice as many waves to wait for memory, for those whose parts the Infinity Cache may hold (launch_merge).
  // 32 heads x 8 x 4096 under the causal mask, fp32 parts, us: batches of one, two, three and four ahead 520, 524, 510, 489, one of four at a
  // time 518, of eight 503.
  constexpr int kBatch = 4;
  struct Batch {
    float L[kBatch];
    f32x4 x0[kBatch], x1[kBatch];
  } batch;
  const int n = p.left();
  auto fetch = [&](Batch& t, int first) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (first + u >= n) break;
      const int64_t r = p.take();
      t.L[u] = lse_parts[r];
      PartRow<HP>::ld(o_base + r * D, t.x0[u], t.x1[u]);
    }
  };
  auto merge_batch = [&](const Batch& t, int first) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (first + u < n) merge_in(t.L[u], t.x0[u], t.x1[u]);
  };
  if constexpr (AHEAD) {
    Batch odd;
    fetch(batch, 0);
    for (int i = 0; i < n; i += 2 * kBatch) {
      fetch(odd, i + kBatch);
      merge_batch(batch, i);
      fetch(batch, i + 2 * kBatch);
      merge_batch(odd, i + kBatch);
    }
  } else {
#pragma unroll 1
    for (int i = 0; i < n; i += kBatch) {
      fetch(batch, i);
      merge_batch(batch, i);
    }
  }
  const float inv = st.inverse();
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (inv == 0.f) acc[e] = 0.f;  // no finite LSE, but perhaps a NaN, which is in the sums
    acc[e] *= inv;  // (the last thing before the store: product and conversion are one rounding in every merge)
  }
  Store8<DT>::st((char*)out + (out_row * D + c8 * 8) * 2, acc);
  if (c8 == 0) lse[out_row] = st.lse();
}

// ---- merge ------------------------------------------------------------------------
template <int DT, int D, bool HP, bool AHEAD>
__global__ __launch_bounds__(256) void merge_kernel(const MergeArgs a) {
  constexpr int TPR = D / 8;  // threads per row, 8 columns each
  constexpr int ROWS = 256 / TPR;
  const MergeRegion reg = a.regions ? a.regions[blockIdx.y] : a.single;
  const int64_t idx = (int64_t)blockIdx.x * ROWS + threadIdx.x / TPR;  // over heads x reg.len
  if (idx >= (int64_t)a.heads * reg.len) return;
  const int64_t row = (idx / reg.len) * a.S + reg.start + idx % reg.len;
  // slot-major partials: slot s of a row lies part_stride_rows rows further on; row-major: at entry row_mul row + s
  const int first = a.slot0_last;
  SlotParts parts{first ? reg.active >> 1 | reg.active << 63 : reg.active, first, a.row_mul > 0 ? row * a.row_mul : row, a.row_mul > 0 ? (int64_t)1 : a.part_stride_rows};
  merge_row<DT, D, HP, AHEAD>(parts, a.o_parts, a.lse_parts, a.out, a.lse, row, threadIdx.x % TPR);
}

// ---- host launchers -----------------------------------------------------------------
// us with 60 registers and with a batch ahead, 8 ranks unless said, under the causal mask: fp32 partials, d = 128, 8 heads x 1024 (152 MB of
// parts) 26.7, 27.3, 16 x 1024 (304 MB) 58.1, 59.1, 16 x 4096 (1.2 GB) 266, 246; d = 64, 8 x 2048 (153 MB) 27.1, 27.9, 16 x 4096 (613 MB) 132, 125;
// fp16, d = 128, 8 heads x 4 x 2048 (43 MB) 10.9, 12.3, 16 x 3 x 5160 (129 MB) 30.3, 34.9, 3 x 11384 (320 MB) 72.7, 74.5, 32 x 4096 (1.2 GB) 297, 277;
// no mask, 3 heads x 12 x 7312 (821 MB) 171, 163, 16 x 5 x 3352, causal (196 MB) 45.5, 53.1.  Between 256 and 512 MB either may be ahead.
constexpr int64_t kMergeAheadBytes = (int64_t)256 << 20;
hipError_t launch_merge(const MergeArgs& a, int dtype, int dim, hipStream_t stream) {
  if (a.n_regions <= 0 || a.max_len <= 0 || a.heads <= 0) return hipSuccess;
  const int rows_per_block = 256 / (dim / 8);
  const int64_t cols = ((int64_t)a.heads * a.max_len + rows_per_block - 1) / rows_per_block;
  if (cols > INT32_MAX || a.n_regions > 65535) return hipErrorInvalidValue;
  const dim3 grid((unsigned)cols, (unsigned)a.n_regions);
  const bool ahead = a.part_rows * (dim * (a.half_partials ? 2 : 4) + (int64_t)sizeof(float)) > kMergeAheadBytes;
#define RA_LAUNCH_MERGE_OF(DT_, D_, HP_)                                                     \
  do {                                                                                      \
    if (ahead) merge_kernel<DT_, D_, HP_, true><<<grid, 256, 0, stream>>>(a);                \
    else merge_kernel<DT_, D_, HP_, false><<<grid, 256, 0, stream>>>(a);                     \
  } while (0)
#define RA_LAUNCH_MERGE(DT_, D_)                           \
  do {                                                    \
    if (a.half_partials) RA_LAUNCH_MERGE_OF(DT_, D_, true); \
    else RA_LAUNCH_MERGE_OF(DT_, D_, false);               \
  } while (0)
  if (dtype == 0 && dim == 64) RA_LAUNCH_MERGE(0, 64);
  else if (dtype == 0 && dim == 128) RA_LAUNCH_MERGE(0, 128);
  else if (dtype == 1 && dim == 64) RA_LAUNCH_MERGE(1, 64);
  else if (dtype == 1 && dim == 128) RA_LAUNCH_MERGE(1, 128);
#undef RA_LAUNCH_MERGE
#undef RA_LAUNCH_MERGE_OF
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
