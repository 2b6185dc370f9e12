// gfx950 (CDNA4) kernel: ring_walk_kernel with the softmax state carried through all chunks, and with a stored partial per chunk
// (ringattn_walk_rows.h holds the program; ringattn_steps.hip the kernel that merges the partials as they come).
#include "ringattn_walk_rows.h"

namespace ringattn {

// KEEP: the softmax state is carried through the chunks (kBlockCarryState); otherwise a partial is stored per
// chunk (kBlockPartials; HP: partial O as fp16).
template <int DT, int D, bool HP, bool KEEP>
__global__ __launch_bounds__(512, KEEP || D == 128 ? 1 : 4) void ring_walk_kernel(const BlockArgs a) {
  constexpr int MODE = KEEP ? kBlockCarryState : kBlockPartials;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kWalkLds<D, MODE>];
  walk_rows<DT, D, HP, MODE>(a, smem);
}

// Single ring steps at d = 64: a compute unit holds two workgroups, which gains where there are plenty.  Few of them are better off one
// at a time: the second of two long walks waits for no compute unit to come free, and places without a workgroup (segments
// shorter than the longest) put two on one compute unit while others idle.  us, one at a time and two: a step of a zigzag ring
// (walks of half and of whole chunks), 11 heads x 8 x 1024 (198 workgroups) 23.8, 34.7; 8 x 4 x 4096 (320) 82, 111; 11 x 8 x 2048 (396) 76,
// 67; the masked step of one rank, 24 heads x 4096 (384) 77, 81; 52 x 2048 (416) 52, 48; of all ranks, 12 x 4 x 1500 (288) 35, 42; 11 x 4
// x 2048 (352) 54, 61; 12 x 4 x 2048 (384) 62, 57.
constexpr int kOneAtATime = 81 * 1024;  // bytes of LDS of which a compute unit has no second lot
static bool one_at_a_time(const BlockArgs& a, const Walks& w) {
  const int64_t jobs = (int64_t)w.tiles * a.BH;
  if (jobs <= kComputeUnits) return true;
  if (!w.uneven) return false;
  return jobs <= (w.longest >= 64 ? (a.n_segs == 1 ? 400 : 360) : w.longest >= 32 ? 288 : 0);
}
// The masked step of one rank with more of them: the XCD's second 32 run shortest first (lap_order).  us, one at a time, two as they come
// and two that way: 16 heads x 8192 172, 189, 174; 17 219, 227, 195; 24 257, 276, 235; 32 346, 328, 314; 32 heads x 4096 93, 101, 92; 64 heads x
// 2048 53, 54, 49; 128 118, 106, 101.  Shorter walks: 72 heads x 777 (288) 23.6, 21.3, 23.2; 104 28, 27.6, 28.8.
static bool second_lap_reversed(const BlockArgs& a, const Walks& w) { return w.masked && a.n_segs == 1 && w.longest >= 64; }

hipError_t launch_walk(BlockArgs a, const Walks& walks, int dtype, int dim, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int q_tiles = a.q_tiles_max;  // kWalkM-row tiles of the longest segment
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (q_tiles <= 0 || blocks > INT32_MAX) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  unsigned more_lds = 0;
  if (dim == 64 && a.mode == kBlockPartials) {
    if (one_at_a_time(a, walks)) more_lds = kOneAtATime - kWalkLds<64, kBlockPartials>;
    else if (second_lap_reversed(a, walks)) a.second_lap = (int)(blocks < 2 * kComputeUnits ? blocks : 2 * kComputeUnits) / kXcds;
  }
  if (a.mode == kBlockPartialsMerged) return launch_steps(a, grid, dtype, dim, stream);
  if (a.mode != kBlockCarryState && a.mode != kBlockPartials) return hipErrorInvalidValue;
#define RA_LAUNCH_WALK(DT_, D_)                                                                          \
  do {                                                                                                \
    if (a.mode == kBlockCarryState) ring_walk_kernel<DT_, D_, false, true><<<grid, 512, 0, stream>>>(a);   \
    else if (a.half_partials) ring_walk_kernel<DT_, D_, true, false><<<grid, 512, more_lds, stream>>>(a);  \
    else ring_walk_kernel<DT_, D_, false, false><<<grid, 512, more_lds, stream>>>(a);                      \
  } while (0)
  if (dtype == 0 && dim == 64) RA_LAUNCH_WALK(0, 64);
  else if (dtype == 0 && dim == 128) RA_LAUNCH_WALK(0, 128);
  else if (dtype == 1 && dim == 64) RA_LAUNCH_WALK(1, 64);
  else if (dtype == 1 && dim == 128) RA_LAUNCH_WALK(1, 128);
#undef RA_LAUNCH_WALK
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
