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

hipError_t launch_walk(BlockArgs a, int dtype, int dim, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int q_tiles = a.q_tiles_max;  // kWalkM-row tiles of the longest segment
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (q_tiles <= 0 || blocks > INT32_MAX) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  if (a.mode == kBlockPartialsMerged) return launch_steps(a, grid, dtype, dim, stream);
  if (a.mode != kBlockCarryState && a.mode != kBlockPartials) return hipErrorInvalidValue;
#define RA_LAUNCH_WALK(DT_, D_)                                                                          \
  do {                                                                                                \
    if (a.mode == kBlockCarryState) ring_walk_kernel<DT_, D_, false, true><<<grid, 512, 0, stream>>>(a);   \
    else if (a.half_partials) ring_walk_kernel<DT_, D_, true, false><<<grid, 512, 0, stream>>>(a);         \
    else ring_walk_kernel<DT_, D_, false, false><<<grid, 512, 0, stream>>>(a);                             \
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
