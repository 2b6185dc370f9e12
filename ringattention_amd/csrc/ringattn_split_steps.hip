// gfx950 (CDNA4) kernel: ring_split_kernel (ringattn_split_rows.h) for the ring steps apart.  The waves take runs of tiles of one key range
// instead of every eighth tile of all; a workgroup goes through as many whole ranges at once as it has waves for, and puts
// the states of each range together to that range's partial.  A step of a ring is a launch of few rows on most of the device's
// compute units idle: 8 heads x 1024 rows are 32 workgroups of ring_walk_kernel or 64 of thin::ring_walk_kernel, whose walk of 32 tiles is a
// chain (0.32 us a tile), and 256 here with four tiles a wave.  us before and after, a step of one rank, one of all, all steps merged: d = 64,
// 4 x 4 x 512 9.9, 10.1, 29.9 and 6.2, 6.9, 17.7; d = 128, 2 x 4 x 2048 46, 49, 163 and 15.3, 36, 123; which plans run on it:
// small_steps in ringattn_api.hip.
// What bounds it: start and combination of a round of ranges (3 us next to 0.5 to 0.7 a tile), and beyond small plans the
// tiles' way from L2, as without the steps.  With 64 rows a wave, or two tiles of a wave in flight, it was no faster.
#include "ringattn_split_rows.h"

namespace ringattn {
namespace steps {

template <int DT, int D, bool HP, int MODE>
__global__ __launch_bounds__(512, D == 64 ? 4 : 2) void ring_split_kernel(const BlockArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[MODE == kBlockPartialsMerged ? kSplitStepsLds<D> : 8 * kSplitWaveLds<D>];
  __shared__ float2 stat[8][kSplitM];
  split_rows<DT, D, D, 8, HP, MODE>(a, smem, stat);
}

}  // namespace steps

hipError_t launch_split_steps(BlockArgs a, int dtype, int dim, int columns, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (a.q_tiles_max <= 0 || blocks > INT32_MAX || a.mode == kBlockCarryState) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  if (columns != dim) return launch_split_columns(a, grid, dtype, dim, false, columns, stream);
#define RA_LAUNCH_OF(DT_, D_, HP_)                                                                                      \
  do {                                                                                                                 \
    if (a.mode == kBlockPartials) steps::ring_split_kernel<DT_, D_, HP_, kBlockPartials><<<grid, 512, 0, stream>>>(a);  \
    else steps::ring_split_kernel<DT_, D_, HP_, kBlockPartialsMerged><<<grid, 512, 0, stream>>>(a);                     \
  } while (0)
#define RA_LAUNCH(DT_, D_)                          \
  do {                                             \
    if (a.half_partials) RA_LAUNCH_OF(DT_, D_, true); \
    else RA_LAUNCH_OF(DT_, D_, false);              \
  } while (0)
  if (dtype == 0 && dim == 64) RA_LAUNCH(0, 64);
  else if (dtype == 0 && dim == 128) RA_LAUNCH(0, 128);
  else if (dtype == 1 && dim == 64) RA_LAUNCH(1, 64);
  else if (dtype == 1 && dim == 128) RA_LAUNCH(1, 128);
#undef RA_LAUNCH
#undef RA_LAUNCH_OF
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
