// gfx950 (CDNA4) kernel: ring_walk_kernel (ringattn_walk_rows.h) for the forward that keeps the ring steps apart.  A workgroup meets all steps
// of its rows, so their partials need not leave it: each is normalised, rounded as a stored one would be and merged at the
// end of its chunk, by the merge kernel's arithmetic in the merge kernel's order.
#include "ringattn_walk_rows.h"

namespace ringattn {
namespace steps {

template <int DT, int D, bool HP>
__global__ __launch_bounds__(512, 1) void ring_walk_kernel(const BlockArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kWalkLds<D, kBlockPartialsMerged>];
  walk_rows<DT, D, HP, kBlockPartialsMerged>(a, smem);
}

}  // namespace steps

hipError_t launch_steps(const BlockArgs& a, unsigned grid, int dtype, int dim, hipStream_t stream) {
#define RA_LAUNCH_STEPS(DT_, D_)                                                                \
  do {                                                                                         \
    if (a.half_partials) steps::ring_walk_kernel<DT_, D_, true><<<grid, 512, 0, stream>>>(a);  \
    else steps::ring_walk_kernel<DT_, D_, false><<<grid, 512, 0, stream>>>(a);                 \
  } while (0)
  if (dtype == 0 && dim == 64) RA_LAUNCH_STEPS(0, 64);
  else if (dtype == 0 && dim == 128) RA_LAUNCH_STEPS(0, 128);
  else if (dtype == 1 && dim == 64) RA_LAUNCH_STEPS(1, 64);
  else if (dtype == 1 && dim == 128) RA_LAUNCH_STEPS(1, 128);
#undef RA_LAUNCH_STEPS
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
