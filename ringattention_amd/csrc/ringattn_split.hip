// gfx950 (CDNA4) kernel: ring_split_kernel (ringattn_split_rows.h holds the program) with the softmax state carried through all keys.
#include "ringattn_split_rows.h"

namespace ringattn {

template <int DT, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES, D == 64 ? 4 : 2) void ring_split_kernel(const BlockArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[WAVES * kSplitWaveLds<D>];
  __shared__ float2 stat[WAVES][kSplitM];
  split_rows<DT, D, D, WAVES, false, kBlockCarryState>(a, smem, stat);
}

hipError_t launch_split(BlockArgs a, int dtype, int dim, bool many_waves, int columns, hipStream_t stream) {
  if (a.n_segs <= 0) return hipSuccess;
  const int64_t blocks = job_grid(a, a.causal != 0);
  if (a.q_tiles_max <= 0 || blocks > INT32_MAX || a.mode != kBlockCarryState) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)blocks;
  if (many_waves && dim != 64) return hipErrorInvalidValue;
  if (columns != dim) return launch_split_columns(a, grid, dtype, dim, many_waves, columns, stream);
  if (dtype == 0 && many_waves) ring_split_kernel<0, 64, 16><<<grid, 1024, 0, stream>>>(a);
  else if (dtype == 1 && many_waves) ring_split_kernel<1, 64, 16><<<grid, 1024, 0, stream>>>(a);
  else if (dtype == 0 && dim == 64) ring_split_kernel<0, 64, 8><<<grid, 512, 0, stream>>>(a);
  else if (dtype == 1 && dim == 64) ring_split_kernel<1, 64, 8><<<grid, 512, 0, stream>>>(a);
  else if (dtype == 0 && dim == 128) ring_split_kernel<0, 128, 8><<<grid, 512, 0, stream>>>(a);
  else if (dtype == 1 && dim == 128) ring_split_kernel<1, 128, 8><<<grid, 512, 0, stream>>>(a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ringattn
