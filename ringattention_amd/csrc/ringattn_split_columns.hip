// gfx950 (CDNA4) kernel: ring_split_kernel (ringattn_split_rows.h) with 64 or 32 columns of V and O in a workgroup, for launches of so few row
// tiles that compute units are left over: the state carried through all keys, or the partial of one key range.  The bits are those
// of the form with all columns; what it gains stands in ringattn_split_rows.h, how many columns in split_columns (ringattn_api.hip).
#include "ringattn_split_rows.h"

namespace ringattn {
namespace columns {

template <int DT, int D, int C, int WAVES, bool HP, int MODE>
__global__ __launch_bounds__(64 * WAVES, D == 64 ? 4 : 2) void ring_split_kernel(const BlockArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[WAVES * kSplitWaveLds<D, C>];
  __shared__ float2 stat[WAVES][kSplitM];
  split_rows<DT, D, C, WAVES, HP, MODE>(a, smem, stat);
}

}  // namespace columns

hipError_t launch_split_columns(const BlockArgs& a, unsigned grid, int dtype, int dim, bool many_waves, int cols, hipStream_t stream) {
#define RA_LAUNCH(DT_, D_, C_, W_, HP_, MODE_) \
  columns::ring_split_kernel<DT_, D_, C_, W_, HP_, MODE_><<<dim3(grid, (D_) / (C_)), 64 * (W_), 0, stream>>>(a)
#define RA_LAUNCH_MODES(DT_, D_, C_)                                                                            \
  do {                                                                                                         \
    if (a.mode == kBlockCarryState && many_waves && D_ == 64) RA_LAUNCH(DT_, D_, C_, D_ == 64 ? 16 : 8, false, kBlockCarryState); \
    else if (a.mode == kBlockCarryState && !many_waves) RA_LAUNCH(DT_, D_, C_, 8, false, kBlockCarryState);     \
    else if (a.mode == kBlockPartials && a.half_partials) RA_LAUNCH(DT_, D_, C_, 8, true, kBlockPartials);      \
    else if (a.mode == kBlockPartials) RA_LAUNCH(DT_, D_, C_, 8, false, kBlockPartials);                        \
    else return hipErrorInvalidValue;                                                                          \
  } while (0)
#define RA_LAUNCH_COLUMNS(DT_)                                   \
  do {                                                          \
    if (dim == 64 && cols == 32) RA_LAUNCH_MODES(DT_, 64, 32);  \
    else if (dim == 128 && cols == 32) RA_LAUNCH_MODES(DT_, 128, 32); \
    else if (dim == 128 && cols == 64) RA_LAUNCH_MODES(DT_, 128, 64); \
    else return hipErrorInvalidValue;                           \
  } while (0)
  if (dtype == 0) RA_LAUNCH_COLUMNS(0);
  else if (dtype == 1) RA_LAUNCH_COLUMNS(1);
  else return hipErrorInvalidValue;
#undef RA_LAUNCH
#undef RA_LAUNCH_MODES
#undef RA_LAUNCH_COLUMNS
  return hipGetLastError();
}

}  // namespace ringattn
