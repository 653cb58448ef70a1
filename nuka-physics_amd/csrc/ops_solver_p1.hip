// Paired instantiations of the block-descent kernel (wide blocks of contact heads without contact rows, two waves a SIMD) for padded
// widths 56 ... 64.
#define NKH_SOLVER_PAIRED
#include "ops_solver_kernel.h"
namespace nkh {
namespace solver {
namespace paired {
template __global__ void BlockDescentTileKernel<56, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
template __global__ void BlockDescentTileKernel<60, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
template __global__ void BlockDescentTileKernel<64, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
}  // namespace paired
}  // namespace solver
}  // namespace nkh
