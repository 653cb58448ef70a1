// Paired instantiations of the block-descent kernel (wide blocks of contact heads without contact rows, two waves a SIMD) for padded
// widths 40 ... 52, and the LDS a paired block takes.
#define NKH_SOLVER_PAIRED
#include "ops_solver_kernel.h"
namespace nkh {
namespace solver {
namespace paired {
template __global__ void BlockDescentTileKernel<40, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
template __global__ void BlockDescentTileKernel<44, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
template __global__ void BlockDescentTileKernel<48, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
template __global__ void BlockDescentTileKernel<52, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
uint32_t BlockFloats(uint32_t n, uint32_t staged) { return SolverLdsFloats(n, staged, staged, true); }
}  // namespace paired
}  // namespace solver
}  // namespace nkh
