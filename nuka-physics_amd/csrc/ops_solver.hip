// Launch side of the block-descent solve: head capacity, LDS sizing and the table of kernels, one per padded width.
// The kernel template lives in ops_solver_kernel.h; its instantiations are spread over ops_solver_w*.hip, ops_solver_g*.hip (general)
// and ops_solver_s*.hip (contact heads only) so that they compile in parallel.
#include "ops_solver_kernel.h"

namespace nkh {
namespace solver {
#define NKH_DECLARE_WIDTH(N) \
    extern template __global__ void BlockDescentTileKernel<N, false>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t); \
    extern template __global__ void BlockDescentTileKernel<N, false, N, false>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t); \
    extern template __global__ void BlockDescentTileKernel<N, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
NKH_DECLARE_WIDTH(4) NKH_DECLARE_WIDTH(8) NKH_DECLARE_WIDTH(12) NKH_DECLARE_WIDTH(16) NKH_DECLARE_WIDTH(20) NKH_DECLARE_WIDTH(24)
NKH_DECLARE_WIDTH(28) NKH_DECLARE_WIDTH(32) NKH_DECLARE_WIDTH(36) NKH_DECLARE_WIDTH(40) NKH_DECLARE_WIDTH(44) NKH_DECLARE_WIDTH(48)
NKH_DECLARE_WIDTH(52) NKH_DECLARE_WIDTH(56) NKH_DECLARE_WIDTH(60) NKH_DECLARE_WIDTH(64)
#undef NKH_DECLARE_WIDTH
// with a queue
#define NKH_DECLARE_QUEUE(N) \
    extern template __global__ void BlockDescentTileKernel<N, false, N, false, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
NKH_DECLARE_QUEUE(4) NKH_DECLARE_QUEUE(8) NKH_DECLARE_QUEUE(12) NKH_DECLARE_QUEUE(16) NKH_DECLARE_QUEUE(20) NKH_DECLARE_QUEUE(24) NKH_DECLARE_QUEUE(28)
NKH_DECLARE_QUEUE(32) NKH_DECLARE_QUEUE(36)
#undef NKH_DECLARE_QUEUE
// reduced blocks (contact heads only): width N with the sweeps K wide
#define NKH_DECLARE_REDUCED(N, K) \
    extern template __global__ void BlockDescentTileKernel<N, true, K>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t); \
    extern template __global__ void BlockDescentTileKernel<N, true, K, false, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
NKH_DECLARE_REDUCED(24, 12) NKH_DECLARE_REDUCED(28, 16) NKH_DECLARE_REDUCED(32, 16) NKH_DECLARE_REDUCED(36, 20) NKH_DECLARE_REDUCED(40, 20)
NKH_DECLARE_REDUCED(44, 24) NKH_DECLARE_REDUCED(48, 24) NKH_DECLARE_REDUCED(52, 28) NKH_DECLARE_REDUCED(56, 28) NKH_DECLARE_REDUCED(60, 32)
NKH_DECLARE_REDUCED(64, 32)
#undef NKH_DECLARE_REDUCED
// the same for worlds under the elliptic cone
#define NKH_DECLARE_ELLIPTIC(N, K) \
    extern template __global__ void BlockDescentTileKernel<N, true, K, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
NKH_DECLARE_ELLIPTIC(4, 4) NKH_DECLARE_ELLIPTIC(8, 8) NKH_DECLARE_ELLIPTIC(12, 12) NKH_DECLARE_ELLIPTIC(16, 16) NKH_DECLARE_ELLIPTIC(20, 20)
NKH_DECLARE_ELLIPTIC(24, 12) NKH_DECLARE_ELLIPTIC(28, 16) NKH_DECLARE_ELLIPTIC(32, 16) NKH_DECLARE_ELLIPTIC(36, 20) NKH_DECLARE_ELLIPTIC(40, 20)
NKH_DECLARE_ELLIPTIC(44, 24) NKH_DECLARE_ELLIPTIC(48, 24) NKH_DECLARE_ELLIPTIC(52, 28) NKH_DECLARE_ELLIPTIC(56, 28) NKH_DECLARE_ELLIPTIC(60, 32)
NKH_DECLARE_ELLIPTIC(64, 32)
#undef NKH_DECLARE_ELLIPTIC
// The dense build of the same template (ops_solver_kernel.h compiled with NKH_SOLVER_DENSE: three or four waves a SIMD), for the
// widths it is instantiated at in ops_solver_d*.hip.
namespace dense {
template <int N, bool kContactsOnly, int K = N, bool kElliptic = !kContactsOnly, bool kQueue = true>
__global__ void BlockDescentTileKernel(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
#define NKH_DECLARE_DENSE(N, K) \
    extern template __global__ void BlockDescentTileKernel<N, true, K>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
NKH_DECLARE_DENSE(4, 4) NKH_DECLARE_DENSE(8, 8) NKH_DECLARE_DENSE(12, 12) NKH_DECLARE_DENSE(16, 16) NKH_DECLARE_DENSE(20, 20)
NKH_DECLARE_DENSE(24, 12) NKH_DECLARE_DENSE(28, 16) NKH_DECLARE_DENSE(32, 16) NKH_DECLARE_DENSE(36, 20) NKH_DECLARE_DENSE(40, 20)
#undef NKH_DECLARE_DENSE
}  // namespace dense
// The paired build (NKH_SOLVER_PAIRED, ops_solver_p*.hip): wide blocks of contact heads without contact rows, two waves a SIMD.
namespace paired {
template <int N, bool kContactsOnly, int K = N, bool kElliptic = !kContactsOnly, bool kQueue = false>
__global__ void BlockDescentTileKernel(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
#define NKH_DECLARE_PAIRED(N) \
    extern template __global__ void BlockDescentTileKernel<N, true>(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
NKH_DECLARE_PAIRED(40) NKH_DECLARE_PAIRED(44) NKH_DECLARE_PAIRED(48) NKH_DECLARE_PAIRED(52) NKH_DECLARE_PAIRED(56) NKH_DECLARE_PAIRED(60)
NKH_DECLARE_PAIRED(64)
#undef NKH_DECLARE_PAIRED
uint32_t BlockFloats(uint32_t n, uint32_t staged);   // words of LDS
}  // namespace paired
__host__ __device__ uint32_t PackedEnvFloats(uint32_t staged);
__global__ void PackedDescentKernel(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t);
}  // namespace solver


// Heads the solver's LDS holds: the contact heads (each stages three Jacobian rows) plus one unit head per joint row
// slot.  Returns the contact-head capacity that fits the budget, 0 when not even one does.  The line lies where it was when a
// contact head took 60 words beside its rows, a joint row's 31 and the unit heads' lists a word a place: an environment
// past it is flagged and solved with the heads that fit, and stays so though the records have shrunk since.
constexpr size_t kHeadLdsBytes = 150u * 1024u;
static uint32_t CapacityFloats(uint32_t dof, uint32_t staged, uint32_t joint_heads) {
    const uint32_t fields = (31u * (staged + joint_heads) + 29u * (staged + 1u) + 3u) & ~3u;
    return solver::FactorRegionFloats(dof) + solver::RowFloats(solver::PaddedWidth(dof), staged, false) + fields + 256u +
           (joint_heads != 0u ? solver::kUnitSlots * uint32_t(solver::kWave) : 0u) + solver::LinkAxisFloats(dof);
}
static_assert(kHeadLdsBytes + 32u * 32u * sizeof(float) <= 160u * 1024u, "the largest tile and its kept rows fit a compute unit");
static_assert(solver::kWideStride <= 31u && solver::kWideStride + solver::kNarrowStride <= 60u, "a head takes no more than the capacity allows for");
// a contact point is one head, or four under the pyramidal cone of the MuJoCo law (one scalar head an edge)
static uint32_t HeadsAPoint(const ModelView& m) { return m.any_mujoco != 0u && m.contact_cone == 0u ? kRowsPerPoint : 1u; }
uint32_t SolverHeadCapacity(const ModelView& m, uint32_t slots) {
    const uint32_t want = slots * (m.max_points_per_slot == 0u ? kPointsPerSlot : m.max_points_per_slot) * HeadsAPoint(m);
    const uint32_t joint_heads = m.joint_limit_rows + m.joint_friction_rows + m.joint_drive_rows;
    for (uint32_t staged = want; staged >= 1u; --staged)
        if (size_t{CapacityFloats(m.dof, staged, joint_heads)} * sizeof(float) <= kHeadLdsBytes) return staged;
    return 0u;
}

namespace {
using namespace solver;

// OrderTilesKernel (block_descent_tile.cuh:3097-3121 orders tiles for its persistent kernel; here the order feeds the
// grid): environments sorted by the work their solve is taken to be (solve_cost), costliest first, so that the few long solves
// start at once instead of trailing the launch.  Each of B workgroups sorts every B-th environment, a counting sort on a
// 256-level key, and puts its i-th costliest to place i B + its own number: the costliest of all of them come first, then
// the second ones.  The order inside a level is arbitrary, which changes when an environment runs and nothing it computes.
// One workgroup for all of them was bound by its LDS atomics: 80 us for 65536 environments, 22 for 16384 and 9.5 for 4096,
// 7, 5 and 5 with one for every kOrderEnvs.
constexpr uint32_t kOrderEnvs = 1024u;
__global__ void __launch_bounds__(1024) OrderTilesKernel(DataView d, uint32_t env_count, bool by_points) {
    __shared__ uint32_t bins[256];
    __shared__ uint32_t top;
    const uint32_t t = threadIdx.x, first = blockIdx.x, blocks = gridDim.x;
    if (t < 256u) bins[t] = 0u;
    if (t == 0u) top = 0u;
    __syncthreads();
    if (first == 0u && t == 0u && d.solver_queue != nullptr) *d.solver_queue = 0u;   // the next launch's first place
    const uint32_t mine = first + t * blocks;   // (no workgroup has more environments than threads)
    const bool there = mine < env_count;
    uint32_t cost = 0u;
    if (there) cost = by_points ? solve_cost(d.solver_cost[mine], d.solver_points[mine]) : d.solver_cost[mine];
    const uint32_t largest = wave_max_u(cost);
    if ((t & 63u) == 0u) atomicMax(&top, largest);
    __syncthreads();
    const uint32_t level = 255u - min(cost / (top / 256u + 1u), 255u);
    if (there) atomicAdd(&bins[level], 1u);
    __syncthreads();
    // exclusive prefix of the 256 counts: a scan inside each of the first four wavefronts, then their totals
    __shared__ uint32_t wave_total[4];
    uint32_t count = 0u, through = 0u;
    if (t < 256u) {
        count = bins[t];
        through = count;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t other = __shfl_up(through, o, 64);
            if (int(t & 63u) >= o) through += other;
        }
        if ((t & 63u) == 63u) wave_total[t >> 6u] = through;
    }
    __syncthreads();
    if (t < 256u) {
        uint32_t before = 0u;
        for (uint32_t w = 0u; w < (t >> 6u); ++w) before += wave_total[w];
        bins[t] = before + through - count;
    }
    __syncthreads();
    if (there) d.tile_order[atomicAdd(&bins[level], 1u) * blocks + first] = mine;
}


using SolverKernel = void (*)(ModelView, DataView, BlockDescentSolveParams, uint32_t, uint32_t, uint32_t, uint32_t);
// Three instantiations per padded width, in the order of the first three of Heads (contact heads under the elliptic cone have the two
// tables after it): the general one without and with the elliptic cone's response
// (whose functions and coupled curvatures the other then has no registers and lane reads for: four steps of 1000 servo-driven
// quadrupeds 1934 -> 1880 us, 4096 servo-driven humanoids 1388 -> 1380), and the one for worlds whose heads
// are contact heads only, at most one a lane.
enum Heads : uint32_t { kAnyHeads, kAnyElliptic, kContactHeads, kContactElliptic };
const SolverKernel kSolverKernels[3][16] = {
    {BlockDescentTileKernel<4, false, 4, false>, BlockDescentTileKernel<8, false, 8, false>, BlockDescentTileKernel<12, false, 12, false>,
     BlockDescentTileKernel<16, false, 16, false>, BlockDescentTileKernel<20, false, 20, false>, BlockDescentTileKernel<24, false, 24, false>,
     BlockDescentTileKernel<28, false, 28, false>, BlockDescentTileKernel<32, false, 32, false>, BlockDescentTileKernel<36, false, 36, false>,
     BlockDescentTileKernel<40, false, 40, false>, BlockDescentTileKernel<44, false, 44, false>, BlockDescentTileKernel<48, false, 48, false>,
     BlockDescentTileKernel<52, false, 52, false>, BlockDescentTileKernel<56, false, 56, false>, BlockDescentTileKernel<60, false, 60, false>,
     BlockDescentTileKernel<64, false, 64, false>},
    {BlockDescentTileKernel<4, false>, BlockDescentTileKernel<8, false>, BlockDescentTileKernel<12, false>, BlockDescentTileKernel<16, false>,
     BlockDescentTileKernel<20, false>, BlockDescentTileKernel<24, false>, BlockDescentTileKernel<28, false>, BlockDescentTileKernel<32, false>,
     BlockDescentTileKernel<36, false>, BlockDescentTileKernel<40, false>, BlockDescentTileKernel<44, false>, BlockDescentTileKernel<48, false>,
     BlockDescentTileKernel<52, false>, BlockDescentTileKernel<56, false>, BlockDescentTileKernel<60, false>, BlockDescentTileKernel<64, false>},
    {BlockDescentTileKernel<4, true>, BlockDescentTileKernel<8, true>, BlockDescentTileKernel<12, true>, BlockDescentTileKernel<16, true>,
     BlockDescentTileKernel<20, true>, BlockDescentTileKernel<24, true>, BlockDescentTileKernel<28, true>, BlockDescentTileKernel<32, true>,
     BlockDescentTileKernel<36, true>, BlockDescentTileKernel<40, true>, BlockDescentTileKernel<44, true>, BlockDescentTileKernel<48, true>,
     BlockDescentTileKernel<52, true>, BlockDescentTileKernel<56, true>, BlockDescentTileKernel<60, true>, BlockDescentTileKernel<64, true>}};
// One reduced instantiation per padded width from 24 on: the sweeps run at about half the width.  A world takes it
// when no contact can reach a coordinate from that width on (ModelView::contact_dof_end).
struct ReducedKernel { uint32_t width, reduced; SolverKernel kernel, queue; };   // queue: the instantiation with one, if any
// Contact heads under the elliptic cone at the full widths 4 to 20; wider ones that are not reduced take the general kernel
// (the general kernel keeps what joint rows need: 4096 quadrupeds under the cone 363 -> 347 us a step, 16384 1150 -> 1096, 500 245
// -> 234, the bits the same)
const SolverKernel kEllipticFull[] = {BlockDescentTileKernel<4, true, 4, true>, BlockDescentTileKernel<8, true, 8, true>, BlockDescentTileKernel<12, true, 12, true>,
                                      BlockDescentTileKernel<16, true, 16, true>, BlockDescentTileKernel<20, true, 20, true>};
constexpr uint32_t kEllipticFullMost = 20u;
const ReducedKernel kReducedKernels[] = {
    {24u, 12u, BlockDescentTileKernel<24, true, 12>, BlockDescentTileKernel<24, true, 12, false, true>}, {28u, 16u, BlockDescentTileKernel<28, true, 16>, BlockDescentTileKernel<28, true, 16, false, true>},
    {32u, 16u, BlockDescentTileKernel<32, true, 16>, BlockDescentTileKernel<32, true, 16, false, true>}, {36u, 20u, BlockDescentTileKernel<36, true, 20>, BlockDescentTileKernel<36, true, 20, false, true>},
    {40u, 20u, BlockDescentTileKernel<40, true, 20>, BlockDescentTileKernel<40, true, 20, false, true>}, {44u, 24u, BlockDescentTileKernel<44, true, 24>, BlockDescentTileKernel<44, true, 24, false, true>},
    {48u, 24u, BlockDescentTileKernel<48, true, 24>, BlockDescentTileKernel<48, true, 24, false, true>}, {52u, 28u, BlockDescentTileKernel<52, true, 28>, BlockDescentTileKernel<52, true, 28, false, true>},
    {56u, 28u, BlockDescentTileKernel<56, true, 28>, BlockDescentTileKernel<56, true, 28, false, true>}, {60u, 32u, BlockDescentTileKernel<60, true, 32>, BlockDescentTileKernel<60, true, 32, false, true>},
    {64u, 32u, BlockDescentTileKernel<64, true, 32>, BlockDescentTileKernel<64, true, 32, false, true>}};
// the same with the elliptic cone's response: 2048 humanoids under it 493 -> 408 us a step, by the general kernel at the full
// width before
const ReducedKernel kEllipticKernels[] = {
    {24u, 12u, BlockDescentTileKernel<24, true, 12, true>, nullptr}, {28u, 16u, BlockDescentTileKernel<28, true, 16, true>, nullptr},
    {32u, 16u, BlockDescentTileKernel<32, true, 16, true>, nullptr}, {36u, 20u, BlockDescentTileKernel<36, true, 20, true>, nullptr},
    {40u, 20u, BlockDescentTileKernel<40, true, 20, true>, nullptr}, {44u, 24u, BlockDescentTileKernel<44, true, 24, true>, nullptr},
    {48u, 24u, BlockDescentTileKernel<48, true, 24, true>, nullptr}, {52u, 28u, BlockDescentTileKernel<52, true, 28, true>, nullptr},
    {56u, 28u, BlockDescentTileKernel<56, true, 28, true>, nullptr}, {60u, 32u, BlockDescentTileKernel<60, true, 32, true>, nullptr},
    {64u, 32u, BlockDescentTileKernel<64, true, 32, true>, nullptr}};
// The dense kernels: (padded width of the block, width of the sweeps), contact heads only.
const ReducedKernel kDenseKernels[] = {
    {4u, 4u, dense::BlockDescentTileKernel<4, true, 4>, dense::BlockDescentTileKernel<4, true, 4>}, {8u, 8u, dense::BlockDescentTileKernel<8, true, 8>, dense::BlockDescentTileKernel<8, true, 8>},
    {12u, 12u, dense::BlockDescentTileKernel<12, true, 12>, dense::BlockDescentTileKernel<12, true, 12>}, {16u, 16u, dense::BlockDescentTileKernel<16, true, 16>, dense::BlockDescentTileKernel<16, true, 16>},
    {20u, 20u, dense::BlockDescentTileKernel<20, true, 20>, dense::BlockDescentTileKernel<20, true, 20>}, {24u, 12u, dense::BlockDescentTileKernel<24, true, 12>, dense::BlockDescentTileKernel<24, true, 12>},
    {28u, 16u, dense::BlockDescentTileKernel<28, true, 16>, dense::BlockDescentTileKernel<28, true, 16>}, {32u, 16u, dense::BlockDescentTileKernel<32, true, 16>, dense::BlockDescentTileKernel<32, true, 16>},
    {36u, 20u, dense::BlockDescentTileKernel<36, true, 20>, dense::BlockDescentTileKernel<36, true, 20>}, {40u, 20u, dense::BlockDescentTileKernel<40, true, 20>, dense::BlockDescentTileKernel<40, true, 20>}};
// Batches from this many environments on take a dense kernel where there is one: twice the 3072 wave slots three waves
// a SIMD make of 256 compute units.  A dense wave runs slower than a two-wave one (fewer registers, some spilled), so
// below that the launch is over sooner with the two-wave kernel: its length is then the longest environment's, not the
// machine's throughput.  Measured on the 36-coordinate humanoid: 4096 environments +9 % with the dense kernel, 5120
// +1 %, 6144 -8 %, 8192 -8 %, 65536 -9 %; the 18-coordinate quadruped -9 % at 6144 and -14 % at 65536.
#ifndef NKH_DENSE_BATCH
#define NKH_DENSE_BATCH 6144
#endif
constexpr uint32_t kDenseBatch = NKH_DENSE_BATCH;
// The general kernels without the elliptic cone that run two waves a SIMD, with a queue.
const SolverKernel kQueueKernels[] = {BlockDescentTileKernel<4, false, 4, false, true>, BlockDescentTileKernel<8, false, 8, false, true>,
                                      BlockDescentTileKernel<12, false, 12, false, true>, BlockDescentTileKernel<16, false, 16, false, true>,
                                      BlockDescentTileKernel<20, false, 20, false, true>, BlockDescentTileKernel<24, false, 24, false, true>,
                                      BlockDescentTileKernel<28, false, 28, false, true>, BlockDescentTileKernel<32, false, 32, false, true>,
                                      BlockDescentTileKernel<36, false, 36, false, true>};
// The paired kernels: the seven padded widths from 40 on.
const SolverKernel kPairedKernels[] = {paired::BlockDescentTileKernel<40, true>, paired::BlockDescentTileKernel<44, true>, paired::BlockDescentTileKernel<48, true>,
                                       paired::BlockDescentTileKernel<52, true>, paired::BlockDescentTileKernel<56, true>, paired::BlockDescentTileKernel<60, true>,
                                       paired::BlockDescentTileKernel<64, true>};
// Batches from this many environments on take a paired kernel where there is one.  Below, an environment with a SIMD to itself is over
// sooner.  With as many heads as coordinates or more it is as many as the machine holds at once that way: ropes of 40 to 64 links, all of them
// on the ground, take 0.83 to 0.85 of the plain kernel's step for 2048, 0.87 to 0.92 for 3072 (64 links: 1024 2.36 and 2.53 ms, plain and
// paired, 1536 2.85 and 3.08, 2048 3.33 and 3.23 in steps in a row, 8192 12.22 and 9.90).  With fewer, a block is a shorter one and waits less
// for its matrix products: 26 trees of 37 to 64 coordinates and 2 to 40 heads take 0.83 to 1.18 of the plain kernel's step for 2048, 0.74 to
// 1.07 for 3072, the plain kernel's third round, and 0.77 to 0.96 for 3328.
constexpr uint32_t kPairedBatch = 2048u, kPairedFewHeads = 3328u;
// Compute units, and the rounds of environments over them from which launches of fewer heads pay (OpBlockDescentSolve).
constexpr size_t kUnits = 256u, kManyRounds = 9u;
}  // namespace

void InitSolverKernels() {
    for (const auto& variant : kSolverKernels) {
        for (SolverKernel kernel : variant) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            (void)hipGetLastError();
        }
    }
    for (const ReducedKernel& reduced : kReducedKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(reduced.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    for (SolverKernel elliptic : kEllipticFull) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(elliptic), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    for (const ReducedKernel& elliptic : kEllipticKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(elliptic.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    for (const ReducedKernel& dense : kDenseKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(dense.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    for (const ReducedKernel& reduced : kReducedKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(reduced.queue), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    for (SolverKernel queue : kQueueKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(queue), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    for (SolverKernel paired : kPairedKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(paired), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
}


// The heads a world's solve meets: anything or contact heads only, at most one a lane, either with or without the elliptic cone
// of the MuJoCo law (contact heads under it take the general kernel at full widths past 20).
static Heads HeadsOf(const ModelView& m, uint32_t staged) {
    const uint32_t joint_heads = m.joint_limit_rows + m.joint_friction_rows + m.joint_drive_rows;
    const bool elliptic = m.any_mujoco != 0u && m.contact_cone == 1u;
    if (joint_heads != 0u || staged > uint32_t(solver::kWave)) return elliptic ? kAnyElliptic : kAnyHeads;
    return elliptic ? kContactElliptic : kContactHeads;
}
// The width the sweeps of a world's solve run at: its coordinates, or the K of a reduced block where no contact of the
// world reaches the coordinates from K on and a kernel is compiled for that.
static uint32_t SolverWorkingWidth(const ModelView& m, Heads heads) {
    if (heads == kContactHeads || heads == kContactElliptic)
        for (const ReducedKernel& reduced : kReducedKernels)
            if (reduced.width == solver::PaddedWidth(m.dof) && m.contact_dof_end != 0u && m.contact_dof_end <= reduced.reduced &&
                reduced.reduced <= m.dof) return reduced.reduced;   // (0: a host that did not say; the full width is always right)
    return m.dof;
}
// The kernel of a world's solve, the same with a queue, where there is one, and how many of its waves share a SIMD
struct ChosenKernel { SolverKernel kernel, queue; int waves; bool paired; };
static ChosenKernel KernelOfWidth(const ModelView& m, Heads heads, uint32_t width, uint32_t env_count, uint32_t staged) {
    const uint32_t padded = solver::PaddedWidth(m.dof);
    const int waves = solver::WavesPerSimd(int(solver::PaddedWidth(width)));
    if (heads == kContactHeads && env_count >= kDenseBatch)
        for (const ReducedKernel& dense : kDenseKernels)
            if (dense.width == padded && dense.reduced == solver::PaddedWidth(width) && (width == m.dof || dense.reduced == width))
                return {dense.kernel, dense.queue, solver::DenseWavesPerSimd(int(dense.reduced)), false};
    if (width == m.dof && env_count >= (staged >= m.dof ? kPairedBatch : kPairedFewHeads) && solver::RowsFromLinks(width, heads == kContactHeads, m.rows_from_links))
        return {kPairedKernels[padded / 4u - 10u], nullptr, 2, true};
    if (width != m.dof) {
        static_assert(sizeof(kReducedKernels) == sizeof(kEllipticKernels), "the same pairs of widths");
        for (const ReducedKernel& reduced : heads == kContactElliptic ? kEllipticKernels : kReducedKernels)
            if (reduced.width == padded && reduced.reduced == width) return {reduced.kernel, reduced.queue, waves, false};
    }
    if (heads == kContactElliptic && padded <= kEllipticFullMost) return {kEllipticFull[padded / 4u - 1u], nullptr, waves, false};
    return {kSolverKernels[heads == kContactElliptic ? kAnyElliptic : heads][padded / 4u - 1u],
            heads == kAnyHeads && padded <= uint32_t(solver::kTwoWaveWidth) ? kQueueKernels[padded / 4u - 1u] : nullptr, waves, false};
}
// LDS of a block of that kernel with room for so many contact heads
static size_t BlockLdsBytes(const ModelView& m, Heads heads, uint32_t width, const ChosenKernel& chosen, uint32_t staged) {
    const uint32_t joint_heads = m.joint_limit_rows + m.joint_friction_rows + m.joint_drive_rows;
    return sizeof(float) * (chosen.paired ? paired::BlockFloats(m.dof, staged)
                                          : solver::ReducedSolverLdsFloats(m.dof, width, staged + joint_heads, staged,
                                                                           solver::RowsFromLinks(width, heads == kContactHeads, m.rows_from_links)));
}
// Worlds whose environments are solved four a wavefront (ops_solver_packed.hip): contact heads only, no more of them and no
// more coordinates than a row of sixteen lanes takes.  From a batch on that has wavefronts enough that way: a wavefront
// of four takes longer than any of them alone: 4096 free boxes step in 269 us one a wavefront and 295 packed, 8192 in 336
// and 339 (374 and 364 where every state is new), 16384 in 526 and 418.
//   Sixteen heads take 24.8 KB of LDS a wavefront, six of them a compute unit, where four take 10.5 KB and the registers allow
// twelve: a body of eight coordinates on sixteen points still gains from 8192 on (732 -> 635 us; 1292 -> 1078 at 16384), its sweeps
// are long.  A free body's four points under the pyramidal cone, sixteen heads of short sweeps, gain from half as many again:
// 8192 boxes 271 and 290, 9216 289 and 302, 10240 302 and 312, 11264 322 and 298, 12288 339 and 321, 16384 411 and 363.  With
// eight heads or fewer, or on a tree, that cone gains from 8192 on too (capsules 223 and 223, four-point trees 243 and 236).
constexpr uint32_t kPackedBatch = 8192u, kPackedEdgesBatch = kPackedBatch + kPackedBatch / 2u;
static bool PackedSolverTakes(const ModelView& m, Heads heads, uint32_t staged, uint32_t env_count) {
    const bool edges = m.free_body != 0u && HeadsAPoint(m) != 1u && staged > 8u;
    return heads == kContactHeads && m.dof <= uint32_t(solver::kPackedWidth) && m.max_dof <= 16u && staged <= solver::kPackedHeads &&
        env_count >= (edges ? kPackedEdgesBatch : kPackedBatch);
}
// Environments that have a wavefront to themselves, the costliest: one a compute unit until the others' wavefronts take
// longer than they do (12288 free boxes 395 us without them, 368 with, 16384 444 and 418, 24576 475 and 477, 65536 976 and 989).
static uint32_t PackedAlone(uint32_t env_count) { return env_count < 3u * kPackedBatch ? uint32_t(kUnits) : 0u; }
static size_t PackedLdsBytes(uint32_t staged) { return size_t{kPackedEnvs} * PackedEnvFloats(staged) * sizeof(float); }
// Blocks (one wavefront each, one environment or four) of a world's full-capacity solve launch that a compute unit holds at
// once, as the runtime's occupancy query answers for the kernel and the LDS the launch asks for; 0 without a solve.
uint32_t SolverBlocksPerUnit(const ModelView& m, uint32_t env_count) {
    if (m.rows_per_env == 0u || m.dof == 0u) return 0u;
    const uint32_t staged = SolverHeadCapacity(m, std::max(m.contact_slots, 1u));
    if (staged == 0u) return 0u;
    const Heads heads = HeadsOf(m, staged);
    const uint32_t width = SolverWorkingWidth(m, heads);
    int blocks = 0;
    if (PackedSolverTakes(m, heads, staged, env_count)) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(PackedDescentKernel), solver::kWave, PackedLdsBytes(staged)) != hipSuccess) {
            (void)hipGetLastError();
            return 0u;
        }
        return uint32_t(std::max(blocks, 0));
    }
    const ChosenKernel chosen = KernelOfWidth(m, heads, width, env_count, staged);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(chosen.kernel), solver::kWave,
                                                     BlockLdsBytes(m, heads, width, chosen, staged)) != hipSuccess) {
        (void)hipGetLastError();
        return 0u;
    }
    return uint32_t(std::max(blocks, 0));
}
uint32_t SolverMassFactorFloats(const ModelView& m) {
    if (m.rows_per_env == 0u || m.dof == 0u) return 0u;
    const uint32_t width = SolverSweepWidth(m);
    return solver::MassFactorInMemory(width) ? solver::FactorFloats(solver::PaddedWidth(width)) : 0u;
}
uint32_t SolverSweepWidth(const ModelView& m) {
    if (m.rows_per_env == 0u || m.dof == 0u) return m.dof;
    const uint32_t staged = SolverHeadCapacity(m, std::max(m.contact_slots, 1u));
    return SolverWorkingWidth(m, staged != 0u ? HeadsOf(m, staged) : kAnyHeads);
}

Status OpBlockDescentSolve(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const BlockDescentSolveParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (p->env_count == 0u || p->rows_per_env == 0u || p->articulation_count == 0u) return Status::Ok;
    if (p->articulation_count != p->env_count || m.dof == 0u || m.dof > kMaxDof || p->max_dof != m.max_dof ||
        p->iterations == 0u) return Status::InvalidArgument;
    const uint32_t staged = SolverHeadCapacity(m, p->contact_slots_per_env == 0u ? 1u : p->contact_slots_per_env);
    if (staged == 0u) return Status::InvalidArgument;
    const uint32_t joint_heads = m.joint_limit_rows + m.joint_friction_rows + m.joint_drive_rows;
    const Heads heads = HeadsOf(m, staged);
    const uint32_t width = SolverWorkingWidth(m, heads);
    const ChosenKernel chosen = KernelOfWidth(m, heads, width, p->env_count, staged);
    const SolverKernel kernel = chosen.kernel;
    const auto lds_bytes = [&](uint32_t contact_heads) { return BlockLdsBytes(m, heads, width, chosen, contact_heads); };
    // blocks a compute unit holds at most, whatever their LDS: four a wave of a SIMD
    const size_t most_blocks = 4u * size_t(chosen.waves);
    const auto blocks_per_unit = [&](uint32_t contact_heads) { return std::min<size_t>(most_blocks, (160u * 1024u) / lds_bytes(contact_heads)); };
    // The LDS a block needs grows with the contact heads it can stage, and a scene's slots (every pair that may ever
    // touch, at its largest manifold) outnumber the contacts an environment usually has.  Where a smaller capacity
    // lets more blocks share a compute unit, environments with few contact points go to a launch of that capacity:
    // a launch each for sixteen, twelve, eight, four and two blocks a unit, those the waves allow, before the full one.  Each launch takes the
    // environments whose contact points fall in its range; an environment's results do not depend on its launch.  It has to
    // let half as many blocks again share a unit, for one launch waits for the other's longest environment: 4096 servo-driven
    // humanoids take 2525 us a step in launches of eight and of seven blocks a unit and 1476 us in one of seven; 16384 walkers
    // under the native laws 1.42 ms in launches of eight and five and 1.80 in one of five, 4096 0.58 and 0.67, 1000 0.47 either
    // way.  Twice as many where a point is four heads, for a launch of as many heads then takes fewer of the environments:
    // humanoids under the pyramidal cone in launches of eight and five blocks 506 us for 400 of them, 604 for 2500 and 771 for
    // 6000, in one of five 338, 430 and 756; 4096 walkers in launches of eight, four, two and one 292 us, 685 in one of one.
    // What waiting for that other longest environment costs has to come back over the rounds of the full launch: those humanoids
    // in launches of twelve and five 828 us for 6144 (under five rounds of 1280), 1037 for 8192, 1144 for 9500, 1351 for 11519
    // and 3561 for 32768, in one of five 763, 980, 1117, 1355 and 3616.  Four times as many blocks make it good in fewer rounds:
    // 1000 walkers, eight blocks for one and four rounds, 244 us in their launches and 289 in one.
    // A contact point is at most `a_point` heads, so `few` heads hold few / a_point points whatever their friction: four
    // edges a point under the pyramidal cone.  (While those worlds went to the one full launch, a walker's 304 heads left a
    // compute unit one block for environments of a handful of points: a step of 4096 with a twentieth reset 768 -> 438 us.)
    // Whether the order goes by the counted points in a state that is new.  Under the pyramidal cone the points say how many heads an
    // environment has and little of its Newton steps - some of any count take three times the others' - so that the many-headed
    // ones together ahead of the rest start those later than any order would: four states in turn, by the work alone and by the
    // points, 4096 humanoids 583 and 623 us, 2500 433 and 464, 16384 1855 and 1876, 6000 quadrupeds 462 and 472, 12288 boxes 359 and
    // 370.  Not so where a full launch leaves a compute unit fewer blocks than it has SIMDs, which the few environments of many
    // points have to themselves: 4096 walkers (one block) 305 and 289, 8192 464 and 442.
    const uint32_t a_point = HeadsAPoint(m);
    const bool by_points = d.solver_points != nullptr && (a_point == 1u || blocks_per_unit(staged) < 4u);
    hipLaunchKernelGGL(OrderTilesKernel, dim3((p->env_count + kOrderEnvs - 1u) / kOrderEnvs), dim3(1024), 0, stream, d, p->env_count, by_points);
    if (PackedSolverTakes(m, heads, staged, p->env_count)) {
        const uint32_t alone = PackedAlone(p->env_count);
        hipLaunchKernelGGL(PackedDescentKernel, dim3(alone + (p->env_count - alone + kPackedEnvs - 1u) / kPackedEnvs), dim3(solver::kWave),
                           PackedLdsBytes(staged), stream, m, d, *p, staged, alone);
        return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
    }
    uint32_t first_points = 0u;
    const bool few_rounds = p->env_count < kManyRounds * kUnits * blocks_per_unit(staged);
    if (p->contact_slots_per_env != 0u) {
        for (const size_t blocks : {size_t{16u}, size_t{12u}, size_t{8u}, size_t{4u}, size_t{2u}}) {
            if (blocks > most_blocks) continue;                            // more blocks than the waves allow
            if (blocks_per_unit(staged) >= blocks) break;                  // the full capacity does as well,
            if (2u * blocks < (a_point == 1u ? 3u : 4u) * blocks_per_unit(staged)) continue;   // or nearly
            if (a_point != 1u && few_rounds && first_points == 0u && blocks < 4u * blocks_per_unit(staged)) break;   // too few rounds to split at all
            uint32_t few = staged;
            while (few > 8u && blocks_per_unit(few) < blocks) --few;
            const uint32_t points = few / a_point;
            if (blocks_per_unit(few) < blocks || points < first_points) continue;   // not even eight heads fit that often
            hipLaunchKernelGGL(kernel, dim3(p->env_count), dim3(solver::kWave), lds_bytes(few), stream, m, d, *p, few + joint_heads, few,
                               first_points, points);
            first_points = points + 1u;
        }
    }
    // One launch of more blocks than the machine holds takes as many as it holds, and a queue (ops_solver_kernel.h).  Steps from the same
    // state, and from eight states in turn: 4096 humanoids 682 -> 672 and 800 -> 777 us, 65536 7540 -> 7353 and 7620 -> 7320; 4096 servo-driven
    // ones 1351 -> 1320 and 1551 -> 1508, 16384 4715 -> 4534; 65536 quadrupeds 4547 -> 4459 and 4580 -> 4457.  Blocks of contact heads that are
    // neither reduced nor dense, and those under the elliptic cone, have no kernel for it (4096 quadrupeds 466 and 466, 531 -> 521 in turn; under
    // the cone 595 -> 592), and paired blocks lose by it: eight that start together are better there than eight at any
    // time (8192 ropes 9.87 ms and 10.06).  Nor where the points send environments to several launches, whose blocks are mostly over at once.
    // From a third more environments than blocks on: of fewer most blocks take none from it, and the kernel that has it is a little the
    // slower (twenty trees of every width that has one, as many blocks as are held and a queue against a block an environment: just past the
    // blocks held 0.99 to 1.01 of the step, a quarter past them 0.99 to 1.01, half 0.99 to 1.02, three quarters 0.92 to 1.02, twice 0.96 to 1.00,
    // eight times 0.85 to 0.96).
    const size_t held = kUnits * blocks_per_unit(staged);
    const bool queued = chosen.queue != nullptr && first_points == 0u && d.solver_queue != nullptr && p->env_count > held + held / 3u;
    hipLaunchKernelGGL(queued ? chosen.queue : kernel, dim3(queued ? uint32_t(held) : p->env_count), dim3(solver::kWave), lds_bytes(staged), stream, m, d, *p, staged + joint_heads,
                       staged, queued ? uint32_t(held) : first_points, queued ? kQueued : kInvalid);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

}  // namespace nkh
