// UABD block-descent contact solve for gfx950.  One 64-lane wavefront owns one environment for the whole solve:
// every velocity sweep, the dual updates and the split-impulse position pass run in a single launch with the
// staged Jacobian rows and per-head state resident in LDS.  A lane is a block coordinate in the matrix phases and
// owns one matrix row IN REGISTERS: the kernel is compiled per padded width N (a multiple of 4, nv <= N <= 64), the
// mass row, the Newton Hessian row and its Cholesky factor row are fully unrolled register arrays, pivots and
// multipliers travel between lanes as scalar lane reads, and LDS only carries what must be read transposed (the
// factor columns of the backward substitution) or broadcast (Jacobian rows, small vectors, read as 16-byte words).
// The mass matrix is constant over a solve, so its factor is built once.  A lane is a head row in the per-head
// phases.  Sums that the reference carries as compensated two-float pairs are double accumulators here (a double
// multiply-add issues at the rate of a float one on this device); nothing is exchanged between environments.
// Two instantiations go beyond the plain block.  A reduced block (template argument K < N) eliminates, once per
// solve, the coordinates from K on that no contact of the world reaches, and sweeps K wide (described above
// mass_times).  A wide block (more than kTwoWaveWidth coordinates) of a world whose contact rows each act through one
// link keeps no Jacobian rows: every entry follows from the row's wrench and the coordinates' motion axes (described
// above link_motion and add_heads_through_links).
//
// Replaces src/phi/backend_cuda/ops/block_descent_tile.cuh (DescendTile :2941-3087 and everything it calls) and
// the helpers it takes from block_descent.cu (:735-820, 1593-1621, 1726-1753) and nk/solve/augmented_row.hpp.
// Blocks: one articulation per environment.  Rows on a single coordinate (joint limit, friction and drive rows) are
// "unit" rows (:799-833): they stage no Jacobian row and touch one diagonal entry and one force entry.
// Not built: free rigid 6x6 blocks, mimic couplings.
#pragma once

#include "nk_device_math.h"
#include "backend.h"
#include "nk_ops.h"

namespace nkh {
namespace solver {
// This header compiles three ways.  Plainly, a block of up to kTwoWaveWidth coordinates runs two waves a SIMD with up to 256
// registers each.  With NKH_SOLVER_DENSE defined (ops_solver_d*.hip) everything below sits in namespace `dense` and a block
// of up to twenty coordinates is compiled for three waves a SIMD, of up to eight for four (DenseWavesPerSimd): 168 or 128
// registers, up to twenty values a lane in scratch memory at some widths (80 bytes at 36/20, 76 at 40/20, 36 at 28/16 and 32/16, 12 at 20 and 24/12),
// the same arithmetic.  A long environment runs a tenth slower that way and a full machine gets a tenth more done, so the
// launcher takes the dense kernels for batches that fill the machine several times over.
//   With NKH_SOLVER_PAIRED defined (ops_solver_p*.hip) it sits in namespace `paired`: wide blocks of contact heads without contact
// rows (Tile::from_links), two waves a SIMD.  A wide wave alone on its SIMD issues an instruction in less than half of its cycles, whatever
// it waits for, and what kept a second one away was LDS, 28 KB a block, not registers: 256 hold the sweeps' rows with some
// forty values a Newton step in scratch memory.  The build keeps no factor in LDS - the substitution hands its columns round
// eight at a time (substitute_by_turns) and a Hessian met again is factored again - and no field that such a head has
// no use for: 20.4 KB, eight blocks a compute unit, and the bits of the plain build (8192 ropes 12.2 -> 9.7 ms a step).
#ifdef NKH_SOLVER_DENSE
namespace dense {
constexpr bool kDense = true;
#else
constexpr bool kDense = false;
#endif
#ifdef NKH_SOLVER_PAIRED
namespace paired {
constexpr bool kPaired = true;
#else
constexpr bool kPaired = false;
#endif

constexpr int kWave = 64;
// Widths up to this run two waves per SIMD (at most 256 registers each); wider rows need the whole register file.
#ifndef NKH_TWO_WAVE_WIDTH
#define NKH_TWO_WAVE_WIDTH 36
#endif
constexpr int kTwoWaveWidth = NKH_TWO_WAVE_WIDTH;
// Waves per SIMD of the dense build at widths it is instantiated at: four where 128 registers hold the block without
// scratch memory (eight coordinates need 126, twelve spill 12 bytes a lane), else three.  A step of 16384 free boxes
// (six coordinates) 642 -> 588 us, of 65536 2128 -> 1904 us, with a fourth wave, while batches of that size took these
// kernels; blocks of up to eight coordinates take them from 6144 to 8191 environments now, or with more than sixteen heads.
constexpr int DenseWavesPerSimd(int width) { return width <= 8 ? 4 : width <= 20 ? 3 : 0; }
#ifdef NKH_SOLVER_DENSE
constexpr int WavesPerSimd(int width) { return DenseWavesPerSimd(width) != 0 ? DenseWavesPerSimd(width) : (width <= kTwoWaveWidth ? 2 : 1); }
#else
constexpr int WavesPerSimd(int width) { return width <= kTwoWaveWidth || kPaired ? 2 : 1; }
#endif
// From this width on a block widens its mass rows to double where it uses them; below it the widened rows are kept over
// the solve (two registers an entry), which pays while they fit.  In the dense build's 168 registers they never do:
// kept, they are what spills (96 B a lane at 20 coordinates, none widened at use; 65536 quadrupeds 6.74 -> 6.48 ms).
#ifndef NKH_WIDEN_AT_USE
#ifdef NKH_SOLVER_DENSE
#define NKH_WIDEN_AT_USE 0
#else
#define NKH_WIDEN_AT_USE 24
#endif
#endif
constexpr int kWidenAtUse = NKH_WIDEN_AT_USE;
// The blocks that are solved four a wavefront (ops_solver_packed.hip): the coordinates and heads a row of sixteen lanes takes
constexpr int kPackedWidth = 8;
constexpr uint32_t kPackedHeads = 16u, kPackedEnvs = 4u;
constexpr int kPackedWaves = 3;   // a SIMD
// Orders the block's LDS words between its lanes.  A block is one wavefront, whose LDS accesses are taken in order, so nothing
// has to be waited for; a barrier of the workgroup waits for the writes all the same, some twenty times a Newton step (333
// humanoids 567 -> 557 us, 4096 743 -> 732, 65536 7758 -> 7678).  A wide block keeps the barrier where matrix rows are read
// behind it: without it those reads move up past it into registers the block does not have (8192 ropes 12.70 -> 12.86 ms).  Where a
// loop over heads has written their fields (apply_moves, update_duals) the fence is taken at every width.
template <int N>
__device__ __forceinline__ void lds_sync() {
    if constexpr (N > kTwoWaveWidth) __syncthreads();
    else wave_sync();
}
constexpr uint32_t kNewtonSteps = 16u;        // block_descent_dense.cuh:14
constexpr uint32_t kLineSearchSteps = 32u;    // block_descent_dense.cuh:15
constexpr float kLineTolerance = 1.0e-6f;     // block_descent_dense.cuh:17
constexpr float kRoundings = 8.0f;            // block_descent_dense.cuh:19
constexpr float kPenaltyConditionCap = 1.0e2f;   // block_descent.cu:71
// Unit heads a coordinate can list for itself (lower limit, upper limit, friction, drive, and room to spare); a block
// with more on one coordinate walks its unit heads serially instead.
constexpr uint32_t kUnitSlots = 6u;
// contributing heads from which a wide block takes the heads' curvature by way of the links (add_heads_through_links)
constexpr uint32_t kLinkHeads = 4u;
// words a head of Tile::wrench: 3 x 6 wrench components, one more for an odd stride
constexpr uint32_t kWrenchStride = 19u;

// Phase timers for development builds (-DNKH_SOLVER_PROFILE): cycles per phase and event counts per environment,
// written over the environment's solver_penalty words at the end of the solve.
#ifdef NKH_SOLVER_PROFILE
#define PROF_BEGIN(c, i) const long long prof_start_##i = clock64()
#define PROF_END(c, i) (c).prof[i] += clock64() - prof_start_##i
#define PROF_COUNT(c, i) (c).prof_count[i] += 1u
#else
#define PROF_BEGIN(c, i)
#define PROF_END(c, i)
#define PROF_COUNT(c, i)
#endif

// The reference sums its gradients, slopes and decrements as two-float compensated sums (TileSum, block_descent_tile.cuh
// :15-46).  Here the same sums run in double: a product of two floats is exact in double, the vector unit executes a
// double multiply-add at the rate of a float one, and one instruction replaces the nine of a compensated step.  The
// rounded result is at least as close to the exact sum as the two-float one.
struct TileSum { double value; };
__device__ __forceinline__ void tile_add(TileSum& s, float x) { s.value += double(x); }
__device__ __forceinline__ void tile_add_product(TileSum& s, float a, float b) { s.value = fma(double(a), double(b), s.value); }
template <int Ctrl>
__device__ __forceinline__ double dpp_move_d(double v) {
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    return double_of(dpp_move_u<Ctrl>(uint32_t(bits)), dpp_move_u<Ctrl>(uint32_t(bits >> 32u)));
}
__device__ __forceinline__ double row_value_d(double v, int row) {
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    const uint32_t low = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(bits)), 16 * row));
    const uint32_t high = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(bits >> 32u)), 16 * row));
    return __longlong_as_double((long long)((uint64_t(high) << 32u) | uint64_t(low)));
}
__device__ __forceinline__ double lane_value_d(double v, int lane) {   // `lane` a compile-time constant at every call site
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    const uint32_t low = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(bits)), lane));
    const uint32_t high = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(bits >> 32u)), lane));
    return __longlong_as_double((long long)((uint64_t(high) << 32u) | uint64_t(low)));
}
// every lane of a row of sixteen ends with the row's sum
__device__ __forceinline__ double row_total_d(double v) {
    v += dpp_move_d<kDppXor1>(v); v += dpp_move_d<kDppXor2>(v); v += dpp_move_d<kDppHalfMirror>(v); v += dpp_move_d<kDppMirror>(v);
    return v;
}
// the sum over the wave: rows of 16 by DPP, then the four rows as scalars; uniform result
__device__ __forceinline__ float wave_total(TileSum s, bool first_row_only = false) {
    const double v = row_total_d(s.value);
    const double a = row_value_d(v, 0);
    // the copies of the first row's heads in lanes 16..63 are left out when only the first sixteen lanes carry terms
    if (first_row_only) return float(a);
    return float((a + row_value_d(v, 1)) + (row_value_d(v, 2) + row_value_d(v, 3)));
}
// the same where only the first N lanes carry terms: the rows past them would add exact zeros
template <int N>
__device__ __forceinline__ float coordinate_total(TileSum s) {
    const double v = row_total_d(s.value);
    const double first = row_value_d(v, 0);
    if constexpr (N <= 16) return float(first);
    else if constexpr (N <= 32) return float(first + row_value_d(v, 1));
    else return float((first + row_value_d(v, 1)) + (row_value_d(v, 2) + row_value_d(v, 3)));
}
__device__ __forceinline__ float first_row_sum(float v) {
    v += dpp_move<kDppXor1>(v); v += dpp_move<kDppXor2>(v); v += dpp_move<kDppHalfMirror>(v); v += dpp_move<kDppMirror>(v);
    return row_value(v, 0);
}

struct Response { float dual_scale, residual_scale; };
// augmented_row.hpp:226-229
__device__ __forceinline__ Response scalar_response(float cap, float compliance) {
    const float product = cap * compliance;
    return product >= 1.0f ? Response{0.0f, 1.0f / compliance} : Response{1.0f - product, cap};
}
// augmented_row.hpp:232-247
__device__ __forceinline__ void scalar_impulse(float dual, float rho, float residual, float compliance, float lower, float upper,
                                               Response r, float* impulse, float* curvature) {
    *impulse = 0.0f; *curvature = 0.0f;
    if (rho <= 0.0f) return;
    if (dual != dual || rho != rho || residual != residual || compliance != compliance || lower != lower || upper != upper) {
        const float invalid = dual + rho + residual + compliance + lower + upper;
        *impulse = invalid; *curvature = invalid;
        return;
    }
    const float k = r.residual_scale;
    const float x = fmaf(k, residual, r.dual_scale * dual);
    *impulse = x < lower ? lower : (x > upper ? upper : x);
    *curvature = x != x ? x : (lower < upper && x >= lower && x <= upper ? k : 0.0f);
}
// augmented_row.hpp:302-318, in two parts: what depends on the dual, the penalty and the friction ratio only, and
// the rest, which takes the residual.  A line search evaluates the second part at every probe and the first once.
struct ConeAxis { float dd, d_low, p, p_low; };
__device__ __forceinline__ ConeAxis cone_axis(float dual, float rho, float mu) {
    // a friction ratio of exactly one (equal coefficients) divides to the dividend itself: skip the two divisions
    const bool unit = mu == 1.0f;
    const bool dual_zero = dual == 0.0f;
    const Recip by_mu = make_recip(mu);   // a ratio of zero gives values that every caller discards
    const float dual_quotient = unit ? dual + float(dual_zero) : div_by(dual + float(dual_zero), by_mu);
    const float dd = dual_zero ? dual : dual_quotient;
    const float low = fmaf(-dd, mu, dual);
    const bool low_zero = low == 0.0f;
    const float low_quotient = unit ? low + float(low_zero) : div_by(low + float(low_zero), by_mu);
    const float d_low = low_zero ? low : low_quotient;
    const float p = rho * mu;
    return ConeAxis{dd, d_low, p, fmaf(rho, mu, -p)};
}
__device__ __forceinline__ float cone_value(ConeAxis a, float residual) {
    const float t = a.p * residual;
    const float t_low = fmaf(a.p, residual, -t) + a.p_low * residual;
    const float sum = a.dd + t;
    const float t_part = sum - a.dd;
    const float sum_low = (a.dd - (sum - t_part)) + (t - t_part);
    return sum + (sum_low + a.d_low + t_low);
}
__device__ __forceinline__ float cone_argument(float dual, float rho, float mu, float residual) {
    return cone_value(cone_axis(dual, rho, mu), residual);
}
// augmented_row.hpp:321-348; curvature entries yy, zz, yz.  The friction ratios depend on the row only, so callers
// that evaluate one row many times compute them once (tangent_ratios) and pass them in.
struct TangentRatios { float mu_y, mu_z, scale; };
__device__ __forceinline__ TangentRatios tangent_ratios(float mu_first, float mu_second) {
    const float scale = fmaxf(mu_first, mu_second);
    return TangentRatios{mu_first <= 0.0f ? 0.0f : mu_first / scale, mu_second <= 0.0f ? 0.0f : mu_second / scale, scale};
}
__device__ __forceinline__ void tangent_impulse(V3 dual, float rho, float res_y, float res_z, float normal_impulse, TangentRatios t,
                                float* fy, float* fz, float* cyy, float* czz, float* cyz) {
    *fy = *fz = *cyy = *czz = *cyz = 0.0f;
    if (rho <= 0.0f) return;
    const float mu_y = t.mu_y, mu_z = t.mu_z;
    const float q_y = mu_y == 0.0f ? 0.0f : cone_argument(dual.y, rho, mu_y, res_y);
    const float q_z = mu_z == 0.0f ? 0.0f : cone_argument(dual.z, rho, mu_z, res_z);
    const float radius = (normal_impulse < 0.0f ? 0.0f : normal_impulse) * fmaxf(t.scale, 0.0f);
    if (q_y != q_y || q_z != q_z || radius != radius || rho != rho) {
        const float invalid = q_y + q_z + radius + rho;
        *fy = *fz = *cyy = *czz = *cyz = invalid;
        return;
    }
    if (radius == 0.0f) return;
    const float norm = hypotf(q_y, q_z);
    if (norm <= radius) {
        *fy = mu_y * q_y; *fz = mu_z * q_z; *cyy = rho * mu_y * mu_y; *czz = rho * mu_z * mu_z;
        return;
    }
    const float dy = q_y / norm, dz = q_z / norm;
    const float cs = rho * radius / norm;
    *fy = mu_y * radius * dy; *fz = mu_z * radius * dz;
    *cyy = cs * mu_y * mu_y * dz * dz; *czz = cs * mu_z * mu_z * dy * dy; *cyz = -cs * mu_y * mu_z * dy * dz;
}
__device__ __forceinline__ void tangent_impulse(V3 dual, float rho, float res_y, float res_z, float normal_impulse, float mu_first, float mu_second,
                                float* fy, float* fz, float* cyy, float* czz, float* cyz) {
    tangent_impulse(dual, rho, res_y, res_z, normal_impulse, tangent_ratios(mu_first, mu_second), fy, fz, cyy, czz, cyz);
}

// ComputeEllipticResponse (augmented_row.hpp:48-55): residual scale k and dual scale s of the three axes
struct EllipticResponse { float kx, ky, kz, sx, st; };
__device__ __forceinline__ EllipticResponse elliptic_response(float cap, float cn, float cy, float cz) {
    const double tangent = fmin(double(cy), double(cz));
    const double normal_scale = 1.0 / (1.0 + double(cap) * cn);
    const double tangent_scale = 1.0 / (1.0 + double(cap) * tangent);
    return EllipticResponse{float(cap * normal_scale), float(cap * tangent_scale * tangent / cy), float(cap * tangent_scale * tangent / cz),
                            float(normal_scale), float(tangent_scale)};
}
// What of EvaluateEllipticImpulse (augmented_row.hpp:58-80) depends on the row alone: the response, the roots of its residual
// scales, the cone's slope in the metric that makes its cross section a circle, and 1 / (1 + slope^2).  A head keeps them from
// its set-up on (three double-precision quotients and four roots, some 350 instructions, were made again at every probe of
// a line: 3.0 k cycles a probe of the elliptic humanoid's longest environment, 1.2 k of a Coulomb one).
struct EllipticCone { EllipticResponse e; float root_x, root_y, root_z, slope, share; };
__device__ __forceinline__ EllipticCone elliptic_cone(float cap, float cn, float cy, float cz, float mu_first) {
    EllipticCone k;
    k.e = elliptic_response(cap, cn, cy, cz);
    k.root_x = sqrtf(k.e.kx); k.root_y = sqrtf(k.e.ky); k.root_z = sqrtf(k.e.kz);
    k.slope = mu_first * k.root_x / k.root_y;
    k.share = 1.0f / (1.0f + k.slope * k.slope);
    return k;
}
// The rest: the projection onto the friction cone; curvature xx yy zz xy xz yz.  Inside, outside and on the cone are
// computed side by side and one is selected, so that a probe carries no branch; the quotients by one divisor share its reciprocal
// and are finished as the division's are, so that they hold over the whole range of the operands.
struct EllipticLine { EllipticCone k; float scaled[3]; Recip by_x, by_y, by_z; };   // with the scaled duals, over a block descent
__device__ __forceinline__ EllipticLine elliptic_line(const EllipticCone& k, V3 dual) {
    return EllipticLine{k, {k.e.sx * dual.x, k.e.st * dual.y, k.e.st * dual.z}, make_recip(k.root_x), make_recip(k.root_y), make_recip(k.root_z)};
}
__device__ __forceinline__ void elliptic_impulse(const EllipticLine& l, float rx, float ry, float rz, float* f, float* cv) {
    const EllipticResponse& e = l.k.e;
    const float root_x = l.k.root_x, root_y = l.k.root_y, root_z = l.k.root_z, m = l.k.slope, a = l.k.share;
    const float xx = fmaf(e.kx, rx, l.scaled[0]), xy = fmaf(e.ky, ry, l.scaled[1]), xz = fmaf(e.kz, rz, l.scaled[2]);
    const float p = quotient_by(xx, l.by_x), q1 = quotient_by(xy, l.by_y), q2 = quotient_by(xz, l.by_z);
    const float t = hypotf(q1, q2);
    const bool inside = t <= m * p, outside = !inside && m * t + p <= 0.0f;
    const float projected = (p + m * t) * a;
    // (t has any size down to a subnormal number, whose reciprocal is none: its exponent comes off it and off the dividends, which
    // are no larger on the cone)
    const int exponent = -__builtin_amdgcn_frexp_expf(t);
    const Recip by_t = make_recip(__builtin_ldexpf(t, exponent));
    const auto over_t = [&](float v) { return quotient_by(__builtin_ldexpf(v, exponent), by_t); };
    const float u1 = over_t(q1), u2 = over_t(q2);
    const float b = over_t(m * projected), along = m * m * a;
    const auto one_of = [&](float within, float on) { return inside ? within : outside ? 0.0f : on; };
    f[0] = one_of(xx, projected * root_x); f[1] = one_of(xy, m * projected * u1 * root_y); f[2] = one_of(xz, m * projected * u2 * root_z);
    cv[0] = one_of(e.kx, e.kx * a);
    cv[1] = one_of(e.ky, e.ky * (along * u1 * u1 + b * u2 * u2));
    cv[2] = one_of(e.kz, e.kz * (along * u2 * u2 + b * u1 * u1));
    cv[3] = one_of(0.0f, root_x * root_y * m * a * u1);
    cv[4] = one_of(0.0f, root_x * root_z * m * a * u2);
    cv[5] = one_of(0.0f, root_y * root_z * (along - b) * u1 * u2);
}

__device__ __forceinline__ uint32_t residual_bits(float value) { return __float_as_uint(value <= FLT_MAX ? fabsf(value) : FLT_MAX); }
__device__ __forceinline__ float along_axis(float impulse, float velocity) { return impulse > 0.0f ? velocity : impulse < 0.0f ? -velocity : 0.0f; }

// Per-head state in LDS, head-major with an odd stride so lane = head reads without bank conflicts.
enum HeadField : uint32_t {
    hSlot,               // the head's row of the environment-major records; kUnowned beside it: the head acts on nothing
    hStride, hAxes, hRho, hCompliance, hLower, hUpper, hMu1, hMu2, hNormalBound,
    hRes, hDual = hRes + 3, hMove = hDual + 3, hStep = hMove + 3, hBase = hStep + 3, hDualScale = hBase + 3, hResidualScale,
    hRelaxStep, hRelaxWeight = hRelaxStep + 3, hRelaxPoint, hC = hRelaxPoint + 3, hColumnsLow = hC + (kPaired ? 0 : 6), hColumnsHigh,
    hRow,                // first of the head's three staged Jacobian rows; kInvalid for a unit head
    hSecond,             // the side that moves is the row's second
    hUnit = hSecond + (kPaired ? 0 : 1),      // the one coordinate a unit head acts on; kInvalid for a staged head
    hUnitValue = hUnit + (kPaired ? 0 : 1),   // its Jacobian entry there
    hFieldCount = hUnitValue + 1
};
// (paired: a contact head's curvature is in its lane's registers, and no head is a unit head: neither has words, and what reads
// or writes them stands behind kPaired or Tile::units)
// Fields that share their words: the rows' sources are done with when a head's residual and base are first written, and an
// assembly's impulses when the next steps are.
constexpr uint32_t hSourceA = hRes, hSourceB = hBase, hF = hStep;
constexpr uint32_t kUnowned = 0x80000000u;

// A contact head under the elliptic cone of the MuJoCo law (block_descent_tile.cuh:645, 778) carries 4 in hAxes: three
// axes, answered by elliptic_impulse.  Such a head has no relaxation state (its dual update takes the projection as it
// is), so the first two words of hRelaxStep hold what it needs instead: the compliances of its two tangent rows.
constexpr uint32_t kAxesElliptic = 4u;
constexpr uint32_t hTangentCompliance = hRelaxStep;
// ... and one of the first 64 its cone's constants (EllipticCone, ten words) in the rest of that state and where only heads
// past the 64th and unit heads keep their curvature.
constexpr uint32_t kConeWords = 10u;
__device__ __forceinline__ constexpr uint32_t cone_field(uint32_t word) { return word < 5u ? hRelaxStep + 2u + word : hC + (word - 5u); }
static_assert(hRelaxPoint == hRelaxStep + 4u && hC == hRelaxPoint + 3u, "five words of the relaxation state from its third on");
__device__ __forceinline__ bool block_axes(uint32_t axes) { return axes >= 3u; }

// A head on one axis uses the first component of every three-component field and none of the block-only fields;
// only block heads (three axes: contact points, which are listed first) use the rest.  The fields are therefore kept
// in two tables: "wide" fields have room for every head, "narrow" fields for the first `narrow` heads and one more
// word that every later head shares.  What is written to that word is the same for all of them: zero for the second and third
// components, the relaxation state, the friction and the column masks, one for the axes and the stride, no row (the
// normal bound apart, which no head on one axis reads).  A head's place in a narrow field is min(h, narrow), one operation
// whatever the number of fields read.
//   A joint row's head takes fifteen words so, and with joint rows on every coordinate the tables are most of a block's LDS:
// 31 words a head (and words where its unit heads are listed) let five blocks of the servo-driven humanoid share a
// compute unit, where fifteen let seven: a step of 4096 of them 1749 -> 1476 us.
__host__ __device__ constexpr uint32_t clamped_span(uint32_t f, uint32_t first, uint32_t end) {   // fields of [first, end) below f
    return f <= first ? 0u : (f >= end ? end - first : f - first);
}
// the narrow fields are these ranges of field ids
__host__ __device__ constexpr uint32_t narrow_below(uint32_t f) {
    return clamped_span(f, hStride, hAxes + 1) + clamped_span(f, hMu1, hNormalBound + 1) +
           clamped_span(f, hRes + 1, hRes + 3) + clamped_span(f, hDual + 1, hDual + 3) + clamped_span(f, hMove + 1, hMove + 3) +
           clamped_span(f, hStep + 1, hStep + 3) + clamped_span(f, hBase + 1, hBase + 3) + clamped_span(f, hRelaxStep, hC) +
           (kPaired ? 0u : clamped_span(f, hC + 1, hC + 6)) + clamped_span(f, hColumnsLow, hSecond + 1);
}
__host__ __device__ constexpr bool narrow_field(uint32_t f) { return narrow_below(f + 1u) != narrow_below(f); }
constexpr uint32_t kNarrowFields = narrow_below(hFieldCount);
constexpr uint32_t kWideFields = hFieldCount - kNarrowFields;
static_assert(kNarrowFields <= 64u, "one lane clears the shared word of each narrow field");
// Both tables are head-major with an odd number of words a head: a field of head h sits at h * stride + its index, so
// every access is one base register (the head's) plus a constant offset, and lanes that read one field of consecutive
// heads fall on different banks.
constexpr uint32_t kWideStride = kWideFields | 1u, kNarrowStride = kNarrowFields | 1u;

struct Tile {
    uint32_t env, lane, n, ldj, heads, cap, narrow, iteration;
    uint32_t n_all;   // n, or past it the coordinates that follow the block's own (a reduced block, described above mass_times)
    float tolerance;
    float* mfac;     // FactorFloats(N) words: Cholesky factor of the mass matrix (rows; columns are read transposed); device memory for a wide block
    float* hfac;     // FactorFloats(N) words: Cholesky factor of the current Newton Hessian (paired: none)
    float* jac;      // 3 * staged capacity rows x ldj, ldj = N
    float* fields;   // cap x kWideStride, then (narrow + 1) x kNarrowStride
    float* vec;      // 4 x 64 scratch vectors (paired: kTurnFloats words), 16-byte aligned
    float* hrows;    // blocks of at most 32 coordinates: N x N words, the Hessian of the last assembly in full
    float* low;      // a reduced block: N x N words, the second floats of its mass rows
    float mass_inverse;   // 1 / diagonal of the mass factor, lane = row
    mutable float curvature[6];      // of lane's own head at the last assembly
    mutable float factor_root;       // the diagonal of that factor, lane = row
    mutable bool rows_current;       // ... and since hrows was written
    mutable bool factor_current;     // no head's curvature has changed since hfac was factored: the Hessian is the same
    mutable uint32_t work;   // Newton steps and line probes of this solve, the next solve's scheduling key
    bool mass_valid;
    bool elliptic;   // some head is under the elliptic cone: every response goes through the general functions
    bool smooth;     // the kernel answers the elliptic cone
    bool units;      // some head is a unit head
    bool scalar_later;   // the heads past the first 64 are on one axis, and two a lane hold them
    bool block_heads;   // every staged head of the first 64 has three axes and reaches no further than the first columns (add_block_heads)
    bool near_heads; // no staged head's rows reach past the coordinates two tiles hold (add_heads_by_tiles)
    bool unit_lists; // every coordinate's unit heads fit its list
    uint16_t* unit_list;      // kUnitSlots x 64: lane's unit heads in head order, slot-major
    uint32_t unit_count;      // lane's own count
    uint32_t unit_most;       // the largest
    uint32_t staged_end;      // one past the last staged head
    uint32_t individual_end;  // one past the last head whose inertial response is computed for itself
    float momentum, residual;
    bool failed;
    // what add_heads_through_links needs (wide blocks only)
    bool from_links;          // the block keeps no contact rows: their entries follow from `wrench` and `axes` wherever a row is read
    float* wrench;            // cap x kWrenchStride: a head's three rows as wrenches about `pivot` (its way to the root takes the words of its column mask)
    bool through_links;       // every staged head acts on the block through one link: the heads' curvature may go by way of the links
    float* axes;              // 64 x 12: a coordinate's motion axis about `pivot`, then the contact stiffness it carries times that axis
    uint32_t path_low, path_high;     // lane = coordinate: the coordinates on the way from its link to the root, itself included
    uint32_t under_low, under_high;   // the coordinates whose way to the root passes through lane's
    uint32_t over_low, over_high;     // the heads whose way to the root passes through lane's coordinate
    bool over_runs;                   // those are neighbours in the list of heads, for every coordinate (a chain, or limbs in turn)
    bool way_runs;                    // and every head's way to the root is a run of coordinates (a chain)
    mutable bool stiffness_current;   // no head's curvature has changed since the stiffness in `axes` was summed
    V3 pivot;                 // the point the axes and the heads' wrenches are taken about: the root link's origin
    const float* rows;        // the environment-major row records and row points of device memory
    const float* row_point_a, *row_point_b;
#ifdef NKH_SOLVER_PROFILE
    mutable long long prof[32];
    mutable uint32_t prof_count[4];
#endif
    // with a constant field, as at nearly every call, the place of the field folds to a constant
    __device__ __forceinline__ uint32_t at(uint32_t field, uint32_t h) const {
        const uint32_t below = narrow_below(field);
        if (!narrow_field(field)) return h * kWideStride + (field - below);
        return kWideStride * cap + min(h, narrow) * kNarrowStride + below;
    }
    __device__ __forceinline__ float& F(uint32_t field, uint32_t h) const { return fields[at(field, h)]; }
    __device__ __forceinline__ uint32_t& U(uint32_t field, uint32_t h) const { return reinterpret_cast<uint32_t*>(fields)[at(field, h)]; }
    __device__ __forceinline__ uint32_t slot(uint32_t h) const { return U(hSlot, h) & ~kUnowned; }
    __device__ __forceinline__ bool owned(uint32_t h) const { return (U(hSlot, h) & kUnowned) == 0u; }
};

// the cone of head h, which is under the elliptic cone
__device__ __forceinline__ void keep_cone(const Tile& c, uint32_t h, const EllipticCone& k) {
    const float words[kConeWords] = {k.e.kx, k.e.ky, k.e.kz, k.e.sx, k.e.st, k.root_x, k.root_y, k.root_z, k.slope, k.share};
#pragma unroll
    for (uint32_t w = 0u; w < kConeWords; ++w) c.F(cone_field(w), h) = words[w];
}
__device__ __forceinline__ EllipticCone cone_of(const Tile& c, uint32_t h) {
    if (h >= uint32_t(kWave))
        return elliptic_cone(c.F(hRho, h), c.F(hCompliance, h), c.F(hTangentCompliance, h), c.F(hTangentCompliance + 1, h), c.F(hMu1, h));
    float w[kConeWords];
#pragma unroll
    for (uint32_t k = 0u; k < kConeWords; ++k) w[k] = c.F(cone_field(k), h);
    return EllipticCone{EllipticResponse{w[0], w[1], w[2], w[3], w[4]}, w[5], w[6], w[7], w[8], w[9]};
}

// lane's row of Tile::low, as sixteen-byte words
template <int N>
__device__ __forceinline__ const float4* low_row(const Tile& c) { return reinterpret_cast<const float4*>(c.low + min(c.lane, uint32_t(N - 1)) * uint32_t(N)); }

// TileResponse (block_descent_tile.cuh:678-681) with the Coulomb branch of EvaluateAugmentedResponse (block_descent.cu:1593-1621)
__device__ __forceinline__ void head_response(const Tile& c, uint32_t h, float mx, float my, float mz, float* f, float* cv) {
    const float rho = c.F(hRho, h);
    if (c.elliptic && c.U(hAxes, h) == kAxesElliptic) {   // block_descent.cu:1595-1601
        elliptic_impulse(elliptic_line(cone_of(c, h), V3{c.F(hDual, h), c.F(hDual + 1, h), c.F(hDual + 2, h)}), c.F(hRes, h) - mx,
                         c.F(hRes + 1, h) - my, c.F(hRes + 2, h) - mz, f, cv);
        return;
    }
    float ni, nc;
    scalar_impulse(c.F(hDual, h), rho, c.F(hRes, h) - mx, c.F(hCompliance, h), c.F(hLower, h), c.F(hUpper, h),
                   Response{c.F(hDualScale, h), c.F(hResidualScale, h)}, &ni, &nc);
    f[0] = ni; f[1] = f[2] = 0.0f;
    cv[0] = nc; cv[1] = cv[2] = cv[3] = cv[4] = cv[5] = 0.0f;
    if (!block_axes(c.U(hAxes, h))) return;
    tangent_impulse(V3{c.F(hDual, h), c.F(hDual + 1, h), c.F(hDual + 2, h)}, rho, c.F(hRes + 1, h) - my, c.F(hRes + 2, h) - mz,
                    c.F(hNormalBound, h), c.F(hMu1, h), c.F(hMu2, h), &f[1], &f[2], &cv[1], &cv[2], &cv[5]);
}

// A pivot's reciprocal square root by the hardware approximation (an ulp or so): the pivot's place in the factor is
// pivot * scale and its reciprocal is scale, two instructions on the chain every later pivot waits for where a
// correctly rounded root and quotient take about fifteen.  The factor differs from the correctly rounded one by a
// backward error of a few ulp in the matrix, which a Newton direction does not see.
__device__ __forceinline__ float pivot_scale(float pivot) { return __builtin_amdgcn_rsqf(pivot); }

// FactorTileBlock (:1622-1645) on register rows: lane i holds row i of the symmetric matrix; on return its entries
// k < i are row i of the strict lower triangle of the Cholesky factor and every other entry is zero, so that a
// substitution takes each entry without a condition; the diagonal is `root`, with `inverse` the scale its pivot gave.
// Element (i, j) loses L_ik L_jk for k = 0, 1, ... in that order, as the reference's serial inner loop does; each product
// and subtraction is one fused multiply-add (the reference is built with its compiler's default contraction, so it fuses
// these too).  A pivot that is not positive and finite gives a scale that is not: one look at the scales at the end
// (uniform result, false on a bad pivot) instead of a test a pivot.  A lane takes the scale of every pivot up to its
// own and keeps the last, so one comparison a pivot serves the mask and, a pivot later, the diagonal.
__device__ __forceinline__ bool pivots_valid(uint32_t lane, uint32_t N, float inverse) {
    return __all(lane >= N || (inverse > 0.0f && inverse <= FLT_MAX));
}
// Four columns go as a panel: within it a column's update takes lane reads, and the columns past it lose each of the
// panel's four on the matrix cores.  v_mfma_f32_4x4x1 multiplies, in each block of four lanes, four values a block with one a
// lane, and its broadcast of one block's four to all sixteen (cbsz 4, abid q) takes the column's own register for both
// sides: the words of rows 4 q .. 4 q + 3 against the lane's own come out in the rows' layout, columns 4 q .. 4 q + 3 of
// the lane's row, with nothing passed through LDS.  An instruction for four columns where a lane read and a multiply-add an entry
// go otherwise, each the fused multiply-add it was and in the same order, bit for bit.  (With the panel's words handed round
// through LDS, an exchange and two waits a panel, a step of 8192 ropes took 17.45 ms, 16.62 as it is; 1000 servo-driven
// quadrupeds, four steps, 2062 and 2026 us; 4096 humanoids, whose reduced blocks took lane reads throughout, 784 and 780.)
typedef float Vec4 __attribute__((ext_vector_type(4)));
// v where bit `at` of the mask is set, else zero: two instructions, no comparison
__device__ __forceinline__ uint32_t bit_spread(uint32_t mask, uint32_t at) { return uint32_t(__builtin_amdgcn_sbfe(int(mask), at, 1u)); }
__device__ __forceinline__ float kept_if(uint32_t mask, uint32_t at, float v) { return __uint_as_float(bit_spread(mask, at) & __float_as_uint(v)); }
// columns 4 Q .. 4 Q + 3 lose own x the `column` of rows 4 Q .. 4 Q + 3
template <int Q, int N>
__device__ __forceinline__ void subtract_product(float column, float own, float (&row)[N]) {
    const Vec4 four = __builtin_amdgcn_mfma_f32_4x4x1f32(column, -own, Vec4{row[4 * Q], row[4 * Q + 1], row[4 * Q + 2], row[4 * Q + 3]}, 4, Q, 0);
#pragma unroll
    for (int t = 0; t < 4; ++t) row[4 * Q + t] = four[t];
}
// the groups of columns First .. End - 1 (a matrix instruction names the block it broadcasts in its encoding)
template <int First, int End, int N>
__device__ __forceinline__ void subtract_products(float column, float own, float (&row)[N]) {
    if constexpr (First < End) {
        subtract_product<First>(column, own, row);
        subtract_products<First + 1, End>(column, own, row);
    }
}
template <int Q, int N>   // from group Q down to the first
__device__ __forceinline__ void subtract_products_down(float column, float own, float (&row)[N]) {
    if constexpr (Q >= 0) {
        subtract_product<Q>(column, own, row);
        subtract_products_down<Q - 1>(column, own, row);
    }
}
template <int K, int N>
__device__ __forceinline__ void factor_pivots(uint32_t lane, float (&row)[N], float* inverse, float* root) {
    if constexpr (K < N) {
        const float scale = pivot_scale(lane_value(row[K], K));
        const float scaled = row[K] * scale;
        if (lane >= uint32_t(K)) { *inverse = scale; *root = scaled; }
        row[K] = lane > uint32_t(K) ? scaled : 0.0f;
#pragma unroll
        for (int j = K + 1; j < K / 4 * 4 + 4; ++j) row[j] = fmaf(-row[K], lane_value(row[K], j), row[j]);
        subtract_products<K / 4 + 1, N / 4>(row[K], row[K], row);
        factor_pivots<K + 1>(lane, row, inverse, root);
    }
}
template <int N>
__device__ __forceinline__ bool factor_rows(uint32_t lane, float (&row)[N], float* inverse_out, float* root_out) {
    lane = local_lane(lane);
    float inverse = 0.0f, root = 0.0f;
    factor_pivots<0>(lane, row, &inverse, &root);
    *inverse_out = inverse; *root_out = root;
    return pivots_valid(lane, uint32_t(N), inverse);
}

// Past 32 coordinates the reference's tile is "wide" (TileSpan > 1, :71-73) and factors H = U U^T from the last
// coordinate down, "so a tree's leaves go first" (FactorTileColumns :209-252); its substitutions run up the columns of
// U and then down its rows (SolveWideTileBlock :1866-1895).  Which end the elimination starts from decides whether a
// long chain's block can be factored in single precision at all, so the order is part of the path's arithmetic.
template <int N>
constexpr bool kLeavesFirst = N > 32;

// Where a factor is kept for its transposed reads, the diagonal's place holding zero.  Root first: rows of N words, moved
// sixteen bytes at a time.  Leaves first: lane i's row of U holds the entries k >= i only, and the rows are packed - row i
// starts at i N - i (i - 1) / 2 and is N - i words long - which halves the storage; a column's words for consecutive
// lanes are consecutive.
__host__ __device__ constexpr uint32_t FactorFloats(uint32_t N) { return N > 32u ? (N * (N + 1u) / 2u + 3u) & ~3u : N * N; }
template <int N>
__device__ __forceinline__ uint32_t factor_at(uint32_t i, uint32_t k) {   // leaves first: k >= i
    if constexpr (kLeavesFirst<N>) return i * uint32_t(N) - (i * (i - 1u)) / 2u + (k - i);
    else return i * uint32_t(N) + k;
}

// FactorTileColumns on register rows: lane i holds row i of the symmetric matrix; on return its entries k > i are
// row i of U, every other entry is zero, and `root` is the diagonal.  Panels of four columns as above.
template <int K, int N>
__device__ __forceinline__ void factor_pivots_up(uint32_t lane, float (&row)[N], float* inverse, float* root) {
    if constexpr (K >= 0) {
        const float scale = pivot_scale(lane_value(row[K], K));
        const float scaled = row[K] * scale;
        if (lane <= uint32_t(K)) { *inverse = scale; *root = scaled; }
        row[K] = lane < uint32_t(K) ? scaled : 0.0f;
#pragma unroll
        for (int j = K - 1; j >= K / 4 * 4; --j) row[j] = fmaf(-row[K], lane_value(row[K], j), row[j]);
        subtract_products_down<K / 4 - 1>(row[K], row[K], row);
        factor_pivots_up<K - 1>(lane, row, inverse, root);
    }
}
template <int N>
__device__ __forceinline__ bool factor_rows_up(uint32_t lane, float (&row)[N], float* inverse_out, float* root_out) {
    lane = local_lane(lane);
    float inverse = 0.0f, root = 0.0f;
    factor_pivots_up<N - 1>(lane, row, &inverse, &root);
    *inverse_out = inverse; *root_out = root;
    return pivots_valid(lane, uint32_t(N), inverse);
}

// SolveWideTileBlock: U w = g with lane's own row (entries right of the diagonal), then U^T d = w with the columns,
// read from the factor several at a time.  The rows hold zeros from the diagonal on, so no step asks which lanes it
// is for: a lane whose entry is final loses an exact zero.
template <int N>
__device__ __forceinline__ float substitute_up(uint32_t lane, const float (&row)[N], const float* factor, float inverse, float g) {
    lane = local_lane(lane);
    float r = g;
#pragma unroll
    for (int j = N - 1; j >= 0; --j) r = fmaf(row[j], -lane_value(r * inverse, j), r);
    r *= inverse;
    const uint32_t mine = lane < uint32_t(N) ? lane : 0u;
    constexpr int kAhead = N > kTwoWaveWidth ? 16 : 8;   // a wide block has the registers for twice the reads in flight
#pragma unroll
    for (int j0 = 0; j0 < N; j0 += kAhead) {
        float u[kAhead];
#pragma unroll
        for (int t = 0; t < kAhead; ++t)   // U[j][lane] for the lanes past j; the others read the first diagonal's word, a zero
            u[t] = j0 + t < N ? factor[mine >= uint32_t(j0 + t) ? factor_at<N>(uint32_t(j0 + t), mine) : 0u] : 0.0f;
#pragma unroll
        for (int t = 0; t < kAhead; ++t)
            if (j0 + t < N) r = fmaf(u[t], -lane_value(r * inverse, j0 + t), r);
    }
    return r * inverse;
}

// The same from the rows alone: the lanes of eight rows at a time put them into `turn`, where every lane finds its
// column's eight words, the next eight under way while these are used.  A block's LDS accesses are taken in order: nothing is
// waited for but the words.  72 writes of sixteen bytes where a stored factor takes 64 of four, and a quarter of its LDS.  Lanes
// ahead of the eight find what an earlier turn left: their own entries have been taken (`solved`) by then.
constexpr uint32_t kTurnRows = 8u, kTurnStride = 68u, kTurnFloats = kTurnRows * kTurnStride;   // (the eight rows' words in different banks)
template <int First, int N>
__device__ __forceinline__ void take_turn(uint32_t lane, const float (&row)[N], float* turn, float (&u)[kTurnRows]) {
    if ((lane >> 3u) == uint32_t(First) / kTurnRows) {
        float4* words = reinterpret_cast<float4*>(turn + (lane & 7u) * kTurnStride);
#pragma unroll
        for (int q = First / 4; q < N / 4; ++q) words[q] = float4{row[4 * q], row[4 * q + 1], row[4 * q + 2], row[4 * q + 3]};
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < int(kTurnRows); ++t) u[t] = First + t < N ? turn[uint32_t(t) * kTurnStride + lane] : 0.0f;   // U[j][lane], zero up to the diagonal
    wave_sync();
}
template <int First, int N>
__device__ __forceinline__ void substitute_turns(uint32_t lane, const float (&row)[N], float* turn, float inverse, const float (&u)[kTurnRows], float& r, float& solved) {
    if constexpr (First < N) {
        float next[kTurnRows];
        if constexpr (First + int(kTurnRows) < N) take_turn<First + int(kTurnRows)>(lane, row, turn, next);
#pragma unroll
        for (int t = 0; t < int(kTurnRows); ++t)
            if (First + t < N) r = fmaf(u[t], -lane_value(r * inverse, First + t), r);
        solved = (lane >> 3u) == uint32_t(First) / kTurnRows ? r * inverse : solved;
        substitute_turns<First + int(kTurnRows)>(lane, row, turn, inverse, next, r, solved);
    }
}
template <int N>
__device__ __forceinline__ float substitute_by_turns(uint32_t lane, const float (&row)[N], float* turn, float inverse, float g) {
    lane = local_lane(lane);
    float r = g, solved = 0.0f, u[kTurnRows];
    take_turn<0>(lane, row, turn, u);
#pragma unroll
    for (int j = N - 1; j >= 0; --j) r = fmaf(row[j], -lane_value(r * inverse, j), r);
    r *= inverse;
    substitute_turns<0>(lane, row, turn, inverse, u, r, solved);
    return lane < uint32_t(N) ? solved : 0.0f;
}

// SolveTileBlock (:1647-1666): forward with the factor's rows, backward with its columns (col[j] = L_j,lane), both zero
// from the diagonal on.
template <int N>
__device__ __forceinline__ float substitute(const float (&row)[N], const float (&col)[N], float inverse, float g) {
    // Lane j's entry is final once the steps before it have run, so it is scaled by its reciprocal pivot where it is
    // read (the same product that would be stored back) and the lanes take it in one multiplication after the sweep.
    float r = g;
#pragma unroll
    for (int j = 0; j < N; ++j) r = fmaf(row[j], -lane_value(r * inverse, j), r);
    r *= inverse;
#pragma unroll
    for (int j = N - 1; j >= 0; --j) r = fmaf(col[j], -lane_value(r * inverse, j), r);
    return r * inverse;
}

template <int N>
__device__ __forceinline__ void store_rows(float* a, uint32_t lane, const float (&row)[N]) {
    lane = local_lane(lane);
    if (lane >= uint32_t(N)) return;
    if constexpr (kLeavesFirst<N>) {
        // the entries left of the diagonal are zeros and go to the diagonal's place, a zero too: no condition a word
        float* diagonal = a + factor_at<N>(lane, lane);
#pragma unroll
        for (int k = 0; k < N; ++k) diagonal[max(k - int(lane), 0)] = row[k];
    } else {
        float4* words = reinterpret_cast<float4*>(a + lane * uint32_t(N));
#pragma unroll
        for (int q = 0; q < N / 4; ++q) words[q] = float4{row[4 * q], row[4 * q + 1], row[4 * q + 2], row[4 * q + 3]};
    }
}
// (A packed row's words are read without a condition, which compiles to a branch a word: left of the diagonal the
// diagonal's place answers, a zero; a lane past the rows reads the last row's.)
template <int N>
__device__ __forceinline__ void load_rows(const float* a, uint32_t lane, float (&row)[N]) {
    lane = local_lane(lane);
    const uint32_t from = lane < uint32_t(N) ? lane : uint32_t(N - 1);
    if constexpr (!kLeavesFirst<N>) {
        const float4* words = reinterpret_cast<const float4*>(a + from * uint32_t(N));
#pragma unroll
        for (int q = 0; q < N / 4; ++q) {
            const float4 w = words[q];
            row[4 * q] = w.x; row[4 * q + 1] = w.y; row[4 * q + 2] = w.z; row[4 * q + 3] = w.w;
        }
        return;
    }
    const float* diagonal = a + factor_at<N>(from, from);
#pragma unroll
    for (int k = 0; k < N; ++k) row[k] = diagonal[max(k - int(from), 0)];
}
// A leaves-first factor in device memory four columns at a time, its rows side by side: words that neighbouring lanes read and
// write together, sixteen bytes a lane.  (Rows one after the other, packed, are 64 words of 64 different lines a lane; with them
// and the transposed reads the mass solves were a tenth of the solve of 8192 ropes.)  It takes no more words than the
// packed rows, whose room a caller gives: a quad's last two rows hold one entry between them, which goes behind all of them
// with four zeros that the lanes past a quad's rows read.
__host__ __device__ constexpr uint32_t quads_before(uint32_t q) { return 8u * q * q; }   // 4 q + 2 rows of four words a quad
template <int N>
__device__ __forceinline__ void store_quads(float* a, uint32_t lane, const float (&row)[N]) {
    static_assert(quads_before(N / 4) + 4u + N / 4 <= FactorFloats(N), "no more than the packed rows");
    lane = local_lane(lane);
    float last = 0.0f;   // of a quad's third row, its entry
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const float4 words{row[4 * q], row[4 * q + 1], row[4 * q + 2], row[4 * q + 3]};
        if (lane <= 4u * uint32_t(q) + 1u) reinterpret_cast<float4*>(a + quads_before(uint32_t(q)))[lane] = words;
        last = lane == 4u * uint32_t(q) + 2u ? words.w : last;
    }
    float* behind = a + quads_before(uint32_t(N / 4));
    if (lane < 4u) behind[lane] = 0.0f;
    if ((lane & 3u) == 2u && lane < uint32_t(N)) behind[4u + lane / 4u] = last;
}
template <int N>
__device__ __forceinline__ void load_quads(const float* a, uint32_t lane, float (&row)[N]) {
    lane = local_lane(lane);
    const float last = a[quads_before(uint32_t(N / 4)) + 4u + min(lane, uint32_t(N - 1)) / 4u];
    const float4* words = reinterpret_cast<const float4*>(a);
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const float4 w = words[lane <= 4u * uint32_t(q) + 1u ? quads_before(uint32_t(q)) / 4u + lane : quads_before(uint32_t(N / 4)) / 4u];
        row[4 * q] = w.x; row[4 * q + 1] = w.y; row[4 * q + 2] = w.z;
        row[4 * q + 3] = lane == 4u * uint32_t(q) + 2u ? last : w.w;
    }
}
template <int N>
__device__ __forceinline__ void load_columns(const float* a, uint32_t lane, float (&col)[N]) {
    lane = local_lane(lane);
    const uint32_t from = lane < uint32_t(N) ? lane : uint32_t(N - 1);
#pragma unroll
    for (int j = 0; j < N; ++j) col[j] = a[uint32_t(j) * uint32_t(N) + from];
}

// Cholesky of the Newton Hessian held in `hrow`, then d = H^-1 g.  The factor passes through LDS once, for the
// transposed read of the backward substitution.
template <int N, bool kFollow>
__device__ __forceinline__ bool cholesky_solve(const Tile& c, float (&hrow)[N], float g, float* d_out) {
    float inverse = 0.0f;
    if constexpr (kPaired) {
        if (!factor_rows_up<N>(c.lane, hrow, &inverse, &c.factor_root)) return false;
        if (c.factor_current) inverse = 1.0f / c.factor_root;   // the Hessian is the one factored last: as a kept factor answers
        c.factor_current = true;
        *d_out = substitute_by_turns<N>(c.lane, hrow, c.vec, inverse, c.lane < c.n ? g : 0.0f);
        lds_sync<N>();
        return true;
    }
    if (!c.factor_current) {   // otherwise the Hessian is the one factored last: its factor is still in hfac
        PROF_BEGIN(c, 14);
        const bool valid = kLeavesFirst<N> ? factor_rows_up<N>(c.lane, hrow, &inverse, &c.factor_root) : factor_rows<N>(c.lane, hrow, &inverse, &c.factor_root);
        PROF_END(c, 14);
        if (!valid) return false;
        PROF_BEGIN(c, 24);
        store_rows<N>(c.hfac, c.lane, hrow);
        lds_sync<N>();
        PROF_END(c, 24);
        c.factor_current = true;
    } else {
        PROF_COUNT(c, 3);
        // the rows come back from hfac; the reciprocal of the diagonal is its quotient
        inverse = 1.0f / c.factor_root;
        load_rows<N>(c.hfac, c.lane, hrow);
    }
    PROF_BEGIN(c, 15);
    if constexpr (kLeavesFirst<N>) {
        *d_out = substitute_up<N>(c.lane, hrow, c.hfac, inverse, c.lane < c.n ? g : 0.0f);
    } else {
        float col[N];
        load_columns<N>(c.hfac, c.lane, col);
        *d_out = substitute<N>(hrow, col, inverse, c.lane < c.n ? g : 0.0f);
    }
    lds_sync<N>();
    PROF_END(c, 15);
    return true;
}

// SolveTileMass (:1898-1931).  The mass matrix does not change during a solve, so its factor (same arithmetic as the
// reference's per-call factorisation, hence the same numbers) is built once by factor_mass and reused here.
template <int N, bool kFollow>
__device__ __forceinline__ bool factor_mass(Tile& c, const float (&mrow)[N]) {
    float row[N];
#pragma unroll
    for (int k = 0; k < N; ++k) row[k] = mrow[k];
    float inverse = 0.0f, root = 0.0f;
    const bool valid = kLeavesFirst<N> ? factor_rows_up<N>(c.lane, row, &inverse, &root) : factor_rows<N>(c.lane, row, &inverse, &root);
    c.mass_inverse = inverse;
    if constexpr (kPaired) store_quads<N>(c.mfac, c.lane, row);
    else store_rows<N>(c.mfac, c.lane, row);
    lds_sync<N>();
    return valid;
}
template <int N>
__device__ __forceinline__ float solve_tile_mass(const Tile& c, float force) {
    float row[N];
    if constexpr (kPaired) {
        load_quads<N>(c.mfac, c.lane, row);
        return substitute_by_turns<N>(c.lane, row, c.vec, c.mass_inverse, c.lane < c.n ? force : 0.0f);
    }
    load_rows<N>(c.mfac, c.lane, row);
    if constexpr (kLeavesFirst<N>) return substitute_up<N>(c.lane, row, c.mfac, c.mass_inverse, c.lane < c.n ? force : 0.0f);
    float col[N];
    load_columns<N>(c.mfac, c.lane, col);
    return substitute<N>(row, col, c.mass_inverse, c.lane < c.n ? force : 0.0f);
}

// Columns 4 q .. 4 q + 3 of a head's Hessian term in lane's row, on the matrix cores: v_mfma_f32_4x4x1 multiplies, in each
// of the wavefront's sixteen blocks of four lanes, four values a block with one a lane, so with the Jacobian row's words
// 4 q + (lane & 3) on the one side and the lane's entry of C J on the other, register r of a lane comes out as the
// term's entry (lane's row, 4 q + r) - the register rows' own layout, whatever head each block of lanes is at.  An axis an
// instruction, each the fused multiply-add it would be on the vector unit (bit for bit), then one sum into the row.  A
// head's words come in one round trip of fifteen four-byte reads; written as vector code the columns took four times
// the arithmetic and a wait for three sixteen-byte reads each (12 heads of 20 columns: 5.7 k cycles a Newton step).
template <int N>
__device__ __forceinline__ void add_columns(int q, float x0, float x1, float x2, float a0, float a1, float a2, float (&hrow)[N]) {
    Vec4 term = {};
    term = __builtin_amdgcn_mfma_f32_4x4x1f32(x0, a0, term, 0, 0, 0);
    term = __builtin_amdgcn_mfma_f32_4x4x1f32(x1, a1, term, 0, 0, 0);
    term = __builtin_amdgcn_mfma_f32_4x4x1f32(x2, a2, term, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) hrow[4 * q + r] += term[r];
}
template <int N>
__device__ __forceinline__ void add_columns(int q, const float* rows, float a0, float a1, float a2, float (&hrow)[N]) {
    const float* x = rows + 4 * q;
    add_columns<N>(q, x[0], x[N], x[2 * N], a0, a1, a2, hrow);
}
// the same for a head on one axis, straight into the row
template <int N>
__device__ __forceinline__ void add_columns_single(int q, float x0, float a0, float (&hrow)[N]) {
    Vec4 term = {hrow[4 * q], hrow[4 * q + 1], hrow[4 * q + 2], hrow[4 * q + 3]};
    term = __builtin_amdgcn_mfma_f32_4x4x1f32(x0, a0, term, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) hrow[4 * q + r] = term[r];
}
// The column groups a head adds to without a test, their reads in flight together: all of them up to twenty coordinates, the
// first half of a wider block, where a floating root and what stands on the ground come first (the half a reduced block
// keeps).  Past them a head that reaches no further leaves with one test, another tests group by group.  With 36
// coordinates, of which the contacts reach 20: 1000 driven humanoids 1.57 ms a step, 1.74 with a test for every group, 1.62
// with all nine taken; 4096, 2.08, 2.17 and 2.09 ms.
template <int N>
constexpr int kFirstColumns = N > 20 ? (N / 2 + 3) / 4 : N / 4;

// One head's part of the block: g += J^T f and H += J^T C J for lane's row, skipping the column groups past the first
// ones that the head's Jacobian rows leave at exact zero.  All head values are uniform.
template <int N>
__device__ __forceinline__ void add_head(const Tile& c, uint32_t h, bool coordinate, const float (&f)[3], const float (&cv)[6],
                                         const float (&noise)[3], uint32_t axes, uint64_t columns, float (&hrow)[N], TileSum& g,
                                         float& scale) {
    const float* j0r = c.jac + c.U(hRow, h) * uint32_t(N);
    const float* words = j0r + (c.lane & 3u);
    // (the lane's words read whether or not it is a coordinate: a read under a condition compiles to a branch a word)
    const uint32_t column = c.lane < uint32_t(N) ? c.lane : uint32_t(N - 1);
    const float w0 = j0r[column];
    const float j0 = coordinate ? w0 : 0.0f;
    tile_add_product(g, j0, f[0]);
    scale += fabsf(j0) * noise[0];
    if (axes == 1u) {
        const float a0 = j0 * cv[0];
        if constexpr (N > kTwoWaveWidth) {
            const float4* r0 = reinterpret_cast<const float4*>(j0r);
#pragma unroll
            for (int q = 0; q < N / 4; ++q) {
                if (((columns >> (4 * q)) & 0xFull) == 0ull) continue;
                const float4 x0 = r0[q];
                hrow[4 * q] = fmaf(a0, x0.x, hrow[4 * q]); hrow[4 * q + 1] = fmaf(a0, x0.y, hrow[4 * q + 1]);
                hrow[4 * q + 2] = fmaf(a0, x0.z, hrow[4 * q + 2]); hrow[4 * q + 3] = fmaf(a0, x0.w, hrow[4 * q + 3]);
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < kFirstColumns<N>; ++q) add_columns_single<N>(q, words[4 * q], a0, hrow);
        if ((columns >> (4 * kFirstColumns<N>)) == 0ull) return;
#pragma unroll
        for (int q = kFirstColumns<N>; q < N / 4; ++q)
            if (((columns >> (4 * q)) & 0xFull) != 0ull) add_columns_single<N>(q, words[4 * q], a0, hrow);
        return;
    }
    const float w1 = j0r[N + column], w2 = j0r[2 * N + column];
    const float j1 = coordinate ? w1 : 0.0f, j2 = coordinate ? w2 : 0.0f;
    const float cxx = cv[0], cyy = cv[1], czz = cv[2], cxy = cv[3], cxz = cv[4], cyz = cv[5];
    tile_add_product(g, j1, f[1]);
    tile_add_product(g, j2, f[2]);
    scale += fabsf(j1) * noise[1] + fabsf(j2) * noise[2];
    const float a0 = (j0 * cxx + j1 * cxy) + j2 * cxz;
    const float a1 = (j1 * cyy + j2 * cyz) + j0 * cxy;
    const float a2 = (j2 * czz + j1 * cyz) + j0 * cxz;
    if constexpr (N > kTwoWaveWidth) {   // with the whole register file in use, the terms' registers would spill
        const float4* r0 = reinterpret_cast<const float4*>(j0r);
        const float4* r1 = reinterpret_cast<const float4*>(j0r + N);
        const float4* r2 = reinterpret_cast<const float4*>(j0r + 2 * N);
#pragma unroll
        for (int q = 0; q < N / 4; ++q) {
            if (((columns >> (4 * q)) & 0xFull) == 0ull) continue;
            const float4 x0 = r0[q], x1 = r1[q], x2 = r2[q];
            hrow[4 * q] += fmaf(a2, x2.x, fmaf(a1, x1.x, a0 * x0.x));
            hrow[4 * q + 1] += fmaf(a2, x2.y, fmaf(a1, x1.y, a0 * x0.y));
            hrow[4 * q + 2] += fmaf(a2, x2.z, fmaf(a1, x1.z, a0 * x0.z));
            hrow[4 * q + 3] += fmaf(a2, x2.w, fmaf(a1, x1.w, a0 * x0.w));
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < kFirstColumns<N>; ++q) add_columns<N>(q, words, a0, a1, a2, hrow);
    if ((columns >> (4 * kFirstColumns<N>)) == 0ull) return;
#pragma unroll
    for (int q = kFirstColumns<N>; q < N / 4; ++q)
        if (((columns >> (4 * q)) & 0xFull) != 0ull) add_columns<N>(q, words, a0, a1, a2, hrow);
}

// The heads' curvature on the matrix cores, for blocks of at most 32 coordinates and those of 36 whose heads reach no further
// than 32 (Tile::near_heads: a robot on two feet, whose arms come last): H += sum over heads and axes of
// (C J)_r^T J_r, four heads a pass.  The wavefront's four groups of sixteen lanes take a head each; a lane holds, for
// its head, the three entries of a coordinate of every sixteen (column = lane & 15 of tile t), forms the entries of C J
// from them and hands both to v_mfma_f32_16x16x4, whose four products of one instruction are the four heads.  Three
// instructions (the axes) a tile and pass, T x T tiles.  The same loads give the heads' part of the force and its
// rounding scale, in double, a partial sum a group.
//   The block's rows need the tiles as lane = row, a register a column.  Tile (J, I) holds H[16 J + 4 g + r][16 I + x] in
// register r of lane 16 g + x; H is symmetric, so that is entry 16 J + 4 g + r of row 16 I + x, and one exchange of lane
// rows between tiles (J, 0) and (J, 1) (v_permlane16_swap) puts rows 0-15 and 16-31 side by side: g = 0 and 1 in the
// lower half of the wavefront, g = 2 and 3 in the upper, which v_permlane32_swap brings down.
//   The rows the heads add to - the mass matrix - come after the sums over the heads, except beside unit heads, whose
// worlds are actuated robots: there the tiles start from them, in the order of the loop this replaces.  A walker's steps
// (contact edges on one axis beside joint rows) ended 2.6 % further from a double-precision solve with the mass matrix
// last (196608 environments, the spread 0.3 %) and end as near as that loop's with it first, for 0.6 % of their time (4096:
// 734 -> 739 us).  The worlds without joint rows are as near either way: 0.999 to 1.007 of the loop's error, spreads
// of 0.1 % (quadrupeds) and 1.2 % (boxes).
//   Bound by the latency of one wave (LDS words of a pass, then the matrix instructions in line).  It takes the place of
// a loop that added heads to register rows by broadcast reads of their Jacobian words, a head a pass with unit heads present
// and two to four without: 1000 servo-driven quadrupeds, four steps, 2.58 -> 2.23 ms; 4096 walkers 1.06 -> 1.01 ms.
template <int N>
constexpr int kTileSpan = N > 32 ? 2 : (N + 15) / 16;   // tiles of sixteen coordinates a side
__device__ __forceinline__ float lane_permute(int source, float v) {   // v of lane `source`, a byte address (4 x lane)
    return __int_as_float(__builtin_amdgcn_ds_bpermute(source, __float_as_int(v)));
}
// rows of sixteen lanes: {a0, b0, a2, b2} in a and {a1, b1, a3, b3} in b
__device__ __forceinline__ void swap_lane_rows(float& a, float& b) {
    const auto pair = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(pair[0]); b = __uint_as_float(pair[1]);
}
__device__ __forceinline__ void swap_lane_rows(double& a, double& b) {
    const uint64_t x = uint64_t(__double_as_longlong(a)), y = uint64_t(__double_as_longlong(b));
    const auto low = __builtin_amdgcn_permlane16_swap(uint32_t(x), uint32_t(y), false, false);
    const auto high = __builtin_amdgcn_permlane16_swap(uint32_t(x >> 32u), uint32_t(y >> 32u), false, false);
    a = __longlong_as_double((long long)((uint64_t(high[0]) << 32u) | uint64_t(low[0])));
    b = __longlong_as_double((long long)((uint64_t(high[1]) << 32u) | uint64_t(low[1])));
}
// v[32 + (lane & 31)] in every lane
__device__ __forceinline__ float upper_half(float v) {
    return __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false)[1]);
}
// v[lane & 31] below lane 32, w[lane & 31] from there on
__device__ __forceinline__ float halves_beside(float v, float w) {
    return __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(w), false, false)[0]);
}
// v[lane & 31] + v[32 + (lane & 31)] in every lane: the two halves of the wavefront swapped against each other
__device__ __forceinline__ float halves_sum(float v) {
    const auto pair = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(pair[0]) + __uint_as_float(pair[1]);
}
__device__ __forceinline__ double halves_sum(double v) {
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    const auto low = __builtin_amdgcn_permlane32_swap(uint32_t(bits), uint32_t(bits), false, false);
    const auto high = __builtin_amdgcn_permlane32_swap(uint32_t(bits >> 32u), uint32_t(bits >> 32u), false, false);
    return __longlong_as_double((long long)((uint64_t(high[0]) << 32u) | uint64_t(low[0]))) +
           __longlong_as_double((long long)((uint64_t(high[1]) << 32u) | uint64_t(low[1])));
}
// lane = head on the way in (mf, mc, mn, my_first; `heads` the uniform mask of those to add), lane = row on return
template <int N, bool kRows>
__device__ __forceinline__ void add_heads_by_tiles(const Tile& c, uint64_t heads, const float (&mf)[3], const float (&mc)[6], const float (&mn)[3],
                                                   uint32_t my_first, float (&hrow)[N], TileSum& g, float& scale) {
    constexpr int T = kTileSpan<N>, kReach = N < 16 * T ? N : 16 * T;   // the coordinates the tiles hold
    const uint32_t group = c.lane >> 4u, x = c.lane & 15u;
    const bool reached = N <= 16 * T || c.lane < uint32_t(kReach);   // a wider block: its last rows are no tile's
    uint32_t column[T];
#pragma unroll
    for (int t = 0; t < T; ++t) column[t] = min(uint32_t(16 * t) + x, uint32_t(N - 1));   // (entries past the width are never read back)
    Vec4 tile[T][T] = {};
    if (kRows && c.units) {   // from the rows as they come, by the exchange at the end backwards; the tiles then hold them
#pragma unroll
        for (int J = 0; J < T; ++J) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const auto entry = [&](int k) { return k < kReach ? hrow[k < kReach ? k : 0] : 0.0f; };
                float low = halves_beside(entry(16 * J + r), entry(16 * J + 8 + r)), high = halves_beside(entry(16 * J + 4 + r), entry(16 * J + 12 + r));
                swap_lane_rows(low, high);
                tile[J][0][r] = low;
                if (T > 1) tile[J][T - 1][r] = high;
            }
        }
#pragma unroll
        for (int k = 0; k < kReach; ++k) hrow[k] = reached ? 0.0f : hrow[k];
    }
    double force[T] = {};
    float bound[T] = {};
    while (heads != 0ull) {
        const uint32_t first = uint32_t(__builtin_ctzll(heads));   // what a group without a head reads: its rows are staged
        uint32_t mine = kInvalid;
#pragma unroll
        for (uint32_t k = 0u; k < 4u; ++k) {
            const uint32_t h = heads != 0ull ? uint32_t(__builtin_ctzll(heads)) : kInvalid;
            heads &= heads - 1ull;   // zero stays zero
            mine = group == k ? h : mine;
        }
        const bool live = mine != kInvalid;
        const int source = int((live ? mine : first) * 4u);
        const float* rows = c.jac + uint32_t(__builtin_amdgcn_ds_bpermute(source, int(my_first))) * uint32_t(N);
        float f[3], cv[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, noise[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) { f[k] = lane_permute(source, mf[k]); noise[k] = lane_permute(source, mn[k]); }
        if constexpr (kRows) {
#pragma unroll
            for (int k = 0; k < 6; ++k) cv[k] = lane_permute(source, mc[k]);
        }
        float j[T][3], a[T][3];
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float word = rows[uint32_t(k) * uint32_t(N) + column[t]];
                j[t][k] = live ? word : 0.0f;
            }
            a[t][0] = fmaf(j[t][2], cv[4], fmaf(j[t][1], cv[3], j[t][0] * cv[0]));
            a[t][1] = fmaf(j[t][2], cv[5], fmaf(j[t][0], cv[3], j[t][1] * cv[1]));
            a[t][2] = fmaf(j[t][1], cv[5], fmaf(j[t][0], cv[4], j[t][2] * cv[2]));
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                force[t] = fma(double(j[t][k]), double(f[k]), force[t]);
                bound[t] = fmaf(fabsf(j[t][k]), noise[k], bound[t]);
            }
        }
        if constexpr (!kRows) continue;
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int J = 0; J < T; ++J)
#pragma unroll
                for (int I = 0; I < T; ++I) tile[J][I] = __builtin_amdgcn_mfma_f32_16x16x4f32(j[J][k], a[I][k], tile[J][I], 0, 0, 0);
    }
#pragma unroll
    for (int J = 0; J < (kRows ? T : 0); ++J) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (16 * J + r >= kReach) continue;
            float low = tile[J][0][r], high = tile[J][T - 1][r];
            swap_lane_rows(low, high);
            const auto add = [&](int k, float v) { if (k < kReach) hrow[k < kReach ? k : 0] += reached ? v : 0.0f; };
            add(16 * J + r, low);
            add(16 * J + 4 + r, high);
            add(16 * J + 8 + r, upper_half(low));
            add(16 * J + 12 + r, upper_half(high));
        }
    }
    double force_low = force[0], force_high = force[T - 1];
    float bound_low = bound[0], bound_high = bound[T - 1];
    swap_lane_rows(force_low, force_high); swap_lane_rows(bound_low, bound_high);
    const double force_sum = halves_sum(force_low + force_high);
    const float bound_sum = halves_sum(bound_low + bound_high);
    g.value += reached ? force_sum : 0.0;
    scale += reached ? bound_sum : 0.0f;
}

// The same as add_head for the heads of `heads` (a uniform mask of the first 64), in head order, where all of them have three
// axes and reach no further than the first columns (Tile::block_heads): nothing is asked of a head, and the next one's words
// are on their way while this one's are worked on.  About half of add_head's instructions, which with its three waits made
// 1.1 k cycles a head: 1000 servo-driven humanoids 1262 -> 1210 us a step, 4096 1432 -> 1409.
template <int N>
__device__ __forceinline__ void add_block_heads(const Tile& c, uint64_t heads, bool coordinate, const float (&mf)[3], const float (&mc)[6], const float (&mn)[3],
                                                uint32_t my_first, float (&hrow)[N], TileSum& g, float& scale) {
    constexpr int kFirst = kFirstColumns<N>;
    const uint32_t column = min(c.lane, uint32_t(N - 1));
    struct Words { float own[3], x[kFirst][3]; };
    auto fetch = [&](uint32_t h) {
        const float* rows = c.jac + uint32_t(__builtin_amdgcn_readlane(int(my_first), int(h))) * uint32_t(N);
        Words w;
#pragma unroll
        for (int k = 0; k < 3; ++k) w.own[k] = rows[uint32_t(k * N) + column];
#pragma unroll
        for (int q = 0; q < kFirst; ++q)
#pragma unroll
            for (int k = 0; k < 3; ++k) w.x[q][k] = rows[uint32_t(k * N + 4 * q) + (c.lane & 3u)];
        return w;
    };
    // (widened once: a lane's two words are read for a conversion a head, which takes four times an instruction's time)
    const double wide[3] = {double(mf[0]), double(mf[1]), double(mf[2])};
    auto force_of = [&](int k, uint32_t h) {
        const uint64_t bits = uint64_t(__double_as_longlong(wide[k]));
        const uint32_t low = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(bits)), int(h))), high = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(bits >> 32u)), int(h)));
        return __longlong_as_double((long long)((uint64_t(high) << 32u) | uint64_t(low)));
    };
    auto value_of = [&](float v, uint32_t h) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), int(h))); };
    uint32_t h = uint32_t(__builtin_ctzll(heads));
    // (two sets of words in turn: with one the compiler moves the reads of both places to where they meet, ahead of their use)
    Words even = fetch(h), odd;
    auto add = [&](const Words& w, Words& next) {   // true after the last head
        heads &= heads - 1ull;
        const uint32_t after = heads != 0ull ? uint32_t(__builtin_ctzll(heads)) : h;
        next = fetch(after);
        __builtin_amdgcn_sched_barrier(0);
        float j[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            j[k] = coordinate ? w.own[k] : 0.0f;
            g.value = fma(double(j[k]), force_of(k, h), g.value);
        }
        scale += fabsf(j[0]) * value_of(mn[0], h);
        scale += fabsf(j[1]) * value_of(mn[1], h) + fabsf(j[2]) * value_of(mn[2], h);
        const float cxx = value_of(mc[0], h), cyy = value_of(mc[1], h), czz = value_of(mc[2], h), cxy = value_of(mc[3], h), cxz = value_of(mc[4], h), cyz = value_of(mc[5], h);
        const float a0 = (j[0] * cxx + j[1] * cxy) + j[2] * cxz;
        const float a1 = (j[1] * cyy + j[2] * cyz) + j[0] * cxy;
        const float a2 = (j[2] * czz + j[1] * cyz) + j[0] * cxz;
#pragma unroll
        for (int q = 0; q < kFirst; ++q) add_columns<N>(q, w.x[q][0], w.x[q][1], w.x[q][2], a0, a1, a2, hrow);
        h = after;
        return heads == 0ull;
    };
#pragma unroll 1
    while (!add(even, odd) && !add(odd, even)) {}
}

// A reduced block of plain contacts adds its heads to register rows instead, in an order of its own (below): its worlds are robots on two
// many-sphered feet, of which some do not converge within their sweeps, and an environment that has not converged hands
// a last place of its Hessian on as the fourth decimal of its velocities.
// Heads a pass: as many copies of the block's rows as fit the wavefront, kGroups<N> of them, a group of lanes kGroupLanes
// wide each - or two where that takes as few passes, or the one that contributes.  The contributing heads are listed a lane
// each once; in a pass the lanes of group k add the k-th head of the pass's to rows of their own, which start at zero past the
// first group; a head's values come from its own lane (lane = head) through the lane permute.  The groups' rows are added
// together at the end, in group order, through LDS (hrows and hfac, which a changed Hessian frees), and stay in hrows.  With
// kRows false only the force and its scale are taken: the Hessian of the last assembly stands.
//   Bound by the LDS trips of one wave, so a pass's words are asked for a pass ahead; a kernel of three waves a SIMD has no
// registers for that, and its other waves fill the wait.  A pass of three heads took 1.25 k cycles while it found its heads
// by scalar code, asked for the first row, the values and the words one behind the other and handed the rows over in two
// exchanges: 333 humanoids 536 -> 510 us, 4096 722 -> 708, 65536 7630 -> 7500, the bits the same.
template <int N>
constexpr int kGroups = N <= 16 ? 4 : (N <= 20 ? 3 : 2);
template <int N>
constexpr uint32_t kGroupLanes = kGroups<N> == 2 ? 32u : uint32_t(N);
template <int N>
__device__ __forceinline__ float groups_sum(uint32_t lane, float v) {
    float total = v;
#pragma unroll
    for (int k = 1; k < kGroups<N>; ++k) total += __shfl(v, int(lane + uint32_t(k) * kGroupLanes<N>), kWave);
    return total;
}
template <int N>
__device__ __forceinline__ double groups_sum(uint32_t lane, double v) {
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    double total = v;
#pragma unroll
    for (int k = 1; k < kGroups<N>; ++k) {
        const int from = int(lane + uint32_t(k) * kGroupLanes<N>);
        const uint32_t low = uint32_t(__shfl(int(uint32_t(bits)), from, kWave));
        const uint32_t high = uint32_t(__shfl(int(uint32_t(bits >> 32u)), from, kWave));
        total += __longlong_as_double((long long)((uint64_t(high) << 32u) | uint64_t(low)));
    }
    return total;
}
template <int N, bool kRows>
__device__ __forceinline__ void add_heads_by_groups(const Tile& c, uint64_t heads, const float (&mf)[3], const float (&mc)[6], const float (&mn)[3],
                                                    uint32_t my_first, float (&hrow)[N], TileSum& g, float& scale) {
    static_assert(N <= 32, "two copies of the rows fit the wavefront");
    constexpr int G = kGroups<N>;
    const uint32_t lane = c.lane, group = lane / kGroupLanes<N>, row = lane - group * kGroupLanes<N>;
    const uint32_t contributing = uint32_t(__popcll(heads));
    const uint32_t taken_a_pass = contributing == 1u ? 1u : ((contributing + G - 1u) / G < (contributing + 1u) / 2u ? G : 2u);
    const bool single = contributing == 1u && c.U(hAxes, uint32_t(__builtin_ctzll(heads))) == 1u;
    const uint32_t column = min(row, uint32_t(N - 1));
    // the contributing heads in order, one a lane from lane 0 on, each with its first row
    const uint32_t below = __builtin_amdgcn_mbcnt_hi(uint32_t(heads >> 32u), __builtin_amdgcn_mbcnt_lo(uint32_t(heads), 0u));
    const uint32_t place = ((heads >> lane) & 1ull) != 0ull ? below : contributing + (lane - below);
    const int listed = __builtin_amdgcn_ds_permute(int(4u * place), int((my_first << 8u) | lane));
    if (group != 0u) {
        if constexpr (kRows) {
#pragma unroll
            for (int k = 0; k < N; ++k) hrow[k] = 0.0f;
        }
        g.value = 0.0; scale = 0.0f;
    }
    // What a lane needs of its group's head in a pass; the next pass's words are on their way while this one's are worked on.
    // Lanes without a head read the last one's: its rows are staged, and add_columns multiplies a word of theirs by zero, which
    // must be a finite word.
    struct Words { float f[3], noise[3], cv[4], j[3]; const float* rows; bool live; };   // cv: xx yy zz yz
    const auto fetch = [&](int entry, uint32_t rank) {
        Words w;
        const int source = (entry & 0xFF) * 4;
        const float* rows = c.jac + (uint32_t(entry) >> 8u) * uint32_t(N);
        w.live = group < taken_a_pass && rank < contributing && row < c.n;   // (the lanes past the last group have none)
#pragma unroll
        for (int k = 0; k < 3; ++k) w.j[k] = rows[uint32_t(k) * uint32_t(N) + column];
        if constexpr (kRows) {
#pragma unroll
            for (int k = 0; k < 3; ++k) w.cv[k] = lane_permute(source, mc[k]);
            w.cv[3] = lane_permute(source, mc[5]);
            w.rows = rows + (lane & 3u);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) { w.f[k] = lane_permute(source, mf[k]); w.noise[k] = lane_permute(source, mn[k]); }
        return w;
    };
    const auto entry_of = [&](uint32_t rank) { return __builtin_amdgcn_ds_bpermute(int(4u * min(rank, contributing - 1u)), listed); };
    const auto take = [&](const Words& w, bool alone) {
        const float j0 = w.live ? w.j[0] : 0.0f, j1 = w.live ? w.j[1] : 0.0f, j2 = w.live ? w.j[2] : 0.0f;
        if constexpr (kRows) {
            const float a0 = j0 * w.cv[0], a1 = j1 * w.cv[1] + j2 * w.cv[3], a2 = j2 * w.cv[2] + j1 * w.cv[3];   // (no plain head couples its normal to a tangent)
            if (alone && single) {
#pragma unroll
                for (int q = 0; q < N / 4; ++q) add_columns_single<N>(q, w.rows[4 * q], a0, hrow);
            } else {
#pragma unroll
                for (int q = 0; q < N / 4; ++q) add_columns<N>(q, w.rows, a0, a1, a2, hrow);
            }
        }
        tile_add_product(g, j0, w.f[0]);
        tile_add_product(g, j1, w.f[1]);
        tile_add_product(g, j2, w.f[2]);
        scale += (fabsf(j0) * w.noise[0] + fabsf(j1) * w.noise[1]) + fabsf(j2) * w.noise[2];
    };
    uint32_t rank = group, done = 0u;
    if constexpr (WavesPerSimd(N) > 2) {
        for (; done < contributing; done += taken_a_pass, rank += taken_a_pass) take(fetch(entry_of(rank), rank), true);
        if (contributing == 1u) return;
    } else {
        if (contributing == 1u) {
            take(fetch(entry_of(rank), rank), true);
            return;
        }
        Words even = fetch(entry_of(rank), rank), odd;
        int entry = entry_of(rank + taken_a_pass);
        const auto pass = [&](const Words& here, Words& next) {   // true after the last one
            done += taken_a_pass; rank += taken_a_pass;
            if (done < contributing) {
                next = fetch(entry, rank);
                entry = entry_of(rank + taken_a_pass);
            }
            take(here, false);
            return done >= contributing;
        };
        while (!pass(even, odd) && !pass(odd, even)) {}
    }
    g.value = groups_sum<N>(lane, g.value); scale = groups_sum<N>(lane, scale);
    if constexpr (kRows) {
        // the second group's rows by way of hrows, the third's by way of hfac, a fourth's behind them; what the lanes
        // past the first group add to theirs is read by nobody
        constexpr int kRound = 2;   // groups an exchange
#pragma unroll
        for (int k = 1; k < G; k += kRound) {
            if (group - uint32_t(k) < uint32_t(kRound) && group < uint32_t(G) && row < uint32_t(N)) {
                float4* to = reinterpret_cast<float4*>((group == uint32_t(k) ? c.hrows : c.hfac) + row * uint32_t(N));
#pragma unroll
                for (int q = 0; q < N / 4; ++q) to[q] = float4{hrow[4 * q], hrow[4 * q + 1], hrow[4 * q + 2], hrow[4 * q + 3]};
            }
            lds_sync<N>();
#pragma unroll
            for (int other = k; other < k + kRound && other < G; ++other) {
                const float4* from = reinterpret_cast<const float4*>((other == k ? c.hrows : c.hfac) + column * uint32_t(N));
#pragma unroll
                for (int q = 0; q < N / 4; ++q) {
                    const float4 w = from[q];
                    const bool adds = G <= kRound + 1 || group == 0u;   // (a group that is still to hand its rows over keeps them)
                    hrow[4 * q] += adds ? w.x : 0.0f; hrow[4 * q + 1] += adds ? w.y : 0.0f;
                    hrow[4 * q + 2] += adds ? w.z : 0.0f; hrow[4 * q + 3] += adds ? w.w : 0.0f;
                }
            }
            lds_sync<N>();
        }
    }
}

// One head's line-search inputs in registers: nothing in them changes between the probes of one search, and neither
// do the parts of its response that do not depend on the probe (plain_line).
struct HeadLine {
    uint32_t head;
    bool owned, contact, bounded, cone, elliptic;
    EllipticLine on_cone;   // of an elliptic head
    float rho, compliance, lower, upper, bound;
    Response response;
    TangentRatios ratios;
    float dual[3], res[3], move[3], step[3];
    float dual_part, radius, rho_radius, radius_y, radius_z, inside_yy, inside_zz;
    ConeAxis y, z;
};
__device__ __forceinline__ HeadLine load_head_line(const Tile& c, uint32_t h) {
    HeadLine l{};
    l.head = h;
    l.owned = h < c.heads && c.owned(h);
    if (!l.owned) return l;
    l.contact = block_axes(c.U(hAxes, h));
    l.elliptic = c.elliptic && c.U(hAxes, h) == kAxesElliptic;
    if (l.elliptic) l.on_cone = elliptic_line(cone_of(c, h), V3{c.F(hDual, h), c.F(hDual + 1, h), c.F(hDual + 2, h)});
    l.rho = c.F(hRho, h); l.compliance = c.F(hCompliance, h); l.lower = c.F(hLower, h); l.upper = c.F(hUpper, h);
    l.bound = c.F(hNormalBound, h);
    l.response = Response{c.F(hDualScale, h), c.F(hResidualScale, h)};
    l.ratios = tangent_ratios(c.F(hMu1, h), c.F(hMu2, h));
#pragma unroll
    for (int k = 0; k < 3; ++k) { l.dual[k] = c.F(hDual + k, h); l.res[k] = c.F(hRes + k, h); l.move[k] = c.F(hMove + k, h); l.step[k] = c.F(hStep + k, h); }
    l.bounded = l.lower < l.upper;
    l.dual_part = l.response.dual_scale * l.dual[0];
    if (l.contact) {
        l.radius = (l.bound < 0.0f ? 0.0f : l.bound) * fmaxf(l.ratios.scale, 0.0f);
        l.cone = l.radius != 0.0f;
        l.y = cone_axis(l.dual[1], l.rho, l.ratios.mu_y);
        l.z = cone_axis(l.dual[2], l.rho, l.ratios.mu_z);
        l.rho_radius = l.rho * l.radius;
        l.radius_y = l.ratios.mu_y * l.radius; l.radius_z = l.ratios.mu_z * l.radius;
        l.inside_yy = l.rho * l.ratios.mu_y * l.ratios.mu_y; l.inside_zz = l.rho * l.ratios.mu_z * l.ratios.mu_z;
    }
    return l;
}

// What the rounding of a head's residual and trial move does to its term of the slope: the impulse is curvature times
// (residual - move) plus a constant, so each of the two carries its own ulp into the impulse at the rate of the
// curvature - the noise the reference's block assembly allows its forces (AssembleTileBlock :1568-1572: impulse plus
// curvature times (|residual| + |move|)).  The reference's line search measures its slopes against the impulses alone
// (:2075-2083): where a stiff row nearly cancels its residual the slope then moves in steps many times the tolerance, no
// point of the line meets it, and the search halves its bracket down to one ulp, some twenty probes for nothing.
// Here the tolerance sees that noise; the accepted step differs from the reference's below the slope's own rounding.
__device__ __forceinline__ float line_noise(const float (&r)[6], float rx, float ry, float rz, float mx, float my, float mz, float sx, float sy, float sz) {
    return r[0] * (fabsf(rx) + fabsf(mx)) * fabsf(sx) + r[1] * (fabsf(ry) + fabsf(my)) * fabsf(sy) + r[2] * (fabsf(rz) + fabsf(mz)) * fabsf(sz);
}
__device__ __forceinline__ void add_line_terms(const float (&f)[3], const float (&r)[6], float sx, float sy, float sz, TileSum& row_slope,
                                               float& row_curvature, float& row_magnitude) {
    tile_add_product(row_slope, f[0], sx);
    tile_add_product(row_slope, f[1], sy);
    tile_add_product(row_slope, f[2], sz);
    row_magnitude += fabsf(f[0] * sx) + fabsf(f[1] * sy) + fabsf(f[2] * sz);
    row_curvature += r[0] * sx * sx + r[1] * sy * sy + r[2] * sz * sz + 2.0f * r[5] * sy * sz + 2.0f * r[3] * sx * sy +
                     2.0f * r[4] * sx * sz;
}
// TileLineDerivatives (:2048-2086); lane = head, heads beyond the first 64 go through `extra`
__device__ __forceinline__ void line_terms(const HeadLine& l, float alpha, TileSum& row_slope, float& row_curvature, float& row_magnitude) {
    const float sx = l.step[0], sy = l.step[1], sz = l.step[2];
    float f[3] = {0.0f, 0.0f, 0.0f}, r[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (l.elliptic) {
        elliptic_impulse(l.on_cone, l.res[0] - fmaf(alpha, sx, l.move[0]), l.res[1] - fmaf(alpha, sy, l.move[1]), l.res[2] - fmaf(alpha, sz, l.move[2]), f, r);
        add_line_terms(f, r, sx, sy, sz, row_slope, row_curvature, row_magnitude);
        row_magnitude += line_noise(r, l.res[0], l.res[1], l.res[2], fmaf(alpha, sx, l.move[0]), fmaf(alpha, sy, l.move[1]), fmaf(alpha, sz, l.move[2]), sx, sy, sz);
        return;
    }
    scalar_impulse(l.dual[0], l.rho, l.res[0] - fmaf(alpha, sx, l.move[0]), l.compliance, l.lower, l.upper, l.response, &f[0], &r[0]);
    if (l.contact)
        tangent_impulse(V3{l.dual[0], l.dual[1], l.dual[2]}, l.rho, l.res[1] - fmaf(alpha, sy, l.move[1]),
                        l.res[2] - fmaf(alpha, sz, l.move[2]), l.bound, l.ratios, &f[1], &f[2], &r[1], &r[2], &r[5]);
    add_line_terms(f, r, sx, sy, sz, row_slope, row_curvature, row_magnitude);
    row_magnitude += line_noise(r, l.res[0], l.res[1], l.res[2], fmaf(alpha, sx, l.move[0]), fmaf(alpha, sy, l.move[1]), fmaf(alpha, sz, l.move[2]), sx, sy, sz);
}
// A head's line-search constants as numbers only, so that the probes run without a branch: every selection the
// response makes on a constant of the head (a single-axis head has no tangent part, a friction ratio of zero takes no
// cone argument, a cone of radius zero gives no tangent impulse and no curvature) is made here once, by handing the
// probe constants on which the general formulas give those results exactly - zeros for what must come out as zero.
// A lane without an owned head gets zeros throughout and adds exact zeros to every sum.
// The cone argument dual / mu + rho mu residual (ConeArgument, augmented_row.hpp:302-318) is kept by the reference as
// compensated float pairs; here the same two constants are doubles (the sums of the reference's pairs) and the
// argument is one double multiply-add.  Everything but `move` and `step` is constant over a block descent.
struct PlainLine {
    float k, k_bounded, dual_part, lower, upper;
    float res[3], move[3], step[3];
    double cone_y, cone_z, gain_y, gain_z;
    float mu_y, mu_z, radius, rho_radius, radius_y, radius_z, inside_yy, inside_zz;
    uint32_t head;   // the head the constants belong to, kInvalid for none: `move` and `step` are then never read
};
__device__ __forceinline__ PlainLine plain_line(const HeadLine& l) {
    PlainLine p{};
    p.head = kInvalid;
    if (!l.owned || l.rho <= 0.0f) return p;   // no penalty: no impulse and no curvature (scalar_impulse, tangent_impulse)
    p.head = l.head;
    p.k = l.response.residual_scale; p.k_bounded = l.bounded ? p.k : 0.0f; p.dual_part = l.dual_part; p.lower = l.lower; p.upper = l.upper;
#pragma unroll
    for (int k = 0; k < 3; ++k) { p.res[k] = l.res[k]; p.move[k] = l.move[k]; p.step[k] = l.step[k]; }
    // a constant that is not a number makes the general response not a number; here it is handed on through the sum
    if (!(l.rho == l.rho && l.dual[0] == l.dual[0] && l.compliance == l.compliance && l.lower == l.lower && l.upper == l.upper)) p.dual_part = nanf("");
    if (!l.contact) return p;
    p.mu_y = l.ratios.mu_y; p.mu_z = l.ratios.mu_z;
    if (p.mu_y != 0.0f) { p.cone_y = double(l.y.dd) + double(l.y.d_low); p.gain_y = double(l.y.p) + double(l.y.p_low); }
    if (p.mu_z != 0.0f) { p.cone_z = double(l.z.dd) + double(l.z.d_low); p.gain_z = double(l.z.p) + double(l.z.p_low); }
    p.radius = l.radius; p.rho_radius = l.rho_radius; p.radius_y = l.radius_y; p.radius_z = l.radius_z;
    if (l.cone) { p.inside_yy = l.inside_yy; p.inside_zz = l.inside_zz; }
    return p;
}
// The response of a head from its constants: scalar_impulse and tangent_impulse operation for operation, both sides
// of the cone computed and one selected, the three quotients by the tangent norm sharing one reciprocal (the answers
// differ from the general functions' in the last place or two).  A residual
// that is not a number comes out as an impulse that is not a number, as in the general functions.  plain_line_terms
// is TileLineDerivatives (:2048-2086) on it, with at most one head a lane.
__device__ __forceinline__ void plain_response(const PlainLine& p, float mx, float my, float mz, float (&f)[3], float (&r)[6]) {
    const float x = fmaf(p.k, p.res[0] - mx, p.dual_part);
    f[0] = x < p.lower ? p.lower : (x > p.upper ? p.upper : x);
    r[0] = x >= p.lower && x <= p.upper ? p.k_bounded : 0.0f;
    const float q_y = float(fma(p.gain_y, double(p.res[1] - my), p.cone_y));
    const float q_z = float(fma(p.gain_z, double(p.res[2] - mz), p.cone_z));
    // the norm and its reciprocal by the hardware root and reciprocal (an ulp each): impulses lie far inside the range
    // where the squares neither overflow nor vanish
    const float norm = __builtin_amdgcn_sqrtf(fmaf(q_y, q_y, q_z * q_z));
    const bool inside = norm <= p.radius;
    const float by_norm = __builtin_amdgcn_rcpf(inside ? 1.0f : norm);
    const float dy = q_y * by_norm, dz = q_z * by_norm, cs = p.rho_radius * by_norm;
    f[1] = inside ? p.mu_y * q_y : p.radius_y * dy;
    f[2] = inside ? p.mu_z * q_z : p.radius_z * dz;
    r[1] = inside ? p.inside_yy : cs * p.mu_y * p.mu_y * dz * dz;
    r[2] = inside ? p.inside_zz : cs * p.mu_z * p.mu_z * dy * dy;
    r[3] = 0.0f; r[4] = 0.0f;
    r[5] = inside ? 0.0f : -cs * p.mu_y * p.mu_z * dy * dz;
}
// A head on one axis as numbers: what of a PlainLine such a head has.  Lanes keep their later heads (the second and third
// sixty-four) so where all of those are on one axis, as joint rows are: a probe of 97 heads 3.7 k cycles with the later
// ones' fields read and their general response taken each time, and a step of 4096 servo-driven humanoids, whose longest
// environment makes 340 probes, 2002 -> 1832 us with it and with the row steps below (row_steps).
struct ScalarLine { float k, k_bounded, dual_part, lower, upper, res, move, step; };
constexpr uint32_t kLaterHeads = 2u;   // a lane
__device__ __forceinline__ ScalarLine scalar_line(const Tile& c, uint32_t h) {
    const uint32_t at = min(h, c.heads - 1u);   // (read whether or not there is such a head)
    const float rho = c.F(hRho, at), dual = c.F(hDual, at), compliance = c.F(hCompliance, at), lower = c.F(hLower, at), upper = c.F(hUpper, at);
    const float k = c.F(hResidualScale, at), scaled = c.F(hDualScale, at) * dual, res = c.F(hRes, at), move = c.F(hMove, at), step = c.F(hStep, at);
    const bool live = h < c.heads && c.owned(at) && !(rho <= 0.0f);
    ScalarLine s{};
    s.k = live ? k : 0.0f; s.k_bounded = live && lower < upper ? k : 0.0f;
    s.dual_part = live ? scaled : 0.0f; s.lower = live ? lower : 0.0f; s.upper = live ? upper : 0.0f;
    s.res = live ? res : 0.0f; s.move = live ? move : 0.0f; s.step = live ? step : 0.0f;
    if (live && !(rho == rho && dual == dual && compliance == compliance && lower == lower && upper == upper)) s.dual_part = nanf("");
    return s;
}
__device__ __forceinline__ void scalar_line_response(const ScalarLine& s, float move, float* f, float* r) {
    const float x = fmaf(s.k, s.res - move, s.dual_part);
    *f = x < s.lower ? s.lower : (x > s.upper ? s.upper : x);
    *r = x >= s.lower && x <= s.upper ? s.k_bounded : 0.0f;
}
// The constants of lane's own head for one block descent.  With at most sixteen heads the four rows of sixteen lanes
// hold copies of the heads (lane & 15), which the line search uses to evaluate several points of a line in one pass;
// the block assembly then takes the copies of the first row only.  `move` and `step` change with every Newton step
// and are read again where they are used.
// The constants stay in registers over the whole block descent (while the factor's panels went through registers of their
// own, widths of 28 to 36 had no room for them and computed them again at each use).
__device__ __forceinline__ PlainLine own_line(const Tile& c) {
    return plain_line(load_head_line(c, c.heads <= 16u ? (c.lane & 15u) : c.lane));
}
// (read whether or not the lane has a head, from the first one's place then, and taken as zero: a read under a condition
// compiles to a branch)
__device__ __forceinline__ void refresh_moves(const Tile& c, PlainLine& p) {
    const bool live = p.head != kInvalid;
    const uint32_t h = live ? p.head : 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) { const float move = c.F(hMove + k, h); p.move[k] = live ? move : 0.0f; }
}
__device__ __forceinline__ void refresh_steps(const Tile& c, PlainLine& p) {
    const bool live = p.head != kInvalid;
    const uint32_t h = live ? p.head : 0u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float move = c.F(hMove + k, h), step = c.F(hStep + k, h);
        p.move[k] = live ? move : 0.0f; p.step[k] = live ? step : 0.0f;
    }
}
// A head's response at its current move with the rounding noise of each axis; false when nothing of it is non-zero.
__device__ __forceinline__ bool head_terms(const Tile& c, uint32_t h, float (&f)[3], float (&cv)[6], float (&noise)[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) { f[k] = 0.0f; noise[k] = 0.0f; }
#pragma unroll
    for (int k = 0; k < 6; ++k) cv[k] = 0.0f;
    if (h >= c.heads || !c.owned(h)) return false;
    head_response(c, h, c.F(hMove, h), c.F(hMove + 1, h), c.F(hMove + 2, h), f, cv);
#pragma unroll
    for (int k = 0; k < 3; ++k) noise[k] = fabsf(f[k]) + cv[k] * (fabsf(c.F(hRes + k, h)) + fabsf(c.F(hMove + k, h)));
    return f[0] != 0.0f || f[1] != 0.0f || f[2] != 0.0f || cv[0] != 0.0f || cv[1] != 0.0f || cv[2] != 0.0f || cv[5] != 0.0f ||
           cv[3] != 0.0f || cv[4] != 0.0f || noise[0] != 0.0f || noise[1] != 0.0f || noise[2] != 0.0f;
}

__device__ __forceinline__ float uniform_lane_value(float v, uint32_t lane) {   // `lane` is uniform, not a constant
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), int(lane)));
}

// The heads' part of the force only: g += J^T f for lane's coordinate, with the rounding scale of that sum.  A staged
// head has three rows in LDS whatever its axes (those it does not have hold zeros, as its response does), and the
// padded columns hold zeros: every head reads its three words without a condition, the next head's ahead of this
// one's arithmetic.  lane = head on the way in (mf, mn, my_first), lane = coordinate for the sums.
template <int N>
__device__ __forceinline__ void add_heads_force(const Tile& c, uint64_t heads, const float (&mf)[3], const float (&mn)[3], uint32_t my_first,
                                                TileSum& g, float& scale) {
    const uint32_t column = c.lane < uint32_t(N) ? c.lane : uint32_t(N - 1);
    auto rows_of = [&](uint32_t h, float (&j)[3]) {
        const float* at = c.jac + uint32_t(__builtin_amdgcn_readlane(int(my_first), int(h))) * uint32_t(N) + column;
        j[0] = at[0]; j[1] = at[N]; j[2] = at[2 * N];
    };
    float next[3] = {0.0f, 0.0f, 0.0f};
    if (heads != 0ull) rows_of(uint32_t(__builtin_ctzll(heads)), next);
    while (heads != 0ull) {
        const uint32_t h = uint32_t(__builtin_ctzll(heads));
        heads &= heads - 1ull;
        const float j[3] = {next[0], next[1], next[2]};
        if (heads != 0ull) rows_of(uint32_t(__builtin_ctzll(heads)), next);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            tile_add_product(g, j[k], uniform_lane_value(mf[k], h));
            scale += fabsf(j[k]) * uniform_lane_value(mn[k], h);
        }
    }
}

// Sums over runs of neighbouring lanes, as differences of the running sum over the wavefront, in double.  A running sum takes
// eighteen instructions, where the sum of every lane's own choice of 64 takes three a lane: a step of 8192 ropes 15.98 ->
// 13.64 ms with the force so (rows_transposed_times), where the heads past every coordinate are neighbours in their list
// (Tile::over_runs), and 13.64 -> 13.31 with the motion of the links (link_motion), where every way to the root is a run of
// coordinates.  The motions are rounded once where 64 single-precision multiply-adds were; how near a step ends to a
// double-precision solve is the same (12288 environments: 0.993 +- 0.011 and 1.001 +- 0.007 of the mean errors before).
template <int Ctrl, int Rows>
__device__ __forceinline__ double dpp_rows_d(double v) {   // lanes without a source, and rows outside the mask, get zero
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    const uint32_t low = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(bits)), Ctrl, Rows, 0xF, true));
    const uint32_t high = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(bits >> 32u)), Ctrl, Rows, 0xF, true));
    return __longlong_as_double((long long)((uint64_t(high) << 32u) | uint64_t(low)));
}
__device__ __forceinline__ double running_sum(double v) {
    v += dpp_rows_d<0x111, 0xF>(v); v += dpp_rows_d<0x112, 0xF>(v); v += dpp_rows_d<0x114, 0xF>(v); v += dpp_rows_d<0x118, 0xF>(v);   // within sixteen lanes
    v += dpp_rows_d<0x142, 0xA>(v);   // lane 15 of a row to the next row,
    v += dpp_rows_d<0x143, 0xC>(v);   // lane 31 to the upper two
    return v;
}
__device__ __forceinline__ bool one_run(uint64_t lanes) {
    const uint64_t from = lanes == 0ull ? 0ull : lanes >> __builtin_ctzll(lanes);
    return (from & (from + 1ull)) == 0ull;
}
struct LaneRun {   // the lanes of a mask that are one run
    bool some, from_start;
    int before, last;      // byte addresses (4 x lane) of the lane ahead of the run and of its last
    __device__ __forceinline__ LaneRun(uint32_t low, uint32_t high) {
        const uint64_t lanes = (uint64_t(high) << 32u) | uint64_t(low);
        some = lanes != 0ull;
        const uint32_t first = some ? uint32_t(__builtin_ctzll(lanes)) : 0u, end = some ? 64u - uint32_t(__builtin_clzll(lanes)) : 1u;
        from_start = first == 0u;
        before = int(4u * (from_start ? 0u : first - 1u)); last = int(4u * (end - 1u));
    }
    __device__ __forceinline__ double sum(double v) const {
        const uint64_t bits = uint64_t(__double_as_longlong(running_sum(v)));
        auto at = [&](int source) {
            const uint32_t low = uint32_t(__builtin_amdgcn_ds_bpermute(source, int(uint32_t(bits)))), high = uint32_t(__builtin_amdgcn_ds_bpermute(source, int(uint32_t(bits >> 32u))));
            return __longlong_as_double((long long)((uint64_t(high) << 32u) | uint64_t(low)));
        };
        const double through = at(last), ahead = at(before);
        return some ? (from_start ? through : through - ahead) : 0.0;
    }
};

// What lanes of coordinates and lanes of heads hand each other on the matrix cores, without a word through LDS.
// v_mfma_f32_4x4x1 takes the four lanes of block q for every block's left side (cbsz 4, abid q).  Where those four
// lanes hold one value each - the motion axes of four coordinates - their registers serve as they are.  Where a lane holds four
// values that belong side by side - four components of one head - each four lanes transpose theirs first: four products with
// unit vectors, exact.  (Through LDS, a table a use, a wait a group of columns and 4.9 KB a block: a step of 8192 ropes
// 12.49 ms, as it is 12.28, bit for bit.)
struct FourUnits {
    float one[4];   // one[k]: one in the lanes of place k among their four, else zero
    __device__ __forceinline__ explicit FourUnits(uint32_t lane) {
#pragma unroll
        for (uint32_t k = 0u; k < 4u; ++k) one[k] = (lane & 3u) == k ? 1.0f : 0.0f;
    }
    // entry t of a lane of place k: v[k] of its four's lane of place t
    __device__ __forceinline__ Vec4 transposed(const float (&v)[4]) const {
        Vec4 out = {};
#pragma unroll
        for (uint32_t k = 0u; k < 4u; ++k) out = __builtin_amdgcn_mfma_f32_4x4x1f32(v[k], one[k], out, 0, 0, 0);
        return out;
    }
};
// Blocks that keep no contact rows (Tile::from_links).  Entry j of a head's row is s_j . w where j lies on the head's
// way to the root, s_j the coordinate's motion axis (Tile::axes) and w the row's wrench (Tile::wrench); elsewhere zero.
// columns 4 Q .. on: their coordinates' axes, transposed, against the lane's own weights
template <int Q, int N>
__device__ __forceinline__ void add_motions(uint32_t on_low, uint32_t on_high, const Vec4& first, const Vec4& last, const float* x, Vec4& low, Vec4& high) {
    if constexpr (Q < N / 4) {
        const Vec4 xs = reinterpret_cast<const Vec4*>(x)[Q];
#pragma unroll
        for (uint32_t t = 0u; t < 4u; ++t) {
            const float on = kept_if(Q < 8 ? on_low : on_high, (4u * uint32_t(Q) + t) & 31u, xs[t]);
            low = __builtin_amdgcn_mfma_f32_4x4x1f32(first[t], on, low, 4, Q, 0);
            high = __builtin_amdgcn_mfma_f32_4x4x1f32(last[t], on, high, 4, Q, 0);   // (and two components nobody reads)
        }
        add_motions<Q + 1, N>(on_low, on_high, first, last, x, low, high);
    }
}
// lane = head: the motion of the head's link, sum over the coordinates j on its way of s_j x_j, for a vector x in LDS.
template <int N>
__device__ __forceinline__ void link_motion(const Tile& c, uint64_t way, const float* x, float (&motion)[6]) {
    if (c.way_runs) {
        const LaneRun run(uint32_t(way), uint32_t(way >> 32u));
        const float4* table = reinterpret_cast<const float4*>(c.axes);
        const float4 a = table[3u * c.lane], b = table[3u * c.lane + 1u];
        const float s[6] = {a.x, a.y, a.z, a.w, b.x, b.y};
        const double own = double(x[c.lane]);   // (a lane past the coordinates holds zeros on both sides)
#pragma unroll
        for (int k = 0; k < 6; ++k) motion[k] = float(run.sum(double(s[k]) * own));
        return;
    }
    // Every lane of the wavefront, those without a head with a way of none: v_mfma_f32_4x4x1 takes a coordinate's axis, a
    // component a lane of four, against the lane's own weight, and register r of a lane is the sum of component r.  (The axes word by
    // word from the table in LDS: 2048 trees of 64 coordinates in limbs of three 1938 us a step, as it is 1793.)
    const FourUnits units(c.lane);
    const float4* table = reinterpret_cast<const float4*>(c.axes);
    const float4 a = table[3u * c.lane], b = table[3u * c.lane + 1u];
    const float four[4] = {a.x, a.y, a.z, a.w}, two[4] = {b.x, b.y, 0.0f, 0.0f};
    const Vec4 first = units.transposed(four), last = units.transposed(two);
    Vec4 low = {}, high = {};
    add_motions<0, N>(opaque_word(uint32_t(way)), opaque_word(uint32_t(way >> 32u)), first, last, x, low, high);
    motion[0] = low[0]; motion[1] = low[1]; motion[2] = low[2]; motion[3] = low[3]; motion[4] = high[0]; motion[5] = high[1];
}
// lane = head: row `axis` of head h times the vector whose link motion is `motion`
__device__ __forceinline__ float wrench_dot(const Tile& c, uint32_t h, uint32_t axis, const float (&motion)[6]) {
    const float* w = c.wrench + h * kWrenchStride + 6u * axis;
    return fmaf(w[5], motion[5], fmaf(w[4], motion[4], fmaf(w[3], motion[3], fmaf(w[2], motion[2], fmaf(w[1], motion[1], w[0] * motion[0])))));
}
__device__ __forceinline__ uint64_t way_of(const Tile& c, uint32_t h) {
    return (uint64_t(c.U(hColumnsHigh, h)) << 32u) | uint64_t(c.U(hColumnsLow, h));
}
// lane = head holds 4 kGroups values; lane = coordinate comes back with their sums over the heads of `heads` (a uniform mask of
// the first 64) whose way holds the coordinate, added to `sum` in head order: an instruction a head and group, a head's four
// values of a group, a lane of four each, against the coordinates' own ones and zeros.  The lanes of heads outside `heads`
// hold zeros.
template <int Q, int kGroups>
__device__ __forceinline__ void add_over_ways(uint32_t over_low, uint32_t over_high, uint64_t heads, const Vec4 (&words)[kGroups], Vec4 (&sum)[kGroups]) {
    if constexpr (Q < int(kWave) / 4) {
        if constexpr (Q % 4 == 0) if ((heads >> (4 * Q)) == 0ull) return;
        const uint32_t over = Q < 8 ? over_low : over_high;
#pragma unroll
        for (uint32_t t = 0u; t < 4u; ++t) {
            const float through = kept_if(over, (4u * uint32_t(Q) + t) & 31u, 1.0f);
#pragma unroll
            for (uint32_t g = 0u; g < uint32_t(kGroups); ++g) sum[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(words[g][t], through, sum[g], 4, Q, 0);
        }
        add_over_ways<Q + 1>(over_low, over_high, heads, words, sum);
    }
}
template <int kGroups>
__device__ __forceinline__ void sums_over_ways(const Tile& c, uint64_t heads, const float (&v)[4 * kGroups], Vec4 (&sum)[kGroups]) {
    const FourUnits units(c.lane);
    Vec4 words[kGroups];
#pragma unroll
    for (uint32_t g = 0u; g < uint32_t(kGroups); ++g) {
        const float four[4] = {v[4u * g], v[4u * g + 1u], v[4u * g + 2u], v[4u * g + 3u]};
        words[g] = units.transposed(four);
    }
    // (through the barrier so that the sixty-four ones and zeros are made here, not ahead of the sweeps and kept)
    add_over_ways<0>(opaque_word(c.over_low), opaque_word(c.over_high), heads, words, sum);
}
// lane = coordinate: sum over the heads `heads` (a uniform mask of the first 64) of J^T x, x one value an axis held by
// lane = head, in double: the heads' wrenches weighted by x summed over the heads whose way holds the coordinate, then
// taken against the coordinate's motion axis.  With `weights` (the magnitudes that go with x) also the rounding scale
// of that sum, an upper bound: sum |s_j| . sum |w| weights.
template <bool kScale>
__device__ __forceinline__ double rows_transposed_times(const Tile& c, uint64_t heads, const float (&x)[3], const float (&weights)[3], float* scale) {
    const uint32_t lane = c.lane;
    float sum[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, bound[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (lane < c.heads && ((heads >> lane) & 1ull) != 0ull) {
        const float* w = c.wrench + lane * kWrenchStride;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            sum[k] = (w[k] * x[0] + w[6 + k] * x[1]) + w[12 + k] * x[2];
            if constexpr (kScale) bound[k] = (fabsf(w[k]) * weights[0] + fabsf(w[6 + k]) * weights[1]) + fabsf(w[12 + k]) * weights[2];
        }
    }
    double carried[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    Vec4 carried_bound[2] = {};
    if (c.over_runs) {
        const LaneRun run(c.over_low, c.over_high);
#pragma unroll
        for (int k = 0; k < 6; ++k) carried[k] = run.sum(double(sum[k]));
        if constexpr (kScale) {
#pragma unroll
            for (int k = 0; k < 6; ++k) carried_bound[k / 4][k % 4] = float(run.sum(double(bound[k])));
        }
    } else {
        // (in double from here: two lane reads a component and head, where one and its widening took a quarter-rate conversion;
        // eight heads a turn at constant lanes, those outside `heads` holding zeros)
        double wide[6];
    #pragma unroll
        for (int k = 0; k < 6; ++k) wide[k] = double(sum[k]);
    #pragma unroll
        for (int first = 0; first < int(kWave); first += 8) {
            if (((heads >> first) & 0xFFull) == 0ull) continue;
            const uint32_t eight = (first < 32 ? c.over_low : c.over_high) >> (first & 31);
    #pragma unroll
            for (int t = 0; t < 8; ++t) {
                const double through = __hiloint2double(int(bit_spread(eight, uint32_t(t)) & 0x3ff00000u), 0);   // one or zero
    #pragma unroll
                for (int k = 0; k < 6; ++k) carried[k] = fma(through, lane_value_d(wide[k], first + t), carried[k]);
            }
        }
        if constexpr (kScale) sums_over_ways<2>(c, heads, bound, carried_bound);
    }
    const float4* table = reinterpret_cast<const float4*>(c.axes);
    const float4 a = table[3u * lane], b = table[3u * lane + 1u];
    const float s[6] = {a.x, a.y, a.z, a.w, b.x, b.y};
    double total = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) total = fma(double(s[k]), carried[k], total);
    if constexpr (kScale) {
        float magnitude = 0.0f;
#pragma unroll
        for (int k = 0; k < 6; ++k) magnitude = fmaf(fabsf(s[k]), carried_bound[k / 4][k % 4], magnitude);
        *scale += magnitude;
    }
    return total;
}

// The heads' curvature sum_h J_h^T C_h J_h by way of the links, for blocks whose staged heads each act through one link.
// A row of such a head is a wrench w = [(p - o) x n; n] about a point o, met by every coordinate j on the way from the
// head's link to the root with its motion axis s_j = [a_j; (r_j - o) x a_j] (a sliding coordinate: [0; a_j]):
// J_j = s_j . w, the entry the row assembly wrote (assemble_rows.cu:122-169).  The head's term in H_ij is therefore
// s_i^T (W C W^T) s_j when both i and j lie on that way, else zero; and of two coordinates that share any head one lies
// on the other's way to the root.  With K_i the sum of W C W^T over the heads whose way to the root holds i - the
// contact stiffness coordinate i carries, as a composite inertia is the inertia it carries -
//     H_ij += (K_i s_i) . s_j   for j on i's way to the root,      (K_j s_j) . s_i   for i on j's,
// which takes 21 words a head and 12 a column where the plain sum over heads takes 3 N words a head.  The two forms
// of one entry multiply and add the same numbers in the same order: the rows stay each other's transposes to the bit.
// lane = head on the way in (mc: its curvature, `mine`: it contributes), lane = coordinate from the sums on.  Both products
// run on the matrix cores with the multiply-adds of the vector form, bit for bit; while no curvature has changed the
// stiffness of the last assembly, left in the table beside the axes, stands.  A
// step of 8192 ropes: 22.1 -> 18.5 ms with the sums of rows_transposed_times and link_motion in the same form.
// columns 4 Q .. on of lane's row: (K_i s_i) . s_j and (K_j s_j) . s_i, each the stiffness-times-axis of the coordinate
// further from the root first, four columns an instruction and component
template <int Q, int N>
__device__ __forceinline__ void add_link_columns(const float (&s)[6], const float (&y)[6], const uint32_t (&path)[2], const uint32_t (&under)[2], float (&hrow)[N]) {
    if constexpr (Q < N / 4) {
        Vec4 mine_first = {}, other_first = {};
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            mine_first = __builtin_amdgcn_mfma_f32_4x4x1f32(s[t], y[t], mine_first, 4, Q, 0);
            other_first = __builtin_amdgcn_mfma_f32_4x4x1f32(y[t], s[t], other_first, 4, Q, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t at = uint32_t(4 * Q + r) & 31u;
            const uint32_t bits = (bit_spread(path[Q / 8], at) & __float_as_uint(mine_first[r])) | (bit_spread(under[Q / 8], at) & __float_as_uint(other_first[r]));
            hrow[4 * Q + r] += __uint_as_float(bits);
        }
        add_link_columns<Q + 1>(s, y, path, under, hrow);
    }
}
template <int N>
__device__ __forceinline__ void add_heads_through_links(const Tile& c, bool mine, const float (&mc)[6], float (&hrow)[N]) {
    const uint32_t lane = c.lane;
    float4* table = reinterpret_cast<float4*>(c.axes);
    if (!c.stiffness_current) {
        float k[24];
#pragma unroll
        for (int e = 0; e < 24; ++e) k[e] = 0.0f;
        if (mine) {
            const uint32_t slot = c.slot(lane), stride = c.U(hStride, lane), axes = c.U(hAxes, lane);
            const bool second = c.U(hSecond, lane) != 0u;
            float w[3][6];
#pragma unroll
            for (uint32_t a = 0u; a < 3u; ++a) {
                if (c.from_links) {
#pragma unroll
                    for (int t = 0; t < 6; ++t) w[a][t] = c.wrench[lane * kWrenchStride + 6u * a + uint32_t(t)];
                    continue;
                }
#pragma unroll
                for (int t = 0; t < 6; ++t) w[a][t] = 0.0f;
                if (a != 0u && axes == 1u) continue;
                const size_t rs = size_t{slot} + a * stride;
                const float* row = c.rows + rs * kRowWords + 12u;          // the first side's direction; the second side's is its negative,
                const float* at = (second ? c.row_point_b : c.row_point_a) + 3u * rs;   // and W C W^T does not see the sign
                const V3 n{row[0], row[1], row[2]};
                const V3 arm = sub3(V3{at[0], at[1], at[2]}, c.pivot);
                const V3 moment = cross3(arm, n);
                w[a][0] = moment.x; w[a][1] = moment.y; w[a][2] = moment.z; w[a][3] = n.x; w[a][4] = n.y; w[a][5] = n.z;
            }
            const float cxx = mc[0], cyy = mc[1], czz = mc[2], cxy = mc[3], cxz = mc[4], cyz = mc[5];
            float u[3][6];
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                u[0][t] = (cxx * w[0][t] + cxy * w[1][t]) + cxz * w[2][t];
                u[1][t] = (cxy * w[0][t] + cyy * w[1][t]) + cyz * w[2][t];
                u[2][t] = (cxz * w[0][t] + cyz * w[1][t]) + czz * w[2][t];
            }
            int e = 0;
#pragma unroll
            for (int r = 0; r < 6; ++r) {
#pragma unroll
                for (int t = r; t < 6; ++t) k[e++] = (w[0][r] * u[0][t] + w[1][r] * u[1][t]) + w[2][r] * u[2][t];
            }
        }
        // lane = coordinate: the stiffness of every head whose way to the root passes through it
        Vec4 carried[6] = {};
        sums_over_ways<6>(c, __ballot(mine), k, carried);
        const float4 a = table[3u * lane], b = table[3u * lane + 1u];
        const float s[6] = {a.x, a.y, a.z, a.w, b.x, b.y};
        float y[6];
        // y = K s, K symmetric with its upper triangle in `carried`, rows first
        const auto entry = [&](int r, int t) {
            const int e = r <= t ? r * 6 - r * (r - 1) / 2 + (t - r) : t * 6 - t * (t - 1) / 2 + (r - t);
            return carried[e / 4][e % 4];
        };
#pragma unroll
        for (int r = 0; r < 6; ++r) {
            float sum = entry(r, 0) * s[0];
#pragma unroll
            for (int t = 1; t < 6; ++t) sum = fmaf(entry(r, t), s[t], sum);
            y[r] = sum;
        }
        table[3u * lane + 1u] = float4{b.x, b.y, y[0], y[1]};
        table[3u * lane + 2u] = float4{y[2], y[3], y[4], y[5]};
        c.stiffness_current = true;
    }
    const float4 la = table[3u * lane], lb = table[3u * lane + 1u], lc = table[3u * lane + 2u];
    const float s[6] = {la.x, la.y, la.z, la.w, lb.x, lb.y}, y[6] = {lb.z, lb.w, lc.x, lc.y, lc.z, lc.w};
    // (through the barrier so that the sixty-four lane masks of each are made here, two instructions a column, instead of
    // ahead of the sweeps and kept in scalar registers the kernel does not have)
    const uint32_t path[2] = {opaque_word(c.path_low), opaque_word(c.path_high)};
    const uint32_t under[2] = {opaque_word(c.under_low) & ~path[0], opaque_word(c.under_high) & ~path[1]};
    add_link_columns<0>(s, y, path, under, hrow);
}

// AssembleTileBlock (:1507-1618): lane i assembles row i of H = M + sum J^T C J in `hrow` and its force g_i.  The
// first 64 heads evaluate their response one per lane and hand it to the row lanes as scalar lane reads; heads beyond
// 64 pass theirs through the head fields.
// In a reduced block (kFollow) the mass row is the sum of two floats, `mrow` and low_row: the Schur complement as it comes
// out of the double-precision elimination.  The force takes both parts, so that the velocity the block converges to
// balances the momentum against the mass matrix itself; the Hessian takes the first.
template <int N, bool kFollow>
__device__ __forceinline__ bool assemble_block(const Tile& c, const float (&mrow)[N], PlainLine& own, float u, float free_v,
                               float (&hrow)[N], float* force, float* inertia, bool* converged) {
    const uint32_t lane = c.lane;
    const bool coordinate = lane < c.n;
    // the difference of two floats, exact in double (the reference carries it as a float and its rounding error)
    double* dvec = reinterpret_cast<double*>(c.vec);
    float* uvec = c.vec + 128;
    dvec[lane] = double(u) - double(free_v); uvec[lane] = fabsf(u);
    PROF_BEGIN(c, 10);
    // lane's own head (the first 64 heads) from its constants, without a branch; a lane without an owned head gets zeros
    float mf[3], mc[6], mn[3];
    if (c.elliptic) head_terms(c, lane, mf, mc, mn);   // the cone's own response; the same values as below for every other head
    else {
        refresh_moves(c, own);
        plain_response(own, own.move[0], own.move[1], own.move[2], mf, mc);
#pragma unroll
        for (int k = 0; k < 3; ++k) mn[k] = fabsf(mf[k]) + mc[k] * (fabsf(own.res[k]) + fabsf(own.move[k]));
    }
    // whether anything of the head is not zero (lanes from the heads' count on hold copies of the first sixteen heads when
    // there are no more than that)
    const auto bits = [](float v) { return __float_as_uint(v); };
    const uint32_t any_bits = ((bits(mf[0]) | bits(mf[1]) | bits(mf[2])) | (bits(mc[0]) | bits(mc[1]) | bits(mc[2]))) |
                              ((bits(mc[3]) | bits(mc[4]) | bits(mc[5])) | (bits(mn[0]) | bits(mn[1]) | bits(mn[2])));
    const bool mine = lane < c.heads && (any_bits << 1u) != 0u;
    // The Hessian M + sum J^T C J changes only through the heads' curvatures: the curvature of a head's last assembly is
    // kept (in the lane of a head below 64, in the fields beyond), and while none differs the factor of the last
    // factorisation still stands.
    uint32_t differs = 0u;
    for (uint32_t h = lane + kWave; c.scalar_later && h < c.heads; h += kWave) {
        const ScalarLine s = scalar_line(c, h);
        float f, cv;
        scalar_line_response(s, s.move, &f, &cv);
        differs |= bits(c.F(hC, h)) ^ bits(cv);
        c.F(hF, h) = f; c.F(hC, h) = cv;
    }
    for (uint32_t h = lane + kWave; !c.scalar_later && h < c.heads; h += kWave) {
        float f[3], cv[6], noise[3];
        head_terms(c, h, f, cv, noise);
#pragma unroll
        for (int k = 0; k < 3; ++k) c.F(hF + k, h) = f[k];
#pragma unroll
        for (int k = 0; k < 6; ++k) { differs |= bits(c.F(hC + k, h)) ^ bits(cv[k]); c.F(hC + k, h) = cv[k]; }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) { differs |= bits(c.curvature[k]) ^ bits(mc[k]); c.curvature[k] = mc[k]; }
    if (__any(lane < c.heads && differs != 0u)) { c.factor_current = false; c.rows_current = false; c.stiffness_current = false; }
    const bool rows_kept = N <= 32 && c.rows_current && c.heads <= uint32_t(kWave);   // only the force is to be summed
    if (c.units && lane < c.heads && c.U(hUnit, lane) != kInvalid) {   // a coordinate reads its unit heads' responses from the fields
        c.F(hF, lane) = mf[0]; c.F(hC, lane) = mc[0];
    }
    lds_sync<N>();
    PROF_END(c, 10);
    PROF_BEGIN(c, 11);
    // Padded columns (k >= n) hold exact zeros in the mass row, the vectors and the Jacobian rows: their terms add
    // nothing to any of the sums below.
    TileSum inertial{0.0};
    double inertial_scale = 0.0;
    const double2* d2 = reinterpret_cast<const double2*>(dvec);
    const float4* low4 = low_row<N>(c);
    float4 low{};
#pragma unroll
    for (int q = 0; q < N / 2; ++q) {
        const double2 dv = d2[q];
        // (the mass rows do not change over the solve: left to itself the compiler widens them to double once, ahead of
        // the sweeps, and holds two registers an entry from there on - which pays while they fit, and a wide block
        // has no room for)
        const double m0 = double(N >= kWidenAtUse ? opaque_with(mrow[2 * q], u) : mrow[2 * q]);
        const double m1 = double(N >= kWidenAtUse ? opaque_with(mrow[2 * q + 1], u) : mrow[2 * q + 1]);
        hrow[2 * q] = mrow[2 * q]; hrow[2 * q + 1] = mrow[2 * q + 1];
        inertial.value = fma(m0, dv.x, inertial.value);
        inertial.value = fma(m1, dv.y, inertial.value);
        if constexpr (kFollow) {
            if (q % 2 == 0) low = low4[q / 2];
            inertial.value = fma(double(q % 2 == 0 ? low.x : low.z), dv.x, inertial.value);
            inertial.value = fma(double(q % 2 == 0 ? low.y : low.w), dv.y, inertial.value);
        }
        inertial_scale = fma(fabs(m0), fabs(dv.x), inertial_scale);
        inertial_scale = fma(fabs(m1), fabs(dv.y), inertial_scale);
    }
    float scale = float(inertial_scale);
    TileSum g{-inertial.value};
    PROF_END(c, 11);
    PROF_BEGIN(c, 12);
    // heads beyond the first 64 hold their responses in the fields, unit heads theirs
    auto noise_of = [&](float f, float curvature, uint32_t h, uint32_t axis) {
        return fabsf(f) + curvature * (fabsf(c.F(hRes + axis, h)) + fabsf(c.F(hMove + axis, h)));
    };
    auto add_later_head = [&](uint32_t h) {
        const float f[3] = {c.F(hF, h), c.F(hF + 1, h), c.F(hF + 2, h)};
        const float cv[6] = {c.F(hC, h), c.F(hC + 1, h), c.F(hC + 2, h), c.F(hC + 3, h), c.F(hC + 4, h), c.F(hC + 5, h)};
        if (f[0] == 0.0f && f[1] == 0.0f && f[2] == 0.0f && cv[0] == 0.0f && cv[1] == 0.0f && cv[2] == 0.0f && cv[3] == 0.0f && cv[4] == 0.0f && cv[5] == 0.0f) return;
        const float noise[3] = {noise_of(f[0], cv[0], h, 0u), noise_of(f[1], cv[1], h, 1u), noise_of(f[2], cv[2], h, 2u)};
        const uint64_t columns = (uint64_t(__builtin_amdgcn_readfirstlane(c.U(hColumnsHigh, h))) << 32u) |
                                 uint64_t(__builtin_amdgcn_readfirstlane(c.U(hColumnsLow, h)));
        add_head<N>(c, h, coordinate, f, cv, noise, c.U(hAxes, h), columns, hrow, g, scale);
    };
    // the staged ones of the first 64
    const uint64_t staged = __ballot(mine && (!c.units || c.U(hUnit, lane) == kInvalid));
    if (N > kTwoWaveWidth && c.from_links) {
        if (staged != 0ull) {
            float weighted = 0.0f;
            g.value += rows_transposed_times<true>(c, staged, mf, mn, &weighted);
            scale += weighted;
            add_heads_through_links<N>(c, mine, mc, hrow);
        }
    } else if (N > kTwoWaveWidth && c.through_links && __popcll(staged) >= int(kLinkHeads)) {
        // enough heads that their curvature is cheaper by way of the links; the force takes the staged rows as ever
        add_heads_force<N>(c, staged, mf, mn, lane < c.heads ? c.U(hRow, lane) : 0u, g, scale);
        add_heads_through_links<N>(c, mine, mc, hrow);
    } else {
        if (N <= 32 || (N <= kTwoWaveWidth && c.near_heads && !c.units)) {
            if constexpr (N <= kTwoWaveWidth) if (staged != 0ull) {
                const uint32_t my_first = c.U(hRow, lane < c.heads ? lane : 0u);
                bool added = false;
                if constexpr (kFollow && N <= 32) {
                    added = !c.smooth;
                    if (added && rows_kept) add_heads_by_groups<N, false>(c, staged, mf, mc, mn, my_first, hrow, g, scale);
                    else if (added) add_heads_by_groups<N, true>(c, staged, mf, mc, mn, my_first, hrow, g, scale);
                }
                if (!added && rows_kept) add_heads_by_tiles<N, false>(c, staged, mf, mc, mn, my_first, hrow, g, scale);
                else if (!added) add_heads_by_tiles<N, true>(c, staged, mf, mc, mn, my_first, hrow, g, scale);
            }
        } else if (N <= kTwoWaveWidth && c.block_heads) {
            if constexpr (N <= kTwoWaveWidth)
                if (staged != 0ull) add_block_heads<N>(c, staged, coordinate, mf, mc, mn, c.U(hRow, lane < c.heads ? lane : 0u), hrow, g, scale);
        } else {
            const uint32_t own_head = lane < c.heads ? lane : 0u;
            const uint32_t my_axes = c.U(hAxes, own_head), my_low = c.U(hColumnsLow, own_head), my_high = c.U(hColumnsHigh, own_head);
            for (uint64_t rest = staged; rest != 0ull; rest &= rest - 1ull) {
                const uint32_t h = uint32_t(__builtin_ctzll(rest));
                float f[3], cv[6], noise[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) { f[k] = uniform_lane_value(mf[k], h); noise[k] = uniform_lane_value(mn[k], h); }
#pragma unroll
                for (int k = 0; k < 6; ++k) cv[k] = uniform_lane_value(mc[k], h);
                const uint32_t axes = uint32_t(__builtin_amdgcn_readlane(int(my_axes), int(h)));
                const uint64_t columns = (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(my_high), int(h)))) << 32u) |
                                         uint64_t(uint32_t(__builtin_amdgcn_readlane(int(my_low), int(h))));
                add_head<N>(c, h, coordinate, f, cv, noise, axes, columns, hrow, g, scale);
            }
        }
        for (uint32_t h = kWave; h < (c.units ? c.staged_end : c.heads); ++h) {
            if (c.units && c.U(hUnit, h) != kInvalid) continue;
            add_later_head(h);
        }
    }
    if (c.units) {
        // a unit head - a row on one coordinate - adds to that coordinate's diagonal and force only: lane = coordinate walks
        // its own short list, or, when some coordinate's list overflowed, the wave walks every unit head in turn
        // (the list and then its heads' words read whether or not the lane has so many, all in flight together: a head that does
        // not contribute holds zeros)
        float diagonal = 0.0f;
        auto add_unit = [&](float v, float curvature, float force, float res, float move) {
            diagonal += v * curvature * v;
            tile_add_product(g, v, force);
            scale += fabsf(v) * (fabsf(force) + curvature * (fabsf(res) + fabsf(move)));
        };
        if (c.unit_lists) {
            uint32_t h[kUnitSlots];
            float v[kUnitSlots], words[kUnitSlots][4];
#pragma unroll
            for (uint32_t k = 0u; k < kUnitSlots; ++k) {
                const uint32_t listed = c.unit_list[k * uint32_t(kWave) + lane];
                h[k] = k < c.unit_count ? listed : 0u;
            }
#pragma unroll
            for (uint32_t k = 0u; k < kUnitSlots; ++k) {
                if (k >= c.unit_most) break;
                v[k] = c.F(hUnitValue, h[k]); words[k][0] = c.F(hC, h[k]); words[k][1] = c.F(hF, h[k]);
                words[k][2] = c.F(hRes, h[k]); words[k][3] = c.F(hMove, h[k]);
            }
#pragma unroll
            for (uint32_t k = 0u; k < kUnitSlots; ++k) {
                if (k >= c.unit_most) break;
                const bool on = k < c.unit_count;
                add_unit(on ? v[k] : 0.0f, on ? words[k][0] : 0.0f, on ? words[k][1] : 0.0f, on ? words[k][2] : 0.0f, on ? words[k][3] : 0.0f);
            }
        } else {
            for (uint32_t h = 0u; h < c.heads; ++h)
                if (c.U(hUnit, h) == lane) add_unit(c.F(hUnitValue, h), c.F(hC, h), c.F(hF, h), c.F(hRes, h), c.F(hMove, h));
        }
        if (!rows_kept) {
#pragma unroll
            for (int k = 0; k < N; ++k) hrow[k] += local_lane(lane) == uint32_t(k) ? diagonal : 0.0f;
        }
    }
    if constexpr (N <= 32) {   // the rows as they stand, for the assemblies that find no curvature changed
        if (!rows_kept) {
            if (lane < uint32_t(N)) {
                float4* words = reinterpret_cast<float4*>(c.hrows + lane * uint32_t(N));
#pragma unroll
                for (int q = 0; q < N / 4; ++q) words[q] = float4{hrow[4 * q], hrow[4 * q + 1], hrow[4 * q + 2], hrow[4 * q + 3]};
            }
            c.rows_current = true;
        } else {
            const float4* words = reinterpret_cast<const float4*>(c.hrows + min(lane, uint32_t(N - 1)) * uint32_t(N));
#pragma unroll
            for (int q = 0; q < N / 4; ++q) {
                const float4 w = words[q];
                hrow[4 * q] = w.x; hrow[4 * q + 1] = w.y; hrow[4 * q + 2] = w.z; hrow[4 * q + 3] = w.w;
            }
        }
    }
    PROF_END(c, 12);
    PROF_BEGIN(c, 13);
    *force = coordinate ? float(g.value) : 0.0f;
    *inertia = coordinate ? float(inertial.value) : 0.0f;
    const float4* u4 = reinterpret_cast<const float4*>(uvec);
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const float4 uv = u4[q];
        const float uk[4] = {uv.x, uv.y, uv.z, uv.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) scale += fabsf(hrow[4 * q + t]) * uk[t];
    }
    // a row entry that is not finite leaves its scale not finite: the entries themselves are looked at only then
    bool finite = isfinite(*force) && isfinite(scale);
    if (!__all(!coordinate || finite)) {
        finite = isfinite(*force);
#pragma unroll
        for (int k = 0; k < N; ++k) finite = finite && isfinite(hrow[k]);
    }
    *converged = __all(!coordinate || fabsf(*force) <= kRoundings * FLT_EPSILON * scale);
    const bool ok = __all(!coordinate || finite);
    lds_sync<N>();
    PROF_END(c, 13);
    return ok;
}

enum Failure : uint32_t { kFailNone = 0u, kFailEquation, kFailFactor, kFailDirection, kFailCandidate };

// A reduced block.  Where no contact of the world reaches the coordinates from K on (the arms of a humanoid that
// stands on its feet), those coordinates enter the block's objective through the mass matrix alone and the minimiser
// over them is linear in the others: u_U = free_U - P (u_T - free_T), P = M_UU^-1 M_UT.  Eliminating them once per
// solve leaves the same problem on the K coordinates T with the Schur complement M_TT - M_TU M_UU^-1 M_UT as its mass
// matrix: every Newton block, factorisation and substitution of the solve is K wide instead of N.  The lanes K..n-1
// ("followers") hold a row of -P where the block's lanes hold a mass row, so that the product every Newton step
// takes with the mass rows (mass_times) hands each follower its own move, and the tests the reference makes over all
// coordinates (step below rounding, largest step, mass-normalised residual) still see all of them.  The minimiser of
// each block is the one the full-width block has; the iterates on the way differ by rounding.
// mass_step_i = sum_k M_ik d_k in coordinate order (:2177-2187, 2228-2238).  In a reduced block the lanes past the
// block's coordinates hold a row of -P instead of a mass row, and get their own move -P d from the same products.
template <int N>
__device__ __forceinline__ float mass_times(const Tile& c, const float (&mrow)[N], float d) {
    float* dvec = c.vec + 192;
    dvec[c.lane] = d;
    lds_sync<N>();
    float out = 0.0f;
    const float4* d4 = reinterpret_cast<const float4*>(dvec);
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const float4 dv = d4[q];
        out += mrow[4 * q] * dv.x; out += mrow[4 * q + 1] * dv.y; out += mrow[4 * q + 2] * dv.z; out += mrow[4 * q + 3] * dv.w;
    }
    lds_sync<N>();
    return c.lane < c.n_all ? out : 0.0f;
}


// TileNewtonDirection (:1935-1992).  The reference re-assembles the block after the mass-normalised
// convergence test because its mass factor overwrites the Hessian storage; here the two live apart and the
// assembled row, force and inertia (which the second assembly would reproduce bit for bit) are simply kept.
template <int N, bool kFollow>
__device__ __forceinline__ Failure newton_direction(const Tile& c, const float (&mrow)[N], PlainLine& line, float u, float free_v,
                                    float* force, float* inertia, float* d, bool* converged) {
    PROF_COUNT(c, 0);
    c.work += 16u;
    float hrow[N];
    PROF_BEGIN(c, 1);
    const bool assembled = assemble_block<N, kFollow>(c, mrow, line, u, free_v, hrow, force, inertia, converged);
    PROF_END(c, 1);
    if (!assembled) return kFailEquation;
    if (*converged && c.tolerance > 0.0f) {
        if (!c.mass_valid) return kFailFactor;
        PROF_BEGIN(c, 3);
        const float direction = solve_tile_mass<N>(c, *force);
        PROF_END(c, 3);
        *d = direction;
        bool small = c.lane >= c.n || fabsf(direction) < c.tolerance;
        if constexpr (kFollow) {
            const float follow = mass_times<N>(c, mrow, c.lane < c.n ? direction : 0.0f);
            if (c.lane >= c.n && c.lane < c.n_all) small = fabsf(follow) < c.tolerance;
        }
        *converged = __all(small);
        if (*converged) return kFailNone;
    }
    if (*converged) return kFailNone;
    PROF_BEGIN(c, 2);
    const bool factored = cholesky_solve<N, kFollow>(c, hrow, *force, d);
    PROF_END(c, 2);
    if (!factored) return kFailFactor;
    return kFailNone;
}

// TileRowSteps (:2018-2044): step = J d per head axis by serial fused multiply-adds, lane = head.  The Jacobian row
// and the direction come in as 16-byte words; padded columns are zeros on both sides.
template <int N>
__device__ __forceinline__ float row_dot_fma(const float* jrow, const float* dvec) {
    const float4* j4 = reinterpret_cast<const float4*>(jrow);
    const float4* d4 = reinterpret_cast<const float4*>(dvec);
    float value = 0.0f;
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const float4 j = j4[q], d = d4[q];
        value = fmaf(j.x, d.x, value); value = fmaf(j.y, d.y, value); value = fmaf(j.z, d.z, value); value = fmaf(j.w, d.w, value);
    }
    return value;
}
template <int N>
__device__ __forceinline__ void row_steps(const Tile& c, float d) {
    float* dvec = c.vec;
    dvec[c.lane] = c.lane < c.n ? d : 0.0f;
    lds_sync<N>();
    if (c.heads <= 16u && !c.units && !c.from_links) {
        // a lane a row: the first three rows of sixteen lanes take an axis each, lane & 15 = head (a head on one axis has
        // zeros in the rows of the others)
        const uint32_t axis = c.lane >> 4u, h = c.lane & 15u;
        if (axis < 3u && h < c.heads && c.U(hRow, h) != kInvalid)
            c.fields[axis == 0u ? c.at(hStep, h) : c.at(hStep + 1, h) + axis - 1u] = row_dot_fma<N>(c.jac + (c.U(hRow, h) + axis) * uint32_t(N), dvec);
        lds_sync<N>();
        return;
    }
    if constexpr (N > kTwoWaveWidth) {
        if (c.from_links) {   // contact heads, one a lane at most, none of them a unit head
            const bool owned = c.lane < c.heads && c.owned(c.lane < c.heads ? c.lane : 0u);
            const uint32_t h = owned ? c.lane : 0u, axes = c.U(hAxes, h);
            float motion[6];
            link_motion<N>(c, owned ? way_of(c, h) : 0ull, dvec, motion);
            if (owned) {
                c.F(hStep, h) = wrench_dot(c, h, 0u, motion);
                c.F(hStep + 1, h) = axes > 1u ? wrench_dot(c, h, 1u, motion) : 0.0f;
                c.F(hStep + 2, h) = axes > 2u ? wrench_dot(c, h, 2u, motion) : 0.0f;
            }
            lds_sync<N>();
            return;
        }
    }
    // a lane a row of the staged heads (a head on one axis has zeros in its other rows), then a lane a unit head, which all
    // come after them.  (A lane a head, its three rows in turn, held the unit heads up behind a dozen contacts.)
    for (uint32_t r = c.lane; r < 3u * c.staged_end; r += kWave) {
        const uint32_t h = r / 3u, axis = r - 3u * h, first = c.U(hRow, h);
        if (first == kInvalid || !c.owned(h)) continue;
        c.fields[axis == 0u ? c.at(hStep, h) : c.at(hStep + 1, h) + axis - 1u] = row_dot_fma<N>(c.jac + (first + axis) * uint32_t(N), dvec);
    }
    if (c.units) {
        for (uint32_t h = c.lane; h < c.heads; h += kWave) {
            const uint32_t unit = c.U(hUnit, h);
            if (c.owned(h) && unit != kInvalid) c.F(hStep, h) = c.F(hUnitValue, h) * dvec[unit];   // :2028-2032
        }
    }
    lds_sync<N>();
}

__device__ __forceinline__ void plain_line_terms(const PlainLine& p, float alpha, TileSum& row_slope, float& row_curvature, float& row_magnitude) {
    const float sx = p.step[0], sy = p.step[1], sz = p.step[2];
    float f[3], r[6];
    const float mx = fmaf(alpha, sx, p.move[0]), my = fmaf(alpha, sy, p.move[1]), mz = fmaf(alpha, sz, p.move[2]);
    plain_response(p, mx, my, mz, f, r);
    tile_add_product(row_slope, f[0], sx);
    tile_add_product(row_slope, f[1], sy);
    tile_add_product(row_slope, f[2], sz);
    row_magnitude += fabsf(f[0] * sx) + fabsf(f[1] * sy) + fabsf(f[2] * sz) + line_noise(r, p.res[0], p.res[1], p.res[2], mx, my, mz, sx, sy, sz);
    row_curvature += r[0] * sx * sx + r[1] * sy * sy + r[2] * sz * sz + 2.0f * r[5] * sy * sz;
}
// The line search runs in one of five modes, the same for every probe of a solve: general (some head is under the elliptic
// cone, or later heads need more than a number a field), general with at most sixteen heads (cone), plain with the terms in
// the first sixteen lanes (narrow), plain over the whole wavefront, plain with the heads past the first 64 as numbers beside
// it (later).  The mode is a template argument so that the probes carry no branch on it.
enum LineMode : int { kLineGeneral = 0, kLineWide = 1, kLineNarrow = 2, kLineLater = 3, kLineCone = 4 };
template <LineMode kMode>
__device__ __forceinline__ void line_derivatives(const Tile& c, const HeadLine& mine, const PlainLine& plain, const ScalarLine (&later)[kLaterHeads], float alpha,
                                 float inertial_slope, float inertial_curvature, float* slope, float* curvature, float* magnitude) {
    PROF_COUNT(c, 1);
    c.work += 1u;
    TileSum row_slope{0.0};
    float row_curvature = 0.0f, row_magnitude = 0.0f;
    if constexpr (kMode == kLineGeneral) {
        if (mine.owned) line_terms(mine, alpha, row_slope, row_curvature, row_magnitude);
        for (uint32_t h = c.lane + kWave; h < c.heads; h += kWave) {
            const HeadLine extra = load_head_line(c, h);
            if (extra.owned) line_terms(extra, alpha, row_slope, row_curvature, row_magnitude);
        }
    } else if constexpr (kMode == kLineCone) {
        if (mine.owned) line_terms(mine, alpha, row_slope, row_curvature, row_magnitude);
    } else {
        plain_line_terms(plain, alpha, row_slope, row_curvature, row_magnitude);
        if constexpr (kMode == kLineLater) {
#pragma unroll
            for (uint32_t e = 0u; e < kLaterHeads; ++e) {
                if (c.heads <= kWave * (e + 1u)) break;
                const ScalarLine& s = later[e];
                float f, r;
                const float move = fmaf(alpha, s.step, s.move);
                scalar_line_response(s, move, &f, &r);
                tile_add_product(row_slope, f, s.step);
                row_magnitude += fabsf(f * s.step) + r * (fabsf(s.res) + fabsf(move)) * fabsf(s.step);
                row_curvature += r * s.step * s.step;
            }
        }
    }
    PROF_BEGIN(c, 25);
    TileSum total{-row_slope.value};
    if (c.lane == 0u) {
        tile_add_product(total, alpha, inertial_curvature);
        tile_add(total, inertial_slope);
    }
    if constexpr (kMode == kLineNarrow || kMode == kLineCone) {
        // with at most sixteen heads every term sits in the first row of lanes; (t + 0) + (0 + 0) is t, so the sums agree
        *slope = wave_total(total, true);
        *curvature = inertial_curvature + first_row_sum(row_curvature);
        *magnitude = fabsf(inertial_slope) + alpha * inertial_curvature + first_row_sum(row_magnitude);
    } else {
        *slope = wave_total(total);
        *curvature = inertial_curvature + wave_sum(row_curvature);
        *magnitude = fabsf(inertial_slope) + alpha * inertial_curvature + wave_sum(row_magnitude);
    }
    PROF_END(c, 25);
}

// The search always evaluates the line at 0 and then at 1.  In the narrow and cone modes the rows of sixteen lanes hold copies of
// the same heads (lane & 15) and the row sums stay within a row: the first row evaluates the line at 0 while the others
// evaluate it at 1, one pass for both points with the numbers either gives alone.  Each point's sums come out in its
// row's lanes.
struct LinePoint { float slope, curvature, magnitude; };
template <LineMode kMode>
__device__ __forceinline__ void line_derivatives_pair(const Tile& c, const HeadLine& mine, const PlainLine& plain, float inertial_slope, float inertial_curvature,
                                                      LinePoint* at_zero, LinePoint* at_one) {
    PROF_COUNT(c, 1);
    const float alpha = c.lane < 16u ? 0.0f : 1.0f;
    TileSum row_slope{0.0};
    float row_curvature = 0.0f, row_magnitude = 0.0f;
    if constexpr (kMode == kLineCone) {
        if (mine.owned) line_terms(mine, alpha, row_slope, row_curvature, row_magnitude);
    } else plain_line_terms(plain, alpha, row_slope, row_curvature, row_magnitude);
    TileSum total{-row_slope.value};
    if ((c.lane & 15u) == 0u) {
        tile_add_product(total, alpha, inertial_curvature);
        tile_add(total, inertial_slope);
    }
    const double slopes = row_total_d(total.value);
    float cv = row_curvature, mg = row_magnitude;
    cv += dpp_move<kDppXor1>(cv); cv += dpp_move<kDppXor2>(cv); cv += dpp_move<kDppHalfMirror>(cv); cv += dpp_move<kDppMirror>(cv);
    mg += dpp_move<kDppXor1>(mg); mg += dpp_move<kDppXor2>(mg); mg += dpp_move<kDppHalfMirror>(mg); mg += dpp_move<kDppMirror>(mg);
    at_zero->slope = float(row_value_d(slopes, 0));
    at_zero->curvature = inertial_curvature + row_value(cv, 0);
    at_zero->magnitude = fabsf(inertial_slope) + 0.0f * inertial_curvature + row_value(mg, 0);
    at_one->slope = float(row_value_d(slopes, 1));
    at_one->curvature = inertial_curvature + row_value(cv, 1);
    at_one->magnitude = fabsf(inertial_slope) + 1.0f * inertial_curvature + row_value(mg, 1);
}

// SearchTileLine (:2089-2125)
template <LineMode kMode>
__device__ __forceinline__ float search_line_in(const Tile& c, PlainLine& plain, float inertial_slope, float inertial_curvature) {
    constexpr bool kPaired = kMode == kLineNarrow || kMode == kLineCone;
    float slope = 0.0f, curvature = 0.0f, magnitude = 0.0f;
    HeadLine mine{};
    ScalarLine later[kLaterHeads] = {};
    if constexpr (kMode == kLineLater) {
#pragma unroll
        for (uint32_t e = 0u; e < kLaterHeads; ++e)
            if (c.heads > kWave * (e + 1u)) later[e] = scalar_line(c, c.lane + kWave * (e + 1u));
    }
    if constexpr (kMode == kLineGeneral) mine = load_head_line(c, c.lane);
    else if constexpr (kMode == kLineCone) mine = load_head_line(c, c.lane & 15u);
    else refresh_steps(c, plain);
    float low = 0.0f, high = 0.0f, alpha = 1.0f;
    bool bounded = false;
    float initial;
    uint32_t step = 0u;
    // one turn of the search on the line's slope and curvature at alpha: true when the search ends, with its answer
    auto turn = [&](float* answer) {
        if (!isfinite(slope) || !isfinite(curvature)) {
            high = alpha; bounded = true; alpha = 0.5f * (low + high);
            return false;
        }
        if (fabsf(slope) <= fmaxf(kLineTolerance * -initial, kRoundings * FLT_EPSILON * magnitude)) { *answer = alpha; return true; }
        if (slope < 0.0f) low = alpha;
        else { high = alpha; bounded = true; }
        if (bounded && high - low <= FLT_EPSILON * high) { *answer = low; return true; }
        float next = alpha - slope * __builtin_amdgcn_rcpf(curvature);
        if (!(next > low && (!bounded || next < high))) next = bounded ? 0.5f * (low + high) : 2.0f * alpha;
        alpha = next;
        return false;
    };
    float answer = 0.0f;
    if constexpr (kPaired) {
        LinePoint at_zero, at_one;
        line_derivatives_pair<kMode>(c, mine, plain, inertial_slope, inertial_curvature, &at_zero, &at_one);
        c.work += 1u;
        initial = at_zero.slope;
        if (!(initial < 0.0f)) return 0.0f;
        slope = at_one.slope; curvature = at_one.curvature; magnitude = at_one.magnitude;
        c.work += 1u;
        if (turn(&answer)) return answer;
        step = 1u;
    } else {
        line_derivatives<kMode>(c, mine, plain, later, 0.0f, inertial_slope, inertial_curvature, &slope, &curvature, &magnitude);
        initial = slope;
        if (!(initial < 0.0f)) return 0.0f;
    }
    for (; step < kLineSearchSteps; ++step) {
        line_derivatives<kMode>(c, mine, plain, later, alpha, inertial_slope, inertial_curvature, &slope, &curvature, &magnitude);
        if (turn(&answer)) return answer;
    }
    return low;
}
__device__ __forceinline__ float search_line(const Tile& c, PlainLine& line, float inertial_slope, float inertial_curvature) {
    if (c.scalar_later) return search_line_in<kLineLater>(c, line, inertial_slope, inertial_curvature);
    if (c.elliptic && c.heads <= 16u) return search_line_in<kLineCone>(c, line, inertial_slope, inertial_curvature);
    if (c.heads > uint32_t(kWave) || c.elliptic) return search_line_in<kLineGeneral>(c, line, inertial_slope, inertial_curvature);
    if (c.heads <= 16u) return search_line_in<kLineNarrow>(c, line, inertial_slope, inertial_curvature);
    return search_line_in<kLineWide>(c, line, inertial_slope, inertial_curvature);
}

__device__ __forceinline__ void apply_moves(const Tile& c, float alpha) {
    for (uint32_t h = c.lane; h < c.heads; h += kWave) {
        if (!c.owned(h)) continue;
#pragma unroll
        for (int k = 0; k < 3; ++k) c.F(hMove + k, h) = fmaf(alpha, c.F(hStep + k, h), c.F(hMove + k, h));
    }
    wave_sync();
}

// DescendTileBlock (:2145-2301).  `u` is lane i's block coordinate; `has_free` is false in the position pass.
template <int N, bool kFollow>
__device__ __forceinline__ void descend_block(Tile& c, const float (&mrow)[N], float* u_io, float free_in, bool has_free,
                                              DataView d) {
    const uint32_t lane = c.lane, n = c.n;
    const bool coordinate = lane < n;
    const bool follower = kFollow && lane >= n && lane < c.n_all;
    const bool moving = coordinate || follower;
    PROF_BEGIN(c, 26);
    for (uint32_t h = lane; h < c.heads; h += kWave) {   // StartTileBlock (:1386-1397)
        if (!c.owned(h)) continue;
        c.F(hNormalBound, h) = c.F(hDual, h);
        c.F(hMove, h) = 0.0f; c.F(hMove + 1, h) = 0.0f; c.F(hMove + 2, h) = 0.0f;
    }
    lds_sync<N>();
    PlainLine line = own_line(c);   // the heads' constants over this block descent
    float start = coordinate ? *u_io : 0.0f;
    const float free_v = moving && has_free ? free_in : 0.0f;
    if constexpr (kFollow) {   // the followers start where the block's coordinates put them
        const float follow = mass_times<N>(c, mrow, coordinate ? start - free_v : 0.0f);
        if (follower) start = free_v + follow;
    }
    float u = start;
    if (c.iteration == 0u && has_free) {   // first-sweep segment search (:2165-2209)
        float dd = coordinate ? free_v - u : 0.0f;
        const float mass_step = mass_times<N>(c, mrow, dd);
        if (follower) dd = mass_step;
        TileSum curvature{0.0};
        if (coordinate) tile_add_product(curvature, dd, mass_step);
        const float inertial_curvature = coordinate_total<N>(curvature);
        if (inertial_curvature > 0.0f && isfinite(inertial_curvature)) {
            row_steps<N>(c, dd);
            const float alpha = search_line(c, line, -inertial_curvature, inertial_curvature);
            if (alpha > 0.0f) {
                u = fmaf(alpha, dd, u);
                apply_moves(c, alpha);
            }
        }
    }
    PROF_END(c, 26);
    Failure failure = kFailNone;
    float primal = FLT_MAX;
    for (uint32_t step = 0u; step < kNewtonSteps; ++step) {
        float force = 0.0f, inertia = 0.0f, dd = 0.0f;
        bool converged = false;
        failure = newton_direction<N, kFollow>(c, mrow, line, u, free_v, &force, &inertia, &dd, &converged);
        if (converged) primal = 0.0f;
        if (failure != kFailNone || converged) break;
        if (!coordinate) dd = 0.0f;
        PROF_BEGIN(c, 8);
        const float mass_step = mass_times<N>(c, mrow, dd);
        if (follower) dd = mass_step;
        PROF_END(c, 8);
        PROF_BEGIN(c, 27);
        TileSum decrement{0.0}, slope{0.0}, curvature{0.0};
        if (coordinate) {
            tile_add_product(decrement, force, dd);
            tile_add_product(slope, inertia, dd);
            tile_add_product(curvature, dd, mass_step);
        }
        const float total_decrement = coordinate_total<N>(decrement);
        const float inertial_slope = coordinate_total<N>(slope);
        const float inertial_curvature = coordinate_total<N>(curvature);
        if (!isfinite(total_decrement) || !isfinite(inertial_slope) || !isfinite(inertial_curvature)) { failure = kFailDirection; break; }
        if (!(total_decrement > 0.0f)) break;
        PROF_END(c, 27);
        PROF_BEGIN(c, 4);
        row_steps<N>(c, dd);
        PROF_END(c, 4);
        PROF_BEGIN(c, 5);
        const float alpha = search_line(c, line, inertial_slope, inertial_curvature);
        PROF_END(c, 5);
        PROF_BEGIN(c, 28);
        const float after = fmaf(alpha, dd, u);
        const bool rounded = __all(!moving || after == u);
        if (!__all(!moving || isfinite(after))) { failure = kFailCandidate; break; }
        primal = 0.0f;
        if (moving && !rounded) primal = fmaxf(primal, fabsf(alpha * dd));
        if (!(alpha > 0.0f)) break;
        u = after;
        apply_moves(c, alpha);
        PROF_END(c, 28);
        if (rounded) break;
    }
    PROF_BEGIN(c, 29);
    for (uint32_t h = lane; h < c.heads; h += kWave) {   // EndTileBlock (:1400-1409)
        if (!c.owned(h)) continue;
#pragma unroll
        for (int k = 0; k < 3; ++k) c.F(hRes + k, h) = c.F(hRes + k, h) - c.F(hMove + k, h);
    }
    lds_sync<N>();
    if (failure != kFailNone) {
        c.failed = true;
        if (lane == 0u) d.env_status[c.env] |= kEnvStatusSolverFailure;
    }
    float moved = failure == kFailNone ? 0.0f : FLT_MAX;
    if (moving) moved = fmaxf(moved, __uint_as_float(residual_bits(u - start)));
    c.momentum = fmaxf(c.momentum, wave_max(moved));
    if (failure != kFailNone) primal = FLT_MAX;
    c.residual = fmaxf(c.residual, wave_max(primal));   // one block per environment: no coupled heads
    if (moving) *u_io = u;
    PROF_END(c, 29);
}

// MeasureTilePrimal (:2378-2489): the mass-normalised momentum balance in double
template <int N, bool kFollow>
__device__ __forceinline__ void measure_primal(Tile& c, const float (&mrow)[N], float* velocity_io, float free_v,
                               const float* lambda_env, uint32_t R, bool reconstruct, DataView d) {
    const uint32_t lane = c.lane, n = c.n;
    const bool coordinate = lane < n;
    const bool follower = kFollow && lane >= n && lane < c.n_all;
    // every coordinate's distance from its free velocity, exact in double, through LDS
    double* apart = reinterpret_cast<double*>(c.vec);
    const float here = coordinate ? *velocity_io : 0.0f;
    apart[lane] = coordinate ? double(here) - double(free_v) : 0.0;
    lds_sync<N>();
    double balance = 0.0;
    const double2* apart2 = reinterpret_cast<const double2*>(apart);
    const float4* low4 = low_row<N>(c);
    float4 low{};
#pragma unroll
    for (int q = 0; q < N / 2; ++q) {
        // the mass row does not change over the solve: left to itself the compiler widens all of it to double once,
        // ahead of the sweeps, and holds two registers an entry from there on
        const double2 dv = apart2[q];   // padded terms are exact zeros
        balance = fma(-double(opaque_with(mrow[2 * q], here)), dv.x, balance);
        balance = fma(-double(opaque_with(mrow[2 * q + 1], here)), dv.y, balance);
        if constexpr (kFollow) {
            if (q % 2 == 0) low = low4[q / 2];
            balance = fma(-double(q % 2 == 0 ? low.x : low.z), dv.x, balance);
            balance = fma(-double(q % 2 == 0 ? low.y : low.w), dv.y, balance);
        }
    }
    // heads with an impulse add J^T lambda in head order (:2402-2436).  A unit head touches one coordinate: that
    // lane takes it from its own list when it comes up between the staged heads
    uint32_t next = 0u;
    auto add_units = [&](uint32_t from, uint32_t below) {
        if (!c.units) return;
        if (c.unit_lists) {
            while (next < c.unit_count) {
                const uint32_t h = c.unit_list[next * uint32_t(kWave) + lane];
                if (h >= below) break;
                ++next;
                if (c.owned(h)) balance += double(c.F(hUnitValue, h)) * lambda_env[c.slot(h) - c.env * R];
            }
            return;
        }
        for (uint32_t h = from; h < below; ++h)
            if (c.owned(h) && c.U(hUnit, h) == lane) balance += double(c.F(hUnitValue, h)) * lambda_env[c.slot(h) - c.env * R];
    };
    uint32_t done = 0u;
    bool rows_taken = false;
    if constexpr (N > kTwoWaveWidth) {
        if (c.from_links) {   // lane = head holds its impulse; the sum goes by way of the links
            float impulse[3] = {0.0f, 0.0f, 0.0f};
            if (lane < c.heads && c.owned(lane)) {
                const uint32_t local = c.slot(lane) - c.env * R, stride = c.U(hStride, lane), axes = c.U(hAxes, lane);
                impulse[0] = lambda_env[local];
                if (block_axes(axes)) { impulse[1] = lambda_env[local + stride]; impulse[2] = lambda_env[local + 2u * stride]; }
            }
            const double sum = rows_transposed_times<false>(c, __ballot(impulse[0] != 0.0f || impulse[1] != 0.0f || impulse[2] != 0.0f), impulse, impulse, nullptr);
            if (coordinate) balance += sum;
            rows_taken = true;
        }
    }
    for (uint32_t h = 0u; h < (rows_taken ? 0u : c.staged_end); ++h) {
        const uint32_t first = c.U(hRow, h);
        if (first == kInvalid || !c.owned(h)) continue;
        add_units(done, h);
        done = h + 1u;
        const uint32_t local = c.slot(h) - c.env * R, stride = c.U(hStride, h), axes = c.U(hAxes, h);
        const float ix = lambda_env[local], iy = block_axes(axes) ? lambda_env[local + stride] : 0.0f,
                    iz = block_axes(axes) ? lambda_env[local + 2u * stride] : 0.0f;
        if (!(ix != 0.0f || iy != 0.0f || iz != 0.0f)) continue;
        if (!coordinate) continue;
        const float* j = c.jac + first * c.ldj;
        balance += double(j[lane]) * ix;
        if (block_axes(axes)) {
            balance += double(j[c.ldj + lane]) * iy;
            balance += double(j[2u * c.ldj + lane]) * iz;
        }
    }
    add_units(done, c.heads);
    lds_sync<N>();
    const float force = float(balance);
    const bool finite = __all(!coordinate || fabs(balance) <= double(FLT_MAX));
    Failure failure = finite ? kFailNone : kFailEquation;
    float direction = 0.0f;
    if (failure == kFailNone) {
        if (c.mass_valid) direction = solve_tile_mass<N>(c, force);
        else failure = kFailFactor;
    }
    float residual = failure == kFailNone ? 0.0f : FLT_MAX;
    if (failure != kFailNone && lane == 0u) d.env_status[c.env] |= kEnvStatusSolverFailure;
    if constexpr (kFollow) {   // the followers' part of M^-1 (balance, 0) is -P times the block's part
        const float follow = failure == kFailNone ? mass_times<N>(c, mrow, coordinate ? direction : 0.0f) : 0.0f;
        if (follower) direction = follow;
    }
    const bool moving = coordinate || follower;
    if (failure == kFailNone && moving) residual = fmaxf(residual, isfinite(direction) ? fabsf(direction) : FLT_MAX);
    residual = wave_max(residual);
    c.residual = fmaxf(c.residual, residual);
    if (reconstruct && failure == kFailNone) {
        if (!__all(!moving || isfinite(*velocity_io + direction))) { c.residual = FLT_MAX; return; }
        if (moving) *velocity_io += direction;
        c.momentum = fmaxf(c.momentum, residual);
    }
}

// InitializeTileResiduals (:890-930) on the staged rows: residual = fl(rhs dt) - J u, products summed in coordinate order
template <int N>
__device__ __forceinline__ void initialize_residuals(const Tile& c, float velocity, const float* urows, float dt) {
    float* dvec = c.vec;
    dvec[c.lane] = c.lane < c.n ? velocity : 0.0f;
    lds_sync<N>();
    const float4* d4 = reinterpret_cast<const float4*>(dvec);
    float motion[6] = {};   // of the link of lane's head, where the rows follow from the links
    if constexpr (N > kTwoWaveWidth) {
        if (c.from_links) link_motion<N>(c, c.lane < c.heads ? way_of(c, c.lane) : 0ull, dvec, motion);
    }
    for (uint32_t h = c.lane; h < c.heads; h += kWave) {
        const uint32_t slot = c.slot(h), stride = c.U(hStride, h), axes = c.U(hAxes, h);
        const uint32_t unit = kPaired ? kInvalid : c.U(hUnit, h), first = c.U(hRow, h);
        if (unit != kInvalid || first == kInvalid) {   // one coordinate (or none): every other product is an exact zero
            const float along = unit != kInvalid ? c.F(hUnitValue, h) * dvec[unit] : 0.0f;
            c.F(hRes, h) = urows[size_t{slot} * kRowWords + 4u] * dt - (0.0f + along);
            c.F(hRes + 1, h) = 0.0f; c.F(hRes + 2, h) = 0.0f;
            continue;
        }
        if constexpr (N > kTwoWaveWidth) {
            if (c.from_links) {
                for (uint32_t axis = 0u; axis < 3u; ++axis)
                    c.F(hRes + axis, h) = axis < axes ? urows[size_t{slot + axis * stride} * kRowWords + 4u] * dt - wrench_dot(c, h, axis, motion) : 0.0f;
                continue;
            }
        }
        for (uint32_t axis = 0u; axis < 3u; ++axis) {
            float residual = 0.0f;
            if (axis < axes) {
                const float rhs = urows[size_t{slot + axis * stride} * kRowWords + 4u];
                const float4* j4 = reinterpret_cast<const float4*>(c.jac + (first + axis) * uint32_t(N));
                float along = 0.0f;
#pragma unroll
                for (int q = 0; q < N / 4; ++q) {
                    const float4 j = j4[q], dv = d4[q];
                    along = along + j.x * dv.x; along = along + j.y * dv.y; along = along + j.z * dv.z; along = along + j.w * dv.w;
                }
                residual = rhs * dt - along;
            }
            c.F(hRes + axis, h) = residual;
        }
    }
    lds_sync<N>();
}

struct DualMomentum { float t, beta; };

// UpdateTileHeadDuals (:2493-2595); classes = {normal, tangent, joint}
__device__ __forceinline__ void update_duals(const Tile& c, float* lambda_env, uint32_t R, const float* urows, DualMomentum* momentum, bool velocity,
                             bool commit, float* classes) {
    uint32_t steps[3] = {0u, 0u, 0u};
    double restart = 0.0;
    for (uint32_t h = c.lane; h < c.heads; h += kWave) {
        const uint32_t slot = c.slot(h), local = slot - c.env * R, stride = c.U(hStride, h), axes = c.U(hAxes, h);
        const bool contact = block_axes(axes);
        const bool elliptic = c.elliptic && axes == kAxesElliptic;
        const float rho = c.F(hRho, h), compliance = c.F(hCompliance, h), lower = c.F(hLower, h), upper = c.F(hUpper, h);
        const float mu1 = c.F(hMu1, h), mu2 = c.F(hMu2, h);
        const Response response{c.F(hDualScale, h), c.F(hResidualScale, h)};
        const V3 residual{c.F(hRes, h), c.F(hRes + 1, h), c.F(hRes + 2, h)};
        const V3 base{c.F(hBase, h), c.F(hBase + 1, h), c.F(hBase + 2, h)};
        const V3 tdual = commit ? V3{c.F(hDual, h), c.F(hDual + 1, h), c.F(hDual + 2, h)} : base;
        float normal, ncurv;
        scalar_impulse(tdual.x, rho, residual.x, compliance, lower, upper, response, &normal, &ncurv);
        V3 dual{normal, 0.0f, 0.0f};
        V3 rstep{0, 0, 0}, rpoint{0, 0, 0};
        float rweight = 0.0f;
        EllipticResponse cone{};
        if (elliptic) {   // :2509-2510: the projection onto the elliptic cone as it is
            const EllipticLine line = elliptic_line(cone_of(c, h), tdual);
            cone = line.k.e;
            float f[3], cv[6];
            elliptic_impulse(line, residual.x, residual.y, residual.z, f, cv);
            dual = V3{f[0], f[1], f[2]};
        } else if (contact) {   // ProjectRowDual (block_descent.cu:799-804) with RelaxContactImpulse (augmented_row.hpp:128-138)
            float fy, fz, cyy, czz, cyz;
            tangent_impulse(tdual, rho, residual.y, residual.z, normal, mu1, mu2, &fy, &fz, &cyy, &czz, &cyz);
            const V3 next{normal, fy, fz};
            V3 last_step{0, 0, 0}, last_point{0, 0, 0};
            float last_weight = 0.0f;
            if (commit) {
                last_step = V3{c.F(hRelaxStep, h), c.F(hRelaxStep + 1, h), c.F(hRelaxStep + 2, h)};
                last_weight = c.F(hRelaxWeight, h);
                last_point = V3{c.F(hRelaxPoint, h), c.F(hRelaxPoint + 1, h), c.F(hRelaxPoint + 2, h)};
            }
            const V3 step{next.x - tdual.x, next.y - tdual.y, next.z - tdual.z};
            const V3 change{step.x - last_step.x, step.y - last_step.y, step.z - last_step.z};
            const V3 moved = sub3(tdual, last_point);
            const float square = change.x * change.x + change.y * change.y + change.z * change.z;
            const float along = -(moved.x * change.x + moved.y * change.y + moved.z * change.z);
            float weight = 1.0f;
            if (last_weight > 0.0f && along > 0.0f && square > 0.0f) weight = fminf(1.0f, along / square);
            rstep = step; rweight = weight; rpoint = tdual;
            dual = V3{tdual.x + weight * step.x, tdual.y + weight * step.y, tdual.z + weight * step.z};
        }
        // MultiplierSteps (block_descent.cu:761-770)
        float step_normal = response.residual_scale > 0.0f && response.dual_scale != 0.0f
            ? fabsf(dual.x - tdual.x) / response.residual_scale : 0.0f;
        float step_tangent = 0.0f;
        if (contact) {
            const float fs = fmaxf(mu1, mu2);
            const float m1 = mu1 <= 0.0f ? 0.0f : mu1 / fs, m2 = mu2 <= 0.0f ? 0.0f : mu2 / fs;
            const float first = m1 > 0.0f && rho > 0.0f ? (dual.y - tdual.y) / (rho * m1 * m1) : 0.0f;
            const float second = m2 > 0.0f && rho > 0.0f ? (dual.z - tdual.z) / (rho * m2 * m2) : 0.0f;
            step_tangent = hypotf(first, second);
        }
        if (!commit && response.residual_scale > 0.0f) step_normal = fabsf(dual.x - tdual.x) / response.residual_scale;
        if (elliptic) {   // EllipticMultiplierStep (augmented_row.hpp:104-108; :2516-2519)
            step_normal = fabsf(dual.x - tdual.x) / cone.kx;
            step_tangent = fmaxf(fabsf(dual.y - tdual.y) / cone.ky, fabsf(dual.z - tdual.z) / cone.kz);
        }
        const V3 physical = commit ? dual : tdual;
        if (!contact) {
            const bool normal_row = (__float_as_uint(urows[size_t{slot} * kRowWords]) & kRowContactNormal) != 0u;
            const float rate = -residual.x + compliance * physical.x;
            const float violation = physical.x > 0.0f ? fabsf(rate) : fmaxf(-rate, 0.0f);
            const float value = normal_row ? fmaxf(step_normal, violation) : step_normal;
            if (normal_row) steps[0] = max(steps[0], residual_bits(value));
            else steps[2] = max(steps[2], residual_bits(value));
        } else {
            if (commit) {
                if (!elliptic) {   // an elliptic head keeps its tangent compliances where the others keep this state
                    c.F(hRelaxStep, h) = rstep.x; c.F(hRelaxStep + 1, h) = rstep.y; c.F(hRelaxStep + 2, h) = rstep.z;
                    c.F(hRelaxWeight, h) = rweight;
                    c.F(hRelaxPoint, h) = rpoint.x; c.F(hRelaxPoint + 1, h) = rpoint.y; c.F(hRelaxPoint + 2, h) = rpoint.z;
                }
                lambda_env[local + stride] = dual.y;
                lambda_env[local + 2u * stride] = dual.z;
            }
            if (elliptic) {   // :2539-2542
                steps[0] = max(steps[0], residual_bits(step_normal));
                steps[1] = max(steps[1], residual_bits(step_tangent));
            } else {
                const V3 v{-residual.x + compliance * physical.x, -residual.y, -residual.z};
                steps[0] = max(steps[0], residual_bits(physical.x > 0.0f ? fabsf(v.x) : fmaxf(-v.x, 0.0f)));
                steps[1] = max(steps[1], residual_bits(fmaxf(step_tangent, fmaxf(along_axis(physical.y, v.y), along_axis(physical.z, v.z)))));
            }
        }
        if (!commit) continue;
        if (velocity) lambda_env[local] = dual.x;
        const bool extrapolate = contact || response.dual_scale != 0.0f;
        if (extrapolate) {   // MultiplierMetric (block_descent.cu:790-795) and MultiplierMomentumRestart (augmented_row.hpp:119-124)
            const float friction = fmaxf(mu1, mu2);
            const float first = contact && mu1 > 0.0f ? mu1 / friction : 0.0f;
            const float second = contact && mu2 > 0.0f ? mu2 / friction : 0.0f;
            V3 metric{response.residual_scale, rho * first * first, rho * second * second};
            if (elliptic) metric = V3{cone.kx, cone.ky, cone.kz};   // :2555-2557
            restart += (metric.x > 0.0f ? (double(tdual.x) - dual.x) * (double(dual.x) - base.x) / metric.x : 0.0) +
                       (metric.y > 0.0f ? (double(tdual.y) - dual.y) * (double(dual.y) - base.y) / metric.y : 0.0) +
                       (metric.z > 0.0f ? (double(tdual.z) - dual.z) * (double(dual.z) - base.z) / metric.z : 0.0);
        }
        if (momentum != nullptr) { c.F(hMove, h) = base.x; c.F(hMove + 1, h) = base.y; c.F(hMove + 2, h) = base.z; }
        c.F(hDual, h) = dual.x; c.F(hDual + 1, h) = dual.y; c.F(hDual + 2, h) = dual.z;
        c.F(hBase, h) = dual.x; c.F(hBase + 1, h) = dual.y; c.F(hBase + 2, h) = dual.z;
    }
    classes[0] = __uint_as_float(wave_max_u(steps[0]));
    classes[1] = __uint_as_float(wave_max_u(steps[1]));
    classes[2] = __uint_as_float(wave_max_u(steps[2]));
    restart = wave_sum_d(restart);
    if (momentum != nullptr) {
        // AdvanceDualMomentum (block_descent.cu:780-788) and ExtrapolateDual (:808-820)
        if (restart > 0.0) momentum->t = 1.0f;
        const float t = 0.5f * (1.0f + sqrtf(fmaf(4.0f * momentum->t, momentum->t, 1.0f)));
        momentum->beta = (momentum->t - 1.0f) / t;
        momentum->t = t;
        for (uint32_t h = c.lane; h < c.heads; h += kWave) {
            const bool contact = block_axes(c.U(hAxes, h));
            const bool extrapolate = contact || c.F(hDualScale, h) != 0.0f;
            const float beta = extrapolate ? momentum->beta : 0.0f;
            const V3 base{c.F(hMove, h), c.F(hMove + 1, h), c.F(hMove + 2, h)};
            const V3 next{c.F(hBase, h), c.F(hBase + 1, h), c.F(hBase + 2, h)};
            V3 out = next;
            if (beta != 0.0f) {
                V3 y{fmaf(beta, next.x - base.x, next.x), fmaf(beta, next.y - base.y, next.y), fmaf(beta, next.z - base.z, next.z)};
                y.x = fminf(fmaxf(y.x, c.F(hLower, h)), c.F(hUpper, h));
                if (!contact) out = V3{y.x, 0.0f, 0.0f};
                else {
                    const float mu1 = c.F(hMu1, h), mu2 = c.F(hMu2, h);
                    const float first = mu1 > 0.0f ? y.y / mu1 : 0.0f, second = mu2 > 0.0f ? y.z / mu2 : 0.0f;
                    const float slip = hypotf(first, second), radius = fmaxf(y.x, 0.0f);
                    const float scale = slip > radius ? radius / slip : 1.0f;
                    out = V3{y.x, mu1 > 0.0f ? y.y * scale : 0.0f, mu2 > 0.0f ? y.z * scale : 0.0f};
                }
            }
            c.F(hDual, h) = out.x; c.F(hDual + 1, h) = out.y; c.F(hDual + 2, h) = out.z;
        }
    }
    wave_sync();
}

__host__ __device__ inline uint32_t PaddedWidth(uint32_t n) { return (n + 3u) & ~3u; }
// `n`: the width the solve works at - the block's coordinates, or the K of a reduced block
// The factor of the Newton Hessian, and at the widths that run two waves a SIMD the factor of the mass matrix beside
// it; wider blocks keep the mass factor, which a solve reads a few times a sweep, in device memory instead
// (DataView::solver_mass_factor), so that two of them fit a compute unit's LDS.
__host__ __device__ inline bool MassFactorInMemory(uint32_t n) { return PaddedWidth(n) > uint32_t(kTwoWaveWidth); }
__host__ __device__ inline uint32_t FactorRegionFloats(uint32_t n) {
    if (kPaired) return 0u;
    const uint32_t N = PaddedWidth(n);
    return (MassFactorInMemory(n) ? 1u : 2u) * FactorFloats(N);   // a multiple of 4
}
// what the set-up of a reduced block passes through LDS ahead of everything else: the eliminated coordinates' factor
// and their coupling to the others, transposed
__host__ __device__ inline uint32_t ReductionScratchFloats(uint32_t full, uint32_t reduced) {
    const uint32_t N = PaddedWidth(full);
    return reduced >= full ? 0u : 2u * (N - reduced) * N;   // doubles
}
// the coordinates' motion axes of a wide block (Tile::axes), twelve words a coordinate
__host__ __device__ inline uint32_t LinkAxisFloats(uint32_t n) { return PaddedWidth(n) > uint32_t(kTwoWaveWidth) ? 12u * uint32_t(kWave) : 0u; }
// the kept Hessian rows of a narrow block (Tile::hrows), and the second floats of a reduced block's mass rows (Tile::low)
__host__ __device__ inline uint32_t KeptRowFloats(uint32_t n, bool reduced) {
    const uint32_t N = PaddedWidth(n);
    return N > 32u ? 0u : (reduced ? 2u : 1u) * N * N;
}
constexpr uint32_t kVectorFloats = kPaired ? kTurnFloats : 4u * uint32_t(kWave);   // Tile::vec
// the coordinates' lists of their unit heads, sixteen bits a place
__host__ __device__ inline uint32_t UnitListFloats(uint32_t cap, uint32_t staged) { return cap > staged ? kUnitSlots * uint32_t(kWave) / 2u : 0u; }
__host__ __device__ inline uint32_t HeadFieldFloats(uint32_t cap, uint32_t narrow) {
    return (kWideStride * cap + kNarrowStride * (narrow + 1u) + 3u) & ~3u;
}
// `cap` heads carry fields; `staged` of them (the contact heads) carry three Jacobian rows each.
// A block that keeps no contact rows (the world's contact rows each act through one link, ModelView::rows_from_links;
// a wide block of contact heads only) holds a wrench record a head in their place.
__host__ __device__ inline bool RowsFromLinks(uint32_t n, bool contacts_only, uint32_t world_flag) {
    return PaddedWidth(n) > uint32_t(kTwoWaveWidth) && contacts_only && world_flag != 0u;
}
__host__ __device__ inline uint32_t RowFloats(uint32_t N, uint32_t staged, bool from_links) {
    return from_links ? (kWrenchStride * staged + 3u) & ~3u : 3u * staged * N;
}
__host__ __device__ inline uint32_t SolverLdsFloats(uint32_t n, uint32_t cap, uint32_t staged, bool from_links = false, bool reduced = false) {
    const uint32_t N = PaddedWidth(n);
    // the per-coordinate unit lists exist only when some head beyond the staged ones can be listed; without joint rows
    // the block keeps the footprint that lets eight of them share a compute unit's LDS
    return FactorRegionFloats(n) + RowFloats(N, staged, from_links) + HeadFieldFloats(cap, staged) + kVectorFloats +
           UnitListFloats(cap, staged) + LinkAxisFloats(n) + KeptRowFloats(n, reduced);
}
__host__ __device__ inline uint32_t ReducedSolverLdsFloats(uint32_t full, uint32_t reduced, uint32_t cap, uint32_t staged, bool from_links = false) {
    const uint32_t solve = SolverLdsFloats(reduced, cap, staged, from_links, reduced < full), scratch = ReductionScratchFloats(full, reduced);
    return solve > scratch ? solve : scratch;
}

// DescendTile (:2941-3087).  kContactsOnly is the instantiation for worlds without joint rows whose heads fit one a
// lane (cap <= 64, every head a staged contact head): the unit-head paths and the loops over heads beyond the first
// 64 are compiled out, which leaves the hot loop shorter and with fewer values to keep live.  kElliptic is whether heads may be
// under the elliptic cone.
// The set-up of a reduced block, in double.  Lane i < n comes with row i of the mass matrix at `mass` (md words a row).
// The coordinates N-1 .. K are eliminated leaves first (FactorTileColumns' order): the lanes below K are left with
// their rows of the Schur complement S = M_TT - M_TU M_UU^-1 M_UT and of U_TU = M_TU U_UU^-T, the followers with their
// rows of the factor M_UU = U_UU U_UU^T.  P = M_UU^-1 M_UT = U_UU^-T U_TU^T then follows by forward substitution over the
// followers in ascending order, a column of P a lane, which passes through LDS to be read by rows.  On return a lane below K
// holds its row of S as the sum of two floats, mrow in registers and the second in LDS at `low` (read by low_row), a
// follower its row of -P rounded to float in mrow.
// Double because these rows stand in for the mass matrix over the whole solve: a Schur complement eliminated in
// single precision moves the velocities the solve converges to by a few 1e-5 of the contact impulse's effect.
template <int N, int K>
__device__ __forceinline__ bool reduce_block(uint32_t lane, uint32_t n, const float* mass, uint32_t md, float* lds, float* low, float (&mrow)[K]) {
    constexpr int kFollowers = N - K;
    const bool row_lane = lane < n;
    double full[N];
    {
        float fetched[N];
        if (md % 4u == 0u && md >= uint32_t(N)) {
#pragma unroll
            for (int q = 0; q < N / 4; ++q) {
                const float4 m4 = reinterpret_cast<const float4*>(mass)[q];
                fetched[4 * q] = m4.x; fetched[4 * q + 1] = m4.y; fetched[4 * q + 2] = m4.z; fetched[4 * q + 3] = m4.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < N; ++k) fetched[k] = uint32_t(k) < n ? mass[k] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < N; ++k)   // rows and columns n..N-1 are those of the identity
            full[k] = row_lane && uint32_t(k) < n ? double(fetched[k]) : (lane == uint32_t(k) && lane < uint32_t(N) ? 1.0 : 0.0);
    }
    const uint32_t at = local_lane(lane);
    bool valid = true;
    double own_scale = 0.0;
#pragma unroll
    for (int k = N - 1; k >= K; --k) {
        const double pivot = lane_value_d(full[k], k);
        valid = valid && pivot > 0.0 && pivot <= double(FLT_MAX);
        // the reciprocal root: the single-precision approximation and two Newton steps
        const double safe = valid ? pivot : 1.0;
        double scale = double(__builtin_amdgcn_rsqf(float(safe)));
        scale = scale * fma(-0.5 * safe, scale * scale, 1.5);
        scale = scale * fma(-0.5 * safe, scale * scale, 1.5);
        full[k] = at == uint32_t(k) ? safe * scale : full[k] * scale;
        if (at == uint32_t(k)) own_scale = scale;
        const uint64_t reach = __ballot(at < uint32_t(k) && full[k] != 0.0);
#pragma unroll
        for (int q = (k - 1) / 4; q >= 0; --q) {
            if (((reach >> (4 * q)) & 0xFull) == 0ull) continue;
            double u[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) u[t] = 4 * q + t <= k - 1 ? lane_value_d(full[k], 4 * q + t) : 0.0;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (4 * q + t <= k - 1) full[4 * q + t] = fma(-full[k], u[t], full[4 * q + t]);
        }
    }
    double* solved = reinterpret_cast<double*>(lds);      // [follower][coordinate below K]: what the substitution ends with
    double* corner = solved + kFollowers * K;             // [follower i][follower k]: U_UU[i][k] right of the diagonal, 1 / U_UU[i][i] on it
    if (lane >= uint32_t(K) && lane < uint32_t(N)) {
#pragma unroll
        for (int k = K; k < N; ++k) corner[(int(lane) - K) * kFollowers + (k - K)] = full[k];
        corner[(int(lane) - K) * (kFollowers + 1)] = own_scale;
    }
    lds_sync<K>();
    // lane = coordinate below K: its own entries of U_TU are a column of the coupling, and the substitution runs down them with the
    // factor's rows the same for every lane, two entries a read.  (A lane a follower, column after column, each a chain of lane
    // reads, took 1.3 k instructions where this takes 250: 65536 humanoids 7570 -> 7512 us, 4096 704 -> 699, the bits the same.)
#pragma unroll
    for (int j = 0; j < kFollowers; ++j) {
        uint32_t from = uint32_t(j * kFollowers);
        if (j > 0) asm volatile("" : "+v"(from) : "v"(full[K + j - 1]));   // (two rows' words in registers at a time, not all of them)
        const double2* row = reinterpret_cast<const double2*>(corner + from);
#pragma unroll
        for (int q = j / 2; q < kFollowers / 2; ++q) {
            const double2 u = row[q];
            if (2 * q == j) full[K + j] *= u.x;
            if (2 * q + 1 == j) full[K + j] *= u.y;
            if (2 * q > j) full[K + 2 * q] = fma(u.x, -full[K + j], full[K + 2 * q]);
            if (2 * q + 1 > j) full[K + 2 * q + 1] = fma(u.y, -full[K + j], full[K + 2 * q + 1]);
        }
    }
    if (lane < uint32_t(K)) {
#pragma unroll
        for (int i = 0; i < kFollowers; ++i) solved[i * K + int(lane)] = full[K + i];
    }
    lds_sync<K>();
    const uint32_t slot = lane >= uint32_t(K) && lane < uint32_t(N) ? lane - uint32_t(K) : 0u;
#pragma unroll
    for (int q = 0; q < K / 2; ++q) {
        const double2 v = reinterpret_cast<const double2*>(solved + slot * uint32_t(K))[q];
        full[2 * q] = lane >= uint32_t(K) ? -v.x : full[2 * q];
        full[2 * q + 1] = lane >= uint32_t(K) ? -v.y : full[2 * q + 1];
    }
    float rest[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double entry = lane < uint32_t(K) || lane < n ? full[k] : 0.0;
        mrow[k] = float(entry);
        rest[k] = float(entry - double(mrow[k]));
        asm volatile("" : "+v"(mrow[k]));   // (or the double stays beside the float over the sweeps, in registers they need)
    }
    if (lane < uint32_t(K)) {   // (the scratch above has been read: its words may be these)
        float4* words = reinterpret_cast<float4*>(low + lane * uint32_t(K));
#pragma unroll
        for (int q = 0; q < K / 4; ++q) words[q] = float4{rest[4 * q], rest[4 * q + 1], rest[4 * q + 2], rest[4 * q + 3]};
    }
    lds_sync<K>();
    return valid;
}

// K < N is a reduced block (described above mass_times): no contact of the world reaches the coordinates K..n-1, which are
// eliminated once in the set-up, and the sweeps run K wide.  K is a multiple of 4 with K <= n, contact heads only.
//   An environment a block, or (kQueue, every dense instantiation), where environments outnumber the blocks the machine holds at once,
// as many blocks as it holds, each of which takes the next place of the launch order (DataView::solver_queue, cleared by the order's
// launch) when it is done.  Blocks of a launch are handed out in turns to the parts of the machine, and one whose part is full holds up those
// behind it: with solves of unequal length a launch of 8192 blocks kept four fifths of the places busy.  The first places are the
// blocks' own, so that the costliest environments start where a launch of all of them would start them.  Instantiations of their own,
// for what a solve keeps in registers over the loop costs the others a per cent (4096 walkers 304 -> 308 us a step).
constexpr uint32_t kQueued = kInvalid - 1u;   // in the place of a launch's largest number of points: points_lo blocks and a queue
struct SolveArguments { ModelView m; DataView d; BlockDescentSolveParams p; };   // the first of the kernel's arguments as they lie in memory
template <int N, bool kContactsOnly, int K = N, bool kElliptic = !kContactsOnly, bool kQueue = kDense>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(WavesPerSimd(K), WavesPerSimd(K))))
BlockDescentTileKernel(ModelView model, DataView data, BlockDescentSolveParams params, uint32_t cap, uint32_t staged_cap, uint32_t lowest,
                       uint32_t highest) {
    constexpr bool kReduced = K < N;
    constexpr int W = K;   // the width of the sweeps
    static_assert(K % 4 == 0 && K <= N && (!kReduced || kContactsOnly), "a reduced block holds contact heads only");
    extern __shared__ __align__(16) float lds[];
    uint32_t place = blockIdx.x;
environment:
    auto arguments = (const __attribute__((address_space(4))) SolveArguments*)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t lane = threadIdx.x;
    if constexpr (kQueue) {
        // They come anew for every environment: what follows from them would otherwise be made once, ahead of the loop, and kept in
        // registers that a solve does not have.
        lane = 0u;
        asm volatile("" : "+s"(arguments), "+s"(lane));
        lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, lane));
    }
    const ModelView& m = kQueue ? ((const SolveArguments*)arguments)->m : model;
    const DataView& d = kQueue ? ((const SolveArguments*)arguments)->d : data;
    const BlockDescentSolveParams& p = kQueue ? ((const SolveArguments*)arguments)->p : params;
    const uint32_t env = d.tile_order[place];
    // A world whose contact slots outnumber the contacts it usually has is solved by two launches of different LDS
    // capacity; each takes the environments whose contact points fall in its range and leaves the others at once.
    if (!(kQueue && highest == kQueued) && (lowest != 0u || highest != kInvalid)) {
        const uint32_t points = d.contact_count[env];
        if (points < lowest || points > highest) return;
    }
    const uint32_t R = p.rows_per_env, md = p.max_dof, n = m.dof, nl = m.links_per_env, S = p.contact_slots_per_env;
    // A narrow block would leave registers free and let more waves share a SIMD than the launch is sized for; one name of
    // the last register holds the kernel to its two (dense build: three or four) waves.  (Behind the place's own words, which
    // are scalar reads only ahead of it.)
    if constexpr (WavesPerSimd(W) == 4) asm volatile("" ::: "v127");
    else if constexpr (WavesPerSimd(W) == 3) asm volatile("" ::: "v163");
    else if constexpr (WavesPerSimd(W) == 2) asm volatile("" ::: "v255");
    Tile c;
    c.env = env; c.lane = lane; c.n = kReduced ? uint32_t(K) : n; c.n_all = n; c.ldj = uint32_t(W); c.cap = cap; c.narrow = staged_cap; c.heads = 0u; c.iteration = 0u;
    c.tolerance = p.velocity_tolerance; c.failed = false; c.momentum = 0.0f; c.residual = 0.0f;
    c.scalar_later = false; c.near_heads = false; c.block_heads = false; c.mass_inverse = 0.0f; c.mass_valid = false; c.work = 0u; c.units = false; c.elliptic = false;
    c.factor_current = false; c.rows_current = false; c.factor_root = 1.0f; c.smooth = kElliptic;
    for (float& entry : c.curvature) entry = 0.0f;
#ifdef NKH_SOLVER_PROFILE
    for (int i = 0; i < 32; ++i) c.prof[i] = 0;
    for (int i = 0; i < 4; ++i) c.prof_count[i] = 0u;
    const long long prof_wall_start = wall_clock64();
#endif
    PROF_BEGIN(c, 9);
    PROF_BEGIN(c, 0);
    if constexpr (W > kTwoWaveWidth) {
        c.mfac = d.solver_mass_factor + size_t{env} * FactorFloats(uint32_t(W));
        c.hfac = lds;
    } else {
        c.mfac = lds;
        c.hfac = c.mfac + FactorFloats(uint32_t(W));
    }
    c.from_links = kPaired || RowsFromLinks(uint32_t(W), kContactsOnly, m.rows_from_links);
    c.jac = lds + FactorRegionFloats(uint32_t(W));
    c.wrench = c.jac;   // one or the other
    c.fields = c.jac + RowFloats(uint32_t(W), staged_cap, c.from_links);
    c.vec = c.fields + HeadFieldFloats(cap, staged_cap);
    if constexpr (kPaired) c.hfac = c.vec;   // what the set-up passes through the factor's place
    c.hrows = c.vec + kVectorFloats + UnitListFloats(cap, staged_cap);
    c.low = c.hrows + uint32_t(W) * uint32_t(W);
    // The block's mass rows: lane's row of M, or in a reduced block lane's row of the Schur complement (lanes below K)
    // and of -P (the followers).
    float mrow[W];
    bool reduction_valid = true;
    if constexpr (kReduced) {
        PROF_BEGIN(c, 30);
        reduction_valid = reduce_block<N, K>(lane, n, d.m + size_t{env} * md * md + size_t{lane < n ? lane : 0u} * md, md, lds, c.low, mrow);
        PROF_END(c, 30);
    }
    if (lane < kNarrowFields) c.fields[kWideStride * cap + staged_cap * kNarrowStride + lane] = 0.0f;   // what a narrow field reads beyond its heads
    c.unit_list = reinterpret_cast<uint16_t*>(c.vec + kVectorFloats);
    c.unit_lists = true; c.unit_count = 0u; c.unit_most = 0u; c.staged_end = 0u; c.individual_end = 0u;
    c.through_links = false; c.over_runs = false; c.way_runs = false;
    c.axes = c.vec + kVectorFloats + UnitListFloats(cap, staged_cap);   // a wide block's; a narrow one keeps rows here
    c.path_low = c.path_high = c.under_low = c.under_high = c.over_low = c.over_high = 0u;
    c.stiffness_current = false;
    c.rows = d.urows; c.row_point_a = d.row_cj_point; c.row_point_b = d.row_cj_point_b;
    c.pivot = V3{0.0f, 0.0f, 0.0f};
    const bool coordinate = lane < n;
    const float* urows = d.urows;
    float* lambda_env = d.lambda + size_t{env} * R;
    const size_t lbase = size_t{env} * nl;
    // InitializeTile (:1327-1350): the free velocity and the constraint velocity carried from the previous solve
    uint32_t my_link = 0u, my_component = kInvalid;
    float free_v = 0.0f, velocity = 0.0f;
    if (coordinate) {
        my_link = m.dof_link[lane]; my_component = m.dof_component[lane];
        const float value = my_component == kInvalid ? d.qdot[lbase + my_link] : d.link_velocity[(lbase + my_link) * 6u + my_component];
        const float carried = d.solver_velocity[size_t{env} * md + lane] - d.solver_free[size_t{env} * md + lane];
        free_v = value;
        velocity = value + (isfinite(carried) ? carried : 0.0f);
    }
    PROF_BEGIN(c, 16);
    // ListTileHeads (:1250-1296): active rows that are not block tangents, in slot order
    // The reference scans the rows below the larger of the last two row extents (all of them when either is unknown,
    // as after a reset).  The rows between this step's extent and that bound were cleared by this step's row assembly
    // and hold no head, so the scan stops at this step's extent: the same heads from a fraction of the row records.
    const uint32_t current = d.contact_row_extent[2u * env + 1u];
    const uint32_t bound = current == 0u ? p.contact_rows_per_env : min(current - 1u, p.contact_rows_per_env);
    const uint32_t total = bound + (R - p.contact_rows_per_env);
    uint32_t heads = 0u, contact_heads = 0u;   // the latter among the former
    bool overflow = false;
    for (uint32_t base = 0u; base < total; base += kWave) {
        const uint32_t index = base + lane;
        const uint32_t slot = env * R + (index < bound ? index : p.contact_rows_per_env + (index - bound));
        bool head = false;
        if (index < total) {
            const uint32_t flags = __float_as_uint(urows[size_t{slot} * kRowWords]);
            head = (flags & kRowActive) != 0u && (flags & kRowBlockTangent) == 0u;
        }
        const uint64_t mask = __ballot(head);
        if (head) {
            const uint32_t at = heads + __popcll(mask & ((uint64_t{1} << lane) - 1u));
            if (at < cap) c.U(hSlot, at) = slot; else overflow = true;
        }
        heads += __popcll(mask);
        contact_heads += __popcll(mask & (bound >= base + kWave ? ~uint64_t{0} : bound > base ? (uint64_t{1} << (bound - base)) - 1u : uint64_t{0}));
    }
    if (__any(overflow)) {   // more heads than the staged LDS holds: fail loudly, solve the ones that fit
        heads = cap;
        contact_heads = min(contact_heads, cap);
        if (lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
    }
    if constexpr (kContactsOnly) __builtin_assume(heads <= uint32_t(kWave));
    c.heads = heads;
    lds_sync<W>();
    PROF_END(c, 16);
    PROF_BEGIN(c, 17);
    // stage Jacobian rows: the sum of the articulated sides' chain rows (TileBlock::Jacobian :555-573, CopyTileRows :836-869).
    // First every (head, axis) row finds its source rows, one per lane; then the copies run with their loads in flight
    // together instead of one row's latency after another.
    // (the contact rows' heads have up to three rows, those of the joint rows, which all come after them, one)
    const uint32_t fan_out = 3u * contact_heads, sources = fan_out + (heads - contact_heads);
    for (uint32_t r = lane; r < sources; r += kWave) {
        const bool contact = r < fan_out;
        const uint32_t h = contact ? r / 3u : r - 2u * contact_heads, axis = contact ? r - 3u * h : 0u;
        const uint32_t slot = c.slot(h);
        const uint32_t flags = __float_as_uint(urows[size_t{slot} * kRowWords]);
        const uint32_t stride = __float_as_uint(urows[size_t{slot} * kRowWords + 2u]);
        const uint32_t axes = contact && h < staged_cap && (flags & kRowBlockNormal) != 0u ? 3u : 1u;   // (one past the staged heads' room)
        uint32_t source_a = kInvalid, source_b = kInvalid;
        if (axis < axes) {
            const uint32_t rs = slot + axis * stride;
            if (__float_as_uint(urows[size_t{rs} * kRowWords + 10u]) == kSideArtic) source_a = rs;
            if (__float_as_uint(urows[size_t{rs} * kRowWords + 18u]) == kSideArtic) source_b = rs;
        }
        c.U(hSourceA + axis, h) = source_a; c.U(hSourceB + axis, h) = source_b;
        if (contact) continue;
#pragma unroll
        for (uint32_t k = 1u; k < 3u; ++k) { c.U(hSourceA + k, h) = kInvalid; c.U(hSourceB + k, h) = kInvalid; }
    }
    lds_sync<W>();
    PROF_BEGIN(c, 22);
    // FindTileRowSupport (:801-833), lane = head: a single-axis head whose Jacobian row has at most one entry is a unit
    // head and stages nothing; every other owned head stages three rows, placed in head order (PlaceTileRows).
    {
        // a single-axis head acting on one coordinate is a unit head; the rows carry that coordinate and its entry
        // from where they were emitted (row_unit, row_unit_value), which is what a scan of the head's Jacobian row
        // for its entries would find
        bool overflow_rows = false;
        for (uint32_t base = 0u; base < heads; base += kWave) {
            const uint32_t h = base + lane;
            if (h >= heads) continue;
            const uint32_t source_a = c.U(hSourceA, h), source_b = c.U(hSourceB, h);
            const bool owned = source_a != kInvalid || source_b != kInvalid;
            // a block head has found the sources of its tangent rows on the sides that move
            const bool single_axis = c.U(hSourceA + 1u, h) == kInvalid && c.U(hSourceB + 1u, h) == kInvalid;
            const uint32_t slot = c.slot(h);
            uint32_t unit = kInvalid;
            float unit_value = 0.0f;
            if (owned && single_axis && d.row_unit[slot] != kInvalid) { unit = d.row_unit[slot]; unit_value = d.row_unit_value[slot]; }
            else if (owned && h >= staged_cap) { overflow_rows = true; unit = 0u; }   // no room for its rows: it acts on nothing, and the solve is flagged
            if constexpr (!kPaired) { c.U(hUnit, h) = unit; c.F(hUnitValue, h) = unit_value; }
            c.U(hRow, h) = owned && unit == kInvalid ? 0u : kInvalid;
            c.U(hColumnsLow, h) = 0u; c.U(hColumnsHigh, h) = 0u;
        }
        if (__any(overflow_rows) && lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
        lds_sync<W>();
        PROF_END(c, 22);
        PROF_BEGIN(c, 23);
        // PlaceTileRows: the staged heads take their rows in head order
        uint32_t staged = 0u, staged_end = 0u, individual_end = 0u, my_units = 0u;
        bool any_unit = false;
        for (uint32_t base = 0u; base < heads; base += kWave) {
            const uint32_t h = base + lane;
            const bool stage = h < heads && c.U(hRow, h) != kInvalid;
            const uint64_t mask = __ballot(stage);
            if (stage) c.U(hRow, h) = 3u * (staged + uint32_t(__popcll(mask & ((uint64_t{1} << lane) - 1ull))));   // no more than h
            staged += uint32_t(__popcll(mask));
            if (mask != 0ull) staged_end = base + uint32_t(64 - __builtin_clzll(mask));
            if constexpr (!kPaired) {
                any_unit = any_unit || (h < heads && c.U(hUnit, h) != kInvalid);
                // heads that need a response of their own: staged ones, and unit heads whose entry is not +-1
                const uint64_t own = __ballot(h < heads && (c.U(hUnit, h) == kInvalid || fabsf(c.F(hUnitValue, h)) != 1.0f));
                if (own != 0ull) individual_end = base + uint32_t(64 - __builtin_clzll(own));
            }
        }
        c.units = !kContactsOnly && __any(any_unit) && cap > staged_cap;   // the lists have room only when the world has joint heads
        c.staged_end = staged_end;
        c.individual_end = individual_end;
        lds_sync<W>();
        // every coordinate lists its own unit heads, in head order
        if (c.units) {
            constexpr uint32_t kAhead = 16u;   // reads in flight
            for (uint32_t h0 = 0u; h0 < heads; h0 += kAhead) {
                uint32_t unit[kAhead];
#pragma unroll
                for (uint32_t t = 0u; t < kAhead; ++t) unit[t] = c.U(hUnit, min(h0 + t, heads - 1u));
#pragma unroll
                for (uint32_t t = 0u; t < kAhead; ++t) {
                    if (unit[t] != lane || h0 + t >= heads) continue;
                    if (my_units < kUnitSlots) c.unit_list[my_units * uint32_t(kWave) + lane] = uint16_t(h0 + t);
                    ++my_units;
                }
            }
            c.unit_lists = !__any(my_units > kUnitSlots);
            c.unit_count = min(my_units, kUnitSlots);
            c.unit_most = wave_max_u(c.unit_count);
        }
        PROF_END(c, 23);
    }
    lds_sync<W>();
    if constexpr (W > kTwoWaveWidth && kContactsOnly) {
        // The coordinates' motion axes about the root link's origin, for add_heads_through_links: a hinge or an angular
        // coordinate of a floating root turns about its axis through the joint's origin, a sliding one moves along it
        // (the columns the row assembly wrote, assemble_rows.cu:122-169, before the dot with a row's direction).
        const float* root = d.link_pose + lbase * 7u;
        c.pivot = V3{root[0], root[1], root[2]};
        float axis[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        uint64_t path = 0ull;
        bool plain = true;
        if (coordinate) {
            V3 along, at;
            bool turning;
            if (my_component == kInvalid) {
                const Xf pose = load_xf(d.link_pose + (lbase + my_link) * 7u);
                along = rotate_normalized(pose.r, V3{m.joint_axis[3u * my_link], m.joint_axis[3u * my_link + 1u], m.joint_axis[3u * my_link + 2u]});
                at = pose.p;
                turning = m.joint_type[my_link] != kPrismatic;
            } else {
                const Xf base = load_xf(d.base_pose + size_t{env} * 7u);
                const uint32_t k = my_component % 3u;
                along = rotate_normalized(base.r, V3{k == 0u ? 1.0f : 0.0f, k == 1u ? 1.0f : 0.0f, k == 2u ? 1.0f : 0.0f});
                at = base.p;
                turning = my_component < 3u;
                plain = my_component < 6u;
            }
            if (turning) {
                const V3 arm = cross3(sub3(at, c.pivot), along);
                axis[0] = along.x; axis[1] = along.y; axis[2] = along.z; axis[3] = arm.x; axis[4] = arm.y; axis[5] = arm.z;
            } else {
                axis[3] = along.x; axis[4] = along.y; axis[5] = along.z;
            }
            path = m.link_dof_mask[my_link];
        }
        float4* table = reinterpret_cast<float4*>(c.axes);
        table[3u * lane] = float4{axis[0], axis[1], axis[2], axis[3]};
        table[3u * lane + 1u] = float4{axis[4], axis[5], 0.0f, 0.0f};
        table[3u * lane + 2u] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        c.path_low = uint32_t(path); c.path_high = uint32_t(path >> 32u);
        uint64_t head_way = 0ull;   // lane = head: the way to the root of the one side that moves
        if (lane < heads) {
            const bool side_a = c.U(hSourceA, lane) != kInvalid, side_b = c.U(hSourceB, lane) != kInvalid;
            if (side_a != side_b) head_way = m.link_dof_mask[(side_a ? d.row_cj_link : d.row_cj_link_b)[c.slot(lane)] - env * nl];
        }
        uint64_t under = 0ull, over = 0ull;
        for (uint32_t i = 0u; i < n; ++i) {   // the coordinates, and the heads, whose way to the root holds i
            const uint64_t holders = __ballot(((path >> i) & 1ull) != 0ull), met = __ballot(((head_way >> i) & 1ull) != 0ull);
            if (lane == i) { under = holders; over = met; }
        }
        c.under_low = uint32_t(under); c.under_high = uint32_t(under >> 32u);
        c.over_low = uint32_t(over); c.over_high = uint32_t(over >> 32u);
        c.over_runs = __all(one_run(over));
        c.way_runs = __all(one_run(head_way));
        // every staged head with exactly one side that moves
        bool one_link = true;
        if (lane < heads) {
            const bool side_a = c.U(hSourceA, lane) != kInvalid, side_b = c.U(hSourceB, lane) != kInvalid;
            one_link = !(side_a && side_b) && (!(side_a || side_b) || c.U(hRow, lane) != kInvalid);
        }
        c.through_links = heads <= uint32_t(kWave) && !c.units && __all(plain && one_link);
        if (c.from_links) {
            // the world was cooked as one whose contact rows each act through one link: an environment that holds
            // anything else was given the wrong kernel
            if (!c.through_links && lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
            // lane = head: its rows as wrenches about the pivot, [(p - o) x n; n] with n the direction of the side that
            // moves, and its way to the root
            if (lane < heads) {
                float* record = c.wrench + lane * kWrenchStride;
                const uint32_t slot = c.slot(lane);
                const float* row = urows + size_t{slot} * kRowWords;
                const uint32_t stride = __float_as_uint(row[2]);
                const uint32_t axes = (__float_as_uint(row[0]) & kRowBlockNormal) != 0u ? 3u : 1u;
                const bool side_a = c.U(hSourceA, lane) != kInvalid, side_b = c.U(hSourceB, lane) != kInvalid;
                const bool second = !side_a;
                for (uint32_t a = 0u; a < 3u; ++a) {
                    float w[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                    if (a < axes && side_a != side_b) {
                        const size_t rs = size_t{slot} + a * stride;
                        const float* side = urows + rs * kRowWords + (second ? 20u : 12u);
                        const float* at = (second ? d.row_cj_point_b : d.row_cj_point) + 3u * rs;
                        const V3 n{side[0], side[1], side[2]};
                        const V3 moment = cross3(sub3(V3{at[0], at[1], at[2]}, c.pivot), n);
                        w[0] = moment.x; w[1] = moment.y; w[2] = moment.z; w[3] = n.x; w[4] = n.y; w[5] = n.z;
                    }
#pragma unroll
                    for (int t = 0; t < 6; ++t) record[6u * a + uint32_t(t)] = w[t];
                }
                c.U(hColumnsLow, lane) = uint32_t(head_way); c.U(hColumnsHigh, lane) = uint32_t(head_way >> 32u);
            }
        }
        lds_sync<W>();
    }
    // CopyTileRows (:836-869): the staged heads' rows, their loads in flight together

    bool stray = false;   // a reduced block: an entry past the block's coordinates
    c.near_heads = true;
    for (uint32_t h0 = 0u; h0 < (c.from_links ? 0u : c.staged_end); h0 += 4u) {   // four heads at a time: 24 reads in flight
        uint32_t first[4];
        float value[4][3];
#pragma unroll
        for (uint32_t t = 0u; t < 4u; ++t) {
            const uint32_t h = h0 + t;
            first[t] = h < c.staged_end ? c.U(hRow, h) : kInvalid;   // a unit head stages nothing and touches no column block
            const bool staged = first[t] != kInvalid;
#pragma unroll
            for (uint32_t axis = 0u; axis < 3u; ++axis) {
                const uint32_t source_a = staged ? c.U(hSourceA + axis, h) : kInvalid, source_b = staged ? c.U(hSourceB + axis, h) : kInvalid;
                const float from_a = coordinate && source_a != kInvalid ? d.chain_jacobian[size_t{source_a} * md + lane] : 0.0f;
                const float from_b = coordinate && source_b != kInvalid ? d.chain_jacobian_b[size_t{source_b} * md + lane] : 0.0f;
                value[t][axis] = (0.0f + from_a) + from_b;
            }
        }
#pragma unroll
        for (uint32_t t = 0u; t < 4u; ++t) {
            const uint32_t h = h0 + t;
            if (h >= c.staged_end) break;
            const bool staged = first[t] != kInvalid;
#pragma unroll
            for (uint32_t axis = 0u; axis < 3u; ++axis)
                if (staged && lane < c.ldj) c.jac[(first[t] + axis) * c.ldj + lane] = value[t][axis];   // padded columns hold zeros
            // the columns this head touches at all: a contact on one limb leaves most coordinates out, and the Hessian
            // update skips their exact-zero products four columns at a time
            uint64_t columns = __ballot(value[t][0] != 0.0f || value[t][1] != 0.0f || value[t][2] != 0.0f);
            if constexpr (kReduced) {
                stray = stray || (columns >> uint32_t(W)) != 0ull;
                columns &= (uint64_t{1} << uint32_t(W)) - 1ull;
            }
            c.near_heads = c.near_heads && (columns >> 32u) == 0ull;
            if (lane == 0u) { c.U(hColumnsLow, h) = uint32_t(columns); c.U(hColumnsHigh, h) = uint32_t(columns >> 32u); }
        }
    }
    // a contact that reaches a coordinate the world's reduction left out: the launch was given the wrong width
    if (stray && lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
    lds_sync<W>();
    PROF_END(c, 17);
    PROF_BEGIN(c, 18);
    // TileInertialResponse (:709-739): J M^-1 J^T of every head's first row through the stored LDL^T factor
    // (ForwardMass + MassDot, articulation_mass.cuh:414-431).  lane = DoF: the unit-lower factor row sits in
    // registers with zeros from the diagonal on, each y_j travels as a scalar lane read, so row i subtracts
    // L_ij y_j for j = 0, 1, ... exactly as the serial loop does; the ordered sum of y_i^2 / D_i follows the same way.
    {
        // Lane's own rows of the mass matrix and of its LDL^T factor (StageTileMass :2127-2142) straight into registers:
        // one row is md contiguous words, so every read of both rows is in flight at once, as 16-byte words where the
        // rows are long enough and aligned for that.
        const size_t tile = size_t{env} * md * md + size_t{coordinate ? lane : 0u} * md;
        const float* factor = d.m_factor + tile;
        const float* mass = d.m + tile;
        float lrow[N];
        if constexpr (kReduced) {   // the mass rows were taken, and reduced, at the start
            if (md % 4u == 0u && md >= uint32_t(N)) {
#pragma unroll
                for (int q = 0; q < N / 4; ++q) {
                    const float4 f4 = reinterpret_cast<const float4*>(factor)[q];
                    lrow[4 * q] = f4.x; lrow[4 * q + 1] = f4.y; lrow[4 * q + 2] = f4.z; lrow[4 * q + 3] = f4.w;
                }
            } else {
#pragma unroll
                for (int k = 0; k < N; ++k) lrow[k] = uint32_t(k) < n ? factor[k] : 0.0f;
            }
        } else {
            float fetched[N];
            if (md % 4u == 0u && md >= uint32_t(N)) {
#pragma unroll
                for (int q = 0; q < N / 4; ++q) {
                    const float4 f4 = reinterpret_cast<const float4*>(factor)[q], m4 = reinterpret_cast<const float4*>(mass)[q];
                    lrow[4 * q] = f4.x; lrow[4 * q + 1] = f4.y; lrow[4 * q + 2] = f4.z; lrow[4 * q + 3] = f4.w;
                    fetched[4 * q] = m4.x; fetched[4 * q + 1] = m4.y; fetched[4 * q + 2] = m4.z; fetched[4 * q + 3] = m4.w;
                }
            } else {
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    lrow[k] = uint32_t(k) < n ? factor[k] : 0.0f;
                    fetched[k] = uint32_t(k) < n ? mass[k] : 0.0f;
                }
            }
#pragma unroll
            for (int k = 0; k < W; ++k)   // rows and columns n..N-1 of the mass matrix are those of the identity
                mrow[k] = coordinate && uint32_t(k) < n ? fetched[k] : (lane == uint32_t(k) && lane < uint32_t(N) ? 1.0f : 0.0f);
        }
        float pivot = 1.0f;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if (coordinate && lane == uint32_t(k)) pivot = lrow[k];
            lrow[k] = coordinate && uint32_t(k) < lane ? lrow[k] : 0.0f;
        }
        // y = L^-1 a, then the ordered sum of y_i^2 / D_i
        auto response = [&](float a) -> float {
#pragma unroll
            for (int j = 0; j < N; ++j) a -= lrow[j] * lane_value(a, j);
            const float term = coordinate ? a * a / pivot : 0.0f;
            float total = 0.0f;
#pragma unroll
            for (int i = 0; i < N; ++i) total += lane_value(term, i);
            return total;
        };
        // Four heads at a time: their substitution chains are independent, and side by side each one's lane reads
        // settle under the others' arithmetic.  A head with one moving side, or with both sides on one owner (:752),
        // wants exactly the staged sum of its two sides' rows.  Unit heads with an entry of +-1 are left to the
        // per-coordinate pass below: y(-e) = -y(e), so every such head of one coordinate has the same response.
        const bool share_units = c.units && c.unit_lists;
        bool by_heads = false;
        if constexpr (W > kTwoWaveWidth && kContactsOnly) {
            if (c.from_links && c.through_links) {
                // Every head at once, lane = head: its first row sits in the lane's registers (the coordinates' axes against
                // the row's wrench), the factor's entries are the same for every lane, and the substitution and the ordered
                // sum run down the coordinates with the operations of the loop below, head beside head instead of
                // four heads a pass.
                by_heads = true;
                const float* factor_rows = d.m_factor + size_t{env} * md * md;
                const bool owned = lane < heads && (c.U(hSourceA, lane) != kInvalid || c.U(hSourceB, lane) != kInvalid);
                const uint64_t way = owned ? way_of(c, lane) : 0ull;
                float w[6];
#pragma unroll
                for (int t = 0; t < 6; ++t) w[t] = owned ? c.wrench[lane * kWrenchStride + uint32_t(t)] : 0.0f;
                const float4* table = reinterpret_cast<const float4*>(c.axes);
                float y[N];
                float total = 0.0f;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    if (uint32_t(i) >= n) { y[i] = 0.0f; continue; }
                    const float4 sa = table[3 * i], sb = table[3 * i + 1];
                    const float entry = fmaf(sb.y, w[5], fmaf(sb.x, w[4], fmaf(sa.w, w[3], fmaf(sa.z, w[2], fmaf(sa.y, w[1], sa.x * w[0])))));
                    float v = ((way >> i) & 1ull) != 0ull ? entry : 0.0f;
                    const float* factor_row = factor_rows + size_t(i) * md;
#pragma unroll
                    for (int j = 0; j < i; ++j) v -= factor_row[j] * y[j];
                    y[i] = v;
                    total += v * v / factor_row[i];
                }
                if (lane < heads) {
                    const bool second = c.U(hSourceA, lane) == kInvalid;
                    c.F(hStep, lane) = second ? 0.0f : total; c.F(hMove, lane) = second ? total : 0.0f;
                }
            }
        }
        for (uint32_t h0 = 0u; h0 < (by_heads ? 0u : share_units ? c.individual_end : heads); h0 += 4u) {
            float a[4], total[4];
            bool second[4], apart[4], skip[4];
#pragma unroll
            for (uint32_t t = 0u; t < 4u; ++t) {
                const uint32_t h = h0 + t;
                a[t] = 0.0f; second[t] = false; apart[t] = false; skip[t] = true;
                if (h >= heads) continue;
                const bool artic_a = c.U(hSourceA, h) != kInvalid, artic_b = c.U(hSourceB, h) != kInvalid;
                if (artic_a && artic_b) {
                    const float* row = urows + size_t{c.slot(h)} * kRowWords;
                    apart[t] = __float_as_uint(row[11]) != __float_as_uint(row[19]);
                }
                second[t] = artic_b && !artic_a;
                const uint32_t first = c.U(hRow, h), unit = kPaired ? kInvalid : c.U(hUnit, h);
                const float unit_value = kPaired ? 0.0f : c.F(hUnitValue, h);
                skip[t] = share_units && unit != kInvalid && fabsf(unit_value) == 1.0f && !apart[t];
                if (coordinate && (artic_a || artic_b) && !apart[t] && !skip[t]) {
                    if (W > kTwoWaveWidth && c.from_links) {   // the first row's entry: the coordinate's axis against the row's wrench
                        const float4* table = reinterpret_cast<const float4*>(c.axes);
                        const float4 sa = table[3u * lane], sb = table[3u * lane + 1u];
                        const float* w = c.wrench + h * kWrenchStride;
                        const float entry = fmaf(sb.y, w[5], fmaf(sb.x, w[4], fmaf(sa.w, w[3], fmaf(sa.z, w[2], fmaf(sa.y, w[1], sa.x * w[0])))));
                        a[t] = ((way_of(c, h) >> lane) & 1ull) != 0ull ? entry : 0.0f;
                    } else {
                        a[t] = first != kInvalid ? (lane < c.ldj ? c.jac[first * c.ldj + lane] : 0.0f) : (lane == unit ? unit_value : 0.0f);
                    }
                }
            }
            if (skip[0] && skip[1] && skip[2] && skip[3]) continue;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                float y[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) y[t] = lane_value(a[t], j);
#pragma unroll
                for (int t = 0; t < 4; ++t) a[t] -= lrow[j] * y[t];
            }
            // the ordered sums, a lane a head: the terms pass through LDS (where the factors will stand, not built yet)
            float* terms = c.hfac;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float term = coordinate ? a[t] * a[t] / pivot : 0.0f;
                if (lane < uint32_t(N)) terms[uint32_t(t * N) + lane] = term;
            }
            lds_sync<W>();
            float mine = 0.0f;
            {
                const float4* words = reinterpret_cast<const float4*>(terms + (lane & 3u) * uint32_t(N));
#pragma unroll
                for (int q = 0; q < N / 4; ++q) { const float4 w = words[q]; mine += w.x; mine += w.y; mine += w.z; mine += w.w; }
            }
            lds_sync<W>();
#pragma unroll
            for (int t = 0; t < 4; ++t) total[t] = lane_value(mine, t);
#pragma unroll
            for (uint32_t t = 0u; t < 4u; ++t) {
                const uint32_t h = h0 + t;
                if (h >= heads || skip[t]) continue;
                float shares[2] = {second[t] ? 0.0f : total[t], second[t] ? total[t] : 0.0f};
                if (apart[t]) {   // two owners: one response each
                    shares[0] = response(coordinate ? d.chain_jacobian[size_t{c.U(hSourceA, h)} * md + lane] : 0.0f);
                    shares[1] = response(coordinate ? d.chain_jacobian_b[size_t{c.U(hSourceB, h)} * md + lane] : 0.0f);
                }
                if (lane == 0u) { c.F(hStep, h) = shares[0]; c.F(hMove, h) = shares[1]; }
            }
        }
        if (share_units) {
            // (M^-1)_uu of every coordinate at once, lane = coordinate u: y = L^-1 e_u down the rows with the factor's entries the
            // same for every lane, and the ordered sum of y^2 / D, with the operations of the loop above (four coordinates a
            // pass of that loop took 40 k cycles of a servo-driven humanoid's set-up, this takes 9 k)
            const Recip by_pivot = make_recip(pivot);   // the quotients to the bit wherever their sum can see them, zero by pivots past 2^126
            float mine = 0.0f, y[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                float v = lane == uint32_t(i) ? 1.0f : 0.0f;
#pragma unroll
                for (int j = 0; j < i; ++j) v -= lane_value(lrow[j], i) * y[j];
                y[i] = v;
                const float term = div_by(v * v, Recip{lane_value(pivot, i), lane_value(by_pivot.value, i)});
                mine += uint32_t(i) < n ? term : 0.0f;
            }
            for (uint32_t k = 0u; k < c.unit_count; ++k) {   // lane = coordinate hands its response to its own unit heads
                const uint32_t h = c.unit_list[k * uint32_t(kWave) + lane];
                if (fabsf(c.F(hUnitValue, h)) != 1.0f) continue;
                const bool artic_a = c.U(hSourceA, h) != kInvalid, artic_b = c.U(hSourceB, h) != kInvalid;
                if (artic_a && artic_b) {   // both sides on one owner (two owners were answered above)
                    const float* row = urows + size_t{c.slot(h)} * kRowWords;
                    if (__float_as_uint(row[11]) != __float_as_uint(row[19])) continue;
                }
                const bool second = artic_b && !artic_a;
                c.F(hStep, h) = second ? 0.0f : mine; c.F(hMove, h) = second ? mine : 0.0f;
            }
        }
        lds_sync<W>();
    }
    PROF_END(c, 18);
    PROF_BEGIN(c, 19);
    // InitializeTileHead (:743-797), lane = head
    bool any_elliptic = false;
    for (uint32_t base = 0u; base < heads; base += kWave) {
        const uint32_t h = base + lane;
        if (h < heads) {
            const uint32_t slot = c.slot(h);
            const float* row = urows + size_t{slot} * kRowWords;
            // (a head past the staged ones' room shares its narrow words with the joint rows' heads, which are on one axis)
            const bool joint = h >= staged_cap;
            const uint32_t flags = __float_as_uint(row[0]), stride = joint ? 1u : __float_as_uint(row[2]);
            const uint32_t axes = !joint && (flags & kRowBlockNormal) != 0u ? 3u : 1u;
            const uint32_t kind_a = __float_as_uint(row[10]), kind_b = __float_as_uint(row[18]);
            const float shares[2] = {c.F(hStep, h), c.F(hMove, h)};
            const bool valid = shares[0] >= 0.0f && isfinite(shares[0]) && shares[1] >= 0.0f && isfinite(shares[1]);
            float response = shares[0] + shares[1];
            const float coupling = shares[0] * shares[1], largest = fmaxf(shares[0], shares[1]);
            if (!(valid && isfinite(response))) response = nanf("");
            const float coupled = coupling > 0.0f ? (response + sqrtf(response * response + 12.0f * coupling)) / (6.0f * coupling) : FLT_MAX;
            const float capv = kPenaltyConditionCap / largest;
            float rho = response > 0.0f ? fminf(capv, coupled) : 0.0f;
            if (!(response == 0.0f || (response > 0.0f && rho > 0.0f && rho <= FLT_MAX))) {
                atomicOr(d.env_status + env, kEnvStatusSolverFailure);
                rho = nanf("");
            }
            d.solver_penalty[slot] = rho;
            const float compliance = row[5];
            const Response sr = scalar_response(rho, compliance);
            const uint32_t local = slot - env * R;
            // three axes of a MuJoCo-law contact: the elliptic cone, with the compliances of the two tangent rows (:778-780)
            const bool elliptic = kElliptic && axes == 3u && (flags & kRowMuJoCo) != 0u;
            any_elliptic = any_elliptic || elliptic;
            c.U(hStride, h) = stride; c.U(hAxes, h) = elliptic ? kAxesElliptic : axes;
            c.U(hSlot, h) = slot | (kind_a == kSideArtic || kind_b == kSideArtic ? 0u : kUnowned);
            c.U(hSecond, h) = joint || kind_a == kSideArtic ? 0u : 1u;
            c.F(hRho, h) = rho; c.F(hCompliance, h) = compliance; c.F(hLower, h) = row[6]; c.F(hUpper, h) = row[7];
            c.F(hMu1, h) = joint ? 0.0f : row[8]; c.F(hMu2, h) = joint ? 0.0f : row[9]; c.F(hNormalBound, h) = 0.0f;
            c.F(hDualScale, h) = sr.dual_scale; c.F(hResidualScale, h) = sr.residual_scale;
            const float dx = lambda_env[local], dy = axes == 3u ? lambda_env[local + stride] : 0.0f,
                        dz = axes == 3u ? lambda_env[local + 2u * stride] : 0.0f;
            c.F(hDual, h) = dx; c.F(hDual + 1, h) = dy; c.F(hDual + 2, h) = dz;
            c.F(hBase, h) = dx; c.F(hBase + 1, h) = dy; c.F(hBase + 2, h) = dz;
#pragma unroll
            for (int k = 0; k < 3; ++k) { c.F(hRes + k, h) = 0.0f; c.F(hMove + k, h) = 0.0f; c.F(hStep + k, h) = 0.0f; c.F(hRelaxStep + k, h) = 0.0f; c.F(hRelaxPoint + k, h) = 0.0f; }
            c.F(hRelaxWeight, h) = 0.0f;
            if (elliptic) {
                c.F(hTangentCompliance, h) = urows[size_t{slot + stride} * kRowWords + 5u];
                c.F(hTangentCompliance + 1, h) = urows[size_t{slot + 2u * stride} * kRowWords + 5u];
                if (h < uint32_t(kWave)) keep_cone(c, h, elliptic_cone(rho, compliance, c.F(hTangentCompliance, h), c.F(hTangentCompliance + 1, h), row[8]));
            }
        }
    }
    c.elliptic = kElliptic && __any(any_elliptic);
    lds_sync<W>();
    {
        const uint32_t own = min(lane, heads == 0u ? 0u : heads - 1u);
        const bool staged = lane < heads && c.U(hRow, own) != kInvalid;
        const bool within = block_axes(c.U(hAxes, own)) && c.U(hColumnsHigh, own) == 0u && (uint64_t(c.U(hColumnsLow, own)) >> (4 * kFirstColumns<W>)) == 0ull;
        c.block_heads = !__any(staged && !within);
    }
    bool later_axes = false;   // a later head on more axes than one
    for (uint32_t h = lane + kWave; h < heads; h += kWave) later_axes = later_axes || c.U(hAxes, h) != 1u;
    c.scalar_later = !kContactsOnly && !c.elliptic && heads > uint32_t(kWave) && heads <= uint32_t(kWave) * (kLaterHeads + 1u) && !__any(later_axes);
    PROF_END(c, 19);
    PROF_BEGIN(c, 20);
    // the one factorisation of the mass matrix
    c.mass_valid = factor_mass<W, kReduced>(c, mrow) && reduction_valid;
    PROF_END(c, 20);
    PROF_BEGIN(c, 21);
    initialize_residuals<W>(c, velocity, urows, p.dt);
    PROF_END(c, 21);
    PROF_END(c, 0);
    float residual4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t sweeps = 0u;
    DualMomentum momentum{1.0f, 0.0f};
    const float tol = c.tolerance;
    while (sweeps < p.iterations) {
        c.iteration = sweeps++;
        c.momentum = 0.0f; c.residual = 0.0f;
        PROF_COUNT(c, 2);
        descend_block<W, kReduced>(c, mrow, &velocity, free_v, true, d);
        float rowsr[3];
        PROF_BEGIN(c, 6);
        update_duals(c, lambda_env, R, urows, &momentum, true, true, rowsr);
        PROF_END(c, 6);
        PROF_BEGIN(c, 7);
        if (sweeps == p.iterations || fmaxf(fmaxf(rowsr[0], rowsr[1]), fmaxf(rowsr[2], c.residual)) < tol)
            measure_primal<W, kReduced>(c, mrow, &velocity, free_v, lambda_env, R, false, d);
        PROF_END(c, 7);
        if (fmaxf(fmaxf(rowsr[0], rowsr[1]), rowsr[2]) < tol && c.residual >= tol && c.residual < FLT_MAX) {
            measure_primal<W, kReduced>(c, mrow, &velocity, free_v, lambda_env, R, true, d);
            if (c.residual < FLT_MAX) {
                initialize_residuals<W>(c, velocity, urows, p.dt);
                update_duals(c, lambda_env, R, urows, nullptr, true, false, rowsr);
                c.residual = 0.0f;
                measure_primal<W, kReduced>(c, mrow, &velocity, free_v, lambda_env, R, false, d);
            }
        }
        residual4[0] = rowsr[0]; residual4[1] = rowsr[1]; residual4[2] = rowsr[2]; residual4[3] = c.residual;
        const float largest = fmaxf(fmaxf(rowsr[0], rowsr[1]), fmaxf(rowsr[2], c.residual));
        if (largest < tol || largest == FLT_MAX) break;
    }
    if constexpr (kReduced && kElliptic) {
        // The followers once more from the block's coordinates as they ended, in double: their moves were single-precision sums,
        // whose rounding nothing corrected on the way (over 65536 humanoids the mean error is 0.9989 of the oracle's with this, 0.9994
        // without it and 0.9990 at the full width).
        double* apart = reinterpret_cast<double*>(c.vec);
        apart[lane] = lane < c.n ? double(velocity) - double(free_v) : 0.0;
        lds_sync<W>();
        double follow = double(free_v);
        const double2* apart2 = reinterpret_cast<const double2*>(apart);
#pragma unroll
        for (int q = 0; q < W / 2; ++q) {
            const double2 dv = apart2[q];
            follow = fma(double(mrow[2 * q]), dv.x, follow);
            follow = fma(double(mrow[2 * q + 1]), dv.y, follow);
        }
        lds_sync<W>();
        if (lane >= c.n && lane < n) velocity = float(follow);
    }
    if (lane < 4u)
        d.solver_residual[size_t{env} * 4u + lane] =
            lane == 0u ? residual4[0] : lane == 1u ? residual4[1] : lane == 2u ? residual4[2] : residual4[3];
    if (lane == 0u) {
        d.vbd_velocity_sweep_count[env] = sweeps;
        d.solver_cost[env] = solve_cost_after(d.solver_cost[env], c.work);   // the scheduling key of the next solves
        if (d.solver_points != nullptr) d.solver_points[env] = points_solved(d.solver_points[env]);
    }
#ifdef NKH_SOLVER_PROFILE
    PROF_END(c, 9);
    if (lane == 0u) {
        for (int i = 0; i < 10; ++i) d.solver_penalty[size_t{env} * R + i] = float(c.prof[i]);
        for (int i = 0; i < 4; ++i) d.solver_penalty[size_t{env} * R + 10 + i] = float(c.prof_count[i]);
        for (int i = 10; i < 26; ++i) d.solver_penalty[size_t{env} * R + 4 + i] = float(c.prof[i]);
        for (int i = 26; i < 32; ++i) if (uint32_t(7 + i) < R) d.solver_penalty[size_t{env} * R + 7 + i] = float(c.prof[i]);
        // launch slot and the wave's first and last moment on the constant 100 MHz clock, as raw words
        d.solver_penalty[size_t{env} * R + 30] = __uint_as_float(uint32_t(prof_wall_start));
        d.solver_penalty[size_t{env} * R + 31] = __uint_as_float(uint32_t(wall_clock64()));
        d.solver_penalty[size_t{env} * R + 32] = __uint_as_float(place);
    }
#endif
    // the block velocities persist for the next solve's carried start
    if (lane < md) {
        d.solver_velocity[size_t{env} * md + lane] = coordinate ? velocity : 0.0f;
        d.solver_free[size_t{env} * md + lane] = coordinate ? free_v : 0.0f;
    }
    // FinishTile (:2607-2650)
    const bool invalid = __any(coordinate && !(fabsf(velocity) <= FLT_MAX));
    if (!invalid) {
        if (lane < md) d.qdot_flat[size_t{env} * md + lane] = coordinate ? velocity : 0.0f;
        if (coordinate) {
            if (my_component == kInvalid) d.qdot[lbase + my_link] = velocity;
            else d.link_velocity[(lbase + my_link) * 6u + my_component] = velocity;
        }
    } else if (lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
    // joint limit impulses (:2658-2668)
    if (p.base_link_count != 0u && p.joint_limit_rows_per_env >= 2u * p.base_link_count) {
        for (uint32_t l = lane; l < nl; l += kWave) {
            const size_t lower = size_t{env} * R + p.contact_rows_per_env + size_t{l} * 2u;
            d.joint_limit_impulse[2u * (lbase + l)] = (__float_as_uint(urows[lower * kRowWords]) & kRowActive) != 0u ? d.lambda[lower] : 0.0f;
            d.joint_limit_impulse[2u * (lbase + l) + 1u] = (__float_as_uint(urows[(lower + 1u) * kRowWords]) & kRowActive) != 0u ? d.lambda[lower + 1u] : 0.0f;
        }
    }
    // split-impulse position pass (:3059-3077; MarkTilePositions :2673-2708; PositionRowBias block_descent.cu:1734-1753)
    if (p.position_iterations != 0u) {
        float* qvec = c.vec + 128;
        qvec[lane] = coordinate ? velocity : 0.0f;   // the final generalized velocity, as qdot_flat
        // The contact slots' first rows, for the heads to find their slot's; a slot without points is nobody's.  (Heads that walked
        // the slots and their Jacobian rows in memory, a trip for every word, were 10 us of the pass's 30 with 4096
        // quadrupeds; a world with compliant contacts, whose heads hardly ever ask, lists none.)
        const uint32_t listed = m.any_mujoco != 0u ? 0u : min(S, 128u);
        uint32_t* slot_rows = reinterpret_cast<uint32_t*>(c.vec);
        for (uint32_t s = lane; s < listed; s += kWave) {
            const size_t at = (size_t{env} * S + s) * 2u;
            const uint32_t first = d.ucontact_row_range[at], points = d.ucontact_row_range[at + 1u];
            slot_rows[s] = points > 0u ? first : kInvalid;
        }
        lds_sync<W>();
        bool push = false;
        for (uint32_t h = lane; h < heads; h += kWave) {
            const uint32_t slot = c.slot(h);
            const float* row = urows + size_t{slot} * kRowWords;
            const uint32_t flags = __float_as_uint(row[0]);
            const float penetration = d.row_penetration[slot];
            const bool speculative = (flags & kRowSpeculative) != 0u;
            const float slop = speculative ? 0.0f : p.position_slop;
            const bool position = (flags & (kRowFriction | kRowVelocityOnly | kRowMuJoCo)) == 0u &&
                (speculative || penetration > slop || c.F(hDual, h) != 0.0f);
            float bias = 0.0f, rounding = 0.0f;
            if (position) {
                const float pen = fmaxf(penetration - slop, 0.0f);
                if (speculative) {
                    // the contact slot whose normal rows hold this row (MapRowContactsKernel, block_descent.cu:1756-1767)
                    const uint32_t group_first = __float_as_uint(row[1]), points = __float_as_uint(row[2]);
                    uint32_t contact = 0u;
                    for (uint32_t s = 0u; s < listed; ++s) contact = slot_rows[s] == group_first ? env * S + s : contact;
                    for (uint32_t s = listed; s < S; ++s)
                        if (d.ucontact_row_range[(size_t{env} * S + s) * 2u] == group_first &&
                            d.ucontact_row_range[(size_t{env} * S + s) * 2u + 1u] > 0u) contact = env * S + s;
                    const size_t point = size_t{contact} * 4u + (slot - group_first) % points;
                    const double depth = double(d.ucontact_depth[point]) - slop;
                    const double reserve = double(penetration) - d.ucontact_depth[point];
                    const double correction = p.position_beta * fmax(depth, 0.0) + reserve;
                    const double target = fmin(depth, 0.0) + correction;
                    double vel = 0.0;   // RowVelocity (block_descent.cu:1051-1082) per articulated side
                    const uint32_t kind_a = __float_as_uint(row[10]), kind_b = __float_as_uint(row[18]), first = c.U(hRow, h);
                    const bool apart = kind_a == kSideArtic && kind_b == kSideArtic && __float_as_uint(row[11]) != __float_as_uint(row[19]);
                    if (!c.from_links && first != kInvalid && !apart) {
                        // one owner: the staged row is the side's own (of two sides with one owner the first holds both), its
                        // entries past the block zeros; each product is exact in double
                        const float4* j4 = reinterpret_cast<const float4*>(c.jac + first * uint32_t(W)), *q4 = reinterpret_cast<const float4*>(qvec);
#pragma unroll
                        for (int q = 0; q < W / 4; ++q) {
                            const float4 j = j4[q], v = q4[q];
                            vel = fma(double(j.x), double(v.x), vel); vel = fma(double(j.y), double(v.y), vel);
                            vel = fma(double(j.z), double(v.z), vel); vel = fma(double(j.w), double(v.w), vel);
                        }
                    } else if (kind_a == kSideArtic) {
                        double value = 0.0;
                        for (uint32_t k = 0u; k < n; ++k) value += double(d.chain_jacobian[size_t{slot} * md + k]) * qvec[k];
                        vel += value;
                    }
                    if (kind_b == kSideArtic && (c.from_links || first == kInvalid || apart)) {
                        double value = 0.0;
                        for (uint32_t k = 0u; k < n; ++k) value += double(d.chain_jacobian_b[size_t{slot} * md + k]) * qvec[k];
                        vel += value;
                    }
                    const double limit = fmin(correction / p.dt, double(p.position_max_velocity));
                    const double absorbed = target > 0.0 ? 0.0 : fmax(reserve, 0.0) / p.dt;
                    bias = float(fmin(target / p.dt - vel, limit));
                    rounding = float(absorbed);
                } else {
                    const float correction = p.position_beta * pen + fmaxf(pen - pen, 0.0f);
                    bias = fminf(correction / p.dt, p.position_max_velocity);
                }
            }
            if (!position) c.U(hSlot, h) = slot | kUnowned;
            const Response sr = scalar_response(c.F(hRho, h), 0.0f);
            c.U(hAxes, h) = 1u;
            c.F(hCompliance, h) = 0.0f; c.F(hLower, h) = 0.0f; c.F(hUpper, h) = FLT_MAX;
            c.F(hDualScale, h) = sr.dual_scale; c.F(hResidualScale, h) = sr.residual_scale;
            c.F(hRes, h) = bias; c.F(hRes + 1, h) = 0.0f; c.F(hRes + 2, h) = 0.0f;
            c.F(hDual, h) = 0.0f; c.F(hDual + 1, h) = 0.0f; c.F(hDual + 2, h) = 0.0f;
            push = push || bias > rounding;
        }
        push = __any(push);
        c.block_heads = false;   // on one axis now
        lds_sync<W>();
        float pseudo = 0.0f;
        if (push) {
            const uint32_t positions = 1u;   // no head couples two moving blocks here, so one solve (:2716)
            for (uint32_t iteration = 0u; iteration < positions; ++iteration) {
                c.iteration = sweeps + iteration;
                descend_block<W, kReduced>(c, mrow, &pseudo, 0.0f, false, d);
            }
        }
        // FinishTilePositions (:2720-2744)
        if (coordinate) {
            if (my_component == kInvalid) d.qdot_pseudo[lbase + my_link] = pseudo;
            else d.link_velocity_pseudo[(lbase + my_link) * 6u + my_component] = pseudo;
        }
    }
    if constexpr (kQueue) {
        if (highest != kQueued) return;
        uint32_t taken = 0u;
        if (lane == 0u) taken = atomicAdd(d.solver_queue, 1u);
        place = lowest + uint32_t(__builtin_amdgcn_readfirstlane(int(taken)));
        if (place >= p.env_count) return;
        __syncthreads();
        goto environment;
    }
}

#ifdef NKH_SOLVER_PAIRED
}  // namespace paired
#endif
#ifdef NKH_SOLVER_DENSE
}  // namespace dense
#endif
}  // namespace solver
}  // namespace nkh
