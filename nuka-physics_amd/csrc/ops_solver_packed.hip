// The block-descent solve of small blocks, four environments a wavefront: a row of sixteen lanes owns an environment, its
// lanes the block's coordinates in the matrix phases (at most kPackedWidth) and its heads in the per-head phases (at most
// sixteen).  For worlds of contact heads only, without the elliptic cone (PackedSolverTakes in ops_solver.hip).
//
// BlockDescentTileKernel gives such an environment a wavefront, and most of its lanes idle: a free box has six coordinates and
// four contact points.  What it passes by scalar lane reads goes by DPP here - row_newbcast hands one lane of a row of
// sixteen to the other fifteen, as an operand of the multiply-add that takes it - so an instruction serves four environments.
// A lane holds its head whole in registers (the wavefront-an-environment kernel keeps heads in LDS, where row lanes and
// head lanes are different lanes); LDS holds the Jacobian rows and the two factors, which are read transposed.  Rows of lanes
// branch on their own: an environment that is done waits for the longest of its wavefront's four, which the launch
// order (sorted by cost) makes much alike.
//
// The arithmetic is that of the narrow block (BlockDescentTileKernel<8, true>) operation for operation, sums in the same
// order, but for where a head stands in the four partial sums of a force: the other kernel places the heads that contribute one
// behind the other, this one every head by its number.  An environment of up to four heads ends with the same bits unless three of
// them contribute and one of the first two does not; then, and with more heads, the last place of a force may differ (in 24 steps of
// 9001 boxes coming to rest one velocity did, by one).
//   Bound by vector issue (20 k instructions a wavefront of 16384 free boxes, of which 256 go alone, where one environment takes
// 12.4 k in the other kernel) and, below 32768 boxes, by the longest wavefronts: the four of one do not take their line searches
// and sweeps alike, which is why the costliest go alone (PackedAlone).  A step of 8192 free boxes in the other kernel and so 336 and
// 339 us (374 and 364 where every state is new), 16384 526 and 418, 32768 915 and 564, 65536 1678 and 979.  Three waves a SIMD, 60
// bytes a lane in scratch memory; with four and the rest in scratch memory 16384 527 and 65536 1250, with two 439 and 1145, where
// three took 392 and 981.
// Replaces what ops_solver_kernel.h replaces (block_descent_tile.cuh), whose line numbers stand there.
#include "ops_solver_kernel.h"

namespace nkh {
namespace solver {
namespace {

constexpr int W = kPackedWidth;

// lane J of the lane's row of sixteen
template <int J>
__device__ __forceinline__ uint32_t row_lane_u(uint32_t v) { return dpp_move_u<0x150 + J>(v); }
template <int J>
__device__ __forceinline__ float row_lane(float v) { return __uint_as_float(row_lane_u<J>(__float_as_uint(v))); }
template <int J>
__device__ __forceinline__ double row_lane(double v) {
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    return double_of(row_lane_u<J>(uint32_t(bits)), row_lane_u<J>(uint32_t(bits >> 32u)));
}
// f(integral constant) for First .. End - 1, in order
template <int First, int End, class F>
__device__ __forceinline__ void each(F&& f) {
    if constexpr (First < End) {
        f(std::integral_constant<int, First>{});
        each<First + 1, End>(f);
    }
}
template <int First, class F>   // from First down to 0
__device__ __forceinline__ void each_down(F&& f) {
    if constexpr (First >= 0) {
        f(std::integral_constant<int, First>{});
        each_down<First - 1>(f);
    }
}
__device__ __forceinline__ float env_sum(float v) {
    v += dpp_move<kDppXor1>(v); v += dpp_move<kDppXor2>(v); v += dpp_move<kDppHalfMirror>(v); v += dpp_move<kDppMirror>(v);
    return v;
}
__device__ __forceinline__ float env_max(float v) {
    v = fmaxf(v, dpp_move<kDppXor1>(v)); v = fmaxf(v, dpp_move<kDppXor2>(v));
    v = fmaxf(v, dpp_move<kDppHalfMirror>(v)); v = fmaxf(v, dpp_move<kDppMirror>(v));
    return v;
}
__device__ __forceinline__ uint32_t env_max_u(uint32_t v) {
    v = max(v, dpp_move_u<kDppXor1>(v)); v = max(v, dpp_move_u<kDppXor2>(v));
    v = max(v, dpp_move_u<kDppHalfMirror>(v)); v = max(v, dpp_move_u<kDppMirror>(v));
    return v;
}
__device__ __forceinline__ double env_sum_rotated(double v) {   // wave_sum_d's order within a row
    v += dpp_move_d<kDppRor8>(v); v += dpp_move_d<kDppRor4>(v); v += dpp_move_d<kDppXor2>(v); v += dpp_move_d<kDppXor1>(v);
    return v;
}

// What of a head a sweep reads once lies in LDS, a record a head, lane = head.  The constants of its line over a block descent
// (PlainLine) lie beside it as sixteen-byte words, taken to registers where a Newton step uses them, twice: kept there
// they and the assembly's sums are more than 168 registers, three waves a SIMD.
enum PackedField : uint32_t {
    pSlot, pStride, pRho, pCompliance, pLower, pUpper, pMu1, pMu2, pDualScale, pResidualScale,
    pRes, pDual = pRes + 3, pBase = pDual + 3, pRelaxStep = pBase + 3, pRelaxPoint = pRelaxStep + 3, pRelaxWeight = pRelaxPoint + 3, kPackedFields
};
constexpr uint32_t kPackedRecord = kPackedFields | 1u;   // lanes' words of one field fall on different banks

constexpr uint32_t kLineStride = 28u;   // of 24 words: sixteen lanes' sixteen-byte words of one place on different banks

// One environment, as its sixteen lanes hold it.
struct Packed {
    uint32_t env, lane;       // lane of the row
    uint32_t shift;           // of the row's votes in the wavefront's
    uint32_t n, heads, iteration, work;
    float tolerance;
    float* jac;               // 3 x capacity rows of W words
    float* mfac;              // W x W words, factor of the mass matrix
    float* hfac;              // W x W words, factor of the Newton Hessian
    float* hrows;             // W x W words, the Hessian of the last assembly
    float* record;            // lane's own head's
    float* line;              // its line's constants; zeros for a lane without a head
    float move[3], step[3];   // of lane's own head
    float* mass;              // W x W words, the mass matrix
    float mass_inverse, factor_root, curvature[6];
    bool mass_valid, factor_current, rows_made;
    float momentum, residual;
    bool live, owned, block;  // lane's own head: there is one; it acts on the block; it has three axes

    __device__ __forceinline__ bool all(bool on) const { return (uint32_t(__builtin_amdgcn_ballot_w64(!on) >> shift) & 0xFFFFu) == 0u; }
    __device__ __forceinline__ bool any(bool on) const { return (uint32_t(__builtin_amdgcn_ballot_w64(on) >> shift) & 0xFFFFu) != 0u; }
    __device__ __forceinline__ float& F(uint32_t field) const { return record[field]; }
    __device__ __forceinline__ uint32_t& U(uint32_t field) const { return reinterpret_cast<uint32_t*>(record)[field]; }
    __device__ __forceinline__ Response response() const { return Response{F(pDualScale), F(pResidualScale)}; }
};

__device__ __forceinline__ float env_total(TileSum s) { return float(row_total_d(s.value)); }

// factor_rows
__device__ __forceinline__ bool factor(const Packed& c, float (&row)[W], float* inverse_out, float* root_out) {
    const uint32_t lane = local_lane(c.lane);
    float inverse = 0.0f, root = 0.0f;
    each<0, W>([&](auto k) {
        constexpr int K = decltype(k)::value;
        const float scale = pivot_scale(row_lane<K>(row[K]));
        const float scaled = row[K] * scale;
        if (lane >= uint32_t(K)) { inverse = scale; root = scaled; }
        row[K] = lane > uint32_t(K) ? scaled : 0.0f;
        const float less = -row[K];
        each<K + 1, W>([&](auto j) { constexpr int J = decltype(j)::value; row[J] = fmaf(less, row_lane<J>(row[K]), row[J]); });
    });
    *inverse_out = inverse; *root_out = root;
    return c.all(c.lane >= uint32_t(W) || (inverse > 0.0f && inverse <= FLT_MAX));
}
__device__ __forceinline__ void store_row(const Packed& c, float* a, const float (&row)[W]) {
    if (c.lane >= uint32_t(W)) return;
    float4* words = reinterpret_cast<float4*>(a + c.lane * uint32_t(W));
#pragma unroll
    for (int q = 0; q < W / 4; ++q) words[q] = float4{row[4 * q], row[4 * q + 1], row[4 * q + 2], row[4 * q + 3]};
}
__device__ __forceinline__ void load_row(const Packed& c, const float* a, float (&row)[W]) {
    const float4* words = reinterpret_cast<const float4*>(a + min(c.lane, uint32_t(W - 1)) * uint32_t(W));
#pragma unroll
    for (int q = 0; q < W / 4; ++q) { const float4 w = words[q]; row[4 * q] = w.x; row[4 * q + 1] = w.y; row[4 * q + 2] = w.z; row[4 * q + 3] = w.w; }
}
// substitute; the columns from the stored factor
__device__ __forceinline__ float substitute_env(const Packed& c, const float (&row)[W], const float* factor_words, float inverse, float g) {
    const uint32_t from = min(c.lane, uint32_t(W - 1));
    float col[W];
#pragma unroll
    for (int j = 0; j < W; ++j) col[j] = factor_words[uint32_t(j * W) + from];
    float r = g;
    each<0, W>([&](auto j) { constexpr int J = decltype(j)::value; r = fmaf(row[J], -row_lane<J>(r * inverse), r); });
    r *= inverse;
    each_down<W - 1>([&](auto j) { constexpr int J = decltype(j)::value; r = fmaf(col[J], -row_lane<J>(r * inverse), r); });
    return r * inverse;
}
__device__ __forceinline__ float solve_mass(const Packed& c, float force) {
    float row[W];
    load_row(c, c.mfac, row);
    return substitute_env(c, row, c.mfac, c.mass_inverse, c.lane < c.n ? force : 0.0f);
}
__device__ __forceinline__ float mass_times_env(const Packed& c, float d) {
    float out = 0.0f, mrow[W];
    load_row(c, c.mass, mrow);
    each<0, W>([&](auto k) { constexpr int K = decltype(k)::value; out += mrow[K] * row_lane<K>(d); });
    return c.lane < c.n ? out : 0.0f;
}
// lane = head: its row `axis`
__device__ __forceinline__ void head_row(const Packed& c, uint32_t h, uint32_t axis, float (&j)[W]) {
    const float4* words = reinterpret_cast<const float4*>(c.jac + (3u * h + axis) * uint32_t(W));
#pragma unroll
    for (int q = 0; q < W / 4; ++q) { const float4 w = words[q]; j[4 * q] = w.x; j[4 * q + 1] = w.y; j[4 * q + 2] = w.z; j[4 * q + 3] = w.w; }
}
// row_steps
__device__ __forceinline__ void take_steps(Packed& c, float d) {
    const float own = c.lane < c.n ? d : 0.0f;
    const uint32_t h = c.owned ? c.lane : 0u;
#pragma unroll
    for (uint32_t axis = 0u; axis < 3u; ++axis) {
        float j[W], value = 0.0f;
        head_row(c, h, axis, j);
        each<0, W>([&](auto k) { constexpr int K = decltype(k)::value; value = fmaf(j[K], row_lane<K>(own), value); });
        c.step[axis] = c.owned ? value : 0.0f;
    }
}
__device__ __forceinline__ void take_moves(Packed& c, float alpha) {   // (a head that acts on nothing has steps of zero)
#pragma unroll
    for (int k = 0; k < 3; ++k) c.move[k] = fmaf(alpha, c.step[k], c.move[k]);
}

// own_line of lane's head at the start of a block descent
__device__ __forceinline__ PlainLine head_line(const Packed& c) {
    HeadLine l{};
    l.head = c.lane;
    l.owned = c.owned;
    if (!l.owned) return plain_line(l);
    l.contact = c.block;
    l.rho = c.F(pRho); l.compliance = c.F(pCompliance); l.lower = c.F(pLower); l.upper = c.F(pUpper);
    l.response = c.response();
    l.ratios = tangent_ratios(c.F(pMu1), c.F(pMu2));
#pragma unroll
    for (int k = 0; k < 3; ++k) { l.dual[k] = c.F(pDual + k); l.res[k] = c.F(pRes + k); }
    l.bound = l.dual[0];
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
    return plain_line(l);
}

__device__ __forceinline__ void store_line(const Packed& c, const PlainLine& p) {
    double2* wide = reinterpret_cast<double2*>(c.line);
    float4* words = reinterpret_cast<float4*>(c.line);
    wide[0] = double2{p.cone_y, p.cone_z}; wide[1] = double2{p.gain_y, p.gain_z};
    words[2] = float4{p.k, p.k_bounded, p.dual_part, p.lower}; words[3] = float4{p.upper, p.res[0], p.res[1], p.res[2]};
    words[4] = float4{p.mu_y, p.mu_z, p.radius, p.rho_radius}; words[5] = float4{p.radius_y, p.radius_z, p.inside_yy, p.inside_zz};
}
__device__ __forceinline__ PlainLine load_line(const Packed& c) {
    const double2* wide = reinterpret_cast<const double2*>(c.line);
    const float4* words = reinterpret_cast<const float4*>(c.line);
    const double2 cone = wide[0], gain = wide[1];
    const float4 a = words[2], b = words[3], e = words[4], g = words[5];
    PlainLine p;
    p.cone_y = cone.x; p.cone_z = cone.y; p.gain_y = gain.x; p.gain_z = gain.y;
    p.k = a.x; p.k_bounded = a.y; p.dual_part = a.z; p.lower = a.w; p.upper = b.x; p.res[0] = b.y; p.res[1] = b.z; p.res[2] = b.w;
    p.mu_y = e.x; p.mu_z = e.y; p.radius = e.z; p.rho_radius = e.w; p.radius_y = g.x; p.radius_z = g.y; p.inside_yy = g.z; p.inside_zz = g.w;
#pragma unroll
    for (int k = 0; k < 3; ++k) { p.move[k] = c.move[k]; p.step[k] = c.step[k]; }
    return p;
}

// assemble_block with add_heads_by_tiles' sums: four heads a pass, axis by axis, to a zeroed row that the mass row then takes
__device__ __forceinline__ bool assemble_env(Packed& c, float u, float free_v, float (&hrow)[W], float* force, float* inertia, bool* converged) {
    const bool coordinate = c.lane < c.n;
    float mf[3], mc[6], mn[3];
    {
        const PlainLine line = load_line(c);
        plain_response(line, c.move[0], c.move[1], c.move[2], mf, mc);
#pragma unroll
        for (int k = 0; k < 3; ++k) mn[k] = fabsf(mf[k]) + mc[k] * (fabsf(line.res[k]) + fabsf(c.move[k]));
    }
    const auto bits = [](float v) { return __float_as_uint(v); };
    uint32_t differs = 0u;
#pragma unroll
    for (int k = 0; k < 6; ++k) { differs |= bits(c.curvature[k]) ^ bits(mc[k]); c.curvature[k] = mc[k]; }
    if (c.any(c.live && differs != 0u)) { c.factor_current = false; c.rows_made = false; }
    const bool rows_kept = c.rows_made;
    const double apart = double(u) - double(free_v);
    TileSum inertial{0.0};
    double inertial_scale = 0.0;
    load_row(c, c.mass, hrow);
    each<0, W>([&](auto k) {
        constexpr int K = decltype(k)::value;
        const double m = double(hrow[K]), dv = row_lane<K>(apart);
        inertial.value = fma(m, dv, inertial.value);
        inertial_scale = fma(fabs(m), fabs(dv), inertial_scale);
    });
    float scale = float(inertial_scale);
    // the heads, four a pass: partial sums of the force a place of the pass each
    double part[4] = {0.0, 0.0, 0.0, 0.0};
    float bound[4] = {0.0f, 0.0f, 0.0f, 0.0f}, sum[W] = {};
    const uint32_t own = min(c.lane, uint32_t(W - 1));
    const bool within = c.lane < uint32_t(W);
#pragma unroll 1
    for (uint32_t first = 0u; first < c.heads; first += 4u) {
        if (first != 0u) {   // the pass's heads to the row's first four lanes
            const auto next = [](float v) { return dpp_move<0x12C>(v); };   // row_ror:12, lane i from lane i + 4
#pragma unroll
            for (int k = 0; k < 3; ++k) { mf[k] = next(mf[k]); mn[k] = next(mn[k]); mc[k] = next(mc[k]); }
            mc[5] = next(mc[5]);
        }
        float a[4][3];
        each<0, 4>([&](auto t) {
            constexpr int T = decltype(t)::value;
            const uint32_t h = first + uint32_t(T);
            const bool there = h < c.heads && within;
            const float* rows = c.jac + (h < c.heads ? 3u * h : 0u) * uint32_t(W) + own;
            float j[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) { const float word = rows[k * W]; j[k] = there ? word : 0.0f; }
            // (no head of these worlds has a curvature between its normal and a tangent: mc[3] and mc[4] are zero)
            a[T][0] = j[0] * row_lane<T>(mc[0]);
            a[T][1] = fmaf(j[2], row_lane<T>(mc[5]), j[1] * row_lane<T>(mc[1]));
            a[T][2] = fmaf(j[1], row_lane<T>(mc[5]), j[2] * row_lane<T>(mc[2]));
            each<0, 3>([&](auto k) {
                constexpr int A = decltype(k)::value;
                part[T] = fma(double(j[A]), double(row_lane<T>(mf[A])), part[T]);
                bound[T] = fmaf(fabsf(j[A]), row_lane<T>(mn[A]), bound[T]);
            });
        });
        if (rows_kept) continue;
#pragma unroll
        for (uint32_t k = 0u; k < 3u; ++k) {
#pragma unroll
            for (uint32_t t = 0u; t < 4u; ++t) {
                const uint32_t h = first + t;
                float row[W];
                head_row(c, h < c.heads ? h : 0u, k, row);
#pragma unroll
                for (int i = 0; i < W; ++i) sum[i] = fmaf(row[i], a[t][k], sum[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    const TileSum g{-inertial.value + ((part[0] + part[1]) + (part[2] + part[3]))};
    scale += (bound[0] + bound[1]) + (bound[2] + bound[3]);
    if (!rows_kept) {
#pragma unroll
        for (int i = 0; i < W; ++i) hrow[i] += sum[i];
        store_row(c, c.hrows, hrow);
        c.rows_made = true;
    } else load_row(c, c.hrows, hrow);
    *force = coordinate ? float(g.value) : 0.0f;
    *inertia = coordinate ? float(inertial.value) : 0.0f;
    const float magnitude = fabsf(u);
    each<0, W>([&](auto k) { constexpr int K = decltype(k)::value; scale += fabsf(hrow[K]) * row_lane<K>(magnitude); });
    bool finite = isfinite(*force) && isfinite(scale);
    if (!c.all(!coordinate || finite)) {
        finite = isfinite(*force);
#pragma unroll
        for (int k = 0; k < W; ++k) finite = finite && isfinite(hrow[k]);
    }
    *converged = c.all(!coordinate || fabsf(*force) <= kRoundings * FLT_EPSILON * scale);
    return c.all(!coordinate || finite);
}

__device__ __forceinline__ Failure direction_env(Packed& c, float u, float free_v, float* force, float* inertia, float* d, bool* converged) {
    c.work += 16u;
    float hrow[W];
    if (!assemble_env(c, u, free_v, hrow, force, inertia, converged)) return kFailEquation;
    if (*converged && c.tolerance > 0.0f) {
        if (!c.mass_valid) return kFailFactor;
        const float direction = solve_mass(c, *force);
        *d = direction;
        *converged = c.all(c.lane >= c.n || fabsf(direction) < c.tolerance);
        if (*converged) return kFailNone;
    }
    if (*converged) return kFailNone;
    float inverse = 0.0f;
    if (!c.factor_current) {
        if (!factor(c, hrow, &inverse, &c.factor_root)) return kFailFactor;
        store_row(c, c.hfac, hrow);
        wave_sync();
        c.factor_current = true;
    } else {
        inverse = 1.0f / c.factor_root;
        load_row(c, c.hfac, hrow);
    }
    *d = substitute_env(c, hrow, c.hfac, inverse, c.lane < c.n ? *force : 0.0f);
    wave_sync();
    return kFailNone;
}

// the line at alpha: plain_line_terms and the narrow sums of line_derivatives
__device__ __forceinline__ void line_at(const Packed& c, const PlainLine& p, float alpha, float inertial_slope, float inertial_curvature, float* slope,
                                        float* curvature, float* magnitude) {
    TileSum row_slope{0.0};
    float row_curvature = 0.0f, row_magnitude = 0.0f;
    plain_line_terms(p, alpha, row_slope, row_curvature, row_magnitude);
    TileSum total{-row_slope.value};
    if (c.lane == 0u) { tile_add_product(total, alpha, inertial_curvature); tile_add(total, inertial_slope); }
    *slope = env_total(total);
    *curvature = inertial_curvature + env_sum(row_curvature);
    *magnitude = fabsf(inertial_slope) + alpha * inertial_curvature + env_sum(row_magnitude);
}
__device__ __forceinline__ float search_env(Packed& c, float inertial_slope, float inertial_curvature) {
    const PlainLine line = load_line(c);
    float slope, curvature, magnitude;
    line_at(c, line, 0.0f, inertial_slope, inertial_curvature, &slope, &curvature, &magnitude);
    c.work += 1u;
    const float initial = slope;
    if (!(initial < 0.0f)) return 0.0f;
    float low = 0.0f, high = 0.0f, alpha = 1.0f;
    bool bounded = false;
    for (uint32_t step = 0u; step < kLineSearchSteps; ++step) {
        line_at(c, line, alpha, inertial_slope, inertial_curvature, &slope, &curvature, &magnitude);
        c.work += 1u;
        if (!isfinite(slope) || !isfinite(curvature)) {
            high = alpha; bounded = true; alpha = 0.5f * (low + high);
            continue;
        }
        if (fabsf(slope) <= fmaxf(kLineTolerance * -initial, kRoundings * FLT_EPSILON * magnitude)) return alpha;
        if (slope < 0.0f) low = alpha;
        else { high = alpha; bounded = true; }
        if (bounded && high - low <= FLT_EPSILON * high) return low;
        float next = alpha - slope * __builtin_amdgcn_rcpf(curvature);
        if (!(next > low && (!bounded || next < high))) next = bounded ? 0.5f * (low + high) : 2.0f * alpha;
        alpha = next;
    }
    return low;
}

// descend_block
__device__ __forceinline__ void descend_env(Packed& c, float* u_io, float free_in, bool has_free, DataView d) {
    const bool coordinate = c.lane < c.n;
    store_line(c, head_line(c));
    for (float& move : c.move) move = 0.0f;
    wave_sync();
    const float start = coordinate ? *u_io : 0.0f, free_v = coordinate && has_free ? free_in : 0.0f;
    float u = start;
    if (c.iteration == 0u && has_free) {
        const float dd = coordinate ? free_v - u : 0.0f;
        const float mass_step = mass_times_env(c, dd);
        TileSum curvature{0.0};
        if (coordinate) tile_add_product(curvature, dd, mass_step);
        const float inertial_curvature = env_total(curvature);
        if (inertial_curvature > 0.0f && isfinite(inertial_curvature)) {
            take_steps(c, dd);
            const float alpha = search_env(c, -inertial_curvature, inertial_curvature);
            if (alpha > 0.0f) { u = fmaf(alpha, dd, u); take_moves(c, alpha); }
        }
    }
    Failure failure = kFailNone;
    float primal = FLT_MAX;
    for (uint32_t step = 0u; step < kNewtonSteps; ++step) {
        float force = 0.0f, inertia = 0.0f, dd = 0.0f;
        bool converged = false;
        failure = direction_env(c, u, free_v, &force, &inertia, &dd, &converged);
        if (converged) primal = 0.0f;
        if (failure != kFailNone || converged) break;
        if (!coordinate) dd = 0.0f;
        const float mass_step = mass_times_env(c, dd);
        TileSum decrement{0.0}, slope{0.0}, curvature{0.0};
        if (coordinate) {
            tile_add_product(decrement, force, dd);
            tile_add_product(slope, inertia, dd);
            tile_add_product(curvature, dd, mass_step);
        }
        const float total_decrement = env_total(decrement), inertial_slope = env_total(slope), inertial_curvature = env_total(curvature);
        if (!isfinite(total_decrement) || !isfinite(inertial_slope) || !isfinite(inertial_curvature)) { failure = kFailDirection; break; }
        if (!(total_decrement > 0.0f)) break;
        take_steps(c, dd);
        const float alpha = search_env(c, inertial_slope, inertial_curvature);
        const float after = fmaf(alpha, dd, u);
        const bool rounded = c.all(!coordinate || after == u);
        if (!c.all(!coordinate || isfinite(after))) { failure = kFailCandidate; break; }
        primal = 0.0f;
        if (coordinate && !rounded) primal = fmaxf(primal, fabsf(alpha * dd));
        if (!(alpha > 0.0f)) break;
        u = after;
        take_moves(c, alpha);
        if (rounded) break;
    }
    if (c.owned) {
#pragma unroll
        for (int k = 0; k < 3; ++k) c.F(pRes + k) = c.F(pRes + k) - c.move[k];
    }
    if (failure != kFailNone && c.lane == 0u) d.env_status[c.env] |= kEnvStatusSolverFailure;
    float moved = failure == kFailNone ? 0.0f : FLT_MAX;
    if (coordinate) moved = fmaxf(moved, __uint_as_float(residual_bits(u - start)));
    c.momentum = fmaxf(c.momentum, env_max(moved));
    if (failure != kFailNone) primal = FLT_MAX;
    c.residual = fmaxf(c.residual, env_max(primal));
    if (coordinate) *u_io = u;
}

// measure_primal; the impulses are the heads' last committed ones (Packed::base), which lambda holds too
__device__ __forceinline__ void measure_env(Packed& c, float* velocity_io, float free_v, bool reconstruct, DataView d) {
    const bool coordinate = c.lane < c.n;
    const double apart = coordinate ? double(*velocity_io) - double(free_v) : 0.0;
    double balance = 0.0;
    float mrow[W];
    load_row(c, c.mass, mrow);
    each<0, W>([&](auto k) { constexpr int K = decltype(k)::value; balance = fma(-double(mrow[K]), row_lane<K>(apart), balance); });
    float mine[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) { const float base = c.F(pBase + k); mine[k] = c.owned && (k == 0 || c.block) ? base : 0.0f; }
    const uint32_t own = min(c.lane, uint32_t(W - 1));
#pragma unroll 1
    for (uint32_t first = 0u; first < c.heads; first += 4u) {
        each<0, 4>([&](auto t) {
            constexpr int T = decltype(t)::value;
            const uint32_t h = first + uint32_t(T);
            const float* j = c.jac + (h < c.heads ? 3u * h : 0u) * uint32_t(W) + own;   // (past the heads: lanes that hold zeros)
            each<0, 3>([&](auto k) { constexpr int A = decltype(k)::value; balance = fma(double(j[A * W]), double(row_lane<T>(mine[A])), balance); });
        });
#pragma unroll
        for (int k = 0; k < 3; ++k) mine[k] = dpp_move<0x12C>(mine[k]);
    }
    const float force = float(balance);
    const bool finite = c.all(!coordinate || fabs(balance) <= double(FLT_MAX));
    Failure failure = finite ? kFailNone : kFailEquation;
    float direction = 0.0f;
    if (failure == kFailNone) {
        if (c.mass_valid) direction = solve_mass(c, force);
        else failure = kFailFactor;
    }
    float residual = failure == kFailNone ? 0.0f : FLT_MAX;
    if (failure != kFailNone && c.lane == 0u) d.env_status[c.env] |= kEnvStatusSolverFailure;
    if (failure == kFailNone && coordinate) residual = fmaxf(residual, isfinite(direction) ? fabsf(direction) : FLT_MAX);
    residual = env_max(residual);
    c.residual = fmaxf(c.residual, residual);
    if (reconstruct && failure == kFailNone) {
        if (!c.all(!coordinate || isfinite(*velocity_io + direction))) { c.residual = FLT_MAX; return; }
        if (coordinate) *velocity_io += direction;
        c.momentum = fmaxf(c.momentum, residual);
    }
}

// initialize_residuals
__device__ __forceinline__ void residuals_env(Packed& c, float velocity, const float* urows, float dt) {
    const float own = c.lane < c.n ? velocity : 0.0f;
    const uint32_t h = c.live ? c.lane : 0u;
#pragma unroll
    for (uint32_t axis = 0u; axis < 3u; ++axis) {
        float j[W], along = 0.0f;
        head_row(c, h, axis, j);
        each<0, W>([&](auto k) { constexpr int K = decltype(k)::value; along = along + j[K] * row_lane<K>(own); });
        float residual = 0.0f;
        if (c.live) {
            if (axis == 0u || c.block) residual = urows[size_t{c.U(pSlot) + axis * c.U(pStride)} * kRowWords + 4u] * dt - along;
            c.F(pRes + axis) = residual;
        }
    }
}

// update_duals of lane's own head (no head here is elliptic)
__device__ __forceinline__ void duals_env(Packed& c, float* lambda_env, uint32_t R, const float* urows, DualMomentum* momentum, bool commit, float* classes) {
    uint32_t steps[3] = {0u, 0u, 0u};
    double restart = 0.0;
    const bool contact = c.block;
    const float lower = c.F(pLower), upper = c.F(pUpper), mu1 = c.F(pMu1), mu2 = c.F(pMu2);
    const Response response = c.response();
    const auto three = [&](uint32_t field) { return V3{c.F(field), c.F(field + 1u), c.F(field + 2u)}; };
    const auto put = [&](uint32_t field, V3 v) { c.F(field) = v.x; c.F(field + 1u) = v.y; c.F(field + 2u) = v.z; };
    V3 earlier{0, 0, 0}, latest{0, 0, 0};
    if (c.live) {
        const uint32_t slot = c.U(pSlot), local = slot - c.env * R, stride = c.U(pStride);
        const float rho = c.F(pRho), compliance = c.F(pCompliance);
        const V3 residual = three(pRes), base = three(pBase);
        const V3 tdual = commit ? three(pDual) : base;
        float normal, ncurv;
        scalar_impulse(tdual.x, rho, residual.x, compliance, lower, upper, response, &normal, &ncurv);
        V3 dual{normal, 0.0f, 0.0f}, rstep{0, 0, 0}, rpoint{0, 0, 0};
        float rweight = 0.0f;
        if (contact) {
            float fy, fz, cyy, czz, cyz;
            tangent_impulse(tdual, rho, residual.y, residual.z, normal, mu1, mu2, &fy, &fz, &cyy, &czz, &cyz);
            const V3 next{normal, fy, fz};
            V3 last_step{0, 0, 0}, last_point{0, 0, 0};
            float last_weight = 0.0f;
            if (commit) {
                last_step = three(pRelaxStep);
                last_weight = c.F(pRelaxWeight);
                last_point = three(pRelaxPoint);
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
        float step_normal = response.residual_scale > 0.0f && response.dual_scale != 0.0f ? fabsf(dual.x - tdual.x) / response.residual_scale : 0.0f;
        float step_tangent = 0.0f;
        if (contact) {
            const float fs = fmaxf(mu1, mu2);
            const float m1 = mu1 <= 0.0f ? 0.0f : mu1 / fs, m2 = mu2 <= 0.0f ? 0.0f : mu2 / fs;
            const float first = m1 > 0.0f && rho > 0.0f ? (dual.y - tdual.y) / (rho * m1 * m1) : 0.0f;
            const float second = m2 > 0.0f && rho > 0.0f ? (dual.z - tdual.z) / (rho * m2 * m2) : 0.0f;
            step_tangent = hypotf(first, second);
        }
        if (!commit && response.residual_scale > 0.0f) step_normal = fabsf(dual.x - tdual.x) / response.residual_scale;
        const V3 physical = commit ? dual : tdual;
        if (!contact) {
            const bool normal_row = (__float_as_uint(urows[size_t{slot} * kRowWords]) & kRowContactNormal) != 0u;
            const float rate = -residual.x + compliance * physical.x;
            const float violation = physical.x > 0.0f ? fabsf(rate) : fmaxf(-rate, 0.0f);
            if (normal_row) steps[0] = residual_bits(fmaxf(step_normal, violation));
            else steps[2] = residual_bits(step_normal);
        } else {
            if (commit) {
                put(pRelaxStep, rstep);
                c.F(pRelaxWeight) = rweight;
                put(pRelaxPoint, rpoint);
                lambda_env[local + stride] = dual.y;
                lambda_env[local + 2u * stride] = dual.z;
            }
            const V3 v{-residual.x + compliance * physical.x, -residual.y, -residual.z};
            steps[0] = residual_bits(physical.x > 0.0f ? fabsf(v.x) : fmaxf(-v.x, 0.0f));
            steps[1] = residual_bits(fmaxf(step_tangent, fmaxf(along_axis(physical.y, v.y), along_axis(physical.z, v.z))));
        }
        if (commit) {
            lambda_env[local] = dual.x;
            if (contact || response.dual_scale != 0.0f) {
                const float friction = fmaxf(mu1, mu2);
                const float first = contact && mu1 > 0.0f ? mu1 / friction : 0.0f;
                const float second = contact && mu2 > 0.0f ? mu2 / friction : 0.0f;
                const V3 metric{response.residual_scale, rho * first * first, rho * second * second};
                restart = (metric.x > 0.0f ? (double(tdual.x) - dual.x) * (double(dual.x) - base.x) / metric.x : 0.0) +
                          (metric.y > 0.0f ? (double(tdual.y) - dual.y) * (double(dual.y) - base.y) / metric.y : 0.0) +
                          (metric.z > 0.0f ? (double(tdual.z) - dual.z) * (double(dual.z) - base.z) / metric.z : 0.0);
            }
            earlier = base;
            latest = dual;
            put(pBase, dual);
        }
    }
    classes[0] = __uint_as_float(env_max_u(steps[0]));
    classes[1] = __uint_as_float(env_max_u(steps[1]));
    classes[2] = __uint_as_float(env_max_u(steps[2]));
    if (!commit) return;
    restart = env_sum_rotated(restart);
    if (restart > 0.0) momentum->t = 1.0f;
    const float t = 0.5f * (1.0f + sqrtf(fmaf(4.0f * momentum->t, momentum->t, 1.0f)));
    momentum->beta = (momentum->t - 1.0f) / t;
    momentum->t = t;
    if (!c.live) return;
    const float beta = contact || response.dual_scale != 0.0f ? momentum->beta : 0.0f;
    const V3 next = latest;
    V3 out = next;
    if (beta != 0.0f) {
        V3 y{fmaf(beta, next.x - earlier.x, next.x), fmaf(beta, next.y - earlier.y, next.y), fmaf(beta, next.z - earlier.z, next.z)};
        y.x = fminf(fmaxf(y.x, lower), upper);
        if (!contact) out = V3{y.x, 0.0f, 0.0f};
        else {
            const float first = mu1 > 0.0f ? y.y / mu1 : 0.0f, second = mu2 > 0.0f ? y.z / mu2 : 0.0f;
            const float slip = hypotf(first, second), radius = fmaxf(y.x, 0.0f);
            const float scale = slip > radius ? radius / slip : 1.0f;
            out = V3{y.x, mu1 > 0.0f ? y.y * scale : 0.0f, mu2 > 0.0f ? y.z * scale : 0.0f};
        }
    }
    put(pDual, out);
}

// lane = head: J M^-1 J^T of the row `a` by way of the LDL^T factor, whose row i lane i holds (`lrow` its unit lower triangle)
__device__ __forceinline__ float response_of(const Packed& c, const float (&lrow)[W], float pivot, const float (&a)[W]) {
    float y[W], total = 0.0f;
    each<0, W>([&](auto i) {
        constexpr int I = decltype(i)::value;
        float v = a[I];
        each<0, I>([&](auto j) { constexpr int J = decltype(j)::value; v -= row_lane<I>(lrow[J]) * y[J]; });
        y[I] = v;
        const float square = v * v / row_lane<I>(pivot);
        if (uint32_t(I) < c.n) total += square;
    });
    return total;
}

}  // namespace

// LDS words of an environment: the mass matrix, two factors, the kept Hessian, the rows, records and lines of `staged` heads, the environments of a wavefront sixteen banks apart
__host__ __device__ uint32_t PackedEnvFloats(uint32_t staged) {
    const uint32_t words = 4u * uint32_t(W * W) + 3u * staged * uint32_t(W) + (staged * kPackedRecord + 3u) / 4u * 4u + (staged + 1u) * kLineStride;
    return (words + 47u) / 64u * 64u + 16u;
}

__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(kPackedWaves, kPackedWaves)))
PackedDescentKernel(ModelView m, DataView d, BlockDescentSolveParams p, uint32_t cap, uint32_t alone) {
    extern __shared__ __align__(16) float lds[];
    // the first `alone` of the launch order have a wavefront each
    const uint32_t row = threadIdx.x >> 4u, place = blockIdx.x < alone ? blockIdx.x : alone + (blockIdx.x - alone) * kPackedEnvs + row;
    if (place >= p.env_count || (blockIdx.x < alone && row != 0u)) return;   // rows of lanes without an environment
    Packed c;
    c.env = d.tile_order[place]; c.lane = threadIdx.x & 15u; c.shift = threadIdx.x & 48u;
    const uint32_t env = c.env, lane = c.lane;
    const uint32_t R = p.rows_per_env, md = p.max_dof, n = m.dof, nl = m.links_per_env;
    c.n = n; c.work = 0u; c.iteration = 0u; c.tolerance = p.velocity_tolerance;
    c.factor_current = false; c.rows_made = false; c.factor_root = 1.0f;
    for (float& entry : c.curvature) entry = 0.0f;
    float* words = lds + (threadIdx.x >> 4u) * PackedEnvFloats(cap);
    c.mfac = words; c.hfac = words + W * W; c.hrows = words + 2 * W * W; c.mass = words + 3 * W * W; c.jac = words + 4 * W * W;
    c.record = c.jac + 3u * cap * uint32_t(W) + min(lane, cap - 1u) * kPackedRecord;   // (a lane past the heads writes none)
    uint32_t* listed = reinterpret_cast<uint32_t*>(words);           // the factors' words hold the set-up's lists first:
    uint32_t* sources = listed + kPackedHeads;                        // the heads' slots, then each row's two source rows
    c.line = c.jac + 3u * cap * uint32_t(W) + (cap * kPackedRecord + 3u) / 4u * 4u + min(lane, cap) * kLineStride;
    for (int k = 0; k < 3; ++k) { c.move[k] = 0.0f; c.step[k] = 0.0f; }
    const bool coordinate = lane < n;
    const float* urows = d.urows;
    float* lambda_env = d.lambda + size_t{env} * R;
    const size_t lbase = size_t{env} * nl;
    uint32_t my_link = 0u, my_component = kInvalid;
    float free_v = 0.0f, velocity = 0.0f;
    if (coordinate) {
        my_link = m.dof_link[lane]; my_component = m.dof_component[lane];
        const float value = my_component == kInvalid ? d.qdot[lbase + my_link] : d.link_velocity[(lbase + my_link) * 6u + my_component];
        const float carried = d.solver_velocity[size_t{env} * md + lane] - d.solver_free[size_t{env} * md + lane];
        free_v = value;
        velocity = value + (isfinite(carried) ? carried : 0.0f);
    }
    // lane's rows of the mass matrix and of its LDL^T factor
    float lrow[W], mrow[W], pivot = 1.0f;
    {
        const size_t tile = size_t{env} * md * md + size_t{coordinate ? lane : 0u} * md;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const bool in = uint32_t(k) < n;
            const float f = in ? d.m_factor[tile + uint32_t(k)] : 0.0f, w = in ? d.m[tile + uint32_t(k)] : 0.0f;
            mrow[k] = coordinate && in ? w : (lane == uint32_t(k) ? 1.0f : 0.0f);
            if (coordinate && lane == uint32_t(k)) pivot = f;
            lrow[k] = coordinate && uint32_t(k) < lane ? f : 0.0f;
        }
    }
    store_row(c, c.mass, mrow);
    // the active rows that are not block tangents, in slot order
    const uint32_t current = d.contact_row_extent[2u * env + 1u];
    const uint32_t bound = current == 0u ? p.contact_rows_per_env : min(current - 1u, p.contact_rows_per_env);
    const uint32_t total = bound + (R - p.contact_rows_per_env);
    uint32_t heads = 0u;
    bool overflow = false;
    for (uint32_t base = 0u; base < total; base += kPackedHeads) {
        const uint32_t index = base + lane;
        const uint32_t slot = env * R + (index < bound ? index : p.contact_rows_per_env + (index - bound));
        bool head = false;
        if (index < total) {
            const uint32_t flags = __float_as_uint(urows[size_t{slot} * kRowWords]);
            head = (flags & kRowActive) != 0u && (flags & kRowBlockTangent) == 0u;
        }
        const uint32_t mask = uint32_t(__builtin_amdgcn_ballot_w64(head) >> c.shift) & 0xFFFFu;
        if (head) {
            const uint32_t at = heads + uint32_t(__popc(mask & ((1u << lane) - 1u)));
            if (at < cap) listed[at] = slot; else overflow = true;
        }
        heads += uint32_t(__popc(mask));
    }
    if (c.any(overflow)) {   // more heads than the staged LDS holds: fail loudly, solve the ones that fit
        heads = cap;
        if (lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
    }
    c.heads = heads; c.live = lane < heads;
    wave_sync();
    const uint32_t slot = c.live ? listed[lane] : 0u;
    uint32_t source_a[3] = {kInvalid, kInvalid, kInvalid}, source_b[3] = {kInvalid, kInvalid, kInvalid};
    uint32_t stride = 1u;
    c.block = false;
    bool apart = false;
    if (c.live) {
        const float* row = urows + size_t{slot} * kRowWords;
        stride = __float_as_uint(row[2]);
        c.block = (__float_as_uint(row[0]) & kRowBlockNormal) != 0u;
#pragma unroll
        for (uint32_t axis = 0u; axis < 3u; ++axis) {
            if (axis != 0u && !c.block) continue;
            const uint32_t rs = slot + axis * stride;
            if (__float_as_uint(urows[size_t{rs} * kRowWords + 10u]) == kSideArtic) source_a[axis] = rs;
            if (__float_as_uint(urows[size_t{rs} * kRowWords + 18u]) == kSideArtic) source_b[axis] = rs;
        }
        apart = source_a[0] != kInvalid && source_b[0] != kInvalid && __float_as_uint(row[11]) != __float_as_uint(row[19]);
#pragma unroll
        for (uint32_t axis = 0u; axis < 3u; ++axis) { sources[2u * (3u * lane + axis)] = source_a[axis]; sources[2u * (3u * lane + axis) + 1u] = source_b[axis]; }
    }
    c.owned = source_a[0] != kInvalid || source_b[0] != kInvalid;
    wave_sync();
    // stage the rows, two of them a turn, a lane a word
    const uint32_t column = lane & 7u;
#pragma unroll 4
    for (uint32_t r = lane >> 3u; r < 3u * heads; r += 2u) {
        const uint32_t from_a = sources[2u * r], from_b = sources[2u * r + 1u];
        const float a = column < n && from_a != kInvalid ? d.chain_jacobian[size_t{from_a} * md + column] : 0.0f;
        const float b = column < n && from_b != kInvalid ? d.chain_jacobian_b[size_t{from_b} * md + column] : 0.0f;
        c.jac[r * uint32_t(W) + column] = (0.0f + a) + b;
    }
    wave_sync();
    float shares[2] = {0.0f, 0.0f};
    {
        float a[W];
        head_row(c, c.live ? lane : 0u, 0u, a);
        const float whole = response_of(c, lrow, pivot, a);
        const bool second = source_b[0] != kInvalid && source_a[0] == kInvalid;
        if (c.owned) { shares[0] = second ? 0.0f : whole; shares[1] = second ? whole : 0.0f; }
        if (c.any(apart)) {   // two owners: one response each
            float sides[2];
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const float* chain = (side == 0 ? d.chain_jacobian : d.chain_jacobian_b) + size_t{apart ? (side == 0 ? source_a[0] : source_b[0]) : 0u} * md;
#pragma unroll
                for (int k = 0; k < W; ++k) a[k] = apart && uint32_t(k) < n ? chain[k] : 0.0f;
                sides[side] = response_of(c, lrow, pivot, a);
            }
            if (apart) { shares[0] = sides[0]; shares[1] = sides[1]; }
        }
    }
    // InitializeTileHead
    if (c.live) {
        const float* row = urows + size_t{slot} * kRowWords;
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
        const Response answer = scalar_response(rho, compliance);
        const uint32_t local = slot - env * R;
        c.U(pSlot) = slot; c.U(pStride) = stride;
        c.F(pRho) = rho; c.F(pCompliance) = compliance; c.F(pLower) = row[6]; c.F(pUpper) = row[7]; c.F(pMu1) = row[8]; c.F(pMu2) = row[9];
        c.F(pDualScale) = answer.dual_scale; c.F(pResidualScale) = answer.residual_scale;
#pragma unroll
        for (uint32_t k = 0u; k < 3u; ++k) {
            const float dual = k == 0u || c.block ? lambda_env[local + k * stride] : 0.0f;
            c.F(pDual + k) = dual; c.F(pBase + k) = dual;
            c.F(pRelaxStep + k) = 0.0f; c.F(pRelaxPoint + k) = 0.0f;
        }
        c.F(pRelaxWeight) = 0.0f;
    }
    wave_sync();
    {
        float row[W], root;
        load_row(c, c.mass, row);
        c.mass_valid = factor(c, row, &c.mass_inverse, &root);
        store_row(c, c.mfac, row);
        wave_sync();
    }
    residuals_env(c, velocity, urows, p.dt);
    float residual4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t sweeps = 0u;
    DualMomentum momentum{1.0f, 0.0f};
    const float tol = c.tolerance;
    while (sweeps < p.iterations) {
        c.iteration = sweeps++;
        c.momentum = 0.0f; c.residual = 0.0f;
        descend_env(c, &velocity, free_v, true, d);
        float rowsr[3];
        duals_env(c, lambda_env, R, urows, &momentum, true, rowsr);
        if (sweeps == p.iterations || fmaxf(fmaxf(rowsr[0], rowsr[1]), fmaxf(rowsr[2], c.residual)) < tol) measure_env(c, &velocity, free_v, false, d);
        if (fmaxf(fmaxf(rowsr[0], rowsr[1]), rowsr[2]) < tol && c.residual >= tol && c.residual < FLT_MAX) {
            measure_env(c, &velocity, free_v, true, d);
            if (c.residual < FLT_MAX) {
                residuals_env(c, velocity, urows, p.dt);
                duals_env(c, lambda_env, R, urows, nullptr, false, rowsr);
                c.residual = 0.0f;
                measure_env(c, &velocity, free_v, false, d);
            }
        }
        residual4[0] = rowsr[0]; residual4[1] = rowsr[1]; residual4[2] = rowsr[2]; residual4[3] = c.residual;
        const float largest = fmaxf(fmaxf(rowsr[0], rowsr[1]), fmaxf(rowsr[2], c.residual));
        if (largest < tol || largest == FLT_MAX) break;
    }
    if (lane < 4u)
        d.solver_residual[size_t{env} * 4u + lane] = lane == 0u ? residual4[0] : lane == 1u ? residual4[1] : lane == 2u ? residual4[2] : residual4[3];
    if (lane == 0u) {
        d.vbd_velocity_sweep_count[env] = sweeps;
        d.solver_cost[env] = solve_cost_after(d.solver_cost[env], c.work);
        if (d.solver_points != nullptr) d.solver_points[env] = points_solved(d.solver_points[env]);
    }
    if (lane < md) {   // (a block of at most W coordinates has no more words a row than lanes)
        d.solver_velocity[size_t{env} * md + lane] = coordinate ? velocity : 0.0f;
        d.solver_free[size_t{env} * md + lane] = coordinate ? free_v : 0.0f;
    }
    const bool invalid = c.any(coordinate && !(fabsf(velocity) <= FLT_MAX));
    if (!invalid) {
        if (lane < md) d.qdot_flat[size_t{env} * md + lane] = coordinate ? velocity : 0.0f;
        if (coordinate) {
            if (my_component == kInvalid) d.qdot[lbase + my_link] = velocity;
            else d.link_velocity[(lbase + my_link) * 6u + my_component] = velocity;
        }
    } else if (lane == 0u) d.env_status[env] |= kEnvStatusSolverFailure;
    if (p.base_link_count != 0u && p.joint_limit_rows_per_env >= 2u * p.base_link_count) {
        for (uint32_t l = lane; l < nl; l += 16u) {
            const size_t lower = size_t{env} * R + p.contact_rows_per_env + size_t{l} * 2u;
            d.joint_limit_impulse[2u * (lbase + l)] = (__float_as_uint(urows[lower * kRowWords]) & kRowActive) != 0u ? d.lambda[lower] : 0.0f;
            d.joint_limit_impulse[2u * (lbase + l) + 1u] = (__float_as_uint(urows[(lower + 1u) * kRowWords]) & kRowActive) != 0u ? d.lambda[lower + 1u] : 0.0f;
        }
    }
    // split-impulse position pass
    if (p.position_iterations != 0u) {
        const float moving = coordinate ? velocity : 0.0f;
        double vel_a = 0.0, vel_b = 0.0;   // of a speculative row's two sides
        float bias = 0.0f, rounding = 0.0f;
        bool position = false, speculative = false;
        if (c.live) {
            const float* row = urows + size_t{slot} * kRowWords;
            const uint32_t flags = __float_as_uint(row[0]);
            speculative = (flags & kRowSpeculative) != 0u;
            position = (flags & (kRowFriction | kRowVelocityOnly | kRowMuJoCo)) == 0u &&
                (speculative || d.row_penetration[slot] > p.position_slop || c.F(pDual) != 0.0f);
        }
        if (c.any(position && speculative)) {
            const bool side_a = position && source_a[0] != kInvalid, side_b = position && source_b[0] != kInvalid;
            const float* from_a = d.chain_jacobian + size_t{side_a ? slot : 0u} * md;
            const float* from_b = d.chain_jacobian_b + size_t{side_b ? slot : 0u} * md;
            each<0, W>([&](auto k) {
                constexpr int K = decltype(k)::value;
                const double v = double(row_lane<K>(moving));
                if (uint32_t(K) >= n) return;
                if (side_a) vel_a += double(from_a[K]) * v;
                if (side_b) vel_b += double(from_b[K]) * v;
            });
        }
        if (position) {
            const float* row = urows + size_t{slot} * kRowWords;
            const float penetration = d.row_penetration[slot], slop = speculative ? 0.0f : p.position_slop;
            if (speculative) {
                const uint32_t group_first = __float_as_uint(row[1]), points = __float_as_uint(row[2]), S = p.contact_slots_per_env;
                uint32_t contact = 0u;
                for (uint32_t s = 0u; s < S; ++s)
                    if (d.ucontact_row_range[(size_t{env} * S + s) * 2u] == group_first &&
                        d.ucontact_row_range[(size_t{env} * S + s) * 2u + 1u] > 0u) contact = env * S + s;
                const size_t point = size_t{contact} * 4u + (slot - group_first) % points;
                const double depth = double(d.ucontact_depth[point]) - slop;
                const double reserve = double(penetration) - d.ucontact_depth[point];
                const double correction = p.position_beta * fmax(depth, 0.0) + reserve;
                const double target = fmin(depth, 0.0) + correction;
                const double vel = vel_a + vel_b;
                const double limit = fmin(correction / p.dt, double(p.position_max_velocity));
                const double absorbed = target > 0.0 ? 0.0 : fmax(reserve, 0.0) / p.dt;
                bias = float(fmin(target / p.dt - vel, limit));
                rounding = float(absorbed);
            } else {
                const float pen = fmaxf(penetration - slop, 0.0f);
                const float correction = p.position_beta * pen + fmaxf(pen - pen, 0.0f);
                bias = fminf(correction / p.dt, p.position_max_velocity);
            }
        }
        c.owned = c.owned && position;
        c.block = false;   // on one axis now
        if (c.live) {
            const Response answer = scalar_response(c.F(pRho), 0.0f);
            c.F(pCompliance) = 0.0f; c.F(pLower) = 0.0f; c.F(pUpper) = FLT_MAX;
            c.F(pDualScale) = answer.dual_scale; c.F(pResidualScale) = answer.residual_scale;
            c.F(pRes) = bias;
#pragma unroll
            for (uint32_t k = 0u; k < 3u; ++k) { c.F(pDual + k) = 0.0f; if (k != 0u) c.F(pRes + k) = 0.0f; }
        }
        float pseudo = 0.0f;
        if (c.any(c.live && bias > rounding)) {
            c.iteration = sweeps;
            descend_env(c, &pseudo, 0.0f, false, d);   // no head couples two moving blocks here, so one solve
        }
        if (coordinate) {
            if (my_component == kInvalid) d.qdot_pseudo[lbase + my_link] = pseudo;
            else d.link_velocity_pseudo[(lbase + my_link) * 6u + my_component] = pseudo;
        }
    }
}

}  // namespace solver
}  // namespace nkh
