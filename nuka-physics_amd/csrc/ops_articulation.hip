// Articulation ops for gfx950: forward kinematics, forward dynamics (RNEA bias + CRBA + LDL^T solve), position
// integration and link twists.  One 64-lane wavefront owns one environment (the forward dynamics runs two, its bias
// forces and its mass matrix side by side): lanes are links in the tree sweeps, matrix entries in the 6x6 inertia
// pushes, and matrix rows in the factorisation; every per-link quantity of the environment lives in LDS between the
// sweeps and reaches HBM once, in contiguous env-major blocks.
//
// Replaces src/phi/backend_cuda/ops/articulation.cu (UpdateWorldLinkPosesKernel :1561-1596,
// ArticulationDynamicsKernel :505-645, IntegratePositionArticulationKernel :764-791, FkLinkVelocitiesKernel
// :647-689) and articulation_mass.cuh (ComputeArticulationMass :124-253, FactorMass :269-335,
// SolveMassBlock :357-396).
#include "nk_device_math.h"
#include "nk_body_pose.h"
#include "backend.h"
#include "nk_ops.h"

#include <type_traits>

namespace nkh {

namespace {

constexpr int kWave = 64;

__device__ __forceinline__ V3 load3(const float* p) { return V3{p[0], p[1], p[2]}; }

// kinematics.cuh:25-42 JointRelativeFrame (revolute / prismatic / fixed)
__device__ Xf joint_relative_frame(uint8_t type, V3 axis, Xf local, V3 parent_offset, float coordinate) {
    Xf result = local;
    result.p = add3(local.p, parent_offset);
    const float l = dot3(axis, axis);
    axis = l > 1.0e-12f ? scale3(axis, rsqrt_exact(l)) : V3{0.0f, 0.0f, 0.0f};
    if (type == kRevolute) {
        const float half = 0.5f * coordinate;
        const float sine = sinf(half);
        const Q4 turn{cosf(half), axis.x * sine, axis.y * sine, axis.z * sine};
        result.r = qnormalize_le(qmul(local.r, turn), 1.0e-12f);
    } else if (type == kPrismatic) {
        result.p = add3(result.p, rotate_normalized(local.r, scale3(axis, coordinate)));
    }
    return result;
}

// articulation.cu:91-124
__device__ void mat3_from_quat(Q4 q, float* m) {
    const float n = q.w * q.w + q.x * q.x + q.y * q.y + q.z * q.z;
    if (n <= 1.0e-12f) {
        m[0] = 1; m[1] = 0; m[2] = 0; m[3] = 0; m[4] = 1; m[5] = 0; m[6] = 0; m[7] = 0; m[8] = 1;
        return;
    }
    const float inv = rsqrt_exact(n);
    q.w *= inv; q.x *= inv; q.y *= inv; q.z *= inv;
    const float xx = q.x * q.x, yy = q.y * q.y, zz = q.z * q.z, xy = q.x * q.y, xz = q.x * q.z, yz = q.y * q.z;
    const float wx = q.w * q.x, wy = q.w * q.y, wz = q.w * q.z;
    m[0] = 1.0f - 2.0f * (yy + zz); m[1] = 2.0f * (xy - wz); m[2] = 2.0f * (xz + wy);
    m[3] = 2.0f * (xy + wz); m[4] = 1.0f - 2.0f * (xx + zz); m[5] = 2.0f * (yz - wx);
    m[6] = 2.0f * (xz - wy); m[7] = 2.0f * (yz + wx); m[8] = 1.0f - 2.0f * (xx + yy);
}

// articulation.cu:126-147
__device__ void mat3_axis_angle(V3 axis, float angle, float* m) {
    const float l = dot3(axis, axis);
    if (l <= 1.0e-12f) {
        m[0] = 1; m[1] = 0; m[2] = 0; m[3] = 0; m[4] = 1; m[5] = 0; m[6] = 0; m[7] = 0; m[8] = 1;
        return;
    }
    axis = scale3(axis, rsqrt_exact(l));
    const float c = cosf(angle), s = sinf(angle), t = 1.0f - c;
    m[0] = t * axis.x * axis.x + c; m[1] = t * axis.x * axis.y - s * axis.z; m[2] = t * axis.x * axis.z + s * axis.y;
    m[3] = t * axis.x * axis.y + s * axis.z; m[4] = t * axis.y * axis.y + c; m[5] = t * axis.y * axis.z - s * axis.x;
    m[6] = t * axis.x * axis.z - s * axis.y; m[7] = t * axis.y * axis.z + s * axis.x; m[8] = t * axis.z * axis.z + c;
}

__device__ void mat3_mul(const float* a, const float* b, float* out) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) out[r * 3 + c] = a[r * 3] * b[c] + a[r * 3 + 1] * b[c + 3] + a[r * 3 + 2] * b[c + 6];
}

// articulation.cu:149-171: X = [[E, 0], [-E skew(t), E]] written to a 36-float LDS tile
__device__ void store_motion_transform(const float* E, V3 t, float* X) {
    const float skew[9] = {0.0f, -t.z, t.y, t.z, 0.0f, -t.x, -t.y, t.x, 0.0f};
    float ll[9];
    mat3_mul(E, skew, ll);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            X[r * 6 + c] = E[r * 3 + c];
            X[r * 6 + c + 3] = 0.0f;
            X[(r + 3) * 6 + c] = -ll[r * 3 + c];
            X[(r + 3) * 6 + c + 3] = E[r * 3 + c];
        }
}

// articulation.cu:259-277 JointTransform
__device__ void joint_transform(const ModelView& m, uint32_t link, float q, float* X) {
    const uint8_t type = m.joint_type[link];
    const V3 axis = load3(m.joint_axis + 3u * link);
    const Xf local = load_xf(m.link_local_pose + 7u * link);
    const V3 offset = load3(m.parent_offset + 3u * link);
    float joint[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    V3 translation = add3(local.p, offset);
    if (type == kRevolute) mat3_axis_angle(axis, q, joint);
    else if (type == kPrismatic) translation = joint_relative_frame(type, axis, local, offset, q).p;
    float lr[9], rot[9], E[9];
    mat3_from_quat(local.r, lr);
    mat3_mul(lr, joint, rot);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) E[r * 3 + c] = rot[c * 3 + r];
    store_motion_transform(E, translation, X);
}

// articulation.cu:194-211
__device__ void motion_subspace(uint8_t type, V3 axis, float* s) {
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] = 0.0f;
    const float l = dot3(axis, axis);
    if (l > 1.0e-12f) axis = scale3(axis, rsqrt_exact(l));
    if (type == kRevolute) { s[0] = axis.x; s[1] = axis.y; s[2] = axis.z; }
    else if (type == kPrismatic) { s[3] = axis.x; s[4] = axis.y; s[5] = axis.z; }
}

// ---- FkWorldPoses ---------------------------------------------------------------------------------------
// The sweeps down the tree give a link a lane, and an environment `G` lanes of a wavefront: where its links need no more
// than half, a quarter or an eighth of one, as many environments share it, and each instruction serves them all
// (the poses of 31 links: 127 us a wavefront each, 70 us two a wavefront, at 65536 environments; of 8 links: 32 and 9 us at
// 20011).  The sharing stops where it would leave one of the chip's 1024 SIMDs without a wavefront.  More than 64 links take
// two each ("128 lanes"): prepared ahead like the first, where a link that is prepared again at every depth of a 65-link
// chain doubled its sweep (227 and 106 us at 8192).
constexpr uint32_t kSimds = 1024u;
inline uint32_t LanesAnEnvironment(uint32_t links, uint32_t envs) {
    if (links > 64u) return 128u;
    uint32_t lanes = 64u;
    while (lanes > 8u && links <= lanes / 2u && uint64_t{envs} * (lanes / 2u) >= uint64_t{kSimds} * 64u) lanes /= 2u;
    return lanes;
}

// One environment by `G` lanes of one wavefront (128: by all 64, two links each); `pose` holds nl * 7 words of LDS.  Every lane of the wavefront is in the
// call, those without an environment with `there` false.
template <int G>
__device__ __forceinline__ void world_poses_of_env(const ModelView& m, const DataView& d, uint32_t env, uint32_t lane, bool there, float* pose) {
    const uint32_t nl = there ? m.links_per_env : 0u;
    const float* q = d.q + size_t{env} * m.links_per_env;
    // A link's frame in its parent does not wait on the tree: every lane computes its own links' before the sweep, which
    // then only composes a depth at a time (links past the second a lane compute theirs when their depth comes).
    struct Placed { uint32_t depth, parent; Xf frame; };
    auto place = [&](uint32_t l) {
        const uint8_t type = m.joint_type[l];
        const uint32_t parent = m.parent_link[l];
        const Xf relative = joint_relative_frame(type, load3(m.joint_axis + 3u * l), load_xf(m.link_local_pose + 7u * l),
                                                 load3(m.parent_offset + 3u * l), q[l]);
        return Placed{m.link_tree_depth[l], parent, parent == kInvalid && type == kFloatingBase ? load_xf(d.base_pose + size_t{env} * 7u) : relative};
    };
    auto compose = [&](uint32_t l, const Placed& t) {
        store_xf(pose + 7u * l, t.parent == kInvalid ? t.frame : compose_frame(load_xf(pose + 7u * t.parent), t.frame));
    };
    constexpr int kOwn = G > kWave ? 2 : 1, kLanes = G / kOwn;   // fewer links than nl only past the second a lane
    Placed own[kOwn];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
        own[i] = Placed{kInvalid, kInvalid, Xf{}};
        if (lane + uint32_t(i * kLanes) < nl) own[i] = place(lane + uint32_t(i * kLanes));
    }
    for (uint32_t depth = 0u; depth <= m.max_depth; ++depth) {
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
            if (own[i].depth == depth) compose(lane + uint32_t(i * kLanes), own[i]);
        if (G > kWave)
            for (uint32_t l = lane + 2u * kWave; l < nl; l += kWave) {
                const Placed t = place(l);
                if (t.depth == depth) compose(l, t);
            }
        wave_sync();
    }
    float* out = d.link_pose + size_t{env} * m.links_per_env * 7u;
    for (uint32_t e = lane; e < nl * 7u; e += kLanes) out[e] = pose[e];
}
template <int G>
__global__ void __launch_bounds__(kWave) FkWorldPosesKernel(ModelView m, DataView d, uint32_t env_count) {
    extern __shared__ float lds[];
    constexpr uint32_t kLanes = G < kWave ? G : kWave;
    const uint32_t group = threadIdx.x / kLanes, env = blockIdx.x * (kWave / kLanes) + group;
    world_poses_of_env<G>(m, d, env, threadIdx.x % kLanes, env < env_count, lds + group * m.links_per_env * 7u);
}

// ---- ArticulationDynamics -------------------------------------------------------------------------------
// Two wavefronts a workgroup, and G lanes of each an environment, so that a workgroup takes 64 / G environments.  The bias
// forces (velocities, bias accelerations, the leaf-to-root force pass) and the mass matrix (composite inertias, columns) do
// not depend on each other, and each is a chain of tree sweeps that keeps a few lanes an environment busy: the first
// wavefront takes the one, the second the other, side by side, each for all environments of the workgroup.  Then they meet,
// and each factors and solves half of the environments, 2 G lanes each (of a workgroup's only one, the second wavefront
// does, while the first carries the matrix and its factor to memory).  Every instruction of a sweep serves 64 / G
// environments: the kernel is bound by the instructions it issues where environments outnumber the wavefronts, not by
// memory.  Fewer lanes give the sweeps fewer links a pass; DynamicsLanes says where that pays.
__host__ __device__ constexpr uint32_t DynamicsSlots(uint32_t lanes) { return lanes >= 64u ? kSweepLinks : lanes >= 32u ? 5u : lanes >= 16u ? 2u : 1u; }
// three places past the links: what a root hangs from, what a floating root does, and one for lanes without a link
constexpr uint32_t kGround = 0u, kBase = 1u, kNobody = 2u, kPlaces = 3u;
// a link's record and its place in the children's list, and the sweeps' list with its length and steps past its end
__host__ __device__ inline uint32_t DynamicsTreeWords(uint32_t nl, uint32_t sweep_passes) {
    return (nl + kPlaces) * 2u + nl + (sweep_passes + 3u) * kSweepLinks + 1u;
}
// links a lane has in the pass over the mass columns, and whether the matrix may take the composite inertias' place: when
// every link's inertia has been read by then
__host__ __device__ constexpr uint32_t DynamicsLinksALane(uint32_t lanes) { return lanes >= 64u ? 2u : 1u; }
__host__ __device__ inline uint32_t DynamicsMatrixWords(uint32_t nl, uint32_t n, uint32_t envs) {   // the inertias and the matrix
    const uint32_t inertias = nl * 36u, matrix = n * (n | 1u), lanes = 64u / envs;
    return nl <= lanes * DynamicsLinksALane(lanes) ? (inertias > matrix ? inertias : matrix) : inertias + matrix;
}
__host__ __device__ inline uint32_t DynamicsEnvWords(uint32_t nl, uint32_t n, uint32_t envs) {
    const uint32_t words = (nl + kPlaces) * (18u + 5u * 6u) + nl + DynamicsMatrixWords(nl, n, envs) + 2u * n + 36u;
    const uint32_t apart = 64u / envs;   // one place of the environments in different banks
    return envs == 1u ? words : (words + 63u - apart) / 64u * 64u + apart;
}

// v of lane K of the L lanes an environment has
template <int L, int K>
__device__ __forceinline__ float group_value(float v) {
    typedef float Vec4 __attribute__((ext_vector_type(4)));
    if constexpr (L == 64) return lane_value(v, K);
    else if constexpr (L == 16) return dpp_move<0x150 + K>(v);   // a row's lane K to the whole row
    else return __builtin_amdgcn_mfma_f32_4x4x1f32(v, 1.0f, Vec4{}, 3, K / 4, 0)[K % 4];   // a block's four to eight blocks
}
// LDL^T of the matrix whose row `lane` is `row`, L lanes a matrix: the strict lower triangle becomes L and the diagonal D
// (:269-335).  Entry (i, j) loses (L_ik L_jk) D_k for k = 0, 1, ... with the three roundings of the serial loop (fused into
// one multiply-add an entry the factor differs in its last place, which an environment that does not converge in its sweeps
// hands on: one of 256 driven humanoids then ends 2.5e-4 from the oracle's).  The products L_ik L_jk come four columns an
// instruction, columns 4 Q .. 4 Q + 3 of lane's row at a time: v_mfma_f32_4x4x1 multiplies four values a block of four lanes
// with one a lane, and its broadcast of block Q's four to the L / 4 blocks (cbsz, abid) takes the multipliers' own register
// for them, where a lane read and a product an entry went before.  What a lane computes above its diagonal is never read.
typedef float Vec4 __attribute__((ext_vector_type(4)));
template <int L>
constexpr int kBlocksLog = L == 64 ? 4 : L == 32 ? 3 : 2;
template <int L, int Q, int K, int N>
__device__ __forceinline__ void subtract_products(float lik, float diagonal, float (&row)[N]) {
    if constexpr (4 * Q < N) {
        const Vec4 product = __builtin_amdgcn_mfma_f32_4x4x1f32(lik, lik, Vec4{}, kBlocksLog<L>, Q, 0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (4 * Q + t > K) row[4 * Q + t] -= product[t] * diagonal;
        subtract_products<L, Q + 1, K>(lik, diagonal, row);
    }
}
template <int L, int K, int N>
__device__ __forceinline__ void ldlt_pivots(uint32_t lane, float (&row)[N]) {
    if constexpr (K < N) {
        const float diagonal = fmaxf(group_value<L, K>(row[K]), 1.0e-6f);
        const float lik = div_by(row[K], make_recip(diagonal));   // the quotient to the bit; zero where an armature past 2^126 holds the joint
        row[K] = lane > uint32_t(K) ? lik : (lane == uint32_t(K) ? diagonal : row[K]);
        subtract_products<L, (K + 1) / 4, K>(lik, diagonal, row);
        ldlt_pivots<L, K + 1>(lane, row);
    }
}
template <int L, int J, int N>
__device__ __forceinline__ void forward_rows(uint32_t lane, uint32_t n, const float (&row)[N], float* x) {
    if constexpr (J < N) {
        const float solved = group_value<L, J>(*x);
        if (lane > uint32_t(J) && lane < n) *x -= row[J] * solved;
        forward_rows<L, J + 1>(lane, n, row, x);
    }
}
template <int L, int I, int N>
__device__ __forceinline__ void backward_columns(uint32_t lane, const float (&col)[N], float* x) {
    if constexpr (I >= 0) {
        const float value = group_value<L, I>(*x);
        if (lane < uint32_t(I)) *x -= col[I] * value;
        backward_columns<L, I - 1>(lane, col, x);
    }
}
// A matrix of LDS to its stride x stride words of memory by a whole wavefront: all of it, or (kLower) the lower triangle of
// a factor, as sixteen-byte words (kWide) where the rows start on them.  Rows and columns past n are zero, but for a factor's
// diagonal.  Row and column of a lane's words step with it, a division by the stride a word costing more than the word.
struct TilePlace {
    uint32_t wide, row, word, rows_a_step, words_a_step;
    __device__ __forceinline__ TilePlace(uint32_t wide_, uint32_t stride, uint32_t lane) : wide(wide_) {
        const uint32_t words = stride / wide;
        row = lane / words; word = lane - row * words;
        rows_a_step = uint32_t(kWave) / words; words_a_step = uint32_t(kWave) - rows_a_step * words;
    }
};
template <bool kLower, bool kWide>
__device__ __forceinline__ void store_tile(const TilePlace& place, float* out, const float* A, uint32_t n, uint32_t ld, uint32_t stride, uint32_t lane) {
    auto word = [&](uint32_t i, uint32_t j) {
        if (kLower) return i < n ? A[i * ld + min(j, i)] : (i == j ? 1.0e-6f : 0.0f);
        const float v = A[min(i, n - 1u) * ld + min(j, n - 1u)];
        return i < n && j < n ? v : 0.0f;
    };
    const uint32_t wide = kWide ? place.wide : 1u, words = stride / wide;
    uint32_t i = place.row, q = place.word;
    for (uint32_t e = lane; e < stride * words; e += kWave) {
        const uint32_t j = wide * q;
        if (wide == 1u) {
            if (!kLower || j <= i) out[e] = word(i, j);
        } else if (!kLower || j + 3u <= i) {
            const float* four = A + i * ld + j;
            reinterpret_cast<float4*>(out)[e] = n == stride ? float4{four[0], four[1], four[2], four[3]}   // (nothing is past the matrix)
                                                            : float4{word(i, j), word(i, j + 1u), word(i, j + 2u), word(i, j + 3u)};
        } else {
            for (uint32_t t = 0u; j + t <= i; ++t) out[i * stride + j + t] = word(i, j + t);
        }
        i += place.rows_a_step; q += place.words_a_step;
        if (q >= words) { q -= words; ++i; }
    }
}
// A link's motion transform X = [[E, 0], [L, E]] as its two blocks, E then L (the products with the zeros add nothing).
// X^T f, each entry summed in the order of the whole product
__device__ __forceinline__ void push_force(const float* X, const float (&f)[6], float (&out)[6]) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        float upper = 0.0f, lower = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; ++c) upper += X[3 * c + r] * f[c];
#pragma unroll
        for (int c = 0; c < 3; ++c) { upper += X[9 + 3 * c + r] * f[3 + c]; lower += X[3 * c + r] * f[3 + c]; }
        out[r] = upper; out[3 + r] = lower;
    }
}
// A row of X as a lane of the sweeps holds it: the words its first three terms take and those of the other three, which
// an angular row does not have; row times x (six words), likewise
struct TransformRow { float first[3], second[3]; };
__device__ __forceinline__ TransformRow load_transform_row(const float* X, uint32_t row) {
    const float* first = X + 3u * row, *second = X + 3u * (row < 3u ? row : row - 3u);   // L's rows follow E's
    return TransformRow{{first[0], first[1], first[2]}, {second[0], second[1], second[2]}};
}
__device__ __forceinline__ float transform_row(const TransformRow& X, uint32_t row, const float (&x)[6]) {
    float value = 0.0f;
#pragma unroll
    for (int c = 0; c < 3; ++c) value += X.first[c] * x[c];
    const float angular = value;
#pragma unroll
    for (int c = 0; c < 3; ++c) value += X.second[c] * x[3 + c];
    return row < 3u ? angular : value;
}

// A link's record in LDS: its parent's place (a root's is one past the links), joint type and first coordinate; the place of
// its children in their list and their number.
struct LinkRecord {
    uint32_t low, high;
    __device__ __forceinline__ uint32_t parent() const { return low & 0xFFFFu; }
    __device__ __forceinline__ uint8_t type() const { return uint8_t(low >> 16u); }
    __device__ __forceinline__ uint32_t dof() const { return low >> 24u; }
    __device__ __forceinline__ uint32_t child_begin() const { return high & 0xFFFFu; }
    __device__ __forceinline__ uint32_t children() const { return high >> 16u; }
};
__device__ __forceinline__ uint32_t times(uint32_t words, uint32_t link) { return __umul24(words, link); }

// Compiled per padded DoF width N (a multiple of 4): the LDL^T factorisation and the solve keep one matrix row per
// lane in registers, fully unrolled, and hand pivots and multipliers round the environment's lanes.
// The tree sweeps run six lanes a link - a lane a row of the link's 6x6 products - and up to ten links a pass, a depth at a
// time from the cooked pass list (ModelView::sweep_links): a pass costs about a third of the instructions of a lane a
// link carrying all six rows, and each row sums in the order the whole product does.  A lone wavefront is bound by the chain
// of a pass, and each dependent read of LDS on it is some 130 cycles: what a pass reads beside the values of the pass before -
// the links, their records, their rows of X - is read a pass or two ahead, roots and lanes without a link have places of
// their own so that no read stands under a condition, and the matrix takes the inertias' place (a pass of 64 arms 900 -> 400
// cycles, the kernel 19.4 -> 16.9 us; 4096 humanoids 118 -> 98 us, 65536 1405 -> 1133 us, 8192 ropes 1633 -> 1031 us).
// With a third wavefront the kernel is FkWorldPoses too (OpPosesAndDynamics): that one places the links beside the other two,
// which ask for a pose only where a link has a wrench on it.
template <int N, int G>
__device__ __forceinline__ void dynamics_of_block(const ModelView& m, const DataView& d, const ArticulationDynamicsParams& p, uint32_t env_count, float* lds) {
    const bool places = blockDim.x > 2u * kWave;
    constexpr uint32_t kEnvs = kWave / G, kRowLanes = G < 32 ? 2u * G : 64u;
    static_assert(N <= int(kRowLanes), "a lane a row");
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, nl = m.links_per_env, n = m.dof, stride = m.max_dof;
    const bool forces = wave == 0u;
    // the tree as the sweeps read it: a record a link, the children's list, and the sweeps' list, kSlots places a step, nobody's
    // where a step has fewer links and in three steps past the end, with its number of steps
    constexpr uint32_t kSlots = DynamicsSlots(G);
    LinkRecord* records = reinterpret_cast<LinkRecord*>(lds);
    uint32_t* t_children = reinterpret_cast<uint32_t*>(records + nl + kPlaces);
    uint32_t* sweep_steps = t_children + nl;
    uint32_t* sweep = sweep_steps + 1u;
    const uint32_t passes = m.sweep_passes;
    const uint32_t ld = n | 1u;
    struct Words { float *xup, *S, *vb, *v, *ic, *a, *pf, *A, *vel, *acc, *tmp, *rate; };
    auto words_of = [&](uint32_t index) {
        float* base = lds + DynamicsTreeWords(nl, passes) + index * DynamicsEnvWords(nl, n, kEnvs);
        Words w;
        const uint32_t places = nl + kPlaces;
        w.xup = base;                    // motion transforms, eighteen words a link
        w.S = w.xup + places * 18u;
        w.vb = w.S + places * 6u;
        w.v = w.vb + places * 6u;
        w.a = w.v + places * 6u;         // link accelerations: bias pass (first wavefront), and again the final pass
        w.pf = w.a + places * 6u;        // bias forces (first wavefront)
        w.ic = w.pf + places * 6u;       // composite inertias (second wavefront)
        // n x ld: mass matrix, then its factor (second wavefront), in the inertias' place where they are read by then
        w.A = nl <= uint32_t(G) * DynamicsLinksALane(G) ? w.ic : w.ic + nl * 36u;
        w.vel = w.ic + DynamicsMatrixWords(nl, n, kEnvs);
        w.acc = w.vel + n;
        w.rate = w.acc + n;
        w.tmp = w.rate + nl;         // 36 words of the inertia push
        return w;
    };
    // of a third wavefront: the links' poses, and whether they stand (a word, its place the environments' poses' last)
    float* poses = lds + DynamicsTreeWords(nl, passes) + kEnvs * DynamicsEnvWords(nl, n, kEnvs);
    volatile uint32_t* posed = reinterpret_cast<uint32_t*>(poses + kEnvs * nl * 7u);
    if (wave == 2u) {
        const uint32_t group = lane / G, env = blockIdx.x * kEnvs + group;
        if (lane == 0u) *posed = 0u;
        __syncthreads();
        world_poses_of_env<G>(m, d, env, lane % G, env < env_count, poses + group * nl * 7u);   // G holds an environment's links
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0u) *posed = 1u;
        __syncthreads();
        if constexpr (kEnvs == 1u) { __syncthreads(); __syncthreads(); }
        return;
    }
    const V3 gravity{p.gravity[0], p.gravity[1], p.gravity[2]};
    // Step by step down the sweeps' list: `fetch` a link's constants one step ahead, `use` them with the values of the step
    // before.  A lane without a link sweeps nobody's place, so that no step asks which lanes it is for.
    const uint32_t nobody = nl + kNobody;
    auto sweep_down = [&](uint32_t steps, uint32_t slot, auto&& fetch, auto&& use) {
        const bool takes = slot < kSlots;
        const uint32_t* list = sweep + (takes ? slot : 0u);
        auto link_at = [&](uint32_t step) { const uint32_t l = list[step * kSlots]; return takes ? l : nobody; };
        uint32_t here = link_at(0u), next = link_at(1u);
        auto constants = fetch(here);
#pragma unroll 1
        for (uint32_t step = 0u; step < steps; ++step) {
            const uint32_t after = link_at(step + 2u);
            const auto ahead = fetch(next);
            use(here, constants);
            wave_sync();
            here = next; next = after; constants = ahead;
        }
    };
    // (where a lane's words of a matrix lie takes divisions: ahead of the first barrier they wait beside reads of memory)
    const uint32_t aligned = uint32_t((reinterpret_cast<uintptr_t>(d.m) | reinterpret_cast<uintptr_t>(d.m_factor)) & 15u);
    const TilePlace place(N > 16 && (stride & 3u) == 0u && aligned == 0u ? 4u : 1u, stride, lane);
    {
        // the tree phase: G lanes an environment; a group past the last environment repeats it and writes nothing
        const uint32_t gl = lane % G, group = lane / G;
        const bool there = blockIdx.x * kEnvs + group < env_count;
        const uint32_t env = min(blockIdx.x * kEnvs + group, env_count - 1u);
        const Words w = words_of(group);
        const size_t lbase = size_t{env} * nl;
        const float* q = d.q + lbase;
        const float* qd = d.qdot + lbase;
        const uint32_t slot = gl / 6u, srow = gl - 6u * slot;   // of the sweeps: lanes past the slots' sit them out
        const uint32_t ri = srow % 3u, rj = (ri + 1u) % 3u, rk = (ri + 2u) % 3u;
        if (!forces) {   // what the mass matrix starts from and the sweeps' tables, while the first wavefront builds the joint transforms
            for (uint32_t e = gl; e < nl * 36u; e += G) w.ic[e] = m.link_inertia[e];
            for (uint32_t l = gl; l < nl; l += G) w.rate[l] = qd[l];
            for (uint32_t l = lane; l < nl; l += kWave) {
                const uint32_t begin = m.link_child_range[2u * l];
                const uint32_t parent = m.parent_link[l], type = m.joint_type[l];
                const uint32_t hangs = parent != kInvalid ? parent : nl + (type == kFloatingBase ? kBase : kGround);
                records[l] = LinkRecord{hangs | (type << 16u) | (m.link_dof[l] << 24u), (begin & 0xFFFFu) | ((m.link_child_range[2u * l + 1u] - begin) << 16u)};
                t_children[l] = m.link_children[l];
            }
            if (lane < kPlaces) records[nl + lane] = LinkRecord{nobody | (kFixed << 16u), 0u};
            if constexpr (G == 64) {
                for (uint32_t e = lane; e < (passes + 3u) * kSweepLinks; e += kWave) sweep[e] = e < passes * kSweepLinks ? min(m.sweep_links[e], nobody) : nobody;
                if (lane == 0u) *sweep_steps = passes;
            } else {   // lane = pass: a pass of `count` links is as many steps as they fill
                uint32_t links[kSweepLinks], count = 0u;
#pragma unroll
                for (uint32_t k = 0u; k < kSweepLinks; ++k) {
                    links[k] = lane < passes ? m.sweep_links[lane * kSweepLinks + k] : kInvalid;
                    count += links[k] != kInvalid ? 1u : 0u;
                }
                const uint32_t mine = (count + kSlots - 1u) / kSlots;
                uint32_t through = mine;
#pragma unroll
                for (int o = 1; o < kWave; o <<= 1) {
                    const uint32_t other = __shfl_up(through, o, kWave);
                    if (int(lane) >= o) through += other;
                }
#pragma unroll
                for (uint32_t k = 0u; k < kSweepLinks; ++k)
                    if (k < mine * kSlots) sweep[(through - mine) * kSlots + k] = min(links[k], nobody);
                const uint32_t all = __shfl(through, kWave - 1, kWave);
                if (lane < 3u * kSlots) sweep[all * kSlots + lane] = nobody;
                if (lane == 0u) *sweep_steps = all;
            }
        } else {
            const V3 base_gravity = rotate_inverse(load_xf(d.base_pose + size_t{env} * 7u).r, gravity);
            // what the roots hang from: at rest, and accelerating against gravity (in the base's own frame for a floating one)
            if (gl < 6u) {
                const uint32_t k = gl % 3u;
                const float world = k == 0u ? gravity.x : k == 1u ? gravity.y : gravity.z, local = k == 0u ? base_gravity.x : k == 1u ? base_gravity.y : base_gravity.z;
                w.v[6u * (nl + kGround) + gl] = 0.0f; w.v[6u * (nl + kBase) + gl] = 0.0f;
                w.a[6u * (nl + kGround) + gl] = gl < 3u ? 0.0f : -world; w.a[6u * (nl + kBase) + gl] = gl < 3u ? 0.0f : -local;
            }
            // link twists of the state enter LDS (a floating root's twist is state; the rest is rebuilt)
            for (uint32_t e = gl; e < nl * 6u; e += G) w.v[e] = d.link_velocity[lbase * 6u + e];
            // joint transforms and motion subspaces (articulation.cu:318-332)
            for (uint32_t l = gl; l < nl; l += G) {
                float X[36];
                if (m.parent_link[l] == kInvalid && m.joint_type[l] == kFloatingBase) {
                    const float id[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
                    store_motion_transform(id, V3{0.0f, 0.0f, 0.0f}, X);
#pragma unroll
                    for (int i = 0; i < 6; ++i) { w.S[6u * l + i] = 0.0f; w.vb[6u * l + i] = 0.0f; }
                } else {
                    joint_transform(m, l, q[l], X);
                    motion_subspace(m.joint_type[l], load3(m.joint_axis + 3u * l), w.S + 6u * l);
                }
#pragma unroll
                for (int e = 0; e < 9; ++e) { w.xup[18u * l + e] = X[(e / 3) * 6 + e % 3]; w.xup[18u * l + 9u + e] = X[(e / 3 + 3) * 6 + e % 3]; }
            }
        }
        __syncthreads();
        const uint32_t steps = *sweep_steps;
        if (forces) {
            struct Constants { LinkRecord record; TransformRow X; float add; };
            // velocities root to leaf (:334-363)
            // (a floating root's twist is state: its joint moves nothing, and its own words are what is added)
            sweep_down(steps, slot, [&](uint32_t l) {
                const LinkRecord record = records[l];
                const float state = w.v[times(6u, l) + srow], moved = w.S[times(6u, l) + srow] * w.rate[min(l, nl - 1u)];
                return Constants{record, load_transform_row(w.xup + times(18u, l), srow), record.parent() == nl + kBase ? state : moved};
            }, [&](uint32_t l, const Constants& k) {
                float x[6];
                const float* parent = w.v + times(6u, k.record.parent());
#pragma unroll
                for (int c = 0; c < 6; ++c) x[c] = parent[c];
                w.v[times(6u, l) + srow] = transform_row(k.X, srow, x) + k.add;
            });
            // each link's twist crossed with its joint's own twist, row by row (motion_cross); a floating root has none
            for (uint32_t l = slot; l < (slot < kSlots ? nl : 0u); l += kSlots) {
                const float* vl = w.v + 6u * l, *s6 = w.S + 6u * l;
                const float rate = w.rate[l];
                const float first = vl[rj] * (s6[(srow < 3u ? 0u : 3u) + rk] * rate) - vl[rk] * (s6[(srow < 3u ? 0u : 3u) + rj] * rate);
                const float second = vl[3u + rj] * (s6[rk] * rate) - vl[3u + rk] * (s6[rj] * rate);
                const bool state = records[l].parent() == nl + kBase;
                w.vb[6u * l + srow] = state ? 0.0f : (srow < 3u ? first : first + second);
            }
            wave_sync();
            // p = v x* (I v) - external wrench (:364-374, 279-295)
            for (uint32_t l = gl; l < nl; l += G) {
                float vl[6], iv[6], bf[6];
#pragma unroll
                for (int i = 0; i < 6; ++i) vl[i] = w.v[6u * l + i];
                mat66_vec(m.link_inertia + 36u * l, vl, iv);
                force_cross(vl, iv, bf);
                if (p.apply_link_wrench != 0u) {
                    const float* wr = d.link_wrench + (lbase + l) * 6u;
                    if (wr[0] != 0.0f || wr[1] != 0.0f || wr[2] != 0.0f || wr[3] != 0.0f || wr[4] != 0.0f || wr[5] != 0.0f) {
                        // (the third wavefront waits for nothing between the barrier above and its word)
                        if (places) while (*posed == 0u) __builtin_amdgcn_s_sleep(1);
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                        const Q4 rot = load_xf(places ? poses + (group * nl + l) * 7u : d.link_pose + (lbase + l) * 7u).r;
                        const V3 force = rotate_inverse(rot, V3{wr[0], wr[1], wr[2]});
                        const V3 torque = rotate_inverse(rot, V3{wr[3], wr[4], wr[5]});
                        const V3 moment = add3(torque, cross3(load_xf(m.link_inertial_frame + 7u * l).p, force));
                        bf[0] -= moment.x; bf[1] -= moment.y; bf[2] -= moment.z; bf[3] -= force.x; bf[4] -= force.y; bf[5] -= force.z;
                    }
                }
#pragma unroll
                for (int i = 0; i < 6; ++i) w.pf[6u * l + i] = bf[i];
            }
            wave_sync();
            // bias accelerations with gravity as base acceleration (:526-547)
            sweep_down(steps, slot, [&](uint32_t l) {
                return Constants{records[l], load_transform_row(w.xup + times(18u, l), srow), w.vb[times(6u, l) + srow]};
            }, [&](uint32_t l, const Constants& k) {
                float x[6];
                const float* parent = w.a + times(6u, k.record.parent());
#pragma unroll
                for (int c = 0; c < 6; ++c) x[c] = parent[c];
                w.a[times(6u, l) + srow] = transform_row(k.X, srow, x) + k.add;
            });
            // p += I a (:548-555)
            for (uint32_t l = gl; l < nl; l += G) {
                float al[6], f[6];
#pragma unroll
                for (int i = 0; i < 6; ++i) al[i] = w.a[6u * l + i];
                mat66_vec(m.link_inertia + 36u * l, al, f);
#pragma unroll
                for (int i = 0; i < 6; ++i) w.pf[6u * l + i] += f[i];
            }
            wave_sync();
            // leaf to root, children in CSR order (:557-569): the passes backwards, a lane a row of every child's X^T p
            {
                const bool takes = slot < kSlots;
                const uint32_t* list = sweep + (takes ? slot : 0u);
                auto link_at = [&](uint32_t back) { const uint32_t l = list[(back < steps ? steps - 1u - back : steps) * kSlots]; return takes ? l : nobody; };
                struct Child { float E[3], L[3]; };
                auto child_of = [&](const LinkRecord& record) { return t_children[min(record.child_begin(), nl - 1u)]; };
                auto push_of = [&](uint32_t child) {
                    const float* E = w.xup + times(18u, child) + ri;
                    return Child{{E[0], E[3], E[6]}, {E[9], E[12], E[15]}};
                };
                auto pushed = [&](uint32_t child, const Child& X) {
                    const float* pc = w.pf + times(6u, child), *first = pc + (srow < 3u ? 0u : 3u);
                    float value = 0.0f;
#pragma unroll
                    for (int c = 0; c < 3; ++c) value += X.E[c] * first[c];
                    const float linear = value;
#pragma unroll
                    for (int c = 0; c < 3; ++c) value += X.L[c] * pc[3 + c];
                    return srow < 3u ? value : linear;
                };
                // two steps ahead the record, one step ahead its first child's columns of X and its own force
                uint32_t here = link_at(0u), next = link_at(1u), after = link_at(2u);
                LinkRecord record = records[here], next_record = records[next];
                uint32_t child = child_of(record), next_child = child_of(next_record);
                Child X = push_of(child);
                float own = w.pf[times(6u, here) + srow];
#pragma unroll 1
                for (uint32_t back = 0u; back < steps; ++back) {
                    const uint32_t later = link_at(back + 3u);
                    const LinkRecord after_record = records[after];
                    const uint32_t after_child = child_of(after_record);
                    const Child next_X = push_of(next_child);
                    const float next_own = w.pf[times(6u, next) + srow];
                    if (record.children() != 0u) {
                        float total = own + pushed(child, X);
                        for (uint32_t i = 1u; i < record.children(); ++i) {
                            const uint32_t other = t_children[record.child_begin() + i];
                            total += pushed(other, push_of(other));
                        }
                        w.pf[times(6u, here) + srow] = total;
                    }
                    wave_sync();
                    here = next; next = after; after = later;
                    record = next_record; next_record = after_record;
                    child = next_child; next_child = after_child;
                    X = next_X; own = next_own;
                }
            }
            // generalized bias and right-hand side, lane = DoF (:570-585)
            float* bias = d.articulation_bias + size_t{env} * stride;
            for (uint32_t i = gl; i < stride; i += G) {
                if (i >= n) { if (there) bias[i] = 0.0f; continue; }
                const uint32_t link = m.dof_link[i], component = m.dof_component[i];
                const bool scalar = component == kInvalid;
                const float velocity = scalar ? qd[link] : w.v[6u * link + component];
                float b = scalar ? dot6(w.S + 6u * link, w.pf + 6u * link) : w.pf[6u * link + component];
                if (scalar) b += d.joint_gravity_force[lbase + link];   // zero unless uploaded
                const float damping = scalar ? m.joint_damping[link] + (p.fold_drive_damping != 0u ? d.drive_dissipation[lbase + link] : 0.0f) : 0.0f;
                const float spring = scalar ? m.joint_stiffness[link] * (q[link] - m.joint_spring_reference[link]) : 0.0f;
                w.vel[i] = velocity;
                if (there) bias[i] = b;
                w.acc[i] = (scalar ? d.tau[lbase + link] : 0.0f) - b - damping * velocity - spring;
            }
        } else {
            // CRBA: composite inertias leaf to root, the push X^T Ic X (articulation_mass.cuh:146-165).
            // deepest parents first, parents of one depth in link order, a parent's children in list order: the cooked visiting
            // list, sixty-four visits at a time - a lane reads one visit's child and parent, the visits take theirs as lane reads.
            // Thirty-six lanes take an entry of each product, or eighteen two that share their words (column c and c + 3 of a
            // row, row r and r + 3 of a column), or six a row and a column each.
            // (lanes past the entries repeat the last one: the same words, the same values)
            const uint32_t push_lane = min(lane, 35u), push_row = push_lane / 6u, push_column = push_lane - 6u * push_row;
            for (uint32_t first = 0u; first < nl; first += kWave) {
                uint32_t my_child = kInvalid, my_parent = 0u;
                if (first + lane < nl) {
                    my_child = m.link_push_order[first + lane];
                    if (my_child != kInvalid) my_parent = m.parent_link[my_child];
                }
                for (uint32_t visit = 0u; visit < uint32_t(kWave); ++visit) {
                    const uint32_t child = uint32_t(__builtin_amdgcn_readlane(int(my_child), int(visit)));
                    if (child == kInvalid) break;
                    const uint32_t l = uint32_t(__builtin_amdgcn_readlane(int(my_parent), int(visit)));
                    const float* E = w.xup + times(18u, child), *C = w.ic + times(36u, child);
                    float* into = w.ic + times(36u, l);
                    if constexpr (G == 64) {
                        // a lane an entry (a pair's second is three products of the six); what does not wait for the first product
                        // is read ahead of it
                        const uint32_t row = push_row, c = push_column, at = c < 3u ? c : c - 3u, out = row < 3u ? row : row - 3u;
                        const float* other = E + (c < 3u ? 9u : 0u), *beside = E + (row < 3u ? 9u : 0u);
                        float left[6], right[6], entry[6];
#pragma unroll
                        for (int k = 0; k < 6; ++k) left[k] = C[row * 6u + uint32_t(k)];
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            right[k] = E[3 * k + at]; right[3 + k] = other[3 * k + at];
                            entry[k] = E[3 * k + out]; entry[3 + k] = beside[3 * k + out];
                        }
                        const float before = into[push_lane];
                        float value = 0.0f;
#pragma unroll
                        for (int k = 0; k < 3; ++k) value += left[k] * right[k];
                        value = c < 3u ? value : 0.0f;
#pragma unroll
                        for (int k = 3; k < 6; ++k) value += left[k] * right[k];
                        w.tmp[push_lane] = value;
                        wave_sync();
                        value = 0.0f;
#pragma unroll
                        for (int k = 0; k < 3; ++k) value += entry[k] * w.tmp[k * 6 + c];
                        value = row < 3u ? value : 0.0f;
#pragma unroll
                        for (int k = 3; k < 6; ++k) value += entry[k] * w.tmp[k * 6 + c];
                        into[push_lane] = before + value;
                    } else {
                        constexpr int kPairs = G == 32 ? 1 : 3;   // a lane
                        constexpr uint32_t kLanes = G == 32 ? 18u : 6u;
                        const uint32_t row = G == 32 ? gl / 3u : gl, column = G == 32 ? gl % 3u : 0u;
                        if (gl < kLanes) {
#pragma unroll
                            for (int t = 0; t < kPairs; ++t) {
                                const uint32_t c = column + uint32_t(t);
                                float left = 0.0f, right = 0.0f;
#pragma unroll
                                for (int k = 0; k < 3; ++k) left += C[row * 6u + k] * E[3 * k + c];
#pragma unroll
                                for (int k = 0; k < 3; ++k) {
                                    left += C[row * 6u + 3u + k] * E[9 + 3 * k + c];
                                    right += C[row * 6u + 3u + k] * E[3 * k + c];
                                }
                                w.tmp[row * 6u + c] = left; w.tmp[row * 6u + 3u + c] = right;
                            }
                        }
                        wave_sync();
                        const uint32_t out_row = G == 32 ? gl / 6u : 0u, out_column = G == 32 ? gl % 6u : gl;
                        if (gl < kLanes) {
#pragma unroll
                            for (int t = 0; t < kPairs; ++t) {
                                const uint32_t r = out_row + uint32_t(t);
                                float upper = 0.0f, lower = 0.0f;
#pragma unroll
                                for (int k = 0; k < 3; ++k) upper += E[3 * k + r] * w.tmp[k * 6 + out_column];
#pragma unroll
                                for (int k = 0; k < 3; ++k) {
                                    upper += E[9 + 3 * k + r] * w.tmp[(3 + k) * 6 + out_column];
                                    lower += E[3 * k + r] * w.tmp[(3 + k) * 6 + out_column];
                                }
                                into[r * 6u + out_column] += upper; into[(r + 3u) * 6u + out_column] += lower;
                            }
                        }
                    }
                    wave_sync();
                }
            }
            // mass columns: each jointed link pushes Ic S to the root (:183-252).  First every link's Ic S and its diagonal entry,
            // and the root's own block, after which the matrix may take the inertias' place.
            const bool floating_root = m.floating_root != 0u;
            constexpr uint32_t kLinks = DynamicsLinksALane(G);
            auto jointed = [&](uint32_t l) { return l < nl && joint_dof(records[l].type()) != 0u && !(l == 0u && floating_root); };
            // (loops that stay loops, one copy of their code each: a lone wavefront waits on instructions it fetches once)
#pragma unroll 1
            for (uint32_t chunk = 0u; chunk < nl; chunk += kLinks * G) {   // past the first the matrix stands apart from the inertias
                float start[kLinks][6], diagonals[kLinks];
#pragma unroll 1
                for (uint32_t o = 0u; o < kLinks; ++o) {
                    const uint32_t l = chunk + o * G + gl;
                    float force[6] = {}, diagonal = 0.0f;
                    if (jointed(l)) {
                        float sl[6];
#pragma unroll
                        for (int i = 0; i < 6; ++i) sl[i] = w.S[6u * l + i];
                        mat66_vec(w.ic + 36u * l, sl, force);
                        diagonal = dot6(sl, force);
                        diagonal += m.joint_armature[l];
                        if (p.fold_drive_damping != 0u) diagonal += p.dt * d.drive_dissipation[lbase + l];   // articulation_mass.cuh:206-208
                    }
#pragma unroll
                    for (uint32_t k = 0u; k < kLinks; ++k) {
                        if (o != k) continue;
#pragma unroll
                        for (int i = 0; i < 6; ++i) start[k][i] = force[i];
                        diagonals[k] = diagonal;
                    }
                    if (chunk + (o + 1u) * G >= nl) break;
                }
                if (chunk == 0u) {
                    float root_block[(36 + G - 1) / G];
#pragma unroll
                    for (int o = 0; o < (36 + G - 1) / G; ++o) root_block[o] = w.ic[min(gl + uint32_t(o * G), 35u)];
                    wave_sync();
                    for (uint32_t e = gl; e < n * ld; e += G) w.A[e] = 0.0f;
                    wave_sync();
                    if (floating_root) {
#pragma unroll
                        for (int o = 0; o < (36 + G - 1) / G; ++o) {
                            const uint32_t e = gl + uint32_t(o * G);
                            if (e < 36u) w.A[(e / 6u) * ld + e % 6u] = root_block[o];
                        }
                    }
                    wave_sync();
                }
#pragma unroll 1
                for (uint32_t o = 0u; o < kLinks; ++o) {
                    const uint32_t l = chunk + o * G + gl;
                    if (chunk + o * G >= nl) break;
                    if (!jointed(l)) continue;
                    float force[6], diagonal = diagonals[0];
#pragma unroll
                    for (int i = 0; i < 6; ++i) force[i] = start[0][i];
                    if (kLinks > 1u && o != 0u) {
#pragma unroll
                        for (int i = 0; i < 6; ++i) force[i] = start[kLinks - 1u][i];
                        diagonal = diagonals[kLinks - 1u];
                    }
                    // a hop ahead: the parent's record, its axis and its transform
                    LinkRecord record = records[l];
                    const uint32_t dof_i = record.dof();
                    w.A[dof_i * ld + dof_i] = diagonal;
                    float X[18];
                    auto fetch_X = [&](uint32_t link) {
#pragma unroll
                        for (int e = 0; e < 18; ++e) X[e] = w.xup[times(18u, link) + e];
                    };
                    fetch_X(l);
                    uint32_t parent = record.parent();
                    record = records[parent];
                    while (parent < nl) {
                        float pushed[6], axis[6];
#pragma unroll
                        for (int i = 0; i < 6; ++i) axis[i] = w.S[times(6u, parent) + i];
                        push_force(X, force, pushed);
                        fetch_X(parent);
                        const LinkRecord further = records[record.parent()];
#pragma unroll
                        for (int i = 0; i < 6; ++i) force[i] = pushed[i];
                        const uint32_t dof_j = record.dof();
                        if (parent == 0u && floating_root) {
#pragma unroll
                            for (int b = 0; b < 6; ++b) { w.A[dof_i * ld + b] = force[b]; w.A[b * ld + dof_i] = force[b]; }
                        } else if (joint_dof(record.type()) != 0u) {
                            const float entry = dot6(axis, force);
                            w.A[dof_i * ld + dof_j] = entry;
                            w.A[dof_j * ld + dof_i] = entry;
                        }
                        parent = record.parent();
                        record = further;
                    }
                }
            }
        }
    }
    __syncthreads();   // the mass matrix (second wavefront) and the right-hand side (first) stand in LDS
    // The matrix phase: kRowLanes lanes an environment, half of the workgroup's environments a wavefront.  A wavefront carries
    // its environments' matrices to memory before their words take the factors.
    constexpr uint32_t kOwn = kEnvs == 1u ? 1u : kEnvs / 2u;
    const uint32_t own_first = kEnvs == 1u ? 0u : wave * kOwn;
    auto store_own = [&](auto lower, float* field) {
        for (uint32_t e = 0u; e < kOwn; ++e) {
            const uint32_t at = blockIdx.x * kEnvs + own_first + e;
            if (at < env_count) store_tile<decltype(lower)::value, (N > 16)>(place, field + size_t{at} * stride * stride, words_of(own_first + e).A, n, ld, stride, lane);
        }
    };
    if (kEnvs > 1u || forces) store_own(std::false_type{}, d.m);
    if (kEnvs == 1u && forces) {
        __syncthreads();   // the other wavefront may now overwrite the matrix with the factor
        __syncthreads();   // ... and has
        store_own(std::true_type{}, d.m_factor);
        return;
    }
    const uint32_t ml = lane % kRowLanes;
    const bool there = blockIdx.x * kEnvs + own_first + lane / kRowLanes < env_count;
    const uint32_t env = min(blockIdx.x * kEnvs + own_first + lane / kRowLanes, env_count - 1u);
    const Words w = words_of(own_first + lane / kRowLanes);
    float row[N];
    {
        // rows and columns n..N-1 are those of the identity
        // (every word read whether or not the lane keeps it, from a place inside the matrix: a read under a condition
        // compiles to a branch a word)
        const uint32_t ll = local_lane(ml);
        const uint32_t from = (ll < n ? ll : 0u) * ld;
        if (n == uint32_t(N)) {   // a lane past the matrix holds its first row, which nothing reads
#pragma unroll
            for (int k = 0; k < N; ++k) row[k] = w.A[from + uint32_t(k)];
        } else {
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const float word = w.A[from + (uint32_t(k) < n ? uint32_t(k) : 0u)];
                row[k] = ll < n && uint32_t(k) < n ? word : (ll == uint32_t(k) ? 1.0f : 0.0f);
            }
        }
    }
    ldlt_pivots<int(kRowLanes), 0>(local_lane(ml), row);
    if (kEnvs == 1u) __syncthreads(); else wave_sync();   // the matrix has been read: its words take the factor
    {
        const uint32_t ll = local_lane(ml);
        if (ll < n) {
#pragma unroll
            for (int k = 0; k < N; ++k)
                if (uint32_t(k) < n) w.A[ll * ld + k] = row[k];
        }
    }
    if (kEnvs == 1u) __syncthreads(); else { wave_sync(); store_own(std::true_type{}, d.m_factor); }
    // solve L D L^T x = rhs: forward by rows, scale, backward by columns (:357-396)
    float x = ml < n ? w.acc[ml] : 0.0f;
    {
        const uint32_t ll = local_lane(ml);
        float col[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float word = w.A[(uint32_t(i) < n ? uint32_t(i) : 0u) * ld + (ll < n ? ll : 0u)];
            col[i] = uint32_t(i) < n ? word : 0.0f;   // (taken by the lanes ahead of the diagonal alone)
        }
        forward_rows<int(kRowLanes), 0>(ll, n, row, &x);
        if (ll < n) x = x / w.A[ll * ld + ll];
        backward_columns<int(kRowLanes), N - 1>(ll, col, &x);
    }
    if (there)
        for (uint32_t i = ml; i < stride; i += kRowLanes) d.articulation_qdd[size_t{env} * stride + i] = i < n ? x : 0.0f;
    if (ml < n) w.acc[ml] = x;
    wave_sync();
    // write back accelerations and the unconstrained velocity update (:597-615)
    const size_t lbase = size_t{env} * nl;
    for (uint32_t l = ml; l < (there ? nl : 0u); l += kRowLanes) {
        float qdd = 0.0f;
        if (joint_dof(records[l].type()) == 1u) {
            const uint32_t dof = records[l].dof();
            qdd = w.acc[dof];
            if (p.integrate_velocity != 0u) d.qdot[lbase + l] = w.vel[dof] + p.dt * qdd;
        }
        d.qddot[lbase + l] = qdd;
        if (p.integrate_velocity != 0u) {
            float* wr = d.link_wrench + (lbase + l) * 6u;
#pragma unroll
            for (int i = 0; i < 6; ++i) wr[i] = 0.0f;
        }
    }
    if (m.floating_root != 0u && p.integrate_velocity != 0u && ml < 6u) {
        const uint32_t component = ml, i = component % 3u, j = (i + 1u) % 3u, k = (i + 2u) % 3u;
        const float transport = component < 3u ? 0.0f : w.vel[j] * w.vel[3u + k] - w.vel[k] * w.vel[3u + j];
        w.v[component] = w.vel[ml] + p.dt * (w.acc[ml] + transport);
    }
    wave_sync();
    // final link accelerations (:617-644)
    {
        const uint32_t slot = ml / 6u, srow = ml - 6u * slot;
        struct Constants { LinkRecord record; TransformRow X; float bias, axis, qdd; };
        sweep_down(*sweep_steps, slot, [&](uint32_t l) {
            const LinkRecord record = records[l];
            const float solved = w.acc[min(record.type() == kFloatingBase ? srow : record.dof(), n - 1u)];
            return Constants{record, load_transform_row(w.xup + times(18u, l), srow), w.vb[times(6u, l) + srow], w.S[times(6u, l) + srow],
                             joint_dof(record.type()) == 1u || record.type() == kFloatingBase ? solved : 0.0f};
        }, [&](uint32_t l, const Constants& k) {
            float x6[6];
            const float* parent = w.a + times(6u, k.record.parent());
#pragma unroll
            for (int c = 0; c < 6; ++c) x6[c] = parent[c];
            float al = transform_row(k.X, srow, x6);
            // a floating root accelerates as solved, in the base's frame
            if (k.record.type() == kFloatingBase) al = srow < 3u ? k.qdd : k.qdd + w.a[6u * (nl + kBase) + srow];
            else al += k.bias + k.axis * k.qdd;
            w.a[times(6u, l) + srow] = al;
        });
    }
    for (uint32_t e = ml; e < (there ? nl * 6u : 0u); e += kRowLanes) {
        d.link_velocity[lbase * 6u + e] = w.v[e];
        d.link_acceleration[lbase * 6u + e] = w.a[e];
    }
}

// ---- IntegratePosition: one thread per (env, link) (articulation.cu:732-791) ------------------------------
__device__ __forceinline__ void integrate_position_of_link(const ModelView& m, const DataView& d, const IntegratePositionParams& p,
                                                            uint32_t env, uint32_t l) {
    const uint32_t gid = env * m.links_per_env + l;
    const float dt = p.dt;
    if (p.pos_pass != 0u) d.q[gid] += (d.qdot[gid] + d.qdot_pseudo[gid]) * dt;
    else d.q[gid] += d.qdot[gid] * dt;
    if (m.parent_link[l] == kInvalid && m.joint_type[l] == kFloatingBase) {
        float* rv = d.link_velocity + size_t{gid} * 6u;
        Xf pose = load_xf(d.base_pose + size_t{env} * 7u);
        float vv[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) vv[i] = p.pos_pass != 0u ? rv[i] + d.link_velocity_pseudo[size_t{gid} * 6u + i] : rv[i];
        const V3 lin_world = rotate_forward(pose.r, V3{vv[3], vv[4], vv[5]});
        pose.p = add3(pose.p, scale3(lin_world, dt));
        const Q4 dq{1.0f, 0.5f * vv[0] * dt, 0.5f * vv[1] * dt, 0.5f * vv[2] * dt};
        pose.r = qnormalize_lt(qmul(pose.r, dq), 1.0e-24f);
        const V3 turned = rotate_inverse(qnormalize_lt(dq, 1.0e-24f), V3{rv[3], rv[4], rv[5]});
        rv[3] = turned.x; rv[4] = turned.y; rv[5] = turned.z;
        store_xf(d.base_pose + size_t{env} * 7u, pose);
    }
}
__global__ void IntegratePositionKernel(ModelView m, DataView d, IntegratePositionParams p) {
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= p.total_link_count) return;
    integrate_position_of_link(m, d, p, gid / m.links_per_env, gid % m.links_per_env);
}

// ---- FkLinkVelocities (articulation.cu:647-689) ---------------------------------------------------------
// One environment by `G` lanes of one wavefront, as world_poses_of_env; `v` holds nl * 6 words of LDS
template <int G>
__device__ __forceinline__ void link_velocities_of_env(const ModelView& m, const DataView& d, uint32_t env, uint32_t lane, bool there, float* v) {
    const uint32_t nl = there ? m.links_per_env : 0u;
    const size_t lbase = size_t{env} * m.links_per_env;
    constexpr int kOwn = G > kWave ? 2 : 1, kLanes = G / kOwn;
    for (uint32_t e = lane; e < nl * 6u; e += kLanes) v[e] = d.link_velocity[lbase * 6u + e];
    wave_sync();
    // the joint transform and the joint's own twist do not wait on the tree: a lane prepares its links' before the sweep
    struct Jointed { uint32_t depth, parent; bool state; float X[36], own[6]; };
    auto prepare = [&](uint32_t l, Jointed& t) {
        const uint8_t type = m.joint_type[l];
        t.depth = m.link_tree_depth[l]; t.parent = m.parent_link[l];
        t.state = t.parent == kInvalid && type == kFloatingBase;   // a floating root's twist is state
        if (t.state) return;
        float s[6];
        joint_transform(m, l, d.q[lbase + l], t.X);
        motion_subspace(type, load3(m.joint_axis + 3u * l), s);
        const float qdl = d.qdot[lbase + l];
#pragma unroll
        for (int c = 0; c < 6; ++c) t.own[c] = s[c] * qdl;
    };
    auto propagate = [&](uint32_t l, const Jointed& t) {
        if (t.state) return;
        float pv[6] = {0, 0, 0, 0, 0, 0}, vl[6];
        if (t.parent != kInvalid) {
#pragma unroll
            for (int i = 0; i < 6; ++i) pv[i] = v[6u * t.parent + i];
        }
        mat66_vec(t.X, pv, vl);
#pragma unroll
        for (int c = 0; c < 6; ++c) v[6u * l + c] = vl[c] + t.own[c];
    };
    Jointed own[kOwn];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
        own[i].depth = kInvalid; own[i].parent = kInvalid; own[i].state = true;
        if (lane + uint32_t(i * kLanes) < nl) prepare(lane + uint32_t(i * kLanes), own[i]);
    }
    for (uint32_t depth = 0u; depth <= m.max_depth; ++depth) {
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
            if (own[i].depth == depth) propagate(lane + uint32_t(i * kLanes), own[i]);
        if (G > kWave)
            for (uint32_t l = lane + 2u * kWave; l < nl; l += kWave) {
                Jointed t;
                prepare(l, t);
                if (t.depth == depth) propagate(l, t);
            }
        wave_sync();
    }
    for (uint32_t e = lane; e < nl * 6u; e += kLanes) d.link_velocity[lbase * 6u + e] = v[e];
}
template <int G>
__global__ void __launch_bounds__(kWave) FkLinkVelocitiesKernel(ModelView m, DataView d, uint32_t env_count) {
    extern __shared__ float lds[];
    constexpr uint32_t kLanes = G < kWave ? G : kWave;
    const uint32_t group = threadIdx.x / kLanes, env = blockIdx.x * (kWave / kLanes) + group;
    link_velocities_of_env<G>(m, d, env, threadIdx.x % kLanes, env < env_count, lds + group * m.links_per_env * 6u);
}

// What follows the solve in a step - positions integrated, world poses, link twists, the bodies' poses - as one kernel,
// `G` lanes of two wavefronts an environment: four kernels that each take about the time of a launch become one, running
// the same device code in the same order (IntegratePosition, FkWorldPoses, FkLinkVelocities, SyncLinkBodyPose).  A plan
// takes this route when its op list holds the four in a row (backend.hip); an op dispatched by itself runs its own kernel.
// (The whole step of a serial chain may be other code, with other last places: ops_chain_kernel.h.)
struct StepTail { IntegratePositionParams integrate; uint32_t runs, sync_bodies; };
template <int G>
__device__ __forceinline__ void step_tail_of_block(const ModelView& m, const DataView& d, const StepTail& t, uint32_t env_count, float* lds) {
    constexpr uint32_t kLanes = G < kWave ? G : kWave, kEnvs = kWave / kLanes;
    const uint32_t lane = threadIdx.x % kLanes, group = threadIdx.x % kWave / kLanes, env = blockIdx.x * kEnvs + group, nl = m.links_per_env;
    const uint32_t wave = threadIdx.x / kWave;   // world poses and link twists do not depend on each other: a wavefront each
    const bool there = env < env_count;
    if (wave == 0u && there) for (uint32_t l = lane; l < nl; l += kLanes) integrate_position_of_link(m, d, t.integrate, env, l);
    __syncthreads();   // the new coordinates, base pose and root twist are in memory for both wavefronts
    if (wave == 1u) link_velocities_of_env<G>(m, d, env, lane, there, lds + kEnvs * nl * 7u + group * nl * 6u);
    if (wave != 0u) return;
    float* pose = lds + group * nl * 7u;
    world_poses_of_env<G>(m, d, env, lane, there, pose);
    if (t.sync_bodies == 0u || !there) return;
    wave_sync();
    for (uint32_t b = lane; b < m.bodies_per_env; b += kLanes) sync_body_pose(m, d, env, b, pose);
}
template <int G>
__global__ void __launch_bounds__(2 * kWave) StepTailKernel(ModelView m, DataView d, StepTail t, uint32_t env_count) {
    extern __shared__ float lds[];
    step_tail_of_block<G>(m, d, t, env_count, lds);
}
// Where nothing stands between the dynamics and the step's tail, as in a world without rows, the workgroup goes on with its own
// environments: their state is its own.
// (Two waves a SIMD at the least, of the five or so that registers allow: a kernel that may have the whole register file gets its matrix
// products in the half of it that other instructions cannot name, and reads each of them back - 630 of 9500 at 36 coordinates.  65536
// humanoids 1064 -> 1030 us, 4096 95.1 -> 91.7, 8192 ropes 962 -> 919, 4096 quadrupeds 38.8 -> 38.3.)
template <int N, int G>
__global__ void __launch_bounds__(3 * kWave) __attribute__((amdgpu_waves_per_eu(2))) ArticulationDynamicsKernel(ModelView m, DataView d, ArticulationDynamicsParams p, uint32_t env_count, StepTail t) {
    extern __shared__ float lds[];
    dynamics_of_block<N, G>(m, d, p, env_count, lds);
    if (t.runs == 0u) return;
    __syncthreads();
    step_tail_of_block<G>(m, d, t, env_count, lds);
}

#include "ops_chain_kernel.h"

// The instantiation for `lanes` lanes an environment and the number of its workgroups
#define NKH_LAUNCH_LANES(lanes, kernel, envs, threads, lds_words_an_env, stream, ...)                                                          \
    do {                                                                                                                                       \
        const uint32_t envs_a_block = (lanes) < 64u ? 64u / (lanes) : 1u, blocks = ((envs) + envs_a_block - 1u) / envs_a_block;                                      \
        const size_t lds_bytes = size_t{envs_a_block} * (lds_words_an_env) * sizeof(float);                                                     \
        if ((lanes) == 8u) hipLaunchKernelGGL(kernel<8>, dim3(blocks), dim3(threads), lds_bytes, stream, __VA_ARGS__);                          \
        else if ((lanes) == 16u) hipLaunchKernelGGL(kernel<16>, dim3(blocks), dim3(threads), lds_bytes, stream, __VA_ARGS__);                   \
        else if ((lanes) == 32u) hipLaunchKernelGGL(kernel<32>, dim3(blocks), dim3(threads), lds_bytes, stream, __VA_ARGS__);                   \
        else if ((lanes) == 64u) hipLaunchKernelGGL(kernel<64>, dim3(blocks), dim3(threads), lds_bytes, stream, __VA_ARGS__);                   \
        else hipLaunchKernelGGL(kernel<128>, dim3(blocks), dim3(threads), lds_bytes, stream, __VA_ARGS__);                                       \
    } while (false)

}  // namespace

// ---- op entry points ------------------------------------------------------------------------------------
Status OpFkWorldPoses(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const FkWorldPosesParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (p->articulation_count == 0u || p->total_link_count == 0u) return Status::Ok;
    if (m.links_per_env == 0u || p->total_link_count != p->articulation_count * m.links_per_env) return Status::InvalidArgument;
    const uint32_t lanes = LanesAnEnvironment(m.links_per_env, p->articulation_count);
    NKH_LAUNCH_LANES(lanes, FkWorldPosesKernel, p->articulation_count, kWave, m.links_per_env * 7u, stream, m, d, p->articulation_count);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

// false when any of the four would not run its kernel as dispatched
static bool StepTailOf(const ModelView& m, const IntegratePositionParams* integrate, const FkWorldPosesParams* poses, const FkLinkVelocitiesParams* twists,
                       const SyncLinkBodyPoseParams* bodies, StepTail* tail) {
    if (integrate == nullptr || poses == nullptr || twists == nullptr) return false;
    const uint32_t E = poses->articulation_count, links = E * m.links_per_env;
    if (E == 0u || m.links_per_env == 0u || integrate->dt <= 0.0f || integrate->total_link_count != links ||
        poses->total_link_count != links || poses->selected_env_count != 0u || twists->articulation_count != E ||
        twists->total_link_count != links) return false;
    if (bodies != nullptr && (bodies->env_count != E || bodies->bodies_per_env != m.bodies_per_env || bodies->bodies_per_env == 0u ||
                              bodies->selected_env_count != 0u)) return false;
    *tail = StepTail{*integrate, 1u, bodies != nullptr ? 1u : 0u};
    return true;
}
// The four ops after the solve as one launch; Unsupported when any of them would not run its kernel as dispatched
// (the caller then dispatches them one by one).
Status OpStepTail(const ModelView& m, const DataView& d, const IntegratePositionParams* integrate, const FkWorldPosesParams* poses,
                  const FkLinkVelocitiesParams* twists, const SyncLinkBodyPoseParams* bodies, hipStream_t stream) {
    StepTail tail;
    if (!StepTailOf(m, integrate, poses, twists, bodies, &tail)) return Status::Unsupported;
    const uint32_t E = poses->articulation_count, lanes = LanesAnEnvironment(m.links_per_env, E);
    NKH_LAUNCH_LANES(lanes, StepTailKernel, E, 2 * kWave, m.links_per_env * 13u, stream, m, d, tail, E);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

using DynamicsKernel = void (*)(ModelView, DataView, ArticulationDynamicsParams, uint32_t, StepTail);
struct DynamicsEntry { uint32_t width, lanes; DynamicsKernel kernel; };
// by lanes an environment, then by width: the first that holds an environment's links and coordinates is the one
#define NKH_DYNAMICS(N, G) {N##u, G##u, ArticulationDynamicsKernel<N, G>}
static const DynamicsEntry kDynamicsKernels[] = {
    NKH_DYNAMICS(8, 8), NKH_DYNAMICS(16, 8),
    NKH_DYNAMICS(12, 16), NKH_DYNAMICS(16, 16), NKH_DYNAMICS(20, 16), NKH_DYNAMICS(24, 16),
    NKH_DYNAMICS(4, 64), NKH_DYNAMICS(8, 64), NKH_DYNAMICS(12, 64), NKH_DYNAMICS(16, 64), NKH_DYNAMICS(20, 64), NKH_DYNAMICS(24, 64),
    NKH_DYNAMICS(28, 64), NKH_DYNAMICS(32, 64), NKH_DYNAMICS(36, 64), NKH_DYNAMICS(40, 64), NKH_DYNAMICS(44, 64), NKH_DYNAMICS(48, 64),
    NKH_DYNAMICS(52, 64), NKH_DYNAMICS(56, 64), NKH_DYNAMICS(60, 64), NKH_DYNAMICS(64, 64)};
#undef NKH_DYNAMICS
// Lanes an environment: all 64 while the environments are few, when the one chain an environment has is what counts and fewer
// lanes lengthen its sweeps; past that as few as hold its links and coordinates.  A step of 1000 arms (8 links, 7 coordinates)
// takes 35.9 us with 64 lanes and 37.0 with 8, 1300 40.9 and 36.9, 2500 54.0 and 40.6; 1000 quadrupeds (13 links, 18
// coordinates) 364 us with 64 and 373 with 16, 2500 399 and 400, 3000 400 and 391, 2000 walkers 261 and 256.  Thirty-two lanes
// gain nothing: two environments of 31 links and 36 coordinates ask for the LDS that two workgroups with 64 lanes each do
// (65536 humanoids 8435 and 8490 us).
constexpr uint32_t kEightLanesFrom = 1152u, kSixteenLanesFrom = 2560u;   // environments
static uint32_t DynamicsLanes(uint32_t links, uint32_t dof, uint32_t envs) {
    if (links <= 8u && dof <= 16u) return envs < kEightLanesFrom ? 64u : 8u;
    return links <= 16u && dof <= 24u && envs >= kSixteenLanesFrom ? 16u : 64u;
}

// LDS of a workgroup of `entry`, with a third wavefront's poses where it `places`
static size_t DynamicsBytes(const ModelView& m, const DynamicsEntry& entry, bool places) {
    const uint32_t envs = kWave / entry.lanes;
    return size_t{DynamicsTreeWords(m.links_per_env, m.sweep_passes) + envs * DynamicsEnvWords(m.links_per_env, m.dof, envs) +
                  (places ? envs * m.links_per_env * 7u + 1u : 0u)} * sizeof(float);
}
// nullptr where the op refuses the world or the parameters
static const DynamicsEntry* DynamicsEntryOf(const ModelView& m, const ArticulationDynamicsParams& p) {
    if (m.dof > kMaxDof || m.dof == 0u || p.max_dof != m.max_dof || p.total_link_count != p.articulation_count * m.links_per_env) return nullptr;
    // the links a world may have: those whose working state, with its transforms in full, fits a compute unit's LDS
    if (size_t{m.links_per_env * 109u + m.dof * (m.dof + 3u) + 64u + m.sweep_passes * kSweepLinks} * sizeof(float) > 160u * 1024u) return nullptr;
    const uint32_t lanes = DynamicsLanes(m.links_per_env, m.dof, p.articulation_count);
    const DynamicsEntry* entry = kDynamicsKernels;
    while (entry->lanes < lanes || entry->width < m.dof) ++entry;
    return entry;
}
static Status LaunchDynamics(const ModelView& m, const DataView& d, const ArticulationDynamicsParams& p, const DynamicsEntry& entry, bool places, const StepTail& tail,
                             hipStream_t stream) {
    const uint32_t envs = kWave / entry.lanes;
    hipLaunchKernelGGL(entry.kernel, dim3((p.articulation_count + envs - 1u) / envs), dim3((places ? 3 : 2) * kWave), DynamicsBytes(m, entry, places), stream, m, d, p,
                       p.articulation_count, tail);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}
Status OpArticulationDynamics(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const ArticulationDynamicsParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (p->articulation_count == 0u || p->total_link_count == 0u) return Status::Ok;
    const DynamicsEntry* entry = DynamicsEntryOf(m, *p);
    return entry == nullptr ? Status::InvalidArgument : LaunchDynamics(m, d, *p, *entry, false, StepTail{}, stream);
}

// The poses in the dynamics' launch: a launch and its gap less, and the sweep of the poses beside the dynamics' longer ones.
// Always where environments share a wavefront (a step of 3500 arms 49 -> 45 us, 65536 229 -> 223; 4096 walkers 343 -> 339, 16384
// quadrupeds 1240 -> 1243).  An environment a wavefront (64 arms 37.3 -> 32.8 us), up to six workgroups a compute unit:
// past that the third wavefront, which has a lane a link and waits on every depth, takes the others' turns (64 humanoids 517
// -> 511 us, 1024 641 -> 637, 1500 621 -> 616, 1800 639 -> 645, 3000 714 -> 723, 65536 7818 -> 8180; 1800 quadrupeds 410 ->
// 408, 2900 435 -> 440).  Not the 65 links of a rope, two a lane (256 of them 2321 -> 2288 us, 1000 2535 -> 2577).
constexpr uint32_t kPlacedBeside = 1536u;
bool PosesAndDynamicsServed(const ModelView& m, const FkWorldPosesParams* poses, const ArticulationDynamicsParams* dynamics) {
    if (poses == nullptr || dynamics == nullptr || dynamics->articulation_count == 0u || m.links_per_env == 0u) return false;
    if (poses->articulation_count != dynamics->articulation_count || poses->total_link_count != dynamics->total_link_count) return false;
    const DynamicsEntry* entry = DynamicsEntryOf(m, *dynamics);
    if (entry == nullptr || DynamicsBytes(m, *entry, true) > 160u * 1024u) return false;
    return m.links_per_env <= entry->lanes && (entry->lanes < uint32_t(kWave) || dynamics->articulation_count <= kPlacedBeside);
}
Status OpPosesAndDynamics(const ModelView& m, const DataView& d, const ArticulationDynamicsParams* dynamics, hipStream_t stream) {
    const DynamicsEntry* entry = DynamicsEntryOf(m, *dynamics);
    return entry == nullptr ? Status::InvalidArgument : LaunchDynamics(m, d, *dynamics, *entry, true, StepTail{}, stream);
}
// Serial chains go a lane an environment (ChainStepKernel), where the host says that the links are one (a chain's depths alone
// do not say that link l hangs from link l - 1)
static bool ChainServed(const ModelView& m, const ArticulationDynamicsParams& dynamics) {
    return m.serial_chain != 0u && m.links_per_env <= kChainLinks && m.max_dof <= kChainLinks && dynamics.articulation_count >= ChainFrom(m.links_per_env);
}
// The step's tail in the dynamics' launch, up to five workgroups a compute unit: past that the shorter kernels fill the chip
// better than one whose workgroups hold the dynamics' LDS to the end (a step of 64 arms 32.8 -> 30.6 us, 1000 37.8 -> 35.4, 8000
// in 1000 workgroups 51.0 -> 46.7, 12000 67.2 -> 67.5, 20011 86 -> 88, 65536 223 -> 234).
constexpr uint32_t kTailWorkgroups = 1280u;
bool StepServed(const ModelView& m, const ArticulationDynamicsParams& dynamics, const IntegratePositionParams* integrate, const FkWorldPosesParams* poses,
                const FkLinkVelocitiesParams* twists, const SyncLinkBodyPoseParams* bodies) {
    StepTail tail;
    const DynamicsEntry* entry = DynamicsEntryOf(m, dynamics);
    if (entry == nullptr || !StepTailOf(m, integrate, poses, twists, bodies, &tail) || poses->articulation_count != dynamics.articulation_count) return false;
    if (ChainServed(m, dynamics)) return true;
    return uint64_t{dynamics.articulation_count} * entry->lanes <= uint64_t{kTailWorkgroups} * kWave;
}
Status OpStep(const ModelView& m, const DataView& d, const ArticulationDynamicsParams* dynamics, const IntegratePositionParams* integrate,
              const FkWorldPosesParams* poses, const FkLinkVelocitiesParams* twists, const SyncLinkBodyPoseParams* bodies, hipStream_t stream) {
    const DynamicsEntry* entry = DynamicsEntryOf(m, *dynamics);
    StepTail tail;
    if (entry == nullptr || !StepTailOf(m, integrate, poses, twists, bodies, &tail)) return Status::InvalidArgument;
    if (ChainServed(m, *dynamics)) {
        hipLaunchKernelGGL(ChainStepKernel, dim3((dynamics->articulation_count + kWave - 1u) / kWave), dim3(kChainWaves * kWave), ChainLdsWords(m.links_per_env, m.max_dof) * sizeof(float), stream, m, d,
                           *dynamics, dynamics->articulation_count, tail);
        return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
    }
    return LaunchDynamics(m, d, *dynamics, *entry, true, tail, stream);
}

namespace {
// SolveMassBlock (articulation_mass.cuh:357-396) by one thread: forward by columns, divide, backward
__device__ void solve_mass_serial(const float* factor, float* value, uint32_t n, uint32_t stride) {
    for (uint32_t j = 0u; j < n; ++j) {
        const float solved = value[j];
        for (uint32_t i = j + 1u; i < n; ++i) value[i] -= factor[size_t{i} * stride + j] * solved;
    }
    for (uint32_t i = 0u; i < n; ++i) value[i] = value[i] / factor[size_t{i} * stride + i];
    for (uint32_t end = n; end > 0u; --end) {
        const uint32_t i = end - 1u;
        float sum = value[i];
        for (uint32_t j = i + 1u; j < n; ++j) sum -= factor[size_t{j} * stride + i] * value[j];
        value[i] = sum;
    }
}

// AccumulateChainJointForce (articulation_types.cuh:193-238): what a force f and a moment at `point` add to the
// generalized force of the joint of `link`
__device__ void accumulate_chain(const ModelView& m, const DataView& d, uint32_t env, uint32_t link, V3 point, V3 f, V3 moment, float* out) {
    const uint32_t dof_index = m.link_dof[link], stride = m.max_dof;
    const uint8_t type = m.joint_type[link];
    if (type == kFloatingBase) {
        const Xf base = load_xf(d.base_pose + size_t{env} * 7u);
        const V3 lever = sub3(point, base.p);
        const V3 e[3] = {rotate_normalized(base.r, V3{1, 0, 0}), rotate_normalized(base.r, V3{0, 1, 0}), rotate_normalized(base.r, V3{0, 0, 1})};
        for (uint32_t b = 0u; b < 3u; ++b) {
            const float angular = dot3(cross3(e[b], lever), f) + dot3(e[b], moment), linear = dot3(e[b], f);
            if (dof_index + b < stride) out[dof_index + b] += angular;
            if (dof_index + 3u + b < stride) out[dof_index + 3u + b] += linear;
        }
        return;
    }
    const Xf pose = load_xf(d.link_pose + (size_t{env} * m.links_per_env + link) * 7u);
    const V3 axis_world = rotate_normalized(pose.r, load3(m.joint_axis + 3u * link));
    float entry;
    if (type == kPrismatic) entry = dot3(axis_world, f);
    else entry = dot3(cross3(axis_world, sub3(point, pose.p)), f) + dot3(axis_world, moment);
    if (dof_index < stride) out[dof_index] += entry;
}

// ArticulationReferenceWeightsKernel (articulation.cu:434-501), one thread an environment as in the reference: the
// diagonal of M^-1 (a floating base's six entries averaged over its rotations and its translations), and for every
// link the mean response of its centre of mass to a unit force and to a unit moment along the three world axes.
// `m_factor` holds the factor of the mass matrix at the current pose (no drive damping folded in).
__global__ void __launch_bounds__(kWave) ReferenceWeightsKernel(ModelView m, DataView d, uint32_t env_count) {
    const uint32_t env = blockIdx.x * kWave + threadIdx.x;
    if (env >= env_count) return;
    const uint32_t nl = m.links_per_env, nb = m.bodies_per_env, md = m.max_dof, dof = m.dof;
    float* weights = d.body_invweight0 + size_t{env} * nb * 2u;
    for (uint32_t b = 0u; b < nb; ++b) weights[2u * b] = weights[2u * b + 1u] = 0.0f;   // static rows move under nothing
    const float* factor = d.m_factor + size_t{env} * md * md;
    float* diagonal = d.dof_invweight0 + size_t{env} * md;
    float row[kMaxDof], solution[kMaxDof];
    for (uint32_t k = 0u; k < dof; ++k) {
        for (uint32_t i = 0u; i < dof; ++i) solution[i] = i == k ? 1.0f : 0.0f;
        solve_mass_serial(factor, solution, dof, md);
        diagonal[k] = solution[k];
    }
    if (m.joint_type[0] == kFloatingBase) {
        const float rotation = (diagonal[0] + diagonal[1] + diagonal[2]) / 3.0f;
        const float translation = (diagonal[3] + diagonal[4] + diagonal[5]) / 3.0f;
        for (uint32_t i = 0u; i < 3u; ++i) { diagonal[i] = rotation; diagonal[i + 3u] = translation; }
    }
    for (uint32_t link = 0u; link < nl; ++link) {
        const Xf pose = load_xf(d.link_pose + (size_t{env} * nl + link) * 7u);
        const V3 point = add3(pose.p, rotate_normalized(pose.r, load3(m.link_inertial_frame + 7u * link)));
        float weight[2] = {0.0f, 0.0f};
        for (uint32_t axis = 0u; axis < 6u; ++axis) {
            for (uint32_t k = 0u; k < dof; ++k) row[k] = 0.0f;
            const V3 unit{axis % 3u == 0u ? 1.0f : 0.0f, axis % 3u == 1u ? 1.0f : 0.0f, axis % 3u == 2u ? 1.0f : 0.0f};
            const V3 none{0.0f, 0.0f, 0.0f};
            for (uint32_t walk = link; walk != kInvalid; walk = m.parent_link[walk])
                if (joint_dof(m.joint_type[walk]) != 0u) accumulate_chain(m, d, env, walk, point, axis < 3u ? unit : none, axis < 3u ? none : unit, row);
            for (uint32_t k = 0u; k < dof; ++k) solution[k] = row[k];
            solve_mass_serial(factor, solution, dof, md);
            for (uint32_t k = 0u; k < dof; ++k) weight[axis / 3u] += row[k] * solution[k];
        }
        const uint32_t body = m.link_body[link];
        if (body < nb) { weights[2u * body] = weight[0] / 3.0f; weights[2u * body + 1u] = weight[1] / 3.0f; }
    }
}
}  // namespace

// ReferenceWeights (op_schema.hpp:123-130; articulation.cu:425-500): the mass matrix at the current poses without
// drive damping, its factor, and the reference weights from it.  World creation and reset dispatch it after the poses
// are refreshed (nk/pipeline/world.cpp:553-561).
// BodyReferenceWeightsKernel (articulation.cu:425-432): a free body's weights are its inverse mass and the mean of its
// inverse principal moments; rows without mass weigh nothing
__global__ void __launch_bounds__(256) BodyReferenceWeightsKernel(DataView d, uint32_t count) {
    const uint32_t body = blockIdx.x * 256u + threadIdx.x;
    if (body >= count) return;
    const float* inverse = d.body_inv_inertia + size_t{body} * 3u;
    d.body_invweight0[2u * body] = d.body_inv_mass[body];
    d.body_invweight0[2u * body + 1u] = (inverse[0] + inverse[1] + inverse[2]) / 3.0f;
}

Status OpReferenceWeights(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const ReferenceWeightsParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (m.free_body != 0u) {
        if (p->total_body_count == 0u) return Status::Ok;
        hipLaunchKernelGGL(BodyReferenceWeightsKernel, dim3((p->total_body_count + 255u) / 256u), dim3(256), 0, stream, d, p->total_body_count);
        return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
    }
    if (p->articulation_count == 0u || p->total_link_count == 0u) return Status::Ok;
    if (p->articulations_per_env != 1u || p->max_dof != m.max_dof || p->bodies_per_env != m.bodies_per_env ||
        p->total_link_count != p->articulation_count * m.links_per_env) return Status::InvalidArgument;
    ArticulationDynamicsParams mass{};   // no velocity update, no wrench, nothing folded into the diagonal
    mass.max_dof = p->max_dof; mass.integrate_velocity = 0u; mass.articulation_count = p->articulation_count;
    mass.total_link_count = p->total_link_count; mass.max_links = m.links_per_env; mass.links_per_env = m.links_per_env;
    mass.bodies_per_env = m.bodies_per_env;
    if (m.dof != 0u) {
        const Status status = OpArticulationDynamics(m, d, &mass, stream);
        if (status != Status::Ok) return status;
    }
    hipLaunchKernelGGL(ReferenceWeightsKernel, dim3((p->articulation_count + kWave - 1u) / kWave), dim3(kWave), 0, stream, m, d,
                       p->articulation_count);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

namespace {
// ActuatorVelocityDerivative (articulation.cu:942-948): what a servo's effort changes per unit joint velocity, none
// while its own force limit clamps it
__device__ float actuator_velocity_derivative(const DataView& d, uint32_t mode, size_t link) {
    if (d.drive_force_limit[link] > 0.0f && fabsf(d.drive_command[link] - d.joint_gravity_force[link]) > d.drive_force_limit[link]) return 0.0f;
    return mode == kDrivePdPosition ? d.drive_damping[link] : mode == kDriveVelocity ? d.drive_stiffness[link] : 0.0f;
}

// ArticulationDampingKernel (articulation.cu:950-1000), one wavefront an environment: contacts were solved with the plain
// mass; the step's velocity change now goes through (M + dt D)^-1 M, D the joint damping and, for the implicit
// integrators, the unclamped servo velocity gains.  M + dt D is factored as L D L^T, lane = row in registers as the forward
// dynamics does it, every entry taking its pivots' updates in pivot order (FactorMass, articulation_mass.cuh:269-335);
// the solve runs forward by columns, divides, and substitutes back with each coordinate's products in ascending order
// (SolveMassBlock :357-396), a product a lane.  A chain of one wavefront: in LDS, with a barrier a column and the last
// substitution on one lane, 4096 robots of twelve coordinates took 22.9 us, 9.4 as it is.
template <int N>
__global__ void __launch_bounds__(kWave) ArticulationDampingKernel(ModelView m, DataView d, ArticulationDampingParams p) {
    const uint32_t env = blockIdx.x, lane = threadIdx.x, n = m.dof, stride = m.max_dof, nl = m.links_per_env;
    const size_t lbase = size_t{env} * nl, base = size_t{env} * stride;
    const bool coordinate = lane < n;
    float row[N];
    {
        const float* own = d.m + (base + (coordinate ? lane : 0u)) * stride;
#pragma unroll
        for (int k = 0; k < N; ++k) row[k] = own[uint32_t(k) < n ? uint32_t(k) : 0u];
    }
    uint32_t link = 0u, component = kInvalid;
    float value = 0.0f, velocity = 0.0f, damping = 0.0f, change = 0.0f;
    if (coordinate) {
        link = m.dof_link[lane]; component = m.dof_component[lane];
        const bool scalar = component == kInvalid;
        value = scalar ? m.joint_damping[link] : 0.0f;
        if (scalar && p.actuator_derivative != 0u) value += actuator_velocity_derivative(d, p.mode, lbase + link);
        velocity = scalar ? d.qdot[lbase + link] : d.link_velocity[(lbase + link) * 6u + component];
        damping = p.dt * value;
        change = damping * (velocity - d.step_qdot_flat[base + lane]);
    }
    if (!__any(coordinate && value != 0.0f)) return;
    const uint32_t ll = local_lane(lane);
#pragma unroll
    for (int k = 0; k < N; ++k) {   // rows and columns n..N-1 are those of the identity
        const float entry = row[k] + (ll == uint32_t(k) ? damping : 0.0f);
        row[k] = coordinate && uint32_t(k) < n ? entry : (ll == uint32_t(k) ? 1.0f : 0.0f);
    }
    ldlt_pivots<64, 0>(ll, row);
    forward_rows<64, 0>(ll, n, row, &change);
    float pivot = 1.0f;
#pragma unroll
    for (int k = 0; k < N; ++k) pivot = ll == uint32_t(k) ? row[k] : pivot;
    change = coordinate ? change / pivot : 0.0f;
#pragma unroll
    for (int i = N - 2; i >= 0; --i) {
        const float product = row[i] * change;
        float sum = lane_value(change, i);
#pragma unroll
        for (int j = i + 1; j < N; ++j) sum -= lane_value(product, j);
        change = ll == uint32_t(i) ? sum : change;
    }
    if (!coordinate) return;
    velocity -= change;
    if (component == kInvalid) d.qdot[lbase + link] = velocity; else d.link_velocity[(lbase + link) * 6u + component] = velocity;
    d.qdot_flat[base + lane] = velocity;
    if (component == kInvalid && p.actuator_derivative != 0u && p.readout_drives != 0u) {
        const float derivative = actuator_velocity_derivative(d, p.mode, lbase + link);
        const float correction = derivative * (velocity - d.step_qdot_flat[base + lane]);
        d.actuator_effort_requested[lbase + link] -= correction;
        d.actuator_effort[lbase + link] -= correction;
        d.tau[lbase + link] -= correction;
    }
}
}  // namespace

// ArticulationDamping (op_schema.hpp:132-141): the op a MuJoCo integrator adds after the constraint solve.
Status OpArticulationDamping(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const ArticulationDampingParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (p->articulation_count == 0u || p->total_link_count == 0u || m.dof == 0u) return Status::Ok;
    if (m.dof > kMaxDof || p->max_dof != m.max_dof || p->total_link_count != p->articulation_count * m.links_per_env) return Status::InvalidArgument;
    using DampingKernel = void (*)(ModelView, DataView, ArticulationDampingParams);
    static const DampingKernel kKernels[16] = {
        ArticulationDampingKernel<4>, ArticulationDampingKernel<8>, ArticulationDampingKernel<12>, ArticulationDampingKernel<16>,
        ArticulationDampingKernel<20>, ArticulationDampingKernel<24>, ArticulationDampingKernel<28>, ArticulationDampingKernel<32>,
        ArticulationDampingKernel<36>, ArticulationDampingKernel<40>, ArticulationDampingKernel<44>, ArticulationDampingKernel<48>,
        ArticulationDampingKernel<52>, ArticulationDampingKernel<56>, ArticulationDampingKernel<60>, ArticulationDampingKernel<64>};
    hipLaunchKernelGGL(kKernels[(m.dof + 3u) / 4u - 1u], dim3(p->articulation_count), dim3(kWave), 0, stream, m, d, *p);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

Status OpIntegratePosition(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const IntegratePositionParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (p->dt <= 0.0f || p->total_link_count == 0u) return Status::Ok;
    if (m.free_body != 0u) return BodyIntegratePosition(m, d, *p, stream);
    const uint32_t blocks = (p->total_link_count + 255u) / 256u;
    hipLaunchKernelGGL(IntegratePositionKernel, dim3(blocks), dim3(256), 0, stream, m, d, *p);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

Status OpFkLinkVelocities(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const FkLinkVelocitiesParams*>(params);
    if (p == nullptr) return Status::InvalidArgument;
    if (p->articulation_count == 0u || p->total_link_count == 0u) return Status::Ok;
    const uint32_t lanes = LanesAnEnvironment(m.links_per_env, p->articulation_count);
    NKH_LAUNCH_LANES(lanes, FkLinkVelocitiesKernel, p->articulation_count, kWave, m.links_per_env * 6u, stream, m, d, p->articulation_count);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}

void InitArticulationKernels() {
    for (const DynamicsEntry& entry : kDynamicsKernels) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(entry.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
    }
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(ChainStepKernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(ChainLdsWords(kChainLinks, kChainLinks) * sizeof(float)));
    (void)hipGetLastError();
}

// ApplyAffineDriveKernel (articulation.cu:836-940): one thread per link turns the controller fields into an affine
// effort `command - dissipation * qdot` and its bounds for the drive row, and overwrites tau with the feedforward
// load.  Gravity compensation (ProjectGravityCompensationKernel :393-423) is not authored on this path:
// joint_gravity_force stays as uploaded.  The inverse-dynamics modes (ComputedTorque, Osc) are not built.
__global__ void __launch_bounds__(256) ApplyAffineDriveKernel(ModelView m, DataView d, ApplyDrivesParams p) {
    const uint32_t link = blockIdx.x * blockDim.x + threadIdx.x;
    if (link >= p.total_link_count) return;
    d.drive_command[link] = d.drive_dissipation[link] = 0.0f;
    d.drive_lower[link] = d.drive_upper[link] = 0.0f;
    d.tau[link] = 0.0f;
    const uint32_t local = link % p.links_per_env;
    if (joint_dof(m.joint_type[local]) != 1u) return;
    const uint32_t mode = p.mode;
    const bool implicit = p.defer_velocity_damping != 0u;
    const bool position_control = mode == kDrivePdPosition, velocity_control = mode == kDriveVelocity;
    const float kp = d.drive_stiffness[link], kd = d.drive_damping[link];
    if ((position_control && (!isfinite(d.drive_target[link]) || !isfinite(kp) || kp < 0.0f || !isfinite(kd) || (implicit && kd < 0.0f))) ||
        ((position_control || velocity_control) && !isfinite(d.velocity_target[link])) ||
        (velocity_control && (!isfinite(kp) || kp < 0.0f)) ||
        (mode == kDriveActuator && !isfinite(d.actuator_noload_speed[link]))) {
        atomicOr(d.env_status + link / p.links_per_env, kEnvStatusControlFailure);
        return;
    }
    const float velocity = d.qdot[link];
    const float limit = d.drive_force_limit[link];
    float lower = limit > 0.0f ? -limit : -FLT_MAX;
    float upper = limit > 0.0f ? limit : FLT_MAX;
    float bias = 0.0f, damping = 0.0f;
    if (mode == kDrivePdPosition) {
        // an implicit spring is evaluated at the end of the step, adding dt kp to the damping
        damping = kd + (implicit ? p.dt * kp : 0.0f);
        bias = kp * (d.drive_target[link] - d.q[link]) + damping * d.velocity_target[link];
    } else if (mode == kDriveVelocity) {
        damping = kp;
        bias = damping * d.velocity_target[link];
    } else {   // torque, actuator
        bias = d.drive_target[link];
        if (mode == kDriveActuator && limit > 0.0f && d.actuator_noload_speed[link] > 0.0f) {
            const float speed_bias = limit * velocity / d.actuator_noload_speed[link];
            lower = fminf(fmaxf(-limit - speed_bias, -limit), limit);
            upper = fminf(fmaxf(limit - speed_bias, -limit), limit);
        }
    }
    const float effort = bias - damping * velocity;
    const float gravity_force = d.joint_gravity_force[link];
    const bool saturated = effort < lower || effort > upper;
    const float joint_limit = d.drive_joint_force_limit[link];
    if (implicit && joint_limit > 0.0f) {
        bias = fminf(fmaxf(fminf(fmaxf(effort, lower), upper) + gravity_force, -joint_limit), joint_limit);
        damping = saturated ? 0.0f : damping;
        bias += damping * velocity;
        lower = -FLT_MAX;
        upper = FLT_MAX;
    } else if (!implicit || saturated) {
        bias = effort + gravity_force;
        damping = 0.0f;
        lower += gravity_force;
        upper += gravity_force;
        if (joint_limit > 0.0f) {
            lower = fminf(fmaxf(lower, -joint_limit), joint_limit);
            upper = fminf(fmaxf(upper, -joint_limit), joint_limit);
        }
    } else {   // the row clamps the command bias = effort + damping * velocity
        bias += gravity_force;
        lower += gravity_force + damping * velocity;
        upper += gravity_force + damping * velocity;
    }
    const float feedforward = d.joint_f[link];
    if (!isfinite(bias) || !isfinite(damping) || damping < 0.0f || !isfinite(limit) || !isfinite(feedforward) || !isfinite(velocity) ||
        !isfinite(d.q[link])) {
        atomicOr(d.env_status + link / p.links_per_env, kEnvStatusControlFailure);
        return;
    }
    d.drive_command[link] = bias;
    d.drive_dissipation[link] = damping;
    d.drive_lower[link] = lower;
    d.drive_upper[link] = upper;
    d.tau[link] = feedforward;
}

// ReadoutDrivesKernel (articulation.cu:999-1016)
__global__ void __launch_bounds__(256) ReadoutDrivesKernel(ModelView m, DataView d, ReadoutDrivesParams p) {
    const uint32_t link = blockIdx.x * blockDim.x + threadIdx.x;
    if (link >= p.total_link_count) return;
    d.actuator_effort_requested[link] = d.actuator_effort[link] = d.actuator_saturated[link] = 0.0f;
    const uint32_t env = link / p.links_per_env, local = link - env * p.links_per_env;
    if (joint_dof(m.joint_type[local]) != 1u) return;
    const size_t row = size_t{env} * p.rows_per_env + p.first_drive_row + local;
    const float effort = d.drive_command[link] - d.drive_dissipation[link] * d.qdot[link];
    d.actuator_effort_requested[link] = effort;
    const float applied = d.lambda[row] / p.dt - d.drive_dissipation[link] * d.qdot[link];
    d.actuator_effort[link] = applied;
    d.actuator_saturated[link] = d.drive_command[link] < d.drive_lower[link] || d.drive_command[link] > d.drive_upper[link] ? 1.0f : 0.0f;
    d.tau[link] += applied;
}

// OpApplyDrives (articulation.cu:1604-1620).  Without drive rows in the cooked world tau is the applied generalized
// force and the op only validates; IntegrateVelocity acts on a free body only (ops_rigid.hip).
Status OpApplyDrives(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const ApplyDrivesParams*>(params);
    if (p == nullptr || p->mode > kDriveActuator) return Status::InvalidArgument;
    // a world cooked without drive rows leaves `tau` as the applied generalized force: nothing to turn into rows
    if (m.joint_drive_rows == 0u) return p->mode == kDriveTorque ? Status::Ok : Status::Unsupported;
    if (p->mode == kDriveComputedTorque || p->mode == kDriveOsc) return Status::Unsupported;
    if (p->total_link_count == 0u) return Status::Ok;
    if (p->links_per_env == 0u || p->links_per_env != m.links_per_env) return Status::InvalidArgument;
    hipLaunchKernelGGL(ApplyAffineDriveKernel, dim3((p->total_link_count + 255u) / 256u), dim3(256), 0, stream, m, d, *p);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}
// OpReadoutDrives (articulation.cu:1654-1667)
Status OpReadoutDrives(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const ReadoutDrivesParams*>(params);
    if (p == nullptr || p->dt <= 0.0f) return Status::InvalidArgument;
    if (p->total_link_count == 0u) return Status::Ok;
    if (p->links_per_env == 0u || p->links_per_env != m.links_per_env || p->first_drive_row + p->links_per_env > p->rows_per_env)
        return Status::InvalidArgument;
    hipLaunchKernelGGL(ReadoutDrivesKernel, dim3((p->total_link_count + 255u) / 256u), dim3(256), 0, stream, m, d, *p);
    return hipGetLastError() == hipSuccess ? Status::Ok : Status::Failed;
}
Status OpIntegrateVelocity(const ModelView& m, const DataView& d, const void* params, hipStream_t stream) {
    const auto* p = static_cast<const IntegrateVelocityParams*>(params);
    if (p == nullptr) return Status::Failed;
    if (p->dt <= 0.0f) return Status::Ok;
    if (m.free_body != 0u && p->total_body_count > 0u) return BodyIntegrateVelocity(m, d, *p, stream);
    return Status::Ok;
}

}  // namespace nkh
