// A whole step of a serial chain in a world without rows, a lane an environment: poses for the links' wrenches, forward
// dynamics, integration, world poses, link twists and body poses (the ops of OpStep, ops_articulation.hip, which includes this).
#pragma once

// ---- A lane an environment ------------------------------------------------------------------------------
// ArticulationDynamicsKernel gives an environment eight lanes or more and sweeps its tree a depth at a time, each depth a trip
// through LDS behind the one before; of a chain a depth is one link, so a sweep keeps six lanes of eight at work on one row
// each.  Here a lane walks its environment's chain alone: link l hangs from link l - 1, so what a sweep hands on is in the lane's
// registers, a wavefront's instruction serves 64 environments and nothing waits but the wavefronts at their barriers.  Four of
// them share a workgroup's environments: each makes the rotations of two links; the first then takes the bias forces and the
// second the composite inertias; each pushes two of the mass columns to the root; the second factors and solves while the
// fourth carries the matrices to memory; the sines of the new coordinates are two links a wavefront's again, and poses, twists and
// accelerations a wavefront's each.  What bounds it is that chain of arithmetic, whatever the batch up to the two workgroups a
// compute unit that LDS holds.  Products and sums are fused, transforms applied by their rotation and offset
// (X = [[E, 0], [-E t x, E]]) and inertias kept symmetric, half the instructions of the general kernel's products; the results
// differ from its in their last places and lie as near a double-precision step.
// Eight: 78 KB of LDS, two workgroups a compute unit; nine links take 86 KB, one.
constexpr uint32_t kChainLinks = 8u;
// From so many environments on: the kernel takes as long for one of them as for sixty-four, so that no fewer are worth it, and a longer
// chain is a longer walk for its one lane while the general kernel's lanes still fill an idle machine (a step, general kernel and this one:
// five links, 64 environments 21.4 and 19.1 us; six, 64 22.6 and 21.5, 256 22.2 and 21.8; seven, 64 23.9 and 24.0, 256 23.4 and 24.3, 320
// 24.8 and 24.3; eight, 64 25.1 and 26.5, 512 26.0 and 27.1, 576 27.8 and 27.1, 1024 29.4 and 27.3).
__host__ __device__ constexpr uint32_t ChainFrom(uint32_t links) { return links <= 6u ? 64u : 256u * (links - 6u) + 1u; }

// a link's constants in LDS
enum ChainWord : uint32_t {
    cRotation = 0u,       // the joint's frame in the parent: nine words, row-major
    cTurns = 9u,          // all bits where the joint turns, else none
    cOffset = 12u,        // ... and its origin
    cSlide = 16u,         // what a slider's coordinate adds to it
    cSlides = 19u,        // all bits where it does, else none
    cAxis = 20u,          // unit axis, zero for none
    cAngular = 24u,       // motion subspace
    cLinear = 28u,
    cInertia = 32u,       // upper triangle of the angular block (6), the coupling block (9), upper triangle of the linear block (6)
    cDamping = 53u, cArmature, cStiffness, cReference,
    cQuat = 57u,
    cDof = 61u,           // as a word; kInvalid where the joint has none
    kChainWords = 64u
};
struct ChainMotion { V3 w, v; };                        // angular, linear
struct ChainFrame { float r[9]; V3 t; };                // child to parent: rotation and the child's origin
__device__ __forceinline__ V3 fma3(V3 a, float s, V3 b) { return V3{fmaf(a.x, s, b.x), fmaf(a.y, s, b.y), fmaf(a.z, s, b.z)}; }
__device__ __forceinline__ V3 add_cross(V3 a, V3 b, V3 c) {   // c + a x b
    return V3{fmaf(a.y, b.z, fmaf(-a.z, b.y, c.x)), fmaf(a.z, b.x, fmaf(-a.x, b.z, c.y)), fmaf(a.x, b.y, fmaf(-a.y, b.x, c.z))};
}
__device__ __forceinline__ V3 negative(V3 a) { return V3{-a.x, -a.y, -a.z}; }
__device__ __forceinline__ float dot_add(V3 a, V3 b, float c) { return fmaf(a.x, b.x, fmaf(a.y, b.y, fmaf(a.z, b.z, c))); }
__device__ __forceinline__ V3 turn(const float* r, V3 a) {      // R a
    return V3{fmaf(r[0], a.x, fmaf(r[1], a.y, r[2] * a.z)), fmaf(r[3], a.x, fmaf(r[4], a.y, r[5] * a.z)), fmaf(r[6], a.x, fmaf(r[7], a.y, r[8] * a.z))};
}
__device__ __forceinline__ V3 turn_back(const float* r, V3 a) { // R^T a
    return V3{fmaf(r[0], a.x, fmaf(r[3], a.y, r[6] * a.z)), fmaf(r[1], a.x, fmaf(r[4], a.y, r[7] * a.z)), fmaf(r[2], a.x, fmaf(r[5], a.y, r[8] * a.z))};
}
__device__ __forceinline__ ChainMotion to_child(const ChainFrame& f, ChainMotion m) {   // X m
    return ChainMotion{turn_back(f.r, m.w), turn_back(f.r, add_cross(m.w, f.t, m.v))};
}
__device__ __forceinline__ ChainMotion to_parent(const ChainFrame& f, ChainMotion p) {  // X^T p of a force (moment, force)
    const V3 force = turn(f.r, p.v);
    return ChainMotion{add_cross(f.t, force, turn(f.r, p.w)), force};
}
__device__ __forceinline__ ChainMotion add_motion(ChainMotion a, ChainMotion b) { return ChainMotion{add3(a.w, b.w), add3(a.v, b.v)}; }
__device__ __forceinline__ float dot_motion(ChainMotion a, ChainMotion b) { return dot_add(a.w, b.w, dot_add(a.v, b.v, 0.0f)); }

struct ChainInertia { float a[6], b[9], d[6]; };        // [[a, b], [b^T, d]]; triangles xx xy xz yy yz zz
__device__ __forceinline__ V3 times_triangle(const float* s, V3 x) {
    return V3{fmaf(s[0], x.x, fmaf(s[1], x.y, s[2] * x.z)), fmaf(s[1], x.x, fmaf(s[3], x.y, s[4] * x.z)), fmaf(s[2], x.x, fmaf(s[4], x.y, s[5] * x.z))};
}
__device__ __forceinline__ ChainMotion times_inertia(const ChainInertia& i, ChainMotion m) {
    return ChainMotion{add3(times_triangle(i.a, m.w), turn(i.b, m.v)), add3(turn_back(i.b, m.w), times_triangle(i.d, m.v))};
}
// R s R^T of a triangle
__device__ __forceinline__ void turn_triangle(const float* r, const float* s, float* out) {
    const V3 rows[3] = {V3{r[0], r[1], r[2]}, V3{r[3], r[4], r[5]}, V3{r[6], r[7], r[8]}};
    const V3 x = times_triangle(s, rows[0]), y = times_triangle(s, rows[1]), z = times_triangle(s, rows[2]);
    out[0] = dot_add(x, rows[0], 0.0f); out[1] = dot_add(x, rows[1], 0.0f); out[2] = dot_add(x, rows[2], 0.0f);
    out[3] = dot_add(y, rows[1], 0.0f); out[4] = dot_add(y, rows[2], 0.0f); out[5] = dot_add(z, rows[2], 0.0f);
}
// `into` += X^T child X
__device__ __forceinline__ void push_inertia(const ChainFrame& f, const ChainInertia& child, ChainInertia& into) {
    float a[6], b[9], d[6];
    turn_triangle(f.r, child.a, a);
    turn_triangle(f.r, child.d, d);
    const V3 rows[3] = {V3{f.r[0], f.r[1], f.r[2]}, V3{f.r[3], f.r[4], f.r[5]}, V3{f.r[6], f.r[7], f.r[8]}};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const V3 x = turn_back(child.b, rows[i]);
#pragma unroll
        for (int j = 0; j < 3; ++j) b[3 * i + j] = dot_add(x, rows[j], 0.0f);
    }
    // with s = t x: the coupling gains s d, the angular block s b^T - (b + s d) s
    const float D[9] = {d[0], d[1], d[2], d[1], d[3], d[4], d[2], d[4], d[5]};
    const V3 t = f.t;
    float moved[9];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        moved[c] = fmaf(t.y, D[6 + c], fmaf(-t.z, D[3 + c], b[c]));
        moved[3 + c] = fmaf(t.z, D[c], fmaf(-t.x, D[6 + c], b[3 + c]));
        moved[6 + c] = fmaf(t.x, D[3 + c], fmaf(-t.y, D[c], b[6 + c]));
    }
    // (s b^T)_rc = (t x column c of b^T)_r = (t x row c of b)_r, ((moved) s)_rc = (row r of moved x t)_c
    const auto before = [&](int r, int c) {
        const float* row = b + 3 * c;
        return r == 0 ? fmaf(t.y, row[2], -t.z * row[1]) : r == 1 ? fmaf(t.z, row[0], -t.x * row[2]) : fmaf(t.x, row[1], -t.y * row[0]);
    };
    const auto behind = [&](int r, int c, float from) {
        const float* row = moved + 3 * r;
        return c == 0 ? fmaf(-row[1], t.z, fmaf(row[2], t.y, from)) : c == 1 ? fmaf(-row[2], t.x, fmaf(row[0], t.z, from)) : fmaf(-row[0], t.y, fmaf(row[1], t.x, from));
    };
    int at = 0;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = r; c < 3; ++c, ++at) { into.a[at] += behind(r, c, a[at] + before(r, c)); into.d[at] += d[at]; }
#pragma unroll
    for (int e = 0; e < 9; ++e) into.b[e] += moved[e];
}

__device__ __forceinline__ V3 chain_vector(const float* words) { return V3{words[0], words[1], words[2]}; }
__device__ __forceinline__ ChainInertia chain_inertia(const float* link) {
    ChainInertia i;
#pragma unroll
    for (int e = 0; e < 6; ++e) { i.a[e] = link[cInertia + e]; i.d[e] = link[cInertia + 15 + e]; }
#pragma unroll
    for (int e = 0; e < 9; ++e) i.b[e] = link[cInertia + 6 + e];
    return i;
}
__device__ __forceinline__ ChainMotion chain_axis(const float* link) { return ChainMotion{chain_vector(link + cAngular), chain_vector(link + cLinear)}; }
__device__ __forceinline__ ChainMotion axis_times(ChainMotion axis, float rate, ChainMotion add) { return ChainMotion{fma3(axis.w, rate, add.w), fma3(axis.v, rate, add.v)}; }
// mat3_axis_angle behind the joint's own frame, from the sine and the cosine of the angle (of zero where the joint does not turn)
__device__ __forceinline__ void chain_rotation(const float* link, float s, float c, float* r) {
#pragma unroll
    for (int e = 0; e < 9; ++e) r[e] = link[cRotation + e];
    const V3 n = chain_vector(link + cAxis);
    const float t = 1.0f - c;
    const V3 tn = scale3(n, t), sn = scale3(n, s);
    const float j[9] = {fmaf(tn.x, n.x, c), fmaf(tn.x, n.y, -sn.z), fmaf(tn.x, n.z, sn.y), fmaf(tn.x, n.y, sn.z), fmaf(tn.y, n.y, c),
                        fmaf(tn.y, n.z, -sn.x), fmaf(tn.x, n.z, -sn.y), fmaf(tn.y, n.z, sn.x), fmaf(tn.z, n.z, c)};
    float out[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) out[3 * i + k] = fmaf(r[3 * i], j[k], fmaf(r[3 * i + 1], j[3 + k], r[3 * i + 2] * j[6 + k]));
#pragma unroll
    for (int e = 0; e < 9; ++e) r[e] = out[e];
}
// A coordinate counts where the joint has a use for it and not otherwise: its bits are taken or left, for zero times a word that is
// not finite is not zero.  (Selected offsets and angles, three instructions for one, cost 20011 arms half a microsecond of 35.5.)
__device__ __forceinline__ float chain_used(const float* link, uint32_t mask, float q) { return __uint_as_float(__float_as_uint(q) & __float_as_uint(link[mask])); }
__device__ __forceinline__ float chain_angle(const float* link, float q) { return chain_used(link, cTurns, q); }
__device__ __forceinline__ V3 chain_offset(const float* link, float q) { return fma3(chain_vector(link + cSlide), chain_used(link, cSlides, q), chain_vector(link + cOffset)); }
// joint_relative_frame from the link's constants and the sine and the cosine of half the angle
__device__ __forceinline__ Xf chain_place(const float* link, float q, float s, float c) {
    Xf place{chain_offset(link, q), Q4{link[cQuat], link[cQuat + 1], link[cQuat + 2], link[cQuat + 3]}};
    const V3 n = chain_vector(link + cAxis);
    const Q4 turned = qnormalize_le(qmul(place.r, Q4{c, n.x * s, n.y * s, n.z * s}), 1.0e-12f);
    if (__float_as_uint(link[cTurns]) != 0u) place.r = turned;
    return place;
}
__device__ __forceinline__ Xf lane_pose(const Xf& x, uint32_t lane) {
    const auto at = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), int(lane))); };
    return Xf{V3{at(x.p.x), at(x.p.y), at(x.p.z)}, Q4{at(x.r.w), at(x.r.x), at(x.r.y), at(x.r.z)}};
}
// consecutive words of a lane's own, sixteen bytes at a time from any word on
typedef float ChainFour __attribute__((ext_vector_type(4), aligned(4)));
typedef float ChainTwo __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ void store_motion(float* to, ChainMotion m) {
    *reinterpret_cast<ChainFour*>(to) = ChainFour{m.w.x, m.w.y, m.w.z, m.v.x};
    *reinterpret_cast<ChainTwo*>(to + 4) = ChainTwo{m.v.y, m.v.z};
}
__device__ __forceinline__ void store_pose(float* to, const Xf& x) {
    *reinterpret_cast<ChainFour*>(to) = ChainFour{x.p.x, x.p.y, x.p.z, x.r.w};
    *reinterpret_cast<ChainTwo*>(to + 4) = ChainTwo{x.r.x, x.r.y};
    to[6] = x.r.z;
}
__device__ __forceinline__ ChainMotion load_motion(const float* from) {
    const ChainFour a = *reinterpret_cast<const ChainFour*>(from);
    const ChainTwo b = *reinterpret_cast<const ChainTwo*>(from + 4);
    return ChainMotion{V3{a[0], a[1], a[2]}, V3{a[3], b[0], b[1]}};
}
// 64 environments' n x n words, laid out in LDS a lane's behind another `apart` words on, to the consecutive words they have in
// memory; of a factor (kLower) the lower triangle alone
template <bool kLower>
__device__ __forceinline__ void store_matrices(float* out, const float* staged, uint32_t apart, uint32_t n, uint32_t envs, uint32_t lane) {
    constexpr uint32_t kAhead = 8u;   // reads in flight
    const uint32_t words = n * n, all = envs * words, by_row = 65536u / n + 1u;
    const uint32_t envs_a_step = uint32_t(kWave) / words, words_a_step = uint32_t(kWave) - envs_a_step * words;
    uint32_t env = lane / words, word = lane - env * words;
    for (uint32_t e = lane; e < all; e += kAhead * kWave) {
        float value[kAhead];
        bool taken[kAhead];
#pragma unroll
        for (uint32_t t = 0u; t < kAhead; ++t) {
            const bool inside = e + t * kWave < all;
            const uint32_t row = (word * by_row) >> 16u;   // word / n, word < 64
            taken[t] = inside && (!kLower || word - row * n <= row);
            value[t] = staged[inside ? env * apart + word : 0u];
            env += envs_a_step; word += words_a_step;
            if (word >= words) { word -= words; ++env; }
        }
#pragma unroll
        for (uint32_t t = 0u; t < kAhead; ++t) if (taken[t]) out[e + t * kWave] = value[t];
    }
}
// What a collidable row's pose follows from (body_pose_of): read in two rounds, whatever the first finds, and looked at last, so that
// nothing waits for either
struct ChainBody {
    uint32_t b, own, proxy, owner, kind;
    Xf local;
    __device__ __forceinline__ void look(const ModelView& m, uint32_t body) {
        b = body;
        own = m.body_to_link[min(b, m.bodies_per_env - 1u)]; proxy = m.body_collidable_link[min(b, m.bodies_per_env - 1u)];
    }
    __device__ __forceinline__ void follow(const ModelView& m) {
        const uint32_t link = own != kInvalid ? own : 0u;
        owner = m.link_body[link]; kind = m.link_geom_kind[link];
        local = load_xf(own != kInvalid ? m.link_geom_local + 7u * link : m.body_collidable_local + 7u * min(b, m.bodies_per_env - 1u));
    }
    __device__ __forceinline__ uint32_t link(const ModelView& m) const {   // kInvalid: the row keeps the pose it has
        const uint32_t follows = own != kInvalid ? (owner == b ? own : kInvalid) : (proxy < m.links_per_env ? proxy : kInvalid);
        return b < m.bodies_per_env ? follows : kInvalid;
    }
    __device__ __forceinline__ uint32_t composed() const { return own == kInvalid || kind != 0u ? 1u : 0u; }
};
// LDS of a workgroup in words: the links' constants; a word or a vector a lane and link each ([link][component][lane]): coordinate,
// rate, right-hand side (the acceleration later), rotation to the parent, bias acceleration, force and mass column; the matrices, a
// lane's behind another's an odd number of words on.  The new coordinates' sines and the poses take the forces' and the columns' place.
__host__ __device__ constexpr uint32_t ChainMatrixWords(uint32_t stride) { return (stride * stride) | 1u; }
__host__ __device__ constexpr uint32_t ChainLdsWords(uint32_t nl, uint32_t stride) { return nl * kChainWords + uint32_t(kWave) * (nl * (3u + 9u + 3u * 6u) + ChainMatrixWords(stride)); }
// (a lane and link's four words of sines and seven of the pose, with a lane's odd word behind them, are no more than its twelve)

__device__ __forceinline__ void put_motion(float* at, ChainMotion m) {
    at[0] = m.w.x; at[kWave] = m.w.y; at[2 * kWave] = m.w.z; at[3 * kWave] = m.v.x; at[4 * kWave] = m.v.y; at[5 * kWave] = m.v.z;
}
__device__ __forceinline__ ChainMotion get_motion(const float* at) {
    return ChainMotion{V3{at[0], at[kWave], at[2 * kWave]}, V3{at[3 * kWave], at[4 * kWave], at[5 * kWave]}};
}

// The walks along the links are loops that stay loops: unrolled, with everything of a link in registers, the kernel's 126 KB of
// code are fetched once a wavefront and the fetches are what it takes (64 arms 31 us a step with the general kernel, 43 so).
constexpr uint32_t kChainWaves = 4u;
__global__ void __launch_bounds__(kChainWaves * kWave)
ChainStepKernel(ModelView m, DataView d, ArticulationDynamicsParams p, uint32_t env_count, StepTail tail) {
    extern __shared__ float lds[];
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave))), lane = threadIdx.x % kWave;
    const uint32_t nl = m.links_per_env, n = m.dof, stride = m.max_dof;
    const uint32_t first = blockIdx.x * uint32_t(kWave), envs = min(env_count - first, uint32_t(kWave));
    const bool there = lane < envs;
    const size_t env = first + min(lane, envs - 1u), lbase = env * nl;
    const float dt = p.dt;
    const uint32_t apart = ChainMatrixWords(stride);
    float* links = lds;
    float* q = links + nl * kChainWords + lane;             // a link's word at l * kWave
    float* qd = q + nl * kWave;
    float* rhs = qd + nl * kWave;                           // by coordinate
    float* rotation = rhs + nl * kWave;                     // at l * 9 * kWave, a component at its number * kWave
    float* bias_motion = rotation + nl * 9u * kWave;        // at l * 6 * kWave
    float* force = bias_motion + nl * 6u * kWave;
    float* column = force + nl * 6u * kWave;                // by coordinate
    float* staged = column - lane + nl * 6u * kWave;
    float* mine = staged + lane * apart;
    float* sines = force;                                   // at l * 4 * kWave: of the whole new angle and of half of it
    float* pose = sines - lane + nl * 4u * kWave + lane * (nl * 7u + 1u);   // (a lane's by itself: nl * 7 + 1 words apart, an odd number or bank conflicts)
    const ChainMotion still{V3{0.0f, 0.0f, 0.0f}, V3{0.0f, 0.0f, 0.0f}};
    const ChainMotion ground{still.w, V3{-p.gravity[0], -p.gravity[1], -p.gravity[2]}};
    // The bodies go round the wavefronts: a lane looks at one of its wavefront's, and those that follow a link take turns at the end.  (One
    // after the other by the poses' wavefront, and each looked up as its turn came, 64 chains of eight links with 100 bodies beside the
    // links' that stand still took 45.6 us a step and with 32 that move 45.5, 31.4 by the general kernel.)
    const bool bodies = tail.sync_bodies != 0u && m.bodies_per_env != 0u;   // uniform
    ChainBody body{};
    if (bodies) body.look(m, lane * kChainWaves + wave);
    // the links' constants by the first wavefront, the state by the second and the third; whether any link has a wrench on it
    bool wrenches = false;
    if (wave == 0u) {
        ChainMotion w[kChainLinks];
        if (p.apply_link_wrench != 0u || p.integrate_velocity != 0u) {
#pragma unroll
            for (uint32_t l = 0u; l < kChainLinks; ++l) w[l] = load_motion(d.link_wrench + (lbase + min(l, nl - 1u)) * 6u);
        }
        if (lane < nl) {
            float* link = links + lane * kChainWords;
            const uint8_t type = m.joint_type[lane];
            const V3 authored = load3(m.joint_axis + 3u * lane);
            const Xf local = load_xf(m.link_local_pose + 7u * lane);
            const float length = dot3(authored, authored);
            const bool directed = length > 1.0e-12f;
            const V3 axis = directed ? scale3(authored, rsqrt_exact(length)) : still.w;
            const V3 offset = add3(local.p, load3(m.parent_offset + 3u * lane));
            const V3 slide = type == kPrismatic ? rotate_normalized(local.r, axis) : still.w;
            const V3 subspace = directed ? axis : authored;   // (motion_subspace keeps an axis too short to normalise)
            const V3 angular = type == kRevolute ? subspace : still.w, linear = type == kPrismatic ? subspace : still.w;
            mat3_from_quat(local.r, link + cRotation);
            link[cTurns] = __uint_as_float(type == kRevolute && directed ? ~0u : 0u);
            link[cSlides] = __uint_as_float(type == kPrismatic ? ~0u : 0u);
            const auto put = [&](uint32_t at, V3 v) { link[at] = v.x; link[at + 1u] = v.y; link[at + 2u] = v.z; };
            put(cOffset, offset); put(cSlide, slide); put(cAxis, axis); put(cAngular, angular); put(cLinear, linear);
            const float* inertia = m.link_inertia + 36u * lane;
            uint32_t at = 0u;
#pragma unroll
            for (uint32_t r = 0u; r < 3u; ++r)
#pragma unroll
                for (uint32_t c = 0u; c < 3u; ++c) {
                    link[cInertia + 6u + 3u * r + c] = inertia[6u * r + 3u + c];
                    if (c >= r) { link[cInertia + at] = inertia[6u * r + c]; link[cInertia + 15u + at] = inertia[6u * (3u + r) + 3u + c]; ++at; }
                }
            link[cDamping] = m.joint_damping[lane]; link[cArmature] = m.joint_armature[lane];
            link[cStiffness] = m.joint_stiffness[lane]; link[cReference] = m.joint_spring_reference[lane];
            link[cQuat] = local.r.w; link[cQuat + 1u] = local.r.x; link[cQuat + 2u] = local.r.y; link[cQuat + 3u] = local.r.z;
            link[cDof] = __uint_as_float(joint_dof(type) == 1u ? m.link_dof[lane] : kInvalid);
        }
        if (p.apply_link_wrench != 0u || p.integrate_velocity != 0u) {
            uint32_t bits = 0u;
#pragma unroll
            for (uint32_t l = 0u; l < kChainLinks; ++l)
                bits |= (__float_as_uint(w[l].w.x) | __float_as_uint(w[l].w.y) | __float_as_uint(w[l].w.z)) | (__float_as_uint(w[l].v.x) | __float_as_uint(w[l].v.y) | __float_as_uint(w[l].v.z));
            wrenches = __any(bits != 0u);
        }
    } else if (wave <= 2u) {
        const float* from = (wave == 1u ? d.q : d.qdot) + lbase;
        float word[kChainLinks];
#pragma unroll
        for (uint32_t l = 0u; l < kChainLinks; ++l) word[l] = from[min(l, nl - 1u)];
#pragma unroll
        for (uint32_t l = 0u; l < kChainLinks; ++l) if (l < nl) (wave == 1u ? q : qd)[l * kWave] = word[l];
    }
    __syncthreads();
    const auto dof_of = [&](uint32_t l) { return uint32_t(__builtin_amdgcn_readfirstlane(int(__float_as_uint(links[l * kChainWords + cDof])))); };
#pragma unroll 1
    for (uint32_t l = wave; l < nl; l += kChainWaves) {
        const float* link = links + l * kChainWords;
        float s, c, r[9];
        sincosf(chain_angle(link, q[l * kWave]), &s, &c);
        chain_rotation(link, s, c, r);
#pragma unroll
        for (int e = 0; e < 9; ++e) rotation[(l * 9u + uint32_t(e)) * kWave] = r[e];
    }
    __syncthreads();
    const auto frame_of = [&](uint32_t l) {
        ChainFrame f;
#pragma unroll
        for (int e = 0; e < 9; ++e) f.r[e] = rotation[(l * 9u + uint32_t(e)) * kWave];
        f.t = chain_offset(links + l * kChainWords, q[l * kWave]);
        return f;
    };
    if (wave == 0u) {
        // root to leaf: twists, bias accelerations, and each link's force; then the forces leaf to root
        ChainMotion v = still, a = ground;
        Xf place{};
#pragma unroll 1
        for (uint32_t l = 0u; l < nl; ++l) {
            const float* link = links + l * kChainWords;
            const ChainFrame f = frame_of(l);
            const float rate = qd[l * kWave];
            const ChainMotion axis = chain_axis(link), own{scale3(axis.w, rate), scale3(axis.v, rate)};
            const ChainInertia inertia = chain_inertia(link);
            v = add_motion(to_child(f, v), own);
            const ChainMotion bias{add_cross(v.w, own.w, still.w), add_cross(v.w, own.v, add_cross(v.v, own.w, still.v))};
            put_motion(bias_motion + l * 6u * kWave, bias);
            a = add_motion(to_child(f, a), bias);
            const ChainMotion momentum = times_inertia(inertia, v), moved = times_inertia(inertia, a);
            ChainMotion acting{add_cross(v.w, momentum.w, add_cross(v.v, momentum.v, moved.w)), add_cross(v.w, momentum.v, moved.v)};
            if (wrenches) {   // (x, y, z: a force, then a torque, on the link in world axes)
                float s, c;
                sincosf(0.5f * q[l * kWave], &s, &c);
                const Xf relative = chain_place(link, q[l * kWave], s, c);
                place = l == 0u ? relative : compose_frame(place, relative);
                if (p.apply_link_wrench != 0u) {
                    const ChainMotion wrench = load_motion(d.link_wrench + (lbase + l) * 6u);
                    const V3 push = rotate_inverse(place.r, wrench.w), torque = rotate_inverse(place.r, wrench.v);
                    const V3 moment = add3(torque, cross3(load_xf(m.link_inertial_frame + 7u * l).p, push));
                    // (nothing of a wrench of zeros: an orientation past the range of floats would make something of it)
                    const bool acts = wrench.w.x != 0.0f || wrench.w.y != 0.0f || wrench.w.z != 0.0f || wrench.v.x != 0.0f || wrench.v.y != 0.0f || wrench.v.z != 0.0f;
                    acting.w = sub3(acting.w, acts ? moment : still.w); acting.v = sub3(acting.v, acts ? push : still.v);
                }
                if (p.integrate_velocity != 0u && there) store_motion(d.link_wrench + (lbase + l) * 6u, still);
            }
            put_motion(force + l * 6u * kWave, acting);
        }
        ChainMotion behind = still;
#pragma unroll 1
        for (uint32_t l = nl; l-- > 0u;) {
            const float* link = links + l * kChainWords;
            const uint32_t dof = dof_of(l);
            const ChainFrame f = frame_of(l);
            const ChainMotion total = add_motion(get_motion(force + l * 6u * kWave), behind);
            if (dof != kInvalid) rhs[dof * kWave] = dot_motion(chain_axis(link), total);   // uniform
            behind = to_parent(f, total);
        }
        // generalized bias and right-hand side
        float* bias = d.articulation_bias + env * stride;
        float gravity[kChainLinks], torque[kChainLinks], drive[kChainLinks];
#pragma unroll
        for (uint32_t k = 0u; k < kChainLinks; ++k) {
            const uint32_t l = min(k, nl - 1u);
            gravity[k] = d.joint_gravity_force[lbase + l]; torque[k] = d.tau[lbase + l];
            drive[k] = p.fold_drive_damping != 0u ? d.drive_dissipation[lbase + l] : 0.0f;
        }
#pragma unroll
        for (uint32_t l = 0u; l < kChainLinks; ++l) {
            if (l >= nl) break;
            const float* link = links + l * kChainWords;
            const uint32_t dof = dof_of(l);
            if (dof == kInvalid) continue;   // uniform
            const float b = rhs[dof * kWave] + gravity[l], spring = link[cStiffness] * (q[l * kWave] - link[cReference]);
            rhs[dof * kWave] = fmaf(-(link[cDamping] + drive[l]), qd[l * kWave], torque[l] - b) - spring;
            if (there) bias[dof] = b;
        }
        if (there) for (uint32_t i = n; i < stride; ++i) bias[i] = 0.0f;
    } else if (wave == 1u) {
        ChainInertia composite{};
#pragma unroll 1
        for (uint32_t l = nl; l-- > 0u;) {
            const float* link = links + l * kChainWords;
            const ChainFrame f = frame_of(l);
            const ChainInertia own = chain_inertia(link);
#pragma unroll
            for (int e = 0; e < 6; ++e) { composite.a[e] += own.a[e]; composite.d[e] += own.d[e]; }
#pragma unroll
            for (int e = 0; e < 9; ++e) composite.b[e] += own.b[e];
            const uint32_t dof = dof_of(l);
            if (dof != kInvalid) {   // uniform
                const ChainMotion axis = chain_axis(link), start = times_inertia(composite, axis);
                float diagonal = dot_motion(axis, start) + link[cArmature];
                if (p.fold_drive_damping != 0u) diagonal = fmaf(dt, d.drive_dissipation[lbase + l], diagonal);
                put_motion(column + dof * 6u * kWave, start);
                mine[dof * stride + dof] = diagonal;
            }
            if (l > 0u) {
                ChainInertia above{};
                push_inertia(f, composite, above);
                composite = above;
            }
        }
    } else if (wave == 2u) {
        for (uint32_t i = n; i < stride; ++i)   // rows and columns past the coordinates
            for (uint32_t j = 0u; j < stride; ++j) { mine[i * stride + j] = 0.0f; mine[j * stride + i] = 0.0f; }
    }
    __syncthreads();
    // each jointed link's column on to the root, the longest walks and the shortest a wavefront
#pragma unroll 1
    for (uint32_t turn = 0u; turn < 2u; ++turn) {
        const uint32_t l0 = turn == 0u ? nl - 1u - min(wave, nl - 1u) : nl - 1u - min(2u * kChainWaves - 1u - wave, nl - 1u);
        const uint32_t k = dof_of(l0);
        if (k == kInvalid || (turn == 0u ? wave : 2u * kChainWaves - 1u - wave) >= nl) continue;   // uniform
        ChainMotion pushed = get_motion(column + k * 6u * kWave);
#pragma unroll 1
        for (uint32_t l = l0; l > 0u; --l) {
            pushed = to_parent(frame_of(l), pushed);
            const uint32_t j = dof_of(l - 1u);
            if (j == kInvalid) continue;   // uniform
            const float entry = dot_motion(chain_axis(links + (l - 1u) * kChainWords), pushed);
            mine[k * stride + j] = entry; mine[j * stride + k] = entry;
        }
    }
    __syncthreads();   // the matrix and the right-hand side stand; forces and columns have been read
    float A[kChainLinks][kChainLinks];   // rows past the coordinates the identity's; lower triangle
    if (wave == 3u) {
        store_matrices<false>(d.m + size_t{first} * stride * stride, staged, apart, stride, envs, lane);
    } else if (wave == 1u) {
#pragma unroll
        for (uint32_t i = 0u; i < kChainLinks; ++i)
#pragma unroll
            for (uint32_t j = 0u; j <= i; ++j) A[i][j] = i < n ? mine[i * stride + j] : (i == j ? 1.0f : 0.0f);
        // L D L^T (ldlt_pivots)
#pragma unroll
        for (uint32_t k = 0u; k < kChainLinks; ++k) {
            A[k][k] = fmaxf(A[k][k], 1.0e-6f);
            const Recip by_pivot = make_recip(A[k][k]);
            float scaled[kChainLinks];
#pragma unroll
            for (uint32_t i = k + 1u; i < kChainLinks; ++i) scaled[i] = div_by(A[i][k], by_pivot);
#pragma unroll
            for (uint32_t i = k + 1u; i < kChainLinks; ++i)
#pragma unroll
                for (uint32_t j = k + 1u; j <= i; ++j) A[i][j] = fmaf(-scaled[i], A[j][k], A[i][j]);
#pragma unroll
            for (uint32_t i = k + 1u; i < kChainLinks; ++i) A[i][k] = scaled[i];
        }
        float x[kChainLinks];
#pragma unroll
        for (uint32_t i = 0u; i < kChainLinks; ++i) x[i] = i < n ? rhs[i * kWave] : 0.0f;
#pragma unroll
        for (uint32_t i = 1u; i < kChainLinks; ++i)
#pragma unroll
            for (uint32_t j = 0u; j < i; ++j) x[i] = fmaf(-A[i][j], x[j], x[i]);
#pragma unroll
        for (uint32_t i = 0u; i < kChainLinks; ++i) x[i] = div_by(x[i], make_recip(A[i][i]));
#pragma unroll
        for (int i = int(kChainLinks) - 2; i >= 0; --i)
#pragma unroll
            for (int k = i + 1; k < int(kChainLinks); ++k) x[i] = fmaf(-A[k][i], x[k], x[i]);
#pragma unroll
        for (uint32_t i = 0u; i < kChainLinks; ++i) if (i < n) rhs[i * kWave] = x[i];
    }
    __syncthreads();   // the accelerations stand, the matrix is in memory
    // the velocities, the coordinates they lead to, and their sines
#pragma unroll 1
    for (uint32_t l = wave; l < nl; l += kChainWaves) {
        const uint32_t dof = dof_of(l);
        const float solved = dof != kInvalid ? rhs[dof * kWave] : 0.0f;
        float rate = qd[l * kWave];
        const bool moves = dof != kInvalid && p.integrate_velocity != 0u;   // uniform
        if (moves) rate = fmaf(dt, solved, rate);
        const float to = fmaf(tail.integrate.pos_pass != 0u ? rate + d.qdot_pseudo[lbase + l] : rate, tail.integrate.dt, q[l * kWave]);
        const float angle = chain_angle(links + l * kChainWords, to);
        float s, c, half_s, half_c;
        sincosf(angle, &s, &c);
        sincosf(0.5f * angle, &half_s, &half_c);
        float* at = sines + l * 4u * kWave;
        at[0] = s; at[kWave] = c; at[2u * kWave] = half_s; at[3u * kWave] = half_c;
        if (!there) continue;
        d.qddot[lbase + l] = solved;
        if (moves) d.qdot[lbase + l] = rate;
        d.q[lbase + l] = to;
    }
    if (wave == 1u) {
#pragma unroll
        for (uint32_t i = 0u; i < kChainLinks; ++i)
#pragma unroll
            for (uint32_t j = 0u; j <= i; ++j) if (i < n) mine[i * stride + j] = A[i][j];
        for (uint32_t i = n; i < stride; ++i) mine[i * stride + i] = 1.0e-6f;
    }
    __syncthreads();
    const auto advanced = [&](uint32_t l, float* rate) {   // as above
        const uint32_t dof = dof_of(l);
        *rate = qd[l * kWave];
        if (dof != kInvalid && p.integrate_velocity != 0u) *rate = fmaf(dt, rhs[dof * kWave], *rate);
        return fmaf(tail.integrate.pos_pass != 0u ? *rate + d.qdot_pseudo[lbase + l] : *rate, tail.integrate.dt, q[l * kWave]);
    };
    if (bodies) body.follow(m);
    if (wave == 0u) {
        Xf place{};
#pragma unroll 1
        for (uint32_t l = 0u; l < nl; ++l) {
            float rate;
            const Xf relative = chain_place(links + l * kChainWords, advanced(l, &rate), sines[(4u * l + 2u) * kWave], sines[(4u * l + 3u) * kWave]);
            place = l == 0u ? relative : compose_frame(place, relative);
            store_xf(pose + 7u * l, place);
            if (there) store_pose(d.link_pose + (lbase + l) * 7u, place);
        }
    } else if (wave == 1u) {
        ChainMotion v = still;
#pragma unroll 1
        for (uint32_t l = 0u; l < nl; ++l) {
            const float* link = links + l * kChainWords;
            float rate;
            ChainFrame f;
            f.t = chain_offset(link, advanced(l, &rate));
            chain_rotation(link, sines[4u * l * kWave], sines[(4u * l + 1u) * kWave], f.r);
            v = axis_times(chain_axis(link), rate, to_child(f, v));
            if (there) store_motion(d.link_velocity + (lbase + l) * 6u, v);
        }
    } else if (wave == 2u) {
        ChainMotion a = ground;
#pragma unroll 1
        for (uint32_t l = 0u; l < nl; ++l) {
            const uint32_t dof = dof_of(l);
            const float solved = dof != kInvalid ? rhs[dof * kWave] : 0.0f;
            a = axis_times(chain_axis(links + l * kChainWords), solved, add_motion(to_child(frame_of(l), a), get_motion(bias_motion + l * 6u * kWave)));
            if (there) store_motion(d.link_acceleration + (lbase + l) * 6u, a);
        }
        float* out = d.articulation_qdd + env * stride;
#pragma unroll
        for (uint32_t i = 0u; i < kChainLinks; ++i) if (there && i < stride) out[i] = i < n ? rhs[i * kWave] : 0.0f;
    } else {
        store_matrices<true>(d.m_factor + size_t{first} * stride * stride, staged, apart, stride, envs, lane);
    }
    if (!bodies) return;
    __syncthreads();   // the poses stand
#pragma unroll 1
    for (uint32_t from = 0u; from < m.bodies_per_env; from += kChainWaves * kWave) {
        if (from != 0u) { body.look(m, from + lane * kChainWaves + wave); body.follow(m); }
        const uint32_t link = body.link(m), composed = body.composed();
        for (uint64_t rest = __ballot(link != kInvalid); rest != 0ull; rest &= rest - 1ull) {
            const uint32_t i = uint32_t(__builtin_ctzll(rest)), b = from + i * kChainWaves + wave;
            Xf place = load_xf(pose + 7u * uint32_t(__builtin_amdgcn_readlane(int(link), int(i))));
            if (__builtin_amdgcn_readlane(int(composed), int(i)) != 0) place = compose_collidable(place, lane_pose(body.local, i));
            if (there) store_pose(d.body_pose + (env * m.bodies_per_env + b) * 7u, place);
        }
    }
}
