// Fused temporalCone control-step kernel for gfx950.
//
// One 64-lane workgroup (one wavefront) owns one world for a whole control
// step: reset/checkpoint, `physics_substeps` microsteps and the transactional
// commit. The world's articulation, colliders, active pairs and solver rows
// live in LDS; persistent state (q, v, scene bodies, manifolds) is read once
// at the start and written once at the end of the control step, so a failed
// step leaves HBM untouched (the checkpoint is the unmodified state). Lanes
// work on independent items (links of one tree level, colliders, compiled
// pairs, manifolds, constraint rows, generalized velocities); every item is
// computed with a fixed scalar evaluation order, and every order-dependent
// accumulation (children into a parent, contact impulses into a velocity)
// is performed by one owner lane in a fixed sequence. Results are therefore
// deterministic and independent of launch shape.
//
// Stage map to the reference (paths relative to the reference repository):
//   drive refresh        src/metal/MetalWorld.metal:280-366
//   kinematics + ABA     src/metal/ArticulatedABA.metal:352-1440
//   scene prediction     src/metal/MetalWorldContact.metal:2509-2567
//   collider projection  src/metal/Collision.metal:321-600, 5666-5712
//   pair flags / scan    src/metal/Collision.metal:796-858, 7905-8176
//   narrowphase          src/metal/Collision.metal:1003-1720, 4379-4830
//   manifolds            src/metal/Collision.metal:5108-5530, 9557-9830
//   emission             src/metal/Collision.metal:9180-9470
//   responses            src/metal/ArticulatedInverseMass.metal:1652-1700
//   IR evaluation        src/metal/MetalWorldContact.metal:3800-3995
//   cone solve           src/metal/MetalWorldContact.metal:482-720, 7856-8316
//   joint limits         src/metal/MetalWorldContact.metal:2878-2960
//   integration          src/metal/MetalWorldContact.metal:8876-9043
//   latch / commit       src/metal/MetalWorldContact.metal:9051-9082, MetalWorld.metal:372-519

#include "mr_device_math.h"
#include "mr_kernel_args.h"
#include "../../include/mr_c_api.h"
#include "mr_mlp_tile.h"

#include <mutex>

using namespace mrd;
using mr::ColdConstraint;
using mr::HotConstraint;
using mr::SolveBlock;
using mr::KernelArgs;

namespace {

constexpr float kTiny = 1.0e-14f;
constexpr float kFloatEps = 1.1920928955078125e-7f;
constexpr float kAbsolutePivotFloor = 1.0e-12f;
constexpr float kMatrixFloor = 1.0e-10f;
constexpr float kConeEpsilon = 1.0e-7f;
constexpr float kContactRegularization = 1.0e-2f;
constexpr uint32_t kLanes = 64u;

MRD_INL V3 f3(const mr_float4& v) { return V3{v.x, v.y, v.z}; }
MRD_INL Q4 q4(const mr_float4& v) { return Q4{v.x, v.y, v.z, v.w}; }
MRD_INL uint32_t feature_key(uint32_t t, uint32_t l) { return ((t & 0x0fu) << 28u) | (l & 0x0fffffffu); }

struct Collider {
    uint32_t type, body, disabled;
    V3 center;
    Q4 rotation;
    V3 lower, upper;
    float radius, half_length, contact_offset;
    V3 half_extents, p0, p1, plane_normal;
};

struct RawContact {
    V3 normal;
    float separation;
    V3 point_a, point_b;
    uint32_t feature_a, feature_b;
};

struct RawBatch {
    RawContact c[MR_RAW_CONTACTS_PER_PAIR];
    uint32_t count;
};

// Where a pair's raw contacts go: straight into the pair's manifold staging
// records (global), from which the eight lanes that build its manifold take
// them, one each. stage_p: eight words a contact (points, features); stage_h:
// the eight separations, then the deepest contact's normal. Nothing is kept in
// a private array, whose dynamic index would put it in scratch memory.
struct ContactSink {
    float* head;    // stage_h record of the pair
    float* points;  // stage_p records of the pair
    uint32_t count;
    // the deepest contact so far: smallest separation, then smallest features
    float deepest;
    uint32_t deepest_a, deepest_b;
    V3 normal;
    float rest, penetration;  // rest distance of the pair; largest rest - separation, at least 0
    bool bad;                 // some contact is not finite
};

MRD_INL V3 sym_mul(const float* s, V3 w) {
    return V3{s[0] * w.x + s[1] * w.y + s[2] * w.z, s[1] * w.x + s[3] * w.y + s[4] * w.z,
              s[2] * w.x + s[4] * w.y + s[5] * w.z};
}

// ------------------------------------------------------------ environment

// A float known to live in LDS: where one access may go to LDS or to global
// memory, the type keeps the compiler from folding the two into a flat access,
// which waits for both memories at once.
using LdsFloat = __attribute__((address_space(3))) float;

struct Env {
    const KernelArgs* a;
    uint32_t env;
    const MRModelHeaderC* hd;
    const MRBodyC* bodies;
    const MRDofC* dofs;
    const MRActuatorProfileC* acts;  // [nv] or null: every DoF inactive
    const MRShapeC* shapes;
    const MRMaterialC* mats;
    const MRCompiledPairC* pairs;
    uint32_t nlinks, nbodies, nv, nq, nshapes, npairs, nscene, levels, root_type;
    float h;
    V3 gravity;
    // LDS
    mr::TopoCache* topo;
    mr::LinkConst* lconst;
    float* arm;  // effective armature per DoF (constant for the launch)
    float *q, *v, *vcand, *effort, *accel, *cmd;
    V3 *pos, *w, *vl, *sa, *sl, *ca, *cl, *r;
    Q4* rot;
    float* I;            // [links][6][6]: articulated inertias of the inward pass, column-major
    float* p;            // [links][6]: bias torque and force of the inward pass
    V3 *Ut, *Ub;
    float *D, *u, *L;
    MRBodyStateC* scene;
    Collider *col, *ccol;  // ccol: swept colliders of the time-of-impact queries
    uint32_t* swept;       // [2 kLanes]: pairs waiting for their time-of-impact query
    uint32_t *active, *npts, *moff, *okey;
    uint32_t* hfitem;  // [kHfSlots]: active pair | query << 16
    mr::HfHit* hfq;    // [kHfSlots]: heightfield query results
    HotConstraint* hot;  // global scratch
    float* lam;          // LDS [ccap][3]
    uint32_t* cpair;     // LDS [ccap]: body_a | body_b << 8 | kind << 16
    float *rslot, *rstack;
    float* resid;
    float4* sbody;       // LDS [nscene][5]: SolverBody records of the ordered sweeps
    uint16_t* sord;      // LDS [ccap]: contacts in schedule order (schedule_contacts)
    LdsFloat* rows;      // LDS, unscheduled sweeps: rows and solve block of the first contacts
    float *jrelax, *jdelta;  // relaxed-Jacobi damping per contact and impulse deltas
    // MLP instance only
    unsigned char* mlp_lds;  // warm-start MLP tile scratch
    float* mlp_lam;          // [ccap][3] plain warm start, kept for the fallback
    MRBodyStateC* mlp_scene; // scene bodies before the warm start
    // global scratch of this environment
    MRManifoldHeaderC* stage_h;
    MRManifoldPointC* stage_p;
    float* jrow;
    float* resp;
    ColdConstraint* cold;
};

template <typename T>
MRD_INL T* lds_at(unsigned char* base, uint32_t off) {
    return reinterpret_cast<T*>(base + off);
}

MRD_INL bool is_link(const Env& e, uint32_t b) { return b < e.nlinks; }
MRD_INL uint32_t link_parent(const Env& e, uint32_t i) {
    const uint32_t p = e.topo->parent[i];
    return p == 0xffu ? MR_INVALID_INDEX : p;
}
MRD_INL uint32_t link_vidx(const Env& e, uint32_t i) {
    const uint32_t v = e.topo->vidx[i];
    return v == 0xffu ? MR_INVALID_INDEX : v;
}
MRD_INL bool is_dynamic_scene(const Env& e, uint32_t b) {
    return b >= e.nlinks && e.topo->motion[b] == MR_MOTION_DYNAMIC;
}

MRD_INL void body_pose(const Env& e, uint32_t b, V3& p, Q4& q) {
    if (b < e.nlinks) {
        p = e.pos[b];
        q = e.rot[b];
    } else {
        const MRBodyStateC& s = e.scene[b - e.nlinks];
        p = f3(s.position);
        q = q4(s.orientation);
    }
}

// Packed failure key: (order << 32) | (code << 24) | index (24 bits).
MRD_INL void report_failure(unsigned long long* slot, uint32_t order, uint32_t code, uint32_t index) {
    const unsigned long long key = ((unsigned long long)order << 32) | ((unsigned long long)(code & 0xffu) << 24) |
        (unsigned long long)(index & 0xffffffu);
    atomicMin(slot, key);
}

// -------------------------------------------------------------- wave ops

// The lane index, opaque to the optimiser from here on. Taken anew at the start of
// every stage, it keeps each stage's addresses and masks out of the others: hoisted
// out of the microstep loop, several hundred of them were live across all stages
// and their reloads from scratch sat inside the sweep loop, where each waits for
// every load in flight.
MRD_INL uint32_t stage_lane(uint32_t lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

MRD_INL uint32_t wave_prefix_sum(uint32_t value, uint32_t lane, uint32_t& total) {
    uint32_t x = value;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, (unsigned)d, 64);
        if (lane >= (uint32_t)d) x += y;
    }
    total = __shfl(x, 63, 64);
    return x - value;
}

// One butterfly step through a DPP lane permutation: x + x[perm(lane)].
template <int kCtrl>
MRD_INL float dpp_fold_step(float x) {
    const int y = __builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, false);
    return x + __int_as_float(y);
}

// Canonical 64-lane pairwise sum x[i] + x[i ^ d] for d = 1, 2, 4, ..., 32.
// d = 1 and 2 are quad permutations; after them every lane of a quad holds
// the same bits (IEEE addition commutes), so the half-row mirror pairs quad 0
// with quad 1 exactly as xor 4 would, and the row mirror then pairs the two
// halves of a row as xor 8. A 16-lane row swap then gives every lane the even
// and the odd row of its row pair (xor 16), and a 32-lane swap the two halves
// (xor 32): the four row sums combine as (r0 + r1) + (r2 + r3).
// Must be called with all 64 lanes active; every lane returns the same value.
MRD_INL float wave_fold(float x) {
    x = dpp_fold_step<0xB1>(x);   // quad_perm [1,0,3,2]: xor 1
    x = dpp_fold_step<0x4E>(x);   // quad_perm [2,3,0,1]: xor 2
    x = dpp_fold_step<0x141>(x);  // row_half_mirror: xor 4 on quad-uniform data
    x = dpp_fold_step<0x140>(x);  // row_mirror: xor 8 on half-row-uniform data
    const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);  // even row + odd row
    const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);  // lower half + upper half
}

// The last three steps of wave_fold (xor 8, 16, 32) on data that repeats every
// eight lanes or less: the row rotation by 8 and the two lane swaps keep the
// position within eight lanes, so up to eight different sums, one per lane of
// every eight, finish in one chain.
MRD_INL float wave_fold_high(float x) {
    x = dpp_fold_step<0x128>(x);  // row_ror:8: xor 8
    const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
    const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

// wave_fold of N values: the first three steps for each of them, interleaved;
// then every lane keeps value lane % P (P = 4 or 8 slots, the last value filling
// the spare ones) and one chain finishes them all. Lane i returns the bits
// wave_fold gives for value min(i % P, N - 1).
template <int N, int P> MRD_INL float wave_fold_packed(float (&x)[N], uint32_t lane) {
    static_assert((P == 4 || P == 8) && N <= P, "a packed fold holds one value per slot");
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = dpp_fold_step<0xB1>(x[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = dpp_fold_step<0x4E>(x[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = dpp_fold_step<0x141>(x[i]);
    const uint32_t slot = lane & (uint32_t)(P - 1);
    float y = x[N - 1];
#pragma unroll
    for (int i = N - 2; i >= 0; --i) y = slot == (uint32_t)i ? x[i] : y;
    return wave_fold_high(y);
}

// The value of lane kLane of each lane's quad.
template <int kLane> MRD_INL float quad_broadcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kLane * 0x55, 0xf, 0xf, true));
}

MRD_INL uint32_t uniform_u32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
// The value of one lane, the same for all, as a scalar.
MRD_INL uint32_t read_lane(uint32_t v, uint32_t lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane); }
MRD_INL float read_lane(float v, uint32_t lane) { return __uint_as_float(read_lane(__float_as_uint(v), lane)); }
MRD_INL V3 read_lane(V3 v, uint32_t lane) { return V3{read_lane(v.x, lane), read_lane(v.y, lane), read_lane(v.z, lane)}; }

// The value of lane `from` (below 64), for every lane's own `from`.
MRD_INL float wave_get(float x, uint32_t from) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute((int)(from << 2), __float_as_int(x)));
}
MRD_INL V3 wave_get(V3 v, uint32_t from) { return V3{wave_get(v.x, from), wave_get(v.y, from), wave_get(v.z, from)}; }
MRD_INL Q4 wave_get(Q4 q, uint32_t from) {
    return Q4{wave_get(q.x, from), wave_get(q.y, from), wave_get(q.z, from), wave_get(q.w, from)};
}

// True on every lane when `bad` holds on any active lane: a uniform branch
// condition for values every lane computes alike.
MRD_INL bool wave_any(bool bad) { return __builtin_amdgcn_ballot_w64(bad) != 0ull; }

// A compile-time flag passed to a generic lambda.
template <bool B> struct BoolTag { static constexpr bool value = B; };

MRD_INL float wave_max(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxd(v, __shfl_xor(v, d, 64));
    return v;
}

MRD_INL uint32_t wave_sum_u32(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

MRD_INL uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const uint32_t o = __shfl_xor(v, d, 64);
        v = v > o ? v : o;
    }
    return v;
}

MRD_INL uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const uint32_t o = __shfl_xor(v, d, 64);
        v = v < o ? v : o;
    }
    return v;
}

// ----------------------------------------------------------------- drives

MRD_INL float effective_armature(const Env& e, uint32_t j) {
    const MRDofC& dof = e.dofs[j];
    float value = dof.drive.z;
    if (e.a->cfg.actuation_mode == MR_ACTUATION_IMPLICIT_POSITION_DRIVE && (dof.flags & MR_DOF_FLAG_DRIVE) != 0u)
        value += e.h * dof.drive.y + e.h * e.h * dof.drive.x;
    return value;
}

// Torque-speed envelope of DoF j at joint velocity vel (MetalWorld.metal:
// 252-269): min(effort limit, stall x efficiency x (1 - speed fraction)). An
// inactive profile executes as no-load speed FLT_MAX, efficiency 1 and stall
// torque = the effort limit, or FLT_MAX without one (MetalWorld.mm:1376-1410).
MRD_INL float actuator_envelope(const MRDofC& dof, const MRActuatorProfileC* act, float vel) {
    constexpr float kFloatMax = 3.40282346638528859812e38f;
    float no_load = kFloatMax, efficiency = 1.0f;
    float stall = ((dof.flags & MR_DOF_FLAG_EFFORT_LIMIT) != 0u && dof.limits.w > 0.0f) ? dof.limits.w : kFloatMax;
    if (act != nullptr && (act->identity[1] & MR_ACTUATOR_PROFILE_ACTIVE) != 0u) {
        no_load = act->motor_and_speed.z;
        efficiency = act->motor_and_speed.w;
        stall = act->transmission_and_envelope.z;
    }
    const float speed_fraction = clampd(fabs_(vel) / fmaxd(no_load, 1.175494351e-38f), 0.0f, 1.0f);
    return fmind(dof.limits.w, stall * efficiency * (1.0f - speed_fraction));
}

// Actuator command of DoF j from the current q / v, clamped to the envelope
// (MetalWorld.metal:184-270 prepare, 280-366 refresh).
MRD_INL float drive_effort(const Env& e, uint32_t j) {
    const MRDofC& dof = e.dofs[j];
    const float command = e.cmd[j];
    const float envelope = actuator_envelope(dof, e.acts != nullptr ? &e.acts[j] : nullptr, e.v[j]);
    if (e.a->cfg.actuation_mode == MR_ACTUATION_EFFORT) return clampd(command, -envelope, envelope);
    float cmd = 0.0f;
    if ((dof.flags & MR_DOF_FLAG_DRIVE) != 0u && dof.q_index != MR_INVALID_INDEX) {
        float target = command;
        if ((dof.flags & MR_DOF_FLAG_POSITION_LIMIT) != 0u) target = clampd(target, dof.limits.x, dof.limits.y);
        const float vel = e.v[j];
        cmd = dof.drive.x * (target - e.q[dof.q_index] - e.h * vel) - dof.drive.y * vel;
        const float dry = dof.drive.w;
        if (dry > 0.0f) {
            if (fabs_(vel) > 1.0e-4f) cmd -= vel > 0.0f ? dry : -dry;
            else cmd -= clampd(cmd, -dry, dry);
        }
        if ((dof.flags & MR_DOF_FLAG_EFFORT_LIMIT) != 0u && dof.limits.w > 0.0f)
            cmd = clampd(cmd, -dof.limits.w, dof.limits.w);
    }
    return clampd(cmd, -envelope, envelope);
}

// ------------------------------------------------------------- kinematics

// Forward kinematics, one lane per link (a tree has at most 48). Only four
// quantities recur along the tree: the orientation, the position, and the two
// velocities. Each is carried level by level in registers, a lane reading its
// parent's value by a lane permutation, and everything else about a link (joint
// sine and cosine, anchors in world axes, motion subspace, bias terms) is
// computed once for all links before or after those chains. The level loops are
// serial latency, so they hold as few instructions as the recurrences allow.
// Measured, one robot's control step: kinematics 177 -> 86 K cycles.
MRD_INL void forward_kinematics(const Env& e, uint32_t lane, unsigned long long* fail) {
    const V3 zero{0.0f, 0.0f, 0.0f};
    const uint32_t n = e.nlinks;
    const bool link = lane < n && lane > 0u;
    Q4 rot{0.0f, 0.0f, 0.0f, 1.0f};
    V3 pos = zero, w = zero, vl = zero;
    if (e.root_type == MR_ROOT_FLOATING) {
        Q4 rq;
        if (!checked_quat(Q4{e.q[3], e.q[4], e.q[5], e.q[6]}, rq)) {
            if (lane == 0u) report_failure(fail, 0u, MR_STEP_NONFINITE_INPUT, 3u);
            rq = Q4{0.0f, 0.0f, 0.0f, 1.0f};
        }
        rot = rq;
        pos = V3{e.q[0], e.q[1], e.q[2]};
        vl = V3{e.v[0], e.v[1], e.v[2]};
        w = V3{e.v[3], e.v[4], e.v[5]};
    }
    // lanes without a parent follow link 0 and are not written
    const uint32_t self = link ? lane : 0u;
    const mr::LinkConst lc = e.lconst[self];
    const uint32_t parent = link ? e.topo->parent[lane] : 0u;
    const uint32_t depth = link ? e.topo->depth[lane] : 0u;
    const uint32_t jt = e.topo->jtype[self];
    const bool moving = link && (jt == MR_JOINT_REVOLUTE || jt == MR_JOINT_CONTINUOUS);
    const Q4 prot{lc.prot[0], lc.prot[1], lc.prot[2], lc.prot[3]};
    const Q4 crot{lc.crot_conj[0], lc.crot_conj[1], lc.crot_conj[2], lc.crot_conj[3]};
    const V3 axis_n{lc.axis[0], lc.axis[1], lc.axis[2]};
    float qd = 0.0f;
    Q4 motion{0.0f, 0.0f, 0.0f, 1.0f};
    if (moving) {
        qd = e.v[e.topo->vidx[lane]];
        motion = axis_angle(axis_n, e.q[e.topo->qidx[lane]]);
    }
    bool ok = true;
    for (uint32_t d = 1; d < e.levels; ++d) {
        const Q4 pjr = qmul(wave_get(rot, parent), prot);
        Q4 child;
        const bool good = normalized_quat(qmul(qmul(pjr, motion), crot), child);
        if (depth == d) {
            ok = good;
            if (good) rot = child;
        }
    }
    const Q4 prr = wave_get(rot, parent);
    const Q4 pjr = qmul(prr, prot);
    const V3 axis_w = qrot(pjr, axis_n);
    const V3 parent_anchor = qrot(prr, V3{lc.panchor[0], lc.panchor[1], lc.panchor[2]});
    const V3 child_anchor = qrot(rot, V3{lc.canchor[0], lc.canchor[1], lc.canchor[2]});
    const V3 spin = mul(qd, axis_w);
    for (uint32_t d = 1; d < e.levels; ++d) {
        const V3 np = sub(add(wave_get(pos, parent), parent_anchor), child_anchor);
        const V3 wp = wave_get(w, parent);
        const V3 nw = moving ? add(wp, spin) : wp;
        if (depth == d) {
            pos = np;
            w = nw;
        }
    }
    const V3 pp = wave_get(pos, parent), wp = wave_get(w, parent);
    const V3 p2j = sub(add(pp, parent_anchor), pp);
    const V3 joint_v = cross(wp, p2j), child_v = cross(w, child_anchor);
    for (uint32_t d = 1; d < e.levels; ++d) {
        const V3 nv = sub(add(wave_get(vl, parent), joint_v), child_v);
        if (depth == d) vl = nv;
    }
    const V3 ca = moving ? mul(qd, cross(wp, axis_w)) : zero;
    const V3 cl = sub(sub(cross(wp, joint_v), cross(ca, child_anchor)), cross(w, child_v));
    if (lane < n) {
        e.rot[lane] = rot;
        e.pos[lane] = pos;
        e.w[lane] = w;
        e.vl[lane] = vl;
        e.r[lane] = link ? sub(pos, pp) : zero;
        e.sa[lane] = moving ? axis_w : zero;
        e.sl[lane] = moving ? neg(cross(axis_w, child_anchor)) : zero;
        e.ca[lane] = ca;
        e.cl[lane] = link ? cl : zero;
    }
    if (link && !(ok && finite3(pos) && finite4(rot) && finite3(w) && finite3(vl) && finite3(cl) && finite3(ca)))
        report_failure(fail, 1u + lane, MR_STEP_NONFINITE_RESULT, lane);
}

MRD_INL void world_inertia(const MRBodyC& b, Q4 rot, float out[6]) {
    const V3 c0 = qrot(rot, V3{1.0f, 0.0f, 0.0f});
    const V3 c1 = qrot(rot, V3{0.0f, 1.0f, 0.0f});
    const V3 c2 = qrot(rot, V3{0.0f, 0.0f, 1.0f});
    const float R[3][3] = {{c0.x, c1.x, c2.x}, {c0.y, c1.y, c2.y}, {c0.z, c1.z, c2.z}};
    const float Ib[3][3] = {{b.inertia_row0.x, b.inertia_row0.y, b.inertia_row0.z},
                            {b.inertia_row1.x, b.inertia_row1.y, b.inertia_row1.z},
                            {b.inertia_row2.x, b.inertia_row2.y, b.inertia_row2.z}};
    const int si[6] = {0, 0, 0, 1, 1, 2};
    const int sj[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int rr = si[k], cc = sj[k];
        float acc = 0.0f;
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
            for (int y = 0; y < 3; ++y) acc += R[rr][x] * Ib[x][y] * R[cc][y];
        out[k] = acc;
    }
}

MRD_INL void world_inverse_inertia(const MRBodyC& b, Q4 rot, MRBodyStateC& s) {
    const V3 c0 = qrot(rot, V3{1.0f, 0.0f, 0.0f});
    const V3 c1 = qrot(rot, V3{0.0f, 1.0f, 0.0f});
    const V3 c2 = qrot(rot, V3{0.0f, 0.0f, 1.0f});
    const float R[3][3] = {{c0.x, c1.x, c2.x}, {c0.y, c1.y, c2.y}, {c0.z, c1.z, c2.z}};
    const float Ib[3][3] = {{b.inverse_inertia_row0.x, b.inverse_inertia_row0.y, b.inverse_inertia_row0.z},
                            {b.inverse_inertia_row1.x, b.inverse_inertia_row1.y, b.inverse_inertia_row1.z},
                            {b.inverse_inertia_row2.x, b.inverse_inertia_row2.y, b.inverse_inertia_row2.z}};
    float o[3][3];
#pragma unroll
    for (int rr = 0; rr < 3; ++rr)
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
            float acc = 0.0f;
#pragma unroll
            for (int x = 0; x < 3; ++x)
#pragma unroll
                for (int y = 0; y < 3; ++y) acc += R[rr][x] * Ib[x][y] * R[cc][y];
            o[rr][cc] = acc;
        }
    s.inverse_inertia_world_row0 = mr_float4{o[0][0], o[0][1], o[0][2], 0.0f};
    s.inverse_inertia_world_row1 = mr_float4{o[1][0], o[1][1], o[1][2], 0.0f};
    s.inverse_inertia_world_row2 = mr_float4{o[2][0], o[2][1], o[2][2], 0.0f};
}

// ABA initialisation of one link: rigid inertia and bias force; a floating
// root also takes its DoFs' armature and efforts.
MRD_INL void aba_init_link(const Env& e, uint32_t i) {
    const MRBodyC& b = e.bodies[i];
    float A[6];
    world_inertia(b, e.rot[i], A);
    const float m = b.mass.x;
    const V3 wi = e.w[i];
    V3 bt = cross(wi, sym_mul(A, wi));
    V3 bf = neg(mul(m, e.gravity));
    if (e.a->cfg.apply_body_damping != 0u) {
        bt = add(bt, mul(b.damping.y, wi));
        bf = add(bf, mul(b.damping.x, e.vl[i]));
    }
    V3 C{m, m, m};
    if (i == 0u && e.root_type == MR_ROOT_FLOATING) {
        C = V3{m + e.arm[0], m + e.arm[1], m + e.arm[2]};
        A[0] += e.arm[3];
        A[3] += e.arm[4];
        A[5] += e.arm[5];
        bt = sub(bt, V3{e.effort[3], e.effort[4], e.effort[5]});
        bf = sub(bf, V3{e.effort[0], e.effort[1], e.effort[2]});
    }
    float* M = e.I + 36u * i;
    const float cols[36] = {A[0], A[1], A[2], 0.0f, 0.0f, 0.0f, A[1], A[3], A[4], 0.0f, 0.0f, 0.0f,
                            A[2], A[4], A[5], 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, C.x,  0.0f, 0.0f,
                            0.0f, 0.0f, 0.0f, 0.0f, C.y,  0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, C.z};
#pragma unroll
    for (int k = 0; k < 36; ++k) M[k] = cols[k];
    float* p = e.p + 6u * i;
    p[0] = bt.x; p[1] = bt.y; p[2] = bt.z;
    p[3] = bf.x; p[4] = bf.y; p[5] = bf.z;
}

// Column j of link i's articulated inertia and component j of its bias: its own
// plus what its children (all finished) passed on, in decreasing child index.
MRD_INL void aba_gather_column(const Env& e, uint32_t i, uint32_t j, float (&c)[6], float& p) {
    const float* own = e.I + 36u * i + 6u * j;
#pragma unroll
    for (int k = 0; k < 6; ++k) c[k] = own[k];
    p = e.p[6u * i + j];
    unsigned long long kids = e.topo->children[i];
    while (kids != 0ull) {
        const uint32_t ch = 63u - (uint32_t)__builtin_clzll(kids);  // decreasing index
        kids &= ~(1ull << ch);
        const float* in = e.I + 36u * ch + 6u * j;
#pragma unroll
        for (int k = 0; k < 6; ++k) c[k] += in[k];
        p += e.p[6u * ch + j];
    }
}

// One level of the inward pass: every link of `links` (a lane mask) is projected
// on its joint and shifted to its parent, in place. A level holds few links (one
// to five of a humanoid's 30), so sixteen lanes share a link instead of one lane
// working through its 6x6 matrix: lanes 0-2 of the sixteen own its angular
// columns and lanes 4-6 its linear ones (lanes 3 and 7 repeat a neighbour, lanes
// 8-15 repeat 0-7), so that a three-component dot product is a sum within a quad
// and the two halves meet through a half-row mirror. Lane 0-14 then each shift
// one element of the two changed blocks. Every element keeps the expression and
// the order of the scalar form.
// Measured, one robot's control step: ABA 350 -> 186 K cycles (with the outward
// pass in registers); the step 692 -> 585 us.
MRD_INL void aba_inward_level(const Env& e, uint32_t lane, unsigned long long links, float& min_piv, float& max_piv,
                              unsigned long long* fail) {
    const uint32_t t = lane & 15u, group = lane >> 4;
    const uint32_t m = (t & 3u) < 2u ? (t & 3u) : 2u;   // component within the half
    const bool linear = (t & 4u) != 0u;
    const uint32_t j = linear ? 3u + m : m;
    while (links != 0ull) {
        // group g takes the g-th link of the mask; spare groups repeat the first
        unsigned long long mine = links, rest = links;
#pragma unroll
        for (uint32_t g = 0; g < 4u; ++g) {
            if (group == g) mine = rest;
            rest &= rest - 1ull;
        }
        const bool active = mine != 0ull;
        const uint32_t i = (uint32_t)__builtin_ctzll(active ? mine : links);
        links = rest;
        const uint32_t vi = e.topo->vidx[i];
        const bool has = vi != 0xffu;
        float c[6], p;
        aba_gather_column(e, i, j, c, p);
        const V3 sa = e.sa[i], sl = e.sl[i], ca = e.ca[i], cl = e.cl[i];
        const float arm = has ? e.arm[vi] : 0.0f, effort = has ? e.effort[vi] : 0.0f;
        p += (c[0] * ca.x + c[1] * ca.y + c[2] * ca.z) + (c[3] * cl.x + c[4] * cl.y + c[5] * cl.z);
        const float U = (c[0] * sa.x + c[1] * sa.y + c[2] * sa.z) + (c[3] * sl.x + c[4] * sl.y + c[5] * sl.z);
        // S_j: this column's component of the motion subspace
        const V3 s3 = linear ? sl : sa;
        const float S = m == 0u ? s3.x : (m == 1u ? s3.y : s3.z);
        const auto mirror = [](float x) {
            return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, true));
        };
        const auto dot_half = [](float x) { return (quad_broadcast<0>(x) + quad_broadcast<1>(x)) + quad_broadcast<2>(x); };
        const float du = dot_half(S * U), dp = dot_half(S * p);
        const float D = (du + mirror(du)) + arm;
        const float dp_other = mirror(dp);
        const float u = (effort - (linear ? dp_other : dp)) - (linear ? dp : dp_other);
        float big = fmaxd(fmaxd(fabs_(c[0]), fabs_(c[1])), fabs_(c[2]));
        big = fmaxd(fmaxd(big, fabs_(c[3])), fmaxd(fabs_(c[4]), fabs_(c[5])));
        big = fmaxd(fmaxd(quad_broadcast<0>(big), quad_broadcast<1>(big)), quad_broadcast<2>(big));
        big = fmaxd(big, mirror(big));
        const float floor_ = fmaxd(kAbsolutePivotFloor, big * 6.0f * kFloatEps);
        if (t == 0u && active && has) {
            if (!(D > floor_) || !isfin(D))
                report_failure(fail, 0xffffu - i, MR_STEP_FACTORIZATION_FAILED, vi);
            const float piv = sqrt_rn(D);
            if (piv >= 0.0f) {
                min_piv = fmind(min_piv, piv);
                max_piv = fmaxd(max_piv, piv);
            }
        }
        // every lane gets U's six components: its own half's by broadcasts, the
        // other half's mirrored (component k sits at position 3 - k there)
        const float V = mirror(U);
        const float own[3] = {quad_broadcast<0>(U), quad_broadcast<1>(U), quad_broadcast<2>(U)};
        const float oth[3] = {quad_broadcast<3>(V), quad_broadcast<2>(V), quad_broadcast<1>(V)};
        if (has) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                c[k] -= ((linear ? oth[k] : own[k]) * U) / D;
                c[3 + k] -= ((linear ? own[k] : oth[k]) * U) / D;
            }
            p += (u / D) * U;
        }
        __syncthreads();
        if (active && t < 7u && t != 3u) {
            float* col = e.I + 36u * i + 6u * j;
#pragma unroll
            for (int k = 0; k < 6; ++k) col[k] = c[k];
            e.p[6u * i + j] = p;
            if (has) {
                reinterpret_cast<float*>(linear ? e.Ub + i : e.Ut + i)[m] = U;
                if (t == 0u) {
                    e.D[i] = D;
                    e.u[i] = u;
                }
            }
        }
        __syncthreads();
        // Shift by r to the parent: A' = A - (Q + Q^T) - P and B' = B + T with
        // T = r~ C, Q row i = B row i x r, P row i = T row i x r; C stays.
        const float* M = e.I + 36u * i;
        const float* rv = reinterpret_cast<const float*>(e.r + i);
        const auto B = [&](uint32_t x, uint32_t y) { return M[6u * x + 3u + y]; };
        const auto C = [&](uint32_t x, uint32_t y) { return M[6u * (3u + x) + 3u + y]; };
        const auto next = [](uint32_t x) { return x == 2u ? 0u : x + 1u; };
        const auto T = [&](uint32_t x, uint32_t y) {
            const uint32_t x1 = next(x), x2 = next(x1);
            return rv[x1] * C(x2, y) - rv[x2] * C(x1, y);
        };
        const auto Q = [&](uint32_t x, uint32_t y) {
            const uint32_t y1 = next(y), y2 = next(y1);
            return B(x, y1) * rv[y2] - B(x, y2) * rv[y1];
        };
        float value = 0.0f, bias = 0.0f;
        uint32_t x = 0u, y = 0u;
        if (t < 6u) {
            x = t < 3u ? 0u : (t < 5u ? 1u : 2u);
            y = t < 3u ? t : (t < 5u ? t - 2u : 2u);
            const uint32_t y1 = next(y), y2 = next(y1);
            const float P = T(x, y1) * rv[y2] - T(x, y2) * rv[y1];
            value = M[6u * y + x] - (Q(x, y) + Q(y, x)) - P;
        } else if (t < 15u) {
            x = (t - 6u) / 3u;
            y = (t - 6u) % 3u;
            value = B(x, y) + T(x, y);
            if (t < 9u) {
                // lanes 6-8 also shift the bias: pt' = pt + r x pb
                const float* pv = e.p + 6u * i;
                const uint32_t k = t - 6u, k1 = next(k), k2 = next(k1);
                bias = pv[k] + (rv[k1] * pv[3u + k2] - rv[k2] * pv[3u + k1]);
            }
        }
        __syncthreads();
        if (active && t < 15u) {
            float* W = e.I + 36u * i;
            if (t < 6u) {
                W[6u * y + x] = value;
                W[6u * x + y] = value;
            } else {
                W[6u * x + 3u + y] = value;
                W[6u * (3u + y) + x] = value;
                if (t < 9u) e.p[6u * i + (t - 6u)] = bias;
            }
        }
        __syncthreads();
    }
}

// Cholesky factor of the floating root's articulated inertia M (column-major,
// symmetric) into L (row-major), held in registers throughout.
MRD_INL bool root_factor(const float* M, float* Lout, float& minp, float& maxp, uint32_t& fail_row) {
    float m[6][6], L[6][6];
    float big = 0.0f;
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int c = 0; c <= r; ++c) {
            m[r][c] = M[6 * c + r];
            big = fmaxd(big, fabs_(m[r][c]));
        }
    const float floor_ = fmaxd(kAbsolutePivotFloor, big * 6.0f * kFloatEps);
    bool ok = true;
#pragma unroll
    for (int row = 0; row < 6; ++row) {
#pragma unroll
        for (int col = 0; col <= row; ++col) {
            float val = m[row][col];
#pragma unroll
            for (int k = 0; k < col; ++k) val -= L[row][k] * L[col][k];
            if (row == col) {
                if (ok && (!(val > floor_) || !isfin(val))) {
                    ok = false;
                    fail_row = (uint32_t)row;
                }
                L[row][col] = sqrt_rn(val);
                minp = fmind(minp, L[row][col]);
                maxp = fmaxd(maxp, L[row][col]);
            } else {
                L[row][col] = val / L[col][col];
            }
            Lout[row * 6 + col] = L[row][col];
        }
    }
    return ok;
}

MRD_INL void root_solve(const float* L, const float rhs[6], float x[6]) {
    float y[6];
    for (int row = 0; row < 6; ++row) {
        float val = rhs[row];
        for (int col = 0; col < row; ++col) val -= L[row * 6 + col] * y[col];
        y[row] = val / L[row * 6 + row];
    }
    for (int row = 5; row >= 0; --row) {
        float val = y[row];
        for (int col = row + 1; col < 6; ++col) val -= L[col * 6 + row] * x[col];
        x[row] = val / L[row * 6 + row];
    }
}

// Inverse ABA for the point forces of one constraint row on up to two links:
// out[nv] = M_eff^{-1} J^T f, one row per lane.
//
// Inward pass: only links on the root paths of `la` / `lb` carry a bias. Every
// other link's bias and contribution is exactly +0 in every component (the
// accumulators start at +0, +0 - y and x + y never produce -0 from operands
// without -0, and u = (0 - s.t) - s.f is +0 for a +0 bias), so visiting only
// path links in decreasing index order, and adding the at most two pending
// child contributions of a merge link in decreasing child order, reproduces
// the dense pass bit for bit. The joint terms u of path links are pushed on a
// per-lane LDS stack; the outward pass visits all links in increasing index
// order and pops them in reverse.
//
// The outward pass is the same walk for every row, so what it needs of a link
// is wave-uniform: lane i holds link i's constants (ResponseLink) and the walk
// reads them as scalars. A link whose parent was visited just before takes its
// acceleration from registers (most links of a tree numbered depth first);
// others read the LDS slot the topology cache's plan gave the parent. All lanes
// stay active throughout (a lane without a row has no endpoint links and
// stores nothing): scalar reads of a lane need it. Measured with the Jacobian
// rows moved to the evaluation pass, one robot's control step: responses and
// evaluation 284 -> 238 K cycles; 1500 random trees, 2 steps, 5.40 -> 5.13 ms.
struct ResponseLink {
    V3 r, Ut, Ub, sa, sl;
    float D;
    uint32_t plan;  // parent | velocity index << 8 | own slot << 16 | parent's slot << 24 (0xff: none)
};

MRD_INL ResponseLink response_link(const Env& e, uint32_t lane) {
    const mr::TopoCache& T = *e.topo;
    const uint32_t i = lane < e.nlinks ? lane : 0u;
    const uint32_t parent = T.parent[i];
    const uint32_t pslot = parent != 0xffu ? T.slot[parent] : 0xffu;
    return ResponseLink{e.r[i], e.Ut[i], e.Ub[i], e.sa[i], e.sl[i], e.D[i],
                        parent | ((uint32_t)T.vidx[i] << 8) | ((uint32_t)T.slot[i] << 16) | (pslot << 24)};
}

MRD_INL void inverse_aba(const Env& e, uint32_t lane, const ResponseLink& own, bool row, uint32_t la, V3 xa, V3 fa,
                         uint32_t lb, V3 xb, V3 fb, float* out) {
    const mr::TopoCache& T = *e.topo;
    const uint32_t n = e.nlinks;
    const V3 zero{0.0f, 0.0f, 0.0f};
    const unsigned long long path = (la != MR_INVALID_INDEX ? T.anc[la] : 0ull) |
                                    (lb != MR_INVALID_INDEX ? T.anc[lb] : 0ull);
    float* ustack = e.rstack + lane;
    uint32_t sp = 0;
    // pending child contributions: target link, child index, torque, force
    uint32_t tg0 = MR_INVALID_INDEX, ch0 = 0u, tg1 = MR_INVALID_INDEX, ch1 = 0u;
    V3 c0t = zero, c0f = zero, c1t = zero, c1f = zero;
    auto gather = [&](uint32_t i, V3& t, V3& f) {
        t = zero;
        f = zero;
        if (i == la) {
            t = sub(t, cross(sub(xa, e.pos[i]), fa));
            f = sub(f, fa);
        }
        if (i == lb) {
            t = sub(t, cross(sub(xb, e.pos[i]), fb));
            f = sub(f, fb);
        }
        const bool m0 = tg0 == i, m1 = tg1 == i;
        if (m0 && m1) {
            const bool first0 = ch0 > ch1;
            t = add(t, first0 ? c0t : c1t);
            f = add(f, first0 ? c0f : c1f);
            t = add(t, first0 ? c1t : c0t);
            f = add(f, first0 ? c1f : c0f);
        } else if (m0) {
            t = add(t, c0t);
            f = add(f, c0f);
        } else if (m1) {
            t = add(t, c1t);
            f = add(f, c1f);
        }
        if (m0) tg0 = MR_INVALID_INDEX;
        if (m1) tg1 = MR_INVALID_INDEX;
    };
    unsigned long long rest = path;
    while (rest != 0ull) {
        const uint32_t i = 63u - (uint32_t)__builtin_clzll(rest);
        rest &= ~(1ull << i);
        V3 t, f;
        gather(i, t, f);
        if (link_vidx(e, i) != MR_INVALID_INDEX) {
            const float u = (0.0f - dot(e.sa[i], t)) - dot(e.sl[i], f);
            const float uD = u / e.D[i];
            t = add(t, mul(uD, e.Ut[i]));
            f = add(f, mul(uD, e.Ub[i]));
            ustack[sp * 64u] = u;
            ++sp;
        }
        const V3 ct = add(t, cross(e.r[i], f));
        if (tg0 == MR_INVALID_INDEX) {
            tg0 = link_parent(e, i);
            ch0 = i;
            c0t = ct;
            c0f = f;
        } else {
            tg1 = link_parent(e, i);
            ch1 = i;
            c1t = ct;
            c1f = f;
        }
    }
    V3 ap, lp;
    if (e.root_type == MR_ROOT_FLOATING) {
        V3 t0, f0;
        gather(0u, t0, f0);
        const float rhs[6] = {-t0.x, -t0.y, -t0.z, -f0.x, -f0.y, -f0.z};
        float x[6];
        root_solve(e.L, rhs, x);
        ap = V3{x[0], x[1], x[2]};
        lp = V3{x[3], x[4], x[5]};
        if (row) {
            out[0] = x[3]; out[1] = x[4]; out[2] = x[5];
            out[3] = x[0]; out[4] = x[1]; out[5] = x[2];
        }
    } else {
        ap = zero;
        lp = zero;
    }
    const auto slot_store = [&](uint32_t s, V3 a, V3 l) {
        float* p = e.rslot + s * 6u * 64u + lane;
        p[0] = a.x; p[64] = a.y; p[128] = a.z;
        p[192] = l.x; p[256] = l.y; p[320] = l.z;
    };
    const uint32_t root_slot = (read_lane(own.plan, 0u) >> 16) & 0xffu;
    if (root_slot != 0xffu) slot_store(root_slot, ap, lp);
    // the next joint term to pop, read one pop ahead
    float top = sp > 0u ? ustack[(sp - 1u) * 64u] : 0.0f;
    V3 a_prev = ap, l_prev = lp;
    for (uint32_t i = 1; i < n; ++i) {
        const uint32_t plan = read_lane(own.plan, i);
        const uint32_t parent = plan & 0xffu, vi = (plan >> 8) & 0xffu, slot = (plan >> 16) & 0xffu;
        V3 a_par = a_prev, l_par = l_prev;
        if (parent + 1u != i) {
            const float* p = e.rslot + (plan >> 24) * 6u * 64u + lane;
            a_par = V3{p[0], p[64], p[128]};
            l_par = V3{p[192], p[256], p[320]};
        }
        const V3 lpi = add(l_par, cross(a_par, read_lane(own.r, i)));
        V3 ai = a_par, li = lpi;
        if (vi != 0xffu) {
            float uu = 0.0f;
            if (((path >> i) & 1ull) != 0ull) {
                --sp;
                uu = top;
                top = sp > 0u ? ustack[(sp - 1u) * 64u] : 0.0f;
            }
            const float proj = dot(read_lane(own.Ut, i), a_par) + dot(read_lane(own.Ub, i), lpi);
            const float qdd = (uu - proj) / read_lane(own.D, i);
            if (row) out[vi] = qdd;
            ai = add(a_par, mul(qdd, read_lane(own.sa, i)));
            li = add(lpi, mul(qdd, read_lane(own.sl, i)));
        }
        if (slot != 0xffu) slot_store(slot, ai, li);
        a_prev = ai;
        l_prev = li;
    }
}

// One DoF's part in the Jacobian columns of any contact point x on a link it
// moves: a root translation's column is `lin`, a root rotation's ang x (x - at),
// a joint's lin + ang x (x - at).
struct DofColumn {
    V3 lin, ang, at;
    uint32_t owner;  // owning link, 0xff without one
    uint32_t kind;   // 0 root translation, 1 root rotation, 2 joint
};

MRD_INL DofColumn dof_column(const Env& e, uint32_t j) {
    DofColumn d;
    if (e.root_type == MR_ROOT_FLOATING && j < 6u) {
        const uint32_t k = j < 3u ? j : j - 3u;
        const V3 ev{k == 0u ? 1.0f : 0.0f, k == 1u ? 1.0f : 0.0f, k == 2u ? 1.0f : 0.0f};
        d.lin = ev;
        d.ang = ev;
        d.at = e.pos[0];
        d.owner = 0xffu;
        d.kind = j < 3u ? 0u : 1u;
        return d;
    }
    const uint32_t owner = j < e.nv ? e.topo->dof_body[j] : 0xffu;
    const bool has = owner < 64u;
    const uint32_t link = has ? owner : 0u;  // read, not used, without an owner
    d.lin = e.sl[link];
    d.ang = e.sa[link];
    d.at = e.pos[link];
    d.owner = has ? owner : 0xffu;
    d.kind = 2u;
    return d;
}

MRD_INL V3 jacobian_column(const DofColumn& d, unsigned long long anc, V3 x) {
    const V3 turn = cross(d.ang, sub(x, d.at));
    const V3 joint = add(d.lin, turn);
    const bool moves = d.owner != 0xffu && ((anc >> d.owner) & 1ull) != 0ull;
    const V3 zero{0.0f, 0.0f, 0.0f};
    return d.kind == 0u ? d.lin : (d.kind == 1u ? turn : (moves ? joint : zero));
}

// ------------------------------------------------------------ colliders

MRD_INL void inflate_bounds(Collider& c) {
    const V3 scale = add(vmax(vabs(c.lower), vabs(c.upper)), V3{1.0f, 1.0f, 1.0f});
    const V3 pad = mul(MR_COLLISION_AABB_RELATIVE_PAD, scale);
    c.lower = sub(c.lower, pad);
    c.upper = add(c.upper, pad);
}

// Collider of shape s with its body at (bpos, borient). Convex hulls and
// meshes are projected by the kGeo instances only.
template <bool kGeo = false>
MRD_INL bool project_collider_pose(const Env& e, uint32_t s, V3 bpos, Q4 borient, Collider& c) {
    const MRShapeC& sh = e.shapes[s];
    Q4 br, lr;
    if (!checked_quat(borient, br) || !checked_quat(q4(sh.local_rotation), lr)) return false;
    c.type = sh.shape_type;
    c.body = sh.body;
    c.disabled = (sh.flags & MR_SHAPE_FLAG_SIMULATION_DISABLED) != 0u ? 1u : 0u;
    c.rotation = qmul(br, lr);
    c.center = add(bpos, qrot(br, f3(sh.local_position)));
    c.contact_offset = sh.contact_rest_radius.x;
    c.radius = 0.0f;
    c.half_length = 0.0f;
    const V3 zero{0.0f, 0.0f, 0.0f};
    c.half_extents = zero;
    c.p0 = zero;
    c.p1 = zero;
    c.plane_normal = zero;
    c.lower = zero;
    c.upper = zero;
    if (!finite3(c.center) || !finite4(c.rotation)) return false;
    if (c.disabled) return true;
    const float co = c.contact_offset;
    if (sh.shape_type == MR_SHAPE_SPHERE) {
        c.radius = sh.dimensions.x;
        const float ex = c.radius + co;
        c.lower = sub(c.center, V3{ex, ex, ex});
        c.upper = add(c.center, V3{ex, ex, ex});
        inflate_bounds(c);
    } else if (sh.shape_type == MR_SHAPE_CAPSULE) {
        c.radius = sh.dimensions.x;
        c.half_length = sh.dimensions.y;
        const V3 axis = qrot(c.rotation, V3{0.0f, c.half_length, 0.0f});
        c.p0 = sub(c.center, axis);
        c.p1 = add(c.center, axis);
        const float ex = c.radius + co;
        c.lower = sub(vmin(c.p0, c.p1), V3{ex, ex, ex});
        c.upper = add(vmax(c.p0, c.p1), V3{ex, ex, ex});
        inflate_bounds(c);
    } else if (sh.shape_type == MR_SHAPE_BOX) {
        c.half_extents = f3(sh.dimensions);
        const V3 bx = qrot(c.rotation, V3{1.0f, 0.0f, 0.0f});
        const V3 by = qrot(c.rotation, V3{0.0f, 1.0f, 0.0f});
        const V3 bz = qrot(c.rotation, V3{0.0f, 0.0f, 1.0f});
        const V3 ext = add(add(add(mul(c.half_extents.x, vabs(bx)), mul(c.half_extents.y, vabs(by))),
                               mul(c.half_extents.z, vabs(bz))),
                           V3{co, co, co});
        c.lower = sub(c.center, ext);
        c.upper = add(c.center, ext);
        inflate_bounds(c);
    } else if (sh.shape_type == MR_SHAPE_PLANE) {
        c.plane_normal = normalize(qrot(c.rotation, V3{0.0f, 1.0f, 0.0f}));
    } else if (sh.shape_type == MR_SHAPE_HEIGHTFIELD) {
        const MRHeightfieldC& hf = e.a->heightfield;
        c.lower = sub(f3(hf.bounds_lower), V3{co, co, co});
        c.upper = add(f3(hf.bounds_upper), V3{co, co, co});
        inflate_bounds(c);
    } else if (kGeo && (sh.shape_type == MR_SHAPE_CONVEX || sh.shape_type == MR_SHAPE_TRIANGLE_MESH)) {
        // half_extents carries the vertex scale; bounds of the transformed
        // vertices (convex) or of the transformed local bounds (mesh)
        c.half_extents = f3(sh.dimensions);
        const MRGeometryC g = e.a->geometries[sh.geometry];
        const V3 sc = c.half_extents;
        V3 lo{__builtin_inff(), __builtin_inff(), __builtin_inff()};
        V3 hi{-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
        const bool convex = sh.shape_type == MR_SHAPE_CONVEX;
        const uint32_t count = convex ? g.vertex_count : 8u;
        for (uint32_t i = 0; i < count; ++i) {
            V3 l;
            if (convex) {
                const mr_float4 v = e.a->geometry_vertices[g.vertex_offset + i];
                l = V3{v.x, v.y, v.z};
            } else {
                l = V3{(i & 1u) ? g.local_upper.x : g.local_lower.x, (i & 2u) ? g.local_upper.y : g.local_lower.y,
                       (i & 4u) ? g.local_upper.z : g.local_lower.z};
            }
            const V3 w = add(c.center, qrot(c.rotation, V3{sc.x * l.x, sc.y * l.y, sc.z * l.z}));
            lo = vmin(lo, w);
            hi = vmax(hi, w);
        }
        c.lower = sub(lo, V3{co, co, co});
        c.upper = add(hi, V3{co, co, co});
        inflate_bounds(c);
    } else {
        return false;
    }
    return finite3(c.lower) && finite3(c.upper);
}

template <bool kGeo = false>
MRD_INL bool project_collider(const Env& e, uint32_t s, Collider& c) {
    V3 bpos;
    Q4 borient;
    body_pose(e, e.shapes[s].body, bpos, borient);
    return project_collider_pose<kGeo>(e, s, bpos, borient, c);
}

MRD_INL float collider_scale(const Collider& c) {
    return fmaxd(fmaxd(maxabs3(c.center), maxabs3(c.half_extents)),
                 fmaxd(fmaxd(maxabs3(c.p0), maxabs3(c.p1)),
                       fmaxd(fmaxd(fabs_(c.radius), fabs_(c.half_length)),
                             fmaxd(fabs_(c.contact_offset), fmaxd(maxabs3(c.lower), maxabs3(c.upper))))));
}

MRD_INL float pair_query_padding(const Collider& a, const Collider& b) {
    return (fmaxd(collider_scale(a), collider_scale(b)) + 1.0f) * MR_COLLISION_QUERY_RELATIVE_PAD;
}

MRD_INL bool pair_may_overlap(const Collider& a, const Collider& b) {
    if (a.disabled || b.disabled) return false;
    if (a.type != MR_SHAPE_PLANE && b.type != MR_SHAPE_PLANE) {
        return a.lower.x <= b.upper.x && a.lower.y <= b.upper.y && a.lower.z <= b.upper.z &&
            a.upper.x >= b.lower.x && a.upper.y >= b.lower.y && a.upper.z >= b.lower.z;
    }
    const Collider& plane = a.type == MR_SHAPE_PLANE ? a : b;
    const Collider& fin = a.type == MR_SHAPE_PLANE ? b : a;
    const V3 center = mul(0.5f, add(fin.lower, fin.upper));
    const V3 half = mul(0.5f, sub(fin.upper, fin.lower));
    const float scale = fmaxd(fmaxd(maxabs3(plane.center), maxabs3(fin.lower)),
                              fmaxd(maxabs3(fin.upper), fmaxd(fabs_(plane.contact_offset), fabs_(fin.contact_offset))));
    const float pad = (scale + 1.0f) * MR_COLLISION_QUERY_RELATIVE_PAD;
    const float dist = dot(plane.plane_normal, sub(center, plane.center)) - dot(vabs(plane.plane_normal), half);
    return dist <= plane.contact_offset + pad;
}

// ------------------------------------------------------------ narrowphase

MRD_INL RawContact make_contact(V3 n, float sep, V3 pa, V3 pb, uint32_t fa, uint32_t fb) {
    RawContact c;
    c.normal = n;
    c.separation = sep;
    c.point_a = pa;
    c.point_b = pb;
    c.feature_a = fa;
    c.feature_b = fb;
    return c;
}

MRD_INL RawContact swapped(const RawContact& in) {
    RawContact c = in;
    c.normal = neg(in.normal);
    c.point_a = in.point_b;
    c.point_b = in.point_a;
    c.feature_a = in.feature_b;
    c.feature_b = in.feature_a;
    return c;
}

MRD_INL V3 coincident_normal(uint32_t a, uint32_t b) {
    const uint32_t hash = (a * 73856093u) ^ (b * 19349663u);
    V3 r{0.0f, 0.0f, 0.0f};
    setcomp(r, (int)(hash % 3u), (hash & 4u) == 0u ? 1.0f : -1.0f);
    return r;
}

MRD_INL V3 stable_segment_normal(V3 da, V3 db, uint32_t ca, uint32_t cb) {
    const V3 cr = cross(da, db);
    if (dot(cr, cr) > kTiny) return normalize(cr);
    V3 d;
    if (dot(da, da) > kTiny) d = normalize(da);
    else if (dot(db, db) > kTiny) d = normalize(db);
    else return coincident_normal(ca, cb);
    const V3 ad = vabs(d);
    V3 ref;
    if (ad.x <= ad.y && ad.x <= ad.z) ref = V3{1.0f, 0.0f, 0.0f};
    else if (ad.y <= ad.z) ref = V3{0.0f, 1.0f, 0.0f};
    else ref = V3{0.0f, 0.0f, 1.0f};
    V3 res = normalize(cross(d, ref));
    if ((((ca * 73856093u) ^ (cb * 19349663u)) & 4u) != 0u) res = neg(res);
    return res;
}

struct SegPoint {
    V3 point;
    float t;
};

MRD_INL SegPoint closest_on_segment(V3 p, V3 e0, V3 e1) {
    const V3 seg = sub(e1, e0);
    const float l2 = dot(seg, seg);
    if (!(l2 > kTiny)) return SegPoint{e0, 0.0f};
    const float t = clampd(dot(sub(p, e0), seg) / l2, 0.0f, 1.0f);
    return SegPoint{add(e0, mul(t, seg)), t};
}

struct SegPair {
    V3 pa, pb;
    float ta, tb;
};

MRD_INL SegPair closest_segments(V3 a0, V3 a1, V3 b0, V3 b1) {
    const V3 da = sub(a1, a0), db = sub(b1, b0), off = sub(a0, b0);
    const float sa = dot(da, da), sb = dot(db, db);
    const float pa = dot(da, off), pb = dot(db, off);
    float ta = 0.0f, tb = 0.0f;
    if (!(sa > kTiny) && !(sb > kTiny)) return SegPair{a0, b0, 0.0f, 0.0f};
    if (!(sa > kTiny)) {
        tb = clampd(pb / sb, 0.0f, 1.0f);
    } else {
        const float cp = dot(da, db);
        if (!(sb > kTiny)) {
            ta = clampd(-pa / sa, 0.0f, 1.0f);
        } else {
            const float den = sa * sb - cp * cp;
            if (den > kTiny * sa * sb) ta = clampd((cp * pb - pa * sb) / den, 0.0f, 1.0f);
            tb = (cp * ta + pb) / sb;
            if (tb < 0.0f) {
                tb = 0.0f;
                ta = clampd(-pa / sa, 0.0f, 1.0f);
            } else if (tb > 1.0f) {
                tb = 1.0f;
                ta = clampd((cp - pa) / sa, 0.0f, 1.0f);
            }
        }
    }
    return SegPair{add(a0, mul(ta, da)), add(b0, mul(tb, db)), ta, tb};
}

MRD_INL uint32_t capsule_feature(float t) {
    if (t <= 0.0f) return 0u;
    return t >= 1.0f ? 1u : 2u;
}

MRD_INL uint32_t box_region(float c, float h) {
    if (c < -h) return 0u;
    return c > h ? 2u : 1u;
}

MRD_INL void sphere_box(const Collider& sphere, const Collider& box, V3& normal, V3& box_point, float& sep,
                        uint32_t& feature) {
    const V3 lc = qrot_inv(box.rotation, sub(sphere.center, box.center));
    const V3 he = box.half_extents;
    V3 closest{clampd(lc.x, -he.x, he.x), clampd(lc.y, -he.y, he.y), clampd(lc.z, -he.z, he.z)};
    const V3 ld = sub(closest, lc);
    const float dist = length(ld);
    if (dist > kTiny) {
        normal = qrot(box.rotation, mul(1.0f / dist, ld));
        sep = dist - sphere.radius;
        feature = box_region(lc.x, he.x) + 3u * box_region(lc.y, he.y) + 9u * box_region(lc.z, he.z);
    } else {
        const V3 d = sub(he, vabs(lc));
        int axis = 0;
        if (d.y < comp(d, axis)) axis = 1;
        if (d.z < comp(d, axis)) axis = 2;
        const float sign = comp(lc, axis) >= 0.0f ? 1.0f : -1.0f;
        V3 outward{0.0f, 0.0f, 0.0f};
        setcomp(outward, axis, sign);
        setcomp(closest, axis, sign * comp(he, axis));
        normal = qrot(box.rotation, neg(outward));
        sep = -comp(d, axis) - sphere.radius;
        feature = 27u + 2u * (uint32_t)axis + (sign > 0.0f ? 1u : 0u);
    }
    box_point = add(box.center, qrot(box.rotation, closest));
}

MRD_INL void consider_capsule_box(V3 seg_point, V3 box_point, float t, uint32_t feat, float& best_sq, V3& best_seg,
                                  V3& best_box, float& best_t, uint32_t& best_feat) {
    const V3 d = sub(box_point, seg_point);
    const float sq = dot(d, d);
    const float tol = 1.0e-12f * (1.0f + fmaxd(best_sq, sq));
    if (!isfin(best_sq) || sq < best_sq - tol || (fabs_(sq - best_sq) <= tol && feat < best_feat)) {
        best_sq = sq;
        best_seg = seg_point;
        best_box = box_point;
        best_t = t;
        best_feat = feat;
    }
}

MRD_INL void capsule_box(const Collider& cap, const Collider& box, uint32_t cap_index, uint32_t box_index,
                         V3& normal, V3& cap_point, V3& box_point, float& sep, float& t_out, uint32_t& feature) {
    const V3 s0 = qrot_inv(box.rotation, sub(cap.p0, box.center));
    const V3 s1 = qrot_inv(box.rotation, sub(cap.p1, box.center));
    const V3 dir = sub(s1, s0);
    const V3 he = box.half_extents;
    float enter = 0.0f, exit_ = 1.0f;
    bool inter = true;
    for (int axis = 0; axis < 3; ++axis) {
        const float da = comp(dir, axis), sa = comp(s0, axis), ha = comp(he, axis);
        if (fabs_(da) <= kTiny) {
            if (sa < -ha || sa > ha) inter = false;
            continue;
        }
        float first = (-ha - sa) / da;
        float second = (ha - sa) / da;
        if (first > second) {
            const float tmp = first;
            first = second;
            second = tmp;
        }
        enter = fmaxd(enter, first);
        exit_ = fmind(exit_, second);
        if (enter > exit_) inter = false;
    }
    if (inter) {
        t_out = clampd(0.5f * (enter + exit_), 0.0f, 1.0f);
        const V3 core = add(s0, mul(t_out, dir));
        const V3 d = sub(he, vabs(core));
        int axis = 0;
        if (d.y < d.x) axis = 1;
        if (d.z < comp(d, axis)) axis = 2;
        const float sign = comp(core, axis) >= 0.0f ? 1.0f : -1.0f;
        V3 outward{0.0f, 0.0f, 0.0f};
        setcomp(outward, axis, sign);
        V3 bp = core;
        setcomp(bp, axis, sign * comp(he, axis));
        const V3 ln = neg(outward);
        normal = qrot(box.rotation, ln);
        cap_point = add(box.center, qrot(box.rotation, add(core, mul(cap.radius, ln))));
        box_point = add(box.center, qrot(box.rotation, bp));
        sep = -comp(d, axis) - cap.radius;
        feature = 27u + 2u * (uint32_t)axis + (sign > 0.0f ? 1u : 0u);
        return;
    }
    float best_sq = __builtin_inff();
    V3 best_seg{0.0f, 0.0f, 0.0f}, best_box{0.0f, 0.0f, 0.0f};
    float best_t = 0.0f;
    uint32_t best_feat = 0xffffffffu;
    for (uint32_t en = 0; en < 2u; ++en) {
        const V3 sp = en == 0u ? s0 : s1;
        const V3 bp{clampd(sp.x, -he.x, he.x), clampd(sp.y, -he.y, he.y), clampd(sp.z, -he.z, he.z)};
        consider_capsule_box(sp, bp, (float)en, en, best_sq, best_seg, best_box, best_t, best_feat);
    }
    uint32_t edge_feature = 2u;
    for (int va = 0; va < 3; ++va) {
        const int f0 = (va + 1) % 3, f1 = (va + 2) % 3;
        for (uint32_t signs = 0; signs < 4u; ++signs) {
            V3 e0{0.0f, 0.0f, 0.0f}, e1{0.0f, 0.0f, 0.0f};
            setcomp(e0, va, -comp(he, va));
            setcomp(e1, va, comp(he, va));
            const float sg0 = (signs & 1u) == 0u ? -1.0f : 1.0f;
            const float sg1 = (signs & 2u) == 0u ? -1.0f : 1.0f;
            setcomp(e0, f0, sg0 * comp(he, f0));
            setcomp(e1, f0, comp(e0, f0));
            setcomp(e0, f1, sg1 * comp(he, f1));
            setcomp(e1, f1, comp(e0, f1));
            const SegPair cl = closest_segments(s0, s1, e0, e1);
            consider_capsule_box(cl.pa, cl.pb, cl.ta, edge_feature, best_sq, best_seg, best_box, best_t, best_feat);
            ++edge_feature;
        }
    }
    const float dist = sqrt_rn(fmaxd(best_sq, 0.0f));
    const V3 ln = dist > kTiny ? mul(1.0f / dist, sub(best_box, best_seg))
                               : qrot_inv(box.rotation, coincident_normal(cap_index, box_index));
    normal = qrot(box.rotation, ln);
    cap_point = add(box.center, qrot(box.rotation, add(best_seg, mul(cap.radius, ln))));
    box_point = add(box.center, qrot(box.rotation, best_box));
    sep = dist - cap.radius;
    t_out = best_t;
    feature = 64u + best_feat;
}

MRD_INL V3 box_axis(const Collider& box, int axis) {
    V3 l{0.0f, 0.0f, 0.0f};
    setcomp(l, axis, 1.0f);
    return qrot(box.rotation, l);
}

MRD_INL float box_projection_radius(const Collider& box, V3 axis) {
    return fabs_(dot(axis, box_axis(box, 0))) * box.half_extents.x +
        fabs_(dot(axis, box_axis(box, 1))) * box.half_extents.y +
        fabs_(dot(axis, box_axis(box, 2))) * box.half_extents.z;
}

MRD_INL V3 box_vertex(const Collider& box, uint32_t v) {
    const V3 he = box.half_extents;
    const V3 l{(v & 1u) == 0u ? -he.x : he.x, (v & 2u) == 0u ? -he.y : he.y, (v & 4u) == 0u ? -he.z : he.z};
    return add(box.center, qrot(box.rotation, l));
}

MRD_INL bool point_in_inflated_box(V3 p, const Collider& box, float infl) {
    const V3 l = vabs(qrot_inv(box.rotation, sub(p, box.center)));
    return l.x <= box.half_extents.x + infl && l.y <= box.half_extents.y + infl && l.z <= box.half_extents.z + infl;
}

MRD_INL V3 box_support(const Collider& box, V3 d) {
    V3 res = box.center;
    for (int axis = 0; axis < 3; ++axis) {
        const V3 basis = box_axis(box, axis);
        const float he = comp(box.half_extents, axis);
        res = add(res, mul(dot(d, basis) >= 0.0f ? he : -he, basis));
    }
    return res;
}

MRD_INL void append(RawBatch& out, const RawContact& c) {
    if (out.count < MR_RAW_CONTACTS_PER_PAIR) out.c[out.count++] = c;
}

MRD_INL void append(ContactSink& out, const RawContact& c) {
    if (out.count >= MR_RAW_CONTACTS_PER_PAIR) return;
    float* p = out.points + 8u * out.count;
    p[0] = c.point_a.x; p[1] = c.point_a.y; p[2] = c.point_a.z;
    p[3] = c.point_b.x; p[4] = c.point_b.y; p[5] = c.point_b.z;
    p[6] = __uint_as_float(c.feature_a);
    p[7] = __uint_as_float(c.feature_b);
    out.head[out.count] = c.separation;
    if (out.count == 0u || c.separation < out.deepest ||
        (c.separation == out.deepest &&
         (c.feature_a < out.deepest_a || (c.feature_a == out.deepest_a && c.feature_b < out.deepest_b)))) {
        out.deepest = c.separation;
        out.deepest_a = c.feature_a;
        out.deepest_b = c.feature_b;
        out.normal = c.normal;
    }
    out.penetration = fmaxd(out.penetration, fmaxd(out.rest - c.separation, 0.0f));
    out.bad = out.bad || !finite3(c.normal) || !isfin(c.separation) || !finite3(c.point_a) || !finite3(c.point_b);
    ++out.count;
}

template <class Out>
MRD_INL void box_box(uint32_t ia, uint32_t ib, const Collider& A, const Collider& B, float accepted, Out& out) {
    // the six face axes, made once; a loop picks them by selects, so that no
    // array with a dynamic index (scratch memory) holds them or the candidates
    const V3 a0 = box_axis(A, 0), a1 = box_axis(A, 1), a2 = box_axis(A, 2);
    const V3 b0 = box_axis(B, 0), b1 = box_axis(B, 1), b2 = box_axis(B, 2);
    const auto pick = [](uint32_t i, V3 x, V3 y, V3 z) { return i == 0u ? x : (i == 1u ? y : z); };
    const auto radius = [](V3 axis, V3 x, V3 y, V3 z, V3 he) {
        return fabs_(dot(axis, x)) * he.x + fabs_(dot(axis, y)) * he.y + fabs_(dot(axis, z)) * he.z;
    };
    const V3 delta = sub(B.center, A.center);
    float best_sep = -__builtin_inff();
    V3 best_n = coincident_normal(ia, ib);
    uint32_t best_axis = 0, k = 0;
#pragma unroll 1
    for (uint32_t i = 0; i < 15u; ++i) {
        V3 axis;
        if (i < 6u) {
            axis = i < 3u ? pick(i, a0, a1, a2) : pick(i - 3u, b0, b1, b2);
        } else {
            const uint32_t x = (i - 6u) / 3u, y = (i - 6u) % 3u;
            const V3 cr = cross(pick(x, a0, a1, a2), pick(y, b0, b1, b2));
            const float sq = dot(cr, cr);
            if (!(sq > 1.0e-12f)) continue;
            axis = mul(1.0f / sqrt_rn(sq), cr);
        }
        const float proj = dot(delta, axis);
        if (proj < 0.0f || (proj == 0.0f && dot(axis, best_n) < 0.0f)) axis = neg(axis);
        const float sep = fabs_(proj) - radius(axis, a0, a1, a2, A.half_extents) - radius(axis, b0, b1, b2, B.half_extents);
        if (sep > accepted) return;
        const float tie = 1.0e-7f * (1.0f + fmaxd(fabs_(best_sep), fabs_(sep)));
        if (!isfin(best_sep) || sep > best_sep + tie || (fabs_(sep - best_sep) <= tie && k < best_axis)) {
            best_sep = sep;
            best_n = axis;
            best_axis = k;
        }
        ++k;
    }
    const float ra = radius(best_n, a0, a1, a2, A.half_extents);
    const float rb = radius(best_n, b0, b1, b2, B.half_extents);
    const float near_b = dot(B.center, best_n) - rb;
    const float far_a = dot(A.center, best_n) + ra;
    for (uint32_t vi = 0; vi < 8u; ++vi) {
        const V3 pa = box_vertex(A, vi);
        if (!point_in_inflated_box(pa, B, accepted)) continue;
        const float sep = near_b - dot(pa, best_n);
        if (sep <= accepted)
            append(out, make_contact(best_n, sep, pa, add(pa, mul(sep, best_n)), feature_key(MR_SHAPE_BOX, vi),
                                     feature_key(MR_SHAPE_BOX, 128u + best_axis)));
    }
    for (uint32_t vi = 0; vi < 8u; ++vi) {
        const V3 pb = box_vertex(B, vi);
        if (!point_in_inflated_box(pb, A, accepted)) continue;
        const float sep = dot(pb, best_n) - far_a;
        if (sep <= accepted)
            append(out, make_contact(best_n, sep, sub(pb, mul(sep, best_n)), pb,
                                     feature_key(MR_SHAPE_BOX, 128u + best_axis), feature_key(MR_SHAPE_BOX, vi)));
    }
    if (out.count == 0u) {
        const V3 pa = box_support(A, best_n);
        const V3 pb = box_support(B, neg(best_n));
        append(out, make_contact(best_n, dot(sub(pb, pa), best_n), pa, pb, feature_key(MR_SHAPE_BOX, 256u + best_axis),
                                 feature_key(MR_SHAPE_BOX, 256u + best_axis)));
    }
}

template <class Out>
MRD_INL void append_surface_contact(Out& out, bool surface_is_a, V3 n, V3 finite_point, float sep,
                                    uint32_t finite_feature, uint32_t surface_feature) {
    const V3 sp = sub(finite_point, mul(sep, n));
    RawContact c = make_contact(neg(n), sep, finite_point, sp, finite_feature, surface_feature);
    if (surface_is_a) c = swapped(c);
    append(out, c);
}

// One query point of a finite shape against the heightfield: the triangle
// under x, its unit normal n, the signed distance d of the shape surface
// (x minus rho along n) and that surface point. d is NaN when x lies outside
// the representable grid, so no threshold accepts it.
MRD_INL mr::HfHit heightfield_query(const Env& e, V3 x, float rho) {
    mr::HfHit h;
    h.d = __builtin_nanf("");
    const MRHeightfieldC& hf = e.a->heightfield;
    const float s = hf.origin_spacing.z;
    const float fx = (x.x - hf.origin_spacing.x) / s;
    const float fy = (x.y - hf.origin_spacing.y) / s;
    if (!isfin(fx) || !isfin(fy)) return h;
    const int ix = (int)__builtin_floorf(clampd(fx, 0.0f, (float)(hf.nx - 2u)));
    const int iy = (int)__builtin_floorf(clampd(fy, 0.0f, (float)(hf.ny - 2u)));
    const float tx = fx - (float)ix;
    const float ty = fy - (float)iy;
    const uint32_t nx = hf.nx;
    const float* H = e.a->heights;
    const float h00 = H[(uint32_t)iy * nx + (uint32_t)ix];
    const float h10 = H[(uint32_t)iy * nx + (uint32_t)ix + 1u];
    const float h01 = H[((uint32_t)iy + 1u) * nx + (uint32_t)ix];
    const float h11 = H[((uint32_t)iy + 1u) * nx + (uint32_t)ix + 1u];
    const V3 v00{hf.origin_spacing.x + (float)ix * s, hf.origin_spacing.y + (float)iy * s, h00};
    const uint32_t tri = tx >= ty ? 0u : 1u;
    V3 e1, e2;
    if (tri == 0u) {
        e1 = V3{s, 0.0f, h10 - h00};
        e2 = V3{s, s, h11 - h00};
    } else {
        e1 = V3{s, s, h11 - h00};
        e2 = V3{0.0f, s, h01 - h00};
    }
    const V3 n = normalize(cross(e1, e2));
    const float d = dot(n, sub(x, v00)) - rho;
    const V3 p = sub(x, mul(rho, n));
    const uint32_t cell = (uint32_t)iy * (nx - 1u) + (uint32_t)ix;
    h.n[0] = n.x; h.n[1] = n.y; h.n[2] = n.z;
    h.d = d;
    h.p[0] = p.x; h.p[1] = p.y; h.p[2] = p.z;
    h.feature = feature_key(MR_SHAPE_HEIGHTFIELD, 2u * cell + tri);
    return h;
}

// Query points of a finite shape against the heightfield (Collision.metal
// meshContacts on a heightfield): a sphere's center; a capsule's two segment
// ends and its center; a box's eight vertices.
MRD_INL uint32_t hf_query_count(uint32_t type) {
    return type == MR_SHAPE_SPHERE ? 1u : type == MR_SHAPE_CAPSULE ? 3u : type == MR_SHAPE_BOX ? 8u : 0u;
}

MRD_INL V3 hf_query_point(const Collider& fs, uint32_t q) {
    if (fs.type == MR_SHAPE_CAPSULE) return q == 0u ? fs.p0 : q == 1u ? fs.p1 : fs.center;
    if (fs.type == MR_SHAPE_BOX) return box_vertex(fs, q);
    return fs.center;
}

MRD_INL float hf_query_radius(const Collider& fs) { return fs.type == MR_SHAPE_BOX ? 0.0f : fs.radius; }

// ------------------------------------------- convex hulls and triangle meshes
//
// Shapes with a support-mapped core (a point set plus a radius): sphere
// (centre), capsule (segment ends), box (8 vertices), convex hull (its
// vertices, scaled) and a mesh triangle (3 vertices). Separated cores get
// GJK's distance and witness points (Voronoi-region simplex reduction, Ericson
// 5.1.5); overlapping cores, or cores closer than float resolution at their
// coordinates, get the Minkowski portal refinement (XenoCollide) along the
// ray from the centre difference through the origin. The contact patch then
// takes both cores' features within a slab of their support planes along the
// normal: two faces give the corners of their intersection polygon (A's face
// clipped by B's, Sutherland-Hodgman in the plane normal to the contact, with
// B's face normal replacing the query normal when within ~8 degrees), an edge
// on a face the clipped segment's ends, anything else the witness pair; the
// deepest MR_RAW_CONTACTS_PER_PAIR points are kept. Per lane: the cores,
// simplices and patch polygons live in private memory, so this code is
// compiled into its own kernel instances, used only by worlds with convex or
// mesh shapes (Collision.metal:2298-3740 is the reference's GJK / EPA / MPR /
// support-mapped patch; the algorithm here is the published one named above).

struct Core {
    uint32_t type;  // MR_SHAPE_* of the collider (MR_SHAPE_TRIANGLE_MESH for a triangle)
    uint32_t n;     // points
    float radius;
    V3 center;
    Q4 rotation;
    V3 scale;       // convex: vertex scale; box: half extents
    V3 p0, p1, p2;  // capsule endpoints / triangle vertices
    const mr_float4* verts;  // convex: the geometry's vertices
};

MRD_INL V3 core_point(const Core& c, uint32_t i) {
    if (c.type == MR_SHAPE_SPHERE) return c.center;
    if (c.type == MR_SHAPE_CAPSULE) return i == 0u ? c.p0 : c.p1;
    if (c.type == MR_SHAPE_TRIANGLE_MESH) return i == 0u ? c.p0 : (i == 1u ? c.p1 : c.p2);
    if (c.type == MR_SHAPE_BOX) {
        const V3 he = c.scale;
        const V3 l{(i & 1u) == 0u ? -he.x : he.x, (i & 2u) == 0u ? -he.y : he.y, (i & 4u) == 0u ? -he.z : he.z};
        return add(c.center, qrot(c.rotation, l));
    }
    const mr_float4 v = c.verts[i];
    return add(c.center, qrot(c.rotation, V3{c.scale.x * v.x, c.scale.y * v.y, c.scale.z * v.z}));
}

// Index of the point with the largest projection on d (the lowest on ties).
MRD_INL uint32_t core_support(const Core& c, V3 d) {
    uint32_t best = 0u;
    float bv = dot(d, core_point(c, 0u));
    for (uint32_t i = 1u; i < c.n; ++i) {
        const float v = dot(d, core_point(c, i));
        if (v > bv) {
            bv = v;
            best = i;
        }
    }
    return best;
}

MRD_INL Core make_core(const Env& e, uint32_t s, const Collider& col) {
    Core c;
    c.type = col.type;
    c.radius = 0.0f;
    c.center = col.center;
    c.rotation = col.rotation;
    c.scale = col.half_extents;
    c.p0 = col.p0;
    c.p1 = col.p1;
    c.p2 = V3{0.0f, 0.0f, 0.0f};
    c.verts = nullptr;
    if (col.type == MR_SHAPE_SPHERE) {
        c.n = 1u;
        c.radius = col.radius;
    } else if (col.type == MR_SHAPE_CAPSULE) {
        c.n = 2u;
        c.radius = col.radius;
    } else if (col.type == MR_SHAPE_BOX) {
        c.n = 8u;
    } else {
        const MRGeometryC& g = e.a->geometries[e.shapes[s].geometry];
        c.n = g.vertex_count;
        c.verts = e.a->geometry_vertices + g.vertex_offset;
    }
    return c;
}

struct Mv {
    V3 w, a, b;
    uint32_t ia, ib;
};

MRD_INL Mv minkowski_support(const Core& A, const Core& B, V3 d) {
    Mv m;
    m.ia = core_support(A, d);
    m.ib = core_support(B, neg(d));
    m.a = core_point(A, m.ia);
    m.b = core_point(B, m.ib);
    m.w = sub(m.a, m.b);
    return m;
}

// Closest point to the origin of simplex s[0..n) (n = 1..3), reducing it in
// place to the sub-simplex whose interior holds that point; lam are the
// barycentric weights of the kept points.
MRD_INL V3 simplex_closest(Mv* s, uint32_t& n, float* lam) {
    if (n == 1u) {
        lam[0] = 1.0f;
        return s[0].w;
    }
    if (n == 2u) {
        const V3 a = s[0].w, b = s[1].w, ab = sub(b, a);
        const float den = dot(ab, ab);
        const float t = den > kTiny ? -dot(a, ab) / den : 0.0f;
        if (t <= 0.0f) {
            n = 1u;
            lam[0] = 1.0f;
            return a;
        }
        if (t >= 1.0f) {
            s[0] = s[1];
            n = 1u;
            lam[0] = 1.0f;
            return b;
        }
        lam[0] = 1.0f - t;
        lam[1] = t;
        return add(a, mul(t, ab));
    }
    const V3 a = s[0].w, b = s[1].w, c = s[2].w;
    const V3 ab = sub(b, a), ac = sub(c, a), ap = neg(a);
    const float d1 = dot(ab, ap), d2 = dot(ac, ap);
    if (d1 <= 0.0f && d2 <= 0.0f) {
        n = 1u;
        lam[0] = 1.0f;
        return a;
    }
    const V3 bp = neg(b);
    const float d3 = dot(ab, bp), d4 = dot(ac, bp);
    if (d3 >= 0.0f && d4 <= d3) {
        s[0] = s[1];
        n = 1u;
        lam[0] = 1.0f;
        return b;
    }
    const float vc = d1 * d4 - d3 * d2;
    if (vc <= 0.0f && d1 >= 0.0f && d3 <= 0.0f) {
        const float t = d1 / (d1 - d3);
        n = 2u;
        lam[0] = 1.0f - t;
        lam[1] = t;
        return add(a, mul(t, ab));
    }
    const V3 cp = neg(c);
    const float d5 = dot(ab, cp), d6 = dot(ac, cp);
    if (d6 >= 0.0f && d5 <= d6) {
        s[0] = s[2];
        n = 1u;
        lam[0] = 1.0f;
        return c;
    }
    const float vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0f && d2 >= 0.0f && d6 <= 0.0f) {
        const float t = d2 / (d2 - d6);
        s[1] = s[2];
        n = 2u;
        lam[0] = 1.0f - t;
        lam[1] = t;
        return add(a, mul(t, ac));
    }
    const float va = d3 * d6 - d5 * d4;
    if (va <= 0.0f && (d4 - d3) >= 0.0f && (d5 - d6) >= 0.0f) {
        const float t = (d4 - d3) / ((d4 - d3) + (d5 - d6));
        s[0] = s[1];
        s[1] = s[2];
        n = 2u;
        lam[0] = 1.0f - t;
        lam[1] = t;
        return add(b, mul(t, sub(c, b)));
    }
    const float den = 1.0f / (va + vb + vc);
    const float v = vb * den, w = vc * den;
    lam[0] = 1.0f - v - w;
    lam[1] = v;
    lam[2] = w;
    return add(a, add(mul(v, ab), mul(w, ac)));
}

// True when the origin lies inside (or on) tetrahedron s[0..4).
MRD_INL bool tetra_contains_origin(const Mv* s) {
    for (int f = 0; f < 4; ++f) {
        const V3 a = s[(f + 1) % 4].w, b = s[(f + 2) % 4].w, c = s[(f + 3) % 4].w, d = s[f].w;
        const V3 nrm = cross(sub(b, a), sub(c, a));
        const float sd = dot(nrm, sub(d, a)), so = dot(nrm, neg(a));
        if (sd * so < 0.0f) return false;
    }
    return true;
}

struct ConvexHit {
    uint32_t status;  // 0 ok, 1 no result
    bool overlap;
    V3 n;             // A -> B
    float sep;        // core separation (negative: depth)
    V3 pa, pb;        // core witness points
};

MRD_INL ConvexHit gjk(const Core& A, const Core& B) {
    ConvexHit r;
    r.status = 0u;
    r.overlap = false;
    r.n = r.pa = r.pb = V3{0.0f, 0.0f, 0.0f};
    r.sep = 0.0f;
    Mv s[4];
    float lam[4] = {1.0f, 0.0f, 0.0f, 0.0f};
    uint32_t n = 0u;
    V3 v = sub(A.center, B.center);
    if (!(dot(v, v) > kTiny)) v = V3{1.0f, 0.0f, 0.0f};
    for (uint32_t it = 0; it < 64u; ++it) {
        const Mv m = minkowski_support(A, B, neg(v));
        const float vv = dot(v, v);
        if (n > 0u && vv - dot(v, m.w) <= 1.0e-6f * vv) break;
        bool repeat = false;
        for (uint32_t k = 0; k < n; ++k) repeat = repeat || (s[k].ia == m.ia && s[k].ib == m.ib);
        if (repeat) break;
        s[n++] = m;
        if (n == 4u) {
            if (tetra_contains_origin(s)) {
                r.overlap = true;
                return r;
            }
            float best = __builtin_inff();
            Mv keep[3];
            float kl[3];
            uint32_t kn = 0u;
            for (int f = 0; f < 4; ++f) {
                Mv t[3] = {s[(f + 1) % 4], s[(f + 2) % 4], s[(f + 3) % 4]};
                uint32_t tn = 3u;
                float tl[3];
                const V3 p = simplex_closest(t, tn, tl);
                const float d = dot(p, p);
                if (d < best) {
                    best = d;
                    kn = tn;
                    for (uint32_t k = 0; k < tn; ++k) {
                        keep[k] = t[k];
                        kl[k] = tl[k];
                    }
                    v = p;
                }
            }
            n = kn;
            for (uint32_t k = 0; k < kn; ++k) {
                s[k] = keep[k];
                lam[k] = kl[k];
            }
        } else {
            v = simplex_closest(s, n, lam);
        }
        if (dot(v, v) <= 1.0e-14f) {
            r.overlap = true;
            return r;
        }
    }
    V3 pa{0.0f, 0.0f, 0.0f}, pb{0.0f, 0.0f, 0.0f};
    for (uint32_t k = 0; k < n; ++k) {
        pa = add(pa, mul(lam[k], s[k].a));
        pb = add(pb, mul(lam[k], s[k].b));
    }
    const V3 d = sub(pb, pa);
    const float dist = length(d);
    const V3 ca = vabs(A.center), cb = vabs(B.center);
    const float coord = fmaxd(fmaxd(fmaxd(ca.x, ca.y), ca.z), fmaxd(fmaxd(cb.x, cb.y), cb.z));
    if (!(dist > 1.0e-6f * (1.0f + coord))) {
        r.overlap = true;
        return r;
    }
    r.pa = pa;
    r.pb = pb;
    r.sep = dist;
    r.n = dist > kTiny ? mul(1.0f / dist, d) : normalize(neg(v));
    return r;
}

MRD_INL ConvexHit mpr(const Core& A, const Core& B) {
    ConvexHit r;
    r.status = 1u;
    r.overlap = true;
    r.n = r.pa = r.pb = V3{0.0f, 0.0f, 0.0f};
    r.sep = 0.0f;
    Mv v0;
    v0.a = A.center;
    v0.b = B.center;
    v0.w = sub(A.center, B.center);
    v0.ia = v0.ib = 0u;
    if (!(dot(v0.w, v0.w) > 1.0e-12f)) v0.w = V3{1.0e-5f, 0.0f, 0.0f};
    V3 n = neg(v0.w);
    Mv v1 = minkowski_support(A, B, n);
    n = cross(v1.w, v0.w);
    if (!(dot(n, n) > 1.0e-14f)) {
        const V3 d = normalize(sub(v1.w, v0.w));
        r.status = 0u;
        r.n = d;
        r.sep = -dot(v1.w, d);
        r.pa = v1.a;
        r.pb = sub(v1.a, mul(-r.sep, d));
        return r;
    }
    Mv v2 = minkowski_support(A, B, n);
    if (dot(v2.w, n) < 0.0f) return r;
    n = cross(sub(v1.w, v0.w), sub(v2.w, v0.w));
    if (dot(n, v0.w) > 0.0f) {
        const Mv t = v1;
        v1 = v2;
        v2 = t;
        n = neg(n);
    }
    Mv v3;
    bool portal = false;
    for (uint32_t it = 0; it < 32u; ++it) {
        v3 = minkowski_support(A, B, n);
        if (dot(v3.w, n) < 0.0f) return r;
        if (dot(cross(v1.w, v3.w), v0.w) < 0.0f) {
            v2 = v3;
            n = cross(sub(v1.w, v0.w), sub(v3.w, v0.w));
            continue;
        }
        if (dot(cross(v3.w, v2.w), v0.w) < 0.0f) {
            v1 = v3;
            n = cross(sub(v3.w, v0.w), sub(v2.w, v0.w));
            continue;
        }
        portal = true;
        break;
    }
    if (!portal) return r;
    for (uint32_t it = 0; it < 32u; ++it) {
        n = cross(sub(v2.w, v1.w), sub(v3.w, v1.w));
        const float nl = length(n);
        if (!(nl > kTiny)) return r;
        n = mul(1.0f / nl, n);
        const Mv v4 = minkowski_support(A, B, n);
        const float delta = dot(sub(v4.w, v3.w), n);
        const float depth = dot(v4.w, n);
        if (delta <= 1.0e-5f * fmaxd(1.0f, fabs_(depth)) || it == 31u) {
            const float dist = dot(v1.w, n);
            const V3 p = mul(dist, n);
            const V3 e1 = sub(v2.w, v1.w), e2 = sub(v3.w, v1.w), ep = sub(p, v1.w);
            const float d00 = dot(e1, e1), d01 = dot(e1, e2), d11 = dot(e2, e2);
            const float d20 = dot(ep, e1), d21 = dot(ep, e2);
            const float den = d00 * d11 - d01 * d01;
            float b2 = 0.0f, b3 = 0.0f;
            if (fabs_(den) > kTiny) {
                b2 = (d11 * d20 - d01 * d21) / den;
                b3 = (d00 * d21 - d01 * d20) / den;
            }
            const float b1 = 1.0f - b2 - b3;
            r.status = 0u;
            r.n = n;
            r.sep = -depth;
            r.pa = add(add(mul(b1, v1.a), mul(b2, v2.a)), mul(b3, v3.a));
            r.pb = sub(r.pa, mul(depth, n));
            return r;
        }
        if (dot(cross(v4.w, v1.w), v0.w) < 0.0f) {
            if (dot(cross(v4.w, v2.w), v0.w) < 0.0f) v1 = v4;
            else v3 = v4;
        } else {
            if (dot(cross(v4.w, v3.w), v0.w) < 0.0f) v2 = v4;
            else v1 = v4;
        }
    }
    return r;
}

MRD_INL void plane_basis(V3 n, V3& t1, V3& t2) {
    const V3 an = vabs(n);
    V3 ref;
    if (an.x <= an.y && an.x <= an.z) ref = V3{1.0f, 0.0f, 0.0f};
    else if (an.y <= an.z) ref = V3{0.0f, 1.0f, 0.0f};
    else ref = V3{0.0f, 0.0f, 1.0f};
    t1 = normalize(cross(n, ref));
    t2 = cross(n, t1);
}

constexpr uint32_t kFeatureCap = 16u;
constexpr uint32_t kPatchCap = 2u * kFeatureCap;

// Points of core c within `slab` of its support plane along d, in index
// order (at most kFeatureCap), and the plane's offset.
MRD_INL uint32_t core_feature(const Core& c, V3 d, float slab, uint32_t* idx, float& top) {
    top = -__builtin_inff();
    for (uint32_t i = 0; i < c.n; ++i) top = fmaxd(top, dot(d, core_point(c, i)));
    uint32_t k = 0u;
    for (uint32_t i = 0; i < c.n && k < kFeatureCap; ++i)
        if (dot(d, core_point(c, i)) >= top - slab) idx[k++] = i;
    return k;
}

MRD_INL float core_extent(const Core& c) {
    float e = 0.0f;
    for (uint32_t i = 0; i < c.n; ++i) e = fmaxd(e, length(sub(core_point(c, i), c.center)));
    return e;
}

// Convex hull of planar points (gift wrapping from the lowest index of the
// leftmost point), counter-clockwise indices into pts; returns its size.
MRD_INL uint32_t hull2d(const float (*pts)[2], uint32_t n, uint32_t* out) {
    uint32_t start = 0u;
    for (uint32_t i = 1; i < n; ++i)
        if (pts[i][0] < pts[start][0] || (pts[i][0] == pts[start][0] && pts[i][1] < pts[start][1])) start = i;
    uint32_t h = 0u, p = start;
    do {
        out[h++] = p;
        uint32_t q = p == 0u ? 1u : 0u;
        for (uint32_t r = 0; r < n; ++r) {
            if (r == p) continue;
            const float cr = (pts[q][0] - pts[p][0]) * (pts[r][1] - pts[p][1]) -
                (pts[q][1] - pts[p][1]) * (pts[r][0] - pts[p][0]);
            const float dq = (pts[q][0] - pts[p][0]) * (pts[q][0] - pts[p][0]) +
                (pts[q][1] - pts[p][1]) * (pts[q][1] - pts[p][1]);
            const float dr = (pts[r][0] - pts[p][0]) * (pts[r][0] - pts[p][0]) +
                (pts[r][1] - pts[p][1]) * (pts[r][1] - pts[p][1]);
            if (cr < 0.0f || (cr == 0.0f && dr > dq)) q = r;
        }
        p = q;
    } while (p != start && h < n);
    return h;
}

// Clips segment (x0,y0)-(x1,y1) against a counter-clockwise convex polygon;
// the kept parameter interval is [t0, t1] (empty when t0 > t1).
MRD_INL void clip_segment(const float (*pts)[2], const uint32_t* poly, uint32_t m, float x0, float y0, float x1,
                          float y1, float& t0, float& t1) {
    t0 = 0.0f;
    t1 = 1.0f;
    for (uint32_t k = 0; k < m && t0 <= t1; ++k) {
        const float* a = pts[poly[k]];
        const float* b = pts[poly[(k + 1) % m]];
        const float ex = b[0] - a[0], ey = b[1] - a[1];
        const float f0 = ex * (y0 - a[1]) - ey * (x0 - a[0]);
        const float f1 = ex * (y1 - a[1]) - ey * (x1 - a[0]);
        if (f0 < 0.0f && f1 < 0.0f) {
            t0 = 1.0f;
            t1 = 0.0f;
        } else if (f0 < 0.0f) {
            t0 = fmaxd(t0, f0 / (f0 - f1));
        } else if (f1 < 0.0f) {
            t1 = fmind(t1, f0 / (f0 - f1));
        }
    }
}

// Keeps the deepest MR_RAW_CONTACTS_PER_PAIR contacts (replacing the
// shallowest, the earlier kept on ties).
MRD_INL void append_deepest(RawBatch& out, const RawContact& c) {
    if (out.count < MR_RAW_CONTACTS_PER_PAIR) {
        out.c[out.count++] = c;
        return;
    }
    uint32_t worst = 0u;
    for (uint32_t k = 1; k < out.count; ++k)
        if (out.c[k].separation > out.c[worst].separation) worst = k;
    if (c.separation < out.c[worst].separation) out.c[worst] = c;
}

MRD_INL uint32_t core_feature_key(const Core& c, uint32_t local, uint32_t tri_feature) {
    if (c.type == MR_SHAPE_TRIANGLE_MESH) return feature_key(MR_SHAPE_TRIANGLE_MESH, tri_feature);
    return feature_key(c.type, local);
}

// One vertex of the clipped patch polygon: plane coordinates, the point on
// A's feature, its feature keys, and the tag of the polygon edge leaving it
// (k < kFeatureCap: A's hull edge k; kFeatureCap + k: B's clip line k).
struct PatchVertex {
    float x, y;
    V3 p;
    uint32_t feat_a, feat_b, tag;
};

MRD_INL void convex_contacts(const Core& A, const Core& B, uint32_t tri_a, uint32_t tri_b, float accepted,
                             RawBatch& out) {
    ConvexHit h = gjk(A, B);
    if (h.overlap) h = mpr(A, B);
    if (h.status != 0u) return;
    const float sep = h.sep - A.radius - B.radius;
    if (!(sep <= accepted)) return;
    V3 n = h.n;
    const float ext_a = fmaxd(core_extent(A), 1.0e-3f), ext_b = fmaxd(core_extent(B), 1.0e-3f);
    uint32_t fa[kFeatureCap], fb[kFeatureCap];
    float top_a, top_b;
    const uint32_t na = core_feature(A, n, 2.0e-3f * ext_a, fa, top_a);
    const uint32_t nb = core_feature(B, neg(n), 2.0e-3f * ext_b, fb, top_b);
    float plane_b = -top_b;  // B's support plane: dot(n, x) = plane_b
    const uint32_t face_a = core_feature_key(A, 128u + fa[0], tri_a), face_b = core_feature_key(B, 128u + fb[0], tri_b);
    if (na == 1u || nb == 1u || (na == 2u && nb == 2u)) {
        const uint32_t feat_a = na == 1u ? core_feature_key(A, fa[0], tri_a) : face_a;
        const uint32_t feat_b = nb == 1u ? core_feature_key(B, fb[0], tri_b) : face_b;
        append_deepest(out, make_contact(n, h.sep - A.radius - B.radius, add(h.pa, mul(A.radius, n)),
                                         sub(h.pb, mul(B.radius, n)), feat_a, feat_b));
        return;
    }
    V3 t1, t2;
    plane_basis(n, t1, t2);
    float pa2[kFeatureCap][2], pb2[kFeatureCap][2];
    V3 wa[kFeatureCap], wb[kFeatureCap];
    for (uint32_t k = 0; k < na; ++k) {
        wa[k] = core_point(A, fa[k]);
        pa2[k][0] = dot(t1, wa[k]);
        pa2[k][1] = dot(t2, wa[k]);
    }
    for (uint32_t k = 0; k < nb; ++k) {
        wb[k] = core_point(B, fb[k]);
        pb2[k][0] = dot(t1, wb[k]);
        pb2[k][1] = dot(t2, wb[k]);
    }
    uint32_t hull_a[kFeatureCap], hull_b[kFeatureCap];
    const uint32_t ma = na >= 3u ? hull2d(pa2, na, hull_a) : 0u;
    const uint32_t mb = nb >= 3u ? hull2d(pb2, nb, hull_b) : 0u;
    const uint32_t before = out.count;
    if (ma >= 3u && mb >= 3u) {
        V3 fnrm{0.0f, 0.0f, 0.0f};
        for (uint32_t k = 0; k < mb; ++k) fnrm = add(fnrm, cross(wb[hull_b[k]], wb[hull_b[(k + 1u) % mb]]));
        const float fl = length(fnrm);
        if (fl > kTiny && dot(fnrm, n) >= 0.99f * fl) {
            n = mul(1.0f / fl, fnrm);
            plane_b = __builtin_inff();
            for (uint32_t k = 0; k < nb; ++k) plane_b = fmind(plane_b, dot(n, wb[k]));
        }
        PatchVertex poly[kPatchCap], next[kPatchCap];
        uint32_t m = ma;
        for (uint32_t k = 0; k < ma; ++k) {
            const uint32_t i = hull_a[k];
            poly[k] = PatchVertex{pa2[i][0], pa2[i][1], wa[i], core_feature_key(A, fa[i], tri_a), face_b, k};
        }
        for (uint32_t k = 0; k < mb && m > 0u; ++k) {
            const float* a = pb2[hull_b[k]];
            const float* b = pb2[hull_b[(k + 1u) % mb]];
            const float ex = b[0] - a[0], ey = b[1] - a[1];
            uint32_t q = 0u;
            for (uint32_t j = 0; j < m; ++j) {
                const PatchVertex P = poly[j];
                const PatchVertex Q = poly[(j + 1u) % m];
                const float fp = ex * (P.y - a[1]) - ey * (P.x - a[0]);
                const float fq = ex * (Q.y - a[1]) - ey * (Q.x - a[0]);
                const bool in_p = fp >= 0.0f, in_q = fq >= 0.0f;
                if (in_p != in_q && q < kPatchCap) {
                    const float t = fp / (fp - fq);
                    PatchVertex c;
                    c.x = P.x + t * (Q.x - P.x);
                    c.y = P.y + t * (Q.y - P.y);
                    c.p = add(P.p, mul(t, sub(Q.p, P.p)));
                    if (P.tag < kFeatureCap) {
                        c.feat_a = core_feature_key(A, 64u + fa[hull_a[P.tag]], tri_a);
                        c.feat_b = core_feature_key(B, 64u + fb[hull_b[k]], tri_b);
                    } else {
                        const uint32_t j_line = P.tag - kFeatureCap;
                        const uint32_t shared = j_line + 1u == k ? hull_b[k]
                            : (j_line == 0u && k + 1u == mb) ? hull_b[0] : MR_INVALID_INDEX;
                        c.feat_a = face_a;
                        c.feat_b = shared != MR_INVALID_INDEX ? core_feature_key(B, fb[shared], tri_b)
                                                              : core_feature_key(B, 64u + fb[hull_b[k]], tri_b);
                    }
                    c.tag = in_p ? kFeatureCap + k : P.tag;
                    next[q++] = c;
                }
                if (in_q && q < kPatchCap) next[q++] = Q;
            }
            m = q;
            for (uint32_t j = 0; j < m; ++j) poly[j] = next[j];
        }
        const float tol = 4.0e-6f * (1.0f + fmaxd(ext_a, ext_b));
        for (uint32_t j = 0; j < m; ++j) {
            bool dup = false;
            for (uint32_t i = 0; i < j; ++i) {
                const float dx = poly[j].x - poly[i].x, dy = poly[j].y - poly[i].y;
                dup = dup || dx * dx + dy * dy <= tol * tol;
            }
            if (dup) continue;
            const float s = plane_b - dot(n, poly[j].p);
            append_deepest(out, make_contact(n, s - A.radius - B.radius, add(poly[j].p, mul(A.radius, n)),
                                             sub(add(poly[j].p, mul(s, n)), mul(B.radius, n)), poly[j].feat_a,
                                             poly[j].feat_b));
        }
    } else if (na == 2u && mb >= 3u) {
        float t0, tt1;
        clip_segment(pb2, hull_b, mb, pa2[0][0], pa2[0][1], pa2[1][0], pa2[1][1], t0, tt1);
        if (t0 <= tt1)
            for (int ei = 0; ei < 2; ++ei) {
                const float t = ei == 0 ? t0 : tt1;
                const V3 p = add(wa[0], mul(t, sub(wa[1], wa[0])));
                const float s = plane_b - dot(n, p);
                append_deepest(out, make_contact(n, s - A.radius - B.radius, add(p, mul(A.radius, n)),
                                                 sub(add(p, mul(s, n)), mul(B.radius, n)),
                                                 core_feature_key(A, 64u + fa[ei], tri_a), face_b));
            }
    } else if (nb == 2u && ma >= 3u) {
        float t0, tt1;
        clip_segment(pa2, hull_a, ma, pb2[0][0], pb2[0][1], pb2[1][0], pb2[1][1], t0, tt1);
        if (t0 <= tt1)
            for (int ei = 0; ei < 2; ++ei) {
                const float t = ei == 0 ? t0 : tt1;
                const V3 p = add(wb[0], mul(t, sub(wb[1], wb[0])));
                const float s = dot(n, p) - top_a;
                append_deepest(out, make_contact(n, s - A.radius - B.radius, add(sub(p, mul(s, n)), mul(A.radius, n)),
                                                 sub(p, mul(B.radius, n)), face_a,
                                                 core_feature_key(B, 64u + fb[ei], tri_b)));
            }
    }
    if (out.count == before)
        append_deepest(out, make_contact(n, h.sep - A.radius - B.radius, add(h.pa, mul(A.radius, n)),
                                         sub(h.pb, mul(B.radius, n)), face_a, face_b));
}

// A convex hull against a plane: every vertex within `accepted` (deepest 8).
MRD_INL void convex_plane_contacts(const Core& hull, const Collider& plane, bool plane_is_a, float accepted,
                                   RawBatch& out) {
    for (uint32_t i = 0; i < hull.n; ++i) {
        const V3 p = core_point(hull, i);
        const float sep = dot(plane.plane_normal, sub(p, plane.center));
        if (!(sep <= accepted)) continue;
        const V3 sp = sub(p, mul(sep, plane.plane_normal));
        RawContact c = make_contact(neg(plane.plane_normal), sep, p, sp, feature_key(MR_SHAPE_CONVEX, i),
                                    feature_key(MR_SHAPE_PLANE, 0u));
        if (plane_is_a) c = swapped(c);
        append_deepest(out, c);
    }
}

constexpr uint32_t kBvhStack = 48u;

// A static mesh against a finite collider: BVH4 traversal with the finite
// collider's bounds (padded by the accepted distance) in the mesh's unscaled
// local frame, then every overlapping triangle as a 3-point core. One-sided
// meshes keep the contacts whose normal (finite -> mesh) opposes the
// triangle's front normal (counter-clockwise vertices).
MRD_INL void mesh_contacts(const Env& e, uint32_t mesh_shape, const Collider& mesh, const Core& fin,
                           const Collider& fin_col, bool mesh_is_a, float accepted, RawBatch& out) {
    const MRShapeC& ms = e.shapes[mesh_shape];
    const MRGeometryC g = e.a->geometries[ms.geometry];
    const mr_float4* vt = e.a->geometry_vertices + g.vertex_offset;
    const MRTriangleC* tris = e.a->triangles + g.triangle_offset;
    const MRBvhNodeC* nodes = e.a->bvh_nodes + g.node_offset;
    const bool two_sided = (ms.flags & MR_SHAPE_FLAG_MESH_TWO_SIDED) != 0u;
    const V3 scale = mesh.half_extents;
    V3 lo{__builtin_inff(), __builtin_inff(), __builtin_inff()};
    V3 hi{-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
    for (uint32_t k = 0; k < 8u; ++k) {
        const V3 w{(k & 1u) ? fin_col.upper.x + accepted : fin_col.lower.x - accepted,
                   (k & 2u) ? fin_col.upper.y + accepted : fin_col.lower.y - accepted,
                   (k & 4u) ? fin_col.upper.z + accepted : fin_col.lower.z - accepted};
        const V3 l = qrot_inv(mesh.rotation, sub(w, mesh.center));
        const V3 u{l.x / scale.x, l.y / scale.y, l.z / scale.z};
        lo = vmin(lo, u);
        hi = vmax(hi, u);
    }
    uint32_t stack[kBvhStack];
    uint32_t top = 0u;
    stack[top++] = 0u;
    while (top > 0u) {
        const MRBvhNodeC& nd = nodes[stack[--top]];
        const float lx[4] = {nd.lower_x.x, nd.lower_x.y, nd.lower_x.z, nd.lower_x.w};
        const float ly[4] = {nd.lower_y.x, nd.lower_y.y, nd.lower_y.z, nd.lower_y.w};
        const float lz[4] = {nd.lower_z.x, nd.lower_z.y, nd.lower_z.z, nd.lower_z.w};
        const float ux[4] = {nd.upper_x.x, nd.upper_x.y, nd.upper_x.z, nd.upper_x.w};
        const float uy[4] = {nd.upper_y.x, nd.upper_y.y, nd.upper_y.z, nd.upper_y.w};
        const float uz[4] = {nd.upper_z.x, nd.upper_z.y, nd.upper_z.z, nd.upper_z.w};
        uint32_t child[4], count[4];
        for (int c = 0; c < 4; ++c) {
            child[c] = nd.child[c];
            count[c] = nd.count[c];
        }
        for (int c = 3; c >= 0; --c) {  // pushed in reverse: children leave the stack in index order
            if (child[c] == MR_INVALID_INDEX || count[c] != 0u) continue;
            if (lx[c] <= hi.x && ux[c] >= lo.x && ly[c] <= hi.y && uy[c] >= lo.y && lz[c] <= hi.z && uz[c] >= lo.z &&
                top < kBvhStack)
                stack[top++] = child[c];
        }
        for (uint32_t c = 0; c < 4u; ++c) {
            if (child[c] == MR_INVALID_INDEX || count[c] == 0u) continue;
            if (!(lx[c] <= hi.x && ux[c] >= lo.x && ly[c] <= hi.y && uy[c] >= lo.y && lz[c] <= hi.z && uz[c] >= lo.z))
                continue;
            for (uint32_t t = child[c]; t < child[c] + count[c]; ++t) {
                const MRTriangleC tr = tris[t];
                Core tc;
                tc.type = MR_SHAPE_TRIANGLE_MESH;
                tc.n = 3u;
                tc.radius = 0.0f;
                tc.rotation = mesh.rotation;
                tc.scale = scale;
                tc.verts = nullptr;
                V3 p[3];
                for (int k = 0; k < 3; ++k) {
                    const mr_float4 v = vt[tr.vertices[k]];
                    p[k] = add(mesh.center, qrot(mesh.rotation, V3{scale.x * v.x, scale.y * v.y, scale.z * v.z}));
                }
                tc.p0 = p[0];
                tc.p1 = p[1];
                tc.p2 = p[2];
                tc.center = mul(1.0f / 3.0f, add(add(p[0], p[1]), p[2]));
                RawBatch one;
                one.count = 0u;
                convex_contacts(fin, tc, 0u, tr.feature, accepted, one);
                const V3 front = cross(sub(p[1], p[0]), sub(p[2], p[0]));
                for (uint32_t k = 0; k < one.count; ++k) {
                    const RawContact& rc = one.c[k];
                    if (!two_sided && !(dot(rc.normal, front) < 0.0f)) continue;
                    append_deepest(out, mesh_is_a ? swapped(rc) : rc);
                }
            }
        }
    }
}

// hf_first: index of this pair's first precomputed heightfield query in e.hfq,
// or ~0 to evaluate the queries here. Convex and mesh pairs are generated by
// the kGeo instances only.
template <bool kGeo = false>
MRD_INL void generate_contacts(const Env& e, uint32_t ia, uint32_t ib, uint32_t cls, const Collider& A,
                               const Collider& B, ContactSink& out, uint32_t hf_first) {
    const float accepted = (A.contact_offset + B.contact_offset) + pair_query_padding(A, B);
    if (cls == MR_PAIR_SPHERE_SPHERE) {
        const V3 d = sub(B.center, A.center);
        const float dist = length(d);
        const V3 n = dist > kTiny ? mul(1.0f / dist, d) : coincident_normal(ia, ib);
        const float sep = dist - A.radius - B.radius;
        if (sep > accepted) return;
        append(out, make_contact(n, sep, add(A.center, mul(A.radius, n)), sub(B.center, mul(B.radius, n)),
                                 feature_key(MR_SHAPE_SPHERE, 0u), feature_key(MR_SHAPE_SPHERE, 0u)));
    } else if (cls == MR_PAIR_SPHERE_CAPSULE) {
        const bool sphere_a = A.type == MR_SHAPE_SPHERE;
        const Collider& sp = sphere_a ? A : B;
        const Collider& cp = sphere_a ? B : A;
        const uint32_t si = sphere_a ? ia : ib, ci = sphere_a ? ib : ia;
        const SegPoint cl = closest_on_segment(sp.center, cp.p0, cp.p1);
        const V3 d = sub(cl.point, sp.center);
        const float dist = length(d);
        const V3 n = dist > kTiny ? mul(1.0f / dist, d)
                                  : stable_segment_normal(sub(cp.p1, cp.p0), V3{0.0f, 0.0f, 0.0f}, si, ci);
        const float sep = dist - sp.radius - cp.radius;
        if (sep <= accepted) {
            RawContact c = make_contact(n, sep, add(sp.center, mul(sp.radius, n)), sub(cl.point, mul(cp.radius, n)),
                                        feature_key(MR_SHAPE_SPHERE, 0u),
                                        feature_key(MR_SHAPE_CAPSULE, capsule_feature(cl.t)));
            if (!sphere_a) c = swapped(c);
            append(out, c);
        }
    } else if (cls == MR_PAIR_CAPSULE_CAPSULE) {
        const SegPair cl = closest_segments(A.p0, A.p1, B.p0, B.p1);
        const V3 d = sub(cl.pb, cl.pa);
        const float dist = length(d);
        const V3 n = dist > kTiny ? mul(1.0f / dist, d) : stable_segment_normal(sub(A.p1, A.p0), sub(B.p1, B.p0), ia, ib);
        const float sep = dist - A.radius - B.radius;
        if (sep <= accepted)
            append(out, make_contact(n, sep, add(cl.pa, mul(A.radius, n)), sub(cl.pb, mul(B.radius, n)),
                                     feature_key(MR_SHAPE_CAPSULE, capsule_feature(cl.ta)),
                                     feature_key(MR_SHAPE_CAPSULE, capsule_feature(cl.tb))));
    } else if (cls == MR_PAIR_SPHERE_BOX) {
        const bool sphere_a = A.type == MR_SHAPE_SPHERE;
        const Collider& sp = sphere_a ? A : B;
        const Collider& bx = sphere_a ? B : A;
        V3 n, bp;
        float sep;
        uint32_t feat;
        sphere_box(sp, bx, n, bp, sep, feat);
        if (sep <= accepted) {
            RawContact c = make_contact(n, sep, add(sp.center, mul(sp.radius, n)), bp, feature_key(MR_SHAPE_SPHERE, 0u),
                                        feature_key(MR_SHAPE_BOX, feat));
            if (!sphere_a) c = swapped(c);
            append(out, c);
        }
    } else if (cls == MR_PAIR_CAPSULE_BOX) {
        const bool cap_a = A.type == MR_SHAPE_CAPSULE;
        const Collider& cp = cap_a ? A : B;
        const Collider& bx = cap_a ? B : A;
        V3 n, cpp, bp;
        float sep, t;
        uint32_t feat;
        capsule_box(cp, bx, cap_a ? ia : ib, cap_a ? ib : ia, n, cpp, bp, sep, t, feat);
        if (sep <= accepted) {
            RawContact c = make_contact(n, sep, cpp, bp, feature_key(MR_SHAPE_CAPSULE, capsule_feature(t)),
                                        feature_key(MR_SHAPE_BOX, feat));
            if (!cap_a) c = swapped(c);
            append(out, c);
        }
    } else if (cls == MR_PAIR_BOX_BOX) {
        box_box(ia, ib, A, B, accepted, out);
    } else if (cls == MR_PAIR_SPHERE_PLANE || cls == MR_PAIR_CAPSULE_PLANE || cls == MR_PAIR_BOX_PLANE) {
        const bool plane_a = A.type == MR_SHAPE_PLANE;
        const Collider& pl = plane_a ? A : B;
        const Collider& fs = plane_a ? B : A;
        const uint32_t pf = feature_key(MR_SHAPE_PLANE, 0u);
        if (cls == MR_PAIR_SPHERE_PLANE) {
            const V3 surf = sub(fs.center, mul(fs.radius, pl.plane_normal));
            const float sep = dot(pl.plane_normal, sub(surf, pl.center));
            if (sep <= accepted)
                append_surface_contact(out, plane_a, pl.plane_normal, surf, sep, feature_key(MR_SHAPE_SPHERE, 0u), pf);
        } else if (cls == MR_PAIR_CAPSULE_PLANE) {
            for (uint32_t en = 0; en < 2u; ++en) {
                const V3 ep = en == 0u ? fs.p0 : fs.p1;
                const V3 surf = sub(ep, mul(fs.radius, pl.plane_normal));
                const float sep = dot(pl.plane_normal, sub(surf, pl.center));
                if (sep <= accepted)
                    append_surface_contact(out, plane_a, pl.plane_normal, surf, sep, feature_key(MR_SHAPE_CAPSULE, en),
                                           pf);
            }
        } else {
            for (uint32_t vi = 0; vi < 8u; ++vi) {
                const V3 wv = box_vertex(fs, vi);
                const float sep = dot(pl.plane_normal, sub(wv, pl.center));
                if (sep <= accepted)
                    append_surface_contact(out, plane_a, pl.plane_normal, wv, sep, feature_key(MR_SHAPE_BOX, vi), pf);
            }
        }
    } else if (cls == MR_PAIR_HEIGHTFIELD) {
        const bool hf_a = A.type == MR_SHAPE_HEIGHTFIELD;
        const Collider& fs = hf_a ? B : A;
        const uint32_t nq = hf_query_count(fs.type);
        for (uint32_t q = 0; q < nq; ++q) {
            const mr::HfHit h = hf_first != 0xffffffffu ? e.hfq[hf_first + q]
                                                        : heightfield_query(e, hf_query_point(fs, q), hf_query_radius(fs));
            if (h.d <= accepted)
                append_surface_contact(out, hf_a, V3{h.n[0], h.n[1], h.n[2]}, V3{h.p[0], h.p[1], h.p[2]}, h.d,
                                       feature_key(fs.type, q), h.feature);
        }
    } else if (kGeo && (cls == MR_PAIR_CONVEX || cls == MR_PAIR_MESH)) {
        RawBatch batch;
        batch.count = 0;
        if (cls == MR_PAIR_CONVEX) {
            if (A.type == MR_SHAPE_PLANE || B.type == MR_SHAPE_PLANE) {
                const bool plane_a = A.type == MR_SHAPE_PLANE;
                convex_plane_contacts(make_core(e, plane_a ? ib : ia, plane_a ? B : A), plane_a ? A : B, plane_a,
                                      accepted, batch);
            } else {
                convex_contacts(make_core(e, ia, A), make_core(e, ib, B), 0u, 0u, accepted, batch);
            }
        } else {
            const bool mesh_a = A.type == MR_SHAPE_TRIANGLE_MESH;
            mesh_contacts(e, mesh_a ? ia : ib, mesh_a ? A : B, make_core(e, mesh_a ? ib : ia, mesh_a ? B : A),
                          mesh_a ? B : A, mesh_a, accepted, batch);
        }
        for (uint32_t c = 0; c < batch.count; ++c) append(out, batch.c[c]);
    }
}


// ------------------------------------------------ continuous collision
//
// The hybrid mode splits a microstep at the earliest time of impact (TOI) of
// the CCD-enabled compiled pairs (mr_world_resolve_ccd and the event select /
// finalize kernels, Collision.metal:6707-6950, 7157-7330, 7657-7900). Over the
// remaining time T of the microstep every body moves rigidly: links with the
// COM and angular velocity of the current kinematics, dynamic scene bodies
// with their velocity plus T * gravity, kinematic bodies with theirs, static
// bodies not at all; rotations follow exp(t w) at a constant rate. A pair whose
// swept bounds overlap and whose colliders start farther apart than their
// contact distance (the sum of the contact offsets; within it the segment's
// speculative contacts hold the pair at any normal speed) gets a TOI: closed
// form for two spheres (centres moving linearly),
// conservative advancement otherwise, stepping t by distance / (closing-speed
// bound), at least the minimum advance, and reporting the first t at which the
// pair is within the tolerance. A step never closes the gap past contact, so
// the pair is touching there without penetrating (up to speed x minimum
// advance). The closing-speed bound is |v_a - v_b| + |w_a| r_a + |w_b| r_b, r
// the largest distance from a body's COM to a point of its shape (exact for
// the constant-rate rotation); against a static plane only the normal
// component of the velocity counts. A pair that does not resolve within the iteration
// cap is safe when both bodies move less than their contact offset plus the
// tolerance (the speculative contacts cover it), and fails the step otherwise.

struct CcdMotion {
    V3 p0;
    Q4 r0;
    V3 v, w;
};

MRD_INL CcdMotion ccd_motion(const Env& e, uint32_t b, float T) {
    const V3 zero{0.0f, 0.0f, 0.0f};
    CcdMotion m;
    if (b < e.nlinks) {
        m.p0 = e.pos[b];
        m.r0 = e.rot[b];
        m.v = e.vl[b];
        m.w = e.w[b];
        return m;
    }
    const MRBodyStateC& s = e.scene[b - e.nlinks];
    m.p0 = f3(s.position);
    m.r0 = q4(s.orientation);
    const uint32_t mt = e.topo->motion[b];
    if (mt == MR_MOTION_DYNAMIC) {
        m.v = add(f3(s.linear_velocity_inv_mass), mul(T, e.gravity));
        m.w = f3(s.angular_velocity);
    } else if (mt == MR_MOTION_KINEMATIC) {
        m.v = f3(s.linear_velocity_inv_mass);
        m.w = f3(s.angular_velocity);
    } else {
        m.v = zero;
        m.w = zero;
    }
    return m;
}

template <bool kGeo>
MRD_INL bool ccd_collider(const Env& e, uint32_t s, const CcdMotion& m, float t, Collider& c) {
    const V3 p = add(m.p0, mul(t, m.v));
    Q4 r;
    if (!normalized_quat(qmul(rotation_increment(mul(t, m.w)), m.r0), r)) return false;
    return project_collider_pose<kGeo>(e, s, p, r, c);
}

// Largest distance from the body's COM to a point of shape s; planes and
// heightfields are unbounded.
MRD_INL float ccd_reach(const MRShapeC& sh) {
    const float offset = length(f3(sh.local_position));
    if (sh.shape_type == MR_SHAPE_SPHERE) return offset + sh.dimensions.x;
    if (sh.shape_type == MR_SHAPE_CAPSULE) return offset + sh.dimensions.x + sh.dimensions.y;
    if (sh.shape_type == MR_SHAPE_BOX) return offset + length(f3(sh.dimensions));
    return __builtin_inff();
}

// Distance bound of a body's shape point over the remaining time T.
MRD_INL float ccd_motion_bound(const CcdMotion& m, const MRShapeC& sh, float T) {
    const float wl = length(m.w), vl = length(m.v);
    if (!(wl > 0.0f) && !(vl > 0.0f)) return 0.0f;
    const float reach = wl > 0.0f ? ccd_reach(sh) : 0.0f;
    return T * (vl + wl * reach);
}

// Separation of two colliders at any distance (negative when they overlap):
// the analytic pair functions without the contact-distance cut-off. For two
// boxes the largest separation over the 15 separating axes, a lower bound of
// their distance. Heightfields have no such query.
MRD_INL float box_box_separation(const Collider& A, const Collider& B) {
    const V3 d = sub(B.center, A.center);
    float best = -__builtin_inff();
    for (int i = 0; i < 3; ++i) {
        const V3 ax = box_axis(A, i);
        best = fmaxd(best, fabs_(dot(d, ax)) - comp(A.half_extents, i) - box_projection_radius(B, ax));
    }
    for (int j = 0; j < 3; ++j) {
        const V3 ax = box_axis(B, j);
        best = fmaxd(best, fabs_(dot(d, ax)) - box_projection_radius(A, ax) - comp(B.half_extents, j));
    }
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) {
            const V3 c = cross(box_axis(A, i), box_axis(B, j));
            const float l = length(c);
            if (!(l > 1.0e-6f)) continue;
            const V3 ax = mul(1.0f / l, c);
            best = fmaxd(best, fabs_(dot(d, ax)) - box_projection_radius(A, ax) - box_projection_radius(B, ax));
        }
    return best;
}

MRD_INL bool ccd_separation(uint32_t ia, uint32_t ib, uint32_t cls, const Collider& A, const Collider& B, float& d) {
    if (cls == MR_PAIR_SPHERE_SPHERE) {
        d = length(sub(B.center, A.center)) - A.radius - B.radius;
    } else if (cls == MR_PAIR_SPHERE_CAPSULE) {
        const Collider& sp = A.type == MR_SHAPE_SPHERE ? A : B;
        const Collider& cp = A.type == MR_SHAPE_SPHERE ? B : A;
        const SegPoint cl = closest_on_segment(sp.center, cp.p0, cp.p1);
        d = length(sub(cl.point, sp.center)) - sp.radius - cp.radius;
    } else if (cls == MR_PAIR_CAPSULE_CAPSULE) {
        const SegPair cl = closest_segments(A.p0, A.p1, B.p0, B.p1);
        d = length(sub(cl.pb, cl.pa)) - A.radius - B.radius;
    } else if (cls == MR_PAIR_SPHERE_BOX) {
        const bool sphere_a = A.type == MR_SHAPE_SPHERE;
        V3 n, bp;
        uint32_t feat;
        sphere_box(sphere_a ? A : B, sphere_a ? B : A, n, bp, d, feat);
    } else if (cls == MR_PAIR_CAPSULE_BOX) {
        const bool cap_a = A.type == MR_SHAPE_CAPSULE;
        V3 n, cpp, bp;
        float t;
        uint32_t feat;
        capsule_box(cap_a ? A : B, cap_a ? B : A, cap_a ? ia : ib, cap_a ? ib : ia, n, cpp, bp, d, t, feat);
    } else if (cls == MR_PAIR_BOX_BOX) {
        d = box_box_separation(A, B);
    } else if (cls == MR_PAIR_SPHERE_PLANE || cls == MR_PAIR_CAPSULE_PLANE || cls == MR_PAIR_BOX_PLANE) {
        const Collider& pl = A.type == MR_SHAPE_PLANE ? A : B;
        const Collider& fs = A.type == MR_SHAPE_PLANE ? B : A;
        if (cls == MR_PAIR_SPHERE_PLANE) {
            d = dot(pl.plane_normal, sub(fs.center, pl.center)) - fs.radius;
        } else if (cls == MR_PAIR_CAPSULE_PLANE) {
            d = fmind(dot(pl.plane_normal, sub(fs.p0, pl.center)), dot(pl.plane_normal, sub(fs.p1, pl.center))) -
                fs.radius;
        } else {
            d = __builtin_inff();
            for (uint32_t vi = 0; vi < 8u; ++vi) d = fmind(d, dot(pl.plane_normal, sub(box_vertex(fs, vi), pl.center)));
        }
    } else {
        return false;
    }
    return isfin(d);
}

enum : uint32_t { kCcdNone = 0u, kCcdImpact = 1u, kCcdUnsafe = 2u };

// Collider s at the start of the remaining time T, its bounds those of the whole
// motion (the union of the start's and the end's); body = MR_INVALID_INDEX where a
// pose is not finite.
template <bool kGeo>
MRD_INL void ccd_sweep_collider(const Env& e, uint32_t s, float T, Collider& c) {
    const CcdMotion m = ccd_motion(e, e.shapes[s].body, T);
    Collider end;
    const bool valid = ccd_collider<kGeo>(e, s, m, 0.0f, c) && ccd_collider<kGeo>(e, s, m, T, end);
    if (!valid) {
        c.body = MR_INVALID_INDEX;
        return;
    }
    c.lower = vmin(c.lower, end.lower);
    c.upper = vmax(c.upper, end.upper);
}

// Whether compiled pair k has a TOI query to run: a CCD flag, both shapes taking
// part, and swept bounds that overlap (or a pose that is not finite, which the
// query judges).
MRD_INL bool ccd_pair_swept(const Env& e, uint32_t k) {
    const MRCompiledPairC& pr = e.pairs[k];
    const uint32_t flags = e.shapes[pr.collider_a].flags | e.shapes[pr.collider_b].flags;
    if ((flags & MR_SHAPE_FLAG_ENABLE_CCD) == 0u || (flags & MR_SHAPE_FLAG_SIMULATION_DISABLED) != 0u) return false;
    const Collider& a = e.ccol[pr.collider_a];
    const Collider& b = e.ccol[pr.collider_b];
    return a.body == MR_INVALID_INDEX || b.body == MR_INVALID_INDEX || pair_may_overlap(a, b);
}

// TOI query of compiled pair k (ccd_pair_swept) over the remaining time T.
// Returns kCcdImpact with toi (seconds), kCcdUnsafe for an unresolved pair the
// speculative contacts do not cover, kCcdNone otherwise (apart over the whole
// interval, or touching already: the discrete contacts handle that).
template <bool kGeo>
MRD_INL uint32_t ccd_pair(const Env& e, uint32_t k, float T, float& toi) {
    const MRWorldStepConfigC& cfg = e.a->cfg;
    const MRCompiledPairC& pr = e.pairs[k];
    const MRShapeC& sa = e.shapes[pr.collider_a];
    const MRShapeC& sb = e.shapes[pr.collider_b];
    const CcdMotion ma = ccd_motion(e, sa.body, T), mb = ccd_motion(e, sb.body, T);
    const float tol = cfg.ccd_distance_tolerance;
    const float motion_a = ccd_motion_bound(ma, sa, T), motion_b = ccd_motion_bound(mb, sb, T);
    const bool speculative_safe = motion_a <= sa.contact_rest_radius.x + tol && motion_b <= sb.contact_rest_radius.x + tol;
    const Collider a0 = e.ccol[pr.collider_a], b0 = e.ccol[pr.collider_b];
    float d;
    if (a0.body == MR_INVALID_INDEX || b0.body == MR_INVALID_INDEX || !ccd_separation(pr.collider_a, pr.collider_b, pr.pair_class, a0, b0, d))
        return speculative_safe ? kCcdNone : kCcdUnsafe;
    // within the contact distance the segment's speculative contacts hold the pair
    if (d <= fmaxd(tol, sa.contact_rest_radius.x + sb.contact_rest_radius.x)) return kCcdNone;
    if (pr.pair_class == MR_PAIR_SPHERE_SPHERE) {
        Collider a1, b1;
        ccd_collider<kGeo>(e, pr.collider_a, ma, T, a1);
        ccd_collider<kGeo>(e, pr.collider_b, mb, T, b1);
        const V3 rel0 = sub(b0.center, a0.center);
        const V3 drel = sub(sub(b1.center, b0.center), sub(a1.center, a0.center));
        const float radius = a0.radius + b0.radius;
        const float aa = dot(drel, drel), bb = 2.0f * dot(rel0, drel), cc = dot(rel0, rel0) - radius * radius;
        const float disc = bb * bb - 4.0f * aa * cc;
        if (aa > kTiny && disc >= 0.0f) {
            const float alpha = (-bb - sqrt_rn(disc)) / (2.0f * aa);
            if (alpha >= 0.0f && alpha <= 1.0f) {
                toi = alpha * T;
                return kCcdImpact;
            }
        }
        return kCcdNone;
    }
    // Closing-speed bound: |v_a - v_b| + |w_a| r_a + |w_b| r_b; against a
    // static plane only the motion along its normal closes the gap.
    const bool plane_a = a0.type == MR_SHAPE_PLANE, plane_b = b0.type == MR_SHAPE_PLANE;
    float total;
    if ((plane_a && !(motion_a > 0.0f)) || (plane_b && !(motion_b > 0.0f))) {
        const V3 n = plane_a ? a0.plane_normal : b0.plane_normal;
        const CcdMotion& fm = plane_a ? mb : ma;
        const float wl = length(fm.w);
        const float reach = wl > 0.0f ? ccd_reach(plane_a ? sb : sa) : 0.0f;
        total = T * (fabs_(dot(fm.v, n)) + wl * reach);
    } else {
        const float wa = length(ma.w), wb = length(mb.w);
        const float spin = (wa > 0.0f ? wa * ccd_reach(sa) : 0.0f) + (wb > 0.0f ? wb * ccd_reach(sb) : 0.0f);
        total = T * (length(sub(ma.v, mb.v)) + spin);
    }
    total = fmaxd(total, tol);
    const float min_alpha = fmind(1.0f, cfg.ccd_minimum_advance / T);
    float alpha = 0.0f;
    for (uint32_t it = 0; it < cfg.max_ccd_iterations; ++it) {
        if (d <= tol) {
            toi = alpha * T;
            return kCcdImpact;
        }
        alpha += fmaxd(d / total, min_alpha);
        if (alpha > 1.0f) return kCcdNone;
        Collider a, b;
        if (!ccd_collider<kGeo>(e, pr.collider_a, ma, alpha * T, a) || !ccd_collider<kGeo>(e, pr.collider_b, mb, alpha * T, b) ||
            !ccd_separation(pr.collider_a, pr.collider_b, pr.pair_class, a, b, d))
            return speculative_safe ? kCcdNone : kCcdUnsafe;
    }
    if (d <= tol || !speculative_safe) {
        // Within the tolerance: the time of impact. Otherwise the iterations ran
        // out with the pair separated up to alpha T: the segment ends there and
        // the pair is queried again from that state.
        toi = alpha * T;
        return kCcdImpact;
    }
    return kCcdNone;
}

// --------------------------------------------------------------- manifold

MRD_INL V3 stable_tangent(V3 n) {
    const V3 a = vabs(n);
    V3 ref;
    if (a.x <= a.y && a.x <= a.z) ref = V3{1.0f, 0.0f, 0.0f};
    else if (a.y <= a.z) ref = V3{0.0f, 1.0f, 0.0f};
    else ref = V3{0.0f, 0.0f, 1.0f};
    return normalize(cross(ref, n));
}

MRD_INL mr_float4 anchor_from_world(V3 bpos, Q4 rot, V3 x) {
    const V3 l = qrot_inv(rot, sub(x, bpos));
    return mr_float4{l.x, l.y, l.z, 0.0f};
}

// The value x of one of a pair's lanes: lane `from` (below 8) of this lane's eight.
template <class T> MRD_INL T group_get(T x, uint32_t lane, uint32_t from) { return wave_get(x, (lane & 56u) + from); }
MRD_INL uint32_t group_get(uint32_t x, uint32_t lane, uint32_t from) {
    return __float_as_uint(wave_get(__uint_as_float(x), (lane & 56u) + from));
}
// One bit per lane of this lane's eight.
MRD_INL uint32_t group_bits(bool b, uint32_t lane) {
    const unsigned long long m = __ballot(b);
    const uint32_t half = (lane & 32u) != 0u ? (uint32_t)(m >> 32) : (uint32_t)m;
    return (half >> (lane & 24u)) & 0xffu;
}

// One candidate point of a manifold, held by one lane.
struct ManifoldCandidate {
    bool valid;
    V3 a, b;        // local anchors
    float aw, bw;   // their unused fourth components, kept as read
    V3 world;
    float separation, drift;
    uint32_t fa, fb;
    MRD_INL unsigned long long feature() const { return ((unsigned long long)fa << 32u) | (unsigned long long)fb; }
};

// Manifold of active pair k from its raw contacts (in the staging records, as
// ContactSink left them) and its previous manifold, written over the staging
// records: eight lanes a pair, eight pairs at once. A manifold has at most
// twelve candidates: lane t of the eight holds raw contact t, the candidate it
// opens if it matches none, and (t < 4) the previous point t. Their index order,
// which the matching and the reduction follow, is previous points first, then
// opened ones.
//
// Matching is sequential in the raw contacts (a contact may match a point an
// earlier contact moved), but the tests it makes are not: whether contact k
// matches previous point i or contact j by feature or by distance is 24 bits per
// contact, found for all contacts at once, and the sequence then only picks bits.
// Sorting is by counted ranks; the greedy spread selection, only with more than
// four candidates, scans scores in rank order, the candidates first brought to
// the lanes of their ranks. Every comparison is the one the serial form makes,
// with its ties. The loops stay rolled: unrolled they spill 200 registers more.
//
// One lane a pair held candidates and contacts in private arrays: their dynamic
// indices made every access a scratch load, 217 K of a robot's 1154 K cycles a
// control step with two lanes at work. Measured: one robot 540 -> 500 us, 4096
// humanoids 3.29 -> 2.59 ms (2 steps), at residual 1e-5 50.5 -> 47.1 ms (20 steps).
// Candidates in rank order in the selection, and loops over the contacts there
// are: 1024 chain-and-boxes worlds 2.70 -> 2.63 ms, 1500 tree worlds 5.03 -> 4.91.
//
// All 64 lanes call it (spare groups with on = false).
MRD_INL void build_manifolds(const Env& e, uint32_t lane, uint32_t k, bool on, const MRManifoldHeaderC* old_h,
                             const MRManifoldPointC* old_p, uint32_t mcount_src, uint32_t& retained, uint32_t& fresh,
                             unsigned long long* fail) {
    const uint32_t t = lane & 7u;
    const MRWorldStepConfigC& cfg = e.a->cfg;
    const uint32_t compiled = e.active[k];
    const MRCompiledPairC pair = e.pairs[compiled];
    const MRShapeC& sa = e.shapes[pair.collider_a];
    const MRShapeC& sb = e.shapes[pair.collider_b];
    float* head = reinterpret_cast<float*>(e.stage_h + k);
    MRManifoldPointC* points = e.stage_p + (size_t)k * MR_MANIFOLD_POINT_CAPACITY;
    // raw contact t (lanes past the count read what the records held before)
    const float* raw = reinterpret_cast<const float*>(points) + 8u * t;
    const V3 raw_a{raw[0], raw[1], raw[2]}, raw_b{raw[3], raw[4], raw[5]};
    const uint32_t raw_fa = __float_as_uint(raw[6]), raw_fb = __float_as_uint(raw[7]);
    const float raw_sep = head[t];
    const V3 n = normalize(V3{head[8], head[9], head[10]});
    V3 pa_pos, pb_pos;
    Q4 pa_q, pb_q;
    body_pose(e, sa.body, pa_pos, pa_q);
    body_pose(e, sb.body, pb_pos, pb_q);
    Q4 ra, rb;
    const bool posed = checked_quat(pa_q, ra) & checked_quat(pb_q, rb);
    if (on && (!posed || !finite3(n) || dot(n, n) < 0.9999f)) {
        if (t == 0u) {
            report_failure(fail, k, MR_STEP_NONFINITE_RESULT, compiled);
            e.npts[k] = 0u;
        }
        on = false;
    }
    const uint32_t raw_count = on ? e.npts[k] : 0u;
    // ---- the pair's previous manifold
    const uint32_t key = pair.collider_a | (pair.collider_b << 16);
    uint32_t found = MR_INVALID_INDEX;
    for (uint32_t m0 = 0; m0 < mcount_src; m0 += 8u) {
        const uint32_t m = m0 + t;
        const uint32_t bits = group_bits(m < mcount_src && e.okey[m] == key, lane);
        if (found == MR_INVALID_INDEX && bits != 0u) found = m0 + (uint32_t)__builtin_ctz(bits);
    }
    const bool had = on && found != MR_INVALID_INDEX;
    const uint32_t mi = had ? found : 0u;
    const MRManifoldHeaderC oh = old_h[mi];
    const MRManifoldPointC op = old_p[(size_t)mi * MR_MANIFOLD_POINT_CAPACITY + (t & 3u)];
    const V3 on_w = normalize(qrot(ra, f3(oh.normal_and_age)));
    const bool compatible = had && oh.generations_and_flags[0] == sa.slot_generation &&
        oh.generations_and_flags[1] == sb.slot_generation && oh.pair_and_count[3] <= MR_MANIFOLD_POINT_CAPACITY &&
        finite3(on_w) && dot(on_w, n) >= cfg.manifold_normal_cosine;
    const V3 ot = qrot(ra, f3(oh.tangent_and_metric));
    const V3 transported = sub(ot, mul(dot(ot, n), n));
    ManifoldCandidate prev;
    {
        const V3 pa = add(pa_pos, qrot(ra, f3(op.local_anchor_a)));
        const V3 pb = add(pb_pos, qrot(rb, f3(op.local_anchor_b)));
        const V3 d = sub(pb, pa);
        prev.separation = dot(d, n);
        prev.drift = length(sub(d, mul(prev.separation, n)));
        prev.valid = compatible && t < 4u && t < oh.pair_and_count[3] &&
            !(prev.separation > cfg.manifold_breaking_separation || prev.drift > cfg.manifold_breaking_tangential);
        prev.a = f3(op.local_anchor_a);
        prev.b = f3(op.local_anchor_b);
        prev.aw = op.local_anchor_a.w;
        prev.bw = op.local_anchor_b.w;
        prev.world = mul(0.5f, add(pa, pb));
        prev.fa = op.feature_and_life[0];
        prev.fb = op.feature_and_life[1];
    }
    const uint32_t prev_life = op.feature_and_life[2] == 0xffffffffu ? 0xffffffffu : op.feature_and_life[2] + 1u;
    ManifoldCandidate own;  // raw contact t as a candidate
    {
        const mr_float4 la = anchor_from_world(pa_pos, ra, raw_a), lb = anchor_from_world(pb_pos, rb, raw_b);
        own.valid = false;
        own.a = f3(la);
        own.b = f3(lb);
        own.aw = 0.0f;
        own.bw = 0.0f;
        own.world = mul(0.5f, add(raw_a, raw_b));
        own.separation = raw_sep;
        own.drift = 0.0f;
        own.fa = raw_fa;
        own.fb = raw_fb;
    }
    // ---- which candidates contact t could match: bits 0-3 previous point i by
    // feature, 4-7 by distance, 8-15 contact j by feature, 16-23 by distance
    const uint32_t most = uniform_u32(wave_max_u32(raw_count));  // contacts j past it open no candidate
    const float merge = 2.0f * (cfg.manifold_merge_distance * cfg.manifold_merge_distance);
    uint32_t matches = 0u;
    const auto test = [&](const ManifoldCandidate& c, uint32_t from, uint32_t bit_f, uint32_t bit_d) {
        // fetched before any branch: a lane permutation reads active lanes only
        const uint32_t fa = group_get(c.fa, lane, from), fb = group_get(c.fb, lane, from);
        const bool f = fa == own.fa && fb == own.fb;
        const V3 da = sub(group_get(c.a, lane, from), own.a), db = sub(group_get(c.b, lane, from), own.b);
        matches |= (f ? 1u << bit_f : 0u) | (dot(da, da) + dot(db, db) <= merge ? 1u << bit_d : 0u);
    };
#pragma unroll 1
    for (uint32_t i = 0; i < 4u; ++i) test(prev, i, i, 4u + i);
#pragma unroll 1
    for (uint32_t j = 0; j < most; ++j) test(own, j, 8u + j, 16u + j);
    // ---- the matching sequence: each candidate remembers the last contact that
    // moved it (8: none yet; an opened one starts with its own)
    uint32_t prev_owner = 8u, own_owner = t;
    for (uint32_t c = 0; c < most; ++c) {
        const uint32_t mk = group_get(matches, lane, c);
        const uint32_t fr = mk >> 8u, dr = mk >> 16u;
        const bool pf = prev.valid && ((prev_owner < 8u ? fr >> prev_owner : mk >> t) & 1u) != 0u;
        const bool pd = prev.valid && ((prev_owner < 8u ? dr >> prev_owner : mk >> (4u + t)) & 1u) != 0u;
        const bool of = own.valid && ((fr >> own_owner) & 1u) != 0u;
        const bool od = own.valid && ((dr >> own_owner) & 1u) != 0u;
        const uint32_t by_feature = group_bits(pf, lane) | (group_bits(of, lane) << 8);
        const uint32_t by_distance = group_bits(pd, lane) | (group_bits(od, lane) << 8);
        const uint32_t hits = by_feature != 0u ? by_feature : by_distance;
        const uint32_t pick = hits != 0u ? (uint32_t)__builtin_ctz(hits) : 8u + c;
        if (c < raw_count) {
            if (pick == t) prev_owner = c;
            if (pick == 8u + t) {
                own.valid = true;
                own_owner = c;
            }
        }
    }
    const uint32_t prev_bits = group_bits(prev.valid, lane), own_bits = group_bits(own.valid, lane);
    if (t == 0u) {
        retained += (uint32_t)__builtin_popcount(prev_bits);
        fresh += (uint32_t)__builtin_popcount(own_bits);
    }
    // ---- moved candidates take the contact's geometry
    const ManifoldCandidate contact = own;
    const auto take = [&](ManifoldCandidate& c, uint32_t owner) {
        const uint32_t from = owner < 8u ? owner : t;
        const V3 a = group_get(contact.a, lane, from), b = group_get(contact.b, lane, from);
        const V3 w = group_get(contact.world, lane, from);
        const float sep = group_get(contact.separation, lane, from);
        const uint32_t fa = group_get(contact.fa, lane, from), fb = group_get(contact.fb, lane, from);
        if (owner < 8u) {
            c.a = a;
            c.b = b;
            c.aw = 0.0f;
            c.bw = 0.0f;
            c.world = w;
            c.separation = sep;
            c.drift = 0.0f;
            c.fa = fa;
            c.fb = fb;
        }
    };
    take(prev, prev_owner);
    take(own, own_owner);
    const uint32_t prev_flags = prev_owner < 8u ? 0u : op.feature_and_life[3];
    uint32_t count = (uint32_t)__builtin_popcount(prev_bits) + (uint32_t)__builtin_popcount(own_bits);
    // ---- ranks by separation, then feature, then index
    uint32_t prev_rank = 0u, own_rank = 0u;
    const auto rank_against = [&](const ManifoldCandidate& c, uint32_t from, uint32_t index) {
        const bool valid = ((index < 4u ? prev_bits : own_bits) >> from & 1u) != 0u;
        const float sep = group_get(c.separation, lane, from);
        const uint32_t fa = group_get(c.fa, lane, from), fb = group_get(c.fb, lane, from);
        const unsigned long long f = ((unsigned long long)fa << 32u) | (unsigned long long)fb;
        const auto before = [&](const ManifoldCandidate& me, uint32_t my_index) {
            if (sep != me.separation) return sep < me.separation;
            return f < me.feature() || (f == me.feature() && index < my_index);
        };
        prev_rank += valid && before(prev, t) ? 1u : 0u;
        own_rank += valid && before(own, 4u + t) ? 1u : 0u;
    };
#pragma unroll 1
    for (uint32_t i = 0; i < 4u; ++i) rank_against(prev, i, i);
#pragma unroll 1
    for (uint32_t j = 0; j < most; ++j) rank_against(own, j, 4u + j);
    bool prev_keep = prev.valid, own_keep = own.valid;
    // ---- more than four: greedy spread selection from the deepest point
    if (wave_any(count > MR_MANIFOLD_POINT_CAPACITY)) {
        // sorted position -> candidate index, one nibble each, the same in all eight lanes
        unsigned long long order = (prev.valid ? (unsigned long long)t << (4u * prev_rank) : 0ull) |
                                   (own.valid ? (unsigned long long)(4u + t) << (4u * own_rank) : 0ull);
        uint32_t lo = (uint32_t)order, hi = (uint32_t)(order >> 32);
#pragma unroll
        for (uint32_t d = 1; d < 8u; d <<= 1) {
            lo |= group_get(lo, lane, t ^ d);
            hi |= group_get(hi, lane, t ^ d);
        }
        order = ((unsigned long long)hi << 32) | lo;
        // from here on lane t holds the candidates of positions t and 8 + t % 4
        const uint32_t low = (uint32_t)(order >> (4u * t)) & 0xfu, high = (uint32_t)(order >> (32u + 4u * (t & 3u))) & 0xfu;
        const auto at = [&](auto p, auto o, uint32_t index) {
            const auto x = group_get(p, lane, index & 3u);
            const auto y = group_get(o, lane, (index - 4u) & 7u);
            return index < 4u ? x : y;
        };
        const V3 low_world = at(prev.world, own.world, low), high_world = at(prev.world, own.world, high);
        const uint32_t low_fa = at(prev.fa, own.fa, low), low_fb = at(prev.fb, own.fb, low);
        const uint32_t high_fa = at(prev.fa, own.fa, high), high_fb = at(prev.fb, own.fb, high);
        const uint32_t longest = uniform_u32(wave_max_u32(count));
        uint32_t selected = 1u, chosen = 0u, nch = 1u;
        const V3 w0 = group_get(low_world, lane, 0u);
        V3 w1 = w0, w2 = w0;
#pragma unroll 1
        for (uint32_t stage = 1; stage < MR_MANIFOLD_POINT_CAPACITY; ++stage) {
            const auto score_of = [&](V3 w) {
                const auto spread = [&](V3 from) {
                    const V3 d = sub(w, from);
                    const V3 tn = sub(d, mul(dot(d, n), n));
                    return dot(tn, tn);
                };
                if (stage == 1u) return spread(w0);
                if (stage == 2u) return fabs_(dot(cross(sub(w1, w0), sub(w, w0)), n));
                float score = fmind(__builtin_inff(), spread(w0));
                if (nch > 1u) score = fmind(score, spread(w1));
                if (nch > 2u) score = fmind(score, spread(w2));
                return score;
            };
            const float low_score = score_of(low_world), high_score = score_of(high_world);
            uint32_t best = MR_INVALID_INDEX;
            float best_score = -1.0f;
            unsigned long long best_feature = ~0ull;
#pragma unroll 1
            for (uint32_t i = 0; i < longest; ++i) {
                const float score = group_get(i < 8u ? low_score : high_score, lane, i & 7u);
                const unsigned long long f =
                    ((unsigned long long)group_get(i < 8u ? low_fa : high_fa, lane, i & 7u) << 32u) |
                    (unsigned long long)group_get(i < 8u ? low_fb : high_fb, lane, i & 7u);
                const bool free = i < count && ((selected >> i) & 1u) == 0u;
                if (free && (score > best_score + 1.0e-12f ||
                             (fabs_(score - best_score) <= 1.0e-12f && f < best_feature))) {
                    best = i;
                    best_score = score;
                    best_feature = f;
                }
            }
            const bool any = best != MR_INVALID_INDEX;
            const uint32_t from = any ? best : 0u;
            const V3 wl = group_get(low_world, lane, from & 7u), wh = group_get(high_world, lane, from & 3u);
            const V3 w = from < 8u ? wl : wh;
            if (any) {
                if (nch == 1u) w1 = w;
                if (nch == 2u) w2 = w;
                chosen |= best << (4u * nch);
                ++nch;
                selected |= 1u << best;
            }
        }
        if (count > MR_MANIFOLD_POINT_CAPACITY) {
            count = nch;
            prev_keep = false;
            own_keep = false;
            uint32_t prev_pick = 0u, own_pick = 0u;
            for (uint32_t q = 0; q < nch; ++q) {
                const uint32_t position = (chosen >> (4u * q)) & 0xfu;
                if (prev.valid && prev_rank == position) {
                    prev_keep = true;
                    prev_pick = q;
                }
                if (own.valid && own_rank == position) {
                    own_keep = true;
                    own_pick = q;
                }
            }
            prev_rank = prev_pick;
            own_rank = own_pick;
        }
    }
    // ---- output order: by feature, ties in the order of the ranks (or picks)
    const uint32_t prev_kept = group_bits(prev_keep, lane), own_kept = group_bits(own_keep, lane);
    uint32_t prev_pos = 0u, own_pos = 0u;
    const auto place_against = [&](const ManifoldCandidate& c, uint32_t rank, uint32_t kept, uint32_t from) {
        const bool valid = (kept >> from & 1u) != 0u;
        const uint32_t r = group_get(rank, lane, from);
        const uint32_t fa = group_get(c.fa, lane, from), fb = group_get(c.fb, lane, from);
        const unsigned long long f = ((unsigned long long)fa << 32u) | (unsigned long long)fb;
        prev_pos += valid && (f < prev.feature() || (f == prev.feature() && r < prev_rank)) ? 1u : 0u;
        own_pos += valid && (f < own.feature() || (f == own.feature() && r < own_rank)) ? 1u : 0u;
    };
#pragma unroll 1
    for (uint32_t i = 0; i < 4u; ++i) place_against(prev, prev_rank, prev_kept, i);
#pragma unroll 1
    for (uint32_t j = 0; j < most; ++j) place_against(own, own_rank, own_kept, j);
    float metric = 0.0f;
    if (prev_keep) metric = fmaxd(metric, fmaxd(fmaxd(prev.separation, 0.0f), prev.drift));
    if (own_keep) metric = fmaxd(metric, fmaxd(fmaxd(own.separation, 0.0f), own.drift));
#pragma unroll
    for (uint32_t d = 1; d < 8u; d <<= 1) metric = fmaxd(metric, group_get(metric, lane, t ^ d));
    V3 tangent = transported;
    if (!compatible || !finite3(tangent) || dot(tangent, tangent) <= 1.0e-12f) tangent = stable_tangent(n);
    else tangent = normalize(tangent);
    if (!on) return;
    const auto store = [&](uint32_t pos, const ManifoldCandidate& c, mr_float4 impulses, uint32_t life, uint32_t flags) {
        if (pos >= MR_MANIFOLD_POINT_CAPACITY) return;
        MRManifoldPointC o;
        o.local_anchor_a = mr_float4{c.a.x, c.a.y, c.a.z, c.aw};
        o.local_anchor_b = mr_float4{c.b.x, c.b.y, c.b.z, c.bw};
        o.impulses = impulses;
        o.feature_and_life[0] = c.fa;
        o.feature_and_life[1] = c.fb;
        o.feature_and_life[2] = life;
        o.feature_and_life[3] = flags;
        points[pos] = o;
    };
    const mr_float4 zero4{0.0f, 0.0f, 0.0f, 0.0f};
    if (prev_keep) store(prev_pos, prev, op.impulses, prev_life, prev_flags);
    if (own_keep) store(own_pos, own, zero4, 0u, 0u);
    if (t < MR_MANIFOLD_POINT_CAPACITY && t >= count) {
        ManifoldCandidate none;
        none.a = none.b = V3{0.0f, 0.0f, 0.0f};
        none.aw = none.bw = 0.0f;
        none.fa = none.fb = 0u;
        store(t, none, zero4, 0u, 0u);
    }
    if (t == 0u) {
        MRManifoldHeaderC o;
        o.pair_and_count[0] = e.env;
        o.pair_and_count[1] = pair.collider_a;
        o.pair_and_count[2] = pair.collider_b;
        o.pair_and_count[3] = count;
        o.generations_and_flags[0] = sa.slot_generation;
        o.generations_and_flags[1] = sb.slot_generation;
        o.generations_and_flags[2] = 0u;
        o.generations_and_flags[3] = 0u;
        const V3 ln = qrot_inv(ra, n), lt = qrot_inv(ra, tangent);
        o.normal_and_age = mr_float4{ln.x, ln.y, ln.z, compatible ? fmind(oh.normal_and_age.w + 1.0f, 65535.0f) : 0.0f};
        o.tangent_and_metric = mr_float4{lt.x, lt.y, lt.z, metric};
        e.stage_h[k] = o;
        e.npts[k] = count;
    }
}

// ------------------------------------------------------------ cone solve

// Normal clamp (and the optional maximum normal impulse), then radial scaling
// of the tangents onto the elliptic cone (MetalWorldContact.metal:482-509).
MRD_INL void project_cone(float lam[3], float mu_u, float mu_v, float max_normal) {
    lam[0] = fmaxd(lam[0], 0.0f);
    if (max_normal > 0.0f) lam[0] = fmind(lam[0], max_normal);
    const float lu = mu_u * lam[0];
    const float lv = mu_v * lam[0];
    if (!(lu > 0.0f) || !(lv > 0.0f)) {
        lam[1] = 0.0f;
        lam[2] = 0.0f;
        return;
    }
    const float ns = (lam[1] * lam[1]) / (lu * lu) + (lam[2] * lam[2]) / (lv * lv);
    if (ns > 1.0f) {
        const float s = 1.0f / sqrt_rn(ns);
        lam[1] *= s;
        lam[2] *= s;
    }
}

// One contact's block update from its relative velocity: cand = the projected
// impulse, and the sweep's largest change. False when any of it is not finite
// (the results are meaningless then).
MRD_INL bool block_update(const HotConstraint& sb, const float rel[3], float lam0, float lam1, float lam2,
                          float max_normal, float cand[3], float& sweep_delta) {
    const float lamc[3] = {lam0, lam1, lam2};
    // the tangent rows' stored target and regularisation are +0
    const float tgt[3] = {sb.target0, 0.0f, 0.0f}, reg[3] = {sb.reg0, 0.0f, 0.0f};
    float rhs[3];
    for (int r = 0; r < 3; ++r) rhs[r] = (tgt[r] - rel[r]) - reg[r] * lamc[r];
    for (int r = 0; r < 3; ++r) {
        cand[r] = lamc[r];
        for (int q = 0; q < 3; ++q) cand[r] += sb.winv[3 * r + q] * rhs[q];
    }
    project_cone(cand, sb.mu_u, sb.mu_v, max_normal);
    const float d0 = cand[0] - lam0, d1 = cand[1] - lam1, d2 = cand[2] - lam2;
    sweep_delta = fmaxd(sweep_delta, fmaxd(fabs_(d0), fmaxd(fabs_(d1), fabs_(d2))));
    return isfin(cand[0]) & isfin(cand[1]) & isfin(cand[2]) & isfin(d0) & isfin(d1) & isfin(d2);
}

MRD_INL bool invert3x3(const float m[3][3], float inv[9]) {
    float scale = 0.0f;
    for (int rr = 0; rr < 3; ++rr)
        for (int cc = 0; cc < 3; ++cc) {
            if (!isfin(m[rr][cc])) return false;
            scale = fmaxd(scale, fabs_(m[rr][cc]));
        }
    if (!(scale > kMatrixFloor)) return false;
    float g[3][3];
    for (int rr = 0; rr < 3; ++rr)
        for (int cc = 0; cc < 3; ++cc) {
            g[rr][cc] = 0.5f * (m[rr][cc] + m[cc][rr]) / scale;
            if (rr == cc) g[rr][cc] += kContactRegularization;
        }
    const float c00 = g[1][1] * g[2][2] - g[1][2] * g[2][1];
    const float c01 = g[1][2] * g[2][0] - g[1][0] * g[2][2];
    const float c02 = g[1][0] * g[2][1] - g[1][1] * g[2][0];
    const float det = g[0][0] * c00 + g[0][1] * c01 + g[0][2] * c02;
    if (!(det > kMatrixFloor) || !isfin(det)) return false;
    const float rcp = 1.0f / (det * scale);
    inv[0] = c00 * rcp;
    inv[1] = (g[0][2] * g[2][1] - g[0][1] * g[2][2]) * rcp;
    inv[2] = (g[0][1] * g[1][2] - g[0][2] * g[1][1]) * rcp;
    inv[3] = c01 * rcp;
    inv[4] = (g[0][0] * g[2][2] - g[0][2] * g[2][0]) * rcp;
    inv[5] = (g[0][2] * g[1][0] - g[0][0] * g[1][2]) * rcp;
    inv[6] = c02 * rcp;
    inv[7] = (g[0][1] * g[2][0] - g[0][0] * g[2][1]) * rcp;
    inv[8] = (g[0][0] * g[1][1] - g[0][1] * g[1][0]) * rcp;
    for (int k = 0; k < 9; ++k)
        if (!isfin(inv[k])) return false;
    return true;
}

MRD_INL V3 inv_inertia_mul(const MRBodyStateC& b, V3 x) {
    return V3{dot(f3(b.inverse_inertia_world_row0), x), dot(f3(b.inverse_inertia_world_row1), x),
              dot(f3(b.inverse_inertia_world_row2), x)};
}

MRD_INL V3 scene_response(const MRBodyStateC& b, V3 x, V3 d) {
    const V3 lever = sub(x, f3(b.position));
    const V3 dw = inv_inertia_mul(b, cross(lever, d));
    return add(mul(b.linear_velocity_inv_mass.w, d), cross(dw, lever));
}

MRD_INL V3 scene_point_velocity(const MRBodyStateC& b, V3 x) {
    return add(f3(b.linear_velocity_inv_mass), cross(f3(b.angular_velocity), sub(x, f3(b.position))));
}

MRD_INL void apply_scene_impulse(MRBodyStateC& b, V3 x, V3 imp) {
    const V3 lever = sub(x, f3(b.position));
    const V3 dv = mul(b.linear_velocity_inv_mass.w, imp);
    b.linear_velocity_inv_mass.x += dv.x;
    b.linear_velocity_inv_mass.y += dv.y;
    b.linear_velocity_inv_mass.z += dv.z;
    const V3 dw = inv_inertia_mul(b, cross(lever, imp));
    b.angular_velocity.x += dw.x;
    b.angular_velocity.y += dw.y;
    b.angular_velocity.z += dw.z;
}

MRD_INL V3 hot_dir(const HotConstraint& h, int r) { return V3{h.dir[3 * r], h.dir[3 * r + 1], h.dir[3 * r + 2]}; }

// Point velocities of a constraint's scene endpoints at the contact point
// (zero for links and static bodies).
MRD_INL void scene_point_velocities(const Env& e, uint32_t kind, uint32_t ba, uint32_t bb, V3 x, V3& va, V3& vb) {
    const V3 zero{0.0f, 0.0f, 0.0f};
    va = (kind & mr::kHotDynamicA) != 0u ? scene_point_velocity(e.scene[ba - e.nlinks], x) : zero;
    vb = (kind & mr::kHotDynamicB) != 0u ? scene_point_velocity(e.scene[bb - e.nlinks], x) : zero;
}

// Relative velocity of one constraint row: the articulation part `art_dot`
// (J v, already folded across the DoF lanes) plus the point velocity of a
// dynamic body B minus that of a dynamic body A (static and link endpoints
// add nothing), in the oracle's order.
MRD_INL float rel_row(uint32_t kind, V3 d, V3 va, V3 vb, float art_dot) {
    float rel = art_dot;
    if ((kind & mr::kHotDynamicB) != 0u) rel = rel + dot(d, vb);
    if ((kind & mr::kHotDynamicA) != 0u) rel = rel - dot(d, va);
    return rel;
}


// ------------------------------------------------ contact schedule
//
// An ordered sweep updates the contacts in index order, and an update reads and
// writes only the velocities of its own nodes: the articulation and its dynamic
// scene bodies. Contacts without a common node therefore commute, and any order
// that keeps the index order at every node gives the same bits. A contact's level
// is one more than the largest level of the earlier contacts at its nodes; the
// contacts of a level share no node, so those between scene bodies run one per
// lane, and the at most one articulated contact of a level runs on the whole wave
// (its dot products are folds over the DoF lanes). A pile of 20 boxes still
// landing has about 58 contacts (2.5 of them articulated) in 7 levels, a settled
// one 93. An update is a serial chain of
// LDS reads and about 250 instructions whatever the number of active lanes, so the
// levels, not the contacts, set the sweep's time. Measured, 2 control steps: 1024
// chain-and-boxes worlds 6.00 -> 2.90 ms, 1500 random trees 13.2 -> 5.95 ms, 300
// chain worlds with hybrid CCD 8.39 -> 6.59 ms (one contact at a time before).
// Contacts that all join the articulation to static geometry are one chain and
// take no schedule.

// A scene body's part in the sweeps, five float4 at a stride of 20 words, so that
// 16 bodies' reads of one float4 touch distinct LDS banks (the 128-byte body record
// puts every body on the same ones): {lin, 1/m}, {ang, pos.x},
// {pos.y, pos.z, I0, I1}, {I2 .. I5}, {I6, I7, I8, -}; I = world inverse inertia rows.
constexpr uint32_t kSolverBodyVectors = 5u;
// The leading words of a HotConstraint that the unscheduled sweeps read: winv, target0, reg0, mu_u, mu_v.
constexpr uint32_t kBlockWords = 13u;
static_assert(offsetof(HotConstraint, mu_v) == (kBlockWords - 1u) * 4u, "leading words");

MRD_INL void load_solver_body(const Env& e, uint32_t s) {
    const MRBodyStateC& b = e.scene[s];
    float4* o = e.sbody + s * kSolverBodyVectors;
    const mr_float4 &r0 = b.inverse_inertia_world_row0, &r1 = b.inverse_inertia_world_row1,
                    &r2 = b.inverse_inertia_world_row2;
    o[0] = make_float4(b.linear_velocity_inv_mass.x, b.linear_velocity_inv_mass.y, b.linear_velocity_inv_mass.z,
                       b.linear_velocity_inv_mass.w);
    o[1] = make_float4(b.angular_velocity.x, b.angular_velocity.y, b.angular_velocity.z, b.position.x);
    o[2] = make_float4(b.position.y, b.position.z, r0.x, r0.y);
    o[3] = make_float4(r0.z, r1.x, r1.y, r1.z);
    o[4] = make_float4(r2.x, r2.y, r2.z, 0.0f);
}

MRD_INL void store_solver_body(const Env& e, uint32_t s) {
    MRBodyStateC& b = e.scene[s];
    const float4 l = e.sbody[s * kSolverBodyVectors], a = e.sbody[s * kSolverBodyVectors + 1u];
    b.linear_velocity_inv_mass.x = l.x;
    b.linear_velocity_inv_mass.y = l.y;
    b.linear_velocity_inv_mass.z = l.z;
    b.angular_velocity.x = a.x;
    b.angular_velocity.y = a.y;
    b.angular_velocity.z = a.z;
}

// scene_point_velocity and apply_scene_impulse on a solver body.
MRD_INL V3 solver_point_velocity(const float4* b, V3 x) {
    const float4 l = b[0], a = b[1], p = b[2];
    return add(V3{l.x, l.y, l.z}, cross(V3{a.x, a.y, a.z}, sub(x, V3{a.w, p.x, p.y})));
}

MRD_INL void solver_apply_impulse(float4* b, V3 x, V3 imp) {
    float4 l = b[0], a = b[1];
    const float4 p = b[2], i0 = b[3], i1 = b[4];
    const V3 lever = sub(x, V3{a.w, p.x, p.y});
    const V3 dv = mul(l.w, imp);
    l.x += dv.x;
    l.y += dv.y;
    l.z += dv.z;
    const V3 t = cross(lever, imp);
    a.x += dot(V3{p.z, p.w, i0.x}, t);
    a.y += dot(V3{i0.y, i0.z, i0.w}, t);
    a.z += dot(V3{i1.x, i1.y, i1.z}, t);
    b[0] = l;
    b[1] = a;
}

// Builds the schedule: e.sord gets the contacts between scene bodies sorted by level (index order
// within one), then the articulated contacts in index order; e.resid gets one word per level and
// one behind the last: the level's first entry in e.sord | (its articulated contact + 1) << 16.
// Returns the number of levels; the total of the last word is the number of contacts between
// scene bodies. Needs nscene < 64 (MR_MAX_BODIES counts the links too).
//
// The schedule takes no LDS of its own at a large contact capacity c: its 4 (c + 1) bytes of level
// words, 2 c of order and, while it is built, 2 c of the contacts' levels lie in the residual
// arrays' 8 c + 4, which are written when it is no longer read (the first half with the last
// sweep done, the second after the pass that still reads e.sord).
MRD_INL uint32_t schedule_contacts(const Env& e, uint32_t lane, uint32_t ncons, uint32_t ccap) {
    uint32_t* pack = reinterpret_cast<uint32_t*>(e.resid);
    uint16_t* lev = e.sord + ccap;
    uint32_t body_level = 0u;  // lane s: the first level scene body s is free at
    uint32_t art_level = 0u, levels = 0u;
    for (uint32_t base = 0; base < ncons; base += kLanes) {
        const uint32_t n = ncons - base < kLanes ? ncons - base : kLanes;
        const uint32_t pairs = lane < n ? e.cpair[base + lane] : 0u;
        uint32_t mine = 0u;
        for (uint32_t i = 0; i < n; ++i) {
            const uint32_t p = read_lane(pairs, i);
            const bool art = ((p >> 16) & mr::kHotArticulated) != 0u;
            const bool da = ((p >> 16) & mr::kHotDynamicA) != 0u, db = ((p >> 16) & mr::kHotDynamicB) != 0u;
            const uint32_t a = da ? (p & 0xffu) - e.nlinks : 0u, b = db ? ((p >> 8) & 0xffu) - e.nlinks : 0u;
            const uint32_t la = da ? read_lane(body_level, a) : 0u, lb = db ? read_lane(body_level, b) : 0u;
            uint32_t l = art ? art_level : 0u;
            l = l > la ? l : la;
            l = l > lb ? l : lb;
            mine = lane == i ? l : mine;
            ++l;
            art_level = art ? l : art_level;
            body_level = ((da && lane == a) || (db && lane == b)) ? l : body_level;
            levels = levels > l ? levels : l;
        }
        if (lane < n) lev[base + lane] = (uint16_t)mine;
    }
    __syncthreads();
    uint32_t at = 0u;
    for (uint32_t l = 0; l < levels; ++l) {
        const uint32_t start = at;
        uint32_t art_contact = 0u;
        for (uint32_t base = 0; base < ncons; base += kLanes) {
            const uint32_t c = base + lane;
            const bool in = c < ncons && lev[c] == l;
            const bool art = in && ((e.cpair[c] >> 16) & mr::kHotArticulated) != 0u;
            const unsigned long long bal = __ballot(in && !art), abal = __ballot(art);
            if (in && !art) e.sord[at + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)c;
            at += (uint32_t)__popcll(bal);
            if (abal != 0ull) art_contact = base + (uint32_t)__builtin_ctzll(abal) + 1u;
        }
        if (lane == 0u) pack[l] = start | (art_contact << 16);
    }
    if (lane == 0u) pack[levels] = at;
    for (uint32_t base = 0; base < ncons; base += kLanes) {
        const uint32_t c = base + lane;
        const bool art = c < ncons && ((e.cpair[c] >> 16) & mr::kHotArticulated) != 0u;
        const unsigned long long abal = __ballot(art);
        if (art) e.sord[at + (uint32_t)__popcll(abal & ((1ull << lane) - 1ull))] = (uint16_t)c;
        at += (uint32_t)__popcll(abal);
    }
    __syncthreads();
    return levels;
}

// Optional per-stage shader-clock counters: lane 0 adds each stage's elapsed
// cycles straight into the environment's global counters (no register array
// held across the kernel when profiling is off).
// ------------------------------------------------ relaxed block Jacobi
// (mrWorldWave32SolvePacket, MetalWorldContact.metal:6142-7213). Articulated
// dot products are serial in DoF order and sums over contacts run in
// constraint order; contacts of other islands add exact zeros, so these are
// the island sums.

// Velocity change at point xc of scene body b from a unit impulse along d at
// point xj (the scene part of typedNormalCrossContactResponse, :6740-6784).
MRD_INL V3 scene_cross_response(const MRBodyStateC& b, V3 xc, V3 xj, V3 d) {
    const V3 dw = inv_inertia_mul(b, cross(sub(xj, f3(b.position)), d));
    return add(mul(b.linear_velocity_inv_mass.w, d), cross(dw, sub(xc, f3(b.position))));
}

// sum_k x[k] * y[k] added in index order (the order the oracle uses), with
// the loads of eight terms issued before their products are added, so that
// their memory latencies overlap instead of following one another.
MRD_INL float serial_dot(const float* x, const float* y, uint32_t n) {
    float a = 0.0f;
    uint32_t k = 0;
    for (; k + 8u <= n; k += 8u) {
        float xs[8], ys[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            xs[i] = x[k + i];
            ys[i] = y[k + i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) a = a + xs[i] * ys[i];
    }
    for (; k < n; ++k) a = a + x[k] * y[k];
    return a;
}

// W_nn(c, j): normal velocity at contact c per unit normal impulse of contact j.
MRD_INL float jacobi_normal_cross(const Env& e, uint32_t c, uint32_t j, uint32_t mnv) {
    const uint32_t pc = e.cpair[c], pj = e.cpair[j];
    float w = 0.0f;
    if (((pc >> 16) & mr::kHotArticulated) != 0u && ((pj >> 16) & mr::kHotArticulated) != 0u) {
        w = serial_dot(e.jrow + (size_t)c * 3u * mnv, e.resp + (size_t)j * 3u * mnv, e.nv);
    }
    const uint32_t cb[2] = {pc & 0xffu, (pc >> 8) & 0xffu}, jb[2] = {pj & 0xffu, (pj >> 8) & 0xffu};
    for (int x = 0; x < 2; ++x) {
        if (!is_dynamic_scene(e, cb[x])) continue;
        for (int y = 0; y < 2; ++y) {
            if (jb[y] != cb[x]) continue;
            const HotConstraint& hc = e.hot[c];
            const HotConstraint& hj = e.hot[j];
            const float t = dot(hot_dir(hc, 0), scene_cross_response(e.scene[cb[x] - e.nlinks],
                                                                     V3{hc.point[0], hc.point[1], hc.point[2]},
                                                                     V3{hj.point[0], hj.point[1], hj.point[2]},
                                                                     hot_dir(hj, 0)));
            w = (x == y) ? w + t : w - t;
        }
    }
    return w;
}

// All impulse deltas of e.jdelta at once: a DoF lane sums its responses in
// constraint order and applies the sum when any response touches it; a scene
// lane accumulates linear and angular impulse over its contacts and applies
// them once (:6858-6990).
MRD_INL void jacobi_apply(Env& e, uint32_t lane, uint32_t ncons, uint32_t mnv, bool dof_lane, float& vj) {
    const float* jd = e.jdelta;
    if (dof_lane) {
        float vd = 0.0f;
        bool part = false;
        for (uint32_t c = 0; c < ncons; ++c) {
            if (((e.cpair[c] >> 16) & mr::kHotArticulated) == 0u) continue;
            const float* rb = e.resp + (size_t)c * 3u * mnv + lane;
            const float r0 = rb[0], r1 = rb[mnv], r2 = rb[2u * mnv];
            part = part || r0 != 0.0f || r1 != 0.0f || r2 != 0.0f;
            vd = vd + ((r0 * jd[3u * c] + r1 * jd[3u * c + 1u]) + r2 * jd[3u * c + 2u]);
        }
        if (part) vj = vj + vd;
    }
    for (uint32_t s = lane; s < e.nscene; s += kLanes) {
        const uint32_t b = e.nlinks + s;
        if (!is_dynamic_scene(e, b)) continue;
        MRBodyStateC st = e.scene[s];
        V3 lin{0.0f, 0.0f, 0.0f}, ang{0.0f, 0.0f, 0.0f};
        bool touched = false;
        for (uint32_t c = 0; c < ncons; ++c) {
            const uint32_t pr = e.cpair[c];
            if ((pr & 0xffu) != b && ((pr >> 8) & 0xffu) != b) continue;
            touched = true;
            const HotConstraint& hk = e.hot[c];
            const float* d = jd + 3u * c;
            const V3 imp = add(add(mul(d[0], hot_dir(hk, 0)), mul(d[1], hot_dir(hk, 1))), mul(d[2], hot_dir(hk, 2)));
            const V3 lever = sub(V3{hk.point[0], hk.point[1], hk.point[2]}, f3(st.position));
            if (hk.body_a == b) {
                lin = sub(lin, imp);
                ang = add(ang, cross(lever, neg(imp)));
            }
            if (hk.body_b == b) {
                lin = add(lin, imp);
                ang = add(ang, cross(lever, imp));
            }
        }
        if (!touched) continue;
        const V3 dv = mul(st.linear_velocity_inv_mass.w, lin);
        st.linear_velocity_inv_mass.x += dv.x;
        st.linear_velocity_inv_mass.y += dv.y;
        st.linear_velocity_inv_mass.z += dv.z;
        const V3 dw = inv_inertia_mul(st, ang);
        st.angular_velocity.x += dw.x;
        st.angular_velocity.y += dw.y;
        st.angular_velocity.z += dw.z;
        e.scene[s] = st;
    }
}

struct StageClock {
    unsigned long long* out;
    unsigned long long last;
    MRD_INL void init(unsigned long long* o, uint32_t lane) {
        out = lane == 0u ? o : nullptr;
        last = out != nullptr ? (unsigned long long)clock64() : 0ull;
    }
    MRD_INL void mark(uint32_t stage) {
        if (out == nullptr) return;
        const unsigned long long now = (unsigned long long)clock64();
        out[stage] += now - last;
        last = now;
    }
};

} // namespace

// ------------------------------------------------ learned warm start

static_assert(mr::kMlpTileLdsBytes == mr::kMlpLdsBytes, "MLP tile LDS size");
static_assert(mr::kMlpTileLdsBytes >= 4u * mr::kMaxConstraints, "a second attempt's residual terms fit the MLP tile");
// Normalized features beyond this many training standard deviations keep the
// plain warm start.
constexpr float kMlpFeatureBound = 8.0f;

// Features of constraint c at the start of its cone solve: normal relative
// velocity (J v_free, the evaluation's staged row), penetration depth, the
// Euclidean norms of the normal and tangent Jacobian rows (articulated DoFs
// plus the twist coordinates (dir, r x dir) of each dynamic scene endpoint)
// and the projected previous-step impulse the plain path warm-starts from.
MRD_INL void contact_features(const Env& e, uint32_t c, uint32_t mnv, float f[mr::kMlpIn]) {
    const HotConstraint& hk = e.hot[c];
    const ColdConstraint& ck = e.cold[c];
    const uint32_t kind = e.cpair[c] >> 16;
    f[0] = hk.stage[0];
    f[1] = -ck.separation;
    const V3 x{hk.point[0], hk.point[1], hk.point[2]};
    for (int r = 0; r < 3; ++r) {
        float s2 = 0.0f;
        if ((kind & mr::kHotArticulated) != 0u) {
            const float* row = e.jrow + ((size_t)c * 3u + (uint32_t)r) * mnv;
            for (uint32_t j = 0; j < e.nv; ++j) s2 += row[j] * row[j];
        }
        const V3 d = hot_dir(hk, r);
        if ((kind & mr::kHotDynamicA) != 0u) {
            const V3 t = cross(sub(x, f3(e.scene[hk.body_a - e.nlinks].position)), d);
            s2 += dot(d, d) + dot(t, t);
        }
        if ((kind & mr::kHotDynamicB) != 0u) {
            const V3 t = cross(sub(x, f3(e.scene[hk.body_b - e.nlinks].position)), d);
            s2 += dot(d, d) + dot(t, t);
        }
        f[2 + r] = sqrt_rn(s2);
    }
    f[5] = e.lam[3u * c];
    f[6] = e.lam[3u * c + 1u];
    f[7] = e.lam[3u * c + 2u];
}

MRD_INL mr::MlpView mlp_view(const MRMlpWeightsC& w) {
    mr::MlpView m;
    m.w1 = reinterpret_cast<const __bf16*>(w.w1);
    m.b1 = w.b1;
    m.w2 = reinterpret_cast<const __bf16*>(w.w2);
    m.b2 = w.b2;
    m.w3 = reinterpret_cast<const __bf16*>(w.w3);
    m.b3 = w.b3;
    m.in_shift = w.in_shift;
    m.in_scale = w.in_scale;
    m.out_scale = w.out_scale;
    return m;
}

// Features of every constraint, 16 at a time: written to `samples` (the
// environment's capture rows, or null) and, with `infer`, run through the
// MLP, which predicts the correction to the previous-step impulse:
// lambda = lambda_prev + out_scale * y_hat, projected onto the cone. The
// prediction replaces the plain warm start (kept in e.mlp_lam, as are the
// scene bodies, for the fallback) when some component of the correction
// exceeds the weights' min_correction, unless a normalized feature lies
// beyond kMlpFeatureBound (outside what the network was trained on) or the
// result is not finite; otherwise the warm start stays untouched, bit for bit.
// Returns whether any warm start was replaced. Uniform in `infer`; all 64
// lanes must be active.
MRD_INL bool mlp_warm_start(const Env& e, uint32_t lane, uint32_t ncons, uint32_t mnv, bool infer, float* samples) {
    const mr::MlpLds s = mr::mlp_lds(e.mlp_lds);
    const mr::MlpView m = mlp_view(e.a->mlp);
    if (infer) {
        for (uint32_t i = lane; i < 3u * ncons; i += kLanes) e.mlp_lam[i] = e.lam[i];
        for (uint32_t b = lane; b < e.nscene; b += kLanes) e.mlp_scene[b] = e.scene[b];
    }
    bool replaced = false;  // this lane replaced a warm start
    for (uint32_t t0 = 0; t0 < ncons; t0 += mr::kMlpRows) {
        bool in_range = false;  // lanes 0-15: their row's features are all within bounds
        __syncthreads();
        if (lane < mr::kMlpRows) {
            const uint32_t c = t0 + lane;
            float f[mr::kMlpIn] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            if (c < ncons) {
                contact_features(e, c, mnv, f);
                if (samples != nullptr) {
                    float* row = samples + (size_t)c * mr::kMlpSampleFloats;
                    for (uint32_t k = 0; k < mr::kMlpIn; ++k) row[k] = f[k];
                    // the warm start the solve begins from, unless the network replaces it below
                    for (uint32_t k = 0; k < 3u; ++k) row[12u + k] = e.lam[3u * c + k];
                    row[15] = 0.0f;
                    for (uint32_t k = 16u; k < 20u; ++k) row[k] = 0.0f;
                }
            }
            if (infer) {
                in_range = true;
                for (uint32_t k = 0; k < mr::kMlpIn; ++k) {
                    const float xn = c < ncons ? (f[k] - m.in_shift[k]) * m.in_scale[k] : 0.0f;
                    in_range = in_range && fabs_(xn) <= kMlpFeatureBound;
                    s.x[lane * mr::kMlpIn + k] = in_range ? xn : 0.0f;
                }
            }
        }
        __syncthreads();
        if (!infer) continue;
        float y[4];
        mr::mlp_tile_forward(m, s, lane, y);
        __syncthreads();
        const uint32_t col = lane & 15u;
        if (col < mr::kMlpOut) {
            const float scale = m.out_scale[col];
            for (uint32_t r = 0; r < 4u; ++r) s.x[((lane >> 4) * 4u + r) * mr::kMlpIn + col] = y[r] * scale;
        }
        __syncthreads();
        if (samples != nullptr && lane < mr::kMlpRows && t0 + lane < ncons && in_range) {
            float* row = samples + (size_t)(t0 + lane) * mr::kMlpSampleFloats;
            for (uint32_t k = 0; k < 3u; ++k) row[16u + k] = s.x[lane * mr::kMlpIn + k];
            row[19] = 1.0f;
        }
        if (lane < mr::kMlpRows && t0 + lane < ncons && in_range) {
            const uint32_t c = t0 + lane;
            float lam[3];
            bool changed = false;
            const float gate = e.a->mlp.min_correction;
            for (uint32_t k = 0; k < 3u; ++k) changed = changed || fabs_(s.x[lane * mr::kMlpIn + k]) > gate;
            for (uint32_t k = 0; k < 3u; ++k) {
                const float prev = e.lam[3u * c + k], d = s.x[lane * mr::kMlpIn + k];
                lam[k] = changed ? prev + d : prev;
            }
            const HotConstraint& hk = e.hot[c];
            if (changed) project_cone(lam, hk.mu_u, hk.mu_v, e.a->cfg.maximum_normal_impulse);
            if (changed && isfin(lam[0]) && isfin(lam[1]) && isfin(lam[2])) {
                e.lam[3u * c] = lam[0];
                e.lam[3u * c + 1u] = lam[1];
                e.lam[3u * c + 2u] = lam[2];
                replaced = true;
                if (samples != nullptr) {
                    float* row = samples + (size_t)c * mr::kMlpSampleFloats;
                    for (uint32_t k = 0; k < 3u; ++k) row[12u + k] = lam[k];
                    row[15] = 1.0f;
                }
            }
        }
    }
    __syncthreads();
    return __ballot(replaced) != 0ull;
}

// --------------------------------------------------------------- kernel

// One control step of one environment (one wavefront per workgroup). kMlp
// selects the instance with the learned warm start and its sample capture;
// the plain instance carries none of that code.
// `step` selects the control step of a multi-step launch: the command, reset
// mask and status records of step `step` ([steps][E] each); 0 elsewhere.
template <bool kMlp, bool kCcd = false, bool kGeo = false>
__device__ __forceinline__ void control_step(const KernelArgs& args, uint32_t env,
                                                                 uint32_t step = 0u) {
    extern __shared__ __align__(16) unsigned char lds_base[];
    __shared__ unsigned long long s_fail;
    __shared__ float s_fmax[2];
    __shared__ float s_root[7];
    __shared__ MRContactStatusC s_cs;
    __shared__ unsigned long long s_t0;  // start of this control step on the constant-rate clock (step timing)
    // with the queue instances' next entry; the world's capacities are checked against what is left
    static_assert(sizeof(s_fail) + sizeof(s_fmax) + sizeof(s_root) + sizeof(s_cs) + sizeof(s_t0) + sizeof(uint32_t) <=
                      mr::kStepStaticLdsBytes, "static LDS of a control step");

    uint32_t lane = stage_lane(threadIdx.x);
    if (env >= args.environment_count) return;
    const KernelArgs& A = args;

    Env e;
    e.a = &A;
    e.env = env;
    e.hd = &A.models[A.environment_model[env]];
    const MRModelHeaderC& hd = *e.hd;
    e.bodies = A.bodies + hd.body_offset;
    e.dofs = A.dofs + hd.dof_offset;
    e.acts = A.actuators != nullptr ? A.actuators + hd.dof_offset : nullptr;
    e.shapes = A.shapes + hd.shape_offset;
    e.mats = A.materials + hd.material_offset;
    e.pairs = A.pairs + hd.pair_offset;
    e.nlinks = hd.link_count;
    e.nbodies = hd.body_count;
    e.nv = hd.nv;
    e.nq = hd.nq;
    e.nshapes = hd.shape_count;
    e.npairs = hd.pair_count;
    e.nscene = hd.scene_body_count;
    e.levels = hd.level_count;
    e.root_type = hd.root_type;
    e.h = A.h;
    e.gravity = V3{A.gravity[0], A.gravity[1], A.gravity[2]};
    const mr::LdsLayout& L = A.lds;
    e.topo = lds_at<mr::TopoCache>(lds_base, L.topo);
    e.lconst = lds_at<mr::LinkConst>(lds_base, L.lconst);
    e.arm = lds_at<float>(lds_base, L.arm);
    e.q = lds_at<float>(lds_base, L.q);
    e.v = lds_at<float>(lds_base, L.v);
    e.vcand = lds_at<float>(lds_base, L.vcand);
    e.effort = lds_at<float>(lds_base, L.effort);
    e.accel = lds_at<float>(lds_base, L.accel);
    e.cmd = lds_at<float>(lds_base, L.cmd);
    e.pos = lds_at<V3>(lds_base, L.pos);
    e.rot = lds_at<Q4>(lds_base, L.rot);
    e.w = lds_at<V3>(lds_base, L.w);
    e.vl = lds_at<V3>(lds_base, L.vl);
    e.sa = lds_at<V3>(lds_base, L.sa);
    e.sl = lds_at<V3>(lds_base, L.sl);
    e.ca = lds_at<V3>(lds_base, L.ca);
    e.cl = lds_at<V3>(lds_base, L.cl);
    e.r = lds_at<V3>(lds_base, L.r);
    e.I = lds_at<float>(lds_base, L.I);
    e.p = lds_at<float>(lds_base, L.p);
    e.Ut = lds_at<V3>(lds_base, L.Ut);
    e.Ub = lds_at<V3>(lds_base, L.Ub);
    e.D = lds_at<float>(lds_base, L.D);
    e.u = lds_at<float>(lds_base, L.u);
    e.L = lds_at<float>(lds_base, L.L);
    e.scene = lds_at<MRBodyStateC>(lds_base, L.scene);
    e.col = lds_at<Collider>(lds_base, L.col);
    if constexpr (kCcd) {
        e.ccol = lds_at<Collider>(lds_base, L.ccol);
        e.swept = lds_at<uint32_t>(lds_base, L.swept);
    }
    e.active = lds_at<uint32_t>(lds_base, L.active);
    e.npts = lds_at<uint32_t>(lds_base, L.npts);
    e.moff = lds_at<uint32_t>(lds_base, L.moff);
    e.okey = lds_at<uint32_t>(lds_base, L.okey);
    e.hfitem = lds_at<uint32_t>(lds_base, L.hfitem);
    e.hfq = lds_at<mr::HfHit>(lds_base, L.hfq);
    e.lam = lds_at<float>(lds_base, L.lam);
    e.cpair = lds_at<uint32_t>(lds_base, L.cpair);
    e.rslot = lds_at<float>(lds_base, L.rslot);
    e.rstack = lds_at<float>(lds_base, L.rstack);
    e.resid = lds_at<float>(lds_base, L.resid);
    e.sbody = lds_at<float4>(lds_base, L.sbody);
    e.sord = lds_at<uint16_t>(lds_base, L.sord);
    e.rows = (LdsFloat*)lds_at<float>(lds_base, L.rows);
    e.jrelax = lds_at<float>(lds_base, L.jrelax);
    e.jdelta = lds_at<float>(lds_base, L.jdelta);
    if constexpr (kMlp) {
        e.mlp_lds = lds_base + L.mlp;
        e.mlp_lam = lds_at<float>(lds_base, L.mlp_lam);
        e.mlp_scene = lds_at<MRBodyStateC>(lds_base, L.mlp_scene);
    }
    const uint32_t pcap = A.pair_capacity, mcap = A.manifold_capacity, ccap = A.constraint_capacity;
    e.stage_h = A.stage_h + (size_t)env * pcap;
    e.stage_p = A.stage_p + (size_t)env * pcap * MR_MANIFOLD_POINT_CAPACITY;
    e.jrow = A.jrow + (size_t)env * ccap * 3u * A.row_stride;
    e.resp = A.resp + (size_t)env * ccap * 3u * A.row_stride;
    e.cold = A.cold + (size_t)env * ccap;
    e.hot = A.hot + (size_t)env * ccap;

    // ---- topology cache (one lane per body / DoF; 64 lanes cover the limits)
    {
        mr::TopoCache& T = *e.topo;
        uint8_t par = 0xffu, vi = 0xffu, qi = 0xffu, dep = 0u, mot = 0u, jt = 0u;
        if (lane < e.nbodies) {
            const MRBodyC& b = e.bodies[lane];
            mot = (uint8_t)b.motion_type;
            if (lane < e.nlinks) {
                par = b.parent == MR_INVALID_INDEX ? (uint8_t)0xffu : (uint8_t)b.parent;
                vi = b.v_index == MR_INVALID_INDEX ? (uint8_t)0xffu : (uint8_t)b.v_index;
                qi = b.q_index == MR_INVALID_INDEX ? (uint8_t)0xffu : (uint8_t)b.q_index;
                dep = (uint8_t)b.depth;
                jt = (uint8_t)b.joint_type;
            }
        }
        T.qidx[lane] = qi;
        T.jtype[lane] = jt;
        T.parent[lane] = par;
        T.vidx[lane] = vi;
        T.depth[lane] = dep;
        T.motion[lane] = mot;
        T.dof_body[lane] = lane < e.nv ? (uint8_t)e.dofs[lane].body : (uint8_t)0xffu;
        if (lane < e.nlinks) {
            const MRBodyC& b = e.bodies[lane];
            mr::LinkConst lc;
            const Q4 cc = qconj(q4(b.child_rotation));
            const V3 ax = normalize(f3(b.axis));
            lc.prot[0] = b.parent_rotation.x; lc.prot[1] = b.parent_rotation.y;
            lc.prot[2] = b.parent_rotation.z; lc.prot[3] = b.parent_rotation.w;
            lc.crot_conj[0] = cc.x; lc.crot_conj[1] = cc.y; lc.crot_conj[2] = cc.z; lc.crot_conj[3] = cc.w;
            lc.axis[0] = ax.x; lc.axis[1] = ax.y; lc.axis[2] = ax.z;
            lc.panchor[0] = b.parent_anchor.x; lc.panchor[1] = b.parent_anchor.y; lc.panchor[2] = b.parent_anchor.z;
            lc.canchor[0] = b.child_anchor.x; lc.canchor[1] = b.child_anchor.y; lc.canchor[2] = b.child_anchor.z;
            e.lconst[lane] = lc;
        }
        if (lane < e.nv) e.arm[lane] = effective_armature(e, lane);
        __syncthreads();
        // model validation guarantees parent < child, so both walks end
        unsigned long long anc = 0ull, ch = 0ull;
        if (lane < e.nlinks) {
            for (uint32_t b = lane; b != 0u && b != 0xffu; b = T.parent[b]) anc |= 1ull << b;
            for (uint32_t c = lane + 1u; c < e.nlinks; ++c)
                if (T.parent[c] == lane) ch |= 1ull << c;
        }
        T.anc[lane] = anc;
        T.children[lane] = ch;
        T.slot[lane] = A.response_slots[(size_t)A.environment_model[env] * MR_MAX_BODIES + lane];
    }

    const uint32_t nv = e.nv, nq = e.nq, nl = e.nlinks, nsc = e.nscene;
    float* gq = A.q + (size_t)env * A.max_nq;
    float* gv = A.v + (size_t)env * A.max_nv;
    MRBodyStateC* gs = A.scene + (size_t)env * A.max_scene;
    const uint32_t cur = A.mcurrent[env];
    const size_t E = A.environment_count;

    // ---- prepare: reset, load state (the HBM state is the checkpoint)
    const size_t step_rec = (size_t)step * E + env;  // this step's record of this environment
    if (A.step_us != nullptr && lane == 0u) s_t0 = __builtin_amdgcn_s_memrealtime();
    const bool reset = A.reset_mask != nullptr && A.reset_mask[step_rec] != 0u;
    for (uint32_t i = lane; i < nq; i += kLanes) {
        const float val = reset ? A.reset_q[(size_t)env * A.max_nq + i] : gq[i];
        e.q[i] = val;
        if (reset) gq[i] = val;
    }
    for (uint32_t i = lane; i < nv; i += kLanes) {
        const float val = reset ? A.reset_v[(size_t)env * A.max_nv + i] : gv[i];
        e.v[i] = val;
        if (reset) gv[i] = val;
        e.cmd[i] = A.command[step_rec * A.max_nv + i];
    }
    for (uint32_t s = lane; s < nsc; s += kLanes) {
        const MRBodyStateC val = reset ? A.reset_scene[(size_t)env * A.max_scene + s] : gs[s];
        e.scene[s] = val;
        if (reset) gs[s] = val;
    }
    if (lane == 0u) {
        if (reset) A.mcount[(size_t)cur * E + env] = 0u;
        s_fail = ~0ull;
    }
    __syncthreads();

    StageClock clk;
    clk.init(A.stage_cycles != nullptr ? A.stage_cycles + (size_t)env * mr::kStageCount : nullptr, lane);
    uint32_t src_buf = cur;
    uint32_t dst_buf = (cur + 1u) % 3u;
    const uint32_t alt_buf = (cur + 2u) % 3u;
    uint32_t mcount_src = A.mcount[(size_t)cur * E + env];
    if (mcount_src > mcap) mcount_src = mcap;

    // Contact status lives in LDS (uniform fields are written with identical
    // values by every lane; lane-0-only fields by lane 0).
    MRContactStatusC& cs = s_cs;
    if (lane == 0u) {
        unsigned char* p = reinterpret_cast<unsigned char*>(&cs);
        for (uint32_t k = 0; k < sizeof(cs); ++k) p[k] = 0;
        cs.first_failing_pair = MR_INVALID_INDEX;
        cs.first_failing_constraint = MR_INVALID_INDEX;
    }
    __syncthreads();
    uint32_t successful = 0u;
    float min_piv = __builtin_inff(), max_piv = 0.0f, max_acc = 0.0f;
    uint32_t failing_substep = MR_INVALID_INDEX;
    float h = e.h;
    const MRWorldStepConfigC& cfg = A.cfg;
    const bool floating = e.root_type == MR_ROOT_FLOATING;
    uint32_t impact_segments = 0u;  // segments that ended at a time of impact (hybrid CCD)

    // A microstep is one segment, or (hybrid CCD) a sequence of segments ending
    // at successive times of impact; each segment runs every stage below with
    // h = its duration, and the microstep counts once its last segment commits.
    float remaining = A.h;
    uint32_t segment = 0u;
    for (uint32_t substep = 0; substep < cfg.physics_substeps;) {
        if constexpr (kCcd) {
            h = remaining;
            e.h = h;
        }
        bool impact = false;
        // ---------------------------------------------------------- drives
        lane = stage_lane(lane);
        // Implicit drives refresh from the current state every microstep; an
        // effort command is clamped once, at the control step's start velocity,
        // and held (MetalWorld.metal:184-270 prepare, 280-366 refresh). They
        // depend on h, so the hybrid mode refreshes them once the segment's
        // duration is known, below.
        if constexpr (!kCcd) {
            if (substep == 0u || cfg.actuation_mode == MR_ACTUATION_IMPLICIT_POSITION_DRIVE)
                for (uint32_t j = lane; j < nv; j += kLanes) e.effort[j] = drive_effort(e, j);
            __syncthreads();
        }
        // ------------------------------------------------------ kinematics
        lane = stage_lane(lane);
        forward_kinematics(e, lane, &s_fail);
        __syncthreads();
        clk.mark(mr::kStageKinematics);
        if (s_fail != ~0ull) break;
        // ----------------------------------------------- time of impact
        if constexpr (kCcd) {
            // Three passes, bound by the instructions of a query (conservative
            // advancement through every pair class a wave holds): the swept
            // bounds once per shape, the pairs against them, and the queries of
            // the pairs that overlap, which are few, packed to 64 at a time.
            // With the bounds and the query of each pair in one pass, 372 pairs
            // took 250,000 cycles a segment; 90,000 now (chain of 7 links, 20 boxes).
            for (uint32_t s = lane; s < e.nshapes; s += kLanes) {
                Collider c;
                ccd_sweep_collider<kGeo>(e, s, remaining, c);
                e.ccol[s] = c;
            }
            __syncthreads();
            uint32_t my_bits = ~0u, my_pair = ~0u, my_unsafe = ~0u;
            uint32_t waiting = 0u;
            for (uint32_t base = 0u, more = 1u; more != 0u; base += kLanes) {
                more = base + kLanes < e.npairs ? 1u : 0u;
                const bool swept = base + lane < e.npairs && ccd_pair_swept(e, base + lane);
                const unsigned long long bal = __ballot(swept);
                if (swept) e.swept[waiting + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull))] = base + lane;
                waiting = uniform_u32(waiting + (uint32_t)__popcll(bal));
                __syncthreads();
                while (waiting >= kLanes || (more == 0u && waiting > 0u)) {
                    if (lane < waiting) {
                        const uint32_t k = e.swept[lane];
                        float toi = 0.0f;
                        const uint32_t r = ccd_pair<kGeo>(e, k, remaining, toi);
                        if (r == kCcdImpact) {
                            const uint32_t bits = __float_as_uint(fmaxd(toi, 0.0f));
                            if (bits < my_bits) {
                                my_bits = bits;
                                my_pair = k;
                            }
                        } else if (r == kCcdUnsafe && my_unsafe == ~0u) {
                            my_unsafe = k;
                        }
                    }
                    waiting -= waiting < kLanes ? waiting : kLanes;
                    const uint32_t next = e.swept[kLanes + lane];
                    __syncthreads();
                    e.swept[lane] = next;
                    __syncthreads();
                }
            }
            // earliest (TOI bits, pair) over the wave: non-negative floats order as their bits
            const uint32_t best_bits = wave_min_u32(my_bits);
            const uint32_t best_pair = wave_min_u32(my_bits == best_bits ? my_pair : ~0u);
            const uint32_t unsafe = wave_min_u32(my_unsafe);
            if (unsafe != ~0u) report_failure(&s_fail, unsafe, MR_STEP_DID_NOT_CONVERGE, unsafe);
            if (best_bits != ~0u) {
                const float tau = fmaxd(__uint_as_float(best_bits), cfg.ccd_time_tolerance);
                if (tau < remaining - cfg.ccd_time_tolerance) {
                    if (segment >= cfg.max_ccd_events)
                        report_failure(&s_fail, best_pair, MR_STEP_CCD_EVENT_BUDGET_EXHAUSTED, best_pair);
                    impact = true;
                    h = tau;
                    e.h = h;
                }
            }
            __syncthreads();
            if (s_fail != ~0ull) break;
        }
        const bool final_sub = substep + 1u == cfg.physics_substeps && !impact;
        const bool capture = cfg.capture_evidence != 0u && substep == cfg.capture_substep && segment == 0u &&
            A.evidence_pairs != nullptr;
        if constexpr (kCcd) {
            if ((substep == 0u && segment == 0u) || cfg.actuation_mode == MR_ACTUATION_IMPLICIT_POSITION_DRIVE)
                for (uint32_t j = lane; j < nv; j += kLanes) e.effort[j] = drive_effort(e, j);
            __syncthreads();
        }
        // -------------------------------------------------------------- ABA
        lane = stage_lane(lane);
        if (lane < nl) aba_init_link(e, lane);
        const uint32_t my_depth = lane < nl ? e.topo->depth[lane] : 0xffu;
        __syncthreads();
        float lane_min_piv = __builtin_inff(), lane_max_piv = 0.0f;
        for (uint32_t d = e.levels - 1u; d >= 1u; --d)
            aba_inward_level(e, lane, __ballot(my_depth == d), lane_min_piv, lane_max_piv, &s_fail);
        if (s_fail != ~0ull) break;
        lane_min_piv = -wave_max(-lane_min_piv);
        lane_max_piv = wave_max(lane_max_piv);
        // the root: its gathered inertia, factored and solved by every lane alike
        V3 alpha{0.0f, 0.0f, 0.0f}, acc{0.0f, 0.0f, 0.0f};
        if (floating) {
            float c[6], p;
            aba_gather_column(e, 0u, lane < 6u ? lane : 0u, c, p);
            __syncthreads();
            if (lane < 6u) {
#pragma unroll
                for (int k = 0; k < 6; ++k) e.I[6u * lane + k] = c[k];
                e.p[lane] = p;
            }
            __syncthreads();
            uint32_t fail_row = 0;
            if (!root_factor(e.I, e.L, lane_min_piv, lane_max_piv, fail_row) && lane == 0u)
                report_failure(&s_fail, 0x10000u, MR_STEP_FACTORIZATION_FAILED, fail_row);
            __syncthreads();
            const float rhs[6] = {-e.p[0], -e.p[1], -e.p[2], -e.p[3], -e.p[4], -e.p[5]};
            float x[6];
            root_solve(e.L, rhs, x);
            alpha = V3{x[0], x[1], x[2]};
            acc = V3{x[3], x[4], x[5]};
            if (lane == 0u) {
                e.accel[0] = x[3]; e.accel[1] = x[4]; e.accel[2] = x[5];
                e.accel[3] = x[0]; e.accel[4] = x[1]; e.accel[5] = x[2];
            }
        }
        if (lane == 0u) {
            s_fmax[0] = lane_min_piv;
            s_fmax[1] = lane_max_piv;
        }
        __syncthreads();
        if (s_fail != ~0ull) break;
        // outward, one lane per link: what a link needs besides its parent's
        // acceleration is in registers before the level loop
        {
            const bool link = lane < nl && lane > 0u;
            const uint32_t i = link ? lane : 0u;
            const uint32_t parent = link ? e.topo->parent[lane] : 0u, vi = link ? e.topo->vidx[lane] : 0xffu;
            const bool has = vi != 0xffu;
            const V3 r = e.r[i], Ut = e.Ut[i], Ub = e.Ub[i], sa = e.sa[i], sl = e.sl[i], ca = e.ca[i], cl = e.cl[i];
            const float D = e.D[i], u = e.u[i];
            float qdd = 0.0f;
            for (uint32_t d = 1; d < e.levels; ++d) {
                const V3 ap = wave_get(alpha, parent);
                const V3 lp = add(wave_get(acc, parent), cross(ap, r));
                V3 ai = add(ap, ca);
                V3 li = add(lp, cl);
                const float proj = dot(Ut, ap) + dot(Ub, lp);
                const float q2 = (u - proj) / D;
                if (has) {
                    ai = add(ai, mul(q2, sa));
                    li = add(li, mul(q2, sl));
                }
                if (my_depth == d) {
                    alpha = ai;
                    acc = li;
                    qdd = q2;
                }
            }
            if (has) e.accel[vi] = qdd;
        }
        __syncthreads();
        for (uint32_t j = lane; j < nv; j += kLanes) {
            const float a = e.accel[j];
            const float nvv = e.v[j] + h * a;
            if (!isfin(a) || !isfin(nvv)) report_failure(&s_fail, j, MR_STEP_NONFINITE_RESULT, j);
            e.vcand[j] = nvv;
        }
        __syncthreads();
        clk.mark(mr::kStageABA);
        if (s_fail != ~0ull) break;
        // ------------------------------------------- scene prediction
        lane = stage_lane(lane);
        for (uint32_t s = lane; s < nsc; s += kLanes) {
            const uint32_t b = nl + s;
            const MRBodyC& bp = e.bodies[b];
            MRBodyStateC st = e.scene[s];
            Q4 rq;
            if (!normalized_quat(q4(st.orientation), rq) || !finite3(f3(st.position)) ||
                !finite3(f3(st.linear_velocity_inv_mass)) || !finite3(f3(st.angular_velocity))) {
                report_failure(&s_fail, b, MR_STEP_NONFINITE_INPUT, b);
                continue;
            }
            st.position.w = 1.0f;
            st.orientation = mr_float4{rq.x, rq.y, rq.z, rq.w};
            st.linear_velocity_inv_mass.w = bp.motion_type == MR_MOTION_DYNAMIC ? bp.mass.y : 0.0f;
            st.angular_velocity.w = 0.0f;
            st.flags_indices[0] = bp.motion_type;
            st.flags_indices[1] = MR_INVALID_INDEX;
            st.flags_indices[2] = b;
            world_inverse_inertia(bp, rq, st);
            if (bp.motion_type == MR_MOTION_DYNAMIC) {
                // velocity damping is a per-microstep factor: its first segment applies it
                const float dl = !kCcd || segment == 0u ? bp.damping_scale.x : 1.0f;
                const float da = !kCcd || segment == 0u ? bp.damping_scale.y : 1.0f;
                const V3 lv = add(mul(dl, f3(st.linear_velocity_inv_mass)), mul(h, e.gravity));
                const V3 av = mul(da, f3(st.angular_velocity));
                st.linear_velocity_inv_mass.x = lv.x;
                st.linear_velocity_inv_mass.y = lv.y;
                st.linear_velocity_inv_mass.z = lv.z;
                st.angular_velocity.x = av.x;
                st.angular_velocity.y = av.y;
                st.angular_velocity.z = av.z;
            } else {
                st.linear_velocity_inv_mass.x = 0.0f;
                st.linear_velocity_inv_mass.y = 0.0f;
                st.linear_velocity_inv_mass.z = 0.0f;
                st.angular_velocity.x = 0.0f;
                st.angular_velocity.y = 0.0f;
                st.angular_velocity.z = 0.0f;
            }
            e.scene[s] = st;
        }
        __syncthreads();
        if (s_fail != ~0ull) break;
        // ------------------------------------------- collider projection
        lane = stage_lane(lane);
        for (uint32_t s = lane; s < e.nshapes; s += kLanes) {
            Collider c;
            if (!project_collider<kGeo>(e, s, c)) report_failure(&s_fail, s, MR_STEP_NONFINITE_INPUT, s);
            e.col[s] = c;
        }
        __syncthreads();
        clk.mark(mr::kStageProjection);
        if (s_fail != ~0ull) break;
        // ----------------------------------------------- broadphase flags
        lane = stage_lane(lane);
        uint32_t nact = 0;
        for (uint32_t base = 0; base < e.npairs; base += kLanes) {
            const uint32_t p = base + lane;
            bool flag = false;
            if (p < e.npairs) {
                const MRCompiledPairC pr = e.pairs[p];
                flag = pair_may_overlap(e.col[pr.collider_a], e.col[pr.collider_b]);
            }
            const unsigned long long bal = __ballot(flag);
            const uint32_t before = (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
            if (flag) {
                const uint32_t slot = nact + before;
                if (slot < pcap) e.active[slot] = p;
            }
            nact += (uint32_t)__popcll(bal);
        }
        __syncthreads();
        if (capture) {
            const uint32_t nrec = nact < pcap ? nact : pcap;
            for (uint32_t k = lane; k < nrec; k += kLanes) {
                const MRCompiledPairC pr = e.pairs[e.active[k]];
                MRPairRecordC rec;
                rec.environment = env;
                rec.collider_a = pr.collider_a;
                rec.collider_b = pr.collider_b;
                rec.pair_class = pr.pair_class;
                A.evidence_pairs[(size_t)env * pcap + k] = rec;
            }
            if (lane == 0u && A.evidence_counts != nullptr) A.evidence_counts[env] = nact;
        }
        nact = uniform_u32(nact);
        cs.required_pairs = nact;
        cs.active_pairs = nact;
        if (cs.max_active_pairs < nact) cs.max_active_pairs = nact;
        if (nact > pcap) {
            if (lane == 0u) report_failure(&s_fail, 0u, MR_STEP_PAIR_CAPACITY_OVERFLOW, 0u);
            // first overflowing compiled pair is the (pcap+1)-th flagged pair
            uint32_t seen = 0, idx = 0;
            for (uint32_t base = 0; base < e.npairs; base += kLanes) {
                const uint32_t p = base + lane;
                bool flag = false;
                if (p < e.npairs) {
                    const MRCompiledPairC pr = e.pairs[p];
                    flag = pair_may_overlap(e.col[pr.collider_a], e.col[pr.collider_b]);
                }
                const unsigned long long bal = __ballot(flag);
                const uint32_t before = (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
                if (flag && seen + before == pcap) idx = p + 1u;
                seen += (uint32_t)__popcll(bal);
            }
            idx = wave_max_u32(idx);
            if (lane == 0u) cs.first_failing_pair = idx - 1u;
            __syncthreads();
            if (lane == 0u) s_fail = ((unsigned long long)MR_STEP_PAIR_CAPACITY_OVERFLOW << 24) | ((idx - 1u) & 0xffffffu);
            __syncthreads();
            break;
        }
        clk.mark(mr::kStageBroadphase);
        // ---------------------------------- narrowphase + manifold refresh
        lane = stage_lane(lane);
        const MRManifoldHeaderC* old_h = A.mh + ((size_t)src_buf * E + env) * mcap;
        const MRManifoldPointC* old_p = A.mp + ((size_t)src_buf * E + env) * mcap * MR_MANIFOLD_POINT_CAPACITY;
        mcount_src = uniform_u32(mcount_src);
        uint32_t my_raw = 0, my_ret = 0, my_fresh = 0;
        float my_pen = 0.0f;
        // collider keys of the previous manifolds, staged once for the lookups
        for (uint32_t m = lane; m < mcount_src; m += kLanes) {
            const uint32_t ka = old_h[m].pair_and_count[1], kb = old_h[m].pair_and_count[2];
            e.okey[m] = (ka < 0x10000u && kb < 0x10000u) ? (ka | (kb << 16)) : 0xffffffffu;
        }
        // Heightfield queries of all active pairs, one lane per query point
        // (a sphere has one, a capsule three, a box eight), into e.hfq; moff
        // holds each pair's first query until the manifold prefix below. A pair
        // whose queries do not fit the table evaluates them in its own lane.
        // Query offsets grow with the pair index, so the pairs that fit own
        // exactly the slots [0, used); the slots of a pair that straddles the
        // table end are never written and never read.
        {
            uint32_t nhf = 0, used = 0;
            for (uint32_t base = 0; base < nact; base += kLanes) {
                const uint32_t k = base + lane;
                uint32_t nq = 0;
                if (k < nact) {
                    const MRCompiledPairC pr = e.pairs[e.active[k]];
                    if (pr.pair_class == MR_PAIR_HEIGHTFIELD) {
                        const uint32_t fsi = e.col[pr.collider_a].type == MR_SHAPE_HEIGHTFIELD ? pr.collider_b
                                                                                              : pr.collider_a;
                        nq = hf_query_count(e.col[fsi].type);
                    }
                }
                uint32_t tot;
                const uint32_t before = wave_prefix_sum(nq, lane, tot);
                uint32_t end = 0;
                if (k < nact) {
                    const uint32_t first = nhf + before;
                    const bool fits = nq > 0u && first + nq <= mr::kHfSlots;
                    e.moff[k] = fits ? first : 0xffffffffu;
                    if (fits) {
                        for (uint32_t q = 0; q < nq; ++q) e.hfitem[first + q] = k | (q << 16);
                        end = first + nq;
                    }
                }
                const uint32_t chunk_end = wave_max_u32(end);
                used = chunk_end > used ? chunk_end : used;
                nhf += tot;
            }
            __syncthreads();
            const uint32_t items = used;
            for (uint32_t i = lane; i < items; i += kLanes) {
                const uint32_t k = e.hfitem[i] & 0xffffu, q = e.hfitem[i] >> 16;
                const MRCompiledPairC pr = e.pairs[e.active[k]];
                const uint32_t fsi = e.col[pr.collider_a].type == MR_SHAPE_HEIGHTFIELD ? pr.collider_b : pr.collider_a;
                const Collider& fs = e.col[fsi];
                e.hfq[i] = heightfield_query(e, hf_query_point(fs, q), hf_query_radius(fs));
            }
        }
        __syncthreads();
        for (uint32_t k = lane; k < nact; k += kLanes) {
            const MRCompiledPairC pr = e.pairs[e.active[k]];
            const Collider ca_ = e.col[pr.collider_a];
            const Collider cb_ = e.col[pr.collider_b];
            ContactSink raw;
            raw.head = reinterpret_cast<float*>(e.stage_h + k);
            raw.points = reinterpret_cast<float*>(e.stage_p + (size_t)k * MR_MANIFOLD_POINT_CAPACITY);
            raw.count = 0u;
            raw.deepest = 0.0f;
            raw.deepest_a = 0u;
            raw.deepest_b = 0u;
            raw.normal = V3{0.0f, 0.0f, 0.0f};
            raw.rest = e.shapes[pr.collider_a].contact_rest_radius.y + e.shapes[pr.collider_b].contact_rest_radius.y;
            raw.penetration = 0.0f;
            raw.bad = false;
            generate_contacts<kGeo>(e, pr.collider_a, pr.collider_b, pr.pair_class, ca_, cb_, raw, e.moff[k]);
            uint32_t contacts = 0;
            if (raw.bad) {
                report_failure(&s_fail, k, MR_STEP_NONFINITE_RESULT, e.active[k]);
            } else if (raw.count > 0u) {
                contacts = raw.count;
                my_raw += raw.count;
                my_pen = fmaxd(my_pen, raw.penetration);
                raw.head[8] = raw.normal.x;
                raw.head[9] = raw.normal.y;
                raw.head[10] = raw.normal.z;
            }
            e.npts[k] = contacts;  // the manifold's points from build_manifolds on
        }
        __syncthreads();
        // the pairs in contact, compacted (moff's queries are used up), eight at a time
        uint32_t touching = 0;
        for (uint32_t base = 0; base < nact; base += kLanes) {
            const uint32_t k = base + lane;
            const bool in = k < nact && e.npts[k] > 0u;
            const unsigned long long bal = __ballot(in);
            if (in) e.moff[touching + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull))] = k;
            touching += (uint32_t)__popcll(bal);
        }
        __syncthreads();
        for (uint32_t base = 0; base < touching; base += kLanes / 8u) {
            const uint32_t slot = base + (lane >> 3);
            const bool on = slot < touching;
            build_manifolds(e, lane, e.moff[on ? slot : base], on, old_h, old_p, mcount_src, my_ret, my_fresh, &s_fail);
        }
        const uint32_t raw_total = wave_sum_u32(my_raw);
        const uint32_t ret_total = wave_sum_u32(my_ret);
        const uint32_t fresh_total = wave_sum_u32(my_fresh);
        const float pen = wave_max(my_pen);
        __syncthreads();
        clk.mark(mr::kStageNarrowphase);
        if (s_fail != ~0ull) break;
        // prefix over manifolds (count>0) and constraint offsets
        uint32_t nman = 0, ncons = 0;
        for (uint32_t base = 0; base < nact; base += kLanes) {
            const uint32_t k = base + lane;
            const uint32_t pts = k < nact ? e.npts[k] : 0u;
            const unsigned long long bal = __ballot(pts > 0u);
            const uint32_t mbefore = (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
            uint32_t tot;
            const uint32_t cbefore = wave_prefix_sum(pts, lane, tot);
            if (k < nact) e.moff[k] = pts > 0u ? ((nman + mbefore) | ((ncons + cbefore) << 16u)) : 0xffffffffu;
            nman += (uint32_t)__popcll(bal);
            ncons += tot;
        }
        // wave-uniform by construction; said so, every loop over the contacts
        // below is a scalar loop instead of an exec-masked one
        nman = uniform_u32(nman);
        ncons = uniform_u32(ncons);
        cs.raw_contacts = raw_total;
        cs.required_manifolds = nman;
        cs.manifolds = nman;
        cs.retained_points = ret_total;
        cs.new_points = fresh_total;
        cs.diagnostics.x = pen;
        if (nman > mcap) {
            if (lane == 0u) s_fail = ((unsigned long long)MR_STEP_MANIFOLD_CAPACITY_OVERFLOW << 24) | (nman & 0xffffffu);
            __syncthreads();
            break;
        }
        cs.required_constraints = ncons;
        if (ncons > ccap) {
            if (lane == 0u) s_fail = ((unsigned long long)MR_STEP_CONSTRAINT_CAPACITY_OVERFLOW << 24) | (ncons & 0xffffffu);
            __syncthreads();
            break;
        }
        cs.constraints = ncons;
        if (cs.max_constraints < ncons) cs.max_constraints = ncons;
        __syncthreads();
        // ---------------------------------------- compact + emission
        lane = stage_lane(lane);
        MRManifoldHeaderC* new_h = A.mh + ((size_t)dst_buf * E + env) * mcap;
        MRManifoldPointC* new_p = A.mp + ((size_t)dst_buf * E + env) * mcap * MR_MANIFOLD_POINT_CAPACITY;
        for (uint32_t k = lane; k < nact; k += kLanes) {
            const uint32_t mo = e.moff[k];
            if (mo == 0xffffffffu) continue;
            const uint32_t m = mo & 0xffffu, c0 = mo >> 16u;
            const MRManifoldHeaderC mh = e.stage_h[k];
            new_h[m] = mh;
            for (uint32_t p = 0; p < MR_MANIFOLD_POINT_CAPACITY; ++p)
                new_p[(size_t)m * MR_MANIFOLD_POINT_CAPACITY + p] = e.stage_p[(size_t)k * MR_MANIFOLD_POINT_CAPACITY + p];
            const MRShapeC& sa = e.shapes[mh.pair_and_count[1]];
            const MRShapeC& sb = e.shapes[mh.pair_and_count[2]];
            V3 pa_pos, pb_pos;
            Q4 pa_q, pb_q;
            body_pose(e, sa.body, pa_pos, pa_q);
            body_pose(e, sb.body, pb_pos, pb_q);
            Q4 ra, rb;
            checked_quat(pa_q, ra);
            checked_quat(pb_q, rb);
            const V3 n = normalize(qrot(ra, f3(mh.normal_and_age)));
            V3 t = qrot(ra, f3(mh.tangent_and_metric));
            t = sub(t, mul(dot(t, n), n));
            t = dot(t, t) > 1.0e-12f ? normalize(t) : stable_tangent(n);
            const V3 bt = cross(n, t);
            const MRMaterialC& ma = e.mats[sa.material];
            const MRMaterialC& mb = e.mats[sb.material];
            const float rest = sa.contact_rest_radius.y + sb.contact_rest_radius.y;
            for (uint32_t p = 0; p < mh.pair_and_count[3]; ++p) {
                const MRManifoldPointC mp = e.stage_p[(size_t)k * MR_MANIFOLD_POINT_CAPACITY + p];
                const uint32_t c = c0 + p;
                HotConstraint hk;
                ColdConstraint ck;
                hk.body_a = sa.body;
                hk.body_b = sb.body;
                hk.flags = mp.feature_and_life[2] == 0u ? MR_CONSTRAINT_FLAG_NEW_IMPACT : MR_CONSTRAINT_FLAG_WARM_STARTED;
                hk.kind = ((is_link(e, sa.body) || is_link(e, sb.body)) ? mr::kHotArticulated : 0u) |
                          (is_dynamic_scene(e, sa.body) ? mr::kHotDynamicA : 0u) |
                          (is_dynamic_scene(e, sb.body) ? mr::kHotDynamicB : 0u);
                const V3 pa = add(pa_pos, qrot(ra, f3(mp.local_anchor_a)));
                const V3 pb = add(pb_pos, qrot(rb, f3(mp.local_anchor_b)));
                const V3 pw = mul(0.5f, add(pa, pb));
                hk.point[0] = pw.x; hk.point[1] = pw.y; hk.point[2] = pw.z;
                hk.dir[0] = n.x; hk.dir[1] = n.y; hk.dir[2] = n.z;
                hk.dir[3] = t.x; hk.dir[4] = t.y; hk.dir[5] = t.z;
                hk.dir[6] = bt.x; hk.dir[7] = bt.y; hk.dir[8] = bt.z;
                ck.pa[0] = pa.x; ck.pa[1] = pa.y; ck.pa[2] = pa.z;
                ck.pb[0] = pb.x; ck.pb[1] = pb.y; ck.pb[2] = pb.z;
                ck.separation = dot(sub(pb, pa), n) - rest;
                ck.manifold = m;
                ck.point = p;
                ck.flags = hk.flags;
                const float fa[4] = {ma.friction.x, ma.friction.y, ma.friction.z, ma.friction.w};
                const float fb[4] = {mb.friction.x, mb.friction.y, mb.friction.z, mb.friction.w};
                for (int q = 0; q < 4; ++q) ck.friction[q] = sqrt_rn(fmaxd(0.0f, fa[q] * fb[q]));
                ck.restitution = fmaxd(ma.response.x, mb.response.x);
                ck.restitution_threshold = fmaxd(ma.response.y, mb.response.y);
                ck.compliance = ma.response.z + mb.response.z;
                ck.dissipation = ma.response.w + mb.response.w;
                const bool warm = cfg.warm_start != 0u;
                float wi[3] = {mp.impulses.x, mp.impulses.y, mp.impulses.z};
                if constexpr (kCcd) {
                    // impulses scale with the step: a segment warm-starts from the last
                    // segment's impulses times the ratio of the two durations
                    if (mp.impulses.w > 0.0f) {
                        const float s = h / mp.impulses.w;
                        for (int r = 0; r < 3; ++r) wi[r] = wi[r] * s;
                    }
                }
                e.lam[3u * c + 0u] = warm ? wi[0] : 0.0f;
                e.lam[3u * c + 1u] = warm ? wi[1] : 0.0f;
                e.lam[3u * c + 2u] = warm ? wi[2] : 0.0f;
                e.cpair[c] = sa.body | (sb.body << 8) | (hk.kind << 16);
                e.hot[c] = hk;
                e.cold[c] = ck;
            }
        }
        __syncthreads();
        clk.mark(mr::kStageEmission);
        // --------------------------- Jacobian rows + inverse-ABA responses
        lane = stage_lane(lane);
        // One response row per lane, three lanes per articulated contact, 21 contacts
        // a pass. The contacts of a pass are gathered to its first lanes: contact c
        // of rank r among the articulated ones pushes itself to lane r.
        {
            const ResponseLink own = response_link(e, lane);
            constexpr uint32_t kPerPass = kLanes / 3u;
            uint32_t count = 0u;
            for (uint32_t base = 0; base < ncons; base += kLanes)
                count += (uint32_t)__popcll(
                    __ballot(base + lane < ncons && ((e.cpair[base + lane] >> 16) & mr::kHotArticulated) != 0u));
            for (uint32_t first = 0; first < count; first += kPerPass) {
                uint32_t gathered = 0u, seen = 0u;  // lane k: contact first + k of the articulated ones, plus one
                for (uint32_t base = 0; base < ncons; base += kLanes) {
                    const uint32_t c = base + lane;
                    const bool art = c < ncons && ((e.cpair[c] >> 16) & mr::kHotArticulated) != 0u;
                    const unsigned long long bal = __ballot(art);
                    const uint32_t rank = seen + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
                    const bool in = art && rank >= first && rank < first + kPerPass;
                    gathered |= (uint32_t)__builtin_amdgcn_ds_permute((int)((in ? rank - first : kLanes - 1u) << 2),
                                                                      in ? (int)(c + 1u) : 0);
                    seen += (uint32_t)__popcll(bal);
                }
                const uint32_t slot = lane / 3u, r = lane % 3u;
                const uint32_t got = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(slot << 2), (int)gathered);
                const bool row = slot < kPerPass && got != 0u;
                const uint32_t c = row ? got - 1u : 0u;
                const HotConstraint& hk = e.hot[c];
                const ColdConstraint& ck = e.cold[c];
                const bool la = row && is_link(e, hk.body_a), lb = row && is_link(e, hk.body_b);
                const V3 pa{ck.pa[0], ck.pa[1], ck.pa[2]};
                const V3 pb{ck.pb[0], ck.pb[1], ck.pb[2]};
                const V3 d = hot_dir(hk, (int)r);
                float* rs = e.resp + ((size_t)c * 3u + (size_t)r) * A.row_stride;
                inverse_aba(e, lane, own, row, la ? hk.body_a : MR_INVALID_INDEX, pa, neg(d),
                            lb ? hk.body_b : MR_INVALID_INDEX, pb, d, rs);
            }
        }
        __syncthreads();
        clk.mark(mr::kStageResponses);
        // Ordered sweeps over contacts that all join the articulation to static
        // geometry need no schedule: they form one chain.
        const bool jacobi = cfg.solver == MR_SOLVER_RELAXED_JACOBI;
        bool scene_lane = false;
        for (uint32_t c = lane; c < ncons; c += kLanes) scene_lane |= (e.cpair[c] >> 16) != mr::kHotArticulated;
        const bool scheduled = !jacobi && wave_any(scene_lane);
        uint32_t levels = 0u, nart = ncons;
        if (scheduled) {
            levels = schedule_contacts(e, lane, ncons, ccap);
            nart = ncons - uniform_u32(reinterpret_cast<const uint32_t*>(e.resid)[levels]);
        }
        // articulated contact k of the substep: the k-th in index order (the
        // Jacobi mode keeps no list: its loops pass the others by)
        const uint32_t art_list = scheduled && lane < nart ? e.sord[ncons - nart + lane] : 0u;
        auto art_at = [&](uint32_t k) -> uint32_t {
            if (!scheduled) return k;
            return k < kLanes ? read_lane(art_list, k) : uniform_u32(e.sord[ncons - nart + k]);
        };
        // ------------------------------------------ IR evaluation + blocks
        lane = stage_lane(lane);
        // Lanes own DoFs for every articulation dot product (canonical fold);
        // per-constraint scalars are then evaluated lane-parallel over
        // constraints. target/winv carry rel and J M^-1 J^T between the two
        // passes.
        const uint32_t mnv = A.row_stride;  // >= max(1, max_nv)
        const bool dof_lane = lane < nv;
        float vj = dof_lane ? e.vcand[lane] : 0.0f;
        // Jacobian / response rows of constraint c for this DoF lane; the
        // loops below fetch constraint c + 1 while working on c. Rows of
        // constraints without an articulation endpoint are never written and
        // their (unused) values are ignored.
        // Branch-free on purpose: every lane loads (lanes past the stride read the
        // row's last element, ignored), so the wait counters can leave the
        // prefetch of the next constraint in flight.
        //
        // The unscheduled sweeps keep the rows and the solve block of as many
        // contacts as fit in LDS that is free by now: re-read from L2 in every
        // sweep, a contact's record took longer to arrive than its update to run.
        // Layout per contact: J rows [3][nv], response rows [3][nv], then the block's
        // 13 words. The Jacobi and learned modes read rows by other lanes and keep
        // them in global memory. Measured with the passes above: 4096 humanoids at
        // residual 1e-5, 20 control steps, 56.0 -> 51.1 ms.
        const uint32_t rec_words = 6u * nv + kBlockWords;
        const uint32_t fit = L.rows_words / rec_words;
        const uint32_t cached = (kMlp || scheduled || jacobi) ? 0u : (fit < ncons ? fit : ncons);
        auto row_lane = [&]() -> uint32_t { return lane < mnv ? lane : mnv - 1u; };
        auto lds_lane = [&]() -> uint32_t { return lane < nv ? lane : (nv > 0u ? nv - 1u : 0u); };
        auto load_responses = [&](uint32_t c, float* r3) {
            if (c < cached) {
                const LdsFloat* rec = e.rows + c * rec_words + 3u * nv + lds_lane();
#pragma unroll
                for (uint32_t r = 0; r < 3u; ++r) r3[r] = rec[r * nv];
            } else {
                const float* rb = e.resp + (size_t)c * 3u * mnv;
                const uint32_t at = row_lane();
#pragma unroll
                for (uint32_t r = 0; r < 3u; ++r) r3[r] = rb[r * mnv + at];
            }
        };
        // Pass 1, every lane, articulated constraints only: the DoF-lane folds
        // of J v (rows 0-2) and of the 3x3 block J M^-1 J^T, staged in the
        // record. Constraints between scene bodies need no fold and are left
        // to the constraint-lane pass below, which also adds every constraint's
        // scene endpoint terms.
        // The Jacobian rows are made here, a DoF per lane: what a DoF's columns need
        // is read once, a contact's geometry comes as scalars out of one register
        // (lanes 0-31 the hot record, 32-63 the cold record's head), fetched a
        // contact ahead, and the rows are stored coalesced.
        const DofColumn dof_col = dof_column(e, lane);
        auto load_geometry = [&](uint32_t c) -> uint32_t {
            const uint32_t* hw = reinterpret_cast<const uint32_t*>(e.hot + c);
            const uint32_t* cw = reinterpret_cast<const uint32_t*>(e.cold + c);
            return lane < 32u ? hw[lane] : cw[lane < 38u ? lane - 32u : 0u];
        };
        float nr[3] = {0.0f, 0.0f, 0.0f};
        uint32_t art_next = nart > 0u ? art_at(0u) : 0u;
        uint32_t geometry = 0u;
        auto load_global_responses = [&](uint32_t c) {
            const float* rb = e.resp + (size_t)c * 3u * mnv;
            const uint32_t at = row_lane();
#pragma unroll
            for (uint32_t r = 0; r < 3u; ++r) nr[r] = rb[r * mnv + at];
        };
        if (nart > 0u) {
            load_global_responses(art_next);
            geometry = load_geometry(art_next);
        }
        for (uint32_t k = 0; k < nart; ++k) {
            const uint32_t c = art_next;
            float jr[3], rr[3] = {nr[0], nr[1], nr[2]};
            const uint32_t geo = geometry;
            art_next = art_at(k + 1u < nart ? k + 1u : 0u);
            load_global_responses(art_next);
            geometry = load_geometry(art_next);
            if (jacobi && (uniform_u32(e.cpair[c] >> 16) & mr::kHotArticulated) == 0u) continue;
            {
                auto word = [&](uint32_t w) { return read_lane(__uint_as_float(geo), w); };
                auto vec = [&](uint32_t w) { return V3{word(w), word(w + 1u), word(w + 2u)}; };
                constexpr uint32_t kDir = offsetof(HotConstraint, dir) / 4u;
                const uint32_t ba = read_lane(geo, offsetof(HotConstraint, body_a) / 4u);
                const uint32_t bb = read_lane(geo, offsetof(HotConstraint, body_b) / 4u);
                V3 ca{0.0f, 0.0f, 0.0f}, cb{0.0f, 0.0f, 0.0f};
                if (is_link(e, ba))
                    ca = jacobian_column(dof_col, e.topo->anc[ba], vec(32u + offsetof(ColdConstraint, pa) / 4u));
                if (is_link(e, bb))
                    cb = jacobian_column(dof_col, e.topo->anc[bb], vec(32u + offsetof(ColdConstraint, pb) / 4u));
                const V3 col = sub(cb, ca);
                // lanes past the DoFs hold +0 everywhere: their products are +0
#pragma unroll
                for (uint32_t r = 0; r < 3u; ++r) {
                    jr[r] = dof_lane ? dot(vec(kDir + 3u * r), col) : 0.0f;
                    rr[r] = dof_lane ? rr[r] : 0.0f;
                }
            }
            if (c < cached) {
                LdsFloat* rec = e.rows + c * rec_words + lane;
                if (dof_lane) {
#pragma unroll
                    for (uint32_t r = 0; r < 3u; ++r) {
                        rec[r * nv] = jr[r];
                        rec[(3u + r) * nv] = rr[r];
                    }
                }
            } else if (dof_lane) {
                float* jb = e.jrow + (size_t)c * 3u * mnv + lane;
#pragma unroll
                for (uint32_t r = 0; r < 3u; ++r) jb[r * mnv] = jr[r];
            }
            float lo[8] = {jr[0] * vj, jr[1] * vj, jr[2] * vj, jr[0] * rr[0], jr[0] * rr[1], jr[0] * rr[2],
                           jr[1] * rr[0], jr[1] * rr[1]};
            float hi[4] = {jr[1] * rr[2], jr[2] * rr[0], jr[2] * rr[1], jr[2] * rr[2]};
            const float flo = wave_fold_packed<8, 8>(lo, lane), fhi = wave_fold_packed<4, 4>(hi, lane);
            // lane i of the first twelve holds sum i: rows of J v, then of the block
            if (lane < 12u) {
                float* hw = reinterpret_cast<float*>(e.hot + c);
                hw[lane < 3u ? offsetof(HotConstraint, stage) / 4u + lane : lane - 3u] = lane < 8u ? flo : fhi;
            }
        }
        __syncthreads();
        const float slop = cfg.contact_slop;
        const float maxdep = cfg.max_depenetration_velocity;
        for (uint32_t c = lane; c < ncons; c += kLanes) {
            HotConstraint hk = e.hot[c];
            const ColdConstraint ck = e.cold[c];
            if ((hk.kind & mr::kHotArticulated) == 0u) {
                for (int r = 0; r < 3; ++r) hk.stage[r] = 0.0f;
                for (int k = 0; k < 9; ++k) hk.winv[k] = 0.0f;
            }
            if ((hk.kind & (mr::kHotDynamicA | mr::kHotDynamicB)) != 0u) {
                V3 va, vb;
                scene_point_velocities(e, hk.kind, hk.body_a, hk.body_b, V3{hk.point[0], hk.point[1], hk.point[2]}, va, vb);
                for (int r = 0; r < 3; ++r) hk.stage[r] = rel_row(hk.kind, hot_dir(hk, r), va, vb, hk.stage[r]);
            }
            const float rel[3] = {hk.stage[0], hk.stage[1], hk.stage[2]};
            const float slip = sqrt_rn(rel[1] * rel[1] + rel[2] * rel[2]);
            const bool stat = slip <= 1.0e-3f;
            hk.mu_u = stat ? ck.friction[0] : ck.friction[2];
            hk.mu_v = stat ? ck.friction[1] : ck.friction[3];
            const float src_target = ck.separation > 0.0f ? -ck.separation / h : 0.0f;
            const float tau = 2.0f * h;
            const float err = fmind(ck.separation + slop, 0.0f);
            const float ratio = h / tau;
            const float den = 1.0f + 2.0f * 1.0f * ratio + ratio * ratio;
            float stab = -h * err / (tau * tau * den);
            stab = clampd(fmaxd(stab, 0.0f), 0.0f, maxdep);
            if ((hk.flags & MR_CONSTRAINT_FLAG_NEW_IMPACT) != 0u) {
                const float incoming = rel[0] - src_target;
                if (incoming < -ck.restitution_threshold) stab = fmaxd(stab, -ck.restitution * incoming);
            }
            hk.target0 = src_target + stab;
            hk.reg0 = fmaxd(ck.compliance / (h * h) + ck.dissipation / h, 0.0f);
            bool ok = true;
            if (!isfin(hk.target0) || !isfin(hk.reg0)) {
                report_failure(&s_fail, c, MR_STEP_NONFINITE_RESULT, c);
                ok = false;
            }
            if (ok) {
                const V3 x{hk.point[0], hk.point[1], hk.point[2]};
                const bool sa_dyn = (hk.kind & mr::kHotDynamicA) != 0u, sb_dyn = (hk.kind & mr::kHotDynamicB) != 0u;
                float W[3][3];
                for (int r = 0; r < 3; ++r)
                    for (int q = 0; q < 3; ++q) {
                        float val = hk.winv[3 * r + q];
                        if (sa_dyn) val += dot(hot_dir(hk, r), scene_response(e.scene[hk.body_a - nl], x, hot_dir(hk, q)));
                        if (sb_dyn) val += dot(hot_dir(hk, r), scene_response(e.scene[hk.body_b - nl], x, hot_dir(hk, q)));
                        if (r == q) val += r == 0 ? hk.reg0 : 0.0f;  // tangent rows carry none
                        W[r][q] = val;
                    }
                if (!invert3x3(W, hk.winv)) report_failure(&s_fail, c, MR_STEP_FACTORIZATION_FAILED, c);
            }
            float lam[3] = {e.lam[3u * c], e.lam[3u * c + 1u], e.lam[3u * c + 2u]};
            project_cone(lam, hk.mu_u, hk.mu_v, e.a->cfg.maximum_normal_impulse);
            e.lam[3u * c] = lam[0];
            e.lam[3u * c + 1u] = lam[1];
            e.lam[3u * c + 2u] = lam[2];
            e.hot[c] = hk;
            if (c < cached) {
                LdsFloat* blk = e.rows + c * rec_words + 6u * nv;
                for (int k = 0; k < 9; ++k) blk[k] = hk.winv[k];
                blk[9] = hk.target0;
                blk[10] = hk.reg0;
                blk[11] = hk.mu_u;
                blk[12] = hk.mu_v;
            }
        }
        __syncthreads();
        clk.mark(mr::kStageEvaluation);
        if (s_fail != ~0ull) break;
        // -------------------------------------- learned warm start (MLP)
        const uint32_t base_iters = cfg.velocity_iterations + (final_sub ? cfg.final_velocity_iterations : 0u);
        const bool adaptive = cfg.residual_tolerance > 0.0f;
        const uint32_t max_iters = adaptive ? cfg.max_iterations : base_iters;
        float sweep_delta = 0.0f;
        uint32_t iters = 0, sweeps_run = 0;
        bool solve_failed = false;
        const SolveBlock* solve = reinterpret_cast<const SolveBlock*>(e.hot);
        const uint32_t hot_words = (uint32_t)(sizeof(HotConstraint) / sizeof(SolveBlock));
        bool mlp_now = false;
        float* capture_rows = nullptr;
        const float vj_free = vj;
        if constexpr (kMlp) {
            mlp_now = A.mlp_enabled != 0u && ncons > 0u;
            if (A.mlp_samples != nullptr && substep == cfg.capture_substep)
                capture_rows = A.mlp_samples + (size_t)env * ccap * mr::kMlpSampleFloats;
            if (mlp_now || capture_rows != nullptr)
                mlp_now = mlp_warm_start(e, lane, ncons, mnv, mlp_now, capture_rows) && mlp_now;
        }
        // The plain path runs the attempt below once. When the MLP replaced any
        // warm start, a microstep whose sweeps miss the residual tolerance is
        // solved again from the plain warm start and the same free velocity.
        for (uint32_t attempt = 0;; ++attempt) {
            lane = stage_lane(lane);
            sweep_delta = 0.0f;
            iters = 0;
            if (cfg.solver == MR_SOLVER_RELAXED_JACOBI) {
                // ---------------------------------- relaxed block Jacobi
                // Lanes own contacts for the proposals, DoFs and scene bodies for
                // the velocity update (jacobi_apply).
                // damping per contact: diag / sum_j |W_nn(c, j)| clamped to [1/32, 1] (:6722-6798)
                for (uint32_t c = lane; c < ncons; c += kLanes) {
                    float sum = 0.0f, diag = 0.0f;
                    for (uint32_t j = 0; j < ncons; ++j) {
                        const float w = fabs_(jacobi_normal_cross(e, c, j, mnv));
                        sum = sum + w;
                        if (j == c) diag = w + e.hot[c].reg0;
                    }
                    e.jrelax[c] = sum > fmaxd(diag, kMatrixFloor) ? clampd(diag / sum, 1.0f / 32.0f, 1.0f) : 1.0f;
                }
                // warm start: the projected warm impulses are the first deltas (:6402-6470)
                for (uint32_t i = lane; i < 3u * ncons; i += kLanes) e.jdelta[i] = e.lam[i];
                __syncthreads();
                jacobi_apply(e, lane, ncons, mnv, dof_lane, vj);
                __syncthreads();
                clk.mark(mr::kStageWarmStart);
                float largest = 0.0f;
                for (uint32_t it = 0; it < max_iters && ncons > 0u; ++it) {
                    if (dof_lane) e.vcand[lane] = vj;
                    __syncthreads();
                    float my_delta = 0.0f;
                    uint32_t my_fail = MR_INVALID_INDEX;
                    for (uint32_t c = lane; c < ncons; c += kLanes) {
                        const SolveBlock sb = solve[(size_t)c * hot_words];
                        const uint32_t kind = e.cpair[c] >> 16;
                        const HotConstraint& hk = e.hot[c];
                        float rel[3] = {0.0f, 0.0f, 0.0f};
                        if ((kind & mr::kHotArticulated) != 0u) {
                            const float* jb = e.jrow + (size_t)c * 3u * mnv;
                            for (int r = 0; r < 3; ++r) rel[r] = serial_dot(jb + (size_t)r * mnv, e.vcand, nv);
                        }
                        if ((kind & (mr::kHotDynamicA | mr::kHotDynamicB)) != 0u) {
                            V3 va, vb;
                            scene_point_velocities(e, kind, hk.body_a, hk.body_b, V3{hk.point[0], hk.point[1], hk.point[2]},
                                                   va, vb);
                            for (int r = 0; r < 3; ++r) rel[r] = rel_row(kind, hot_dir(hk, r), va, vb, rel[r]);
                        }
                        const float lam[3] = {e.lam[3u * c], e.lam[3u * c + 1u], e.lam[3u * c + 2u]};
                        const float tgt[3] = {sb.target0, 0.0f, 0.0f}, reg[3] = {sb.reg0, 0.0f, 0.0f};
                        float rhs[3];
                        for (int r = 0; r < 3; ++r) rhs[r] = (tgt[r] - rel[r]) - reg[r] * lam[r];
                        float prop[3] = {lam[0], lam[1], lam[2]};
                        for (int r = 0; r < 3; ++r)
                            for (int q = 0; q < 3; ++q) prop[r] += sb.winv[3 * r + q] * rhs[q];
                        project_cone(prop, sb.mu_u, sb.mu_v, e.a->cfg.maximum_normal_impulse);
                        const float relax = e.jrelax[c];
                        float d[3], cand[3];
                        for (int r = 0; r < 3; ++r) {
                            d[r] = relax * (prop[r] - lam[r]);
                            cand[r] = lam[r] + d[r];
                        }
                        if (!isfin(cand[0]) || !isfin(cand[1]) || !isfin(cand[2]) || !isfin(d[0]) || !isfin(d[1]) ||
                            !isfin(d[2])) {
                            my_fail = c < my_fail ? c : my_fail;
                            continue;
                        }
                        for (int r = 0; r < 3; ++r) {
                            e.lam[3u * c + r] = cand[r];
                            e.jdelta[3u * c + r] = d[r];
                        }
                        my_delta = fmaxd(my_delta, fmaxd(fabs_(d[0]), fmaxd(fabs_(d[1]), fabs_(d[2]))));
                    }
                    const uint32_t first_fail = wave_min_u32(my_fail);
                    if (first_fail != MR_INVALID_INDEX) {
                        if (lane == 0u) s_fail = ((unsigned long long)MR_STEP_NONFINITE_RESULT << 24) | (first_fail & 0xffffffu);
                        solve_failed = true;
                        break;
                    }
                    __syncthreads();
                    jacobi_apply(e, lane, ncons, mnv, dof_lane, vj);
                    __syncthreads();
                    const float it_delta = wave_max(my_delta);
                    largest = fmaxd(largest, it_delta);
                    ++iters;
                    if (adaptive && it_delta <= cfg.residual_tolerance) break;
                }
                sweep_delta = largest;
            } else {
            // ---------------------------------------------------- warm start
            // DoF lanes accumulate the warm-start impulses of the articulated
            // contacts in index order, the next contact's response rows in flight;
            // scene bodies take theirs in schedule order.
            const uint32_t* pack = reinterpret_cast<const uint32_t*>(e.resid);
            const uint32_t pack_lane = scheduled && lane <= levels ? pack[lane] : 0u;
            auto level_pack = [&](uint32_t l) { return l < kLanes ? read_lane(pack_lane, l) : uniform_u32(pack[l]); };
            // the scene contact of this lane in a level of n entries from `first`
            // (a lane past them reads the last one's record and stays idle)
            auto sched_contact = [&](uint32_t first, uint32_t n) -> uint32_t {
                return e.sord[first + (lane < n ? lane : (n > 0u ? n - 1u : 0u))];
            };
            if (nart > 0u) {
                uint32_t an = art_at(0u);
                load_responses(an, nr);
                for (uint32_t k = 0; k < nart; ++k) {
                    const uint32_t c = an;
                    const float c0 = nr[0], c1 = nr[1], c2 = nr[2];
                    an = art_at(k + 1u < nart ? k + 1u : 0u);
                    load_responses(an, nr);
                    const float* lc = e.lam + 3u * c;
                    vj += (c0 * lc[0] + c1 * lc[1]) + c2 * lc[2];
                }
                if (!dof_lane) vj = 0.0f;
            }
            if (scheduled) {
                for (uint32_t b = lane; b < nsc; b += kLanes) load_solver_body(e, b);
                __syncthreads();
                auto warm_contact = [&](uint32_t c) {
                    const HotConstraint& hk = e.hot[c];
                    const float* lc = e.lam + 3u * c;
                    const V3 imp = add(add(mul(lc[0], hot_dir(hk, 0)), mul(lc[1], hot_dir(hk, 1))), mul(lc[2], hot_dir(hk, 2)));
                    const V3 x{hk.point[0], hk.point[1], hk.point[2]};
                    if ((hk.kind & mr::kHotDynamicA) != 0u)
                        solver_apply_impulse(e.sbody + (hk.body_a - nl) * kSolverBodyVectors, x, neg(imp));
                    if ((hk.kind & mr::kHotDynamicB) != 0u)
                        solver_apply_impulse(e.sbody + (hk.body_b - nl) * kSolverBodyVectors, x, imp);
                };
                for (uint32_t l = 0; l < levels; ++l) {
                    const uint32_t pk = level_pack(l);
                    const uint32_t first = pk & 0xffffu, end = level_pack(l + 1u) & 0xffffu;
                    for (uint32_t p = first + lane; p < end; p += kLanes) warm_contact(e.sord[p]);
                    if ((pk >> 16) != 0u && lane == 0u) warm_contact((pk >> 16) - 1u);
                    __builtin_amdgcn_wave_barrier();
                }
            }
            __syncthreads();
            clk.mark(mr::kStageWarmStart);
            // ------------------------------------------ ordered block sweeps
            // The update of one articulated contact, a serial chain of instructions
            // whose number is its time: the three row sums finish in one packed
            // chain, and from there lane r of every quad (row 3 repeating row 2)
            // works on row r alone: its right-hand side, its row of the block, its
            // tangent's share of the cone. Only the values the rows exchange cross
            // lanes, by quad permutations: about 110 instructions instead of 250. DoF
            // lanes keep the candidate velocity in a register, and the next
            // articulated contact's rows and block slice (5 words a lane) are fetched
            // meanwhile. Measured with the stage-local lane index: 4096 humanoids at
            // residual 1e-5, 20 control steps, 77.5 -> 62.4 ms.
            const uint32_t row = (lane & 3u) < 2u ? (lane & 3u) : 2u;
            struct ContactRegs {
                float j[3], r[3];       // this DoF lane's Jacobian and response rows
                float w[3], mu, target; // this lane's row of the block; reg0, mu_u or mu_v; target0
            };
            static_assert(offsetof(HotConstraint, mu_u) == offsetof(HotConstraint, reg0) + 4u &&
                          offsetof(HotConstraint, mu_v) == offsetof(HotConstraint, reg0) + 8u, "reg0, mu_u, mu_v adjoin");
            constexpr uint32_t kMu = offsetof(HotConstraint, reg0) / 4u, kTarget = offsetof(HotConstraint, target0) / 4u;
            auto load_lds_contact = [&](uint32_t c, ContactRegs& g) {
                const LdsFloat* rec = e.rows + c * rec_words;
                const LdsFloat* at = rec + lds_lane();
                const LdsFloat* blk = rec + 6u * nv;
#pragma unroll
                for (uint32_t q = 0; q < 3u; ++q) {
                    g.j[q] = at[q * nv];
                    g.r[q] = at[(3u + q) * nv];
                    g.w[q] = blk[3u * row + q];
                }
                g.mu = blk[kMu + row];
                g.target = blk[kTarget];
            };
            auto load_contact = [&](uint32_t c, ContactRegs& g) {
                const float* jb = e.jrow + (size_t)c * 3u * mnv;
                const float* rb = e.resp + (size_t)c * 3u * mnv;
                const float* hw = reinterpret_cast<const float*>(e.hot + c);
                const uint32_t at = row_lane();
#pragma unroll
                for (uint32_t q = 0; q < 3u; ++q) {
                    g.j[q] = jb[q * mnv + at];
                    g.r[q] = rb[q * mnv + at];
                    g.w[q] = hw[3u * row + q];
                }
                g.mu = hw[kMu + row];
                g.target = hw[kTarget];
            };
            const float max_normal_impulse = cfg.maximum_normal_impulse;
            // Updates contact c from `g`; `prefetch` then refills g with a later
            // contact. Returns false when the update is not finite (nothing is
            // written then).
            auto articulated_update = [&](auto scene_tag, uint32_t c, ContactRegs& g, auto prefetch) -> bool {
                constexpr bool kScene = decltype(scene_tag)::value;
                const float lam = e.lam[3u * c + row];
                float rel3[3];
                float rr[3];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    rel3[r] = dof_lane ? g.j[r] * vj : 0.0f;
                    rr[r] = g.r[r];
                }
                const float w0 = g.w[0], w1 = g.w[1], w2 = g.w[2], mu = g.mu;
                const float target = row == 0u ? g.target : 0.0f, reg = row == 0u ? g.mu : 0.0f;
                prefetch();
                float rel = wave_fold_packed<3, 4>(rel3, lane);
                uint32_t kind = 0u, ba = 0u, bb = 0u;
                V3 x{0.0f, 0.0f, 0.0f}, dir{0.0f, 0.0f, 0.0f};
                if constexpr (kScene) {
                    const uint32_t pr = uniform_u32(e.cpair[c]);
                    kind = pr >> 16;
                    ba = pr & 0xffu;
                    bb = (pr >> 8) & 0xffu;
                    if ((kind & (mr::kHotDynamicA | mr::kHotDynamicB)) != 0u) {
                        const HotConstraint& hk = e.hot[c];
                        x = V3{hk.point[0], hk.point[1], hk.point[2]};
                        dir = V3{hk.dir[3u * row], hk.dir[3u * row + 1u], hk.dir[3u * row + 2u]};
                        V3 va{0.0f, 0.0f, 0.0f}, vb{0.0f, 0.0f, 0.0f};
                        if ((kind & mr::kHotDynamicA) != 0u)
                            va = solver_point_velocity(e.sbody + (ba - nl) * kSolverBodyVectors, x);
                        if ((kind & mr::kHotDynamicB) != 0u)
                            vb = solver_point_velocity(e.sbody + (bb - nl) * kSolverBodyVectors, x);
                        rel = rel_row(kind, dir, va, vb, rel);
                    }
                }
                // the tangent rows' target and regularisation are +0
                const float rhs = (target - rel) - reg * lam;
                float cand = lam;
                cand += w0 * quad_broadcast<0>(rhs);
                cand += w1 * quad_broadcast<1>(rhs);
                cand += w2 * quad_broadcast<2>(rhs);
                // project_cone, a tangent per lane
                float normal = fmaxd(quad_broadcast<0>(cand), 0.0f);
                if (max_normal_impulse > 0.0f) normal = fmind(normal, max_normal_impulse);
                const float bound = mu * normal;
                if (wave_any(row != 0u && !(bound > 0.0f))) {
                    cand = row == 0u ? normal : 0.0f;
                } else {
                    const float share = (cand * cand) / (bound * bound);
                    const float ns = quad_broadcast<1>(share) + quad_broadcast<2>(share);
                    if (wave_any(ns > 1.0f)) cand *= 1.0f / sqrt_rn(ns);
                    cand = row == 0u ? normal : cand;
                }
                const float d = cand - lam;
                if (wave_any(!isfin(cand) | !isfin(d))) return false;
                sweep_delta = fmaxd(sweep_delta, fabs_(d));
                const float d0 = quad_broadcast<0>(d), d1 = quad_broadcast<1>(d), d2 = quad_broadcast<2>(d);
                if (dof_lane) vj += (rr[0] * d0 + rr[1] * d1) + rr[2] * d2;
                // The workgroup is one wavefront and its LDS operations
                // complete in issue order, so the writes below follow every
                // lane's reads above and precede the next contact's reads; the
                // wave barrier only stops the compiler from moving memory
                // operations across these points.
                __builtin_amdgcn_wave_barrier();
                if constexpr (kScene) {
                    if ((kind & (mr::kHotDynamicA | mr::kHotDynamicB)) != 0u) {
                        const V3 m = mul(d, dir);
                        const V3 imp{(quad_broadcast<0>(m.x) + quad_broadcast<1>(m.x)) + quad_broadcast<2>(m.x),
                                     (quad_broadcast<0>(m.y) + quad_broadcast<1>(m.y)) + quad_broadcast<2>(m.y),
                                     (quad_broadcast<0>(m.z) + quad_broadcast<1>(m.z)) + quad_broadcast<2>(m.z)};
                        if (lane == 0u) {
                            if ((kind & mr::kHotDynamicA) != 0u)
                                solver_apply_impulse(e.sbody + (ba - nl) * kSolverBodyVectors, x, neg(imp));
                            if ((kind & mr::kHotDynamicB) != 0u)
                                solver_apply_impulse(e.sbody + (bb - nl) * kSolverBodyVectors, x, imp);
                        }
                    }
                }
                if (lane < 3u) e.lam[3u * c + lane] = cand;
                __builtin_amdgcn_wave_barrier();
                return true;
            };
            if (!scheduled) {
                // every contact joins the articulation to static geometry: one
                // chain, first the contacts whose records LDS holds, then the others
                ContactRegs near_regs, far_regs;
                if (cached > 0u) load_lds_contact(0u, near_regs);
                if (cached < ncons) load_contact(cached, far_regs);
                for (uint32_t it = 0; it < max_iters && ncons > 0u; ++it) {
                    sweep_delta = 0.0f;
                    uint32_t c = 0u;
                    bool ok = true;
                    for (; ok && c < cached; ++c)
                        ok = articulated_update(BoolTag<false>{}, c, near_regs,
                                                [&] { load_lds_contact(c + 1u < cached ? c + 1u : 0u, near_regs); });
                    for (; ok && c < ncons; ++c)
                        ok = articulated_update(BoolTag<false>{}, c, far_regs,
                                                [&] { load_contact(c + 1u < ncons ? c + 1u : cached, far_regs); });
                    if (!ok) {
                        if (lane == 0u) s_fail = ((unsigned long long)MR_STEP_NONFINITE_RESULT << 24) | ((c - 1u) & 0xffffffu);
                        solve_failed = true;
                    }
                    if (solve_failed) break;
                    ++iters;
                    if (adaptive && !wave_any(!(sweep_delta <= cfg.residual_tolerance))) break;
                }
                sweep_delta = wave_max(sweep_delta);
            } else {
                // Level by level: the level's contacts between scene bodies one per
                // lane, their records fetched a level ahead, then its articulated
                // contact. A sweep runs to its end before a failure is reported:
                // contacts before the first failing index are untouched by it, so
                // the smallest failing index is the one the index order meets first.
                uint32_t k_art = 0u;
                uint32_t cn = nart > 0u ? art_at(0u) : 0u;
                ContactRegs regs;
                if (nart > 0u) load_contact(cn, regs);
                uint32_t pk = level_pack(0u), pk_next = level_pack(1u);
                uint32_t cc = sched_contact(pk & 0xffffu, (pk_next & 0xffffu) - (pk & 0xffffu));
                HotConstraint rec = e.hot[cc];
                for (uint32_t it = 0; it < max_iters; ++it) {
                    sweep_delta = 0.0f;
                    uint32_t my_fail = MR_INVALID_INDEX;
                    for (uint32_t l = 0; l < levels; ++l) {
                        const uint32_t first = pk & 0xffffu, end = pk_next & 0xffffu, art_c = pk >> 16;
                        const uint32_t ln = l + 1u < levels ? l + 1u : 0u;
                        pk = level_pack(ln);
                        pk_next = level_pack(ln + 1u);
                        auto scene_contact = [&](uint32_t c, const HotConstraint& hk) {
                            const bool da = (hk.kind & mr::kHotDynamicA) != 0u, db = (hk.kind & mr::kHotDynamicB) != 0u;
                            float4* sa = e.sbody + (da ? hk.body_a - nl : 0u) * kSolverBodyVectors;
                            float4* sbp = e.sbody + (db ? hk.body_b - nl : 0u) * kSolverBodyVectors;
                            const V3 x{hk.point[0], hk.point[1], hk.point[2]};
                            const float lam0 = e.lam[3u * c], lam1 = e.lam[3u * c + 1u], lam2 = e.lam[3u * c + 2u];
                            V3 va{0.0f, 0.0f, 0.0f}, vb{0.0f, 0.0f, 0.0f};
                            if (da) va = solver_point_velocity(sa, x);
                            if (db) vb = solver_point_velocity(sbp, x);
                            float rel[3];
#pragma unroll
                            for (int r = 0; r < 3; ++r) rel[r] = rel_row(hk.kind, hot_dir(hk, r), va, vb, 0.0f);
                            float cand[3];
                            if (!block_update(hk, rel, lam0, lam1, lam2, cfg.maximum_normal_impulse, cand, sweep_delta)) {
                                my_fail = c < my_fail ? c : my_fail;
                                return;
                            }
                            const float d0 = cand[0] - lam0, d1 = cand[1] - lam1, d2 = cand[2] - lam2;
                            const V3 imp = add(add(mul(d0, hot_dir(hk, 0)), mul(d1, hot_dir(hk, 1))), mul(d2, hot_dir(hk, 2)));
                            if (da) solver_apply_impulse(sa, x, neg(imp));
                            if (db) solver_apply_impulse(sbp, x, imp);
                            e.lam[3u * c] = cand[0];
                            e.lam[3u * c + 1u] = cand[1];
                            e.lam[3u * c + 2u] = cand[2];
                        };
                        // Most levels of a robot beside a few objects hold its own
                        // contact only, and fetch no record. (With one fetched for
                        // every level, 512 chains of 20 links and a free box, 2
                        // control steps to residual 1e-5, took 40.1 ms, now 35.1.)
                        if (first < end || (pk & 0xffffu) < (pk_next & 0xffffu)) {
                            const uint32_t c0 = cc;
                            const HotConstraint h0 = rec;
                            cc = sched_contact(pk & 0xffffu, (pk_next & 0xffffu) - (pk & 0xffffu));
                            rec = e.hot[cc];
                            if (first + lane < end) scene_contact(c0, h0);
                            for (uint32_t p = first + kLanes + lane; p < end; p += kLanes) {
                                const uint32_t c = e.sord[p];
                                scene_contact(c, e.hot[c]);
                            }
                            __builtin_amdgcn_wave_barrier();
                        }
                        if (art_c != 0u) {
                            k_art = k_art + 1u < nart ? k_art + 1u : 0u;
                            cn = art_at(k_art);
                            if (!articulated_update(BoolTag<true>{}, art_c - 1u, regs, [&] { load_contact(cn, regs); }))
                                my_fail = art_c - 1u < my_fail ? art_c - 1u : my_fail;
                        }
                    }
                    if (wave_any(my_fail != MR_INVALID_INDEX)) {
                        const uint32_t first_fail = wave_min_u32(my_fail);
                        if (lane == 0u)
                            s_fail = ((unsigned long long)MR_STEP_NONFINITE_RESULT << 24) | (first_fail & 0xffffffu);
                        solve_failed = true;
                        break;
                    }
                    ++iters;
                    if (adaptive && !wave_any(!(sweep_delta <= cfg.residual_tolerance))) break;
                }
                sweep_delta = wave_max(sweep_delta);
                __syncthreads();
                for (uint32_t b = lane; b < nsc; b += kLanes)
                    if (is_dynamic_scene(e, nl + b)) store_solver_body(e, b);
            }
            }
            __syncthreads();
            clk.mark(mr::kStageSweeps);
            sweeps_run += iters;
            if constexpr (kMlp) {
                if (mlp_now && attempt == 0u && adaptive && !solve_failed) {
                    const bool missed = !(sweep_delta <= cfg.residual_tolerance);
                    bool diverged = false;
                    if (!missed && A.mlp.max_normal_residual > 0.0f) {
                        // The learned solve reached the tolerance: its normal
                        // residuals, computed as the residual pass below does,
                        // must also stay within max_normal_residual. (Their
                        // articulated terms go to the MLP tile's LDS, free by
                        // now: a second attempt reads the schedule in e.resid.)
                        float* res_n = reinterpret_cast<float*>(e.mlp_lds);
                        for (uint32_t c = 0; c < ncons; ++c) {
                            if ((uniform_u32(e.cpair[c] >> 16) & mr::kHotArticulated) == 0u) continue;
                            const float j0 = e.jrow[(size_t)c * 3u * mnv + row_lane()];
                            const float a0 = wave_fold(dof_lane ? j0 * vj : 0.0f);
                            if (lane == 0u) res_n[c] = a0;
                        }
                        __syncthreads();
                        bool over = false;
                        for (uint32_t c = lane; c < ncons; c += kLanes) {
                            const HotConstraint hk = e.hot[c];
                            float rel0 = (hk.kind & mr::kHotArticulated) != 0u ? res_n[c] : 0.0f;
                            if ((hk.kind & (mr::kHotDynamicA | mr::kHotDynamicB)) != 0u) {
                                V3 va, vb;
                                scene_point_velocities(e, hk.kind, hk.body_a, hk.body_b,
                                                       V3{hk.point[0], hk.point[1], hk.point[2]}, va, vb);
                                rel0 = rel_row(hk.kind, hot_dir(hk, 0), va, vb, rel0);
                            }
                            const float l0 = e.lam[3u * c];
                            const float eq = (rel0 - hk.target0) + hk.reg0 * l0;
                            const float nres = l0 > kConeEpsilon ? fabs_(eq) : fmaxd(-eq, 0.0f);
                            over = over || !(nres <= A.mlp.max_normal_residual);
                        }
                        diverged = __ballot(over) != 0ull;
                        __syncthreads();
                    }
                    if (missed || diverged) {
                        vj = vj_free;
                        for (uint32_t i = lane; i < 3u * ncons; i += kLanes) e.lam[i] = e.mlp_lam[i];
                        for (uint32_t b = lane; b < nsc; b += kLanes) e.scene[b] = e.mlp_scene[b];
                        if (lane == 0u) {
                            cs.diagnostics.z += 1.0f;
                            if (diverged) cs.diagnostics.w += 1.0f;
                        }
                        __syncthreads();
                        continue;
                    }
                }
            }
            break;
        }
        if constexpr (kMlp) {
            // capture targets: the impulse the solve converged to
            if (capture_rows != nullptr && !solve_failed) {
                for (uint32_t c = lane; c < ccap; c += kLanes) {
                    float* row = capture_rows + (size_t)c * mr::kMlpSampleFloats;
                    if (c < ncons) {
                        row[8] = e.lam[3u * c];
                        row[9] = e.lam[3u * c + 1u];
                        row[10] = e.lam[3u * c + 2u];
                    }
                    row[11] = c < ncons ? 1.0f : 0.0f;
                }
            }
        }
        if (s_fail != ~0ull) break;
        // ------------------------------------- residuals + impulse store
        lane = stage_lane(lane);
        // Pass 1, every lane, articulated constraints only: the DoF-lane fold
        // of the normal row's J v.
        float* res_n = e.resid;                 // [ccap]: articulated J v, then the normal residual
        float* res_c = e.resid + ccap;          // [ccap]: cone violation
        for (uint32_t k0 = 0; k0 < nart; k0 += 4u) {
            // four contacts a pass, one packed fold (Jacobi: rows of the others
            // were never written and their sums are not read)
            float f[4];
            uint32_t mine = 0u;
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) {
                const uint32_t c = art_at(k0 + i < nart ? k0 + i : nart - 1u);
                mine = (lane & 3u) == i ? c : mine;
                float j0;
                if (c < cached) j0 = e.rows[c * rec_words + lds_lane()];
                else j0 = e.jrow[(size_t)c * 3u * mnv + row_lane()];
                f[i] = dof_lane ? j0 * vj : 0.0f;
            }
            const float a = wave_fold_packed<4, 4>(f, lane);
            if (lane < 4u && k0 + lane < nart) res_n[mine] = a;
        }
        __syncthreads();
        // Pass 2, constraint lanes: the dynamic scene endpoints' terms of the
        // normal-row relative velocity, residual terms and the impulse store.
        float lane_normal = 0.0f, lane_cone = 0.0f;
        bool lane_odd = false;
        for (uint32_t c = lane; c < ncons; c += kLanes) {
            const HotConstraint hk = e.hot[c];
            float rel0 = (hk.kind & mr::kHotArticulated) != 0u ? res_n[c] : 0.0f;
            if ((hk.kind & (mr::kHotDynamicA | mr::kHotDynamicB)) != 0u) {
                V3 va, vb;
                scene_point_velocities(e, hk.kind, hk.body_a, hk.body_b, V3{hk.point[0], hk.point[1], hk.point[2]}, va, vb);
                rel0 = rel_row(hk.kind, hot_dir(hk, 0), va, vb, rel0);
            }
            const float lamr[3] = {e.lam[3u * c], e.lam[3u * c + 1u], e.lam[3u * c + 2u]};
            const float eq = (rel0 - hk.target0) + hk.reg0 * lamr[0];
            const float nres = lamr[0] > kConeEpsilon ? fabs_(eq) : fmaxd(-eq, 0.0f);
            const float lu = hk.mu_u * lamr[0], lv = hk.mu_v * lamr[0];
            float viol;
            if (lu > 0.0f && lv > 0.0f)
                viol = fmaxd(sqrt_rn((lamr[1] * lamr[1]) / (lu * lu) + (lamr[2] * lamr[2]) / (lv * lv)) - 1.0f, 0.0f);
            else
                viol = sqrt_rn(lamr[1] * lamr[1] + lamr[2] * lamr[2]);
            res_n[c] = nres;
            res_c[c] = viol;
            lane_normal = fmaxd(lane_normal, nres);
            lane_cone = fmaxd(lane_cone, viol);
            lane_odd = lane_odd || !isfin(nres) || !isfin(viol);
            const ColdConstraint& ck = e.cold[c];
            new_p[(size_t)ck.manifold * MR_MANIFOLD_POINT_CAPACITY + ck.point].impulses =
                mr_float4{lamr[0], lamr[1], lamr[2], kCcd ? h : 0.0f};
        }
        __syncthreads();
        // Pass 3: maxima. Finite non-negative terms have one maximum in any
        // order; a non-finite one is met in constraint order (the oracle's).
        float max_normal, max_cone;
        if (wave_any(lane_odd)) {
            max_normal = 0.0f;
            max_cone = 0.0f;
            for (uint32_t c = 0; c < ncons; ++c) {
                max_normal = fmaxd(max_normal, res_n[c]);
                max_cone = fmaxd(max_cone, res_c[c]);
            }
        } else {
            max_normal = wave_max(lane_normal);
            max_cone = wave_max(lane_cone);
        }
        if (dof_lane) e.vcand[lane] = vj;
        __syncthreads();
        if (!isfin(sweep_delta) || !isfin(max_normal) || !isfin(max_cone)) {
            if (lane == 0u) s_fail = ((unsigned long long)MR_STEP_NONFINITE_RESULT << 24) | 0xffffffu;
            __syncthreads();
            break;
        }
        cs.solver_iterations = ncons > 0u ? iters : 0u;
        cs.residuals = mr_float4{ncons > 0u ? sweep_delta : 0.0f, max_normal, max_cone,
                                 cs.residuals.w + (float)(ncons > 0u ? sweeps_run : 0u)};
        // Islands: components of the contact graph over the used nodes (lane 0
        // the articulation, lane 1 + s scene body s), one label per lane, the
        // smallest node of its component. An edge relabels the larger component
        // label at once; most contacts have one node and touch only `node_used`.
        uint32_t islands = 0u;
        {
            uint32_t label = lane;
            bool node_used = false;
            for (uint32_t base = 0; base < ncons; base += kLanes) {
                const uint32_t n = ncons - base < kLanes ? ncons - base : kLanes;
                const uint32_t pairs = lane < n ? e.cpair[base + lane] : 0u;
                for (uint32_t i = 0; i < n; ++i) {
                    const uint32_t p = read_lane(pairs, i);
                    const uint32_t ba = p & 0xffu, bb = (p >> 8) & 0xffu;
                    const uint32_t na = ba < nl ? 0u : (((p >> 16) & mr::kHotDynamicA) != 0u ? 1u + (ba - nl) : kLanes);
                    const uint32_t nb = bb < nl ? 0u : (((p >> 16) & mr::kHotDynamicB) != 0u ? 1u + (bb - nl) : kLanes);
                    node_used = node_used || lane == na || lane == nb;
                    if (na < kLanes && nb < kLanes) {
                        const uint32_t la = read_lane(label, na), lb = read_lane(label, nb);
                        const uint32_t lo = la < lb ? la : lb, hi = la < lb ? lb : la;
                        label = label == hi ? lo : label;
                    }
                }
            }
            islands = (uint32_t)__popcll(__ballot(node_used && label == lane));
        }
        // ------------------------------------------------- joint limits
        lane = stage_lane(lane);
        for (uint32_t j = lane; j < nv; j += kLanes) {
            const MRDofC& dof = e.dofs[j];
            float vel = e.vcand[j];
            if ((dof.flags & MR_DOF_FLAG_VELOCITY_LIMIT) != 0u) vel = clampd(vel, -dof.limits.z, dof.limits.z);
            if ((dof.flags & MR_DOF_FLAG_POSITION_LIMIT) != 0u && dof.q_index != MR_INVALID_INDEX) {
                const float pos = e.q[dof.q_index];
                vel = clampd(vel, (dof.limits.x - pos) / h, (dof.limits.y - pos) / h);
            }
            if (!isfin(vel)) report_failure(&s_fail, j, MR_STEP_NONFINITE_RESULT, j);
            e.vcand[j] = vel;
        }
        __syncthreads();
        cs.islands = islands;
        clk.mark(mr::kStageResiduals);
        if (s_fail != ~0ull) break;
        // ---------------------------------------------------- integration
        lane = stage_lane(lane);
        // New coordinates are staged in registers / s_root and written after
        // a barrier, because other lanes still read q in this phase.
        float qnew = 0.0f;
        uint32_t qslot = MR_INVALID_INDEX;
        if (lane == 0u && floating) {
            const Q4 inc = rotation_increment(V3{h * e.vcand[3], h * e.vcand[4], h * e.vcand[5]});
            Q4 o;
            if (!normalized_quat(qmul(inc, Q4{e.q[3], e.q[4], e.q[5], e.q[6]}), o)) {
                report_failure(&s_fail, 0u, MR_STEP_NONFINITE_RESULT, 3u);
                o = Q4{e.q[3], e.q[4], e.q[5], e.q[6]};
            }
            for (uint32_t i = 0; i < 3u; ++i) {
                s_root[i] = e.q[i] + h * e.vcand[i];
                if (!isfin(s_root[i])) report_failure(&s_fail, 1u + i, MR_STEP_NONFINITE_RESULT, i);
            }
            s_root[3] = o.x;
            s_root[4] = o.y;
            s_root[5] = o.z;
            s_root[6] = o.w;
        }
        for (uint32_t i = 1u + lane; i < nl; i += kLanes) {
            const MRBodyC& b = e.bodies[i];
            if (b.q_index != MR_INVALID_INDEX) {
                qslot = b.q_index;
                qnew = e.q[b.q_index] + h * e.vcand[b.v_index];
                if (!isfin(qnew)) report_failure(&s_fail, 1u + b.q_index, MR_STEP_NONFINITE_RESULT, b.q_index);
            }
        }
        for (uint32_t s = lane; s < nsc; s += kLanes) {
            const uint32_t b = nl + s;
            const MRBodyC& bp = e.bodies[b];
            if (bp.motion_type != MR_MOTION_DYNAMIC) continue;
            MRBodyStateC st = e.scene[s];
            V3 lin = f3(st.linear_velocity_inv_mass);
            V3 ang = f3(st.angular_velocity);
            const float ll = length(lin), al = length(ang);
            if (bp.damping.z > 0.0f && ll > bp.damping.z) lin = mul(bp.damping.z / ll, lin);
            if (bp.damping.w > 0.0f && al > bp.damping.w) ang = mul(bp.damping.w / al, ang);
            st.linear_velocity_inv_mass.x = lin.x;
            st.linear_velocity_inv_mass.y = lin.y;
            st.linear_velocity_inv_mass.z = lin.z;
            st.angular_velocity.x = ang.x;
            st.angular_velocity.y = ang.y;
            st.angular_velocity.z = ang.z;
            const V3 np = add(f3(st.position), mul(h, lin));
            st.position = mr_float4{np.x, np.y, np.z, 1.0f};
            const Q4 inc = rotation_increment(mul(h, ang));
            Q4 o;
            if (!normalized_quat(qmul(inc, q4(st.orientation)), o) || !finite3(np)) {
                report_failure(&s_fail, 0x10000u + b, MR_STEP_NONFINITE_RESULT, b);
                continue;
            }
            st.orientation = mr_float4{o.x, o.y, o.z, o.w};
            world_inverse_inertia(bp, o, st);
            e.scene[s] = st;
        }
        __syncthreads();
        if (s_fail != ~0ull) break;
        if (qslot != MR_INVALID_INDEX) e.q[qslot] = qnew;
        if (lane == 0u && floating)
            for (uint32_t i = 0; i < 7u; ++i) e.q[i] = s_root[i];
        for (uint32_t j = lane; j < nv; j += kLanes) e.v[j] = e.vcand[j];
        __syncthreads();
        if (s_fail != ~0ull) break;
        // --------------------------------------------- microstep commit
        if (lane == 0u) A.mcount[(size_t)dst_buf * E + env] = nman;
        mcount_src = nman;
        src_buf = dst_buf;
        dst_buf = dst_buf == (cur + 1u) % 3u ? alt_buf : (cur + 1u) % 3u;
        if (!impact) successful = substep + 1u;
        min_piv = fmind(min_piv, s_fmax[0]);
        max_piv = fmaxd(max_piv, s_fmax[1]);
        float my_acc = 0.0f;
        for (uint32_t j = lane; j < nv; j += kLanes) my_acc = fmaxd(my_acc, fabs_(e.accel[j]));
        max_acc = fmaxd(max_acc, wave_max(my_acc));
        __syncthreads();
        clk.mark(mr::kStageIntegration);
        if constexpr (kCcd) {
            if (impact) {
                remaining -= h;
                ++segment;
                ++impact_segments;  // counted once the segment commits
                continue;
            }
            remaining = A.h;
            segment = 0u;
        }
        ++substep;
    }
    if constexpr (kCcd) e.h = A.h;

    // ------------------------------------------- transactional commit
    lane = stage_lane(lane);
    __syncthreads();
    const unsigned long long fk = s_fail;
    const bool failed = fk != ~0ull;
    const uint32_t code = failed ? (uint32_t)((fk >> 24) & 0xffull) : MR_STEP_SUCCESS;
    uint32_t findex = failed ? (uint32_t)(fk & 0xffffffull) : MR_INVALID_INDEX;
    if (findex == 0xffffffu) findex = MR_INVALID_INDEX;
    if (failed) failing_substep = successful;
    if (!failed) {
        for (uint32_t i = lane; i < nq; i += kLanes) gq[i] = e.q[i];
        for (uint32_t j = lane; j < nv; j += kLanes) gv[j] = e.v[j];
        for (uint32_t s = lane; s < nsc; s += kLanes) gs[s] = e.scene[s];
        if (A.acceleration != nullptr)
            for (uint32_t j = lane; j < nv; j += kLanes) A.acceleration[(size_t)env * A.max_nv + j] = e.accel[j];
    } else if (A.acceleration != nullptr) {
        for (uint32_t j = lane; j < nv; j += kLanes) A.acceleration[(size_t)env * A.max_nv + j] = 0.0f;
    }
    if (lane == 0u) {
        if (!failed && successful > 0u) A.mcurrent[env] = src_buf;
        MRWorldStatusC ws;
        ws.code = code;
        ws.environment = env;
        ws.control_step = A.control_step + step;
        ws.successful_substeps = successful;
        ws.aba_code = 0u;
        ws.failing_substep = failed ? failing_substep : MR_INVALID_INDEX;
        ws.failing_index = findex;
        ws.flags = 0u;
        if (!failed) {
            float qerr = 0.0f;
            if (floating) {
                const float n2 = e.q[3] * e.q[3] + e.q[4] * e.q[4] + e.q[5] * e.q[5] + e.q[6] * e.q[6];
                qerr = fabs_(sqrt_rn(n2) - 1.0f);
            }
            ws.diagnostics = mr_float4{isfin(min_piv) ? min_piv : 0.0f, max_piv, max_acc, qerr};
        } else {
            ws.diagnostics = mr_float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        A.status[step_rec] = ws;
        if constexpr (kCcd) cs.diagnostics.w = (float)impact_segments;
        cs.code = code;
        if (failed) {
            if (code == MR_STEP_PAIR_CAPACITY_OVERFLOW) cs.first_failing_pair = findex;
            else cs.first_failing_constraint = findex;
        }
        A.cstatus[step_rec] = cs;
        // wall-clock duration of this control step of this world (the GPU's constant-rate clock)
        if (A.step_us != nullptr)
            A.step_us[step_rec] = A.us_per_tick * (float)(__builtin_amdgcn_s_memrealtime() - s_t0);
    }
}

// Two wavefronts per SIMD: the register budget is capped at 256 so that two
// worlds share each SIMD and hide each other's memory and LDS latency (the
// per-world stages are latency-bound; one wave per SIMD left it idle).
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
mr_control_step_kernel(KernelArgs args) {
    control_step<false>(args, blockIdx.x);
}

// Persistent work-queue instance: a fixed grid of workgroups, each taking the
// next environment of args.queue (in the queue's order) until the queue is
// drained, so the order (heaviest first, say) and the number of resident
// workgroups are the caller's choice. The head is zeroed by
// mr_queue_reset_kernel before every launch.
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
mr_control_step_queue_kernel(KernelArgs args) {
    __shared__ uint32_t s_next;
    for (;;) {
        if (threadIdx.x == 0u) s_next = atomicAdd(args.queue_head, 1u);
        __syncthreads();
        const uint32_t idx = s_next;
        __syncthreads();
        if (idx >= args.queue_count) break;
        control_step<false>(args, args.queue[idx]);
        __syncthreads();
    }
}

// Persistent horizon instance: the work queue of mr_control_step_queue_kernel,
// where each entry is a world advanced through all args.horizon control steps
// back to back (step t's command, reset mask and status records at [t][E]).
// A world's next control step starts as soon as its previous one ends, so
// the launch is not held to the slowest world of every step; each world's
// steps run in order on one workgroup, so its results are those of one
// launch per control step.
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
mr_control_horizon_queue_kernel(KernelArgs args) {
    __shared__ uint32_t s_next;
    for (;;) {
        if (threadIdx.x == 0u) s_next = atomicAdd(args.queue_head, 1u);
        __syncthreads();
        const uint32_t idx = s_next;
        __syncthreads();
        if (idx >= args.queue_count) break;
        const uint32_t env = args.queue[idx];
        for (uint32_t t = 0; t < args.horizon; ++t) {
            control_step<false>(args, env, t);
            __syncthreads();
        }
    }
}

extern "C" __global__ void mr_queue_reset_kernel(uint32_t* head) {
    if (threadIdx.x == 0u && blockIdx.x == 0u) *head = 0u;
}

// Work-queue order for the next control step: the environments of `status`
// (one control step's contact statuses) sorted by the cone sweeps that step
// took (residuals.w), most first, by a counting sort over 1024 sweep bins in
// one workgroup. Only the schedule depends on it: which workgroup takes which
// world never changes a world's results. Environments with equal counts land
// in any order (atomic placement).
//
// With steps > 1 (after a persistent horizon launch, status holding [steps][E]
// records) the key is each world's mean sweeps per control step over the
// horizon, so the worlds that cost most over the whole horizon start first
// (longest-processing-time-first order for the next horizon).
extern "C" __global__ void __launch_bounds__(1024)
mr_queue_order_kernel(const MRContactStatusC* status, uint32_t environments, uint32_t steps, uint32_t* order) {
    __shared__ uint32_t bins[1024];
    __shared__ uint32_t wave_base[16];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    bins[t] = 0u;
    __syncthreads();
    auto key_of = [&](uint32_t e) {
        float sum = 0.0f;
        for (uint32_t s = 0; s < steps; ++s) sum += status[(size_t)s * environments + e].residuals.w;
        const float w = fminf(fmaxf(sum / (float)steps, 0.0f), 1023.0f);  // NaN -> 0
        return 1023u - (uint32_t)w;
    };
    for (uint32_t e = t; e < environments; e += 1024u) atomicAdd(&bins[key_of(e)], 1u);
    __syncthreads();
    // exclusive prefix over the bins: wave scans, then the wave totals
    const uint32_t v = bins[t];
    uint32_t x = v;
#pragma unroll
    for (uint32_t d = 1; d < 64u; d <<= 1) {
        const uint32_t y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63u) wave_base[wave] = x;
    __syncthreads();
    if (t == 0u) {
        uint32_t run = 0;
        for (uint32_t w = 0; w < 16u; ++w) {
            const uint32_t c = wave_base[w];
            wave_base[w] = run;
            run += c;
        }
    }
    __syncthreads();
    bins[t] = (x - v) + wave_base[wave];
    __syncthreads();
    for (uint32_t e = t; e < environments; e += 1024u) order[atomicAdd(&bins[key_of(e)], 1u)] = e;
}

// The learned-warm-start instance: the MLP tile keeps its accumulators and
// operands in registers next to the solver state, so it runs one wavefront
// per SIMD with the full register file.
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1)))
mr_control_step_mlp_kernel(KernelArgs args) {
    control_step<true>(args, blockIdx.x);
}

// The hybrid CCD mode: one workgroup per environment, microsteps split at
// times of impact. A separate instance, so the speculative kernels carry none
// of its registers. Two wavefronts per SIMD: at one, the compiler moves state
// into AGPRs instead of spilling, and the chain7+boxes hybrid workload ran
// 19 % slower (502k against 597k env-steps/s at 4096 worlds).
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
mr_control_step_ccd_kernel(KernelArgs args) {
    control_step<false, true>(args, blockIdx.x);
}

// Worlds with convex hulls or triangle meshes: one workgroup per
// environment, with the GJK / MPR / patch and BVH narrowphase (speculative
// and hybrid CCD modes). Separate instances, so the other kernels carry none
// of its private arrays.
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2)))
mr_control_step_geo_kernel(KernelArgs args) {
    control_step<false, false, true>(args, blockIdx.x);
}

extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2)))
mr_control_step_ccd_geo_kernel(KernelArgs args) {
    control_step<false, true, true>(args, blockIdx.x);
}

// Advance summary: one thread clears it, then a grid-stride pass over the
// [steps][environments] status records folds it with per-wave reductions and
// one atomic per wave (kernels rather than a memset, so the sequence is also
// valid inside a captured graph). With a subset work-queue schedule only the
// listed environments were stepped, so only their records are folded:
// `order` lists them (null for every environment).
extern "C" __global__ void mr_summary_clear_kernel(mr::AdvanceSummaryDev* s) {
    if (threadIdx.x == 0u && blockIdx.x == 0u) {
        s->first_failure = ~0ull;
        s->failed = 0u;
        s->max_active_pairs = 0u;
        s->max_constraints = 0u;
        s->pad = 0u;
    }
}

extern "C" __global__ void __launch_bounds__(256)
mr_summary_reduce_kernel(const MRWorldStatusC* status, const MRContactStatusC* cstatus, uint64_t steps,
                         uint32_t environments, const uint32_t* order, uint32_t order_count,
                         mr::AdvanceSummaryDev* s) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t failed = 0u, pairs = 0u, cons = 0u;
    unsigned long long first = ~0ull;
    const uint32_t stepped = order != nullptr ? order_count : environments;
    const uint64_t count = steps * stepped;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t step = i / stepped;
        const uint64_t env = order != nullptr ? order[i % stepped] : i % stepped;
        const uint64_t rec = step * environments + env;
        const uint32_t code = status[rec].code;
        if (code != MR_STEP_SUCCESS) {
            ++failed;
            const unsigned long long key = (step << 40) | (env << 8) | (unsigned long long)(code & 0xffu);
            first = key < first ? key : first;
        }
        const MRContactStatusC& c = cstatus[rec];
        pairs = c.max_active_pairs > pairs ? c.max_active_pairs : pairs;
        cons = c.max_constraints > cons ? c.max_constraints : cons;
    }
    failed = wave_sum_u32(failed);
    pairs = wave_max_u32(pairs);
    cons = wave_max_u32(cons);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const unsigned long long o = ((unsigned long long)__shfl_xor((int)(first >> 32), d, 64) << 32) |
                                     (unsigned long long)(uint32_t)__shfl_xor((int)(first & 0xffffffffull), d, 64);
        first = o < first ? o : first;
    }
    if (lane == 0u) {
        if (failed != 0u) atomicAdd(&s->failed, failed);
        atomicMax(&s->max_active_pairs, pairs);
        atomicMax(&s->max_constraints, cons);
        if (first != ~0ull) atomicMin(&s->first_failure, first);
    }
}

namespace mr {

hipError_t launch_advance_summary(const MRWorldStatusC* status, const MRContactStatusC* cstatus, uint64_t steps,
                                  uint32_t environments, const uint32_t* order, uint32_t order_count,
                                  AdvanceSummaryDev* summary, hipStream_t stream) {
    hipLaunchKernelGGL(mr_summary_clear_kernel, dim3(1), dim3(64), 0, stream, summary);
    const uint64_t count = steps * (order != nullptr ? order_count : environments);
    const uint64_t blocks = (count + 255u) / 256u;
    const uint32_t grid = (uint32_t)(blocks < 1024u ? (blocks > 0u ? blocks : 1u) : 1024u);
    hipLaunchKernelGGL(mr_summary_reduce_kernel, dim3(grid), dim3(256), 0, stream, status, cstatus, steps,
                       environments, order, order_count, summary);
    return hipGetLastError();
}

static_assert(sizeof(Collider) == 124, "Collider layout");
static_assert(sizeof(HotConstraint) == 128, "HotConstraint layout");
static_assert(sizeof(SolveBlock) == 64 && sizeof(HotConstraint) % sizeof(SolveBlock) == 0, "SolveBlock layout");

hipError_t launch_control_step(const KernelArgs& args, uint32_t lds_bytes, hipStream_t stream, bool mlp,
                               uint32_t queue_grid) {
    if (queue_grid > 0u && args.horizon > 0u) {
        hipLaunchKernelGGL(mr_queue_reset_kernel, dim3(1), dim3(64), 0, stream, args.queue_head);
        hipLaunchKernelGGL(mr_control_horizon_queue_kernel, dim3(queue_grid), dim3(64), lds_bytes, stream, args);
        return hipGetLastError();
    }
    if (queue_grid > 0u) {
        hipLaunchKernelGGL(mr_queue_reset_kernel, dim3(1), dim3(64), 0, stream, args.queue_head);
        hipLaunchKernelGGL(mr_control_step_queue_kernel, dim3(queue_grid), dim3(64), lds_bytes, stream, args);
        return hipGetLastError();
    }
    if (mlp)
        hipLaunchKernelGGL(mr_control_step_mlp_kernel, dim3(args.environment_count), dim3(64), lds_bytes, stream, args);
    else if (args.geometry != 0u && args.cfg.ccd_mode == MR_CCD_HYBRID)
        hipLaunchKernelGGL(mr_control_step_ccd_geo_kernel, dim3(args.environment_count), dim3(64), lds_bytes, stream,
                           args);
    else if (args.geometry != 0u)
        hipLaunchKernelGGL(mr_control_step_geo_kernel, dim3(args.environment_count), dim3(64), lds_bytes, stream, args);
    else if (args.cfg.ccd_mode == MR_CCD_HYBRID)
        hipLaunchKernelGGL(mr_control_step_ccd_kernel, dim3(args.environment_count), dim3(64), lds_bytes, stream, args);
    else
        hipLaunchKernelGGL(mr_control_step_kernel, dim3(args.environment_count), dim3(64), lds_bytes, stream, args);
    return hipGetLastError();
}

// Scratch of the allocation-free entry point (mr_world_enqueue_device_static):
// one file-scope device array, which every GPU the library runs on holds at
// its own address until the process ends. Host code never passes the array's
// name to a kernel (on the host it is a stand-in, not a device address); it
// passes the address static_scratch() looked up for the current device.
static __device__ __align__(256) unsigned char scratch[MR_WORLD_STATIC_SCRATCH_BYTES];

// Device address of `scratch` on the current device: looked up once per
// device with hipGetSymbolAddress, then served from the cache.
hipError_t static_scratch(void** out, size_t* bytes) {
    constexpr int kMaxDevices = 64;
    static std::mutex guard;
    static void* address[kMaxDevices] = {};
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(guard);
    if (address[device] == nullptr) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (ptr == nullptr) return hipErrorInvalidSymbol;
        address[device] = ptr;
    }
    *out = address[device];
    *bytes = MR_WORLD_STATIC_SCRATCH_BYTES;
    return hipSuccess;
}

// Spins one thread until the constant-rate clock (s_memrealtime) has advanced
// `ticks`, or `max_iterations` reads have passed, and reports the ticks it saw;
// timed with events on the host, it gives the clock's rate.
extern "C" __global__ void mr_clock_spin_kernel(unsigned long long ticks, unsigned long long max_iterations,
                                                unsigned long long* seen) {
    if (threadIdx.x != 0u || blockIdx.x != 0u) return;
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    unsigned long long t = t0;
    for (unsigned long long i = 0; i < max_iterations && t - t0 < ticks; ++i) t = __builtin_amdgcn_s_memrealtime();
    *seen = t - t0;
}

// Microseconds per tick of s_memrealtime on the current device, measured once
// per device: a spin of 2^20 ticks (a few milliseconds at the rates GPUs use)
// timed with events.
hipError_t clock_us_per_tick(float* out) {
    constexpr int kMaxDevices = 64;
    static std::mutex guard;
    static float cached[kMaxDevices] = {};
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(guard);
    if (cached[device] == 0.0f) {
        unsigned long long* seen = nullptr;
        hipEvent_t a = nullptr, b = nullptr;
        e = hipMalloc(&seen, sizeof(unsigned long long));
        if (e == hipSuccess) e = hipEventCreate(&a);
        if (e == hipSuccess) e = hipEventCreate(&b);
        float ms = 0.0f;
        unsigned long long ticks = 0ull;
        if (e == hipSuccess) {
            (void)hipEventRecord(a, nullptr);
            hipLaunchKernelGGL(mr_clock_spin_kernel, dim3(1), dim3(64), 0, nullptr, 1ull << 20, 1ull << 26, seen);
            (void)hipEventRecord(b, nullptr);
            e = hipEventSynchronize(b);
        }
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
        if (e == hipSuccess) e = hipMemcpy(&ticks, seen, sizeof(ticks), hipMemcpyDeviceToHost);
        if (a != nullptr) (void)hipEventDestroy(a);
        if (b != nullptr) (void)hipEventDestroy(b);
        if (seen != nullptr) (void)hipFree(seen);
        if (e != hipSuccess) return e;
        if (ticks == 0ull || !(ms > 0.0f)) return hipErrorUnknown;
        cached[device] = 1000.0f * ms / (float)ticks;
    }
    *out = cached[device];
    return hipSuccess;
}

hipError_t launch_queue_order(const MRContactStatusC* status, uint32_t environments, uint32_t steps, uint32_t* order,
                              hipStream_t stream) {
    hipLaunchKernelGGL(mr_queue_order_kernel, dim3(1), dim3(1024), 0, stream, status, environments, steps, order);
    return hipGetLastError();
}

// Workgroups of the plain or work-queue control-step kernel one CU holds.
hipError_t control_step_occupancy(uint32_t lds_bytes, int* blocks_per_cu) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu,
                                                        reinterpret_cast<const void*>(&mr_control_step_queue_kernel),
                                                        64, lds_bytes);
}

// The dynamic-LDS limit is an attribute of the kernel function, shared by
// every world in the process: it only ever grows to the largest world's need.
hipError_t configure_control_step(uint32_t lds_bytes, uint32_t mlp_lds_bytes) {
    static std::mutex guard;
    static uint32_t plain_max = 0u, mlp_max = 0u;
    std::lock_guard<std::mutex> lock(guard);
    if (lds_bytes > plain_max) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&mr_control_step_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&mr_control_step_queue_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&mr_control_horizon_queue_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
        for (const void* k : {reinterpret_cast<const void*>(&mr_control_step_ccd_kernel),
                              reinterpret_cast<const void*>(&mr_control_step_geo_kernel),
                              reinterpret_cast<const void*>(&mr_control_step_ccd_geo_kernel)}) {
            e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
            if (e != hipSuccess) return e;
        }
        plain_max = lds_bytes;
    }
    if (mlp_lds_bytes > mlp_max) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&mr_control_step_mlp_kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)mlp_lds_bytes);
        if (e != hipSuccess) return e;
        mlp_max = mlp_lds_bytes;
    }
    return hipSuccess;
}

} // namespace mr
