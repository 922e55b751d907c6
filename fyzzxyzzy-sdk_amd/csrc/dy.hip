// Dy stage of the GPU step on gfx950: unconstrained pre-integration, solver
// rows, exact first-fit conflict partitions, contact preparation with
// correlated friction and anchor growth, partitioned projected Gauss-Seidel
// (normal rows, then the patch's friction rows under the Coulomb clamp),
// integration and the wake-counter sleep check.
//
// Reference (src/native/scene.cpp):
//   prepare_unconstrained_velocities            10383-10507   k_pre
//   prepare_solver_bodies                       6940-7112     k_rows
//   partition_constraints                       7113-7489     k_part_*
//   prepare_constraints (contact managers)      7490-7515, 7763-8511   k_prep
//   cached_friction_patch_valid                 3981-4010     history_valid
//   solve_constraint_task                       8853-9148     k_pgs
//   publish_solver_bodies, integrate_solver_task, integrate_quaternion
//                                               9509-9549, 10508-10707, 111-146   integrate_body, in k_outputs
//
// Admitted scene class: dynamic boxes and static planes/boxes, PCM
// manifolds (one normal per manager, 1-4 contacts), non-compliant
// materials, no joints, locks, slop or gyroscopic terms; one solver task.
//
// Exactness. Every FP32 expression keeps the reference's operation order
// (the library builds with -ffp-contract=off). Partitions reproduce the
// sequential first-fit over 32-bit masks exactly: a manager's partition
// depends only on the masks its two bodies carry after the earlier managers
// incident to them, so a manager is coloured as soon as its predecessor on
// each body is (one launch, no global rounds). Within a partition no two
// managers share a dynamic body and the static world's solver body keeps a zero state, so
// solving a partition's managers concurrently gives the sequential sweep's
// values bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <string>

#include "../../include/fyzz_hip.h"
#include "context.hpp"
#include "select.hpp"
#include "stages.hpp"
#include "vecmath.hpp"

namespace fyzz_hip::dy {
using namespace fyzz_hip::vm;

constexpr u32 kNone = 0xffffffffu;
constexpr u32 kPending = 0xfffffffeu;
constexpr u32 kMaxParts = 4096;       // partitions per step
constexpr u32 kMaxPending = 65536;    // managers left for overflow waves
constexpr int kBlock = 256;
constexpr int kColorBlocks = 256;     // workgroups of the colouring (64: +60 us on the pile, 1024: +27)
constexpr u32 kListRegs = 16;         // incidence lists up to this length are handled in registers
constexpr int kPgsBlocks = 512;       // workgroups of the sweep (see k_pgs)

constexpr u32 kColorTicket = 0, kColorDone = 1, kBarWords = 2;

// device counters
enum : u32 { kFront0 = 0, kFront1, kFront2, kPend, kNParts, kPosIters, kVelIters, kRounds, kContacts, kFrictionRows,
             kIncidence, kCtrWords = 16 };

// The solver rows of the manager at a partition-sorted position, laid out
// for the eight lanes that solve it (4 lanes per body: three components and
// one for scalars): 4 row pairs (contact rows 0/1, 2/3, the friction rows of
// anchor 0, of anchor 1) of 8 float4, 512 B. Lane q (side q >> 2, component
// c = q & 3) of pair p holds
//   c < 3: (direction_c, lever_c) of the pair's first row, then of its
//          second (direction: contact normal or tangent; lever: the side's
//          angular part of the row), negated for side 1, whose terms enter
//          a row's relative velocity and its own update with a minus
//   c = 3: the scalars of the first row (side 0) or the second (side 1):
//          contact (velocity multiplier, biased error, unbiased error,
//          maximum impulse), friction (velocity multiplier, bias, target, 0)
// so that a pair is one 128-B request of the eight lanes.
constexpr u32 kRowLanes = 8;       // float4 per row pair
constexpr u32 kRowQuads = 4 * kRowLanes;  // float4 per manager

struct Ws {
    // step inputs
    float dt;
    u32 nb, ns, nm, nh;
    fyzz_dy_body* bodies;
    const fyzz_dy_static* statics;
    const fyzz_dy_manager* mg;
    const fyzz_dy_patch* history;
    fyzz_dy_patch* patches;
    float* impulses;
    u32* parts_out;
    const u32* d_nm;  // device manager count (at most nm), or null
    u32 with_rows;    // contact prep ran: order, rows and patches are valid
    // per body
    float4 *pv, *pw;          // pre-integrated velocities
    float4 *lin, *ang;        // solver deltas: lin_delta|inv_mass, ang_state
    float4 *mlin, *mang;      // motion snapshot after the last position iteration
    float4 *rpos, *rq;        // mass pose of the solver row
    float4* sii;              // 3 columns of the world sqrt inverse inertia
    u32* has_row;
    u32 *deg, *off, *fill, *body_mask;  // incidence list of body b: inc[off[b]], deg[b] entries
    // per manager
    u32 *inc, *pred, *part, *pend, *sorted, *order;
    uint8_t* dd;  // [nm] the manager touches two dynamic bodies (a compact copy for the per-body passes)
    u64* entry;  // [2 nm] partition colouring: ready | level << 32 | mask after the manager, per side
    int4* sinfo; // [nm] per partition-sorted position: body0, body1, manager, contact rows | anchors << 8
    u32* pos_of;    // [nm] partition-sorted position of each manager in a partition
    uint4* srank;   // [nm] per position: rank of the manager among body0's / body1's (by partition), their degrees
    u32* erank;     // [2 nm] per incidence entry: rank among the body's managers by partition
    u64* vst;       // [8 nb] sweep state, a 64-byte line per body: 4 chunks of (linear bits, updates applied,
                    // angular bits, updates applied): x, y, z, then the inverse mass
    float4* rows;   // [32 nm] solver rows by partition-sorted position (kRowQuads each)
    float* app;     // [8 nm] applied impulses by position: 4 contact rows, 4 friction rows
    float4* fric;   // [nm] by position: the patch's static and dynamic friction, its flags
    u32 *part_count, *part_off, *part_fill;
    u32* ctr;
    u32* flags;
    u32* bar;  // the colouring's ticket and count of workgroups done
    // adjoint support (tape mode)
    u32 tape;             // record branches and raw row vectors
    u32 tape_iters;       // iterations the tape holds
    uint8_t* tape_c;      // [iter][4 nm] normal rows: 1 free update, 0 clamped to zero, 2 at the maximum
    uint8_t* tape_f;      // [iter][4 nm] friction rows: 0 free, 1 clamped inside, 2 at +max, 3 at -max
    float* tape_ni;       // [iter][nm] the manager's normal impulse sum of the iteration
    float4* craw;         // [4 nm][2] contact rows: (ra x n, kv), (rb x n, 0); d err / d vrel = kv vm
    float4* fraw;         // [4 nm][2] friction rows: (ra x t, 0), (rb x t, 0) unscaled
    // adjoint inputs / outputs and state
    const float* adj_v_out;
    const float* adj_w_out;
    const float* adj_p_out;
    float* adj_v_in;
    float* adj_w_in;
    float* adj_friction;  // per body: d loss / d dynamic friction
    float4* a_side;  // [4 nm] per manager and side: (velocity adjoint, friction adjoint), (angular adjoint, 0)
    // by position: the applied impulses' adjoint, the errors' (contact) and targets' (friction), as app
    float *a_app, *a_acc;
    float* a_df;  // per manager: the dynamic friction's
};

__device__ inline u32 ld(const u32* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void raise_flag(const Ws& W, u32 f) { atomicOr(W.flags, f); }
__device__ inline u32 mcount(const Ws& W) { return W.d_nm ? min(ld(W.d_nm), W.nm) : W.nm; }
constexpr u32 kSpinLimit = 1u << 20;  // polls of one bounded wait; beyond it a status flag is raised
// A wave whose lanes all wait backs off (64, 256, then 1024 cycles per
// poll), so polling leaves the memory system to the waves doing work.
__device__ inline void wait_backoff(u32 idle) {
    if (idle == 0) return;
    if (idle < 8)
        __builtin_amdgcn_s_sleep(1);
    else if (idle < 64)
        __builtin_amdgcn_s_sleep(4);
    else
        __builtin_amdgcn_s_sleep(16);
}
__device__ inline bool finite3(V v) { return isfinite(v.x) && isfinite(v.y) && isfinite(v.z); }
__device__ inline bool finite4(Q q) { return isfinite(q.x) && isfinite(q.y) && isfinite(q.z) && isfinite(q.w); }
__device__ inline V v3(const float* p) { return {p[0], p[1], p[2]}; }
__device__ inline Q q4(const float* p) { return {p[0], p[1], p[2], p[3]}; }
__device__ inline V f3(float4 f) { return {f.x, f.y, f.z}; }
__device__ inline float len2(V v) { return v.x * v.x + v.y * v.y + v.z * v.z; }
__device__ inline void put3(float* d, V s) {
    d[0] = s.x;
    d[1] = s.y;
    d[2] = s.z;
}
// mass pose of a box: identity mass-local frame (scene.cpp:359-365)
__device__ inline V mass_position(V p, Q q) { return vadd(p, srot(q, V{0.0f, 0.0f, 0.0f})); }
__device__ inline Q mass_orientation(Q q) { return qmul(q, Q{0.0f, 0.0f, 0.0f, 1.0f}); }

// ---------------------------------------------------------------- bodies

__device__ inline bool manager_ok(const Ws& W, const fyzz_dy_manager& M) {
    return !((M.body0 < 0 && M.body1 < 0) || M.body0 == M.body1 || M.body0 >= int(W.nb) || M.body1 >= int(W.nb) ||
             (M.body0 < 0 && u32(-1 - M.body0) >= W.ns) || (M.body1 < 0 && u32(-1 - M.body1) >= W.ns) ||
             M.count == 0 || M.count > 4);
}

// Start of a step: status flags, counters, per-body and per-partition
// counts cleared (plain stores, so a captured step records no memset
// node), then the unconstrained velocities, scene.cpp:10383-10507 for
// default dynamics (no pending velocity mods). The flags are raised from
// the next kernel on (k_rows checks these velocities).
__global__ __launch_bounds__(kBlock) void k_pre(Ws W) {
    const u32 i = blockIdx.x * kBlock + threadIdx.x;
    if (i < kCtrWords) W.ctr[i] = 0;
    if (i == 0) *W.flags = 0;
    if (i < kBarWords) W.bar[i] = 0;
    if (i < kMaxParts) {
        W.part_count[i] = 0;
        W.part_fill[i] = 0;
    }
    if (i >= W.nb) return;
    W.has_row[i] = 0;
    W.deg[i] = 0;
    W.fill[i] = 0;
    const fyzz_dy_body& b = W.bodies[i];
    if (b.flags & 1u) return;
    const float dt = W.dt;
    const float gravity = -9.81f;
    float vx = b.linear_velocity[0] + 0.0f + 0.0f * dt;
    float vy = b.linear_velocity[1] + 0.0f + 0.0f * dt;
    float vz = b.linear_velocity[2] + 0.0f + 0.0f * dt;
    vy = vy + ((b.flags & 4u) ? gravity * dt : 0.0f);
    const float lm = smax(1.0f - b.linear_damping * dt, 0.0f);
    vx *= lm;
    vy *= lm;
    vz *= lm;
    V a{b.angular_velocity[0] + 0.0f + 0.0f * dt, b.angular_velocity[1] + 0.0f + 0.0f * dt,
        b.angular_velocity[2] + 0.0f + 0.0f * dt};
    const float am = smax(1.0f - b.angular_damping * dt, 0.0f);
    a.x *= am;
    a.y *= am;
    a.z *= am;
    const float s2 = vx * vx + vy * vy + vz * vz;
    const float ml2 = b.max_linear_velocity * b.max_linear_velocity;
    const float ma2 = b.max_angular_velocity * b.max_angular_velocity;
    if (s2 > ml2) {
        const float f = sqrtf(ml2 / s2);
        vx *= f;
        vy *= f;
        vz *= f;
    }
    const float a2 = a.x * a.x + a.y * a.y + a.z * a.z;
    if (a2 > ma2) {
        const float f = sqrtf(ma2 / a2);
        a.x *= f;
        a.y *= f;
        a.z *= f;
    }
    W.pv[i] = make_float4(vx, vy, vz, 0.0f);
    W.pw[i] = make_float4(a.x, a.y, a.z, 0.0f);
}

// Bodies of touching managers get a solver row (scene.cpp:6987-7013);
// incidence degrees (dynamic sides) and the manager's cleared entries for
// the partitions.
__global__ __launch_bounds__(kBlock) void k_mark(Ws W) {
    const u32 m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= mcount(W)) return;
    const fyzz_dy_manager& M = W.mg[m];
    W.part[m] = kNone;
    W.entry[2 * m] = 0ull;
    W.entry[2 * m + 1] = 0ull;
    const bool ok = manager_ok(W, M);
    W.dd[m] = ok && M.body0 >= 0 && M.body1 >= 0 ? 1u : 0u;
    if (!ok) {
        raise_flag(W, FYZZ_DY_BAD_INPUT);
        return;
    }
    if (M.body0 >= 0) {
        atomicAdd(&W.deg[M.body0], 1u);
        if (!(W.bodies[M.body0].flags & 1u)) W.has_row[M.body0] = 1;
    }
    if (M.body1 >= 0) {
        atomicAdd(&W.deg[M.body1], 1u);
        if (!(W.bodies[M.body1].flags & 1u)) W.has_row[M.body1] = 1;
    }
}

// world sqrt inverse inertia R diag(sqrt I^-1) R^T (scene.cpp:7092-7110)
__global__ __launch_bounds__(kBlock) void k_rows(Ws W) {
    // iteration counts (maximum over bodies with rows): one atomic per
    // workgroup and counter
    __shared__ u32 pos_it, vel_it, base;
    __shared__ u32 scratch[kBlock / kWave + 1];
    if (threadIdx.x == 0) pos_it = vel_it = 0;
    __syncthreads();
    const u32 i = blockIdx.x * kBlock + threadIdx.x;
    // the body's range of the incidence lists: the workgroup's bodies in
    // order, the workgroups in any (a list is found by its offset and
    // degree alone), so one counter takes the place of a scan's launches
    u32 total;
    const u32 before = block_exclusive_scan<kBlock>(i < W.nb ? W.deg[i] : 0u, scratch, &total);
    if (threadIdx.x == 0) base = total ? atomicAdd(&W.ctr[kIncidence], total) : 0u;
    if (i < W.nb && W.has_row[i]) {
        const u32 it = W.bodies[i].iterations;
        atomicMax(&pos_it, it & 0xffu);
        atomicMax(&vel_it, (it >> 8) & 0xffu);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (pos_it) atomicMax(&W.ctr[kPosIters], pos_it);
        if (vel_it) atomicMax(&W.ctr[kVelIters], vel_it);
    }
    if (i >= W.nb) return;
    W.off[i] = base + before;
    const bool row = W.has_row[i];
    {
        // the sweep's state line: no change, no updates, the inverse mass
        const u32 im = row ? __float_as_uint(W.bodies[i].inverse_mass) : 0u;
        uint4* line = reinterpret_cast<uint4*>(W.vst + 8ull * i);
        line[0] = line[1] = line[2] = make_uint4(0u, 0u, 0u, 0u);
        line[3] = make_uint4(im, 0u, 0u, 0u);
    }
    if (!(W.bodies[i].flags & 1u) && (!finite3(f3(W.pv[i])) || !finite3(f3(W.pw[i]))))
        raise_flag(W, FYZZ_DY_NONFINITE);
    float4 c0 = make_float4(0.f, 0.f, 0.f, 0.f), c1 = c0, c2 = c0;
    W.ang[i] = c0;
    W.mlin[i] = c0;
    W.mang[i] = c0;
    if (!row) {
        W.lin[i] = c0;
        W.rpos[i] = c0;
        W.rq[i] = make_float4(0.f, 0.f, 0.f, 1.f);
        W.sii[3 * i] = c0;
        W.sii[3 * i + 1] = c0;
        W.sii[3 * i + 2] = c0;
        return;
    }
    const fyzz_dy_body& b = W.bodies[i];
    const Q q = mass_orientation(q4(b.orientation));
    const V p = mass_position(v3(b.position), q4(b.orientation));
    W.rpos[i] = make_float4(p.x, p.y, p.z, 0.f);
    W.rq[i] = make_float4(q.x, q.y, q.z, q.w);
    W.lin[i] = make_float4(0.f, 0.f, 0.f, b.inverse_mass);
    const V l{sqrtf(b.inverse_inertia[0]), sqrtf(b.inverse_inertia[1]), sqrtf(b.inverse_inertia[2])};
    if (q.x == 0.0f && q.y == 0.0f && q.z == 0.0f && q.w == 1.0f) {
        c0.x = l.x;
        c1.y = l.y;
        c2.z = l.z;
    } else {
        const V rx = srot(q, V{1.f, 0.f, 0.f});
        const V ry = srot(q, V{0.f, 1.f, 0.f});
        const V rz = srot(q, V{0.f, 0.f, 1.f});
        const float xx = l.x * rx.x * rx.x + l.y * ry.x * ry.x + l.z * rz.x * rz.x;
        const float yy = l.x * rx.y * rx.y + l.y * ry.y * ry.y + l.z * rz.y * rz.y;
        const float zz = l.x * rx.z * rx.z + l.y * ry.z * ry.z + l.z * rz.z * rz.z;
        const float xy = l.x * rx.x * rx.y + l.y * ry.x * ry.y + l.z * rz.x * rz.y;
        const float xz = l.x * rx.x * rx.z + l.y * ry.x * ry.z + l.z * rz.x * rz.z;
        const float yz = l.x * rx.y * rx.z + l.y * ry.y * ry.z + l.z * rz.y * rz.z;
        c0 = make_float4(xx, xy, xz, 0.f);
        c1 = make_float4(xy, yy, yz, 0.f);
        c2 = make_float4(xz, yz, zz, 0.f);
    }
    W.sii[3 * i] = c0;
    W.sii[3 * i + 1] = c1;
    W.sii[3 * i + 2] = c2;
}

// ------------------------------------------------------------ partitions

// First-fit partitions over 32-bit masks (scene.cpp:7352-7445) for one task
// spanning the manager list; stable scatter by partition (7447-7489).
//
// The data-parallel phases are plain kernels over bodies or managers:
// degrees, incidence lists by body, each body's list in manager order with
// the predecessor of every dynamic/dynamic entry, static managers after the
// body's dynamic partitions, sizes, offsets and the scatter. The colouring
// is one kernel: a manager's partition depends only on the masks its two
// bodies carry after their earlier managers, so workgroups draw tiles of
// managers in increasing order and colour one as soon as the entries of
// its two predecessors are published. An entry is one 64-bit word (ready
// bit, chain level, mask after the manager) written and read as a single
// relaxed agent-scope atomic, cleared by the degree kernel every step. The
// smallest uncoloured manager is always ready and its thread is resident,
// so the colouring always advances; its waits are bounded regardless.

constexpr u64 kEntryReady = 1ull << 63;

// incidence lists, entry = manager << 1 | side
__global__ __launch_bounds__(kBlock) void k_part_fill(Ws W) {
    const u32 m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= mcount(W)) return;
    const fyzz_dy_manager& M = W.mg[m];
    if (!manager_ok(W, M)) return;
    if (M.body0 >= 0) W.inc[W.off[M.body0] + atomicAdd(&W.fill[M.body0], 1u)] = m << 1;
    if (M.body1 >= 0) W.inc[W.off[M.body1] + atomicAdd(&W.fill[M.body1], 1u)] = (m << 1) | 1u;
}

// One word of lane t (the same t in all lanes) in every lane.
__device__ inline u32 lane_word(u32 x, u32 t) {
    return static_cast<u32>(__builtin_amdgcn_readlane(static_cast<int>(x), static_cast<int>(t)));
}

// each body's list in manager order; predecessor links of the
// dynamic/dynamic entries
//
// An insertion sort in place is a chain of dependent loads and stores, so
// lists are ordered by counting, every load in flight at once: those of up
// to kListRegs entries (almost all of a pile's) in one thread's registers,
// those of up to a wave's width by the wave, a lane per entry. The longest
// list of a launch set its time: a 30,000-box heap 21 -> 15 us.
__global__ __launch_bounds__(kBlock) void k_part_chain(Ws W) {
    const u32 b = blockIdx.x * kBlock + threadIdx.x;
    const u32 lo = b < W.nb ? W.off[b] : 0u, d = b < W.nb ? W.deg[b] : 0u, hi = lo + d;
    for (u64 longs = __ballot(d > kListRegs && d <= kWave); longs; longs &= longs - 1) {
        const u32 src = static_cast<u32>(__builtin_ctzll(longs));
        const u32 at = lane_word(lo, src), len = lane_word(d, src), lane = lane_id();
        const u32 e = lane < len ? W.inc[at + lane] : kNone;
        const bool dyn = lane < len && W.dd[e >> 1];
        const u64 dyns = __ballot(dyn);
        u32 rank = 0, prev = 0;  // entry before + 1, 0: none
        for (u32 t = 0; t < len; ++t) {
            const u32 x = lane_word(e, t);
            const bool less = x < e;
            rank += less ? 1u : 0u;
            prev = less && ((dyns >> t) & 1ull) ? max(prev, x + 1u) : prev;
        }
        if (lane < len) W.inc[at + rank] = e;
        if (dyn) W.pred[e] = prev - 1u;
    }
    if (d <= kListRegs) {
        u32 e[kListRegs], dyn = 0;
#pragma unroll
        for (u32 k = 0; k < kListRegs; ++k) e[k] = k < d ? W.inc[lo + k] : kNone;
#pragma unroll
        for (u32 k = 0; k < kListRegs; ++k)
            if (k < d && W.dd[e[k] >> 1]) dyn |= 1u << k;
#pragma unroll
        for (u32 k = 0; k < kListRegs; ++k) {
            if (k >= d) continue;
            u32 rank = 0, prev = 0;  // as above
#pragma unroll
            for (u32 t = 0; t < kListRegs; ++t) {
                const bool less = e[t] < e[k];  // (absent entries are never less)
                rank += less ? 1u : 0u;
                prev = less && ((dyn >> t) & 1u) ? max(prev, e[t] + 1u) : prev;
            }
            W.inc[lo + rank] = e[k];
            if ((dyn >> k) & 1u) W.pred[e[k]] = prev - 1u;
        }
    } else if (d > kWave) {
        for (u32 i = lo + 1; i < hi; ++i) {
            const u32 e = W.inc[i];
            u32 j = i;
            while (j > lo && W.inc[j - 1] > e) {
                W.inc[j] = W.inc[j - 1];
                --j;
            }
            W.inc[j] = e;
        }
        u32 prev = kNone;
        for (u32 i = lo; i < hi; ++i) {
            const u32 e = W.inc[i];
            if (!W.dd[e >> 1]) continue;
            W.pred[e] = prev;
            prev = e;
        }
    }
}

// Ascending sort of a[0, p) by one workgroup (every thread calls it): a
// bitonic network over the next power of two, in the form whose every
// compare-exchange puts the smaller key at the lower index (each merge
// starts with a flipped half-cleaner), so the virtual padding (+inf keys
// beyond p) never moves and its exchanges are skipped. The pending list
// holds distinct manager indices.
__device__ void sort_pending(u32* a, u32 p) {
    u32 p2 = 1;
    while (p2 < p) p2 <<= 1;
    for (u32 k = 2; k <= p2; k <<= 1) {
        for (u32 j = k >> 1; j > 0; j >>= 1) {
            for (u32 t = threadIdx.x; t < (p2 >> 1); t += blockDim.x) {
                u32 l, r;
                if (j == (k >> 1)) {  // flipped half-cleaner: l pairs with its mirror in the block of k
                    const u32 blk = t / j, o = t % j;
                    l = blk * k + o;
                    r = blk * k + k - 1 - o;
                } else {
                    l = (t / j) * 2 * j + t % j;
                    r = l + j;
                }
                if (r < p) {
                    const u32 x = a[l], y = a[r];
                    if (x > y) {
                        a[l] = y;
                        a[r] = x;
                    }
                }
            }
            __threadfence_block();
            __syncthreads();
        }
    }
}

// The colouring and the overflow waves. A manager is coloured as soon as
// the entries of its two predecessors are published. Workgroups take tiles
// of kBlock managers by a ticket, so a tile's predecessors belong to it or
// to tiles already taken by running workgroups: the colouring advances
// however few of its workgroups are resident (a plain launch). The last
// workgroup to finish runs the overflow waves.
//
// What bounds it: the chain of dependent managers. The list is sorted by
// its lower slot, so most predecessors sit a few managers back: entries of
// the tile are also kept in LDS, where a hop is a fraction of the trip
// through memory, and a predecessor found ready is not polled again. With a
// persistent thread per several managers, every hop through memory and a
// grid barrier at the end (us): a 30,000-box heap 54, the formed pile of
// 100,000 95, 1,024 stacks of 64 boxes 140; so 45, 58 and 76.
__global__ __launch_bounds__(kBlock) void k_part_color(Ws W) {
    __shared__ u64 ent[2 * kBlock];
    __shared__ u32 s_tile, s_depth, s_last;
    const u32 nm = mcount(W);
    const u32 tiles = (nm + kBlock - 1) / kBlock;
    if (threadIdx.x == 0) s_depth = 0;
    bool pended = false;
    for (;;) {
        if (threadIdx.x == 0) s_tile = atomicAdd(&W.bar[kColorTicket], 1u);
        ent[threadIdx.x] = 0ull;
        ent[kBlock + threadIdx.x] = 0ull;
        __syncthreads();
        const u32 tile = s_tile;
        if (tile >= tiles) break;
        const u32 first = tile * kBlock, m = first + threadIdx.x;
        bool todo = m < nm && W.dd[m];  // a valid manager between two dynamic bodies
        u32 p0 = todo ? W.pred[2 * m] : kNone, p1 = todo ? W.pred[2 * m + 1] : kNone;
        u64 a0 = p0 == kNone ? kEntryReady : 0ull, a1 = p1 == kNone ? kEntryReady : 0ull;
        const u32 base = 2 * first;
        const bool local0 = p0 != kNone && p0 >= base, local1 = p1 != kNone && p1 >= base;
        volatile u64* const vent = ent;
        u32 spins = 0, idle = 0;
        while (__ballot(todo)) {
            bool progress = false;
            if (todo) {
                if (!a0)
                    a0 = local0 ? vent[p0 - base]
                                : __hip_atomic_load(&W.entry[p0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (!a1)
                    a1 = local1 ? vent[p1 - base]
                                : __hip_atomic_load(&W.entry[p1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (a0 && a1) {
                    const u32 before0 = static_cast<u32>(a0), before1 = static_cast<u32>(a1);
                    const u32 level = max(static_cast<u32>(a0 >> 32) & 0x7fffffffu,
                                          static_cast<u32>(a1 >> 32) & 0x7fffffffu) + 1u;
                    const u32 avail = ~(before0 | before1);
                    const u32 bit = avail ? 1u << __builtin_ctz(avail) : 0u;
                    const u64 hi = kEntryReady | (static_cast<u64>(level) << 32);
                    const u64 e0 = hi | (before0 | bit), e1 = hi | (before1 | bit);
                    vent[2 * threadIdx.x] = e0;
                    vent[2 * threadIdx.x + 1] = e1;
                    __hip_atomic_store(&W.entry[2 * m], e0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(&W.entry[2 * m + 1], e1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (avail) {
                        W.part[m] = __builtin_ctz(avail);
                    } else {
                        W.part[m] = kPending;
                        const u32 k = atomicAdd(&W.ctr[kPend], 1u);
                        if (k < kMaxPending) W.pend[k] = m;
                        pended = true;
                    }
                    atomicMax(&s_depth, level);
                    todo = false;
                    progress = true;
                } else if (++spins > kSpinLimit) {
                    // (the entries are published all the same, so that the
                    // managers after this one do not wait for it in turn)
                    raise_flag(W, FYZZ_DY_LOGIC);
                    vent[2 * threadIdx.x] = vent[2 * threadIdx.x + 1] = kEntryReady;
                    __hip_atomic_store(&W.entry[2 * m], kEntryReady, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(&W.entry[2 * m + 1], kEntryReady, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    todo = false;
                }
            }
            idle = __ballot(progress) ? 0u : idle + 1u;
            if (idle > 2u) wait_backoff(idle);
        }
        __syncthreads();
    }
    // the pending list is written back before this workgroup counts as done
    if (__syncthreads_or(pended)) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if (threadIdx.x == 0) {
        if (s_depth > ld(&W.ctr[kRounds])) atomicMax(&W.ctr[kRounds], s_depth);
        s_last = atomicAdd(&W.bar[kColorDone], 1u) == gridDim.x - 1 ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last || !ld(&W.ctr[kPend])) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    // overflow waves: the unassigned managers, in order, with fresh masks
    __shared__ u32 s_pending;
    if (threadIdx.x == 0) {
        u32 p = ld(&W.ctr[kPend]);
        if (p > kMaxPending) {
            raise_flag(W, FYZZ_DY_OVERFLOW);
            p = 0;
        }
        s_pending = p;
    }
    __syncthreads();
    sort_pending(W.pend, s_pending);
    if (threadIdx.x == 0) {
        u32 p = s_pending;
        for (u32 wave = 32; p; wave += 32) {
            for (u32 k = 0; k < p; ++k) {
                const fyzz_dy_manager& M = W.mg[W.pend[k]];
                W.body_mask[M.body0] = 0;
                W.body_mask[M.body1] = 0;
            }
            u32 over = 0;
            for (u32 k = 0; k < p; ++k) {
                const u32 mm = W.pend[k];
                const fyzz_dy_manager& M = W.mg[mm];
                const u32 avail = ~(W.body_mask[M.body0] | W.body_mask[M.body1]);
                if (!avail) {
                    W.pend[over++] = mm;
                    continue;
                }
                const u32 bit = __builtin_ctz(avail);
                W.body_mask[M.body0] |= 1u << bit;
                W.body_mask[M.body1] |= 1u << bit;
                W.part[mm] = wave + bit;
            }
            if (over == p) {
                raise_flag(W, FYZZ_DY_LOGIC);
                break;
            }
            p = over;
        }
    }
}

// Dynamic/static managers follow the body's dynamic partitions; then each
// of the body's managers is ranked by partition (the order in which a
// sweep reaches them; a body's managers have distinct partitions). A
// static manager touches one dynamic body, so this thread owns its
// partition; the dynamic ones are final after the colouring.
// Partition sizes are counted here too, each manager by its first dynamic
// side: in LDS per workgroup first (a pile has a few tens of partitions, so
// one global counter per manager would serialize ~10^4 atomics per
// address), then one value per partition the workgroup holds.
__global__ __launch_bounds__(kBlock) void k_part_static(Ws W) {
    __shared__ u32 cnt[kMaxParts];
    __shared__ u32 top;
    for (u32 i = threadIdx.x; i < kMaxParts; i += kBlock) cnt[i] = 0;
    if (threadIdx.x == 0) top = 0;
    __syncthreads();
    auto tally = [&](u32 pm) {
        if (pm >= kMaxParts) {
            raise_flag(W, FYZZ_DY_OVERFLOW);
        } else {
            atomicAdd(&cnt[pm], 1u);
            atomicMax(&top, pm + 1);
        }
    };
    const u32 b = blockIdx.x * kBlock + threadIdx.x;
    const u32 lo = b < W.nb ? W.off[b] : 0u, d = b < W.nb ? W.deg[b] : 0u, hi = lo + d;
    // As in k_part_chain: a lane per manager for lists of up to a wave's
    // width (a thread alone loads every pair of them: a 30,000-box heap
    // 62 -> 17 us), registers for those of up to kListRegs.
    for (u64 longs = __ballot(d > kListRegs && d <= kWave); longs; longs &= longs - 1) {
        const u32 src = static_cast<u32>(__builtin_ctzll(longs));
        const u32 at = lane_word(lo, src), len = lane_word(d, src), lane = lane_id();
        const bool live = lane < len;
        const u32 e = live ? W.inc[at + lane] : 0u, m = e >> 1;
        const bool dyn = live && W.dd[m];
        u32 pc = dyn ? W.part[m] : kNone;
        u32 k = pc < kPending ? pc + 1u : 0u;
        for (int o = kWave / 2; o > 0; o >>= 1) k = max(k, static_cast<u32>(__shfl_xor(static_cast<int>(k), o, kWave)));
        const u64 stat = __ballot(live && !dyn);
        if (live && !dyn) {
            pc = k + lane_rank(stat);
            W.part[m] = pc;
        }
        if (live && (!dyn || !(e & 1u))) tally(pc);
        u32 r = 0;
        for (u32 t = 0; t < len; ++t) r += lane_word(pc, t) < pc ? 1u : 0u;
        if (live) W.erank[e] = r;
    }
    if (d <= kListRegs) {
        u32 pc[kListRegs], ec[kListRegs], dyn = 0, k = 0;
#pragma unroll
        for (u32 q = 0; q < kListRegs; ++q) ec[q] = q < d ? W.inc[lo + q] : 0u;
#pragma unroll
        for (u32 q = 0; q < kListRegs; ++q) {
            pc[q] = kNone;  // absent entries never count as lower
            if (q < d && W.dd[ec[q] >> 1]) {
                dyn |= 1u << q;
                pc[q] = W.part[ec[q] >> 1];
            }
        }
#pragma unroll
        for (u32 q = 0; q < kListRegs; ++q)
            if (pc[q] < kPending) k = max(k, pc[q] + 1u);
#pragma unroll
        for (u32 q = 0; q < kListRegs; ++q) {
            if (q >= d) continue;
            if (!((dyn >> q) & 1u)) {
                W.part[ec[q] >> 1] = k;
                pc[q] = k++;
            }
            if (!((dyn >> q) & 1u) || !(ec[q] & 1u)) tally(pc[q]);
        }
#pragma unroll
        for (u32 q = 0; q < kListRegs; ++q) {
            if (q >= d) continue;
            u32 r = 0;
#pragma unroll
            for (u32 t = 0; t < kListRegs; ++t) r += pc[t] < pc[q] ? 1u : 0u;
            W.erank[ec[q]] = r;
        }
    } else if (d > kWave) {
        u32 k = 0;
        for (u32 i = lo; i < hi; ++i) {
            const u32 m = W.inc[i] >> 1;
            if (W.dd[m] && W.part[m] < kPending) k = max(k, W.part[m] + 1u);
        }
        for (u32 i = lo; i < hi; ++i) {
            const u32 e = W.inc[i], m = e >> 1;
            const bool dyn = W.dd[m];
            if (!dyn) W.part[m] = k++;
            if (!dyn || !(e & 1u)) tally(W.part[m]);
        }
        for (u32 i = lo; i < hi; ++i) {
            const u32 e = W.inc[i];
            const u32 pe = W.part[e >> 1];
            u32 r = 0;
            for (u32 j = lo; j < hi; ++j) r += W.part[W.inc[j] >> 1] < pe ? 1u : 0u;
            W.erank[e] = r;
        }
    }
    __syncthreads();
    const u32 np = top;
    for (u32 i = threadIdx.x; i < np; i += kBlock)
        if (cnt[i]) atomicAdd(&W.part_count[i], cnt[i]);
    if (threadIdx.x == 0 && np) atomicMax(&W.ctr[kNParts], np);
}

// Managers grouped by partition (order inside a partition is free): each
// workgroup scans the partition sizes into offsets (the first one writes
// them out), ranks its managers per partition in LDS, reserves one range
// per partition it holds, then writes.
__global__ __launch_bounds__(kBlock) void k_part_scatter(Ws W) {
    __shared__ u32 cnt[kMaxParts];
    __shared__ u32 base[kMaxParts];
    __shared__ u32 top;
    __shared__ u32 scratch[kBlock / kWave + 1];
    {
        const u32 np = min(W.ctr[kNParts], kMaxParts);
        u32 carry = 0, total;
        for (u32 t0 = 0; t0 < np; t0 += kBlock) {
            const u32 t = t0 + threadIdx.x;
            const u32 ex = carry + block_exclusive_scan<kBlock>(t < np ? W.part_count[t] : 0u, scratch, &total);
            if (t < np) {
                base[t] = ex;
                if (blockIdx.x == 0) W.part_off[t] = ex;
            }
            carry += total;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) W.part_off[np] = carry;
    }
    const u32 m = blockIdx.x * kBlock + threadIdx.x;
    for (u32 i = threadIdx.x; i < kMaxParts; i += kBlock) cnt[i] = 0;
    if (threadIdx.x == 0) top = 0;
    __syncthreads();
    const u32 pm = m < mcount(W) ? W.part[m] : kNone;
    const bool live = pm < kMaxParts;
    u32 local = 0;
    if (live) {
        local = atomicAdd(&cnt[pm], 1u);
        atomicMax(&top, pm + 1);
    }
    __syncthreads();
    const u32 np = top;
    for (u32 i = threadIdx.x; i < np; i += kBlock)
        if (cnt[i]) base[i] += atomicAdd(&W.part_fill[i], cnt[i]);
    __syncthreads();
    if (live) {
        const fyzz_dy_manager& M = W.mg[m];
        const u32 pos = base[pm] + local;
        W.sorted[pos] = m;
        W.pos_of[m] = pos;
        W.sinfo[pos] = make_int4(M.body0, M.body1, static_cast<int>(m), 0);
        W.srank[pos] = make_uint4(M.body0 >= 0 ? W.erank[2 * m] : 0u, M.body1 >= 0 ? W.erank[2 * m + 1] : 0u,
                                  M.body0 >= 0 ? W.deg[M.body0] : 0u, M.body1 >= 0 ? W.deg[M.body1] : 0u);
    }
}

// ----------------------------------------------------- contact preparation

struct Row {
    V pos;
    Q q;
    V v, w;
    float inv_mass;
    V c0, c1, c2;
};
__device__ inline Row load_row(const Ws& W, int id) {
    Row r{};
    r.q = Q{0.f, 0.f, 0.f, 1.f};
    if (id < 0 || !W.has_row[id]) return r;
    r.pos = f3(W.rpos[id]);
    const float4 q = W.rq[id];
    r.q = Q{q.x, q.y, q.z, q.w};
    r.v = f3(W.pv[id]);
    r.w = f3(W.pw[id]);
    r.inv_mass = W.lin[id].w;
    r.c0 = f3(W.sii[3 * id]);
    r.c1 = f3(W.sii[3 * id + 1]);
    r.c2 = f3(W.sii[3 * id + 2]);
    return r;
}
__device__ inline V transform(const Row& d, V v) {
    return {d.c0.x * v.x + d.c1.x * v.y + d.c2.x * v.z, d.c0.y * v.x + d.c1.y * v.y + d.c2.y * v.z,
            d.c0.z * v.x + d.c1.z * v.y + d.c2.z * v.z};
}
struct BodyView {
    V pos;
    Q q;
};
__device__ inline BodyView view_of(const Ws& W, int id) {
    if (id >= 0) return {v3(W.bodies[id].position), q4(W.bodies[id].orientation)};
    const fyzz_dy_static& s = W.statics[-1 - id];
    return {v3(s.position), q4(s.orientation)};
}
__device__ inline V local_point(const BodyView& a, V world) {
    const Q q = mass_orientation(a.q);
    const V p = mass_position(a.pos, a.q);
    return srot(Q{-q.x, -q.y, -q.z, q.w}, vsub(world, p));
}
__device__ inline V local_normal(const BodyView& a, V n) {
    const Q q = mass_orientation(a.q);
    return srot(Q{-q.x, -q.y, -q.z, q.w}, n);
}
__device__ inline V world_point(const BodyView& a, V local) {
    const V r = srot(mass_orientation(a.q), local);
    const V p = mass_position(a.pos, a.q);
    return vadd(r, p);
}

struct Patch {
    V normal, n0, n1;
    float sf, df, rest, damping;
    V a0[2], a1[2];
    V bmin, bmax;
    u32 contacts, anchors;
    bool broken, disable_strong;
};

// Field-by-field copy (a whole-struct copy from a runtime-indexed slot
// would keep the destination in memory as well).
__device__ inline void copy_patch(Patch& d, const Patch& s) {
    d.normal = V{s.normal.x, s.normal.y, s.normal.z};
    d.n0 = V{s.n0.x, s.n0.y, s.n0.z};
    d.n1 = V{s.n1.x, s.n1.y, s.n1.z};
    d.sf = s.sf;
    d.df = s.df;
    d.rest = s.rest;
    d.damping = s.damping;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        d.a0[k] = V{s.a0[k].x, s.a0[k].y, s.a0[k].z};
        d.a1[k] = V{s.a1[k].x, s.a1[k].y, s.a1[k].z};
    }
    d.bmin = V{s.bmin.x, s.bmin.y, s.bmin.z};
    d.bmax = V{s.bmax.x, s.bmax.y, s.bmax.z};
    d.contacts = s.contacts;
    d.anchors = s.anchors;
    d.broken = s.broken;
    d.disable_strong = s.disable_strong;
}

// scene.cpp:3981-4010
__device__ inline bool history_valid(const Patch& old, const BodyView& a0, const BodyView& a1) {
    if (old.broken || old.disable_strong || old.anchors == 0u) return false;
    const float same_normal = 0.999f;
    const float corr = 0.025f;
    const Q q0 = mass_orientation(a0.q), q1 = mass_orientation(a1.q);
    const V n10 = srot_inv(q0, srot(q1, old.n1));
    if (vdot(old.n0, n10) <= same_normal) return false;
    const V p0 = mass_position(a0.pos, a0.q), p1 = mass_position(a1.pos, a1.q);
    // constant anchor indices (at most two), so the patch stays in registers
#pragma unroll
    for (u32 k = 0; k < 2; ++k) {
        if (k >= old.anchors) break;
        const V l = srot(q1, old.a1[k]);
        const V world = vadd(l, p1);
        const V in0 = srot_inv(q0, vsub(world, p0));
        const V d = vsub(old.a0[k], in0);
        if (fabsf(vdot(d, old.n0)) >= corr) return false;
    }
    return true;
}

struct Run {
    u32 start, count;
    V normal, bmin, bmax;
    int next;
};

// A solver row as prepared, and a pair of them in the sweep's lane layout.
struct RowOut {
    V d, ra, rb;
    float4 s;
};
__device__ inline void store_rows(float4* o, const RowOut& x, const RowOut& y) {
    o[0] = make_float4(x.d.x, x.ra.x, y.d.x, y.ra.x);
    o[1] = make_float4(x.d.y, x.ra.y, y.d.y, y.ra.y);
    o[2] = make_float4(x.d.z, x.ra.z, y.d.z, y.ra.z);
    o[3] = x.s;
    o[4] = make_float4(-x.d.x, -x.rb.x, -y.d.x, -y.rb.x);
    o[5] = make_float4(-x.d.y, -x.rb.y, -y.d.y, -y.rb.y);
    o[6] = make_float4(-x.d.z, -x.rb.z, -y.d.z, -y.rb.z);
    o[7] = y.s;
}
// Row r (0-3 contact, 4-7 friction) of a position, read back by one thread.
__device__ inline RowOut read_row(const Ws& W, u32 pos, u32 r) {
    const float4* o = W.rows + static_cast<std::size_t>(kRowQuads) * pos + kRowLanes * (r >> 1);
    const bool second = r & 1u;
    RowOut v;
    const float4 x = o[0], y = o[1], z = o[2], bx = o[4], by = o[5], bz = o[6];
    v.d = second ? V{x.z, y.z, z.z} : V{x.x, y.x, z.x};
    v.ra = second ? V{x.w, y.w, z.w} : V{x.y, y.y, z.y};
    v.rb = second ? V{-bx.w, -by.w, -bz.w} : V{-bx.y, -by.y, -bz.y};
    v.s = o[second ? 7 : 3];
    return v;
}

// One thread per manager: materials, same-normal runs, friction-patch
// correlation with the previous step, contact rows, anchor growth and
// friction rows (scene.cpp:7794-8505).
__global__ __launch_bounds__(128) void k_prep(Ws W) {
    const u32 m = blockIdx.x * 128 + threadIdx.x;
    if (m >= mcount(W)) return;
    const fyzz_dy_manager& M = W.mg[m];
    if (W.part[m] >= kMaxParts) return;
    const float inv_dt = 1.0f / W.dt;
    const BodyView a0 = view_of(W, M.body0), a1 = view_of(W, M.body1);
    const Row a = load_row(W, M.body0);
    const Row b = load_row(W, M.body1);
    float sf0, df0, r0, sf1, df1, r1;
    if (M.body0 >= 0) {
        sf0 = W.bodies[M.body0].static_friction;
        df0 = W.bodies[M.body0].dynamic_friction;
        r0 = W.bodies[M.body0].restitution;
    } else {
        sf0 = W.statics[-1 - M.body0].static_friction;
        df0 = W.statics[-1 - M.body0].dynamic_friction;
        r0 = W.statics[-1 - M.body0].restitution;
    }
    if (M.body1 >= 0) {
        sf1 = W.bodies[M.body1].static_friction;
        df1 = W.bodies[M.body1].dynamic_friction;
        r1 = W.bodies[M.body1].restitution;
    } else {
        sf1 = W.statics[-1 - M.body1].static_friction;
        df1 = W.statics[-1 - M.body1].dynamic_friction;
        r1 = W.statics[-1 - M.body1].restitution;
    }
    if (r0 < 0.0f || r1 < 0.0f) {  // compliant contacts are not admitted
        raise_flag(W, FYZZ_DY_LOGIC);
        return;
    }
    const float rigid_contact_bias = 0.8f;
    const float bounce_threshold = -2.0f;
    const float same_normal = 0.999f;
    const float friction_offset_threshold = 0.04f;
    const float restitution = 0.5f * (r0 + r1);
    const float damping = 0.5f * (0.0f + 0.0f);
    const float dynamic_friction = smax(0.0f, 0.5f * (df0 + df1));
    const float static_friction = smax(dynamic_friction, 0.5f * (sf0 + sf1));
    const float max_pen_bias = -1.0e32f;
    const float rest_distance = 0.0f;
    // the previous step's patch when it correlates (scene.cpp:8007-8030)
    bool have_old = false;
    Patch c{};
    if (M.history != kNone && M.history < W.nh && W.history[M.history].anchor_count > 2u) {
        raise_flag(W, FYZZ_DY_BAD_INPUT);
    } else if (M.history != kNone && M.history < W.nh) {
        const fyzz_dy_patch& h = W.history[M.history];
        Patch old{};
        old.n0 = v3(h.body0_normal);
        old.n1 = v3(h.body1_normal);
        for (int k = 0; k < 2; ++k) {
            old.a0[k] = v3(h.body0_anchors[k]);
            old.a1[k] = v3(h.body1_anchors[k]);
        }
        old.sf = h.static_friction;
        old.df = h.dynamic_friction;
        old.rest = h.restitution;
        old.damping = h.damping;
        old.anchors = h.anchor_count;
        old.broken = h.flags & 1u;
        old.disable_strong = (h.flags >> 1) & 1u;
        if (history_valid(old, a0, a1)) {
            c = old;
            c.normal = srot(mass_orientation(a0.q), old.n0);
            c.contacts = 0;
            c.bmin = {kFltMax, kFltMax, kFltMax};
            c.bmax = {-kFltMax, -kFltMax, -kFltMax};
            have_old = true;
        }
    }
    // The kept patch, its header normal and the contact order (2-bit fields,
    // correlation-list order). A manager whose contacts all continue the
    // first contact's normal (every PCM manager: one published normal)
    // forms one run: the previous patch if it correlates, else one new
    // patch, keeps all contacts in their own order. Only other managers
    // take the general path over runs and candidate patches.
    Patch P;
    V header;
    u32 order_bits = 0, no = 0;
    bool one_run = M.count > 0 && M.count <= 4;
    {
        const V n0c = v3(M.contacts[0].normal);
#pragma unroll
        for (u32 jj = 1; jj < 4; ++jj)
            if (jj < M.count && vdot(n0c, v3(M.contacts[jj].normal)) < same_normal) one_run = false;
    }
    if (one_run) {
        // the run (scene.cpp:7964-7997) and its correlation (8007-8099)
        const V rn = v3(M.contacts[0].normal);
        V rbmin = v3(M.contacts[0].position), rbmax = rbmin;
#pragma unroll
        for (u32 jj = 1; jj < 4; ++jj)
            if (jj < M.count) {
                const V pp = v3(M.contacts[jj].position);
                rbmin = {smin(rbmin.x, pp.x), smin(rbmin.y, pp.y), smin(rbmin.z, pp.z)};
                rbmax = {smax(rbmax.x, pp.x), smax(rbmax.y, pp.y), smax(rbmax.z, pp.z)};
            }
        if (have_old && vdot(c.normal, rn) >= same_normal && c.rest == restitution && c.damping == damping &&
            c.sf == static_friction && c.df == dynamic_friction) {
            P = c;
        } else {
            P = Patch{};
            P.normal = rn;
            P.sf = static_friction;
            P.df = dynamic_friction;
            P.rest = restitution;
            P.damping = damping;
            P.n0 = local_normal(a0, rn);
            P.n1 = local_normal(a1, rn);
        }
        P.bmin = rbmin;
        P.bmax = rbmax;
        P.contacts = M.count;
        header = rn;
        no = M.count;
        order_bits = 0u | (1u << 2) | (2u << 4) | (3u << 6);
    } else {
        // contiguous same-normal runs (scene.cpp:7964-7997)
        Run runs[4];
        u32 nr = 0;
        for (u32 j = 0; j < M.count; ++j) {
            const V pn = v3(M.contacts[j].normal);
            const V pp = v3(M.contacts[j].position);
            if (nr == 0 || vdot(runs[nr - 1].normal, pn) < same_normal) {
                runs[nr++] = Run{j, 1, pn, pp, pp, -1};
            } else {
                Run& r = runs[nr - 1];
                ++r.count;
                r.bmin = {smin(r.bmin.x, pp.x), smin(r.bmin.y, pp.y), smin(r.bmin.z, pp.z)};
                r.bmax = {smax(r.bmax.x, pp.x), smax(r.bmax.y, pp.y), smax(r.bmax.z, pp.z)};
            }
        }
        // correlation against the previous step's patch (scene.cpp:8007-8099)
        Patch local[5];
        u32 nl = 0;
        if (have_old) local[nl++] = c;
        int heads[5] = {-1, -1, -1, -1, -1};
        for (u32 ri = 0; ri < nr; ++ri) {
            Run& cp = runs[ri];
            u32 lp = 0;
            for (; lp < nl; ++lp) {
                const Patch& p = local[lp];
                if (vdot(p.normal, cp.normal) >= same_normal && p.rest == restitution && p.damping == damping &&
                    p.sf == static_friction && p.df == dynamic_friction)
                    break;
            }
            if (lp == nl) {
                Patch p{};
                p.normal = cp.normal;
                p.sf = static_friction;
                p.df = dynamic_friction;
                p.rest = restitution;
                p.damping = damping;
                p.n0 = local_normal(a0, cp.normal);
                p.n1 = local_normal(a1, cp.normal);
                local[nl++] = p;
            }
            Patch& p = local[lp];
            if (p.contacts == 0) {
                p.bmin = cp.bmin;
                p.bmax = cp.bmax;
            } else {
                p.bmin = {smin(p.bmin.x, cp.bmin.x), smin(p.bmin.y, cp.bmin.y), smin(p.bmin.z, cp.bmin.z)};
                p.bmax = {smax(p.bmax.x, cp.bmax.x), smax(p.bmax.y, cp.bmax.y), smax(p.bmax.z, cp.bmax.z)};
            }
            p.contacts += cp.count;
            cp.next = heads[lp];
            heads[lp] = int(ri);
        }
        // exactly one patch keeps contacts: PCM managers publish one normal
        int kept = -1, nkept = 0;
        for (u32 j = 0; j < nl; ++j)
            if (local[j].contacts) {
                if (kept < 0) kept = int(j);
                ++nkept;
            }
        if (nkept != 1) {
            raise_flag(W, FYZZ_DY_LOGIC);
            return;
        }
        copy_patch(P, local[kept]);
        header = v3(M.contacts[runs[heads[kept]].start].normal);
        for (int cp = heads[kept]; cp >= 0; cp = runs[cp].next)
            for (u32 c = runs[cp].start; c < runs[cp].start + runs[cp].count; ++c) {
                order_bits |= c << (2 * no);
                ++no;
            }
    }
    // contact rows in the correlation-list order (scene.cpp:8204-8225, 8237-8330)
    bool bad = false;
    const u32 pos = W.pos_of[m];
    float4* const out = W.rows + static_cast<std::size_t>(kRowQuads) * pos;
    RowOut r[2];
    for (u32 q = 0; q < no; ++q) {
        const fyzz_dy_contact& C = M.contacts[(order_bits >> (2 * q)) & 3u];
        const V n = header;
        const V cpos = v3(C.position);
        const V ra_x_n = vcross(vsub(cpos, a.pos), n);
        const V rb_x_n = vcross(vsub(cpos, b.pos), n);
        const float lin_vrel = vdot(n, vsub(a.v, b.v));
        const V ra = transform(a, ra_x_n);
        const V rb = transform(b, rb_x_n);
        const float ang_vrel = vdot(ra_x_n, a.w) - vdot(rb_x_n, b.w);
        const float vrel = lin_vrel + ang_vrel;
        const float response = (a.inv_mass + vdot(ra, ra)) + (b.inv_mass + vdot(rb, rb));
        const float vm = response > 0.0f ? 1.0f / response : 0.0f;
        const float pen = C.separation - rest_distance;
        const float pen_inv_dt = pen * inv_dt;
        const bool separated = pen >= 0.0f;
        const bool closing = -vrel > pen_inv_dt;
        const bool bouncing = restitution > 0.0f && bounce_threshold > vrel && closing;
        const float target_velocity = bouncing ? -vrel * restitution : 0.0f;
        const float target = target_velocity - vrel;
        const float pen_scaled = separated ? pen_inv_dt : pen * (inv_dt * rigid_contact_bias);
        const float scaled_bias = bouncing ? 0.0f : vm * smax(max_pen_bias, pen_scaled);
        RowOut& o = r[q & 1u];
        const float biased = target * vm - scaled_bias;
        const float unbiased = target * vm - (bouncing ? 0.0f : smax(scaled_bias, 0.0f));
        o.d = n;
        o.ra = ra;
        o.rb = rb;
        o.s = make_float4(vm, biased, unbiased, kFltMax);
        bad |= !isfinite(response) || !isfinite(biased) || !isfinite(unbiased);
        if ((q & 1u) || q + 1 == no) store_rows(out + kRowLanes * (q >> 1), r[0], (q & 1u) ? r[1] : r[0]);
        if (W.tape) {
            // err = target vm - bias with target = -(1 + e) vrel when bouncing, -vrel otherwise
            W.craw[2 * (4 * m + q)] = make_float4(ra_x_n.x, ra_x_n.y, ra_x_n.z, bouncing ? -(1.0f + restitution) : -1.0f);
            W.craw[2 * (4 * m + q) + 1] = make_float4(rb_x_n.x, rb_x_n.y, rb_x_n.z, 0.0f);
        }
    }
    if (bad) raise_flag(W, FYZZ_DY_NONFINITE);
    // anchor growth (scene.cpp:8359-8433)
    {
        const V extent = vsub(P.bmax, P.bmin);
        const float diag2 = len2(extent);
        bool keep_pair = false;
        if (P.anchors == 2) {
            const V d = vsub(P.a0[0], P.a0[1]);
            keep_pair = len2(d) * 4.0f >= diag2;
            if (!keep_pair) P.anchors = 0;
        }
        V anchors[2] = {V{0.f, 0.f, 0.f}, V{0.f, 0.f, 0.f}};
        bool changed[2] = {false, false};
        u32 count = P.anchors;
        if (!keep_pair) {
            if (count == 1) anchors[0] = world_point(a0, P.a0[0]);
            float pd2 = 0.0f;
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                if (q >= no) continue;
                const u32 j = (order_bits >> (2 * q)) & 3u;
                if (M.contacts[j].separation >= friction_offset_threshold + rest_distance) continue;
                const V wp = v3(M.contacts[j].position);
                if (count == 0) {
                    anchors[0] = wp;
                    changed[0] = true;
                    ++count;
                } else if (count == 1) {
                    const float d = len2(vsub(wp, anchors[0]));
                    if (d > 1.0e-8f) {
                        anchors[1] = wp;
                        changed[1] = true;
                        pd2 = d;
                        ++count;
                    }
                } else {
                    const float d0 = len2(vsub(wp, anchors[0]));
                    const float d1 = len2(vsub(wp, anchors[1]));
                    if (d0 > d1 && d0 > pd2) {
                        anchors[1] = wp;
                        changed[1] = true;
                        pd2 = d0;
                    } else if (d1 >= d0 && d1 > pd2) {
                        anchors[0] = wp;
                        changed[0] = true;
                        pd2 = d1;
                    }
                }
            }
#pragma unroll
            for (u32 k = 0; k < 2; ++k) {
                if (k >= count || !changed[k]) continue;
                P.a0[k] = local_point(a0, anchors[k]);
                P.a1[k] = local_point(a1, anchors[k]);
            }
            if (count == 0) {
                P.a0[0] = V{0.f, 0.f, 0.f};
                P.a1[0] = V{0.f, 0.f, 0.f};
            }
        }
        P.anchors = count;
        if (count) {
            const V n = header;
            const V rel = vsub(a.v, b.v);
            V t0 = vsub(rel, V{n.x * vdot(rel, n), n.y * vdot(rel, n), n.z * vdot(rel, n)});
            if (len2(t0) <= 0.0001f) t0 = fabsf(n.x) < 0.70710678f ? V{0.0f, -n.z, n.y} : V{-n.y, n.x, 0.0f};
            const float il = 1.0f / sqrtf(len2(t0));
            t0 = {t0.x * il, t0.y * il, t0.z * il};
            const V t1 = vcross(n, t0);
#pragma unroll
            for (u32 k = 0; k < 2; ++k) {
                if (k >= count) continue;
                const V ra = srot(mass_orientation(a0.q), P.a0[k]);
                const V rb = srot(mass_orientation(a1.q), P.a1[k]);
                const V c0 = mass_position(a0.pos, a0.q), c1 = mass_position(a1.pos, a1.q);
                const V err = vsub(vadd(ra, c0), vadd(rb, c1));
                for (u32 ti = 0; ti < 2; ++ti) {
                    const V tangent = ti ? t1 : t0;
                    const V ax0 = vcross(ra, tangent);
                    const V ax1 = vcross(rb, tangent);
                    const V j0 = transform(a, ax0);
                    const V j1 = transform(b, ax1);
                    const float response = (a.inv_mass + vdot(j0, j0)) + (b.inv_mass + vdot(j1, j1));
                    RowOut& fr = r[ti];
                    fr.d = tangent;
                    fr.ra = j0;
                    fr.rb = j1;
                    fr.s = make_float4(response > 0.0f ? rigid_contact_bias / response : 0.0f,
                                       vdot(tangent, err) * inv_dt,
                                       -(vdot(tangent, rel) + vdot(ax0, a.w) - vdot(ax1, b.w)), 0.0f);
                    if (W.tape) {
                        W.fraw[2 * (4 * m + 2 * k + ti)] = make_float4(ax0.x, ax0.y, ax0.z, 0.0f);
                        W.fraw[2 * (4 * m + 2 * k + ti) + 1] = make_float4(ax1.x, ax1.y, ax1.z, 0.0f);
                    }
                }
                store_rows(out + kRowLanes * (2 + k), r[0], r[1]);
            }
        }
    }
    fyzz_dy_patch o;
    put3(o.body0_normal, P.n0);
    put3(o.body1_normal, P.n1);
    for (int k = 0; k < 2; ++k) {
        put3(o.body0_anchors[k], P.a0[k]);
        put3(o.body1_anchors[k], P.a1[k]);
    }
    o.static_friction = P.sf;
    o.dynamic_friction = P.df;
    o.restitution = P.rest;
    o.damping = P.damping;
    o.anchor_count = P.anchors;
    o.flags = (P.broken ? 1u : 0u) | (P.disable_strong ? 2u : 0u);
    W.patches[m] = o;
    W.order[m] = no | ((order_bits & 3u) << 8) | ((no > 1 ? (order_bits >> 2) & 3u : 0u) << 12) |
                 ((no > 2 ? (order_bits >> 4) & 3u : 0u) << 16) | ((no > 3 ? (order_bits >> 6) & 3u : 0u) << 20);
    // the sweep reads the row counts with the position record
    W.sinfo[pos].w = static_cast<int>(no | (P.anchors << 8));
    W.fric[pos] = make_float4(o.static_friction, o.dynamic_friction, __uint_as_float(o.flags), 0.f);
    float4* const ap = reinterpret_cast<float4*>(W.app + 8ull * pos);
    ap[0] = ap[1] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// ------------------------------------------------------------------ solve

// scene.cpp:8985-9010 (normal rows), 9050-9120 (friction rows)
// Coherent body state: during the sweep a body's velocity change lives in
// one 64-byte line of four 16-byte chunks (x, y, z, inverse mass), each
// value followed by the number of updates applied to the body, moved
// between workgroups on different XCDs by device-coherent (sc1) 16-byte
// loads and stores. The four lanes of a body's side move the whole line as
// one request. A reader takes the state when all counts carry the count it
// waits for: a count is written once per body, so matching counts give the
// values written with it, and a writer needs no wait between its state
// stores and a separate counter.
typedef u32 Chunk __attribute__((ext_vector_type(4)));
constexpr u32 kStateBytes = 64;
constexpr int kDeviceCoherent = 16;  // cache policy: sc1 (device scope)
__device__ inline __amdgpu_buffer_rsrc_t state_rsrc(const Ws& W) {
    // raw buffer over the state lines, range check off (offsets < 2^32)
    return __builtin_amdgcn_make_buffer_rsrc(W.vst, 0, 0xFFFFFFFF, 0x00020000);
}
__device__ inline Chunk load_chunk(__amdgpu_buffer_rsrc_t R, u32 off) {
    return __builtin_amdgcn_raw_buffer_load_b128(R, off, 0, kDeviceCoherent);
}
__device__ inline void store_chunk(__amdgpu_buffer_rsrc_t R, u32 off, float lin, float ang, u32 count) {
    const Chunk a = {__float_as_uint(lin), count, __float_as_uint(ang), count};
    __builtin_amdgcn_raw_buffer_store_b128(a, R, off, 0, kDeviceCoherent);
}
// Clock cycles before a body still (need - seen) updates short of a
// waiting manager is polled again: about one solve hop per missing update
// (kPollHopCycles), at most 32 hops; a body one update short (or a torn
// read, seen == need) is polled on the next pass.
constexpr u32 kPollHopCycles = 1024;
__device__ inline u64 poll_delay(u32 need, u32 seen) {
    const u32 d = need - seen;  // counts only grow up to need
    return d <= 1u ? 0ull : static_cast<u64>(min(d - 1u, 32u)) * kPollHopCycles;
}

// The eight lanes of one manager. Every exchange is a DPP move inside them:
// a quad broadcast (one lane's value to the four of its side) or the
// half-row mirror, which hands each lane a value of the other side (the
// values exchanged are the same in all four lanes of a side). The eight
// lanes always run together, so a DPP source is never an inactive lane.
constexpr int kDppMirror8 = 0x141;  // row_half_mirror
template <int CTRL>
__device__ inline float dpp(float x) {
    return __uint_as_float(
        static_cast<u32>(__builtin_amdgcn_update_dpp(0, static_cast<int>(__float_as_uint(x)), CTRL, 0xf, 0xf, true)));
}
template <int K>
__device__ inline float quad(float x) { return dpp<K * 0x55>(x); }
__device__ inline float other_side(float x) { return dpp<kDppMirror8>(x); }
// A value of side 0 (the same in its four lanes), or of side 1, in all
// eight lanes: the mirror into the other side's quads only (the bank mask
// names a row's quads), the side's own quads keep theirs.
template <int BANKS>
__device__ inline float mirror_into(float x) {
    const int v = static_cast<int>(__float_as_uint(x));
    return __uint_as_float(static_cast<u32>(__builtin_amdgcn_update_dpp(v, v, kDppMirror8, 0xf, BANKS, false)));
}
__device__ inline float of_side0(float x) { return mirror_into<0xa>(x); }
__device__ inline float of_side1(float x) { return mirror_into<0x5>(x); }

// The bits set in any of the four lanes of a side, and of either side
// (values equal in the four lanes).
template <int CTRL>
__device__ inline u32 dpp_or(u32 x) {
    return x | static_cast<u32>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), CTRL, 0xf, 0xf, true));
}
__device__ inline u32 quad_or(u32 x) { return dpp_or<0x4e>(dpp_or<0xb1>(x)); }  // lane ^ 1, then lane ^ 2
__device__ inline u32 sides_or(u32 x) { return dpp_or<kDppMirror8>(x); }

// A row's values in one lane: its component's direction and lever, and the
// row's scalars: velocity multiplier, error (contact) or target less bias
// (friction), maximum impulse.
struct LaneRow {
    float d, r, vm, e, top;
};
// Both rows of a pair from the lane's float4 of it (see Ws::rows); e:
// the scalar lanes' error of the iteration.
__device__ inline void unpack_rows(const float4& x, float e, LaneRow& first, LaneRow& second) {
    first.d = x.x;
    first.r = x.y;
    second.d = x.z;
    second.r = x.w;
    // the scalar lane (3) of each side: the first row's is side 0's
    const float vm = quad<3>(x.x), er = quad<3>(e), top = quad<3>(x.w);
    first.vm = of_side0(vm);
    first.e = of_side0(er);
    first.top = of_side0(top);
    second.vm = of_side1(vm);
    second.e = of_side1(er);
    second.top = of_side1(top);
}
// Applied impulses (lane q holds contact row q or friction row q - 4) of
// contact row K and friction row K in every lane.
template <int K>
__device__ inline void unpack_applied(float x, float& contact, float& friction) {
    const float own = quad<K>(x);
    contact = of_side0(own);
    friction = of_side1(own);
}

// One side's velocity state in its four lanes, and a row's relative
// velocity: direction . (side 0) - direction . (side 1) + lever . (side 0) -
// lever . (side 1), in that order. Side 1 holds its row negated, so its
// terms come with their minus: each product is the exact negative, and so
// is each sum but for the sign of a zero. That sign reaches nothing: the
// relative velocity is only subtracted from an error, scaled and added to
// an applied impulse, which is never -0 (it starts at +0, and a sum is -0
// only of two -0).
struct LaneState {
    float v, w;
};
__device__ inline float relative(const LaneState& s, float d, float r) {
    const float pv = d * s.v, pw = s.w * r;
    const float v0 = quad<0>(pv), w0 = quad<0>(pw);
    const float v1 = v0 + quad<1>(pv), w1 = w0 + quad<1>(pw);
    const float lin = v1 + quad<2>(pv), ang = w1 + quad<2>(pw);
    return ((lin + other_side(lin)) + of_side0(ang)) + of_side1(ang);
}

// The reverse of a row's velocity update: (direction . side 0) im0 -
// (direction . side 1) im1 + lever . (side 0) - lever . (side 1), in that
// order (signs as in relative).
__device__ inline float reverse_relative(const LaneState& s, float d, float r, float im) {
    const float pv = d * s.v, pw = r * s.w;
    const float v0 = quad<0>(pv), w0 = quad<0>(pw);
    const float v1 = v0 + quad<1>(pv), w1 = w0 + quad<1>(pw);
    const float lin = (v1 + quad<2>(pv)) * im, ang = w1 + quad<2>(pw);
    return ((lin + other_side(lin)) + of_side0(ang)) + of_side1(ang);
}

// Position then velocity iterations over the partitions in order, motion
// snapshotted after the last position iteration (scene.cpp:9136-9146),
// without grid barriers. The sweep is the sequence (iteration, sorted
// position); within a partition no two managers share a dynamic body, so
// the Gauss-Seidel result depends only on each body seeing its managers'
// updates in that order. A body's state words count the updates applied
// to it; the manager at rank r among the body's d managers (by partition)
// runs in iteration t once all words carry t*d + r, and publishes its
// result with t*d + r + 1. Eight lanes solve a manager (four per body);
// octet k solves positions k, k + T, ... in every iteration (T octets), in
// sequence order, each as soon as it is ready (an octet waits without
// holding back the rest of its wave). The earliest unsolved (iteration,
// position) always has its predecessors done and its octet resident
// (cooperative launch), so the sweep always advances; waits are bounded
// regardless (a status flag, not a hang).
//
// What bounds it: the chain of dependent managers (partitions x iterations
// hops), each hop a store made visible, a poll that finds it, and the
// solve. With one thread per manager a wave held up to 64 managers that
// became ready a few at a time, and each such group cost a full serial
// solve of both bodies' components (1.8 us); a poll read a body's line in
// two round trips. Eight lanes read the line in one request, solve the
// components side by side and poll for eight managers per wave instead of
// 64. Measured in steps (us per sweep, one thread per manager before): the
// formed pile of 100,000 boxes (230k managers, 19 partitions) 580 -> 317,
// a heap of 3,001 (800 managers, 10 partitions) 229 -> 120, 2,048 scenes
// 146 -> 99. By solve-time stamps on the heap a hop is 1.7 us: 0.7 us of
// solve (0.45 without friction rows), the rest visibility and polls.
// Variants that lost: the next position's rows loaded one position ahead
// (pile 407 -> 437), the solve issued between the polls and their answers
// (341 -> 505). 512 workgroups: pile 382 at 256, 317 at 512, 317 at 768;
// the scenes 91 at 256, 106 at 768.
// kTape: also records each row's branch for the adjoint (a variant of its
// own, so that a plain sweep carries none of it).
template <bool kTape>
__global__ __launch_bounds__(kBlock) void k_pgs(Ws W) {
    const u32 q = threadIdx.x & 7u, c = q & 3u;
    const bool side1 = q >= 4u;
    const u32 slot = (blockIdx.x * kBlock + threadIdx.x) >> 3;
    const u32 nslots = (gridDim.x * kBlock) >> 3;
    const u32 np = min(ld(&W.ctr[kNParts]), kMaxParts);
    const u32 pos_iters = ld(&W.ctr[kPosIters]);
    const u32 vel_iters = max(ld(&W.ctr[kVelIters]), 1u);
    const u32 total = pos_iters + vel_iters;
    const u32 n = np ? W.part_off[np] : 0u;
    u32 iter = 0, i = slot, spins = 0, idle = 0;
    const __amdgpu_buffer_rsrc_t R = state_rsrc(W);
    u64 wake = 0;  // earliest clock at which the side's body is polled again
    u64 now = 0;   // the clock as of the last pass (its read overlaps that pass's polls)
    bool have = false;
    u32 miss = 0;  // zero once the side's body state is taken (or the side is static)
    int4 info = make_int4(-1, -1, 0, 0);
    uint4 rk = make_uint4(0u, 0u, 0u, 0u);
    int body = -1;
    u32 need = 0;
    Chunk st = {0u, 0u, 0u, 0u};
    float4 x[4] = {};
    LaneRow row[8] = {};
    float ap[8] = {};
    float app = 0.f;
    float4 fric = make_float4(0.f, 0.f, 0.f, 0.f);  // static and dynamic friction, patch flags
    // the position record of the octet's next position, loaded while the
    // current manager waits (positions repeat in every iteration)
    u32 next_pos = kNone;
    int4 next_info = info;
    uint4 next_rk = rk;
    for (;;) {
        bool progress = false;
        while (iter < total && i >= n) {
            ++iter;
            i = slot;
        }
        if (iter < total) {
            const bool fresh = !have;
            if (fresh) {
                if (next_pos == i) {
                    info = next_info;
                    rk = next_rk;
                } else {
                    info = W.sinfo[i];
                    rk = W.srank[i];
                }
                have = true;
                body = side1 ? info.y : info.x;
                need = side1 ? iter * rk.w + rk.y : iter * rk.z + rk.x;
                miss = body < 0 ? 0u : 1u;
                wake = 0;
                st = Chunk{0u, 0u, 0u, 0u};
                // the rows are loaded while the bodies are awaited; only
                // this octet writes the applied impulses during the sweep,
                // each lane its own. An octet with a single position keeps
                // its rows and impulses in the lanes.
                if (iter == 0 || n > nslots) {
                    const float4* rows = W.rows + static_cast<std::size_t>(kRowQuads) * i + q;
                    const u32 no = static_cast<u32>(info.w) & 0xffu, anchors = (static_cast<u32>(info.w) >> 8) & 0xffu;
                    x[0] = rows[0];
                    if (no > 2u) x[1] = rows[kRowLanes];
                    if (anchors) x[2] = rows[2 * kRowLanes];
                    if (anchors > 1u) x[3] = rows[3 * kRowLanes];
                    app = W.app[8ull * i + q];
                    fric = W.fric[i];
                    const u32 nx = i + nslots < n ? i + nslots : slot;
                    next_pos = nx;
                    next_info = W.sinfo[nx];
                    next_rk = W.srank[nx];
                }
            }
            // A body whose count reached the awaited value stays there
            // until this manager runs: its state is kept, not polled again.
            // A body still `need - seen` updates short is polled again only
            // after about that many solve hops: waiting lanes would
            // otherwise keep the memory system busy with polls that cannot
            // succeed, slowing the hops they wait for.
            const bool poll = miss && now >= wake;
            if (poll) {
                st = load_chunk(R, static_cast<u32>(body) * kStateBytes + 16u * c);
                miss = quad_or((st.y ^ need) | (st.w ^ need));
                // (the first lane's count for all four)
                const u32 seen = __float_as_uint(quad<0>(__uint_as_float(st.y)));
                if (miss) wake = now + poll_delay(need, seen);
            }
            if (fresh) {
                // off the dependency chain: the wait for the poll covers the
                // row loads issued before it
                const bool pos = iter < pos_iters;
                unpack_rows(x[0], pos ? x[0].y : x[0].z, row[0], row[1]);
                unpack_rows(x[1], pos ? x[1].y : x[1].z, row[2], row[3]);
                unpack_rows(x[2], x[2].z - (pos ? x[2].y : 0.0f), row[4], row[5]);
                unpack_rows(x[3], x[3].z - (pos ? x[3].y : 0.0f), row[6], row[7]);
                unpack_applied<0>(app, ap[0], ap[4]);
                unpack_applied<1>(app, ap[1], ap[5]);
                unpack_applied<2>(app, ap[2], ap[6]);
                unpack_applied<3>(app, ap[3], ap[7]);
            }
            if (!sides_or(miss)) {
                const u32 no = static_cast<u32>(info.w) & 0xffu, anchors = (static_cast<u32>(info.w) >> 8) & 0xffu;
                LaneState s{__uint_as_float(st.x), __uint_as_float(st.z)};
                const float im = quad<3>(s.v);
                [[maybe_unused]] u32 branch = 0;  // tape: the branch of the lane's row
                float normal_impulse = 0.0f;
#pragma unroll
                for (u32 k = 0; k < 4; ++k) {
                    if (k >= no) break;
                    const LaneRow& r = row[k];
                    const float nv = relative(s, r.d, r.r);
                    const float xx = -nv * r.vm + r.e;
                    // max and min as the hardware has them: the operands
                    // differ or are the same bits (an applied impulse is
                    // never -0, so xx and -ap[k] are no mixed zeros), and a
                    // NaN stays in the velocities and is flagged below
                    const float dc = fmaxf(xx, -ap[k]);
                    const float sum = ap[k] + dc;
                    const float next = fminf(r.top, sum);
                    if constexpr (kTape) {
                        const u32 br = r.top < sum ? 2u : (xx < -ap[k] ? 0u : 1u);
                        branch = q == k ? br : branch;
                    }
                    const float delta = next - ap[k];
                    const float dm = delta * im;
                    s.v += r.d * dm;
                    s.w += r.r * delta;
                    app = q == k ? next : app;
                    normal_impulse += next;
                }
                const u32 m = static_cast<u32>(info.z);
                const bool rub = (iter >= pos_iters || pos_iters - iter <= 3u) && anchors;
                if (rub) {
                    const float coef = anchors == 2 ? 0.5f : 1.0f;
                    const float max_static = fric.x * coef * normal_impulse;
                    const float max_dynamic = fric.y * coef * normal_impulse;
                    const float min_dynamic = 0.0f - max_dynamic;
                    bool broken = false;
#pragma unroll
                    for (u32 k = 0; k < 4; ++k) {
                        if (k >= anchors * 2) break;
                        const LaneRow& r = row[4 + k];
                        const float td = relative(s, r.d, r.r);
                        const float cand = ap[4 + k] + (r.e - td) * r.vm;
                        const bool clamped = fabsf(cand) > max_static;
                        // a clamped candidate lies beyond +-max_static,
                        // which is at least max_dynamic: its clamp is the
                        // bound of its sign (+0 when the bound is 0)
                        const float bound = cand > 0.0f ? max_dynamic : min_dynamic;
                        const float next = clamped ? bound : cand;
                        if constexpr (kTape) {
                            const u32 br = !clamped ? 0u : (max_dynamic < cand ? 2u : (cand < -max_dynamic ? 3u : 1u));
                            branch = q == 4 + k ? br : branch;
                        }
                        const float delta = next - ap[4 + k];
                        const float dm = delta * im;
                        s.v += r.d * dm;
                        s.w += r.r * delta;
                        app = q == 4 + k ? next : app;
                        broken |= clamped;
                    }
                    if (iter + 1 == total && q == 0)
                        W.patches[m].flags = (__float_as_uint(fric.z) & ~1u) | (broken ? 1u : 0u);
                }
                if (c == 3u) s = LaneState{im, 0.0f};
                if (body >= 0) store_chunk(R, static_cast<u32>(body) * kStateBytes + 16u * c, s.v, s.w, need + 1u);
                // a velocity component once non-finite stays so through
                // later row updates (sums with finite or non-finite terms),
                // so the final check equals a check after every row
                if (c < 3u && (!isfinite(s.v) || !isfinite(s.w))) raise_flag(W, FYZZ_DY_NONFINITE);
                if (iter + 1 == total || n > nslots) W.app[8ull * i + q] = app;
                const bool end = side1 ? rk.y + 1 == rk.w : rk.x + 1 == rk.z;
                if (body >= 0 && end) {
                    if (iter + 1 == pos_iters) {
                        reinterpret_cast<float*>(W.mlin + body)[c] = s.v;
                        reinterpret_cast<float*>(W.mang + body)[c] = s.w;
                    }
                    if (iter + 1 == total) {
                        reinterpret_cast<float*>(W.lin + body)[c] = s.v;
                        reinterpret_cast<float*>(W.ang + body)[c] = s.w;
                    }
                }
                if (kTape && iter < W.tape_iters) {
                    const std::size_t t = static_cast<std::size_t>(iter) * 4 * W.nm + 4 * m + c;
                    if (!side1) {
                        if (c < no) W.tape_c[t] = static_cast<uint8_t>(branch);
                    } else if (rub && c < 2 * anchors) {
                        W.tape_f[t] = static_cast<uint8_t>(branch);
                    }
                    if (q == 0) W.tape_ni[static_cast<std::size_t>(iter) * W.nm + m] = normal_impulse;
                }
                have = false;
                i += nslots;
                progress = true;
                spins = 0;  // the budget bounds one wait, not the octet's whole sweep
            } else if (sides_or(poll ? 1u : 0u) && ++spins > kSpinLimit) {
                raise_flag(W, FYZZ_DY_LOGIC);
                iter = total;  // give up on this octet's work
            }
        }
        if (!__ballot(iter < total)) break;
        idle = __ballot(progress) ? 0u : idle + 1u;
        wait_backoff(idle);
        now = clock64();
    }
}

inline const void* pgs_kernel(bool tape) {
    return tape ? reinterpret_cast<const void*>(&k_pgs<true>) : reinterpret_cast<const void*>(&k_pgs<false>);
}

// --------------------------------------------------------------- adjoint
//
// Reverse mode through one step's PGS and integration with the step's
// contact rows frozen (normals, lever arms, effective masses, biases and
// friction frames are constants): every row update is then piecewise
// linear in the velocities, with the branch recorded in the tape. Inputs:
// adjoints of the step's outputs (velocity, angular velocity, position);
// outputs: adjoints of its input velocities and of each body's dynamic
// friction. Orientation is not differentiated (it reaches the outputs only
// through the frozen rows).

__device__ inline V ld3(const float* p, u32 i) { return {p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }

// adjoint state at the end of the sweeps, in the state lines (no updates
// yet; the inverse mass as in the sweep)
__global__ __launch_bounds__(kBlock) void k_adj_init(Ws W) {
    const u32 t = blockIdx.x * kBlock + threadIdx.x;
    if (t < W.nb) {
        const V av = ld3(W.adj_v_out, t), aw = ld3(W.adj_w_out, t);
        const float4 c0 = W.sii[3 * t], c1 = W.sii[3 * t + 1], c2 = W.sii[3 * t + 2];
        // v_out = v_pre + lin; w_out = w_pre + S ang (S symmetric)
        const float lin[4] = {av.x, av.y, av.z, W.lin[t].w};
        const float ang[4] = {c0.x * aw.x + c0.y * aw.y + c0.z * aw.z, c1.x * aw.x + c1.y * aw.y + c1.z * aw.z,
                              c2.x * aw.x + c2.y * aw.y + c2.z * aw.z, 0.f};
        for (u32 k = 0; k < 4; ++k) {
            W.vst[8 * t + 2 * k] = __float_as_uint(lin[k]);
            W.vst[8 * t + 2 * k + 1] = __float_as_uint(ang[k]);
        }
        W.adj_friction[t] = 0.0f;
    }
    const u32 nm = mcount(W);
    if (t < 8 * nm) {
        W.a_app[t] = 0.f;
        W.a_acc[t] = 0.f;
    }
    if (t < nm) W.a_df[t] = 0.f;
}

// The sweeps in reverse: iterations and partitions backwards. The motion
// snapshot taken after the last position iteration feeds the position
// update, so its adjoint (dt x adjoint of the position) joins the
// velocity-delta adjoint when the reverse reaches that point: the body's
// first manager of the iteration in reverse order adds it to the state it
// takes. Dataflow and lanes as in k_pgs, with the order reversed: the
// manager ranked r of d takes its body's state after (total - 1 - t)*d +
// d - 1 - r updates. A grid barrier between partitions took 1,535 us per
// step of 1,024 stacks of 64 boxes and 439 us of 5 stacks; this form takes
// 231 and 121 us.
__global__ __launch_bounds__(kBlock) void k_pgs_adjoint(Ws W) {
    const u32 q = threadIdx.x & 7u, c = q & 3u;
    const bool side1 = q >= 4u;
    const u32 slot = (blockIdx.x * kBlock + threadIdx.x) >> 3;
    const u32 nslots = (gridDim.x * kBlock) >> 3;
    const u32 np = min(ld(&W.ctr[kNParts]), kMaxParts);
    const u32 pos_iters = ld(&W.ctr[kPosIters]);
    const u32 vel_iters = max(ld(&W.ctr[kVelIters]), 1u);
    const u32 total = pos_iters + vel_iters;
    if (total > W.tape_iters) {  // the tape does not hold every iteration
        if (slot == 0 && q == 0) raise_flag(W, FYZZ_DY_OVERFLOW);
        return;
    }
    const u32 n = np ? W.part_off[np] : 0u;
    // `step` counts the reversed iterations; j the reversed positions
    u32 step = slot < n ? 0u : total, j = slot, spins = 0, idle = 0;
    const __amdgpu_buffer_rsrc_t R = state_rsrc(W);
    bool have = false;
    u32 miss = 0, need = 0;
    u64 wake = 0, now = 0;  // as in k_pgs
    int4 info = make_int4(-1, -1, 0, 0);
    int body = -1;
    Chunk st = {0u, 0u, 0u, 0u};
    float4 x[4] = {};
    LaneRow row[8] = {};
    float app = 0.f, acc = 0.f, inject = 0.f, ni = 0.f;
    u32 branch = 0;
    u32 anchors = 0;  // the patch's anchors and dynamic friction
    float df = 0.f;
    while (__ballot(step < total)) {
        bool progress = false;
        if (step < total) {
            const u32 i = n - 1u - j, iter = total - 1u - step;
            const bool fresh = !have;
            if (fresh) {
                info = W.sinfo[i];
                const uint4 rk = W.srank[i];
                have = true;
                body = side1 ? info.y : info.x;
                const u32 deg = side1 ? rk.w : rk.z, back = deg - 1u - (side1 ? rk.y : rk.x);
                need = step * deg + back;
                miss = body < 0 ? 0u : 1u;
                wake = 0;
                st = Chunk{0u, 0u, 0u, 0u};
                const float4* rows = W.rows + static_cast<std::size_t>(kRowQuads) * i + q;
                const fyzz_dy_patch& P = W.patches[static_cast<u32>(info.z)];
                anchors = min(P.anchor_count, 2u);
                df = P.dynamic_friction;
                const u32 no = static_cast<u32>(info.w) & 0xffu;
                x[0] = rows[0];
                if (no > 2u) x[1] = rows[kRowLanes];
                if (anchors) x[2] = rows[2 * kRowLanes];
                if (anchors > 1u) x[3] = rows[3 * kRowLanes];
                app = W.a_app[8ull * i + q];
                acc = W.a_acc[8ull * i + q];
                const std::size_t m = static_cast<u32>(info.z), base = static_cast<std::size_t>(iter) * W.nm;
                branch = (side1 ? W.tape_f : W.tape_c)[4 * (base + m) + c];
                ni = W.tape_ni[base + m];
                inject = 0.f;
                if (iter + 1 == pos_iters && back == 0u && body >= 0 && c < 3u && W.has_row[body])
                    inject = W.dt * W.adj_p_out[3 * body + c];
            }
            const bool poll = miss && now >= wake;
            if (poll) {
                st = load_chunk(R, static_cast<u32>(body) * kStateBytes + 16u * c);
                miss = quad_or((st.y ^ need) | (st.w ^ need));
                const u32 seen = __float_as_uint(quad<0>(__uint_as_float(st.y)));
                if (miss) wake = now + poll_delay(need, seen);
            }
            if (fresh) {
                unpack_rows(x[0], 0.f, row[0], row[1]);
                unpack_rows(x[1], 0.f, row[2], row[3]);
                unpack_rows(x[2], 0.f, row[4], row[5]);
                unpack_rows(x[3], 0.f, row[6], row[7]);
            }
            if (!sides_or(miss)) {
                const u32 no = static_cast<u32>(info.w) & 0xffu;
                LaneState s{__uint_as_float(st.x), __uint_as_float(st.z)};
                const float im = quad<3>(s.v);
                if (iter + 1 == pos_iters && c < 3u) s.v += inject;
                float ap[8];
                unpack_applied<0>(app, ap[0], ap[4]);
                unpack_applied<1>(app, ap[1], ap[5]);
                unpack_applied<2>(app, ap[2], ap[6]);
                unpack_applied<3>(app, ap[3], ap[7]);
                // every row's branch in all eight lanes, two bits each
                u32 br = (branch & 3u) << (2u * q);  // (an unsolved row's byte is unset)
                br = sides_or(quad_or(br));
                const u32 m = static_cast<u32>(info.z);
                float a_ni = 0.0f;
                if ((iter >= pos_iters || pos_iters - iter <= 3u) && anchors) {
                    const float coef = anchors == 2 ? 0.5f : 1.0f;
                    float a_maxd = 0.0f;
#pragma unroll
                    for (int k = 3; k >= 0; --k) {
                        if (k >= static_cast<int>(anchors * 2)) continue;
                        const LaneRow& r = row[4 + k];
                        const float a_delta = reverse_relative(s, r.d, r.r, im);
                        const float a_next = ap[4 + k] + a_delta;
                        float a_applied = -a_delta;
                        const u32 b = (br >> (2 * (4 + k))) & 3u;
                        float a_cand = 0.0f;
                        if (b <= 1u)
                            a_cand = a_next;
                        else if (b == 2u)
                            a_maxd += a_next;
                        else
                            a_maxd -= a_next;
                        a_applied += a_cand;
                        const float tgt = acc + r.vm * a_cand;
                        const float a_td = -r.vm * a_cand;
                        s.v += r.d * a_td;
                        s.w += r.r * a_td;
                        app = q == 4u + k ? a_applied : app;
                        acc = q == 4u + k ? tgt : acc;
                    }
                    // max_dynamic = df * coef * ni
                    if (q == 0) W.a_df[m] += coef * ni * a_maxd;
                    a_ni = df * coef * a_maxd;
                }
#pragma unroll
                for (int k = 3; k >= 0; --k) {
                    if (k >= static_cast<int>(no)) continue;
                    const LaneRow& r = row[k];
                    const float a_delta = reverse_relative(s, r.d, r.r, im);
                    const float a_next = ap[k] + a_delta + a_ni;
                    float a_applied = -a_delta;
                    if (((br >> (2 * k)) & 3u) == 1u) {
                        a_applied += a_next;
                        const float a_nv = -r.vm * a_next;
                        const float err = acc + a_next;
                        acc = q == static_cast<u32>(k) ? err : acc;
                        s.v += r.d * a_nv;
                        s.w += r.r * a_nv;
                    }
                    app = q == static_cast<u32>(k) ? a_applied : app;
                }
                if (c == 3u) s = LaneState{im, 0.0f};
                if (body >= 0) store_chunk(R, static_cast<u32>(body) * kStateBytes + 16u * c, s.v, s.w, need + 1u);
                W.a_app[8ull * i + q] = app;
                W.a_acc[8ull * i + q] = acc;
                have = false;
                j += nslots;
                if (j >= n) {
                    ++step;
                    j = slot;
                }
                progress = true;
                spins = 0;
            } else if (sides_or(poll ? 1u : 0u) && ++spins > kSpinLimit) {
                raise_flag(W, FYZZ_DY_LOGIC);
                step = total;  // give up on this octet's work
            }
        }
        idle = __ballot(progress) ? 0u : idle + 1u;
        wait_backoff(idle);
        now = clock64();
    }
}

// Rows' velocity terms back to the bodies' pre-integrated velocities; the
// combined dynamic friction back to each body's (max(0, (df0 + df1) / 2)).
__global__ __launch_bounds__(kBlock) void k_adj_rows(Ws W) {
    const u32 m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= mcount(W) || W.part[m] >= kMaxParts) return;
    const fyzz_dy_manager& M = W.mg[m];
    const int i0 = M.body0, i1 = M.body1;
    const u32 pos = W.pos_of[m];
    V ava{0.f, 0.f, 0.f}, avb{0.f, 0.f, 0.f}, awa{0.f, 0.f, 0.f}, awb{0.f, 0.f, 0.f};
    const u32 no = W.order[m] & 0xffu;
    for (u32 q = 0; q < no; ++q) {
        const RowOut r = read_row(W, pos, q);
        const float4 x0 = W.craw[2 * (4 * m + q)], x1 = W.craw[2 * (4 * m + q) + 1];
        const float a_vrel = x0.w * r.s.x * W.a_acc[8ull * pos + q];
        const V n = r.d;
        ava = vadd(ava, vmul(n, a_vrel));
        avb = vsub(avb, vmul(n, a_vrel));
        awa = vadd(awa, vmul(f3(x0), a_vrel));
        awb = vsub(awb, vmul(f3(x1), a_vrel));
    }
    const fyzz_dy_patch& P = W.patches[m];
    for (u32 k = 0; k < 2 * min(P.anchor_count, 2u); ++k) {
        const V t = read_row(W, pos, 4 + k).d;
        const float a_t = W.a_acc[8ull * pos + 4 + k];
        // target = -(t . (va - vb) + (ra x t) . wa - (rb x t) . wb)
        ava = vsub(ava, vmul(t, a_t));
        avb = vadd(avb, vmul(t, a_t));
        awa = vsub(awa, vmul(f3(W.fraw[2 * (4 * m + k)]), a_t));
        awb = vadd(awb, vmul(f3(W.fraw[2 * (4 * m + k) + 1]), a_t));
    }
    const float a_df = P.dynamic_friction > 0.0f ? 0.5f * W.a_df[m] : 0.0f;
    // each side's terms, summed per body by k_adj_bodies in the body's
    // incidence order (no atomics: the gradients are the same every run)
    W.a_side[4 * m] = make_float4(ava.x, ava.y, ava.z, a_df);
    W.a_side[4 * m + 1] = make_float4(awa.x, awa.y, awa.z, 0.f);
    W.a_side[4 * m + 2] = make_float4(avb.x, avb.y, avb.z, a_df);
    W.a_side[4 * m + 3] = make_float4(awb.x, awb.y, awb.z, 0.f);
}

// Pre-integration backwards: v_pre = lm (v_in + g dt), w_pre = am w_in, and
// v_pre reaches the outputs directly (v_out, and p_out through dt).
__global__ __launch_bounds__(kBlock) void k_adj_bodies(Ws W) {
    const u32 i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= W.nb) return;
    const fyzz_dy_body& b = W.bodies[i];
    const V av = ld3(W.adj_v_out, i), aw = ld3(W.adj_w_out, i), ap = ld3(W.adj_p_out, i);
    if (b.flags & 1u) {  // asleep: the step leaves it unchanged
        for (int k = 0; k < 3; ++k) {
            W.adj_v_in[3 * i + k] = (&av.x)[k];
            W.adj_w_in[3 * i + k] = (&aw.x)[k];
        }
        return;
    }
    // the rows' terms of the body's managers, in incidence order (sorted by
    // manager when the partitions were built)
    V a_rows_v{0.f, 0.f, 0.f}, a_rows_w{0.f, 0.f, 0.f};
    float a_fric = 0.0f;
    if (mcount(W) && W.has_row[i]) {
        for (u32 k = W.off[i]; k < W.off[i] + W.deg[i]; ++k) {
            const u32 e = W.inc[k], m = e >> 1, side = e & 1u;
            if (W.part[m] >= kMaxParts) continue;
            const float4 v = W.a_side[4 * m + 2 * side], w = W.a_side[4 * m + 2 * side + 1];
            a_rows_v = vadd(a_rows_v, f3(v));
            a_rows_w = vadd(a_rows_w, f3(w));
            a_fric += v.w;
        }
    }
    W.adj_friction[i] = a_fric;
    const V a_vpre = vadd(vadd(av, vmul(ap, W.dt)), a_rows_v);
    const V a_wpre = vadd(aw, a_rows_w);
    const float lm = smax(1.0f - b.linear_damping * W.dt, 0.0f);
    const float am = smax(1.0f - b.angular_damping * W.dt, 0.0f);
    W.adj_v_in[3 * i] = lm * a_vpre.x;
    W.adj_v_in[3 * i + 1] = lm * a_vpre.y;
    W.adj_v_in[3 * i + 2] = lm * a_vpre.z;
    W.adj_w_in[3 * i] = am * a_wpre.x;
    W.adj_w_in[3 * i + 1] = am * a_wpre.y;
    W.adj_w_in[3 * i + 2] = am * a_wpre.z;
}

// ------------------------------------------------------------- integrate

// sinf and cosf as the C library the native scene links computes them
// (glibc 2.28 and later ship the ARM optimized-routines sinf/cosf): the
// float argument widened to double; below 0.75 (a test on the top 12 bits
// against pi/4) a double polynomial in x^2 rounded once to float, below
// 2^-12 the argument itself (sin) or 1 (cos); up to 120 a reduction by the
// nearest multiple of pi/2 first. The published minimax coefficients are
// restated here; every float in [2^-13, 120) gives the host library's
// result but 17 arguments above 17 (the nearest-multiple reduction of a
// value close to a multiple of pi/2). Beyond 120 (angular speeds above
// 28,800 rad/s at 120 Hz) the device's own functions are used.
namespace libm {
constexpr double kS1 = -0x1.555545995a603p-3, kS2 = 0x1.1107605230bc4p-7, kS3 = -0x1.994eb3774cf24p-13;
constexpr double kC0 = 0x1p0, kC1 = -0x1.ffffffd0c621cp-2, kC2 = 0x1.55553e1068f19p-5,
                 kC3 = -0x1.6c087e89a359dp-10, kC4 = 0x1.99343027bf8c3p-16;
constexpr double kHalfPiInv = 0x1.45F306DC9C883p+23, kHalfPi = 0x1.921FB54442D18p0;

__device__ inline uint32_t top12(float f) { return (__float_as_uint(f) >> 20) & 0x7ffu; }

// cos_branch: the even polynomial (cos), else the odd one (sin); negate:
// the coefficients' sign flipped (the odd quadrants of the reduction)
__device__ inline double poly(double x, double x2, bool cos_branch, bool negate) {
    if (!cos_branch) {
        const double x3 = x * x2;
        const double s1 = kS2 + x2 * kS3;
        const double x7 = x3 * x2;
        const double s = x + x3 * kS1;
        return s + x7 * s1;
    }
    const double g = negate ? -1.0 : 1.0;
    const double x4 = x2 * x2;
    const double c2 = g * kC3 + x2 * (g * kC4);
    const double c1 = g * kC0 + x2 * (g * kC1);
    const double x6 = x4 * x2;
    const double c = c1 + x4 * (g * kC2);
    return c + x6 * c2;
}

__device__ inline float sin_cos(float y, bool want_cos) {
    const double x = y;
    if (top12(y) < top12(0x1.921FB6p-1f)) {
        if (top12(y) < top12(0x1p-12f)) return want_cos ? 1.0f : y;
        return static_cast<float>(poly(x, x * x, want_cos, false));
    }
    if (top12(y) < top12(120.0f)) {
        const double r = x * kHalfPiInv;
        const int n = (static_cast<int>(r) + 0x800000) >> 24;
        const double xr = x - n * kHalfPi;
        const double sgn = ((n & 3) == 1 || (n & 3) == 2) ? -1.0 : 1.0;
        const int q = want_cos ? n + 1 : n;
        return static_cast<float>(poly(xr * sgn, xr * xr, (q & 1) != 0, (q & 2) != 0));
    }
    return want_cos ? static_cast<float>(cos(static_cast<double>(y))) : sinf(y);
}
}  // namespace libm

// scene.cpp:111-146
__device__ bool integrate_quaternion(Q pose, V w, float dt, Q& out) {
    float ww = w.x * w.x + w.y * w.y + w.z * w.z;
    if (ww != 0.0f) {
        ww = sqrtf(ww);
        const float max_w = 1.0e7f;
        if (ww > max_w) {
            const float s = max_w / ww;
            w = {w.x * s, w.y * s, w.z * s};
            ww = max_w;
        }
        const float v = dt * ww * 0.5f;
        const float s = libm::sin_cos(v, false) / ww;
        const float c = libm::sin_cos(v, true);
        const Q dq = qmul(Q{w.x * s, w.y * s, w.z * s, 0.0f}, pose);
        const Q nx{dq.x + pose.x * c, dq.y + pose.y * c, dq.z + pose.z * c, dq.w + pose.w * c};
        const float len = sqrtf(nx.x * nx.x + nx.y * nx.y + nx.z * nx.z + nx.w * nx.w);
        if (!(len > 0.0f) || !isfinite(len)) return false;
        pose = {nx.x / len, nx.y / len, nx.z / len, nx.w / len};
    }
    out = pose;
    return true;
}

__device__ inline V apply_sii(V w, float4 c0, float4 c1, float4 c2, V s) {
    return {w.x + c0.x * s.x + c1.x * s.y + c2.x * s.z, w.y + c0.y * s.x + c1.y * s.y + c2.y * s.z,
            w.z + c0.z * s.x + c1.z * s.y + c2.z * s.z};
}

// publish (scene.cpp:9509-9549), integrate and sleep check (10508-10707)
__device__ void integrate_body(const Ws& W, u32 i) {
    fyzz_dy_body& B = W.bodies[i];
    if (B.flags & 1u) return;
    const float dt = W.dt;
    V vel = f3(W.pv[i]), ang = f3(W.pw[i]);
    V motion_lin = vel, motion_ang = ang;
    if (W.has_row[i]) {
        const V rv = vel, rw = ang;
        const float4 c0 = W.sii[3 * i], c1 = W.sii[3 * i + 1], c2 = W.sii[3 * i + 2];
        const V ld = f3(W.lin[i]), as = f3(W.ang[i]);
        const V ml = f3(W.mlin[i]), ma = f3(W.mang[i]);
        vel = vadd(rv, ld);
        ang = apply_sii(rw, c0, c1, c2, as);
        motion_lin = vadd(rv, ml);
        motion_ang = apply_sii(rw, c0, c1, c2, ma);
        if (!finite3(vel) || !finite3(ang)) raise_flag(W, FYZZ_DY_NONFINITE);
    }
    const V p0 = v3(B.position);
    const Q q0 = q4(B.orientation);
    const V center = mass_position(p0, q0);
    V p{center.x + motion_lin.x * dt, center.y + motion_lin.y * dt, center.z + motion_lin.z * dt};
    Q q;
    if (!integrate_quaternion(mass_orientation(q0), motion_ang, dt, q)) {
        raise_flag(W, FYZZ_DY_NONFINITE);
        q = q0;
    }
    q = qmul(q, Q{-0.0f, -0.0f, -0.0f, 1.0f});
    const V off = srot(q, V{0.f, 0.f, 0.f});
    p = vsub(p, off);
    if (!finite3(p) || !finite4(q)) raise_flag(W, FYZZ_DY_NONFINITE);
    // sleep check (scene.cpp:10640-10705)
    const float wake_reset = 20.0f * 0.02f;
    const float energy_threshold = 5.0e-5f * 10.0f * 10.0f;
    float wc = B.wake_counter;
    V lin_acc = v3(B.sleep_linear_acc), ang_acc = v3(B.sleep_angular_acc);
    if (wc < wake_reset * 0.5f || wc < dt) {
        const V la = srot_inv(q, motion_ang);
        const V l2 = vadd(lin_acc, motion_lin);
        const V a2 = vadd(ang_acc, la);
        const V ii = v3(B.inverse_inertia);
        const V inertia{ii.x > 0.0f ? 1.0f / ii.x : 1.0f, ii.y > 0.0f ? 1.0f / ii.y : 1.0f,
                        ii.z > 0.0f ? 1.0f / ii.z : 1.0f};
        const float ang_e =
            (a2.x * a2.x * inertia.x + a2.y * a2.y * inertia.y + a2.z * a2.z * inertia.z) * B.inverse_mass;
        const float lin_e = l2.x * l2.x + l2.y * l2.y + l2.z * l2.z;
        const float ne = 0.5f * (ang_e + lin_e);
        const float cluster = 1.0f + float(B.counted_interactions);
        const float th = cluster * energy_threshold;
        if (ne >= th) {
            lin_acc = {0.f, 0.f, 0.f};
            ang_acc = {0.f, 0.f, 0.f};
            const float factor = th == 0.0f ? 2.0f : smin(ne / th, 2.0f);
            wc = factor * 0.5f * wake_reset + dt * (cluster - 1.0f);
        } else {
            lin_acc = l2;
            ang_acc = a2;
            wc = smax(wc - dt, 0.0f);
        }
    } else {
        wc = smax(wc - dt, 0.0f);
    }
    const bool ready = wc == 0.0f;
    if (ready) {
        lin_acc = {0.f, 0.f, 0.f};
        ang_acc = {0.f, 0.f, 0.f};
    }
    put3(B.position, p);
    B.orientation[0] = q.x;
    B.orientation[1] = q.y;
    B.orientation[2] = q.z;
    B.orientation[3] = q.w;
    put3(B.linear_velocity, vel);
    put3(B.angular_velocity, ang);
    B.wake_counter = wc;
    put3(B.sleep_linear_acc, lin_acc);
    put3(B.sleep_angular_acc, ang_acc);
    B.flags = (B.flags & ~2u) | (ready ? 2u : 0u);
}

// impulses per manifold contact and the partition of each manager; the
// step's contact and friction row counts
// (the impulses land in their contact slots through selects, and the row
// totals are summed per workgroup in LDS: one global atomic per workgroup
// instead of one per wave on the same two words)
__global__ __launch_bounds__(kBlock) void k_outputs(Ws W) {
    __shared__ u32 s_rows, s_frows;
    if (threadIdx.x == 0) s_rows = s_frows = 0;
    __syncthreads();
    const u32 m = blockIdx.x * kBlock + threadIdx.x;
    if (W.with_rows && m < W.nb) integrate_body(W, m);
    u32 rows = 0, frows = 0;
    if (m < mcount(W)) {
        if (W.parts_out) W.parts_out[m] = W.part[m];
        float out[4] = {0.f, 0.f, 0.f, 0.f};
        if (W.with_rows && W.part[m] < kMaxParts) {
            const u32 o = W.order[m];
            const u32 no = min(o & 0xffu, 4u);
            const u32 pos = W.pos_of[m];
            const float4 app = *reinterpret_cast<const float4*>(W.app + 8ull * pos);
            const float applied[4] = {app.x, app.y, app.z, app.w};
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                if (q >= no) continue;
                const u32 slot = (o >> (8 + 4 * q)) & 0xfu;
                const float v = applied[q];
#pragma unroll
                for (u32 k = 0; k < 4; ++k) out[k] = slot == k ? v : out[k];
            }
            rows = no;
            frows = 2u * ((static_cast<u32>(W.sinfo[pos].w) >> 8) & 0xffu);
        }
        if (W.impulses)
            for (u32 q = 0; q < 4; ++q) W.impulses[4 * m + q] = out[q];
    }
    for (int d = kWave / 2; d > 0; d >>= 1) {
        rows += __shfl_xor(rows, d, kWave);
        frows += __shfl_xor(frows, d, kWave);
    }
    if (lane_id() == 0 && (rows || frows)) {
        atomicAdd(&s_rows, rows);
        atomicAdd(&s_frows, frows);
    }
    __syncthreads();
    if (threadIdx.x == 0 && (s_rows || s_frows)) {
        atomicAdd(&W.ctr[kContacts], s_rows);
        atomicAdd(&W.ctr[kFrictionRows], s_frows);
    }
}

// Scene::write_back_contacts' friction part (scene.cpp:9339-9388) for
// the last step's managers: each anchor's world position on body0 (the
// manager's first body, whose frame holds the patch's body0 anchors: the
// mass pose the rows were prepared with, centre + rotated local anchor)
// and its world impulse, the two tangent rows' tangent x applied force
// summed in double.
__global__ __launch_bounds__(kBlock) void k_anchors(Ws W, fyzz_friction_anchors* out) {
    const u32 m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= mcount(W)) return;
    fyzz_friction_anchors r{};
    if (W.with_rows && W.part[m] < kMaxParts) {
        const fyzz_dy_patch& P = W.patches[m];
        const u32 na = min(P.anchor_count, 2u);
        r.anchor_count = na;
        r.broken = P.flags & 1u;
        const int b0 = W.mg[m].body0;
        const float4 cp = W.rpos[b0 >= 0 ? b0 : 0];
        const float4 cq = W.rq[b0 >= 0 ? b0 : 0];
        const Q q{cq.x, cq.y, cq.z, cq.w};
        for (u32 k = 0; k < na; ++k) {
            const V local{P.body0_anchors[k][0], P.body0_anchors[k][1], P.body0_anchors[k][2]};
            const V rot = srot(q, local);
            r.position[k][0] = cp.x + rot.x;
            r.position[k][1] = cp.y + rot.y;
            r.position[k][2] = cp.z + rot.z;
            const u32 pos = W.pos_of[m];
            const V x = read_row(W, pos, 4 + 2 * k).d, y = read_row(W, pos, 5 + 2 * k).d;
            const float ax = W.app[8ull * pos + 4 + 2 * k], ay = W.app[8ull * pos + 5 + 2 * k];
            r.impulse[k][0] = static_cast<double>(x.x) * ax + static_cast<double>(y.x) * ay;
            r.impulse[k][1] = static_cast<double>(x.y) * ax + static_cast<double>(y.y) * ay;
            r.impulse[k][2] = static_cast<double>(x.z) * ax + static_cast<double>(y.z) * ay;
        }
    }
    out[m] = r;
}

}  // namespace fyzz_hip::dy

using namespace fyzz_hip;

struct fyzz_hip_dy {
    fyzz_hip_context* ctx = nullptr;
    u32 body_cap = 0, mgr_cap = 0;
    int coop_blocks_partition = 0, coop_blocks_pgs = 0, coop_blocks_adjoint = 0;
    bool plain_launch = false;
    DevBuf<float4> pv, pw, lin, ang, mlin, mang, rpos, rq, sii;
    DevBuf<u32> has_row, deg, off, fill, body_mask;
    DevBuf<u32> inc, pred, part, pend, sorted, order;
    DevBuf<uint8_t> dd;
    DevBuf<u64> entry;
    DevBuf<int4> sinfo;
    DevBuf<uint4> srank;
    DevBuf<u32> erank, pos_of;
    DevBuf<u64> vst;
    DevBuf<float4> rows, fric;
    DevBuf<float> app;
    DevBuf<u32> part_count, part_off, part_fill, ctr, flags, bar;
    // tape mode
    bool tape = false;
    bool taped_step = false;  // the last solved step recorded a tape
    DevBuf<uint8_t> tape_c, tape_f;
    DevBuf<float> tape_ni, a_app, a_acc, a_df;
    DevBuf<float4> craw, fraw, a_side;
    dy::Ws ws{};
    bool prepared = false;
};

namespace {

int resident_blocks(const void* kernel, int device) {
    int per_cu = 0, cus = 0;
    FYZZ_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, dy::kBlock, 0));
    FYZZ_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    FYZZ_REQUIRE(per_cu > 0 && cus > 0, kDeviceError, "dy: cooperative kernel does not fit a compute unit");
    return per_cu * cus;
}
// Cooperative launch (the runtime checks that every workgroup is resident).
// Inside a captured graph the kernels are launched as plain kernels with
// the same small grid (far below the device's resident capacity); the
// sweep's bounded waits turn a non-resident grid into a status flag.
void launch_coop(const void* kernel, int blocks, dy::Ws& ws, hipStream_t st, bool plain) {
    void* args[] = {&ws};
    if (plain)
        FYZZ_HIP_CHECK(hipLaunchKernel(kernel, dim3(blocks), dim3(dy::kBlock), args, 0, st));
    else
        FYZZ_HIP_CHECK(hipLaunchCooperativeKernel(kernel, dim3(blocks), dim3(dy::kBlock), args, 0, st));
}

void dy_prepare(fyzz_hip_dy* d, float dt, uint32_t nb, fyzz_dy_body* bodies, uint32_t ns,
                const fyzz_dy_static* statics, uint32_t nm, const fyzz_dy_manager* managers,
                const fyzz_dy_patch* history, uint32_t nh, fyzz_dy_patch* patches, bool partition_only,
                const u32* d_nm = nullptr) {
    FYZZ_REQUIRE(nb <= d->body_cap, kOverflow, "dy: body count exceeds the capacity given at creation");
    FYZZ_REQUIRE(nm <= d->mgr_cap, kOverflow, "dy: manager count exceeds the capacity given at creation");
    FYZZ_REQUIRE(dt > 0.0f, kInvalidArgument, "dy: dt must be positive");
    FYZZ_REQUIRE(nb == 0 || bodies, kInvalidArgument, "dy: null bodies");
    FYZZ_REQUIRE(nm == 0 || managers, kInvalidArgument, "dy: null managers");
    FYZZ_REQUIRE(ns == 0 || statics, kInvalidArgument, "dy: null statics");
    FYZZ_REQUIRE(nh == 0 || history, kInvalidArgument, "dy: null history");
    FYZZ_REQUIRE(partition_only || nm == 0 || patches, kInvalidArgument, "dy: null patch output");
    dy::Ws& w = d->ws;
    w.dt = dt;
    w.nb = nb;
    w.ns = partition_only ? 0xffffffffu : ns;  // partitions never read statics
    w.nm = nm;
    w.nh = nh;
    w.bodies = bodies;
    w.statics = statics;
    w.mg = managers;
    w.history = history;
    w.patches = patches;
    w.d_nm = d_nm;
    w.with_rows = partition_only ? 0u : 1u;
    w.tape = (d->tape && !partition_only) ? 1u : 0u;
    d->taped_step = false;
    hipStream_t st = d->ctx->stream;
    auto& prof = d->ctx->prof;
    {
        ProfScope ps(&prof, "dy.bodies", st);
        hipLaunchKernelGGL(dy::k_pre, dim3(grid_for(std::max<u32>(nb, dy::kMaxParts), dy::kBlock)), dim3(dy::kBlock), 0,
                           st, w);
        if (nm) hipLaunchKernelGGL(dy::k_mark, dim3(grid_for(nm, dy::kBlock)), dim3(dy::kBlock), 0, st, w);
        if (nb) hipLaunchKernelGGL(dy::k_rows, dim3(grid_for(nb, dy::kBlock)), dim3(dy::kBlock), 0, st, w);
        FYZZ_HIP_CHECK(hipGetLastError());
    }
    {
        ProfScope ps(&prof, "dy.partition", st);
        const dim3 blk(dy::kBlock);
        const dim3 gb(grid_for(std::max<u32>(nb, 1), dy::kBlock)), gm(grid_for(std::max<u32>(nm, 1), dy::kBlock));
        if (nm) {
            hipLaunchKernelGGL(dy::k_part_fill, gm, blk, 0, st, w);
            hipLaunchKernelGGL(dy::k_part_chain, gb, blk, 0, st, w);
            FYZZ_HIP_CHECK(hipGetLastError());
            hipLaunchKernelGGL(dy::k_part_color,
                               dim3(std::min<u32>(d->coop_blocks_partition, grid_for(nm, dy::kBlock))), blk, 0, st, w);
            hipLaunchKernelGGL(dy::k_part_static, gb, blk, 0, st, w);
        }
        hipLaunchKernelGGL(dy::k_part_scatter, gm, blk, 0, st, w);
        FYZZ_HIP_CHECK(hipGetLastError());
    }
    if (!partition_only && nm) {
        ProfScope ps(&prof, "dy.prep", st);
        hipLaunchKernelGGL(dy::k_prep, dim3(grid_for(nm, 128)), dim3(128), 0, st, w);
        FYZZ_HIP_CHECK(hipGetLastError());
    }
    d->prepared = !partition_only;
}

void dy_solve(fyzz_hip_dy* d) {
    FYZZ_REQUIRE(d->prepared, kLogicError, "dy_solve: no prepared step");
    d->taped_step = d->ws.tape != 0;
    if (!d->ws.nm) return;
    ProfScope ps(&d->ctx->prof, "dy.pgs", d->ctx->stream);
    launch_coop(dy::pgs_kernel(d->ws.tape != 0), d->coop_blocks_pgs, d->ws, d->ctx->stream,
                d->plain_launch || !d->ctx->cooperative);
}

void dy_integrate(fyzz_hip_dy* d, float* impulses, uint32_t* partitions) {
    FYZZ_REQUIRE(d->prepared, kLogicError, "dy_integrate: no prepared step");
    hipStream_t st = d->ctx->stream;
    d->ws.impulses = impulses;
    d->ws.parts_out = partitions;
    ProfScope ps(&d->ctx->prof, "dy.integrate", st);
    const u32 span = std::max(d->ws.nb, d->ws.nm);
    if (span) hipLaunchKernelGGL(dy::k_outputs, dim3(grid_for(span, dy::kBlock)), dim3(dy::kBlock), 0, st, d->ws);
    FYZZ_HIP_CHECK(hipGetLastError());
    d->prepared = false;
}

void dy_set_tape(fyzz_hip_dy* d, bool enabled) {
    if (enabled && !d->tape_c.p) {
        const std::size_t nm = std::max<u32>(d->mgr_cap, 1), nb = std::max<u32>(d->body_cap, 1);
        constexpr u32 kTapeIters = 8;
        d->tape_c.reserve(kTapeIters * 4 * nm);
        d->tape_f.reserve(kTapeIters * 4 * nm);
        d->tape_ni.reserve(kTapeIters * nm);
        for (auto* b : {&d->a_app, &d->a_acc}) b->reserve(8 * nm);
        d->a_df.reserve(nm);
        d->craw.reserve(8 * nm);
        d->fraw.reserve(8 * nm);
        d->a_side.reserve(4 * nm);
        dy::Ws& w = d->ws;
        w.tape_iters = kTapeIters;
        w.tape_c = d->tape_c.p;
        w.tape_f = d->tape_f.p;
        w.tape_ni = d->tape_ni.p;
        w.craw = d->craw.p;
        w.fraw = d->fraw.p;
        w.a_app = d->a_app.p;
        w.a_acc = d->a_acc.p;
        w.a_df = d->a_df.p;
        w.a_side = d->a_side.p;
    }
    d->tape = enabled;
}

void dy_adjoint(fyzz_hip_dy* d, const float* adj_v_out, const float* adj_w_out, const float* adj_p_out,
                float* adj_v_in, float* adj_w_in, float* adj_friction) {
    FYZZ_REQUIRE(d->taped_step, kLogicError, "dy_adjoint: the last step was not solved with the tape on");
    FYZZ_REQUIRE(!d->prepared, kLogicError, "dy_adjoint: the last step has not been integrated");
    dy::Ws& w = d->ws;
    FYZZ_REQUIRE(w.nb == 0 || (adj_v_out && adj_w_out && adj_p_out && adj_v_in && adj_w_in && adj_friction),
                 kInvalidArgument, "dy_adjoint: null device pointer");
    w.adj_v_out = adj_v_out;
    w.adj_w_out = adj_w_out;
    w.adj_p_out = adj_p_out;
    w.adj_v_in = adj_v_in;
    w.adj_w_in = adj_w_in;
    w.adj_friction = adj_friction;
    hipStream_t st = d->ctx->stream;
    ProfScope ps(&d->ctx->prof, "dy.adjoint", st);
    const u32 span = std::max<u32>(w.nb, 8 * w.nm);
    if (span) hipLaunchKernelGGL(dy::k_adj_init, dim3(grid_for(span, dy::kBlock)), dim3(dy::kBlock), 0, st, w);
    if (w.nm) {
        launch_coop(reinterpret_cast<const void*>(&dy::k_pgs_adjoint), d->coop_blocks_adjoint, w, st,
                    d->plain_launch || !d->ctx->cooperative);
        hipLaunchKernelGGL(dy::k_adj_rows, dim3(grid_for(w.nm, dy::kBlock)), dim3(dy::kBlock), 0, st, w);
    }
    if (w.nb) hipLaunchKernelGGL(dy::k_adj_bodies, dim3(grid_for(w.nb, dy::kBlock)), dim3(dy::kBlock), 0, st, w);
    FYZZ_HIP_CHECK(hipGetLastError());
}

}  // namespace

namespace fyzz_hip::dy {
const u32* counters(fyzz_hip_dy* d) { return d->ctr.get(); }
void set_plain_launch(fyzz_hip_dy* d, bool plain) { d->plain_launch = plain; }
void set_coop_blocks(fyzz_hip_dy* d, int partition_blocks, int pgs_blocks) {
    const int cap_p = resident_blocks(reinterpret_cast<const void*>(&k_part_color), d->ctx->device);
    // the sweep has no grid barrier: its cap is the resident capacity
    const int cap_s = resident_blocks(pgs_kernel(true), d->ctx->device);
    FYZZ_REQUIRE(partition_blocks > 0 && pgs_blocks > 0, kInvalidArgument, "dy: workgroup counts must be positive");
    d->coop_blocks_partition = std::min(partition_blocks, cap_p);
    d->coop_blocks_pgs = std::min(pgs_blocks, cap_s);
}
void effective_blocks(int device, int partition_blocks, int pgs_blocks, int* partition_out, int* pgs_out) {
    const int cap_p = resident_blocks(reinterpret_cast<const void*>(&k_part_color), device);
    const void* pgs = pgs_kernel(true);
    *partition_out = std::min(partition_blocks > 0 ? partition_blocks : kColorBlocks, cap_p);
    *pgs_out = pgs_blocks > 0 ? std::min(pgs_blocks, resident_blocks(pgs, device)) : std::min(resident_blocks(pgs, device), kPgsBlocks);
}
void coop_blocks_of(fyzz_hip_dy* d, int* partition_blocks, int* pgs_blocks) {
    *partition_blocks = d->coop_blocks_partition;
    *pgs_blocks = d->coop_blocks_pgs;
}

void step_device(fyzz_hip_dy* d, float dt, u32 nb, fyzz_dy_body* bodies, u32 ns, const fyzz_dy_static* statics,
                 u32 nm_cap, const u32* d_nm, const fyzz_dy_manager* managers, const fyzz_dy_patch* history,
                 u32 nh, fyzz_dy_patch* patches, float* impulses, u32* partitions) {
    dy_prepare(d, dt, nb, bodies, ns, statics, nm_cap, managers, history, nh, patches, false, d_nm);
    dy_solve(d);
    dy_integrate(d, impulses, partitions);
}
}  // namespace fyzz_hip::dy

extern "C" {

int fyzz_hip_dy_create(fyzz_hip_context* ctx, uint32_t body_capacity, uint32_t manager_capacity,
                       fyzz_hip_dy** out) {
    return guarded(ctx, [&] {
        FYZZ_REQUIRE(out, kInvalidArgument, "dy_create: null out");
        FYZZ_REQUIRE(manager_capacity < (1u << 30), kInvalidArgument, "dy_create: manager capacity too large");
        // the sweep addresses a body's 64-byte state line with a 32-bit offset
        FYZZ_REQUIRE(body_capacity <= (1u << 26), kInvalidArgument, "dy_create: body capacity too large");
        auto d = std::make_unique<fyzz_hip_dy>();
        d->ctx = ctx;
        d->body_cap = body_capacity;
        d->mgr_cap = manager_capacity;
        const std::size_t nb = std::max<u32>(body_capacity, 1), nm = std::max<u32>(manager_capacity, 1);
        for (auto* b : {&d->pv, &d->pw, &d->lin, &d->ang, &d->mlin, &d->mang, &d->rpos, &d->rq}) b->reserve(nb);
        d->sii.reserve(3 * nb);
        for (auto* b : {&d->has_row, &d->deg, &d->off, &d->fill, &d->body_mask}) b->reserve(nb);
        for (auto* b : {&d->inc, &d->pred}) b->reserve(2 * nm);
        d->entry.reserve(2 * nm);
        d->sinfo.reserve(nm);
        d->srank.reserve(nm);
        d->erank.reserve(2 * nm);
        d->vst.reserve(8ull * nb);
        d->pos_of.reserve(nm);
        for (auto* b : {&d->part, &d->pend, &d->sorted, &d->order}) b->reserve(nm);
        d->dd.reserve(nm);
        d->rows.reserve(dy::kRowQuads * nm);
        d->app.reserve(8 * nm);
        d->fric.reserve(nm);
        d->part_count.reserve(dy::kMaxParts + 1);
        d->part_off.reserve(dy::kMaxParts + 1);
        d->part_fill.reserve(dy::kMaxParts);
        d->ctr.reserve(dy::kCtrWords);
        d->flags.reserve(1);
        d->bar.reserve(dy::kBarWords);
        FYZZ_HIP_CHECK(hipMemset(d->bar.get(), 0, dy::kBarWords * sizeof(u32)));
        d->coop_blocks_partition =
            std::min(resident_blocks(reinterpret_cast<const void*>(&dy::k_part_color), ctx->device), dy::kColorBlocks);
        d->coop_blocks_pgs = std::min(resident_blocks(dy::pgs_kernel(true), ctx->device), dy::kPgsBlocks);
        d->coop_blocks_adjoint =
            std::min(resident_blocks(reinterpret_cast<const void*>(&dy::k_pgs_adjoint), ctx->device), dy::kPgsBlocks);
        FYZZ_HIP_CHECK(hipMemset(d->flags.get(), 0, sizeof(u32)));
        FYZZ_HIP_CHECK(hipMemset(d->ctr.get(), 0, dy::kCtrWords * sizeof(u32)));
        dy::Ws& w = d->ws;
        w.pv = d->pv.get();
        w.pw = d->pw.get();
        w.lin = d->lin.get();
        w.ang = d->ang.get();
        w.mlin = d->mlin.get();
        w.mang = d->mang.get();
        w.rpos = d->rpos.get();
        w.rq = d->rq.get();
        w.sii = d->sii.get();
        w.has_row = d->has_row.get();
        w.deg = d->deg.get();
        w.off = d->off.get();
        w.fill = d->fill.get();
        w.body_mask = d->body_mask.get();
        w.inc = d->inc.get();
        w.pred = d->pred.get();
        w.part = d->part.get();
        w.entry = d->entry.get();
        w.sinfo = d->sinfo.get();
        w.srank = d->srank.get();
        w.erank = d->erank.get();
        w.vst = d->vst.get();
        w.pos_of = d->pos_of.get();
        w.pend = d->pend.get();
        w.sorted = d->sorted.get();
        w.order = d->order.get();
        w.dd = d->dd.get();
        w.rows = d->rows.get();
        w.app = d->app.get();
        w.fric = d->fric.get();
        w.part_count = d->part_count.get();
        w.part_off = d->part_off.get();
        w.part_fill = d->part_fill.get();
        w.ctr = d->ctr.get();
        w.flags = d->flags.get();
        w.bar = d->bar.get();
        // every workspace array the step kernels touch must exist
        const void* need[] = {w.pv, w.pw, w.lin, w.ang, w.mlin, w.mang, w.rpos, w.rq, w.sii, w.has_row,
                              w.deg, w.off, w.fill, w.body_mask, w.inc, w.pred, w.part, w.pend,
                              w.sorted, w.order, w.entry, w.sinfo, w.srank, w.erank, w.vst, w.pos_of, w.rows,
                              w.app, w.fric,
                              w.part_count, w.part_off, w.part_fill, w.ctr, w.flags, w.bar};
        for (const void* q : need) FYZZ_REQUIRE(q != nullptr, kDeviceError, "dy_create: workspace array missing");
        *out = d.release();
    });
}

int fyzz_hip_dy_destroy(fyzz_hip_dy* d) {
    if (!d) return kInvalidArgument;
    (void)hipSetDevice(d->ctx->device);
    (void)hipStreamSynchronize(d->ctx->stream);
    delete d;
    return kOk;
}

int fyzz_hip_dy_partition(fyzz_hip_dy* d, uint32_t n_bodies, fyzz_dy_body* bodies, uint32_t n_managers,
                          const fyzz_dy_manager* managers, uint32_t* partitions) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] {
        FYZZ_REQUIRE(n_managers == 0 || partitions, kInvalidArgument, "dy_partition: null output");
        dy_prepare(d, 1.0f, n_bodies, bodies, 0, nullptr, n_managers, managers, nullptr, 0, nullptr, true);
        d->ws.parts_out = partitions;
        d->ws.impulses = nullptr;
        if (n_managers)
            hipLaunchKernelGGL(dy::k_outputs, dim3(grid_for(n_managers, dy::kBlock)), dim3(dy::kBlock), 0,
                               d->ctx->stream, d->ws);
        FYZZ_HIP_CHECK(hipGetLastError());
    });
}

int fyzz_hip_dy_prepare(fyzz_hip_dy* d, float dt, uint32_t n_bodies, fyzz_dy_body* bodies, uint32_t n_statics,
                        const fyzz_dy_static* statics, uint32_t n_managers, const fyzz_dy_manager* managers,
                        const fyzz_dy_patch* history, uint32_t n_history, fyzz_dy_patch* patches) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] {
        dy_prepare(d, dt, n_bodies, bodies, n_statics, statics, n_managers, managers, history, n_history, patches,
                   false);
    });
}

int fyzz_hip_dy_solve(fyzz_hip_dy* d) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] { dy_solve(d); });
}

int fyzz_hip_dy_integrate(fyzz_hip_dy* d, float* impulses, uint32_t* partitions) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] { dy_integrate(d, impulses, partitions); });
}

int fyzz_hip_dy_step(fyzz_hip_dy* d, float dt, uint32_t n_bodies, fyzz_dy_body* bodies, uint32_t n_statics,
                     const fyzz_dy_static* statics, uint32_t n_managers, const fyzz_dy_manager* managers,
                     const fyzz_dy_patch* history, uint32_t n_history, fyzz_dy_patch* patches, float* impulses,
                     uint32_t* partitions) {
    int rc = fyzz_hip_dy_prepare(d, dt, n_bodies, bodies, n_statics, statics, n_managers, managers, history,
                                 n_history, patches);
    if (rc == kOk) rc = fyzz_hip_dy_solve(d);
    if (rc == kOk) rc = fyzz_hip_dy_integrate(d, impulses, partitions);
    return rc;
}

int fyzz_hip_dy_set_tape(fyzz_hip_dy* d, int enabled) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] { dy_set_tape(d, enabled != 0); });
}

int fyzz_hip_dy_adjoint(fyzz_hip_dy* d, const float* adj_v_out, const float* adj_w_out, const float* adj_p_out,
                        float* adj_v_in, float* adj_w_in, float* adj_friction) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] { dy_adjoint(d, adj_v_out, adj_w_out, adj_p_out, adj_v_in, adj_w_in, adj_friction); });
}

int fyzz_hip_dy_friction_anchors(fyzz_hip_dy* d, fyzz_friction_anchors* out) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] {
        FYZZ_REQUIRE(out || d->ws.nm == 0, kInvalidArgument, "dy: null anchor output");
        if (!d->ws.nm) return;
        hipLaunchKernelGGL(dy::k_anchors, dim3(grid_for(d->ws.nm, dy::kBlock)), dim3(dy::kBlock), 0, d->ctx->stream,
                           d->ws, out);
        FYZZ_HIP_CHECK(hipGetLastError());
    });
}

int fyzz_hip_dy_status(fyzz_hip_dy* d, uint32_t* flags, uint32_t* n_partitions, uint32_t* rounds) {
    if (!d) return kInvalidArgument;
    return guarded(d->ctx, [&] {
        u32 f = 0, c[dy::kCtrWords];
        FYZZ_HIP_CHECK(hipMemcpyAsync(&f, d->flags.get(), sizeof f, hipMemcpyDeviceToHost, d->ctx->stream));
        FYZZ_HIP_CHECK(hipMemcpyAsync(c, d->ctr.get(), sizeof c, hipMemcpyDeviceToHost, d->ctx->stream));
        FYZZ_HIP_CHECK(hipStreamSynchronize(d->ctx->stream));
        if (flags) *flags = f;
        if (n_partitions) *n_partitions = c[dy::kNParts];
        if (rounds) *rounds = c[dy::kRounds];
        FYZZ_REQUIRE(!(f & FYZZ_DY_BAD_INPUT), kInvalidArgument, "dy: malformed manager record");
        FYZZ_REQUIRE(!(f & FYZZ_DY_OVERFLOW), kOverflow, "dy: partition or overflow-wave capacity exceeded");
        FYZZ_REQUIRE(!(f & FYZZ_DY_NONFINITE), kOverflow, "dy: non-finite solver value");
        FYZZ_REQUIRE(!(f & FYZZ_DY_LOGIC), kLogicError, "dy: manager outside the admitted class");
    });
}

}  // extern "C"
