// Single-world pipeline (the plain drop-in for one World::step) and its C ABI.
//
// Per step, on one HIP stream, no host synchronisation:
//   k_integrate        World::updateObjectStatus + applyExternalForce    (thread / body)
//   k_sap_*            sweep-and-prune broadphase over the body store (pe_sap.hpp): stable sort
//                      on aabb_min[axis], candidate runs, load-balanced sweep in the
//                      reference's (i, j) order, next axis
//   k_narrow           thread / pair: shape dispatch + 8-slot contact cache + depth sort
//   k_setup            thread / pair: solver rows (FrictionContactConstraint::initSequentialImpulse)
//   k_solve_small      small worlds (pe_world::one_workgroup): colouring and sweeps in one workgroup, on LDS; else
//   k_jp_*             the constraint graph: per body its pairs
//   k_solve_flow       one launch over the whole GPU: colouring, then the Gauss-Seidel sweeps in
//                      colour order as a data flow between the pairs, and the velocity sync
#include "pe_common.hpp"
#include "pe_device.hpp"
#include "pe_prims.hpp"
#include "pe_pipeline.hpp"
#include "pe_sap.hpp"
#include "pe_joints.hpp"
#include "pe_raycast.hpp"
#include "pe_host.hpp"
#include "../../include/pe_amd.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <vector>

static thread_local std::string g_err;
void pe_set_error(const std::string& msg) { g_err = msg; }

using namespace pe;

namespace {

constexpr int CLAIM_MAX = 12288;     // bodies up to which a caller may ask for the colouring in one workgroup

struct Dev {
    BodyView b;
    PairStore ps;           // pairs [pcap], contact slots and rows [pcap*8]
    SapView sap;            // the broadphase over the body store's AABBs (pairs to ps.pa / ps.pb)
    int32_t* shape_list;    // [pcap] pairs handed from k_narrow to k_narrow_shapes (from the front)
                            // and to k_narrow_sat (from the back)
    int32_t* comp_list;     // [pcap] pairs with a compound body (worlds with compounds; else null)
    // the solve's constraint graph: per dynamic body its active pairs, jp_deg[i] entries from jp_off[i]
    // on in jp_adj [2 pcap] (filled through the cursors jp_fill), per pair its colour and its place in
    // the colour, pairs per colour [pcap + 1]
    int32_t* jp_deg;
    int32_t* jp_off;
    int32_t* jp_fill;
    int2* jp_adj;        // (pair, claim priority)
    int32_t* jp_col;
    int32_t* jp_idx;
    uint64_t* jp_set;       // [pcap] heavy bodies: the set of colours their pairs have, body i's from jp_set_at[i] on
    int32_t* jp_set_at;
    int32_t* jp_ccount;
    int32_t* jp_hist;       // [FLOW_BINS][workgroups] pairs of each of the first colours per workgroup
    int32_t* jp_items;      // [pcap + 1] sweep: first item of each colour (colours beyond those kept in LDS)
    // the sweep (k_solve_flow): temp velocities with the number of updates made to them, and per place in
    // the solve order its pair and its place in its bodies' sequences of updates
    uint64_t* vel;          // [n][VELW]
    int4* q_pair;           // [pcap] pair, bodies A and B (top bit: kinematic), rows
    int4* q_seq;            // [pcap] A's updates before this pair's in an iteration, A's in an iteration; B's
    int32_t* order;         // [pcap]
    int32_t* act;           // [3*pcap] colouring work lists
    int32_t* color_start;   // [pcap+1]
    int32_t* claim;         // [n] claims of the colouring in one workgroup
    DevCounts* cnt;
    int32_t* rows_out;      // host memory: how full the last solve would fill one workgroup (null: not asked for)
    int pcap;
    float dt;
    float g[3];
    int iterations;
    // joints (World::addConstraint): definitions, per-step rows, sweep order grouped by colour
    const JointDef* joints;
    JointRow* jrows;
    const int32_t* jorder;   // [njoints] joint indices, colour by colour
    const int32_t* jcs;      // [njcol + 1] colour starts in jorder
    const int2* jseq;        // [njoints] joints of body A (B) in earlier joint colours
    const int32_t* jdeg;     // [n] joints of a dynamic body (null: no joints)
    int njoints, njcol;
    // sleeping, lifetimes, removals (World::updateObjectStatus) and collision reports
    StatusView st;
    int status_on;           // some body may sleep, end its lifetime or has been removed
    int report_on;           // some body reports its contacts
    float* events;           // [pcap][EVW] the last narrowphase's collision reports, by pair
    int32_t* ev_flag;        // [pcap] 1: pair p has a report
};

// Collision report of a pair (World::execCollisionCallbacks, world.cpp:129-192): bodies A and B (int
// bits), mean contact position, normalised sum of the normals, mean distance, mean relative velocity.
constexpr int EVW = 12;

// ------------------------------------------------------------------ stage 0: integrate
// World::updateObjectStatus (world.cpp:35-119) with zero sleep thresholds, then
// World::applyExternalForce (world.cpp:121-127), then SequentialImpulseSolver::setupSolver's
// clearTempVelocity (sequential_impulse_solver.cpp:17-20).
__global__ void k_integrate(Dev d) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < d.b.n; i += gridDim.x * blockDim.x) integrate_body(d.b, i, d.dt, d.g);
}
// The same with sleeping and lifetimes (world.cpp:85-117).
__global__ void k_integrate_status(Dev d) {
    const StatusView st = d.st;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < d.b.n; i += gridDim.x * blockDim.x)
        integrate_body<true>(d.b, i, d.dt, d.g, &st);
}

// DefaultRaycastSolver::performRaycast (default_raycast_solver.cpp:11-86), one workgroup per ray or RAYS_MAX
// of them over the world's bodies.  Skipped: removed bodies, ignore-collision bodies, the call's ignore
// set (sorted).  The reference walks the bodies in order and ends the query, reporting no hit, at the
// first mesh body whose AABB the unbounded ray misses, its result keeping the best hit of the bodies
// before it; so the first pass finds that body (the lowest such index), the second takes the nearest
// hit among the bodies before it, ties to the lowest index (the reference replaces a hit only by a
// strictly nearer one), as a minimum over (distance key, index).
// Bound by the passes over the bodies: every ray meets every body's record (72 bytes) and nearly all it meets
// are far off.  So a body is read once for several rays, and a box is only tested (some 150 instructions, a dozen
// divisions) for a ray that ray_may_hit_box lets through.  4096 rays against 10 000 boxes: 470 -> 152 us (with the mesh
// walk's stacks in the same kernel 239; the tests left gathered in LDS and done 64 at a time were slower, by their second
// reads and the LDS they take from the waves).
// MESH: the world has meshes.  Their walks take a stack row per thread (bvh_stack_row), so a workgroup has no more
// threads than there are rows; and the one thread that holds a terrain would walk it for each of its workgroup's rays
// in turn, so it has one ray (4096 rays over a terrain: 3.0 ms).
constexpr int RAY_IN = 7;    // start (3), direction (3), length
constexpr int RAY_OUT = 12;  // hit, body (int bits), distance, point (3), normal (3), pad
constexpr int RAYS_MAX = 4;
constexpr int ray_threads(bool mesh) { return mesh ? BVH_ROWS : 256; }
constexpr int ray_share(bool mesh) { return mesh ? 1 : RAYS_MAX; }
// Rays from which on a workgroup takes RAYS_MAX of them: with fewer a workgroup each fills the GPU better.
constexpr int RAYS_SHARED = 1024;
// Whether ray_box could report a hit of the ray, for a ray whose direction is no shorter than 0.5 (dir2 its squared
// length) and a box whose basis is orthonormal to 1e-3.  A hit has a point of the line in the box, up to what
// ray_hit_box adds: direction components below 1e-5 are raised to it (at a distance |m| + r the line is off by less
// than 4e-5 of that) and rounding (1e-6 of it).  The box is within r of its centre, so the line passes the
// centre within r and a margin of 2e-4 (|m| + r) and 1 % of r.  NaNs and infinities let through.
__device__ __forceinline__ bool ray_may_hit_box(f3 start, f3 dir, float dir2, f3 o, float r) {
    const f3 m = sub(o, start);
    const f3 c = cross(m, dir);
    const float bound = r * 1.01f + 2e-4f * (fabsf(m.x) + fabsf(m.y) + fabsf(m.z) + r);
    return !(dot(c, c) > bound * bound * dir2 * 1.001f);
}
__device__ __forceinline__ bool nearly_orthonormal(const m33& R) {
    const f3 a = col(R, 0), b = col(R, 1), c = col(R, 2);
    const float e = 1e-3f;
    return fabsf(dot(a, a) - 1.0f) < e && fabsf(dot(b, b) - 1.0f) < e && fabsf(dot(c, c) - 1.0f) < e && fabsf(dot(a, b)) < e &&
           fabsf(dot(a, c)) < e && fabsf(dot(b, c)) < e;
}
template <bool MESH>
__global__ void __launch_bounds__(ray_threads(MESH)) k_raycast(Dev d, const float* rays, int nrays, int per_group,
                                                               const int32_t* ignore, int nignore, float* out) {
    constexpr int RAY_THREADS = ray_threads(MESH);
    static_assert(!MESH || RAY_THREADS <= BVH_ROWS, "a stack row per thread");
    constexpr int RAYS = ray_share(MESH);
    __shared__ float s_ray[RAYS][8];                         // start, direction, length, squared length of direction
    __shared__ int s_abort[RAYS];
    // a thread's best of each ray: key, and distance, point, normal (of one ray in registers)
    __shared__ uint64_t s_best[RAYS][RAYS > 1 ? RAY_THREADS : 1];
    __shared__ float s_hit[RAYS][7][RAYS > 1 ? RAY_THREADS : 1];
    uint64_t best = ~0ull;
    float hit[7];
    const int tid = threadIdx.x;
    const int ray0 = blockIdx.x * per_group;
    const int nr = nrays - ray0 < per_group ? nrays - ray0 : per_group;
    if (tid < RAYS) s_abort[tid] = 0x7fffffff;
    if (tid < nr) {
        const float* r = rays + (size_t)(ray0 + tid) * RAY_IN;
#pragma unroll
        for (int k = 0; k < RAY_IN; k++) s_ray[tid][k] = r[k];
        s_ray[tid][7] = dot(f3{r[3], r[4], r[5]}, f3{r[3], r[4], r[5]});
    }
    if constexpr (RAYS > 1)
#pragma unroll
        for (int k = 0; k < RAYS; k++) s_best[k][tid] = ~0ull;
    __syncthreads();
    const int n = d.b.n;
    auto skipped = [&](int i) {
        if (d.status_on && (d.st.flags[i] & ST_REMOVED)) return true;
        if (d.b.at(F_SP + 3, i) == COLL_IGNORE) return true;
        int lo = 0, hi = nignore;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (ignore[mid] < i) lo = mid + 1; else hi = mid;
        }
        return lo < nignore && ignore[lo] == i;
    };
    if (MESH) {
        uint32_t open = (1u << nr) - 1u;   // rays whose query no body of this thread has ended yet
        for (int i = tid; i < n && open; i += RAY_THREADS) {
            if (d.b.iat(I_TYPE, i) < SHAPE_CONVEX || skipped(i)) continue;
            const f3 mn = ld3(d.b, F_AMIN, i), mx = ld3(d.b, F_AMAX, i);
            for (uint32_t m = open; m; m &= m - 1) {
                const int k = __ffs(m) - 1;
                const float* r = s_ray[k];
                float t;
                f3 hp, hn;
                if (ray_hit_box(f3{r[0], r[1], r[2]}, f3{r[3], r[4], r[5]}, mn, mx, t, hp, hn)) continue;
                atomicMin(&s_abort[k], i);
                open &= ~(1u << k);
            }
        }
    }
    __syncthreads();
    int lim = 0;
    for (int k = 0; k < nr; k++) lim = s_abort[k] > lim ? s_abort[k] : lim;
    if (lim > n) lim = n;
    for (int i = tid; i < lim; i += RAY_THREADS) {
        if (skipped(i)) continue;
        const int type = d.b.iat(I_TYPE, i);
        const f3 o = ld3(d.b, F_POS, i);
        const m33 R = ld9(d.b, F_ROT, i);
        const float sp[3] = {d.b.at(F_SP, i), d.b.at(F_SP + 1, i), d.b.at(F_SP + 2, i)};
        uint32_t rest = (1u << nr) - 1u;
        if (type == SHAPE_BOX && nearly_orthonormal(R)) {
            const float rad = 0.5f * sqrtf(sp[0] * sp[0] + sp[1] * sp[1] + sp[2] * sp[2]);
#pragma unroll
            for (int k = 0; k < RAYS; k++) {
                const float* r = s_ray[k];
                if (k < nr && r[7] >= 0.25f && !ray_may_hit_box(f3{r[0], r[1], r[2]}, f3{r[3], r[4], r[5]}, r[7], o, rad))
                    rest &= ~(1u << k);
            }
        }
        for (; rest; rest &= rest - 1) {
            const int q = __ffs(rest) - 1;
            if (i >= s_abort[q]) continue;
            const f3 start{s_ray[q][0], s_ray[q][1], s_ray[q][2]}, dir{s_ray[q][3], s_ray[q][4], s_ray[q][5]};
            const float len = s_ray[q][6];
            float t = 0.0f;
            f3 hp, hn;
            bool ret;
            if (type == SHAPE_BOX) ret = ray_box(start, dir, len, sp, R, o, t, hp, hn);
            else if (type == SHAPE_SPHERE) ret = ray_sphere(start, dir, len, sp[0], o, t, hp, hn);
            else if (type == SHAPE_CYLINDER) ret = ray_cylinder(start, dir, len, sp[0], sp[1], R, o, t, hp, hn);
            else if (type != SHAPE_COMPOUND) {
                ret = false;
                if constexpr (MESH) ret = ray_mesh(d.b.ms, __float_as_int(sp[0]), start, dir, len, R, o, t, hp, hn);
            } else {
                // each child in turn writes the same outputs, its hit or-ed in: the last child's distance and
                // point decide (default_raycast_solver.cpp:50-78)
                ret = false;
                const int2 kr = d.b.ms.krange[__float_as_int(sp[0])];
                for (int k = 0; k < kr.y; k++) {
                    float csp[3];
                    m33 Rc;
                    f3 pc;
                    const int ct = child_pose(d.b.ms, kr.x + k, R, o, csp, Rc, pc);
                    if (ct == SHAPE_BOX) ret |= ray_box(start, dir, len, csp, Rc, pc, t, hp, hn);
                    else if (ct == SHAPE_SPHERE) ret |= ray_sphere(start, dir, len, csp[0], pc, t, hp, hn);
                    else if (ct == SHAPE_CYLINDER) ret |= ray_cylinder(start, dir, len, csp[0], csp[1], Rc, pc, t, hp, hn);
                    else if constexpr (MESH) ret |= ray_mesh(d.b.ms, __float_as_int(csp[0]), start, dir, len, Rc, pc, t, hp, hn);
                }
            }
            if (ret && t <= len && t < REAL_MAX) {
                const uint64_t key = ((uint64_t)float_key(t + 0.0f) << 32) | (uint32_t)i;
                const float h[7] = {t, hp.x, hp.y, hp.z, hn.x, hn.y, hn.z};
                if constexpr (RAYS > 1) {
                    if (key < s_best[q][tid]) {
                        s_best[q][tid] = key;
#pragma unroll
                        for (int k = 0; k < 7; k++) s_hit[q][k][tid] = h[k];
                    }
                } else if (key < best) {
                    best = key;
#pragma unroll
                    for (int k = 0; k < 7; k++) hit[k] = h[k];
                }
            }
        }
    }
    __syncthreads();
    // a wave per ray: the least key, and what the thread that found it kept
    const int lane = tid & (WAVE - 1);
    auto least = [](uint64_t& win, int& at) {
#pragma unroll
        for (int m = 1; m < WAVE; m <<= 1) {
            const uint64_t w = (uint64_t)__shfl_xor((unsigned long long)win, m, WAVE);
            const int a = __shfl_xor(at, m, WAVE);
            if (w < win) { win = w; at = a; }
        }
    };
    auto result = [&](int q, uint64_t win, auto&& kept) {
        float e[RAY_OUT] = {0.0f, __int_as_float(-1), REAL_MAX};
        if (win != ~0ull) {
            e[0] = s_abort[q] == 0x7fffffff ? 1.0f : 0.0f;
            e[1] = __int_as_float((int)(uint32_t)win);
#pragma unroll
            for (int k = 0; k < 7; k++) e[2 + k] = kept(k);
        }
        st_rec<RAY_OUT / 4>(out + (size_t)(ray0 + q) * RAY_OUT, e);
    };
    if constexpr (RAYS > 1) {
        for (int q = tid / WAVE; q < nr; q += RAY_THREADS / WAVE) {
            uint64_t win = ~0ull;
            int at = 0;
            for (int k = lane; k < RAY_THREADS; k += WAVE)
                if (s_best[q][k] < win) { win = s_best[q][k]; at = k; }
            least(win, at);
            if (lane == 0) result(q, win, [&](int k) { return s_hit[q][k][at]; });
        }
    } else {
        static_assert(RAYS > 1 || RAY_THREADS == WAVE, "one wave");
        uint64_t win = best;
        int at = lane;
        least(win, at);
        if (win == ~0ull ? lane == 0 : lane == at) result(0, win, [&](int k) { return hit[k]; });
    }
}

// Recomputes AABBs and scales only (after pe_world_set_state); a removed body stays out of the sweep.
__global__ void k_aabb_only(Dev d) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < d.b.n; i += gridDim.x * blockDim.x) {
        if (d.status_on && (d.st.flags[i] & ST_REMOVED)) retire_body(d.b, i);
        else refresh_body(d.b, i);
    }
}

// World::removeRigidBody (world.cpp:223-231) of body i.
__global__ void k_remove_body(Dev d, int i) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    d.st.flags[i] |= ST_REMOVED;
    retire_body(d.b, i);
}

// SimpleNarrowPhase's neighbour counts (simple_narrow_phase.cpp:43-62): for a pair with contact
// points, each non-kinematic body counts a static neighbour when the other sleeps or is kinematic,
// a dynamic one otherwise (integer atomics: the counts do not depend on the order).
__global__ void k_neighbours(Dev d) {
    const int np = d.cnt->npairs;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        if (d.ps.npts[p] == 0) continue;
        const int a = d.ps.pa[p], b = d.ps.pb[p];
        const bool ka = d.b.iat(I_KIN, a) != 0, kb = d.b.iat(I_KIN, b) != 0;
        const bool sa = (d.st.flags[a] & ST_SLEEP) != 0, sb = (d.st.flags[b] & ST_SLEEP) != 0;
        if (!kb) atomicAdd((sa || ka) ? &d.st.scnt[b] : &d.st.dcnt[b], 1);
        if (!ka) atomicAdd((sb || kb) ? &d.st.scnt[a] : &d.st.dcnt[a], 1);
    }
}

// World::execCollisionCallbacks' arithmetic (world.cpp:131-151) for every pair with contact points
// whose bodies report: sums over the points in depth order, then the means and the normalised normal
// (Eigen's normalize: divide by the square root of the squared norm when it is positive).  Velocities
// are RigidBody::getLinearVelocityAtLocalPoint of the points' local positions (rigidbody.cpp:138-140)
// after gravity, as the callbacks see them.
__global__ void k_events(Dev d) {
    const int np = d.cnt->npairs;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        const int n = d.ps.npts[p];
        const int a = d.ps.pa[p], b = d.ps.pb[p];
        int flag = 0;
        if (n > 0 && (d.st.report[a] || d.st.report[b])) {
            flag = 1;
            f3 pos{0.0f, 0.0f, 0.0f}, nor{0.0f, 0.0f, 0.0f}, vel{0.0f, 0.0f, 0.0f};
            float depth = 0.0f;
            const f3 va = ld3(d.b, F_V, a), wa = ld3(d.b, F_W, a), vb = ld3(d.b, F_V, b), wb = ld3(d.b, F_W, b);
            for (int k = 0; k < n; k++) {
                const float* c = d.ps.cp + ((size_t)p * 8 + k) * CW;
                pos = add(pos, f3{c[C_WPOS], c[C_WPOS + 1], c[C_WPOS + 2]});
                nor = add(nor, f3{c[C_N], c[C_N + 1], c[C_N + 2]});
                depth += d.ps.cd[(size_t)p * 8 + k];
                vel = add(vel, add(va, cross(wa, f3{c[C_LA], c[C_LA + 1], c[C_LA + 2]})));
                vel = sub(vel, add(vb, cross(wb, f3{c[C_LB], c[C_LB + 1], c[C_LB + 2]})));
            }
            const float fn = (float)n;
            pos = f3{pos.x / fn, pos.y / fn, pos.z / fn};
            const float z = sqnorm3(nor);
            if (z > 0.0f) {
                const float r = sqrtf(z);
                nor = f3{nor.x / r, nor.y / r, nor.z / r};
            }
            depth = depth / fn;
            vel = f3{vel.x / fn, vel.y / fn, vel.z / fn};
            const float e[EVW] = {__int_as_float(a), __int_as_float(b), pos.x, pos.y, pos.z, nor.x, nor.y, nor.z,
                                  depth, vel.x, vel.y, vel.z};
            st_rec<EVW / 4>(d.events + (size_t)p * EVW, e);
        }
        d.ev_flag[p] = flag;
    }
}

// ------------------------------------------------------------------ stage 1: broadphase (pe_sap.hpp)

// ------------------------------------------------------------------ stage 2: narrowphase
// Box and sphere pairs here; pairs with a cylinder or a mesh are listed for k_narrow_sat (a wave
// each, pair_on_wave) or k_narrow_shapes (a thread each: a box or sphere with a cylinder).
__global__ void __launch_bounds__(128) k_narrow(Dev d) {
    const int np = d.cnt->npairs;
    const int prev = d.cnt->prev_npairs;
    if (blockIdx.x == 0 && threadIdx.x == 0) d.cnt->npoints = 0;   // summed by k_count_points
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        const bool simple = pair_is_simple(d.b, d.ps, p);
        const bool comp = !simple && (d.b.iat(I_TYPE, d.ps.pa[p]) == SHAPE_COMPOUND ||
                                      d.b.iat(I_TYPE, d.ps.pb[p]) == SHAPE_COMPOUND);
        const bool sat = !simple && !comp && pair_on_wave(d.b, d.ps, p);
        const int slot = wave_append(!simple && !sat && !comp, &d.cnt->nshape);
        const int sslot = wave_append(sat, &d.cnt->nsat);
        const int cslot = wave_append(comp && d.comp_list, &d.cnt->ncomp);
        if (simple) narrow_pair<false>(d.b, d.ps, p, prev);
        else if (sat) d.shape_list[d.pcap - 1 - sslot] = p;
        else if (comp) {
            if (d.comp_list) d.comp_list[cslot] = p;
            else { d.ps.npts[p] = 0; d.ps.swap[p] = 0; }   // no compound table: no algorithm
        } else d.shape_list[slot] = p;
    }
}
__global__ void __launch_bounds__(64) k_narrow_shapes(Dev d) {
    const int ns = d.cnt->nshape;
    const int prev = d.cnt->prev_npairs;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < ns; q += gridDim.x * blockDim.x)
        narrow_pair<true>(d.b, d.ps, d.shape_list[q], prev);
}
// One wave per listed wave pair (pair_on_wave: separating-axis pairs, a sphere or cylinder with a
// mesh).  Built for three waves per SIMD (at most 168 VGPRs; a little spilling): the 50k shape mix
// took 4.16 ms per step at two waves (248 VGPRs), 4.12 at three, 4.26 at four.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_narrow_sat(Dev d) {
    const int ns = d.cnt->nsat;
    const int prev = d.cnt->prev_npairs;
    const int nw = gridDim.x * (blockDim.x / WAVE);
    for (int q = blockIdx.x * (blockDim.x / WAVE) + (int)(threadIdx.x / WAVE); q < ns; q += nw)
        narrow_pair<true, WAVE>(d.b, d.ps, d.shape_list[d.pcap - 1 - q], prev);
}
// The pairs with a compound body, one thread each (64-thread workgroups: the contact cache and the
// BVH stacks of the separating-axis and mesh routines live in LDS rows of one lane each).
__global__ void __launch_bounds__(64) k_narrow_compound(Dev d) {
    const int nc = d.cnt->ncomp;
    const int prev = d.cnt->prev_npairs;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < nc; q += gridDim.x * blockDim.x)
        narrow_pair<true, 1, true>(d.b, d.ps, d.comp_list[q], prev);
}

// ------------------------------------------------------------------ stage 3: solver
// Words of a body's temp velocities in d.vel: component c of the linear (c) and angular (4 + c) one, each
// beside the number of updates made to the body in this solve (high half).  64 bytes per body.
constexpr int VELW = 8;
__device__ __forceinline__ uint64_t vel_word(float v, uint32_t seq) { return (uint64_t)seq << 32 | __float_as_uint(v); }

// Clears the solve's per-body and per-colour counters and sets every body's velocity words.
__global__ void k_solve_begin(Dev d) {
    const int n = d.b.n;
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x, gsz = gridDim.x * blockDim.x;
    for (int i = gtid; i < n; i += gsz) {
        d.jp_deg[i] = 0;
        d.jp_fill[i] = 0;
        const float* sb = d.b.sbr(i);
        ulonglong2* w = reinterpret_cast<ulonglong2*>(d.vel + (size_t)i * VELW);
        w[0] = make_ulonglong2(vel_word(sb[SB_TV], 0), vel_word(sb[SB_TV + 1], 0));
        w[1] = make_ulonglong2(vel_word(sb[SB_TV + 2], 0), 0);
        w[2] = make_ulonglong2(vel_word(sb[SB_TW], 0), vel_word(sb[SB_TW + 1], 0));
        w[3] = make_ulonglong2(vel_word(sb[SB_TW + 2], 0), 0);
    }
    for (int c = gtid; c < d.cnt->jp_ncol; c += gsz) d.jp_ccount[c] = 0;   // the colours the last solve counted
    if (gtid == 0) {
        d.cnt->nact = 0;
        d.cnt->nrows = 0;
        d.cnt->adj_total = 0;
        d.cnt->jp_rounds = 0;
        d.cnt->jp_heavy = 0;
        d.cnt->jp_maxdeg = 0;
        d.cnt->jp_words = 0;
        d.cnt->jp_fall = 0;
        d.cnt->fl_arrive = 0;
        d.cnt->fl_state = 0;
        d.cnt->fl_exit = 0;
    }
}

// SequentialImpulseSolver::setupSolver (sequential_impulse_solver.cpp:11-58), thread / pair: the solver
// rows, the list of the pairs to solve (contact points, not both bodies kinematic) and, for the colouring
// over the GPU (GRAPH), their dynamic bodies' degrees.
template <bool GRAPH> __global__ void k_setup(Dev d) {
    const int np = d.cnt->npairs;
    const int gsz = gridDim.x * blockDim.x;
    const int n_iter = (np + gsz - 1) / gsz;
    for (int it = 0; it < n_iter; it++) {
        const int p = it * gsz + blockIdx.x * blockDim.x + threadIdx.x;
        bool act = false;
        if (p < np && d.ps.npts[p] > 0) {
            setup_pair(d.b, d.ps, p, d.dt);
            const int a = d.ps.pa[p], c = d.ps.pb[p];
            const bool ka = d.b.iat(I_KIN, a) != 0, kc = d.b.iat(I_KIN, c) != 0;
            act = !(ka && kc);
            if (GRAPH && act) {
                d.jp_col[p] = -1;
                if (!ka) atomicAdd(&d.jp_deg[a], 1);
                if (!kc) atomicAdd(&d.jp_deg[c], 1);
            }
        }
        const int slot = wave_append(act, &d.cnt->nact);
        if (act) d.act[slot] = p;
    }
}
// Tells the host what a solve's contact points come to beyond those that one workgroup takes a colour at a time (it reads
// it at some later launch: pe_world::one_workgroup).
constexpr int SMALL_COLOUR_POINTS = 160;
__device__ __forceinline__ void report_rows(const Dev& d, int rows, int ncol) {
    if (d.rows_out) __hip_atomic_store(d.rows_out, rows - SMALL_COLOUR_POINTS * ncol, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// A body in more pairs than this is heavy: its pairs, which take different colours one after another, do not look at each
// other but at the set of their colours (jp_colour_heavy).
constexpr int JP_HEAVY = 32;
// Each body's range of the adjacency lists (the ranges' order does not matter); and syncTempVelocity
// (sequential_impulse_solver.cpp:71-80) of the removed bodies: the others' comes with their last update or, where
// there is none, changes nothing, but a removed body's temp velocities are not made anew from those the caller sets.
__global__ void k_jp_alloc(Dev d) {
    const int n = d.b.n;
    const int gsz = gridDim.x * blockDim.x;
    const int lane = threadIdx.x & (WAVE - 1);
    const int n_iter = (n + gsz - 1) / gsz;
    for (int it = 0; it < n_iter; it++) {
        const int i = it * gsz + blockIdx.x * blockDim.x + threadIdx.x;
        const int deg = i < n ? d.jp_deg[i] : 0;
        int incl = deg;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const int y = __shfl_up(incl, o, WAVE);
            if (lane >= o) incl += y;
        }
        int base = 0;
        if (lane == WAVE - 1 && incl > 0) base = (int)atomicAdd(&d.cnt->adj_total, (uint32_t)incl);
        base = __shfl(base, WAVE - 1, WAVE);
        if (i < n) {
            d.jp_off[i] = base + incl - deg;
            if (d.status_on && (d.st.flags[i] & ST_REMOVED) && !d.b.iat(I_KIN, i)) {
                const float* t = d.b.sbr(i);
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    d.b.at(F_V + k, i) = t[SB_TV + k];
                    d.b.at(F_W + k, i) = t[SB_TW + k];
                }
            }
        }
        const uint64_t heavy = __ballot(deg > JP_HEAVY);
        if (heavy) {
            int most = deg;
            for (int o = WAVE / 2; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, WAVE));
            if (lane == 0) {
                atomicAdd(&d.cnt->jp_heavy, (int)__popcll(heavy));
                atomicMax(&d.cnt->jp_maxdeg, most);
            }
        }
    }
}

// The list k_setup<false> adds to, emptied: k_solve_small leaves it so, a solve over the GPU does not.
__global__ void k_no_pairs(Dev d) { d.cnt->nact = 0; }

// BallJointConstraint / HingeJointConstraint / SliderJointConstraint::initSequentialImpulse, thread / joint
// (after the contacts' rows, as setupSolver initialises them, sequential_impulse_solver.cpp:49-51).
__global__ void k_joint_setup(Dev d) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < d.njoints; k += gridDim.x * blockDim.x)
        joint_setup(d.b, d.joints[k], d.jrows[k], d.dt);
}

// Sense-reversing barrier over all workgroups of a launch that are on the GPU together (every wait ends).  The last arrival resets the count and bumps the generation.
// It also orders memory across the grid: the workgroup's writes before the barrier are visible to
// every workgroup after it.  One thread per workgroup fences (a release fence before arriving, an
// acquire fence after the wait: the workgroup barriers around them carry the ordering to its other
// threads), and the arrival and the polling are relaxed atomics, so the caches are written back and
// invalidated once per workgroup and barrier, not once per wave or poll.
__device__ __forceinline__ void grid_barrier(uint32_t* count, uint32_t* gen, uint32_t nblocks) {
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t g = __hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");   // also keeps the load of g before the arrival
        if (__hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nblocks - 1) {
            __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);   // after the reset
        } else {
            while (__hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g) __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}

// Constraint-graph colouring over the whole GPU (Jones-Plassmann), the same colour classes as colour_pairs:
// colour_pairs builds each colour as the independent set its priority claims settle on, which is the
// greedy independent set in priority order of the pairs left (the candidate of lowest priority always
// holds its claims, and a pair joins exactly when no lower-priority neighbour joined); repeating that
// colour after colour gives each pair the first colour no lower-priority neighbour (a pair sharing a
// dynamic body) holds.  Here a pair takes that colour as soon as all its lower-priority neighbours
// have theirs, and the colours read are final when seen, so the result does not depend on timing.
__global__ void k_jp_fill(Dev d) {
    const int nact = d.cnt->nact;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nact; k += gridDim.x * blockDim.x) {
        const int p = d.act[k];
        const int a = d.ps.pa[p], c = d.ps.pb[p];
        const int2 e = make_int2(p, colour::prio(p, d.ps.npts[p]));
        if (!d.b.iat(I_KIN, a)) d.jp_adj[d.jp_off[a] + atomicAdd(&d.jp_fill[a], 1)] = e;
        if (!d.b.iat(I_KIN, c)) d.jp_adj[d.jp_off[c] + atomicAdd(&d.jp_fill[c], 1)] = e;
    }
}
__device__ __forceinline__ int jp_col_load(const int32_t* col, int q) {
    return __hip_atomic_load(&col[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The first colour not in used: a pair of no heavy body has at most 2 (JP_HEAVY - 1) neighbours, so one below 128 is
// free, and colours above that do not matter to it.
__device__ __forceinline__ int jp_first(const uint64_t (&used)[2]) {
    return ~used[0] != 0ull ? __ffsll((unsigned long long)~used[0]) - 1 : 63 + __ffsll((unsigned long long)~used[1]);
}
__device__ __forceinline__ void jp_use(uint64_t (&used)[2], int c) {
    if (c >= 0 && c < 64) used[0] |= 1ull << c;
    else if (c >= 64 && c < 128) used[1] |= 1ull << (c & 63);
}
// Pair p's (of no heavy body) first-fit colour if every lower-priority neighbour is coloured, else -1.  The adjacency
// entries and their colours are loaded eight at a time (independent loads in flight together: a
// neighbour scan is a chain of L2 round trips otherwise).
constexpr int JP_BATCH = 8;
__device__ __forceinline__ int jp_try(const Dev& d, int p) {
    const int pr = colour::prio(p, d.ps.npts[p]);
    const int body[2] = {d.ps.pa[p], d.ps.pb[p]};
    uint64_t used[2] = {0, 0};
    for (int s = 0; s < 2; s++) {
        const int x = body[s];
        if (d.b.iat(I_KIN, x)) continue;
        const int k0 = d.jp_off[x], k1 = k0 + d.jp_deg[x];
        for (int k = k0; k < k1; k += JP_BATCH) {
            int2 q[JP_BATCH];
            int cq[JP_BATCH];
#pragma unroll
            for (int j = 0; j < JP_BATCH; j++) q[j] = k + j < k1 ? d.jp_adj[k + j] : make_int2(p, pr);
#pragma unroll
            for (int j = 0; j < JP_BATCH; j++) {
                const bool lower = q[j].x != p && q[j].y < pr;
                cq[j] = lower ? jp_col_load(d.jp_col, q[j].x) : -2;
            }
            int wait = 0;
#pragma unroll
            for (int j = 0; j < JP_BATCH; j++) {
                wait |= cq[j] == -1;
                jp_use(used, cq[j]);
            }
            if (wait) return -1;
        }
    }
    return jp_first(used);
}
// The lower-priority neighbours of pair p at its bodies that are not heavy to list[JP_KEEP]; their number, or -1 if they are
// more.
constexpr int JP_KEEP = 32;
__device__ __forceinline__ int jp_lower(const Dev& d, int p, int* list) {
    const int pr = colour::prio(p, d.ps.npts[p]);
    const int body[2] = {d.ps.pa[p], d.ps.pb[p]};
    int m = 0;
    for (int s = 0; s < 2; s++) {
        const int x = body[s];
        if (d.b.iat(I_KIN, x)) continue;
        const int k0 = d.jp_off[x], k1 = k0 + d.jp_deg[x];
        if (k1 - k0 > JP_HEAVY) continue;
        for (int k = k0; k < k1; k += JP_BATCH) {
            int2 q[JP_BATCH];
#pragma unroll
            for (int j = 0; j < JP_BATCH; j++) q[j] = k + j < k1 ? d.jp_adj[k + j] : make_int2(p, pr);
#pragma unroll
            for (int j = 0; j < JP_BATCH; j++) {
                if (q[j].x == p || q[j].y >= pr) continue;
                if (m == JP_KEEP) return -1;
                list[m++] = q[j].x;
            }
        }
    }
    return m;
}
// Drops the coloured pairs of list[n] and enters their colours; the number left.
__device__ __forceinline__ int jp_poll(const Dev& d, int* list, int n, uint64_t (&used)[2]) {
    int m = 0;
    for (int k = 0; k < n; k += JP_BATCH) {
        int q[JP_BATCH], cq[JP_BATCH];
#pragma unroll
        for (int j = 0; j < JP_BATCH; j++) q[j] = k + j < n ? list[k + j] : -1;
#pragma unroll
        for (int j = 0; j < JP_BATCH; j++) cq[j] = q[j] >= 0 ? jp_col_load(d.jp_col, q[j]) : 0;
#pragma unroll
        for (int j = 0; j < JP_BATCH; j++) {
            if (q[j] < 0) continue;
            if (cq[j] < 0) list[m++] = q[j];   // at or before the entry read
            else jp_use(used, cq[j]);
        }
    }
    return m;
}
// Pairs of body x (not p) in a colour before c: p's place in x's sequence of updates.  sets: heavy bodies have the sets of
// their colours.
__device__ __forceinline__ int jp_rank(const Dev& d, int x, int p, int c, bool sets) {
    const int k0 = d.jp_off[x], k1 = k0 + d.jp_deg[x];
    int r = 0;
    if (sets && k1 - k0 > JP_HEAVY) {
        const uint64_t* set = d.jp_set + d.jp_set_at[x];
        for (int w = 0; w < c >> 6; w++) r += (int)__popcll(set[w]);
        return r + (int)__popcll(set[c >> 6] & ((1ull << (c & 63)) - 1ull));
    }
    for (int k = k0; k < k1; k += JP_BATCH) {
        int q[JP_BATCH];
#pragma unroll
        for (int j = 0; j < JP_BATCH; j++) q[j] = k + j < k1 ? d.jp_adj[k + j].x : p;
#pragma unroll
        for (int j = 0; j < JP_BATCH; j++) r += q[j] != p && jp_col_load(d.jp_col, q[j]) < c;
    }
    return r;
}

// ---- worlds with heavy bodies
// A heavy body's pairs are coloured in the order of their priorities, and their colours differ: so the pair with r
// of them before it is next when the set of their colours, which each adds its own to, has r members, and
// it then has those colours at hand.  A try reads that set (a word per 64 pairs) where a scan of the body's pairs reads
// all of them, twice.  2 500 bodies of which 40 / 150 / 500 lie on one plate: 0.72 / 2.2 / 6.9 ms a step, most of it
// the sweeps' 40 / 140 / 460 colours (with scans 0.89 ms for 40; every pair by claims in one workgroup 5.5 / 20.0).
struct JpHeavy {
    uint64_t* set;   // the body's set (null: it is not heavy)
    int words, rank;
    int lo;          // leading words seen full: they stay so
};
// Words of the set of a body with deg pairs: a colour is at most the number of the pair's other neighbours.
__device__ __forceinline__ int jp_set_words(int deg, int maxdeg) { return (deg + maxdeg) / 64 + 1; }
// Hands out the sets, empty.
__device__ __forceinline__ void jp_set_alloc(const Dev& d, int gtid, int gsz) {
    for (int i = gtid; i < d.b.n; i += gsz) {
        if (d.jp_deg[i] <= JP_HEAVY) continue;
        const int m = jp_set_words(d.jp_deg[i], d.cnt->jp_maxdeg);
        const uint32_t at = atomicAdd(&d.cnt->jp_words, (uint32_t)m);
        if ((uint64_t)at + m > (uint64_t)d.pcap) {
            d.cnt->jp_fall = 1;
            return;
        }
        d.jp_set_at[i] = (int)at;
        for (int w = 0; w < m; w++) d.jp_set[at + w] = 0;
    }
}
__device__ __forceinline__ uint64_t jp_set_load(const uint64_t* w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool jp_is_heavy(const Dev& d, int x) { return !d.b.iat(I_KIN, x) && d.jp_deg[x] > JP_HEAVY; }
// The set of body x and pair p's place among its pairs (rank < 0: counted here).
__device__ __forceinline__ JpHeavy jp_heavy(const Dev& d, int x, int p, int rank) {
    JpHeavy h{nullptr, 0, 0, 0};
    if (!jp_is_heavy(d, x)) return h;
    h.set = d.jp_set + d.jp_set_at[x];
    h.words = jp_set_words(d.jp_deg[x], d.cnt->jp_maxdeg);
    h.rank = rank;
    if (rank >= 0) return h;
    const int pr = colour::prio(p, d.ps.npts[p]);
    h.rank = 0;
    const int k0 = d.jp_off[x], k1 = k0 + d.jp_deg[x];
    for (int k = k0; k < k1; k += 2 * JP_BATCH) {
        int q[2 * JP_BATCH];
#pragma unroll
        for (int j = 0; j < 2 * JP_BATCH; j++) q[j] = k + j < k1 ? d.jp_adj[k + j].y : pr;
#pragma unroll
        for (int j = 0; j < 2 * JP_BATCH; j++) h.rank += q[j] < pr;
    }
    return h;
}
// How many pairs of a heavy body are still to be coloured before this one.
__device__ __forceinline__ int jp_heavy_missing(const Dev& d, JpHeavy& h) {
    if (!h.set) return 0;
    // with one heavy body a colour is at most its pair's place and what a body that is not heavy adds
    const int hi = d.cnt->jp_heavy == 1 ? min(h.words, (h.rank + JP_HEAVY) / 64 + 1) : h.words;
    int sum = 64 * h.lo;
    bool lead = true;
    for (int w = h.lo; w < hi; w += 4) {
        uint64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = w + u < hi ? jp_set_load(h.set + w + u) : 0ull;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            sum += (int)__popcll(v[u]);
            lead = lead && ~v[u] == 0ull;
            h.lo += lead;
        }
    }
    return h.rank - sum;
}
// The first colour in neither set nor among list[n], which is entered in the sets; -1: none (not reached).
__device__ __forceinline__ int jp_heavy_take(const JpHeavy& a, const JpHeavy& b, const int* list, int n) {
    const int words = !a.set ? b.words : !b.set ? a.words : min(a.words, b.words);
    for (int w = max(a.lo, b.lo); w < words; w++) {
        uint64_t used = 0;
        if (a.set) used |= jp_set_load(a.set + w);
        if (b.set) used |= jp_set_load(b.set + w);
        for (int k = 0; k < n; k++)
            if (list[k] >> 6 == w) used |= 1ull << (list[k] & 63);
        if (~used == 0ull) continue;
        const int bit = __ffsll((unsigned long long)~used) - 1;
        if (a.set) __hip_atomic_fetch_or(a.set + w, 1ull << bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (b.set) __hip_atomic_fetch_or(b.set + w, 1ull << bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return 64 * w + bit;
    }
    return -1;
}
// Puts the colours that are there in the place of the pairs in list whose bits are set in miss; the bits left.
__device__ __forceinline__ uint32_t jp_poll_keep(const Dev& d, int* list, uint32_t miss) {
    for (uint32_t todo = miss; todo;) {
        int at[4], c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            at[u] = todo ? __ffs(todo) - 1 : -1;
            todo &= todo - 1;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) c[u] = at[u] >= 0 ? jp_col_load(d.jp_col, list[at[u]]) : -1;
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (c[u] >= 0) {
                list[at[u]] = c[u];
                miss &= ~(1u << at[u]);
            }
    }
    return miss;
}
// Colours every pair, as the loops of k_solve_flow do where no body is heavy; mine: the thread's JP_KEEP words of LDS.
// The number of tries, negated where pairs of this thread were given up.
__device__ __forceinline__ int jp_colour_heavy(const Dev& d, int nact, int gtid, int gsz, int* mine, int spins) {
    int tries = 0;
    bool left = true;
    if (nact <= gsz) {
        const int p = gtid < nact ? d.act[gtid] : -1;
        JpHeavy a{nullptr, 0, 0, 0}, b = a;
        int n = 0;
        if (p >= 0) {
            a = jp_heavy(d, d.ps.pa[p], p, -1);
            b = jp_heavy(d, d.ps.pb[p], p, -1);
            n = jp_lower(d, p, mine);
        }
        const bool heavy = a.set || b.set;
        uint32_t miss = heavy ? (uint32_t)((1ull << n) - 1ull) : 0u;   // (then n < JP_HEAVY)
        uint64_t used[2] = {0, 0};
        left = p >= 0;
        int skip = 0;   // rounds until the next look: a pair whose turn is far off only loads the fabric
        while (__any(left) && tries < spins) {
            const bool look = left && skip == 0;
            if (left && skip > 0) skip--;
            if (look) {
                int c = -1;
                if (heavy) {
                    if (miss) miss = jp_poll_keep(d, mine, miss);
                    const int before = max(jp_heavy_missing(d, a), jp_heavy_missing(d, b));
                    if (before == 0 && miss == 0) c = jp_heavy_take(a, b, mine, n);
                    skip = before > 4 ? min(before >> 2, 1024) : 0;
                } else if (n < 0) {
                    c = jp_try(d, p);
                } else {
                    n = jp_poll(d, mine, n, used);
                    if (n == 0) c = jp_first(used);
                }
                if (c >= 0) {
                    __hip_atomic_store(&d.jp_col[p], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    left = false;
                }
            }
            if (__any(look)) tries++;
            else __builtin_amdgcn_s_sleep(16);
        }
    } else {
        // several pairs per thread: their places wait in q_seq, which is only made after the colouring
        for (int k = gtid; k < nact; k += gsz) {
            const int p = d.act[k];
            d.q_seq[k] = make_int4(jp_heavy(d, d.ps.pa[p], p, -1).rank, jp_heavy(d, d.ps.pb[p], p, -1).rank, 0, 0);
        }
        for (; __any(left) && tries < spins; tries++) {
            left = false;
            for (int k = gtid; k < nact; k += gsz) {
                const int p = d.act[k];
                if (jp_col_load(d.jp_col, p) >= 0) continue;
                const int4 r = d.q_seq[k];
                JpHeavy a = jp_heavy(d, d.ps.pa[p], p, r.x), b = jp_heavy(d, d.ps.pb[p], p, r.y);
                int c = -1;
                if (!a.set && !b.set) {
                    c = jp_try(d, p);
                } else if (jp_heavy_missing(d, a) == 0 && jp_heavy_missing(d, b) == 0) {
                    const int n = jp_lower(d, p, mine);
                    if (jp_poll_keep(d, mine, (uint32_t)((1ull << n) - 1ull)) == 0) c = jp_heavy_take(a, b, mine, n);
                }
                if (c >= 0) __hip_atomic_store(&d.jp_col[p], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else left = true;
            }
        }
    }
    return left ? -tries : tries;
}

// Colouring and Gauss-Seidel sweeps (SequentialImpulseSolver::solve, sequential_impulse_solver.cpp:60-81)
// over the whole GPU in one launch whose workgroups run at the same time (flow_together), so every wait ends.
//
// The sweeps run as a data flow instead of colour by colour between grid barriers.  The colour order fixes
// for every body the sequence of the pairs (then joints) that update it in an iteration, so a pair only
// has to wait until its two bodies have had the updates before its own: each word of a body's temp
// velocities carries the number of updates made (d.vel), a pair polls its bodies' words until they show
// the number it expects, solves its rows and writes the words back with that number plus one.  The one pair
// that expects a number is the only reader of that version and the next writer, so nothing else orders the
// threads, and the words are relaxed device-scope atomics without fences.  Every body sees the updates
// of the colour-by-colour sweep in the same order: the same bits.
// What bounds it is the chain of dependent updates: iterations x colours x (the rows of a pair, 0.27 us each,
// + about 0.9 us until the next pair of the body has seen the words: a store becomes visible to a polling
// load in 0.5 to 0.67 us, on the same XCD or another).  Colour by colour, each pass also paid a grid
// barrier (2 us at 32 workgroups, 4 to 7 at 256: atomics on one word) and waited for the slowest pair of the
// colour.  10 000 boxes at rest (13 colours, 17 000 pairs, 36 000 points, 10 iterations): colouring 305 ->
// 75 us, sweeps 850 -> 260 us.
//
// A wave works on items of 16 pairs of one colour, a quad of lanes per pair (quad_solve_row), or on 16
// joints; it takes its items (wave, wave + waves, ...) in the order of iterations and colours.  The first
// unfinished item in that order is therefore always at the head of its wave with everything it waits for
// finished.  With an item per wave or less the rows stay in registers throughout.
constexpr int FLOW_THREADS = 512;
constexpr int FLOW_COLORS = 1024;       // colours whose starts every workgroup keeps in LDS
constexpr int FLOW_BINS = 64;           // colours whose pairs every workgroup counts in LDS
constexpr int FLOW_PAIRS = WAVE / 4;    // pairs per item
constexpr int FLOW_JOINTS = 16;         // joints per wave at a time
constexpr int FLOW_SPINS = 1 << 21;     // polls after which a wait is given up (seconds: a fault of this program)

__device__ __forceinline__ uint64_t vel_load(const uint64_t* w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void vel_store(uint64_t* w, float v, uint32_t seq) {
    __hip_atomic_store(w, vel_word(v, seq), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Pause between two polls of a wave that is not ready: by how many updates the farthest of its pairs still
// waits for (polls of waves whose turn is far off only load the fabric: with short pauses throughout the
// sweeps of 10 000 boxes at rest took 283 us, with these 260).
__device__ __forceinline__ void flow_pause(bool waits, uint32_t dist) {
    if (!__any(waits && dist > 1)) __builtin_amdgcn_s_sleep(1);
    else if (!__any(waits && dist > 4)) __builtin_amdgcn_s_sleep(24);
    else __builtin_amdgcn_s_sleep(100);
}
// A quad's pair.  wa, wb: the lane's words of the bodies' linear velocities (the angular ones 4 on).
struct FlowPair {
    int n, ia, ib;
    int4 seq;
    float* rows;
    uint64_t *wa, *wb;
    QuadBody A, B;
};
// Place q of the solve order (an empty pair beyond the colour's end).
__device__ __forceinline__ void flow_load(const Dev& d, int q, bool valid, int c, FlowPair& f) {
    int4 pr = make_int4(0, 1 << 31, 1 << 31, 0);
    f.seq = make_int4(0, 0, 0, 0);
    if (valid) {
        pr = d.q_pair[q];
        f.seq = d.q_seq[q];
    }
    f.n = pr.w;
    f.ia = pr.y & 0x7fffffff;
    f.ib = pr.z & 0x7fffffff;
    f.rows = d.ps.rows + (size_t)pr.x * 8 * RW;
    f.wa = d.vel + (size_t)f.ia * VELW + c;
    f.wb = d.vel + (size_t)f.ib * VELW + c;
    quad_load_body(d.b.sbr(f.ia), c, pr.y < 0, f.A);
    quad_load_body(d.b.sbr(f.ib), c, pr.z < 0, f.B);
}
__device__ __forceinline__ void flow_rows(const FlowPair& f, int k0, int c, QuadRow (&r)[4]) {
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (k0 + u < f.n) quad_load_row(f.rows + (size_t)(k0 + u) * RW, c, r[u]);
}
__device__ __forceinline__ void flow_store_acc(const FlowPair& f, int k0, int c, const QuadRow (&r)[4]) {
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (k0 + u < f.n) f.rows[(size_t)(k0 + u) * RW + R_LN + c] = r[u].acc;
}
// Polls the lane's words of a body that is to have had e updates: whether it has, its velocity words into
// q, and how many updates are missing.
__device__ __forceinline__ void flow_take(QuadBody& q, uint64_t v, uint64_t w, uint32_t e, bool& ready, uint32_t& dist) {
    const uint32_t s0 = (uint32_t)(v >> 32), s1 = (uint32_t)(w >> 32);
    ready = s0 == e && s1 == e;
    dist = max(dist, e - s0);
    q.tv = __uint_as_float((uint32_t)v);
    q.tw = __uint_as_float((uint32_t)w);
}
// Solves the pair's rows from r (its first four) and the row store (the rest, their impulses put back),
// then hands the bodies on.  last_a (last_b): the update after which A (B) is solved, its velocities
// then going to the body store (syncTempVelocity, sequential_impulse_solver.cpp:71-80).
__device__ __forceinline__ void flow_solve(const Dev& d, FlowPair& f, int c, bool first, bool own, QuadRow (&r)[4], uint32_t ea,
                                           uint32_t eb, uint32_t last_a, uint32_t last_b) {
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (u < f.n) quad_solve_row(r[u], first, f.A, f.B);
    for (int k = 4; k < f.n; k++) {
        QuadRow x;
        quad_load_row(f.rows + (size_t)k * RW, c, x);
        quad_solve_row(x, first, f.A, f.B);
        if (own) f.rows[(size_t)k * RW + R_LN + c] = x.acc;
    }
    auto hand_on = [&](const QuadBody& q, int i, uint64_t* w, uint32_t e, uint32_t last) {
        if (q.kin) return;
        vel_store(w, q.tv, e + 1);
        vel_store(w + 4, q.tw, e + 1);
        if (e + 1 == last) {
            d.b.at(F_V + c, i) = q.tv;
            d.b.at(F_W + c, i) = q.tw;
            float* sb = d.b.sbr(i);
            sb[SB_TV + c] = q.tv;
            sb[SB_TW + c] = q.tw;
        }
    };
    if (own) {
        hand_on(f.A, f.ia, f.wa, ea, last_a);
        hand_on(f.B, f.ib, f.wb, eb, last_b);
    }
}
// The joints of lanes j0, j0 + nl, ... of jorder, over all iterations, a joint per lane at a time: each waits for
// its bodies' contacts and earlier joints of the iteration.  False if given up.
__device__ __forceinline__ bool flow_joints(const Dev& d, int j0, int nl) {
    int at = j0, it = 0;
    bool live = at < d.njoints && d.iterations > 0, fresh = true;
    JointDef j{};
    SolvBody S[2];
    int body[2] = {0, 0}, k = 0;
    uint32_t e[2] = {0, 0}, last[2] = {0, 0};
    bool ready[2] = {false, false};
    for (int spin = 0; __any(live); spin++) {
        if (spin == FLOW_SPINS) return false;
        if (live && fresh) {
            fresh = false;
            k = d.jorder[at];
            j = d.joints[k];
            const int2 seq = d.jseq[k];
            body[0] = j.a;
            body[1] = j.b;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                S[s] = load_solv(d.b, body[s]);
                S[s].tv = S[s].tw = f3{0.0f, 0.0f, 0.0f};   // a kinematic body's stay so
                ready[s] = S[s].kin;
                const int deg = d.jp_deg[body[s]], tot = deg + d.jdeg[body[s]];
                e[s] = (uint32_t)(it * tot + deg + (s == 0 ? seq.x : seq.y));
                last[s] = (uint32_t)(d.iterations * tot);
            }
        }
        uint32_t dist = 0;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            if (!live || ready[s]) continue;
            const uint64_t* w = d.vel + (size_t)body[s] * VELW;
            uint64_t x[6];
#pragma unroll
            for (int m = 0; m < 6; m++) x[m] = vel_load(w + (m < 3 ? m : m + 1));
            bool ok = true;
#pragma unroll
            for (int m = 0; m < 6; m++) ok = ok && (uint32_t)(x[m] >> 32) == e[s];
            dist = max(dist, e[s] - (uint32_t)(x[0] >> 32));
            ready[s] = ok;
            auto val = [&](int m) { return __uint_as_float((uint32_t)x[m]); };
            S[s].tv = f3{val(0), val(1), val(2)};
            S[s].tw = f3{val(3), val(4), val(5)};
        }
        const bool go = live && ready[0] && ready[1];
        if (go) {
            joint_solve(j, d.jrows[k], S[0], S[1]);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                if (S[s].kin) continue;
                uint64_t* w = d.vel + (size_t)body[s] * VELW;
                const float v[6] = {S[s].tv.x, S[s].tv.y, S[s].tv.z, S[s].tw.x, S[s].tw.y, S[s].tw.z};
#pragma unroll
                for (int m = 0; m < 6; m++) vel_store(w + (m < 3 ? m : m + 1), v[m], e[s] + 1);
                if (e[s] + 1 == last[s]) {
                    float* sb = d.b.sbr(body[s]);
#pragma unroll
                    for (int m = 0; m < 6; m++) {
                        d.b.at((m < 3 ? F_V : F_W - 3) + m, body[s]) = v[m];
                        sb[SB_TV + m] = v[m];   // SB_TW follows SB_TV
                    }
                }
            }
            fresh = true;
            at += nl;
            if (at >= d.njoints) {
                at = j0;
                live = ++it < d.iterations;
            }
        }
        if (__any(go)) spin = 0;
        else flow_pause(live, dist);
    }
    return true;
}

// The whole solve by one workgroup of FLOW_THREADS on the records in global memory, a pair per thread, the claims in
// LDS or (n bodies, any n) in memory: where a small world's pairs or colours outgrow its workgroup's
// LDS, and where the workgroups of k_solve_flow could not all be had at once.
template <bool LDS_CLAIM>
__device__ __forceinline__ void solve_alone(const Dev& d, int nact, int* claim) {
    __shared__ int wsum[FLOW_THREADS / WAVE + 1];
    const int tid = threadIdx.x;
    for (int i = tid; i < d.b.n; i += FLOW_THREADS) claim_set<LDS_CLAIM>(claim, i, colour::FREE);
    claim_sync<LDS_CLAIM>();
    int* bufs[3] = {d.act, d.act + d.pcap, d.act + 2 * (size_t)d.pcap};
    const int ncol = colour_pairs<LDS_CLAIM>(d.b, d.ps, bufs, nact, d.order, d.color_start, claim, 0, 0, wsum);
    if (tid == 0) {
        d.cnt->ncolors = ncol;
        d.cnt->nordered = d.color_start[ncol];
        d.cnt->jp_rounds = 0;
    }
    for (int it = 0; it < d.iterations; it++) {
        for (int c = 0; c < ncol; c++) {
            for (int q = d.color_start[c] + tid; q < d.color_start[c + 1]; q += FLOW_THREADS) iterate_pair(d.b, d.ps, d.order[q]);
            __syncthreads();
        }
        // the joints after the contacts, colour by colour (sequential_impulse_solver.cpp:66-68)
        for (int c = 0; c < d.njcol; c++) {
            for (int q = d.jcs[c] + tid; q < d.jcs[c + 1]; q += FLOW_THREADS) {
                const int k = d.jorder[q];
                const JointDef j = d.joints[k];
                SolvBody A = load_solv(d.b, j.a), B = load_solv(d.b, j.b);
                joint_solve(j, d.jrows[k], A, B);
                for (int s = 0; s < 2; s++) {
                    const SolvBody& S = s == 0 ? A : B;
                    if (S.kin) continue;
                    float* o = d.b.sbr(s == 0 ? j.a : j.b);
                    o[SB_TV] = S.tv.x; o[SB_TV + 1] = S.tv.y; o[SB_TV + 2] = S.tv.z;
                    o[SB_TW] = S.tw.x; o[SB_TW + 1] = S.tw.y; o[SB_TW + 2] = S.tw.z;
                }
            }
            __syncthreads();
        }
    }
    for (int i = tid; i < d.b.n; i += FLOW_THREADS) {
        if (d.b.iat(I_KIN, i)) continue;
        const float* o = d.b.sbr(i);
        st3(d.b, F_V, i, f3{o[SB_TV], o[SB_TV + 1], o[SB_TV + 2]});
        st3(d.b, F_W, i, f3{o[SB_TW], o[SB_TW + 1], o[SB_TW + 2]});
    }
}

// Whether all workgroups of the launch are on the GPU at once, which their waits on each other need.  The launch is
// an ordinary one (a cooperative one changes queues: 28 us a step, and with several worlds' streams up to
// 170), its grid no more than the GPU holds; but other launches may hold the GPU at the time.  The
// last workgroup to start says so to the others; one that has waited `patience` (ticks of 10 ns) calls the
// launch off instead, and whichever comes first holds for all.  Called off, the workgroups leave
// as they come, nothing done, and the last of them, now alone, solves by itself.
constexpr uint32_t FLOW_GO = 1, FLOW_OFF = 2;
__device__ __forceinline__ bool flow_together(const Dev& d, uint64_t patience, int* alone) {
    __shared__ uint32_t s_state;
    if (threadIdx.x == 0) {
        DevCounts* c = d.cnt;
        uint32_t st = 0;
        if (__hip_atomic_fetch_add(&c->fl_arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
            uint32_t none = 0;
            __hip_atomic_compare_exchange_strong(&c->fl_state, &none, FLOW_GO, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint64_t t0 = wall_clock64();
        while ((st = __hip_atomic_load(&c->fl_state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
            if (wall_clock64() - t0 >= patience) {
                uint32_t none = 0;
                __hip_atomic_compare_exchange_strong(&c->fl_state, &none, FLOW_OFF, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            } else {
                __builtin_amdgcn_s_sleep(1);
            }
        }
        s_state = st;
        if (st == FLOW_OFF)
            *alone = __hip_atomic_fetch_add(&c->fl_exit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    }
    __syncthreads();
    return s_state == FLOW_GO;
}

// claims: the colouring runs in workgroup 0 (colour_pairs), as it does where the heavy bodies' sets outgrow their memory.
__global__ void __launch_bounds__(FLOW_THREADS) k_solve_flow(Dev d, int claims, uint64_t patience) {
    __shared__ int s_cs[FLOW_COLORS + 1], s_is[FLOW_COLORS + 1], s_ncol;
    __shared__ int s_hist[FLOW_BINS];
    __shared__ int s_low[FLOW_THREADS][JP_KEEP + 1];   // rows of odd length: distinct banks
    const int nact = d.cnt->nact;
    const int tid = threadIdx.x, gtid = blockIdx.x * blockDim.x + tid, gsz = gridDim.x * blockDim.x;
    if (!flow_together(d, patience, &s_ncol)) {
        if (s_ncol) solve_alone<false>(d, nact, d.claim);
        return;
    }
    if (tid < FLOW_BINS) s_hist[tid] = 0;
    auto stalled = [&]() { atomicOr(&d.cnt->overflow, OVF_STALL); };
    // The same for every workgroup: heavy bodies have their sets; the colouring is done by claims.  Few worlds have any: said
    // so, their code lies out of the way (else the sweeps of 10 000 boxes at rest take 359 us instead of 354).
    bool sets = !claims && d.cnt->jp_heavy > 0, coloured = claims;
    if (__builtin_expect(sets, 0)) {
        jp_set_alloc(d, gtid, gsz);
        grid_barrier(&d.cnt->bar_count, &d.cnt->bar_gen, gridDim.x);
        coloured = d.cnt->jp_fall != 0;
        sets = !coloured;
    }
    if (!coloured) {
        // Every thread tries its pairs until all have their colours: the uncoloured pair of lowest priority
        // gets its colour whenever it is tried, so the loops end.  With a pair per thread or less, a thread
        // scans its bodies' lists once and keeps the lower-priority neighbours in LDS; a try then reads only
        // the colours still missing, in flight together.
        int tries = 0;
        bool left = true;
        if (__builtin_expect(sets, 0)) {
            tries = jp_colour_heavy(d, nact, gtid, gsz, s_low[tid], FLOW_SPINS);
            left = tries < 0;
            tries = abs(tries);
        } else if (nact <= gsz) {
            const int p = gtid < nact ? d.act[gtid] : -1;
            int* mine = s_low[tid];
            int nlow = p >= 0 ? jp_lower(d, p, mine) : 0;   // neighbours whose colours are missing (-1: too many to keep)
            uint64_t used[2] = {0, 0};   // colours the others hold
            left = p >= 0;
            for (; __any(left) && tries < FLOW_SPINS; tries++) {
                if (!left) continue;
                int c = -1;
                if (nlow < 0) {
                    c = jp_try(d, p);
                } else {
                    nlow = jp_poll(d, mine, nlow, used);
                    if (nlow == 0) c = jp_first(used);
                }
                if (c >= 0) {
                    __hip_atomic_store(&d.jp_col[p], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    left = false;
                }
            }
        } else {
            for (; __any(left) && tries < FLOW_SPINS; tries++) {
                left = false;
                for (int k = gtid; k < nact; k += gsz) {
                    const int p = d.act[k];
                    if (jp_col_load(d.jp_col, p) >= 0) continue;
                    const int c = jp_try(d, p);
                    if (c >= 0) __hip_atomic_store(&d.jp_col[p], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    else left = true;
                }
            }
        }
        if (__any(left)) stalled();
        if ((tid & (WAVE - 1)) == 0) atomicMax(&d.cnt->jp_rounds, tries);
        // the pairs' places in their colours: among the workgroup's for the first colours, counted in LDS
        // (an atomic on each colour's one counter serialises over the whole GPU)
        __syncthreads();
        for (int k = gtid; k < nact; k += gsz) {
            const int p = d.act[k];
            const int c = jp_col_load(d.jp_col, p);
            if (c >= 0) d.jp_idx[p] = c < FLOW_BINS ? atomicAdd(&s_hist[c], 1) : atomicAdd(&d.jp_ccount[c], 1);
        }
        __syncthreads();
        if (tid < FLOW_BINS) d.jp_hist[tid * gridDim.x + blockIdx.x] = s_hist[tid];
    } else {
        if (blockIdx.x == 0) {
            __shared__ int wsum[FLOW_THREADS / WAVE + 1];
            for (int i = tid; i < d.b.n; i += FLOW_THREADS) claim_set<false>(d.claim, i, colour::FREE);
            claim_sync<false>();
            int* bufs[3] = {d.act, d.act + d.pcap, d.act + 2 * (size_t)d.pcap};
            const int nc = colour_pairs<false>(d.b, d.ps, bufs, nact, d.order, d.color_start, d.claim, 0, 0, wsum);
            if (tid == 0) {
                d.cnt->ncolors = nc;
                d.cnt->nordered = d.color_start[nc];
            }
        }
        grid_barrier(&d.cnt->bar_count, &d.cnt->bar_gen, gridDim.x);
        const int ncol = d.cnt->ncolors, nord = d.cnt->nordered;
        for (int q = gtid; q < nord; q += gsz) {
            int lo = 0, hi = ncol;   // last colour starting at or before q
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (d.color_start[mid] <= q) lo = mid; else hi = mid;
            }
            const int p = d.order[q];
            d.jp_col[p] = lo;
            d.jp_idx[p] = q - d.color_start[lo];
            if (q == d.color_start[lo]) d.jp_ccount[lo] = d.color_start[lo + 1] - q;
        }
    }
    grid_barrier(&d.cnt->bar_count, &d.cnt->bar_gen, gridDim.x);   // every colour is set and counted
    // each colour's pairs, and for the colours counted per workgroup those of the workgroups before this one
    if (!coloured) {
        if (tid < FLOW_BINS) s_cs[tid] = 0;
        __syncthreads();
        for (int c = tid / WAVE; c < FLOW_BINS; c += FLOW_THREADS / WAVE) {
            int all = 0, before = 0;
            for (int g = tid & (WAVE - 1); g < (int)gridDim.x; g += WAVE) {
                const int m = d.jp_hist[c * gridDim.x + g];
                all += m;
                before += g < (int)blockIdx.x ? m : 0;
            }
            for (int o = WAVE / 2; o > 0; o >>= 1) {
                all += __shfl_xor(all, o, WAVE);
                before += __shfl_xor(before, o, WAVE);
            }
            s_cs[c] = all;
            s_hist[c] = before;
            if (all == 0) break;   // the colours end at the first empty one at the latest
        }
    }
    // Colour starts in the solve order and in the items.  First-fit colours are dense (a pair of colour c
    // has lower neighbours of every colour below c), so the colours end at the first empty one.
    for (int c = tid + (coloured ? 0 : FLOW_BINS); c < FLOW_COLORS; c += FLOW_THREADS) s_cs[c] = c <= d.pcap ? d.jp_ccount[c] : 0;
    __syncthreads();
    if (tid == 0) {
        int run = 0, items = 0, c = 0;
        for (; c < FLOW_COLORS && s_cs[c] > 0; c++) {
            const int m = s_cs[c];
            s_cs[c] = run;
            s_is[c] = items;
            run += m;
            items += (m + FLOW_PAIRS - 1) / FLOW_PAIRS;
        }
        s_cs[c] = run;
        s_is[c] = items;
        s_ncol = c;
    }
    __syncthreads();
    int ncol = s_ncol;
    if (ncol == FLOW_COLORS) {   // the same for every workgroup: the starts beyond, through memory
        if (gtid == 0) {
            int run = s_cs[ncol], items = s_is[ncol], c = ncol;
            for (; c <= d.pcap && d.jp_ccount[c] > 0; c++) {
                const int m = d.jp_ccount[c];
                d.color_start[c] = run;
                d.jp_items[c] = items;
                run += m;
                items += (m + FLOW_PAIRS - 1) / FLOW_PAIRS;
            }
            d.color_start[c] = run;
            d.jp_items[c] = items;
            d.cnt->jp_ncol = c;
        }
        grid_barrier(&d.cnt->bar_count, &d.cnt->bar_gen, gridDim.x);
        ncol = d.cnt->jp_ncol;
    }
    auto cs = [&](int c) { return c <= FLOW_COLORS ? s_cs[c] : d.color_start[c]; };
    auto is = [&](int c) { return c <= FLOW_COLORS ? s_is[c] : d.jp_items[c]; };
    if (blockIdx.x == 0) {
        for (int c = tid; c <= ncol; c += FLOW_THREADS)
            if (c <= FLOW_COLORS) d.color_start[c] = s_cs[c];
        if (tid == 0) {
            d.cnt->ncolors = ncol;
            d.cnt->jp_ncol = ncol;
            d.cnt->nordered = cs(ncol);
        }
    }
    // the solve order, and each pair's place in its bodies' sequences of updates
    const int32_t* list = coloured ? d.order : d.act;   // (the claims' lists are built in d.act)
    for (int k = gtid; k < nact; k += gsz) {
        const int p = list[k];
        const int c = d.jp_col[p];
        if (c < 0) continue;   // only after a wait given up
        const int q = cs(c) + d.jp_idx[p] + (!coloured && c < FLOW_BINS ? s_hist[c] : 0);
        const int a = d.ps.pa[p], b = d.ps.pb[p];
        const bool ka = d.b.iat(I_KIN, a) != 0, kb = d.b.iat(I_KIN, b) != 0;
        if (d.rows_out) atomicAdd(&d.cnt->nrows, d.ps.npts[p]);
        d.order[q] = p;
        d.q_pair[q] = make_int4(p, ka ? a | 1 << 31 : a, kb ? b | 1 << 31 : b, d.ps.npts[p]);
        d.q_seq[q] = make_int4(ka ? 0 : jp_rank(d, a, p, c, sets), ka ? 0 : d.jp_deg[a] + (d.jdeg ? d.jdeg[a] : 0),
                               kb ? 0 : jp_rank(d, b, p, c, sets), kb ? 0 : d.jp_deg[b] + (d.jdeg ? d.jdeg[b] : 0));
    }
    grid_barrier(&d.cnt->bar_count, &d.cnt->bar_gen, gridDim.x);   // the order is complete
    if (gtid == 0) report_rows(d, d.cnt->nrows, ncol);

    // consecutive items go to different workgroups, so a colour's pairs spread over the CUs; half of the
    // waves take the joints, if there are any
    const int wave = (tid / WAVE) * gridDim.x + blockIdx.x;
    const int all_waves = gridDim.x * (FLOW_THREADS / WAVE), nwaves = d.njoints > 0 ? all_waves / 2 : all_waves;
    const int lane = tid & (WAVE - 1);
    if (wave >= nwaves) {
        const int jw = wave - nwaves, nl = (all_waves - nwaves) * FLOW_JOINTS;
        const int j0 = lane < FLOW_JOINTS ? jw * FLOW_JOINTS + lane : d.njoints;
        if (!flow_joints(d, j0, nl)) stalled();
        return;
    }
    const int quad = lane >> 2, c = (lane & 3) < 2 ? lane & 3 : 2;
    const bool first = (lane & 3) == 0, own = (lane & 3) < 3;
    const int nitems = is(ncol);
    const bool resident = nitems <= nwaves;
    // The wave goes through its places in the order: items wave, wave + nwaves, ... of every iteration, each
    // solved once all its pairs are ready (solving the ready ones of a poll by themselves repeats the row
    // chains, which cost as much as the wait: 380 us instead of 275 for 10 000 boxes at rest).
    int item = wave, it = 0;
    bool live = item < nitems && d.iterations > 0, fresh = true, ra = false, rb = false;
    uint32_t ea = 0, eb = 0;
    QuadRow r[4];
    FlowPair f;
    for (int spin = 0; __any(live); spin++) {
        if (spin == FLOW_SPINS) { stalled(); return; }
        if (live && fresh) {
            if (it == 0 || !resident) {
                int lo = 0, hi = ncol;   // last colour whose first item is at or before this one
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (is(mid) <= item) lo = mid; else hi = mid;
                }
                const int q = cs(lo) + (item - is(lo)) * FLOW_PAIRS + quad;
                flow_load(d, q, q < cs(lo + 1), c, f);
                flow_rows(f, 0, c, r);
            }
            fresh = false;
            ra = f.A.kin;
            rb = f.B.kin;
            f.A.tv = f.A.tw = f.B.tv = f.B.tw = 0.0f;   // a kinematic body's stay so (rigidbody.cpp:72-80, 167)
            ea = (uint32_t)(it * f.seq.y + f.seq.x);
            eb = (uint32_t)(it * f.seq.w + f.seq.z);
        }
        uint64_t a0 = 0, a1 = 0, b0 = 0, b1 = 0;
        const bool pa = live && !ra, pb = live && !rb;
        if (pa) { a0 = vel_load(f.wa); a1 = vel_load(f.wa + 4); }
        if (pb) { b0 = vel_load(f.wb); b1 = vel_load(f.wb + 4); }
        uint32_t dist = 0;
        if (pa) flow_take(f.A, a0, a1, ea, ra, dist);
        if (pb) flow_take(f.B, b0, b1, eb, rb, dist);
        const bool go = !__any(live && !(ra && rb));
        if (go) {
            flow_solve(d, f, c, first, own, r, ea, eb, (uint32_t)(d.iterations * f.seq.y), (uint32_t)(d.iterations * f.seq.w));
            fresh = true;
            item += nwaves;
            if (item >= nitems) {
                item = wave;
                live = ++it < d.iterations;
            }
            if (own && (!resident || !live)) flow_store_acc(f, 0, c, r);
        }
        if (go) spin = 0;
        else flow_pause(!(ra && rb), dist);
    }
}

// ---- the solve of a small world in one workgroup
// The solve of a small world in one workgroup: the bodies' temp velocities in LDS, a workgroup barrier between
// colours (0.1 us) where the flow over the GPU pays 0.9 us for a store to be seen on another CU, and three launches
// less (4.5 us each).  Four lanes per pair as there (quad_solve_row): a colour of up to SMALL_THREADS / 4 pairs is one
// pass as long as its longest pair's row chains; a larger one takes several, which is where the flow becomes faster.
constexpr int SMALL_THREADS = FLOW_THREADS;
constexpr int SMALL_LDS = 152 * 1024;
constexpr int SMALL_COLORS = 128;   // colours counted in LDS (two 64-bit masks per body)
constexpr int SMALL_ROW = RW + 1;   // a row's floats in LDS: an odd stride spreads the quads' rows over the banks

// The sweeps on LDS velocities vel ([n][8]: linear from 0, angular from 4) over the ordered pairs info (pair,
// bodies A and B with the kinematic flag on top, rows | first row in rows << 4); ROWS_LDS: the rows are in
// rows, else in the row store.
template <bool ROWS_LDS>
__device__ __forceinline__ void small_sweeps(const Dev& d, float* vel, const int4* info, float* rows, const int* cs, int ncol) {
    const int tid = threadIdx.x;
    const int quad = tid >> 2, c = (tid & 3) < 2 ? tid & 3 : 2;
    const bool first = (tid & 3) == 0, own = (tid & 3) < 3;
    QuadRow r[4];
    QuadBody A, B;
    int4 f = make_int4(0, 0, 0, 0);
    bool have = false;
    auto row = [&](int k) {
        return ROWS_LDS ? rows + (size_t)((f.w >> 4) + k) * SMALL_ROW : d.ps.rows + ((size_t)f.x * 8 + k) * RW;
    };
    auto load4 = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (k0 + u < (f.w & 15)) quad_load_row(row(k0 + u), c, r[u]);
    };
    auto solve4 = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (k0 + u < (f.w & 15)) {
                quad_solve_row(r[u], first, A, B);
                if (own) row(k0 + u)[R_LN + c] = r[u].acc;
            }
    };
    auto fetch = [&](int q, int end) {
        have = q < end;
        if (!have) return;
        f = info[q];
        quad_load_body(d.b.sbr(f.y & 0x7fffffff), c, f.y < 0, A);
        quad_load_body(d.b.sbr(f.z & 0x7fffffff), c, f.z < 0, B);
        load4(0);
    };
    auto solve = [&]() {
        float* va = vel + (f.y & 0x7fffffff) * 8 + c;
        float* vb = vel + (f.z & 0x7fffffff) * 8 + c;
        A.tv = va[0]; A.tw = va[4];
        B.tv = vb[0]; B.tw = vb[4];
        solve4(0);
        if ((f.w & 15) > 4) {
            load4(4);
            solve4(4);
        }
        if (own && !A.kin) { va[0] = A.tv; va[4] = A.tw; }
        if (own && !B.kin) { vb[0] = B.tv; vb[4] = B.tw; }
    };
    if (ncol > 0) fetch(cs[0] + quad, cs[1]);
    for (int it = 0; it < d.iterations; it++) {
        for (int k = 0; k < ncol; k++) {
            if (have) {
                solve();
                for (int q = cs[k] + quad + SMALL_THREADS / 4; q < cs[k + 1]; q += SMALL_THREADS / 4) {
                    fetch(q, cs[k + 1]);
                    solve();
                }
            }
            const int nx = k + 1 < ncol ? k + 1 : 0;
            fetch(cs[nx] + quad, cs[nx + 1]);   // all but the velocities, ahead of the barrier
            __syncthreads();
        }
        // the joints after the contacts, colour by colour (sequential_impulse_solver.cpp:66-68)
        for (int k = 0; k < d.njcol; k++) {
            for (int q = d.jcs[k] + tid; q < d.jcs[k + 1]; q += SMALL_THREADS) {
                const int id = d.jorder[q];
                const JointDef j = d.joints[id];
                SolvBody S[2] = {load_solv(d.b, j.a), load_solv(d.b, j.b)};
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const float* v = vel + (s == 0 ? j.a : j.b) * 8;
                    S[s].tv = f3{v[0], v[1], v[2]};
                    S[s].tw = f3{v[4], v[5], v[6]};
                }
                joint_solve(j, d.jrows[id], S[0], S[1]);
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    if (S[s].kin) continue;
                    float* v = vel + (s == 0 ? j.a : j.b) * 8;
                    v[0] = S[s].tv.x; v[1] = S[s].tv.y; v[2] = S[s].tv.z;
                    v[4] = S[s].tw.x; v[5] = S[s].tw.y; v[6] = S[s].tw.z;
                }
            }
            __syncthreads();
        }
    }
}
__global__ void __launch_bounds__(SMALL_THREADS) k_solve_small(Dev d) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ int s_cnt[SMALL_COLORS], s_cs[SMALL_COLORS + 1], s_ncol, s_full, wsum[SMALL_THREADS / WAVE + 1];
    const int tid = threadIdx.x, n = d.b.n;
    const int nact = d.cnt->nact;
    // LDS: velocities and ordered pairs; then the colouring's arrays, and over them the rows
    float* vel = (float*)lds;
    int4* info = (int4*)(lds + (size_t)n * 32);
    unsigned char* rest = (unsigned char*)(info + nact);
    uint64_t* mask = (uint64_t*)rest;                  // [n][2] colours of a body's coloured pairs
    int* claim = (int*)(mask + 2 * (size_t)n);         // [2][n] claims of even and odd rounds
    int* prio = claim + 2 * n;                         // per pair: claim priority,
    uint32_t* ab = (uint32_t*)(prio + nact);           // bodies A | B << 16,
    int* col = (int*)(ab + nact);                      // colour | place in the colour << 8 (-1: none yet)
    bool small = (size_t)n * 32 + (size_t)nact * 28 + (size_t)n * 24 <= (size_t)SMALL_LDS;
    if (small) {
        if (tid < SMALL_COLORS) s_cnt[tid] = 0;
        if (tid == 0) s_full = 0;
        for (int i = tid; i < n; i += SMALL_THREADS) {
            const float* s = d.b.sbr(i);
            const float4 q0 = reinterpret_cast<const float4*>(s)[0], q1 = reinterpret_cast<const float4*>(s)[1];
            float4* v = reinterpret_cast<float4*>(vel + (size_t)i * 8);   // tv 0..2, tw 3..5, im, kin in the record
            v[0] = make_float4(q0.x, q0.y, q0.z, 0.0f);
            v[1] = make_float4(q0.w, q1.x, q1.y, q1.w);   // [7]: the kinematic flag
            mask[2 * i] = mask[2 * i + 1] = 0;
            claim[i] = claim[n + i] = colour::FREE;
        }
        for (int k = tid; k < nact; k += SMALL_THREADS) {
            const int p = d.act[k];
            prio[k] = colour::prio(p, d.ps.npts[p]);
            ab[k] = (uint32_t)d.ps.pa[p] | (uint32_t)d.ps.pb[p] << 16;
            col[k] = -1;
        }
        __syncthreads();
        // Rounds of claims: a pair that holds the lowest claim on its dynamic bodies among the uncoloured ones
        // takes the first colour none of their coloured pairs has.  Those are exactly the neighbours of lower
        // priority (one of higher priority cannot have held its claim before), so the classes are those of
        // colour_pairs, all colours in the rounds of one (about 25 for box piles).
        bool left = nact > 0;
        for (int round = 0; __syncthreads_or(left && s_full == 0); round++) {
            int* now = claim + (round & 1) * n;
            int* next = claim + ((round + 1) & 1) * n;
            for (int k = tid; k < nact; k += SMALL_THREADS) {
                if (col[k] >= 0) continue;
                const int a = ab[k] & 0xffff, b = ab[k] >> 16;
                if (vel[8 * a + 7] == 0.0f) atomicMin(&now[a], prio[k]);
                if (vel[8 * b + 7] == 0.0f) atomicMin(&now[b], prio[k]);
            }
            __syncthreads();
            left = false;
            for (int k = tid; k < nact; k += SMALL_THREADS) {
                if (col[k] >= 0) continue;
                const int a = ab[k] & 0xffff, b = ab[k] >> 16;
                const bool ka = vel[8 * a + 7] != 0.0f, kb = vel[8 * b + 7] != 0.0f;
                if (!ka) next[a] = colour::FREE;
                if (!kb) next[b] = colour::FREE;
                if (!((ka || now[a] == prio[k]) && (kb || now[b] == prio[k]))) {
                    left = true;
                    continue;
                }
                const uint64_t u0 = (ka ? 0 : mask[2 * a]) | (kb ? 0 : mask[2 * b]);
                const uint64_t u1 = (ka ? 0 : mask[2 * a + 1]) | (kb ? 0 : mask[2 * b + 1]);
                if (~u0 == 0 && ~u1 == 0) {
                    s_full = 1;
                    continue;
                }
                const int w = ~u0 != 0 ? 0 : 1, c = __ffsll((unsigned long long)~(w == 0 ? u0 : u1)) - 1;
                if (!ka) mask[2 * a + w] |= 1ull << c;
                if (!kb) mask[2 * b + w] |= 1ull << c;
                col[k] = (64 * w + c) | atomicAdd(&s_cnt[64 * w + c], 1) << 8;
            }
        }
        small = s_full == 0;
        __syncthreads();
    }
    if (!small) {   // the same for every thread
        solve_alone<true>(d, nact, (int*)lds);
        if (tid == 0) {
            d.cnt->nact = 0;
            report_rows(d, 8 * nact, 0);
        }
        return;
    }
    if (tid == 0) {
        int run = 0, c = 0;
        for (; c < SMALL_COLORS && s_cnt[c] > 0; c++) {
            s_cs[c] = run;
            run += s_cnt[c];
        }
        s_cs[c] = run;
        s_ncol = c;
    }
    __syncthreads();
    const int ncol = s_ncol;
    for (int k = tid; k < nact; k += SMALL_THREADS) {
        const int p = d.act[k], q = s_cs[col[k] & 0xff] + (col[k] >> 8);
        const int a = ab[k] & 0xffff, b = ab[k] >> 16;
        info[q] = make_int4(p, vel[8 * a + 7] != 0.0f ? a | 1 << 31 : a, vel[8 * b + 7] != 0.0f ? b | 1 << 31 : b, d.ps.npts[p]);
        d.order[q] = p;
    }
    for (int c = tid; c <= ncol; c += SMALL_THREADS) d.color_start[c] = s_cs[c];
    __syncthreads();
    int nrows = 0;
    for (int base = 0; base < nact; base += SMALL_THREADS) {
        const int q = base + tid;
        const int m = q < nact ? info[q].w : 0;
        int tot;
        const int ex = block_exclusive_scan(m, wsum, &tot);
        if (q < nact) info[q].w = m | (nrows + ex) << 4;
        nrows += tot;
    }
    __syncthreads();
    float* rows = (float*)rest;
    if ((size_t)n * 32 + (size_t)nact * 16 + (size_t)nrows * SMALL_ROW * 4 <= (size_t)SMALL_LDS) {
        // a thread per float4 of a pair's rows (8 slots of 6)
        for (int k = tid; k < nact * 48; k += SMALL_THREADS) {
            const int q = k / 48, u = k % 48 / 6, part = k % 6;
            const int4 f = info[q];
            if (u >= (f.w & 15)) continue;
            const float4 v = reinterpret_cast<const float4*>(d.ps.rows + ((size_t)f.x * 8 + u) * RW)[part];
            float* o = rows + (size_t)((f.w >> 4) + u) * SMALL_ROW + 4 * part;
            o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
        }
        __syncthreads();
        small_sweeps<true>(d, vel, info, rows, s_cs, ncol);
        for (int k = tid; k < nact * 8; k += SMALL_THREADS) {   // the accumulated impulses, for the getters
            const int4 f = info[k >> 3];
            if ((k & 7) >= (f.w & 15)) continue;
            const float* o = rows + (size_t)((f.w >> 4) + (k & 7)) * SMALL_ROW + R_LN;
            float* t = d.ps.rows + ((size_t)f.x * 8 + (k & 7)) * RW + R_LN;
            t[0] = o[0]; t[1] = o[1]; t[2] = o[2];
        }
    } else {
        small_sweeps<false>(d, vel, info, rows, s_cs, ncol);
    }
    __syncthreads();
    // syncTempVelocity (sequential_impulse_solver.cpp:71-80)
    for (int i = tid; i < n; i += SMALL_THREADS) {
        const float* v = vel + (size_t)i * 8;
        if (v[7] != 0.0f) continue;
        float* s = d.b.sbr(i);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            d.b.at(F_V + k, i) = s[SB_TV + k] = v[k];
            d.b.at(F_W + k, i) = s[SB_TW + k] = v[4 + k];
        }
    }
    if (tid == 0) {
        d.cnt->ncolors = ncol;
        d.cnt->nordered = nact;
        d.cnt->jp_rounds = 0;
        d.cnt->nact = 0;   // counted from zero by the next step's set-up
        report_rows(d, nrows, ncol);
    }
}

// Ends a narrowphase: its contact points, per-workgroup sums added to the counter k_narrow cleared; a pair whose
// clipper lost points (bit 1 of its swap word) raises OVF_CLIP; the pairs become the previous step's and the
// lists are empty again (no workgroup here reads either; a launch of its own for that was 4.5 us a step).
__global__ void __launch_bounds__(256) k_count_points(Dev d) {
    __shared__ int wsum[256 / WAVE + 1];
    const int np = d.cnt->npairs;
    int acc = 0, lost = 0;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        acc += d.ps.npts[p];
        lost |= d.ps.swap[p] & 2;
    }
    int tot;
    block_exclusive_scan(acc, wsum, &tot);
    if (threadIdx.x == 0 && tot) atomicAdd(&d.cnt->npoints, tot);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        d.cnt->prev_npairs = np;
        d.cnt->nshape = 0;
        d.cnt->nsat = 0;
        d.cnt->ncomp = 0;
    }
    if (lost) atomicOr(&d.cnt->overflow, OVF_CLIP);
}

}  // namespace

// ====================================================================== host side
// Workgroups of the solve over the GPU: enough waves for about an item each (a world at rest has up to
// two pairs with contacts per body, 16 to an item), at most one workgroup per CU of the 256.
static int default_flow_blocks(int n, int max_blocks) { return std::min(max_blocks, std::max(8, std::min(256, n / 80))); }

struct pe_world;
namespace {
// Turns at k_solve_flow between this process's worlds on one GPU.  As long as all of them fit on it at once
// nothing is done; else the worlds that can do without leave it (40 worlds of 500 bodies on their own streams: 3960 us
// a step of all with turns, 2260 in a workgroup each), and if the others still do not fit each launch waits for the one
// before it, so that two of them never share the GPU with neither complete.
struct FlowTurns {
    std::mutex m;
    int blocks[2] = {0, 0};      // workgroups of all live worlds that can do without the flow, that cannot
    hipEvent_t last = nullptr;   // after the last launch (kept for the process)
    uint64_t last_order = 0;     // whose order it came in (pe_world::order)
};
// Those of a world's own device, whichever is current when it is changed or destroyed.
FlowTurns& flow_turns(int device) {
    static FlowTurns t[64];
    return t[device >= 0 && device < 64 ? device : 0];
}
struct FlowTurn {
    explicit FlowTurn(pe_world& w);
    int done();
    pe_world& w;
    FlowTurns& t;
    std::unique_lock<std::mutex> lock;
    bool crowded;
    hipError_t err = hipSuccess;
};
}  // namespace

// The solve runs in one workgroup (k_solve_small) up to SMALL_BODIES bodies, and up to SMALL_MAX while the last solve
// the host knows of had no more contact points than SMALL_POINTS + SMALL_COLOUR_POINTS a colour, or the process's worlds
// crowd the GPU (FlowTurns): more fill a colour's pass of the workgroup more than once, where the flow waits once a
// colour whatever it holds.  us per step in one workgroup / over the GPU (contact points, colours):
//   bodies                  200              260               300                400                590
//   boxes at rest           141 / 144 (716)  162 / 160 (958)   172 / 159 (1043)   210 / 166 (1429)   279 / 181 (2107)
//   boxes, spheres at rest  141 / 145 (447)  153 / 150 (643)   167 / 157 (733)    180 / 157 (877)    237 / 169 (1322)
//   boxes, spheres falling  107 / 127 (279)  125 / 137 (362)   122 / 134 (389)    131 / 135 (472)    162 / 148 (748)
//   joint chains             80 / 121 (0)    250 / 304 (0)     274 / 335 (3)      272 / 325 (5)      293 / 356 (8)
//   bodies                  285                 330                 380                 440                 590
//   a steeper pile, boxes   204 / 215 (994, 6)  214 / 219 (1142, 6) 236 / 228 (1339, 7) 268 / 237 (1539, 6) 328 / 267 (1981, 7)
//   with spheres            181 / 186 (687, 5)  206 / 213 (789, 6)  211 / 212 (885, 6)  234 / 221 (1035, 6) 278 / 239 (1321, 6)
//   a tower struck          233 / 248 (1188, 7) 263 / 263 (1232, 7) 281 / 258 (1240, 6) 305 / 271 (1932, 7) 429 / 306 (3281, 7)
// (of these a line at 650 points gave up to 8 % away, this one up to 6 where it keeps one workgroup and 3 where not).
constexpr int SMALL_BODIES = 280, SMALL_MAX = 600, SMALL_POINTS = 200;

struct pe_world {
    Dev d{};
    int n = 0, stride = 0;
    hipStream_t stream = nullptr;
    std::vector<void*> allocs;
    int flow_blocks = 0;    // workgroups of the solve over the GPU
    int flow_max_blocks = 0;                 // and how many of them the GPU holds at once
    uint64_t flow_patience = 5000000;        // 50 ms
    int device = 0;
    int flow_counted[2] = {0, 0};            // workgroups entered in flow_turns(device)
    hipStream_t own = nullptr;               // the world's own stream (stream: the one it is being stepped on)
    uint64_t id = 0;                         // of this world, never used again
    // Two launches of one order follow each other anyway, those on the world's own stream or on the null stream; 0: on
    // another, whose handle may come to be another stream's.
    uint64_t order() const { return stream == own ? id : stream == nullptr ? 1 : 0; }
    bool flowed = false;                     // the last solve was over the GPU: it leaves its pairs listed
    int colouring = 0;                       // 0: by body count, 1: one workgroup's claims, 2: over the GPU
    int32_t* rows = nullptr;                 // host memory: what report_rows left there last,
    int32_t* rows_dev = nullptr;             // and where a kernel finds it
    int alloc_rows() {
        PE_HIP(hipHostMalloc((void**)&rows, sizeof(int32_t), hipHostMallocMapped));
        *rows = 0;
        PE_HIP(hipHostGetDevicePointer((void**)&rows_dev, rows, 0));
        return PE_OK;
    }
    enum Route { ONE_WORKGROUP = -1, EITHER = 0, FLOW = 1 };
    Route route() const { return colouring != 0 || n > SMALL_MAX ? FLOW : n <= SMALL_BODIES || !rows ? ONE_WORKGROUP : EITHER; }
    bool one_workgroup() const {
        if (route() != EITHER) return route() == ONE_WORKGROUP;
        if (__atomic_load_n(rows, __ATOMIC_RELAXED) <= SMALL_POINTS) return true;
        FlowTurns& t = flow_turns(device);
        std::lock_guard<std::mutex> g(t.m);
        return t.blocks[0] + t.blocks[1] > flow_max_blocks;
    }
    // Enters the world's workgroups for its route (leave: none).
    void count_flow(bool leave = false) {
        FlowTurns& t = flow_turns(device);
        std::lock_guard<std::mutex> g(t.m);
        for (int k = 0; k < 2; k++) {
            const int b = !leave && (int)route() == k ? flow_blocks : 0;
            t.blocks[k] += b - flow_counted[k];
            flow_counted[k] = b;
        }
    }
    bool timing = false;
    hipEvent_t ev[5] = {};
    hipEvent_t order_ev[2] = {};   // orders work on a caller's stream with the world's own stream
    double stage_ms[4] = {0, 0, 0, 0};
    int n_dynamic = 0;
    bool has_shapes = false;   // any cylinder / convex / concave body
    bool has_mesh = false;     // any convex / concave mesh (a compound's children too)
    DevMeshes meshes;
    std::vector<JointDef> joints;            // host copies of the joint definitions
    std::vector<uint64_t> ignore_keys;       // sorted ignore-pair keys
    std::vector<char> kinematic;             // per body (joint colouring)
    std::vector<char> finite_life, has_joint, removed;   // per body (joints and removals exclude each other)
    void* joint_mem[6] = {};                 // device: definitions, rows, order, colour starts, sequence, degrees
    void* ignore_mem = nullptr;
    void* ray_mem = nullptr;                 // raycast inputs, ignore set and results
    size_t ray_bytes = 0;

    ~pe_world() {
        if (stream) hipStreamSynchronize(stream);
        count_flow(true);
        for (void* p : allocs) hipFree(p);
        for (void* p : joint_mem) if (p) hipFree(p);
        if (ignore_mem) hipFree(ignore_mem);
        if (ray_mem) hipFree(ray_mem);
        if (rows) hipHostFree(rows);
        meshes.release();
        for (auto& e : ev) if (e) hipEventDestroy(e);
        for (auto& e : order_ev) if (e) hipEventDestroy(e);
        if (stream) hipStreamDestroy(stream);
    }
    template <class T> int alloc(T** p, size_t count) {
        void* q = nullptr;
        PE_HIP(hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)));
        PE_HIP(hipMemsetAsync(q, 0, std::max<size_t>(count, 1) * sizeof(T), stream));
        allocs.push_back(q);
        *p = (T*)q;
        return PE_OK;
    }
    int grid(int work, int block) const { return std::max(1, std::min((work + block - 1) / block, 4096)); }

    int launch_integrate() {
        if (d.status_on) hipLaunchKernelGGL(k_integrate_status, dim3(grid(n, 256)), dim3(256), 0, stream, d);
        else hipLaunchKernelGGL(k_integrate, dim3(grid(n, 256)), dim3(256), 0, stream, d);
        return PE_OK;
    }
    int launch_broadphase() {
        sap_launch(d.sap, stream);
        return PE_OK;
    }
    int launch_narrowphase() {
        hipLaunchKernelGGL(k_narrow, dim3(grid(d.pcap, 128)), dim3(128), 0, stream, d);
        if (has_shapes) {
            hipLaunchKernelGGL(k_narrow_shapes, dim3(grid(d.pcap, 64)), dim3(64), 0, stream, d);
            hipLaunchKernelGGL(k_narrow_sat, dim3(std::min(grid(d.pcap, 4), 4096)), dim3(256), 0, stream, d);
        }
        if (d.comp_list) hipLaunchKernelGGL(k_narrow_compound, dim3(grid(d.pcap, 64)), dim3(64), 0, stream, d);
        hipLaunchKernelGGL(k_count_points, dim3(grid(d.pcap, 1024)), dim3(256), 0, stream, d);
        if (d.status_on) hipLaunchKernelGGL(k_neighbours, dim3(grid(d.pcap, 256)), dim3(256), 0, stream, d);
        if (d.report_on) hipLaunchKernelGGL(k_events, dim3(grid(d.pcap, 256)), dim3(256), 0, stream, d);
        return PE_OK;
    }
    int launch_solve() {
        d.rows_out = route() == EITHER ? rows_dev : nullptr;
        if (one_workgroup()) {
            if (flowed) hipLaunchKernelGGL(k_no_pairs, dim3(1), dim3(1), 0, stream, d);
            flowed = false;
            hipLaunchKernelGGL(k_setup<false>, dim3(grid(d.pcap, 128)), dim3(128), 0, stream, d);
            if (d.njoints > 0) hipLaunchKernelGGL(k_joint_setup, dim3(grid(d.njoints, 64)), dim3(64), 0, stream, d);
            hipLaunchKernelGGL(k_solve_small, dim3(1), dim3(SMALL_THREADS), SMALL_LDS, stream, d);
            return PE_OK;
        }
        hipLaunchKernelGGL(k_solve_begin, dim3(grid(n, 256)), dim3(256), 0, stream, d);
        hipLaunchKernelGGL(k_setup<true>, dim3(grid(d.pcap, 128)), dim3(128), 0, stream, d);
        if (d.njoints > 0) hipLaunchKernelGGL(k_joint_setup, dim3(grid(d.njoints, 64)), dim3(64), 0, stream, d);
        hipLaunchKernelGGL(k_jp_alloc, dim3(grid(n, 256)), dim3(256), 0, stream, d);
        hipLaunchKernelGGL(k_jp_fill, dim3(grid(d.pcap, 256)), dim3(256), 0, stream, d);
        int claims = colouring == 1;
        flowed = true;
        FlowTurn turn(*this);
        hipLaunchKernelGGL(k_solve_flow, dim3(flow_blocks), dim3(FLOW_THREADS), 0, stream, d, claims, flow_patience);
        return turn.done();
    }
    int step() {
        pe_clear_stale_error();
        if (timing) hipEventRecord(ev[0], stream);
        launch_integrate();
        if (timing) hipEventRecord(ev[1], stream);
        launch_broadphase();
        if (timing) hipEventRecord(ev[2], stream);
        launch_narrowphase();
        if (timing) hipEventRecord(ev[3], stream);
        launch_solve();
        if (timing) hipEventRecord(ev[4], stream);
        PE_HIP(hipGetLastError());
        if (timing) {
            PE_HIP(hipEventSynchronize(ev[4]));
            for (int k = 0; k < 4; k++) {
                float ms = 0;
                hipEventElapsedTime(&ms, ev[k], ev[k + 1]);
                stage_ms[k] += ms;
            }
        }
        return PE_OK;
    }
};

namespace {
FlowTurn::FlowTurn(pe_world& w_) : w(w_), t(flow_turns(w_.device)), lock(t.m), crowded(t.blocks[1] > w_.flow_max_blocks) {
    if (crowded) {   // a stream under capture takes no part: what it waits for then is not this launch's time
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        crowded = hipStreamIsCapturing(w.stream, &st) != hipSuccess || st == hipStreamCaptureStatusNone;
    }
    if (!crowded) {
        lock.unlock();
        return;
    }
    if (!t.last) err = hipEventCreateWithFlags(&t.last, hipEventDisableTiming);
    else if (w.order() == 0 || w.order() != t.last_order) err = hipStreamWaitEvent(w.stream, t.last, 0);
}
int FlowTurn::done() {
    if (crowded && err == hipSuccess) {
        err = hipEventRecord(t.last, w.stream);
        t.last_order = w.order();
    }
    PE_HIP(err);
    return PE_OK;
}
int check_world(pe_world* w) {
    if (!w) { pe_set_error("null world"); return PE_ERR_INVALID; }
    return PE_OK;
}
// Reports the capacity errors the steps since the last report raised (PE_ERR_CAPACITY, with the
// causes in the message) and clears them; c holds counters read after the stream drained.
int report_overflow(pe_world* w, const DevCounts& c) {
    if (c.overflow == 0) return PE_OK;
    std::string m = "capacity exceeded:";
    if (c.overflow & OVF_PAIRS) m += " more broadphase pairs than max_pairs (" + std::to_string(w->d.pcap) + ")";
    if (c.overflow & OVF_CHUNKS) m += " more sweep candidates than the sweep's chunk capacity";
    if (c.overflow & OVF_CLIP) m += " a clipped contact polygon outgrew its buffer";
    if (c.overflow & OVF_STALL) m = "the solver gave up waiting for an update that never came";
    PE_HIP(hipMemsetAsync(&w->d.cnt->overflow, 0, sizeof(int32_t), w->stream));
    PE_HIP(hipStreamSynchronize(w->stream));
    pe_set_error(m);
    return (c.overflow & OVF_STALL) ? PE_ERR_DEVICE : PE_ERR_CAPACITY;
}
}  // namespace

extern "C" {

const char* pe_last_error(void) { return g_err.c_str(); }

int pe_device_count(int32_t* count) {
    int c = 0;
    PE_HIP(hipGetDeviceCount(&c));
    if (count) *count = c;
    return PE_OK;
}

int pe_world_create(const pe_scene_desc* sc, const pe_world_params* prm, int32_t max_pairs, pe_world** out) {
    if (!sc || !prm || !out || sc->n <= 0) { pe_set_error("pe_world_create: invalid argument"); return PE_ERR_INVALID; }
    if (int rc = check_scene(sc)) return rc;
    auto* w = new pe_world();
    const int n = sc->n;
    w->n = n;
    w->stride = (n + 63) & ~63;
    const int64_t want = max_pairs > 0 ? (int64_t)max_pairs : std::max<int64_t>(1024, 16 * (int64_t)n);
    if (want > ((int64_t)1 << colour::PRIO_INDEX_BITS)) {
        delete w;
        pe_set_error("pe_world_create: at most 2^28 pairs per world");
        return PE_ERR_INVALID;
    }
    const int pcap = (int)want;
    auto fail = [&](int rc) { delete w; return rc; };
    if (hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking) != hipSuccess) { pe_set_error("stream create failed"); return fail(PE_ERR_DEVICE); }
    static std::atomic<uint64_t> worlds{2};
    w->id = worlds++;
    w->own = w->stream;
    if (n > SMALL_BODIES && n <= SMALL_MAX && w->alloc_rows() != PE_OK) return fail(PE_ERR_DEVICE);
    Dev& d = w->d;
    d.pcap = pcap;
    d.ps.cs = (size_t)pcap * 8;
    d.dt = (float)prm->dt;
    for (int k = 0; k < 3; k++) d.g[k] = (float)prm->gravity[k];
    d.iterations = prm->iterations;
    d.b.n = n;
    d.b.stride = w->stride;
    const size_t S = w->stride;
    int rc = PE_OK;
    rc |= w->alloc(&d.b.f, NF * S);
    rc |= w->alloc(&d.b.i, NI * S);
    rc |= w->alloc(&d.ps.pa, pcap);
    rc |= w->alloc(&d.ps.pb, pcap);
    rc |= w->alloc(&d.ps.cp, (size_t)CW * pcap * 8);
    rc |= w->alloc(&d.ps.cd, (size_t)pcap * 8);
    rc |= w->alloc(&d.b.cb, (size_t)CBW * S);
    rc |= w->alloc(&d.b.sb, (size_t)SBW * S);
    rc |= w->alloc(&d.b.ab, (size_t)8 * S);
    rc |= w->alloc(&d.ps.npts, pcap);
    rc |= w->alloc(&d.ps.swap, pcap);
    rc |= w->alloc(&d.ps.rows, (size_t)RW * pcap * 8);
    rc |= w->alloc(&d.order, pcap);
    rc |= w->alloc(&d.shape_list, pcap);
    rc |= w->alloc(&d.act, 3 * (size_t)pcap);
    rc |= w->alloc(&d.color_start, pcap + 1);
    rc |= w->alloc(&d.claim, n);
    rc |= w->alloc(&d.cnt, 1);
    rc |= w->alloc(&d.jp_deg, n);
    rc |= w->alloc(&d.jp_off, n);
    rc |= w->alloc(&d.jp_fill, n);
    rc |= w->alloc(&d.jp_adj, 2 * (size_t)pcap);
    rc |= w->alloc(&d.jp_col, pcap);
    rc |= w->alloc(&d.jp_idx, pcap);
    rc |= w->alloc(&d.jp_set, pcap);
    rc |= w->alloc(&d.jp_set_at, n);
    rc |= w->alloc(&d.jp_ccount, (size_t)pcap + 1);
    rc |= w->alloc(&d.jp_items, (size_t)pcap + 1);
    rc |= w->alloc(&d.vel, (size_t)VELW * n);
    rc |= w->alloc(&d.q_pair, pcap);
    rc |= w->alloc(&d.q_seq, pcap);
    rc |= w->alloc(&d.st.flags, n);
    rc |= w->alloc(&d.st.sleep_time, n);
    rc |= w->alloc(&d.st.life, n);
    rc |= w->alloc(&d.st.last, n);
    rc |= w->alloc(&d.st.scnt, n);
    rc |= w->alloc(&d.st.dcnt, n);
    rc |= w->alloc(&d.st.report, n);
    rc |= w->alloc(&d.events, (size_t)EVW * pcap);
    rc |= w->alloc(&d.ev_flag, pcap);
    SapView& sp = d.sap;
    sp.n = n;
    sp.amin = d.b.f + (size_t)F_AMIN * w->stride;
    sp.amax = d.b.f + (size_t)F_AMAX * w->stride;
    sp.fs = w->stride;
    sp.bs = 1;
    sp.rec = d.b.ab;
    sp.cnt = d.cnt;
    sp.pa = d.ps.pa;
    sp.pb = d.ps.pb;
    sp.pcap = pcap;
    rc |= w->alloc(&sp.keys, n);
    rc |= w->alloc(&sp.vals, n);
    rc |= w->alloc(&sp.keys2, n);
    rc |= w->alloc(&sp.vals2, n);
    rc |= w->alloc(&sp.skey, n);
    rc |= w->alloc(&sp.srec, (size_t)8 * n);
    rc |= w->alloc(&sp.end, n);
    rc |= w->alloc(&sp.first, n);
    rc |= w->alloc(&sp.blk, sap_blocks(n));
    rc |= w->alloc(&sp.sub, sap_subs(n));
    sp.axis_in = -1;
    rc |= w->alloc(&sp.hist, 256 * (size_t)sap_radix_blocks(n));
    rc |= w->alloc(&sp.red, SAP_RED_VALUES * (size_t)sap_red_blocks(n));
    // sweep chunks: the candidates (bodies overlapping on the sweep axis) are at most n (n - 1) / 2,
    // and a pile that lands while the axis is still the fall direction comes close to that (the
    // reference's sweep too: the axis is chosen after the sweep); 12 bytes per 64 candidates, so the
    // bound itself is allocated, up to 2^31 candidates
    const int64_t max_cand = std::min<int64_t>((int64_t)n * (n - 1) / 2, (int64_t)1 << 31);
    sp.chunk_cap = (int)std::max<int64_t>(max_cand / SAP_CHUNK + 1, 1024);
    rc |= w->alloc(&sp.owner, sap_units(sp.chunk_cap, n));
    rc |= w->alloc(&sp.unit_hit, sap_units(sp.chunk_cap, n));
    if (rc != PE_OK) return fail(PE_ERR_DEVICE);

    // host staging of the body store (FP32) and of the scene's meshes
    std::vector<float> hf(NF * S, 0.0f);
    std::vector<int32_t> hi(NI * S, 0);
    HostMeshes hm;
    if (int rc2 = stage_bodies(sc, hf, hi, S, 0, hm)) return fail(rc2);
    if (int rc2 = w->meshes.upload(hm, w->stream)) return fail(rc2);
    d.b.ms = w->meshes.view();
    w->has_mesh = hm.count() > 0;
    int ndyn = 0;
    bool has_compound = false;
    w->kinematic.resize(n);
    for (int i = 0; i < n; i++) {
        ndyn += sc->kinematic[i] ? 0 : 1;
        w->kinematic[i] = sc->kinematic[i] ? 1 : 0;
        w->has_shapes |= sc->shape_type[i] > PE_SHAPE_SPHERE;
        has_compound |= sc->shape_type[i] == PE_SHAPE_COMPOUND;
    }
    if (has_compound && w->alloc(&d.comp_list, pcap) != PE_OK) return fail(PE_ERR_DEVICE);
    w->n_dynamic = ndyn;
    // RigidBody::_life_time (rigidbody.cpp:97): FP32 PE_REAL_MAX unless the scene sets one
    std::vector<float> life(n, 1e30f);
    w->finite_life.assign(n, 0);
    for (int i = 0; sc->lifetime && i < n; i++) {
        life[i] = (float)sc->lifetime[i];
        if (!(sc->lifetime[i] >= 1e30)) { w->finite_life[i] = 1; d.status_on = 1; }
    }
    w->has_joint.assign(n, 0);
    w->removed.assign(n, 0);
    if (hipMemcpyAsync(d.b.f, hf.data(), hf.size() * sizeof(float), hipMemcpyHostToDevice, w->stream) != hipSuccess ||
        hipMemcpyAsync(d.b.i, hi.data(), hi.size() * sizeof(int32_t), hipMemcpyHostToDevice, w->stream) != hipSuccess ||
        hipMemcpyAsync(d.st.life, life.data(), n * sizeof(float), hipMemcpyHostToDevice, w->stream) != hipSuccess) {
        pe_set_error("upload failed");
        return fail(PE_ERR_DEVICE);
    }
    for (void* p : {(void*)d.st.flags, (void*)d.st.sleep_time, (void*)d.st.last, (void*)d.st.scnt, (void*)d.st.dcnt,
                    (void*)d.st.report})
        if (hipMemsetAsync(p, 0, n * sizeof(int32_t), w->stream) != hipSuccess) { pe_set_error("upload failed"); return fail(PE_ERR_DEVICE); }
    if (hipMemsetAsync(d.ev_flag, 0, pcap * sizeof(int32_t), w->stream) != hipSuccess) { pe_set_error("upload failed"); return fail(PE_ERR_DEVICE); }
    hipLaunchKernelGGL(k_aabb_only, dim3(w->grid(n, 256)), dim3(256), 0, w->stream, d);
    for (auto& e : w->ev) hipEventCreate(&e);
    for (auto& e : w->order_ev) hipEventCreateWithFlags(&e, hipEventDisableTiming);
    {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_solve_flow, FLOW_THREADS, 0) != hipSuccess || per_cu < 1) {
            pe_set_error("cannot size the solver grid");
            return fail(PE_ERR_DEVICE);
        }
        if (hipFuncSetAttribute((const void*)k_solve_small, hipFuncAttributeMaxDynamicSharedMemorySize, SMALL_LDS) != hipSuccess) {
            pe_set_error("cannot size the small-world solver's LDS");
            return fail(PE_ERR_DEVICE);
        }
        w->device = dev;
        w->flow_max_blocks = cus * per_cu;
        w->flow_blocks = default_flow_blocks(n, w->flow_max_blocks);
        w->count_flow();
        if (w->alloc(&d.jp_hist, (size_t)FLOW_BINS * w->flow_max_blocks) != PE_OK) return fail(PE_ERR_DEVICE);
    }
    if (hipStreamSynchronize(w->stream) != hipSuccess) { pe_set_error("init sync failed"); return fail(PE_ERR_DEVICE); }
    *out = w;
    return PE_OK;
}

int pe_world_add_joints(pe_world* w, int32_t n, const pe_joint_desc* jd) {
    if (int rc = check_world(w)) return rc;
    if (n < 0 || (n > 0 && !jd) || (int64_t)w->joints.size() + n > 65536) { pe_set_error("pe_world_add_joints: invalid argument"); return PE_ERR_INVALID; }
    for (int k = 0; k < n; k++) {
        const pe_joint_desc& s = jd[k];
        if (s.type < PE_JOINT_BALL || s.type > PE_JOINT_SLIDER || s.body_a < 0 || s.body_a >= w->n || s.body_b < 0 ||
            s.body_b >= w->n || s.body_a == s.body_b) {
            pe_set_error("pe_world_add_joints: joint " + std::to_string(k) + " has an unknown type or invalid bodies");
            return PE_ERR_INVALID;
        }
        for (int x : {s.body_a, s.body_b})
            if (w->finite_life[x] || w->removed[x]) {
                pe_set_error("pe_world_add_joints: body " + std::to_string(x) + " has a finite lifetime or was removed");
                return PE_ERR_INVALID;
            }
    }
    for (int k = 0; k < n; k++) {
        const pe_joint_desc& s = jd[k];
        w->has_joint[s.body_a] = w->has_joint[s.body_b] = 1;
        JointDef j{};
        j.type = s.type; j.a = s.body_a; j.b = s.body_b;
        j.flags = (s.use_limits ? JF_LIMITS : 0) | (s.use_motor ? JF_MOTOR : 0);
        for (int c = 0; c < 3; c++) {
            j.anchor_a[c] = (float)s.anchor_a[c]; j.anchor_b[c] = (float)s.anchor_b[c];
            j.axis_a[c] = (float)s.axis_a[c]; j.axis_b[c] = (float)s.axis_b[c];
        }
        j.min_angle = (float)s.min_angle; j.max_angle = (float)s.max_angle; j.target_speed = (float)s.target_speed;
        w->joints.push_back(j);
    }
    // greedy colouring in joint order: joint k takes the lowest colour no earlier joint sharing a
    // dynamic body with it holds
    const int nj = (int)w->joints.size();
    std::vector<int> col(nj, 0), order;
    std::vector<std::vector<int>> body_cols(w->n);
    int ncol = 0;
    for (int k = 0; k < nj; k++) {
        std::vector<char> used(ncol + 1, 0);
        for (int x : {w->joints[k].a, w->joints[k].b})
            if (!w->kinematic[x]) for (int c : body_cols[x]) used[c] = 1;
        int c = 0;
        while (used[c]) c++;
        col[k] = c;
        ncol = std::max(ncol, c + 1);
        for (int x : {w->joints[k].a, w->joints[k].b})
            if (!w->kinematic[x]) body_cols[x].push_back(c);
    }
    std::vector<int32_t> jorder, jcs, jdeg(w->n, 0);
    std::vector<int2> jseq(nj, make_int2(0, 0));   // a joint's place in the sequence of its bodies' joints
    for (int c = 0; c < ncol; c++) {
        jcs.push_back((int32_t)jorder.size());
        for (int k = 0; k < nj; k++) {
            if (col[k] != c) continue;
            jorder.push_back(k);
            const int a = w->joints[k].a, b = w->joints[k].b;
            if (!w->kinematic[a]) jseq[k].x = jdeg[a]++;
            if (!w->kinematic[b]) jseq[k].y = jdeg[b]++;
        }
    }
    jcs.push_back((int32_t)jorder.size());
    PE_HIP(hipStreamSynchronize(w->stream));
    for (void*& p : w->joint_mem) if (p) { hipFree(p); p = nullptr; }
    const size_t bytes[6] = {nj * sizeof(JointDef), nj * sizeof(JointRow), nj * sizeof(int32_t), jcs.size() * sizeof(int32_t),
                             nj * sizeof(int2), jdeg.size() * sizeof(int32_t)};
    const void* src[6] = {w->joints.data(), nullptr, jorder.data(), jcs.data(), jseq.data(), jdeg.data()};
    for (int k = 0; k < 6; k++) {
        PE_HIP(hipMalloc(&w->joint_mem[k], std::max<size_t>(bytes[k], 16)));
        if (src[k] && bytes[k]) PE_HIP(hipMemcpy(w->joint_mem[k], src[k], bytes[k], hipMemcpyHostToDevice));
    }
    w->d.joints = (const JointDef*)w->joint_mem[0];
    w->d.jrows = (JointRow*)w->joint_mem[1];
    w->d.jorder = (const int32_t*)w->joint_mem[2];
    w->d.jcs = (const int32_t*)w->joint_mem[3];
    w->d.jseq = (const int2*)w->joint_mem[4];
    w->d.jdeg = (const int32_t*)w->joint_mem[5];
    w->d.njoints = nj;
    w->d.njcol = ncol;
    return PE_OK;
}

// Marks the bodies in ignore pairs (COLL_PARTNERS in their fourth shape parameter, unless they ignore
// every collision) and refreshes their AABB records.
__global__ void k_mark_partners(Dev d, const uint64_t* keys, int nkeys) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nkeys; k += gridDim.x * blockDim.x) {
        const int i = (int)(keys[k] >> 32), j = (int)(uint32_t)keys[k];
        for (int x : {i, j}) {
            float& f = d.b.at(F_SP + 3, x);
            if (f != COLL_IGNORE) f = COLL_PARTNERS;
            d.b.abr(x)[7] = f;
        }
    }
}

int pe_world_add_ignore_pairs(pe_world* w, int32_t n, const int32_t* pairs) {
    if (int rc = check_world(w)) return rc;
    if (n < 0 || (n > 0 && !pairs)) { pe_set_error("pe_world_add_ignore_pairs: invalid argument"); return PE_ERR_INVALID; }
    for (int k = 0; k < n; k++) {
        const int a = pairs[2 * k], b = pairs[2 * k + 1];
        if (a < 0 || a >= w->n || b < 0 || b >= w->n || a == b) { pe_set_error("pe_world_add_ignore_pairs: invalid body index"); return PE_ERR_INVALID; }
        w->ignore_keys.push_back((uint64_t)std::min(a, b) << 32 | (uint32_t)std::max(a, b));
    }
    std::sort(w->ignore_keys.begin(), w->ignore_keys.end());
    w->ignore_keys.erase(std::unique(w->ignore_keys.begin(), w->ignore_keys.end()), w->ignore_keys.end());
    PE_HIP(hipStreamSynchronize(w->stream));
    if (w->ignore_mem) { hipFree(w->ignore_mem); w->ignore_mem = nullptr; }
    const size_t bytes = w->ignore_keys.size() * sizeof(uint64_t);
    PE_HIP(hipMalloc(&w->ignore_mem, std::max<size_t>(bytes, 16)));
    if (bytes) PE_HIP(hipMemcpy(w->ignore_mem, w->ignore_keys.data(), bytes, hipMemcpyHostToDevice));
    w->d.sap.ignore = (const uint64_t*)w->ignore_mem;
    w->d.sap.nignore = (int)w->ignore_keys.size();
    if (!w->ignore_keys.empty())
        hipLaunchKernelGGL(k_mark_partners, dim3(w->grid((int)w->ignore_keys.size(), 256)), dim3(256), 0, w->stream, w->d,
                           (const uint64_t*)w->ignore_mem, (int)w->ignore_keys.size());
    PE_HIP(hipGetLastError());
    PE_HIP(hipStreamSynchronize(w->stream));
    return PE_OK;
}

static int read_counts(pe_world* w, DevCounts& c);

int pe_world_raycast(pe_world* w, int32_t nrays, const float* rays, int32_t nignore, const int32_t* ignore,
                     pe_ray_hit* out) {
    if (int rc = check_world(w)) return rc;
    if (nrays < 0 || nignore < 0 || (nrays > 0 && (!rays || !out)) || (nignore > 0 && !ignore) || nrays > (1 << 24)) {
        pe_set_error("pe_world_raycast: invalid argument");
        return PE_ERR_INVALID;
    }
    if (nrays == 0) return PE_OK;
    std::vector<int32_t> ig(ignore, ignore + nignore);
    std::sort(ig.begin(), ig.end());
    ig.erase(std::unique(ig.begin(), ig.end()), ig.end());
    pe_clear_stale_error();
    const size_t in_b = (size_t)nrays * RAY_IN * 4, ig_b = std::max<size_t>(ig.size(), 1) * 4, out_b = (size_t)nrays * RAY_OUT * 4;
    if (w->ray_bytes < in_b + ig_b + out_b + 512) {
        if (w->ray_mem) hipFree(w->ray_mem);
        w->ray_mem = nullptr;
        w->ray_bytes = 0;
        PE_HIP(hipMalloc(&w->ray_mem, in_b + ig_b + out_b + 512));
        w->ray_bytes = in_b + ig_b + out_b + 512;
    }
    char* base = (char*)w->ray_mem;
    float* d_rays = (float*)base;
    int32_t* d_ig = (int32_t*)(base + ((in_b + 255) & ~(size_t)255));
    float* d_out = (float*)(base + ((in_b + 255) & ~(size_t)255) + ((ig_b + 255) & ~(size_t)255));
    PE_HIP(hipMemcpyAsync(d_rays, rays, in_b, hipMemcpyHostToDevice, w->stream));
    if (!ig.empty()) PE_HIP(hipMemcpyAsync(d_ig, ig.data(), ig.size() * 4, hipMemcpyHostToDevice, w->stream));
    const int per_group = nrays >= RAYS_SHARED ? ray_share(w->has_mesh) : 1;
    hipLaunchKernelGGL(w->has_mesh ? k_raycast<true> : k_raycast<false>, dim3((nrays + per_group - 1) / per_group),
                       dim3(ray_threads(w->has_mesh)), 0, w->stream, w->d, (const float*)d_rays, nrays, per_group,
                       (const int32_t*)d_ig, (int)ig.size(), d_out);
    PE_HIP(hipGetLastError());
    std::vector<float> res((size_t)nrays * RAY_OUT);
    PE_HIP(hipMemcpyAsync(res.data(), d_out, out_b, hipMemcpyDeviceToHost, w->stream));
    PE_HIP(hipStreamSynchronize(w->stream));
    for (int k = 0; k < nrays; k++) {
        const float* e = &res[(size_t)k * RAY_OUT];
        pe_ray_hit& h = out[k];
        h.hit = e[0] != 0.0f ? 1 : 0;
        std::memcpy(&h.body, &e[1], 4);
        h.distance = e[2];
        for (int c = 0; c < 3; c++) { h.point[c] = e[3 + c]; h.normal[c] = e[6 + c]; }
    }
    return PE_OK;
}

int pe_world_set_sleep(pe_world* w, double lin_vel2, double ang_vel2, double time) {
    if (int rc = check_world(w)) return rc;
    w->d.st.lin2 = (float)lin_vel2;
    w->d.st.ang2 = (float)ang_vel2;
    w->d.st.tsleep = (float)time;
    if (lin_vel2 != 0.0 || ang_vel2 != 0.0) w->d.status_on = 1;
    return PE_OK;
}

int pe_world_remove_body(pe_world* w, int32_t body) {
    if (int rc = check_world(w)) return rc;
    if (body < 0 || body >= w->n) { pe_set_error("pe_world_remove_body: body index out of range"); return PE_ERR_INVALID; }
    if (w->has_joint[body]) { pe_set_error("pe_world_remove_body: the body has joints"); return PE_ERR_INVALID; }
    w->removed[body] = 1;
    w->d.status_on = 1;
    pe_clear_stale_error();
    hipLaunchKernelGGL(k_remove_body, dim3(1), dim3(1), 0, w->stream, w->d, (int)body);
    PE_HIP(hipGetLastError());
    return PE_OK;
}

int pe_world_get_body_status(pe_world* w, int32_t* flags, int32_t* static_count, int32_t* dynamic_count,
                             float* sleep_time) {
    if (int rc = check_world(w)) return rc;
    PE_HIP(hipStreamSynchronize(w->stream));
    const size_t bytes = (size_t)w->n * 4;
    if (flags) PE_HIP(hipMemcpy(flags, w->d.st.flags, bytes, hipMemcpyDeviceToHost));
    if (static_count) PE_HIP(hipMemcpy(static_count, w->d.st.scnt, bytes, hipMemcpyDeviceToHost));
    if (dynamic_count) PE_HIP(hipMemcpy(dynamic_count, w->d.st.dcnt, bytes, hipMemcpyDeviceToHost));
    if (sleep_time) PE_HIP(hipMemcpy(sleep_time, w->d.st.sleep_time, bytes, hipMemcpyDeviceToHost));
    return PE_OK;
}

int pe_world_set_collision_reports(pe_world* w, int32_t n, const int32_t* bodies, int32_t on) {
    if (int rc = check_world(w)) return rc;
    if (n < 0 || (n > 0 && !bodies)) { pe_set_error("pe_world_set_collision_reports: invalid argument"); return PE_ERR_INVALID; }
    for (int k = 0; k < n; k++)
        if (bodies[k] < 0 || bodies[k] >= w->n) { pe_set_error("pe_world_set_collision_reports: body index out of range"); return PE_ERR_INVALID; }
    PE_HIP(hipStreamSynchronize(w->stream));
    std::vector<int32_t> rep(w->n);
    PE_HIP(hipMemcpy(rep.data(), w->d.st.report, (size_t)w->n * 4, hipMemcpyDeviceToHost));
    for (int k = 0; k < n; k++) rep[bodies[k]] = on ? 1 : 0;
    PE_HIP(hipMemcpy(w->d.st.report, rep.data(), (size_t)w->n * 4, hipMemcpyHostToDevice));
    w->d.report_on = 0;
    for (int32_t r : rep) w->d.report_on |= r;
    return PE_OK;
}

int pe_world_get_collision_events(pe_world* w, int32_t cap, pe_collision_event* out, int32_t* count) {
    if (int rc = check_world(w)) return rc;
    if (cap < 0 || (cap > 0 && !out) || !count) { pe_set_error("pe_world_get_collision_events: invalid argument"); return PE_ERR_INVALID; }
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    const int np = std::min(c.npairs, w->d.pcap);
    int total = 0;
    if (w->d.report_on && np > 0) {
        std::vector<int32_t> flag(np);
        std::vector<float> ev((size_t)np * EVW);
        PE_HIP(hipMemcpy(flag.data(), w->d.ev_flag, (size_t)np * 4, hipMemcpyDeviceToHost));
        PE_HIP(hipMemcpy(ev.data(), w->d.events, ev.size() * 4, hipMemcpyDeviceToHost));
        for (int p = 0; p < np; p++) {
            if (!flag[p]) continue;
            if (total < cap) {
                const float* e = &ev[(size_t)p * EVW];
                pe_collision_event& o = out[total];
                std::memcpy(&o.body_a, &e[0], 4);
                std::memcpy(&o.body_b, &e[1], 4);
                for (int k = 0; k < 3; k++) { o.position[k] = e[2 + k]; o.normal[k] = e[5 + k]; o.velocity[k] = e[9 + k]; }
                o.depth = e[8];
            }
            total++;
        }
    }
    *count = total;
    return PE_OK;
}

int pe_world_destroy(pe_world* w) {
    delete w;
    return PE_OK;
}

int pe_world_step(pe_world* w, int32_t nsteps) {
    if (int rc = check_world(w)) return rc;
    for (int s = 0; s < nsteps; s++)
        if (int rc = w->step()) return rc;
    return PE_OK;
}
static int read_counts(pe_world* w, DevCounts& c) {
    PE_HIP(hipMemcpyAsync(&c, w->d.cnt, sizeof(c), hipMemcpyDeviceToHost, w->stream));
    PE_HIP(hipStreamSynchronize(w->stream));
    return PE_OK;
}
int pe_world_step_async(pe_world* w, int32_t nsteps, pe_stream_t stream) {
    if (int rc = check_world(w)) return rc;
    if (nsteps < 0) { pe_set_error("nsteps must be >= 0"); return PE_ERR_INVALID; }
    hipStream_t cs = (hipStream_t)stream;
    // the caller's stream first waits for the world's pending work ...
    PE_HIP(hipEventRecord(w->order_ev[0], w->stream));
    PE_HIP(hipStreamWaitEvent(cs, w->order_ev[0], 0));
    hipStream_t keep = w->stream;
    w->stream = cs;
    int rc = PE_OK;
    for (int s = 0; s < nsteps && rc == PE_OK; s++) rc = w->step();
    w->stream = keep;
    // ... and the world's later calls wait for the steps enqueued on it
    PE_HIP(hipEventRecord(w->order_ev[1], cs));
    PE_HIP(hipStreamWaitEvent(w->stream, w->order_ev[1], 0));
    return rc;
}
int pe_world_get_cache(pe_world* w, float* distances, int32_t cap, int32_t* prev_npairs) {
    if (int rc = check_world(w)) return rc;
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    if (prev_npairs) *prev_npairs = c.prev_npairs;
    const int m = std::min(cap, c.prev_npairs);
    if (distances && m > 0) PE_HIP(hipMemcpy(distances, w->d.ps.cd, (size_t)m * 8 * sizeof(float), hipMemcpyDeviceToHost));
    return PE_OK;
}
int pe_world_set_cache(pe_world* w, const float* distances, int32_t prev_npairs) {
    if (int rc = check_world(w)) return rc;
    if (prev_npairs < 0 || prev_npairs > w->d.pcap || (prev_npairs > 0 && !distances)) {
        pe_set_error("pe_world_set_cache: pair count beyond the world's pair capacity");
        return PE_ERR_INVALID;
    }
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    c.prev_npairs = prev_npairs;
    if (prev_npairs > 0)
        PE_HIP(hipMemcpy(w->d.ps.cd, distances, (size_t)prev_npairs * 8 * sizeof(float), hipMemcpyHostToDevice));
    PE_HIP(hipMemcpy(w->d.cnt, &c, sizeof(c), hipMemcpyHostToDevice));
    return PE_OK;
}
int pe_world_integrate(pe_world* w) {
    if (int rc = check_world(w)) return rc;
    pe_clear_stale_error();
    w->launch_integrate();
    PE_HIP(hipGetLastError());
    return PE_OK;
}
int pe_world_broadphase(pe_world* w, int32_t* npairs) {
    if (int rc = check_world(w)) return rc;
    pe_clear_stale_error();
    w->launch_broadphase();
    PE_HIP(hipGetLastError());
    if (npairs) {
        DevCounts c;
        PE_HIP(hipMemcpyAsync(&c, w->d.cnt, sizeof(c), hipMemcpyDeviceToHost, w->stream));
        PE_HIP(hipStreamSynchronize(w->stream));
        *npairs = c.npairs;
        if (int rc = report_overflow(w, c)) return rc;
    }
    return PE_OK;
}
int pe_world_narrowphase(pe_world* w) {
    if (int rc = check_world(w)) return rc;
    pe_clear_stale_error();
    w->launch_narrowphase();
    PE_HIP(hipGetLastError());
    return PE_OK;
}
int pe_world_solve(pe_world* w) {
    if (int rc = check_world(w)) return rc;
    pe_clear_stale_error();
    w->launch_solve();
    PE_HIP(hipGetLastError());
    return PE_OK;
}
int pe_world_sync(pe_world* w) {
    if (int rc = check_world(w)) return rc;
    PE_HIP(hipStreamSynchronize(w->stream));
    DevCounts c;
    PE_HIP(hipMemcpy(&c, w->d.cnt, sizeof(c), hipMemcpyDeviceToHost));
    return report_overflow(w, c);
}

static int get_field(pe_world* w, int f0, int nf, float* out) {
    const size_t S = w->stride;
    std::vector<float> tmp((size_t)nf * S);
    PE_HIP(hipMemcpyAsync(tmp.data(), w->d.b.f + (size_t)f0 * S, tmp.size() * sizeof(float), hipMemcpyDeviceToHost, w->stream));
    PE_HIP(hipStreamSynchronize(w->stream));
    for (int i = 0; i < w->n; i++)
        for (int k = 0; k < nf; k++) out[(size_t)i * nf + k] = tmp[(size_t)k * S + i];
    return PE_OK;
}
static int set_field(pe_world* w, int f0, int nf, const float* in) {
    const size_t S = w->stride;
    std::vector<float> tmp((size_t)nf * S);
    PE_HIP(hipMemcpyAsync(tmp.data(), w->d.b.f + (size_t)f0 * S, tmp.size() * sizeof(float), hipMemcpyDeviceToHost, w->stream));
    PE_HIP(hipStreamSynchronize(w->stream));
    for (int i = 0; i < w->n; i++)
        for (int k = 0; k < nf; k++) tmp[(size_t)k * S + i] = in[(size_t)i * nf + k];
    PE_HIP(hipMemcpyAsync(w->d.b.f + (size_t)f0 * S, tmp.data(), tmp.size() * sizeof(float), hipMemcpyHostToDevice, w->stream));
    PE_HIP(hipStreamSynchronize(w->stream));
    return PE_OK;
}

int pe_world_get_state(pe_world* w, float* pos, float* rot, float* v, float* av) {
    if (int rc = check_world(w)) return rc;
    int rc = PE_OK;
    if (pos && (rc = get_field(w, F_POS, 3, pos))) return rc;
    if (rot && (rc = get_field(w, F_ROT, 9, rot))) return rc;
    if (v && (rc = get_field(w, F_V, 3, v))) return rc;
    if (av && (rc = get_field(w, F_W, 3, av))) return rc;
    return PE_OK;
}
int pe_world_set_state(pe_world* w, const float* pos, const float* rot, const float* v, const float* av) {
    if (int rc = check_world(w)) return rc;
    int rc = PE_OK;
    if (pos && (rc = set_field(w, F_POS, 3, pos))) return rc;
    if (rot && (rc = set_field(w, F_ROT, 9, rot))) return rc;
    if (v && (rc = set_field(w, F_V, 3, v))) return rc;
    if (av && (rc = set_field(w, F_W, 3, av))) return rc;
    hipLaunchKernelGGL(k_aabb_only, dim3(w->grid(w->n, 256)), dim3(256), 0, w->stream, w->d);
    PE_HIP(hipStreamSynchronize(w->stream));
    return PE_OK;
}
int pe_world_get_aabbs(pe_world* w, float* mn, float* mx) {
    if (int rc = check_world(w)) return rc;
    int rc = PE_OK;
    if (mn && (rc = get_field(w, F_AMIN, 3, mn))) return rc;
    if (mx && (rc = get_field(w, F_AMAX, 3, mx))) return rc;
    return PE_OK;
}
int pe_world_get_pairs(pe_world* w, int32_t* pairs, int32_t cap, int32_t* npairs) {
    if (int rc = check_world(w)) return rc;
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    if (npairs) *npairs = c.npairs;
    const int m = std::min(cap, c.npairs);
    if (pairs && m > 0) {
        std::vector<int32_t> a(m), b(m);
        PE_HIP(hipMemcpy(a.data(), w->d.ps.pa, m * sizeof(int32_t), hipMemcpyDeviceToHost));
        PE_HIP(hipMemcpy(b.data(), w->d.ps.pb, m * sizeof(int32_t), hipMemcpyDeviceToHost));
        for (int i = 0; i < m; i++) { pairs[2 * i] = a[i]; pairs[2 * i + 1] = b[i]; }
    }
    return PE_OK;
}
int pe_world_get_contacts(pe_world* w, int32_t* npoints, float* points, int32_t cap) {
    if (int rc = check_world(w)) return rc;
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    const int m = std::min(cap, c.npairs);
    if (m <= 0) return PE_OK;
    std::vector<int32_t> np(m);
    PE_HIP(hipMemcpy(np.data(), w->d.ps.npts, m * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (npoints) std::copy(np.begin(), np.end(), npoints);
    if (points) {
        // slots at or beyond the point count are reported invalid; every slot's distance is reported
        std::vector<float> rec((size_t)m * 8 * CW), dist((size_t)m * 8);
        PE_HIP(hipMemcpy(rec.data(), w->d.ps.cp, rec.size() * sizeof(float), hipMemcpyDeviceToHost));
        PE_HIP(hipMemcpy(dist.data(), w->d.ps.cd, dist.size() * sizeof(float), hipMemcpyDeviceToHost));
        for (size_t s = 0; s < (size_t)m * 8; s++) {
            float* o = points + s * CF;
            const bool valid = (int)(s % 8) < np[s / 8];
            for (int f = 0; f < CW; f++) o[f] = valid ? rec[s * CW + f] : (f < 3 ? REAL_MAX : 0.0f);
            o[12] = dist[s];
        }
    }
    return PE_OK;
}
int pe_world_get_impulses(pe_world* w, float* impulses, int32_t cap) {
    if (int rc = check_world(w)) return rc;
    if (!impulses) { pe_set_error("null argument"); return PE_ERR_INVALID; }
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    const int m = std::min(cap, c.npairs);
    if (m <= 0) return PE_OK;
    std::vector<int32_t> np(m);
    std::vector<float> rows((size_t)m * 8 * RW);
    PE_HIP(hipMemcpy(np.data(), w->d.ps.npts, m * sizeof(int32_t), hipMemcpyDeviceToHost));
    PE_HIP(hipMemcpy(rows.data(), w->d.ps.rows, rows.size() * sizeof(float), hipMemcpyDeviceToHost));
    for (size_t s = 0; s < (size_t)m * 8; s++) {
        const bool valid = (int)(s % 8) < np[s / 8];
        for (int k = 0; k < 3; k++) impulses[s * 3 + k] = valid ? rows[s * RW + R_LN + k] : 0.0f;
    }
    return PE_OK;
}
int pe_world_get_solve_order(pe_world* w, int32_t* order, int32_t cap, int32_t* nordered, int32_t* color_start,
                             int32_t ccap, int32_t* ncolors) {
    if (int rc = check_world(w)) return rc;
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    if (nordered) *nordered = c.nordered;
    if (ncolors) *ncolors = c.ncolors;
    if (order && cap > 0 && c.nordered > 0)
        PE_HIP(hipMemcpy(order, w->d.order, std::min(cap, c.nordered) * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (color_start && ccap > 0)
        PE_HIP(hipMemcpy(color_start, w->d.color_start, std::min(ccap, c.ncolors + 1) * sizeof(int32_t), hipMemcpyDeviceToHost));
    return PE_OK;
}
int pe_world_get_axis(pe_world* w, int32_t* axis) {
    if (int rc = check_world(w)) return rc;
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    if (axis) *axis = c.axis;
    return PE_OK;
}
int pe_world_set_axis(pe_world* w, int32_t axis) {
    if (int rc = check_world(w)) return rc;
    if (axis < 0 || axis > 2) { pe_set_error("axis out of range"); return PE_ERR_INVALID; }
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    c.axis = axis;
    PE_HIP(hipMemcpy(w->d.cnt, &c, sizeof(c), hipMemcpyHostToDevice));
    return PE_OK;
}
int pe_world_set_timing(pe_world* w, int32_t enable) {
    if (int rc = check_world(w)) return rc;
    w->timing = enable != 0;
    return PE_OK;
}
int pe_world_get_stage_times(pe_world* w, double* ms) {
    if (int rc = check_world(w)) return rc;
    for (int k = 0; k < 4; k++) ms[k] = w->stage_ms[k];
    return PE_OK;
}
int pe_world_set_solver_blocks(pe_world* w, int32_t blocks) {
    if (int rc = check_world(w)) return rc;
    if (blocks < 0) { pe_set_error("blocks must be >= 0"); return PE_ERR_INVALID; }
    w->flow_blocks = blocks == 0 ? default_flow_blocks(w->n, w->flow_max_blocks) : std::min(blocks, w->flow_max_blocks);
    w->count_flow();
    return PE_OK;
}

int pe_world_set_colouring(pe_world* w, int32_t mode) {
    if (int rc = check_world(w)) return rc;
    if (mode < 0 || mode > 2 || (mode == 1 && w->n > CLAIM_MAX)) {
        pe_set_error("pe_world_set_colouring: mode 0, 1 (at most 12288 bodies) or 2");
        return PE_ERR_INVALID;
    }
    w->colouring = mode;
    w->count_flow();
    return PE_OK;
}

int pe_internal_set_flow_patience(pe_world* w, int64_t ticks) {
    if (int rc = check_world(w)) return rc;
    w->flow_patience = (uint64_t)std::max<int64_t>(ticks, 0);
    return PE_OK;
}

int pe_world_get_records(pe_world* w, float* aabb, float* body, float* solver) {
    if (int rc = check_world(w)) return rc;
    const size_t n = (size_t)w->n;
    PE_HIP(hipStreamSynchronize(w->stream));
    if (aabb) PE_HIP(hipMemcpy(aabb, w->d.b.ab, n * 8 * sizeof(float), hipMemcpyDeviceToHost));
    if (body) PE_HIP(hipMemcpy(body, w->d.b.cb, n * CBW * sizeof(float), hipMemcpyDeviceToHost));
    if (solver) PE_HIP(hipMemcpy(solver, w->d.b.sb, n * SBW * sizeof(float), hipMemcpyDeviceToHost));
    return PE_OK;
}

int pe_world_get_counts(pe_world* w, int64_t* counts) {
    if (int rc = check_world(w)) return rc;
    DevCounts c;
    if (int rc = read_counts(w, c)) return rc;
    counts[0] = w->n;
    counts[1] = w->n_dynamic;
    counts[2] = c.npairs;
    counts[3] = c.npoints;
    counts[4] = c.ncolors;
    counts[5] = c.jp_rounds;
    return PE_OK;
}

}  // extern "C"

// ====================================================================== stage entry points
// The three stage seams of the reference's World (broadphase, narrowphase, constraint solver) on
// a caller's device buffers and stream, so a host that keeps the reference's World can replace one
// stage at a time.  A pe_stage is a pe_world used as workspace: each call loads the caller's
// records into its body and pair stores, runs the same kernels as pe_world_step, and writes the
// results back to the caller's buffers; nothing is synchronised (the caller waits on its stream).
namespace {

// Collision records of the caller ([n][CBW]: basis, origin, AABB scale, shape parameters, shape
// type and kinematic flag as int bits, friction, restitution) into the body store; the shape type
// and kinematic flag also into the int fields the pair dispatch and the colouring read.
__global__ void k_stage_bodies(Dev d, const float* __restrict__ body, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float4* s = reinterpret_cast<const float4*>(body + (size_t)i * CBW);
        float4* o = reinterpret_cast<float4*>(d.b.cbr(i));
#pragma unroll
        for (int k = 0; k < CBW / 4; k++) o[k] = s[k];
        d.b.iat(I_TYPE, i) = __float_as_int(body[(size_t)i * CBW + CB_TYPE]);
        d.b.iat(I_KIN, i) = __float_as_int(body[(size_t)i * CBW + CB_KIN]) != 0 ? 1 : 0;
    }
}
// Solver records of the caller ([n][SBW]: inverse mass, kinematic flag, world inverse inertia,
// velocities; the temp velocities are ignored) into the body store, with the temp velocities set
// as SequentialImpulseSolver::setupSolver's clearTempVelocity sets them (the velocities, zero for a
// kinematic body).
__global__ void k_stage_solver_in(Dev d, const float* __restrict__ sb, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float r[SBW];
        ld_rec<SBW / 4>(sb + (size_t)i * SBW, r);
        const bool kin = r[SB_KIN] != 0.0f;
        for (int k = 0; k < 3; k++) {
            r[SB_TV + k] = kin ? 0.0f : r[SB_V + k];
            r[SB_TW + k] = kin ? 0.0f : r[SB_W + k];
        }
        r[SB_KIN] = kin ? 1.0f : 0.0f;
        if (kin) r[SB_IM] = 0.0f;
        st_rec<SBW / 4>(d.b.sbr(i), r);
        d.b.iat(I_KIN, i) = kin ? 1 : 0;
    }
}
// The solved velocities (syncTempVelocity) into the caller's solver records.
__global__ void k_stage_solver_out(Dev d, float* __restrict__ sb, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (d.b.iat(I_KIN, i)) continue;
        const float* t = d.b.sbr(i);
        float* o = sb + (size_t)i * SBW;
        for (int k = 0; k < 3; k++) {
            o[SB_V + k] = t[SB_TV + k];
            o[SB_W + k] = t[SB_TW + k];
        }
    }
}
// Pairs (and, for the solver, point counts and contact slots; for the narrowphase, the distances
// of the slots that survive from the previous call) into the pair store.
__global__ void k_stage_pairs(Dev d, const int32_t* __restrict__ pa, const int32_t* __restrict__ pb, int np, int prev,
                              const int32_t* __restrict__ npts, const float* __restrict__ points) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        d.cnt->npairs = np;
        d.cnt->prev_npairs = prev;
        d.cnt->nshape = 0;
        d.cnt->nsat = 0;
        d.cnt->npoints = 0;
        d.cnt->overflow = 0;
        d.cnt->nact = 0;
    }
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        d.ps.pa[p] = pa[p];
        d.ps.pb[p] = pb[p];
        if (npts) d.ps.npts[p] = npts[p];
        if (!points) continue;
        for (int k = 0; k < 8; k++) {
            const float* c = points + ((size_t)p * 8 + k) * CF;
            const size_t s = (size_t)p * 8 + k;
            if (npts) {
                if (k < npts[p])
                    for (int f = 0; f < CW; f++) d.ps.cp[s * CW + f] = c[f];
                d.ps.cd[s] = c[12];
            } else if (p < prev) {
                d.ps.cd[s] = c[12];
            }
        }
    }
}
// Contact results of the narrowphase into the caller's slots ([np][8][CF]: valid slots in cache
// order, invalid ones with the position at PE_REAL_MAX and their distance kept), point counts and
// swap flags.
__global__ void k_stage_contacts_out(Dev d, int np, float* __restrict__ points, int32_t* __restrict__ npts,
                                     int32_t* __restrict__ swap) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        const int m = d.ps.npts[p];
        if (npts) npts[p] = m;
        if (swap) swap[p] = d.ps.swap[p] & 1;
        for (int k = 0; k < 8; k++) {
            const size_t s = (size_t)p * 8 + k;
            float* o = points + s * CF;
            for (int f = 0; f < CW; f++) o[f] = k < m ? d.ps.cp[s * CW + f] : (f < 3 ? REAL_MAX : 0.0f);
            o[12] = d.ps.cd[s];
        }
    }
}
__global__ void k_stage_impulses_out(Dev d, int np, float* __restrict__ imp) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        const int m = d.ps.npts[p];
        for (int k = 0; k < 8; k++)
            for (int q = 0; q < 3; q++)
                imp[((size_t)p * 8 + k) * 3 + q] = k < m ? d.ps.rows[((size_t)p * 8 + k) * RW + R_LN + q] : 0.0f;
    }
}
__global__ void k_stage_result(Dev d, int32_t* result, int which) {
    result[0] = which == 0 ? d.cnt->overflow : d.cnt->ncolors;
    if (which == 1) result[1] = d.cnt->overflow;
}

// A sweep over a caller's AABB records ([n][8]) with the given working memory and pair outputs.
// result[0] = pairs found (more than the capacity when it overflowed), result[1] = the next axis, result[2] =
// capacity-error bits.
SapView sap_over_records(const SapView& work, int n, const float* aabb, int axis, int32_t* pa, int32_t* pb, int cap,
                         int32_t* result) {
    SapView s = work;
    s.n = n;
    s.amin = aabb;
    s.amax = aabb + 4;
    s.fs = 1;
    s.bs = 8;
    s.rec = aabb;
    s.pa = pa;
    s.pb = pb;
    s.pcap = cap;
    s.axis_in = axis;
    s.result = result;
    return s;
}

int stage_grid(int work, int block) { return std::max(1, std::min((work + block - 1) / block, 4096)); }

}  // namespace

struct pe_stage {
    pe_world* w = nullptr;
    int max_bodies = 0, max_pairs = 0;
    ~pe_stage() { delete w; }
};

extern "C" {

int pe_stage_create(int32_t max_bodies, int32_t max_pairs, pe_stage** out) {
    if (!out || max_bodies < 1 || max_pairs < 1) { pe_set_error("pe_stage_create: invalid argument"); return PE_ERR_INVALID; }
    // the workspace is a world of max_bodies unit spheres (their state is overwritten by each call)
    std::vector<int32_t> type(max_bodies, PE_SHAPE_SPHERE), kin(max_bodies, 1);
    std::vector<double> param(4 * (size_t)max_bodies, 0.0), mass(max_bodies, 1.0), zero3(3 * (size_t)max_bodies, 0.0),
        rot(9 * (size_t)max_bodies, 0.0), mu(max_bodies, 0.5), e(max_bodies, 0.0);
    for (int i = 0; i < max_bodies; i++) {
        param[4 * (size_t)i] = 1.0;
        rot[9 * (size_t)i] = rot[9 * (size_t)i + 4] = rot[9 * (size_t)i + 8] = 1.0;
    }
    pe_scene_desc sc{};
    sc.n = max_bodies;
    sc.shape_type = type.data();
    sc.shape_param = param.data();
    sc.mass = mass.data();
    sc.position = zero3.data();
    sc.rotation = rot.data();
    sc.linear_velocity = zero3.data();
    sc.angular_velocity = zero3.data();
    sc.friction = mu.data();
    sc.restitution = e.data();
    sc.kinematic = kin.data();
    pe_world_params prm{1.0 / 60.0, {0.0, 0.0, 0.0}, 10};
    auto* S = new pe_stage();
    if (int rc = pe_world_create(&sc, &prm, max_pairs, &S->w)) { delete S; return rc; }
    if (max_bodies > SMALL_MAX) {   // it may be handed worlds of those sizes
        if (int rc = S->w->alloc_rows()) { delete S; return rc; }
    }
    S->w->has_shapes = true;
    S->max_bodies = max_bodies;
    S->max_pairs = max_pairs;
    *out = S;
    return PE_OK;
}

int pe_stage_destroy(pe_stage* s) {
    delete s;
    return PE_OK;
}

int pe_stage_set_meshes(pe_stage* s, int32_t n_meshes, const pe_mesh_desc* meshes, const int32_t* concave,
                        int32_t prepared) {
    if (!s || n_meshes < 0 || (n_meshes > 0 && (!meshes || !concave))) { pe_set_error("invalid argument"); return PE_ERR_INVALID; }
    HostMeshes hm;
    for (int k = 0; k < n_meshes; k++)
        if (hm.add(meshes[k], concave[k] != 0, nullptr, nullptr, prepared != 0) < 0) return PE_ERR_INVALID;
    pe_world* w = s->w;
    PE_HIP(hipStreamSynchronize(w->stream));
    w->meshes.release();
    if (int rc = w->meshes.upload(hm, w->stream)) return rc;
    PE_HIP(hipStreamSynchronize(w->stream));
    w->d.b.ms = w->meshes.view();
    return PE_OK;
}

int pe_stage_broadphase(pe_stage* s, int32_t n, const float* aabb, int32_t axis, int32_t* pair_a, int32_t* pair_b,
                        int32_t cap, int32_t* result, pe_stream_t stream) {
    if (!s || n < 0 || n > s->max_bodies || axis < 0 || axis > 2 || cap < 0 || !result || (n > 0 && !aabb) ||
        (cap > 0 && (!pair_a || !pair_b))) {
        pe_set_error("pe_stage_broadphase: invalid argument");
        return PE_ERR_INVALID;
    }
    pe_clear_stale_error();
    hipStream_t st = (hipStream_t)stream;
    const SapView v = sap_over_records(s->w->d.sap, n, aabb, axis, pair_a, pair_b, cap, result);
    if (n >= 2) sap_launch(v, st);   // fewer than 2 bodies: no pairs, the axis stays (broad_phase_sweep_and_prune.cpp:8)
    else hipLaunchKernelGGL(k_sap_none, dim3(1), dim3(1), 0, st, v);
    PE_HIP(hipGetLastError());
    return PE_OK;
}

int pe_stage_narrowphase(pe_stage* s, int32_t n, const float* body, int32_t npairs, const int32_t* pair_a,
                         const int32_t* pair_b, int32_t prev_npairs, float* points, int32_t* npoints, int32_t* swap,
                         int32_t* result, pe_stream_t stream) {
    if (!s || n < 1 || n > s->max_bodies || npairs < 0 || npairs > s->max_pairs || prev_npairs < 0 ||
        prev_npairs > s->max_pairs || !body || !result || (npairs > 0 && (!pair_a || !pair_b || !points))) {
        pe_set_error("pe_stage_narrowphase: invalid argument");
        return PE_ERR_INVALID;
    }
    pe_clear_stale_error();
    pe_world* w = s->w;
    hipStream_t keep = w->stream;
    w->stream = (hipStream_t)stream;
    w->n = n;
    w->d.b.n = n;
    hipLaunchKernelGGL(k_stage_bodies, dim3(stage_grid(n, 256)), dim3(256), 0, w->stream, w->d, body, (int)n);
    hipLaunchKernelGGL(k_stage_pairs, dim3(stage_grid(npairs, 256)), dim3(256), 0, w->stream, w->d, pair_a, pair_b,
                       (int)npairs, (int)prev_npairs, (const int32_t*)nullptr, (const float*)points);
    w->launch_narrowphase();
    if (npairs > 0)
        hipLaunchKernelGGL(k_stage_contacts_out, dim3(stage_grid(npairs, 128)), dim3(128), 0, w->stream, w->d,
                           (int)npairs, points, npoints, swap);
    hipLaunchKernelGGL(k_stage_result, dim3(1), dim3(1), 0, w->stream, w->d, result, 0);
    w->stream = keep;
    PE_HIP(hipGetLastError());
    return PE_OK;
}

int pe_stage_solve(pe_stage* s, int32_t n, const float* body, float* solver_body, int32_t npairs, const int32_t* pair_a,
                   const int32_t* pair_b, const int32_t* npoints, const float* points, float dt, int32_t iterations,
                   float* impulses, int32_t* result, pe_stream_t stream) {
    if (!s || n < 1 || n > s->max_bodies || npairs < 0 || npairs > s->max_pairs || !body || !solver_body || !result ||
        iterations < 0 || (npairs > 0 && (!pair_a || !pair_b || !npoints || !points))) {
        pe_set_error("pe_stage_solve: invalid argument");
        return PE_ERR_INVALID;
    }
    pe_clear_stale_error();
    pe_world* w = s->w;
    hipStream_t keep = w->stream;
    w->stream = (hipStream_t)stream;
    w->n = n;
    w->d.b.n = n;
    w->d.dt = dt;
    w->d.iterations = iterations;
    w->flow_blocks = default_flow_blocks(n, w->flow_max_blocks);
    hipLaunchKernelGGL(k_stage_bodies, dim3(stage_grid(n, 256)), dim3(256), 0, w->stream, w->d, body, (int)n);
    hipLaunchKernelGGL(k_stage_solver_in, dim3(stage_grid(n, 256)), dim3(256), 0, w->stream, w->d, (const float*)solver_body, (int)n);
    hipLaunchKernelGGL(k_stage_pairs, dim3(stage_grid(npairs, 256)), dim3(256), 0, w->stream, w->d, pair_a, pair_b,
                       (int)npairs, 0, npoints, points);
    int rc = w->launch_solve();
    if (rc == PE_OK) {
        hipLaunchKernelGGL(k_stage_solver_out, dim3(stage_grid(n, 256)), dim3(256), 0, w->stream, w->d, solver_body, (int)n);
        if (impulses && npairs > 0)
            hipLaunchKernelGGL(k_stage_impulses_out, dim3(stage_grid(npairs, 128)), dim3(128), 0, w->stream, w->d,
                               (int)npairs, impulses);
        hipLaunchKernelGGL(k_stage_result, dim3(1), dim3(1), 0, w->stream, w->d, result, 1);
    }
    w->stream = keep;
    if (rc != PE_OK) return rc;
    PE_HIP(hipGetLastError());
    return PE_OK;
}

}  // extern "C"
