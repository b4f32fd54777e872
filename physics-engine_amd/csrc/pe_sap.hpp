// Sweep-and-prune broadphase over n AABBs on the whole GPU (BroadPhaseSweepAndPrune::
// calcCollisionPairs, broad_phase_sweep_and_prune.cpp:6-41), shared by the single-world pipeline
// (its body store) and the stage entry points (a caller's AABB records):
//   k_sap_rank           up to SAP_RANK_MAX bodies: stable sort of (aabb_min[axis] + 0, index) by counting,
//                        or k_sap_keys + radix, a stable LSD sort in 4 passes of 8 bits; both leave the
//                        AABB records in sorted order; beside them the next axis's partial sums
//   k_sap_runs           16 or 64 sorted bodies per workgroup (a block): their candidate runs (j > i with
//                        min_j <= max_i), cut into units of 64 candidates
//   k_sap_test           a wave per unit tests its candidates, a lane each (up to SAP_FUSED_MAX bodies
//                        k_sap_runs does so itself)
//   k_sap_emit           the pairs that passed, in the reference's (i, j) sweep order; the next axis =
//                        argmax variance of AABB centres (FP64, fixed blocks)
#pragma once
#include "pe_common.hpp"
#include "pe_prims.hpp"

namespace pe {

struct DevCounts {          // device-side counters of one step
    int32_t npairs;         // pairs emitted by the broadphase (clamped to capacity)
    int32_t prev_npairs;    // pairs of the previous narrowphase (contact slots that survive)
    int32_t axis;           // SAP axis for the next sort
    int32_t overflow;       // sticky capacity-error bits (OVF_*), cleared when the host reports them
    uint32_t nchunk_pairs;  // pairs counted by the sweep (unclamped)
    int32_t ncolors;
    int32_t nordered;       // pairs in the solve order
    int32_t npoints;        // contact points of the last narrowphase
    uint32_t nunits;        // units of candidates handed out to the workgroups of the sweep
    uint32_t bar_count;     // grid barrier: arrivals (0 between barriers)
    uint32_t bar_gen;       // grid barrier: generation
    int32_t nshape;         // pairs of this narrowphase that involve a cylinder or a mesh ...
    int32_t nsat;           // ... of which these run the polyhedral separating-axis routine
    int32_t ncomp;          // ... and these involve a compound body
    int32_t nact;           // pairs the solve orders (contact points, not both bodies kinematic)
    int32_t nrows;          // their contact points, where the host asks for them
    int32_t jp_ncol;        // colours the last sweep over the GPU counted
    uint32_t adj_total;     // colouring: adjacency entries
    uint32_t fl_arrive;     // solve over the GPU: workgroups that have started,
    uint32_t fl_state;      // whether all have in time (FLOW_*),
    uint32_t fl_exit;       // and workgroups that left when not
    int32_t jp_heavy;       // bodies in more than JP_HEAVY pairs,
    int32_t jp_maxdeg;      // the most pairs one of them is in,
    uint32_t jp_words;      // words of their colour sets,
    int32_t jp_fall;        // and whether those are more than there are
    int32_t jp_rounds;      // colouring over the GPU: the most times a thread tried its pairs
};
// Capacity errors, OR-ed into DevCounts::overflow by the step that hits them and kept until the
// host reads and reports them: a result that lost pairs or contact points is never returned as a
// success.
constexpr int OVF_PAIRS = 1;         // the broadphase found more pairs than the pair capacity
constexpr int OVF_CHUNKS = 4;        // the sweep had more candidates than its chunk capacity
constexpr int OVF_CLIP = 8;          // a clipped polygon outgrew its buffer (contact points lost)
constexpr int OVF_STALL = 16;        // the solver gave up a wait (not a capacity: a fault of this program)

// Sorted bodies per workgroup of the sweep: few where its workgroups also test their candidates (FUSED); else more, since
// each takes its units' numbers from one counter, 12 ns after the other (50 000 bodies in blocks of 16: 78 us of
// that, in blocks of 64: 16), and sums up the pairs of those before it.  16 lanes search a run.
constexpr int sap_block(bool fused) { return fused ? 16 : 64; }
constexpr int sap_threads(bool fused) { return 16 * sap_block(fused); }
// Threads of k_sap_emit: 50 000 bodies whose pairs lie along the sort axis take it 67 / 48 / 45 us with 256 / 512 / 1024.
constexpr int sap_emit_threads(bool fused) { return fused ? 256 : 512; }
// Sorted bodies per counter of pairs, which k_sap_test's waves add to (with one per 64 bodies it took 30 us for the 10 000
// boxes at rest, with one per 16 22).
constexpr int SAP_SUB = 16;
constexpr int SAP_UNIT = 64;         // candidates per unit
constexpr int SAP_CHUNK = 32;        // the workspace is sized in chunks of this many candidates
// Units for at most `chunks` chunks of candidates over n bodies' runs.
__host__ __device__ constexpr int64_t sap_units(int64_t chunks, int64_t n) { return chunks * SAP_CHUNK / SAP_UNIT + n + 1; }
constexpr int SAP_RED_THREADS = 256;
constexpr int SAP_RED_VALUES = 7;   // axis reduction: centre sums (3), squared sums (3), bodies

// The AABBs and the working memory of one sweep.  AABB minimum k of body i is
// amin[k * fs + i * bs] (field-major SoA: fs = stride, bs = 1; records: fs = 1, bs = 8); rec holds
// one 8-float record per body: min xyz, kinematic flag, max xyz, ignore-collision flag (non-zero:
// the body is in no pair), read by the sweep's pair test.
struct SapView {
    int n;
    const float* amin;
    const float* amax;
    int fs, bs;
    const float* rec;
    uint32_t* keys;         // [n] x 2 radix buffers
    uint32_t* vals;
    uint32_t* keys2;
    uint32_t* vals2;
    float* skey;            // [n] sorted keys as floats
    float* srec;            // [n][8] the AABB records in sorted order
    uint32_t* end;          // [n] per sorted body: the end of its run
    uint32_t* first;        // [n] and its first unit
    uint32_t* blk;          // [sap_blocks(n)] per block its units
    uint2* sub;             // [sap_subs(n)] per SAP_SUB sorted bodies: candidates, pairs
    uint32_t* owner;        // [sap_units(chunk_cap, n)] per unit its sorted body
    uint64_t* unit_hit;     // [sap_units(chunk_cap, n)] per unit, bit k: its candidate k is a pair
    uint32_t* hist;         // [256 * radix_blocks(n)] radix histograms
    double* red;            // [6 * red_blocks(n)] axis reduction partials
    DevCounts* cnt;
    int32_t* pa;            // [pcap] pair output: body A, body B (sorted position order)
    int32_t* pb;
    int pcap;
    int chunk_cap;          // at most this many times SAP_CHUNK candidates
    int axis_in;            // the sort axis (-1: the one in cnt, left by the last sweep)
    int32_t* result;        // [3] or null: pairs found, next axis, capacity-error bits
    const uint64_t* ignore; // [nignore] sorted keys (lo << 32 | hi) of body pairs that never collide
    int nignore;
    __device__ __forceinline__ int ax() const { return axis_in >= 0 ? axis_in : cnt->axis; }
    __device__ __forceinline__ float mn(int k, int i) const { return amin[(size_t)k * fs + (size_t)i * bs]; }
    __device__ __forceinline__ float mx(int k, int i) const { return amax[(size_t)k * fs + (size_t)i * bs]; }
};

__host__ inline int sap_radix_blocks(int n) { return (n + RS_TILE - 1) / RS_TILE; }
__host__ inline int sap_red_blocks(int n) { return n < 1 ? 1 : (n + SAP_RED_THREADS - 1) / SAP_RED_THREADS < 256 ? (n + SAP_RED_THREADS - 1) / SAP_RED_THREADS : 256; }
__host__ __device__ constexpr int sap_subs(int n) { return (n + sap_block(false) - 1) / sap_block(false) * (sap_block(false) / SAP_SUB); }
__host__ __device__ constexpr int sap_blocks(int n, bool fused = true) { return (n + sap_block(fused) - 1) / sap_block(fused); }

// BroadPhaseBase::validateCollisionPair (broad_phase_base.cpp:5-19) on two AABB records: the
// ignore-collision flags, both kinematic, then closed-interval overlap on x, y, z.  Ignore-id pairs
// (broad_phase_base.cpp:12-13) are tested by sap_pair_allowed.
__device__ __forceinline__ bool sap_pair_ok(const float (&A)[8], const float (&B)[8]) {
    if (A[7] == COLL_IGNORE || B[7] == COLL_IGNORE) return false;
    if (A[3] != 0.0f && B[3] != 0.0f) return false;
    if (A[0] > B[4] || B[0] > A[4]) return false;
    if (A[1] > B[5] || B[1] > A[5]) return false;
    if (A[2] > B[6] || B[2] > A[6]) return false;
    return true;
}
// sap_pair_ok, then for two bodies that both have ignore partners, the ignore-pair list (binary
// search of the pair's key).
__device__ __forceinline__ bool sap_pair_allowed(const SapView& s, const float (&A)[8], const float (&B)[8], int i, int j) {
    if (!sap_pair_ok(A, B)) return false;
    if (A[7] != COLL_PARTNERS || B[7] != COLL_PARTNERS) return true;
    const uint64_t key = i < j ? ((uint64_t)i << 32 | (uint32_t)j) : ((uint64_t)j << 32 | (uint32_t)i);
    int lo = 0, hi = s.nignore;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (s.ignore[mid] < key) lo = mid + 1; else hi = mid;
    }
    return !(lo < s.nignore && s.ignore[lo] == key);
}
__device__ __forceinline__ void sap_ld_rec(const float* src, float (&dst)[8]) {
    const float4* s = reinterpret_cast<const float4*>(src);
    const float4 a = s[0], b = s[1];
    dst[0] = a.x; dst[1] = a.y; dst[2] = a.z; dst[3] = a.w;
    dst[4] = b.x; dst[5] = b.y; dst[6] = b.z; dst[7] = b.w;
}
// The record of the body at sorted position q (contiguous loads along a run of candidates).
__device__ __forceinline__ void sap_ld_sorted(const SapView& s, int q, float (&dst)[8]) { sap_ld_rec(s.srec + (size_t)q * 8, dst); }
// sap_pair_allowed for the bodies at sorted positions qa and qb (their indices are loaded only
// for the ignore-pair search).
__device__ __forceinline__ bool sap_pair_allowed_sorted(const SapView& s, const float (&A)[8], const float (&B)[8],
                                                        int qa, int qb) {
    if (!sap_pair_ok(A, B)) return false;
    if (A[7] != COLL_PARTNERS || B[7] != COLL_PARTNERS) return true;
    return sap_pair_allowed(s, A, B, (int)s.vals[qa], (int)s.vals[qb]);
}

// A sweep over fewer than two bodies through a stage entry point: no pairs, the axis stays.
static __global__ void k_sap_none(SapView s) {
    s.cnt->axis = s.axis_in;
    s.cnt->overflow = 0;
    s.cnt->npairs = 0;
    s.cnt->nchunk_pairs = 0;
    s.result[0] = 0;
    s.result[1] = s.axis_in;
    s.result[2] = 0;
}
// Clears what the sweep counts (a given axis: a stage entry point, whose last call's errors are dropped).
__device__ __forceinline__ void sap_begin(const SapView& s) {
    s.cnt->nunits = 0;
    if (s.axis_in >= 0) s.cnt->overflow = 0;
}
__device__ __forceinline__ void sap_sorted(const SapView& s, uint32_t q, int i, float key) {
    s.skey[q] = key;
    const float4* src = reinterpret_cast<const float4*>(s.rec + (size_t)i * 8);
    float4* dst = reinterpret_cast<float4*>(s.srec + (size_t)q * 8);
    dst[0] = src[0];
    dst[1] = src[1];
}

// Next SAP axis (broad_phase_sweep_and_prune.cpp:37-40): variance of AABB centres, reduced in
// FP64 over fixed blocks (deterministic), argmax with the reference's tie rule.
// A body whose AABB is empty (min > max) has left the world (World::removeRigidBody, an ended
// lifetime): it sorts last with an infinite key, has no candidates and is not in the variance; with
// fewer than two bodies left the axis stays (the reference's sweep returns early).
// The partial sums of block b of nb (SAP_RED_THREADS threads of the workgroup work).
__device__ __forceinline__ void sap_axis_partial(const SapView& s, int b, int nb, double (&sh)[SAP_RED_VALUES][SAP_RED_THREADS]) {
    const int t = threadIdx.x;
    if (t < SAP_RED_THREADS) {
        double acc[SAP_RED_VALUES] = {0, 0, 0, 0, 0, 0, 0};
        for (int i = b * SAP_RED_THREADS + t; i < s.n; i += nb * SAP_RED_THREADS) {
            if (!(s.mn(0, i) <= s.mx(0, i))) continue;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float c = (s.mn(k, i) + s.mx(k, i)) * 0.5f;
                acc[k] += (double)c;
                acc[3 + k] += (double)(c * c);
            }
            acc[6] += 1.0;
        }
#pragma unroll
        for (int k = 0; k < SAP_RED_VALUES; k++) sh[k][t] = acc[k];
    }
    __syncthreads();
    for (int o = SAP_RED_THREADS / 2; o > 0; o >>= 1) {
        if (t < o)
#pragma unroll
            for (int k = 0; k < SAP_RED_VALUES; k++) sh[k][t] += sh[k][t + o];
        __syncthreads();
    }
    if (t < SAP_RED_VALUES) s.red[t * nb + b] = sh[t][0];
}
// The axis from the nb partial sums, by one wave (lane k adds up value k, in block order); returned by
// every lane (-1: it stays).
__device__ __forceinline__ int sap_axis_final(const SapView& s, int nb) {
    const int lane = threadIdx.x & (WAVE - 1);
    double t = 0;
    if (lane < SAP_RED_VALUES) {
        const double* r = s.red + lane * nb;
        int b = 0;
        for (; b + 8 <= nb; b += 8) {   // eight loads in flight, added in order
            double x[8];
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = r[b + j];
#pragma unroll
            for (int j = 0; j < 8; j++) t += x[j];
        }
        for (; b < nb; b++) t += r[b];
    }
    const double cnt = __shfl(t, 6, WAVE);
    double v[3];
    for (int k = 0; k < 3; k++) {
        const double m = __shfl(t, k, WAVE), q = __shfl(t, 3 + k, WAVE);
        v[k] = q - m * m / cnt;
    }
    if (cnt < 2.0) return -1;
    int axis = 0;
    if (v[1] > v[0]) axis = 1;
    if (v[2] > v[axis]) axis = 2;
    return axis;
}

// Stable sort by counting: a body's sorted position is the number of bodies with a smaller key, or an equal
// one and a lower index.  SAP_RANK_BODIES bodies per workgroup, a lane each, the other keys split over its
// waves: n^2 / 64 wave steps of about two instructions, spread over the whole GPU -- 777 bodies 9 us, 10 000 30, in
// one launch, where the radix sort's twelve cost 4.5 us each in a stream whatever they do.  The whole sweep with one / the
// other: 2 000 bodies 27 / 68 us, 10 000 54 / 93, 16 000 79 / 105, 20 000 113 / 117, 30 000 169 / 152.
// The workgroups from nrank on make the axis's partial sums.
constexpr int SAP_RANK_MAX = 16384;
constexpr int SAP_RANK_BODIES = WAVE, SAP_RANK_THREADS = 512, SAP_RANK_TILE = 2048;
static __global__ void __launch_bounds__(SAP_RANK_THREADS) k_sap_rank(SapView s, int nrank) {
    __shared__ double sh[SAP_RED_VALUES][SAP_RED_THREADS];
    if ((int)blockIdx.x >= nrank) {
        sap_axis_partial(s, blockIdx.x - nrank, gridDim.x - nrank, sh);
        return;
    }
    __shared__ __align__(16) uint32_t tile[SAP_RANK_TILE];
    __shared__ int part[SAP_RANK_THREADS / WAVE][WAVE];
    const int ax = s.ax(), n = s.n;
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    const int i0 = blockIdx.x * SAP_RANK_BODIES, i = i0 + lane;
    if (blockIdx.x == 0 && threadIdx.x == 0) sap_begin(s);
    const float key = i < n ? s.mn(ax, i) + 0.0f : 0.0f;
    const uint32_t ki = float_key(key);
    int count = 0;
    for (int base = 0; base < n; base += SAP_RANK_TILE) {
        const int m = min(SAP_RANK_TILE, n - base);
        __syncthreads();
        for (int j = threadIdx.x; j < m; j += SAP_RANK_THREADS) tile[j] = float_key(s.mn(ax, base + j) + 0.0f);
        __syncthreads();
        const int per = ((m + SAP_RANK_THREADS / WAVE - 1) / (SAP_RANK_THREADS / WAVE) + 3) & ~3;
        const int j0 = min(m, w * per), j1 = min(m, j0 + per);
        // before the workgroup's own bodies an equal key counts, after them it does not
        const int own0 = min(max(i0 - base, j0), j1), own1 = min(max(i0 + SAP_RANK_BODIES - base, j0), j1);
        auto run = [&](int a, int b, bool equal) {
            int j = a;
            for (; j < b && (j & 3); j++) count += equal ? tile[j] <= ki : tile[j] < ki;
#pragma unroll 4
            for (; j + 4 <= b; j += 4) {
                const uint4 k = *reinterpret_cast<const uint4*>(&tile[j]);
                if (equal) count += (k.x <= ki) + (k.y <= ki) + (k.z <= ki) + (k.w <= ki);
                else count += (k.x < ki) + (k.y < ki) + (k.z < ki) + (k.w < ki);
            }
            for (; j < b; j++) count += equal ? tile[j] <= ki : tile[j] < ki;
        };
        run(j0, own0, true);
        for (int j = own0; j < own1; j++) count += tile[j] < ki || (tile[j] == ki && base + j < i);
        run(own1, j1, false);
    }
    part[w][lane] = count;
    __syncthreads();
    if (w != 0 || i >= n) return;
    uint32_t q = 0;
#pragma unroll
    for (int k = 0; k < SAP_RANK_THREADS / WAVE; k++) q += (uint32_t)part[k][lane];
    s.vals[q] = (uint32_t)i;
    sap_sorted(s, q, i, key);
}

// The radix sort's keys; the workgroups from nkeys on make the axis's partial sums.
static __global__ void __launch_bounds__(SAP_RED_THREADS) k_sap_keys(SapView s, int nkeys) {
    __shared__ double sh[SAP_RED_VALUES][SAP_RED_THREADS];
    if ((int)blockIdx.x >= nkeys) {
        sap_axis_partial(s, blockIdx.x - nkeys, gridDim.x - nkeys, sh);
        return;
    }
    const int ax = s.ax();
    if (blockIdx.x == 0 && threadIdx.x == 0) sap_begin(s);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < s.n; i += nkeys * blockDim.x) {
        s.keys[i] = float_key(s.mn(ax, i) + 0.0f);
        s.vals[i] = (uint32_t)i;
    }
}
// After the radix sort: the sorted float keys and records.
static __global__ void k_sap_gather(SapView s) {
    const int ax = s.ax();
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < s.n; q += gridDim.x * blockDim.x) {
        const int i = (int)s.vals[q];
        sap_sorted(s, q, i, s.mn(ax, i) + 0.0f);
    }
}

// First sorted position in [lo, hi) whose key is above m, hi if none: the binary search, four of its levels a
// step on 16 lanes (lane l of a group has node l of the levels' tree in heap order), so a run's end costs
// a quarter of the dependent loads.  The same for the 16 lanes.
__device__ __forceinline__ int sap_search(const float* skey, int lo, int hi, float m) {
    const int l = threadIdx.x & 15;
    while (__any(lo < hi)) {
        int a = lo, b = hi;
        const int depth = 31 - __clz(l | 1);
        for (int k = depth - 1; k >= 0; k--) {
            const int mid = (a + b) >> 1;
            if (a < b) {
                if ((l >> k) & 1) a = mid + 1; else b = mid;
            }
        }
        const bool above = l > 0 && a < b && skey[(a + b) >> 1] > m;
        const uint32_t g = (uint32_t)(__ballot(above) >> (threadIdx.x & 48)) & 0xffffu;
        for (int k = 0, node = 1; k < 4; k++) {
            if (lo >= hi) break;
            const int mid = (lo + hi) >> 1;
            if ((g >> node) & 1) { hi = mid; node = 2 * node; } else { lo = mid + 1; node = 2 * node + 1; }
        }
    }
    return lo;
}
// Tests unit k of sorted body q (its run ends before `end`), a lane per candidate -- neighbouring lanes read
// neighbouring records -- and leaves the outcomes in unit_hit[u]; the number of pairs.
__device__ __forceinline__ int sap_test_unit(const SapView& s, uint32_t u, int q, int k, int end) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int j = q + 1 + k * SAP_UNIT + lane;
    bool ok = false;
    if (j < end) {
        float A[8], B[8];
        sap_ld_sorted(s, q, A);
        sap_ld_sorted(s, j, B);
        ok = sap_pair_allowed_sorted(s, A, B, q, j);
    }
    const uint64_t hit = __ballot(ok);
    if (lane == 0) s.unit_hit[u] = hit;
    return (int)__popcll(hit);
}
// The candidate runs of a block's sorted bodies (the reference's sweep breaks at the first key above a body's
// maximum) and their units, numbered from a common counter.  FUSED: the workgroup tests them itself, which
// saves a launch while the longest run (of a ground: every body) stays short; else k_sap_test spreads
// all units over the GPU (10 000 boxes at rest: with every workgroup testing its own, the ground's run alone
// took 40 us).
constexpr int SAP_FUSED_MAX = 2048;
template <bool FUSED>
static __global__ void __launch_bounds__(sap_threads(FUSED)) k_sap_runs(SapView s) {
    constexpr int BLOCK = sap_block(FUSED), THREADS = sap_threads(FUSED);
    static_assert(BLOCK == (FUSED ? SAP_SUB : WAVE), "a lane per body, and whole counters");
    __shared__ uint32_t s_len[BLOCK], s_unit[BLOCK + 1], s_base;
    __shared__ int s_pairs;
    const int n = s.n, q0 = blockIdx.x * BLOCK, nq = min(BLOCK, n - q0);
    const int tid = threadIdx.x, r = tid >> 4, q = q0 + r;
    const float m = r < nq ? s.srec[(size_t)q * 8 + 4 + s.ax()] : 0.0f;
    const int end = sap_search(s.skey, r < nq ? q + 1 : n, n, m);
    if ((tid & 15) == 0) s_len[r] = r < nq ? (uint32_t)(end - q - 1) : 0u;
    __syncthreads();
    uint32_t cand = 0;   // of the lane's SAP_SUB bodies
    if (tid < WAVE) {
        const uint32_t len = tid < BLOCK ? s_len[tid] : 0u, units = (len + SAP_UNIT - 1) / SAP_UNIT;
        uint32_t incl = units;
        cand = len;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, WAVE);
            if (tid >= o) incl += y;
            if (o < SAP_SUB) cand += __shfl_xor(cand, o, WAVE);
        }
        if (!FUSED && tid % SAP_SUB == 0) s.sub[blockIdx.x * (BLOCK / SAP_SUB) + tid / SAP_SUB] = make_uint2(cand, 0u);
        if (tid < BLOCK) s_unit[tid] = incl - units;
        if (tid == BLOCK - 1) {
            s_unit[BLOCK] = incl;
            s_base = atomicAdd(&s.cnt->nunits, incl);
            s_pairs = 0;
        }
    }
    __syncthreads();
    // the units beyond the workspace are dropped (an error that k_sap_emit reports)
    const uint32_t slots = (uint32_t)sap_units(s.chunk_cap, n), base = s_base;
    const uint32_t units = base >= slots ? 0u : min(s_unit[BLOCK], slots - base);
    if (r < nq) {
        if ((tid & 15) == 0) {
            s.end[q] = (uint32_t)end;
            s.first[q] = base + s_unit[r];
        }
        if (!FUSED)
            for (uint32_t u = s_unit[r] + (tid & 15); u < s_unit[r + 1] && u < units; u += 16) s.owner[base + u] = (uint32_t)q;
    }
    if (FUSED) {
        int pairs = 0, o = 0;   // o: the run of the wave's unit
        for (uint32_t u = tid / WAVE; u < units; u += THREADS / WAVE) {
            while (s_unit[o + 1] <= u) o++;
            pairs += sap_test_unit(s, base + u, q0 + o, (int)(u - s_unit[o]), q0 + o + 1 + (int)s_len[o]);
        }
        if ((tid & (WAVE - 1)) == 0 && pairs) atomicAdd(&s_pairs, pairs);
        __syncthreads();
    }
    if (tid == 0) {
        s.blk[blockIdx.x] = units;
        if (FUSED) s.sub[blockIdx.x] = make_uint2(cand, (uint32_t)s_pairs);
    }
}
static __global__ void __launch_bounds__(256) k_sap_test(SapView s) {
    const uint32_t units = min(s.cnt->nunits, (uint32_t)sap_units(s.chunk_cap, s.n));
    const uint32_t wave = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE, nw = gridDim.x * (blockDim.x / WAVE);
    for (uint32_t u = wave; u < units; u += nw) {
        const int q = (int)s.owner[u];
        const int pairs = sap_test_unit(s, u, q, (int)(u - s.first[q]), (int)s.end[q]);
        if ((threadIdx.x & (WAVE - 1)) == 0 && pairs) atomicAdd(&s.sub[q / SAP_SUB].y, (uint32_t)pairs);
    }
}

// The pairs of a block's bodies after those of the blocks before it; the last workgroup knows all of them and sets
// the counts and the next axis from its nred partial sums.
template <bool FUSED>
static __global__ void __launch_bounds__(sap_emit_threads(FUSED)) k_sap_emit(SapView s, int nred) {
    constexpr int BLOCK = sap_block(FUSED), THREADS = sap_emit_threads(FUSED), SUBS = BLOCK / SAP_SUB;
    __shared__ uint32_t s_unit[BLOCK];
    __shared__ int wsum[THREADS / WAVE + 1];
    __shared__ unsigned long long s_cand;
    const int tid = threadIdx.x, q0 = blockIdx.x * BLOCK, nq = min(BLOCK, s.n - q0);
    const bool last = blockIdx.x + 1 == gridDim.x;
    const uint32_t units = s.blk[blockIdx.x], base = s.first[q0];
    uint32_t own = 0;
    uint64_t own_cand = 0;
#pragma unroll
    for (int g = 0; g < SUBS; g++) {
        const uint2 o = s.sub[blockIdx.x * SUBS + g];
        own += o.y;
        own_cand += o.x;
    }
    int before = 0;
    uint64_t cand = 0;
    for (int b = tid; b < (int)blockIdx.x * SUBS; b += THREADS) {
        const uint2 o = s.sub[b];
        before += (int)o.y;
        if (!FUSED) cand += o.x;
    }
    if (tid < nq) s_unit[tid] = s.first[q0 + tid] - base;
    if (!FUSED && tid == 0) s_cand = own_cand;
    int carry;
    block_exclusive_scan(before, wsum, &carry);
    if (!FUSED && last) {
        if (cand) atomicAdd(&s_cand, (unsigned long long)cand);
        __syncthreads();
    }
    if (last && tid < WAVE) {
        const int axis = sap_axis_final(s, nred);
        if (tid == 0) {
            const uint32_t total = (uint32_t)carry + own;
            int32_t ovf = 0;
            // (SAP_FUSED_MAX bodies form fewer candidates than any workspace holds)
            if (!FUSED && s_cand > (uint64_t)s.chunk_cap * SAP_CHUNK) ovf |= OVF_CHUNKS;
            if (total > (uint32_t)s.pcap) ovf |= OVF_PAIRS;
            ovf |= s.cnt->overflow;
            s.cnt->overflow = ovf;
            s.cnt->nchunk_pairs = total;
            s.cnt->npairs = total > (uint32_t)s.pcap ? s.pcap : (int32_t)total;
            if (axis >= 0) s.cnt->axis = axis;
            else if (s.axis_in >= 0) s.cnt->axis = s.axis_in;
            if (s.result) {
                s.result[0] = (int32_t)total;
                s.result[1] = s.cnt->axis;
                s.result[2] = ovf;
            }
        }
    }
    if (own == 0) return;
    for (uint32_t u0 = 0; u0 < units; u0 += THREADS) {
        const uint32_t u = u0 + tid;
        uint64_t hit = u < units ? s.unit_hit[base + u] : 0ull;
        int tot;
        uint32_t out = (uint32_t)(carry + block_exclusive_scan((int)__popcll(hit), wsum, &tot));
        carry += tot;
        if (hit == 0) continue;
        int r = 0;   // the last of the runs that start at or before this unit (empty runs share their starts)
#pragma unroll
        for (int k = BLOCK / 2; k > 0; k >>= 1) r = r + k < nq && s_unit[r + k] <= u ? r + k : r;
        const int a = (int)s.vals[q0 + r], j0 = q0 + r + 1 + (int)(u - s_unit[r]) * SAP_UNIT;
        for (; hit; hit &= hit - 1, out++) {
            if ((int)out >= s.pcap) break;
            s.pa[out] = a;
            s.pb[out] = (int)s.vals[j0 + __ffsll((unsigned long long)hit) - 1];
        }
    }
}

// The whole sweep on stream st (no host synchronisation): pairs to s.pa / s.pb, their count and
// the next axis to s.cnt (and s.result).  n >= 1.
inline void sap_launch(const SapView& s, hipStream_t st) {
    const int n = s.n;
    const int nred = sap_red_blocks(n);
    if (n <= SAP_RANK_MAX) {
        const int nrank = (n + SAP_RANK_BODIES - 1) / SAP_RANK_BODIES;
        hipLaunchKernelGGL(k_sap_rank, dim3(nrank + nred), dim3(SAP_RANK_THREADS), 0, st, s, nrank);
    } else {
        const int rsb = sap_radix_blocks(n), nk = (n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256;
        hipLaunchKernelGGL(k_sap_keys, dim3(nk + nred), dim3(SAP_RED_THREADS), 0, st, s, nk);
        uint32_t *ki = s.keys, *vi = s.vals, *ko = s.keys2, *vo = s.vals2;
        for (int pass = 0; pass < 4; pass++) {
            hipLaunchKernelGGL(k_radix_hist, dim3(rsb), dim3(RS_THREADS), 0, st, ki, n, pass * 8, s.hist, rsb);
            hipLaunchKernelGGL(k_scan_u32, dim3(1), dim3(1024), 0, st, s.hist, 256 * rsb, (uint32_t*)nullptr);
            hipLaunchKernelGGL(k_radix_scatter, dim3(rsb), dim3(RS_THREADS), 0, st, ki, vi, ko, vo, n, pass * 8, s.hist, rsb);
            uint32_t* t = ki; ki = ko; ko = t;
            t = vi; vi = vo; vo = t;
        }
        // after 4 passes the sorted data is back in keys / vals
        hipLaunchKernelGGL(k_sap_gather, dim3(nk), dim3(256), 0, st, s);
    }
    if (n <= SAP_FUSED_MAX) {
        hipLaunchKernelGGL(k_sap_runs<true>, dim3(sap_blocks(n, true)), dim3(sap_threads(true)), 0, st, s);
        hipLaunchKernelGGL(k_sap_emit<true>, dim3(sap_blocks(n, true)), dim3(sap_emit_threads(true)), 0, st, s, nred);
    } else {
        hipLaunchKernelGGL(k_sap_runs<false>, dim3(sap_blocks(n, false)), dim3(sap_threads(false)), 0, st, s);
        hipLaunchKernelGGL(k_sap_test, dim3(2048), dim3(256), 0, st, s);
        hipLaunchKernelGGL(k_sap_emit<false>, dim3(sap_blocks(n, false)), dim3(sap_emit_threads(false)), 0, st, s, nred);
    }
}

}  // namespace pe
