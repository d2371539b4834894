// Multi-source BFS: up to 64 sources advance together, one bit per source in a
// 64-bit mask per vertex (frontier, visited, next).
//
// No reference counterpart: "MBFS" in the reference is multi-GPU BFS
// (HowToBuild:13); the semantics here are those of k independent BFS runs
// (Algorithm/UserOperators.h:17-36 per source), checked against exactly that.
//
// Superstep:
//   push: active vertices (frontier mask != 0) OR their mask into next[v] of every
//         out-neighbour that still lacks some of those bits (64-bit atomicOr); vertices
//         up to `large` out-degree go through the wave-cooperative queue, hubs above it
//         are split over whole workgroups (the threshold is autotunable);
//   pull: every vertex not yet visited by all sources ORs the frontier masks of its
//         in-neighbours, stopping early once every missing bit has been found; vertices are
//         visited in in-degree order over ELL slabs of source ids (the pull layout), so the
//         index loads are coalesced;
//   update: new = next & ~visited; visited |= new; frontier = new; the level of the new bits goes
//         into bit planes (plane p holds bit p of every (vertex, source) level); the two active
//         queues and the counters are rebuilt with ballot + in-workgroup prefix scan;
//   finish: once, after the last superstep: the planes as one level byte per (source, vertex).
//
// Drivers as for BFS: device-driven (the last workgroup of each update writes the next superstep
// into a control block; batches of supersteps are captured as hipGraphs and replayed until done,
// the first batch sized by the previous run on the handle, and each ends with the finish, which
// returns at once unless the run is done) and host-driven (timing or tracing) over the same kernels.

#include <algorithm>
#include <cstring>

#include "engine.h"
#include "sched.h"

namespace medusa {

constexpr uint32_t kMbfsLargeDefault = 1024;
constexpr uint32_t kMbfsGridDefault = 2048;
constexpr uint32_t kMbfsBatch = 8;
constexpr uint32_t kMbfsSplit = 8;  // minimum workgroup items per hub

constexpr uint32_t kMbfsProbeLines = 8;

// Sums of an update, on lines of their own.
enum { kMbfsActive, kMbfsActiveDeg, kMbfsNewBits, kMbfsReachedEdges, kMbfsLargeDeg, kMbfsSums };
struct MbfsLine {
    alignas(128) unsigned long long v;
};
struct MbfsCounters {
    MDS_COUNTER(uint32_t, n_small);   // active vertices with 1 <= outdeg <= large
    MDS_COUNTER(uint32_t, n_large);   // active vertices with outdeg > large
    MDS_COUNTER(uint32_t, ticket);    // workgroups of the update that are done
    MbfsLine sum[kMbfsSums];
    MbfsLine probes[kMbfsProbeLines];  // in-edges examined, by workgroup number
};

struct MbfsCtl {
    int32_t step;
    uint32_t pull, done, n_small, n_large, hub_wgs, mode, saturated;
    uint32_t supersteps, push_steps, pull_steps, k;
    unsigned long long n, m, n_f, m_f, n_u, m_u, reached, reached_edges, kernel_bytes, alg_bytes, full;
    uint8_t* out;  // where the finish of a device-driven run writes the levels, or null
};

struct MbfsArgs {
    const uint32_t *row_ptr, *col, *cptr, *csrc;
    uint32_t *q_small, *q_large;
    unsigned long long *visited, *frontier, *next;
    const PrRun* runs;
    const uint32_t *wg_run, *perm, *ell;
    MbfsCounters* ctr;
    MbfsCtl* ctl;
    const float* policy;
    void* planes;  // kMbfsPlanes of n words each, of the width that holds k bits
    uint32_t n, large, items, grid;
};
constexpr uint32_t kMbfsPlanes = 8;

// Masks cleared, counters and control block set up.
__global__ __launch_bounds__(256) void k_mbfs_fill(MbfsArgs a, unsigned long long m, uint32_t k, uint32_t mode,
                                                   uint8_t* out) {
    const uint64_t tid = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    // visited, frontier and next follow each other
    for (uint64_t i = tid; i < 3ull * a.n; i += stride) a.visited[i] = 0;
    if (blockIdx.x != 0) return;
    for (uint32_t i = threadIdx.x; i < sizeof(MbfsCounters) / 8; i += blockDim.x)
        reinterpret_cast<unsigned long long*>(a.ctr)[i] = 0;
    if (threadIdx.x == 0) {
        MbfsCtl z{};
        z.mode = mode;
        z.n = a.n;
        z.m = m;
        z.k = k;
        z.n_u = (unsigned long long)a.n * k;
        z.m_u = m * k;
        z.full = k == 64 ? ~0ull : ((1ull << k) - 1);
        z.out = out;
        *a.ctl = z;
    }
}

// Workgroups of a push expansion given to the hub queue (as for BFS).
__host__ __device__ inline uint32_t mbfs_hub_wgs(uint32_t grid, uint32_t n_small, uint32_t n_large,
                                                 unsigned long long deg_large, unsigned long long deg_sum) {
    if (!n_large) return 0;
    if (!n_small) return grid;
    unsigned long long h = deg_sum ? (unsigned long long)grid * deg_large / deg_sum : 1ull;
    if (h < 1) h = 1;
    if (h > grid - 1) h = grid - 1;
    return (uint32_t)h;
}

// ---- superstep bodies ---------------------------------------------------------------

// Wave-cooperative push; wave w of the nwaves taking part holds queue entries
// w, w + nwaves, ... one per lane.
__device__ __forceinline__ void mbfs_push_small(const uint32_t* __restrict__ q, uint32_t qn,
                                                const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col,
                                                const unsigned long long* __restrict__ frontier,
                                                const unsigned long long* __restrict__ visited,
                                                unsigned long long* __restrict__ next, uint32_t wave0, uint32_t nwaves) {
    __shared__ uint32_t s_beg[4][kWave], s_off[4][kWave];
    __shared__ unsigned long long s_mask[4][kWave];
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    for (uint64_t r = 0; wave0 + r * kWave * nwaves < qn; ++r) {  // uniform across the wave
        const uint64_t i = wave0 + (r * kWave + lane) * nwaves;
        uint32_t beg = 0, deg = 0;
        unsigned long long fm = 0;
        if (i < qn) {
            const uint32_t u = q[i];
            beg = row_ptr[u];
            deg = row_ptr[u + 1] - beg;
            fm = frontier[u];
        }
        const uint32_t incl = wave_incl_scan(deg);
        const uint32_t total = __shfl(incl, kWave - 1, kWave);
        s_beg[wv][lane] = beg;
        s_off[wv][lane] = incl - deg;
        s_mask[wv][lane] = fm;
        __builtin_amdgcn_wave_barrier();
        for (uint32_t e = lane; e < total; e += kWave) {
            uint32_t lo = 0;
#pragma unroll
            for (uint32_t step = kWave / 2; step; step >>= 1)
                if (s_off[wv][lo + step] <= e) lo += step;
            const uint32_t v = col[s_beg[wv][lo] + (e - s_off[wv][lo])];
            const unsigned long long add = s_mask[wv][lo] & ~visited[v];
            if (add && (next[v] & add) != add) atomicOr(&next[v], add);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Hubs: each queue vertex split into `split` edge ranges, one per workgroup item.
__device__ __forceinline__ void mbfs_push_large(const uint32_t* __restrict__ q, uint32_t qn,
                                                const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col,
                                                const unsigned long long* __restrict__ frontier,
                                                const unsigned long long* __restrict__ visited,
                                                unsigned long long* __restrict__ next, uint32_t wg0, uint32_t nwg) {
    uint32_t split = nwg / qn;
    split = split < kMbfsSplit ? kMbfsSplit : (split > 4096u ? 4096u : split);
    for (uint64_t w = wg0; w < (uint64_t)qn * split; w += nwg) {
        const uint32_t u = q[w / split], part = (uint32_t)(w % split);
        const uint32_t b = row_ptr[u], deg = row_ptr[u + 1] - b;
        const unsigned long long fm = frontier[u];
        const uint32_t per = (deg + split - 1) / split;
        const uint32_t lo = b + min(deg, part * per), hi = b + min(deg, (part + 1) * per);
        for (uint32_t k = lo + threadIdx.x; k < hi; k += blockDim.x) {
            const uint32_t v = col[k];
            const unsigned long long add = fm & ~visited[v];
            if (add && (next[v] & add) != add) atomicOr(&next[v], add);
        }
    }
}

constexpr uint32_t kMbfsPullGroup = 4;  // in-edges a lane probes per round

// Bottom-up over the pull layout: a vertex missing some sources ORs its in-neighbours'
// frontier masks until every missing bit is found.  Work item w of the layout is 256
// lane-vertices of one equal-in-degree run (their k-th sources are one coalesced ELL load;
// kMbfsPullGroup in-edges per round, loads issued together, merged one by one with the same
// early exit and probe count as a plain loop) or 4 wave-vertices of in-degree > 64 (the wave
// scans 64 in-edges per step and ORs them by shuffles).  Workgroups stride over the items.
// `probes` counts in-edges examined up to and including the last one needed.
__device__ __forceinline__ void mbfs_pull_ell(unsigned long long full, const PrRun* __restrict__ runs,
                                              const uint32_t* __restrict__ wg_run, uint32_t items,
                                              const uint32_t* __restrict__ perm, const uint32_t* __restrict__ ell,
                                              const uint32_t* __restrict__ cptr, const uint32_t* __restrict__ csrc,
                                              const unsigned long long* __restrict__ frontier,
                                              const unsigned long long* __restrict__ visited,
                                              unsigned long long* __restrict__ next, MbfsCounters* __restrict__ ctr) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    unsigned long long probes = 0;
    for (uint32_t w = blockIdx.x; w < items; w += gridDim.x) {  // uniform per block
        const PrRun R = runs[wg_run[w]];
        const uint32_t local = w - R.wg_begin;
        if (R.kind == kPrWave) {
            const uint32_t p = R.begin + local * 4 + wave;
            if (p >= R.begin + R.count) continue;  // uniform across the wave
            const uint32_t v = perm[p];
            const unsigned long long vis = visited[v];
            if (vis == full) continue;
            const uint32_t vb = cptr[v], ve = cptr[v + 1];
            unsigned long long acc = 0;
            for (uint32_t k0 = vb; k0 < ve; k0 += kWave) {
                const uint32_t k = k0 + lane;
                unsigned long long x = k < ve ? frontier[csrc[k]] : 0ull;
#pragma unroll
                for (int off = kWave / 2; off >= 1; off >>= 1) x |= __shfl_xor(x, off, kWave);
                acc |= x;
                if (lane == 0) probes += min(ve - k0, (uint32_t)kWave);
                if ((acc | vis) == full) break;
            }
            acc &= ~vis;
            if (lane == 0 && acc) next[v] = acc;
            continue;
        }
        const uint32_t i = local * 256 + threadIdx.x;
        if (i >= R.count) continue;
        const uint32_t v = perm[R.begin + i];
        const unsigned long long vis = visited[v];
        if (vis == full) continue;
        const uint32_t* col = ell + R.ell_base + i;
        const uint32_t deg = R.deg, st = R.ell_stride;
        unsigned long long acc = 0;
        bool all = false;
        for (uint32_t k0 = 0; k0 < deg && !all; k0 += kMbfsPullGroup) {
            uint32_t u[kMbfsPullGroup];
            unsigned long long f[kMbfsPullGroup];
#pragma unroll
            for (uint32_t j = 0; j < kMbfsPullGroup; ++j) u[j] = k0 + j < deg ? col[(size_t)(k0 + j) * st] : 0u;
#pragma unroll
            for (uint32_t j = 0; j < kMbfsPullGroup; ++j) f[j] = k0 + j < deg ? frontier[u[j]] : 0ull;
#pragma unroll
            for (uint32_t j = 0; j < kMbfsPullGroup; ++j) {
                if (all || k0 + j >= deg) continue;
                acc |= f[j];
                ++probes;
                all = (acc | vis) == full;
            }
        }
        acc &= ~vis;
        if (acc) next[v] = acc;
    }
    // one atomic per workgroup (every wave of the block reaches this point)
    __shared__ unsigned long long s_probe[4];
    probes = wave_sum_u64(probes);
    if (lane == 0) s_probe[threadIdx.x / kWave] = probes;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long t = s_probe[0] + s_probe[1] + s_probe[2] + s_probe[3];
        if (t) atomicAdd(&ctr->probes[blockIdx.x % kMbfsProbeLines].v, t);
    }
}

__global__ __launch_bounds__(256) void k_mbfs_expand(MbfsArgs a) {
    const MbfsCtl* ctl = a.ctl;
    if (ctl->done) return;
    if (ctl->pull) {
        mbfs_pull_ell(ctl->full, a.runs, a.wg_run, a.items, a.perm, a.ell, a.cptr, a.csrc, a.frontier, a.visited,
                      a.next, a.ctr);
        return;
    }
    const uint32_t hub = ctl->hub_wgs;
    if (blockIdx.x < hub) {
        mbfs_push_large(a.q_large, ctl->n_large, a.row_ptr, a.col, a.frontier, a.visited, a.next, blockIdx.x, hub);
        return;
    }
    const uint32_t wg = blockIdx.x - hub, nwg = gridDim.x - hub;
    mbfs_push_small(a.q_small, ctl->n_small, a.row_ptr, a.col, a.frontier, a.visited, a.next,
                    wg * 4 + threadIdx.x / kWave, nwg * 4);
}

// Direction of the next superstep, by one wave: fixed, learned, or the direction-optimising
// heuristic.
__device__ __forceinline__ bool mbfs_direction(const MbfsCtl& c, bool pull, const float* __restrict__ policy,
                                               float* s_params) {
    if (c.mode == 1) return false;
    if (c.mode == 2) return true;
    const bool plain = !pull ? (double)c.m_f > (double)c.m_u / Sched::kAlphaMbfs
                             : !((double)c.n_f < (double)c.n / Sched::kBeta);
    if (c.mode != 3 || !policy ||
        !bfs_policy_consulted(pull, (double)c.n_f, (double)c.m_f, (double)c.m_u, (double)c.n, Sched::kAlphaMbfs,
                              Sched::kBeta))
        return plain;
    const double rec[MEDUSA_TRACE_FIELDS] = {(double)c.step, (double)c.n_f, (double)c.m_f, (double)c.n_u,
                                             (double)c.m_u, (double)c.n, (double)c.m, 0.0, 0.0};
    float c_push, c_pull;
    policy_direction_costs_wave(rec, policy, s_params, c_push, c_pull);
    return policy_pull(c_push, c_pull, plain);
}

// One wave, after every workgroup of an update (or the start, when `first`) has added its counters:
// folds them into the control block, decides the next superstep and clears them.
__device__ __forceinline__ void mbfs_decide(const MbfsArgs& a, bool first, float* s_params) {
    MbfsCounters* ctr = a.ctr;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t n_small = load_now(&ctr->n_small), n_large = load_now(&ctr->n_large);
    unsigned long long sum[kMbfsSums];
#pragma unroll
    for (int i = 0; i < kMbfsSums; ++i) sum[i] = load_now(&ctr->sum[i].v);
    const unsigned long long probe = lane < kMbfsProbeLines ? load_now(&ctr->probes[lane].v) : 0ull;
    MbfsCtl c = load_now_block(a.ctl);
    const unsigned long long probes = wave_sum_u64(probe);
    const unsigned long long n = c.n;
    if (!first) {
        // byte model of the superstep just finished: push = queue + offsets + mask per active
        // vertex, col + visited + next probe per edge; pull = offsets + visited per vertex,
        // source + frontier mask per probe; update = 24n
        const unsigned long long kb = c.pull ? 4ull * (n + 1) + 8ull * n + 12ull * probes
                                             : 20ull * c.n_f + 20ull * c.m_f;
        c.kernel_bytes += kb;
        c.alg_bytes += kb + 24ull * n + sum[kMbfsNewBits];
        c.supersteps += 1;
        if (c.pull) c.pull_steps += 1; else c.push_steps += 1;
        c.step += 1;
    }
    const unsigned long long n_active = sum[kMbfsActive];
    if (c.step >= 255 && n_active) c.saturated = 1;
    c.reached += sum[kMbfsNewBits];
    c.reached_edges += sum[kMbfsReachedEdges];
    c.n_u -= sum[kMbfsNewBits];
    c.m_u -= sum[kMbfsReachedEdges];
    c.n_f = n_active;
    c.m_f = sum[kMbfsActiveDeg];
    c.n_small = n_small;
    c.n_large = n_large;
    c.hub_wgs = mbfs_hub_wgs(a.grid, n_small, n_large, sum[kMbfsLargeDeg], c.m_f);
    if (n_active == 0) c.done = 1;
    c.pull = !c.done && mbfs_direction(c, first ? false : c.pull != 0, a.policy, s_params) ? 1u : 0u;
    if (lane == 0) {
        *a.ctl = c;
        ctr->n_small = ctr->n_large = ctr->ticket = 0;
    }
    if (lane < kMbfsSums) ctr->sum[lane].v = 0;
    if (lane < kMbfsProbeLines) ctr->probes[lane].v = 0;
}

struct MbfsSources {
    uint32_t v[64];
};

// The k sources (any of them repeated) at level 0: masks, queues and counters; one workgroup of one
// wave.  `decide`: and the first decision.
__global__ __launch_bounds__(kWave) void k_mbfs_start(MbfsArgs a, MbfsSources src, uint32_t k, uint32_t decide) {
    __shared__ float s_params[kMlpWaveLds];
    const uint32_t lane = threadIdx.x;
    const uint32_t v = lane < k ? src.v[lane] : 0xFFFFFFFFu;  // (vertices are below 2^32 - 1)
    unsigned long long mask = 0;
    for (uint32_t j = 0; j < k; ++j)
        if (v == (uint32_t)__builtin_amdgcn_readlane(v, j)) mask |= 1ull << j;
    const bool one = lane < k && (uint32_t)__builtin_ctzll(mask) == lane;  // the first of its vertex
    uint32_t deg = 0;
    if (one) {
        deg = a.row_ptr[v + 1] - a.row_ptr[v];
        a.frontier[v] = mask;
        a.visited[v] = mask;
    }
    const bool large = deg > a.large, small = deg > 0 && !large;
    const unsigned long long sm = __ballot(small), lm = __ballot(large);
    if (small) a.q_small[lanes_below(sm)] = v;
    if (large) a.q_large[lanes_below(lm)] = v;
    const unsigned long long sum[kMbfsSums] = {(unsigned long long)__popcll(__ballot(one)), wave_sum_u64(deg), k,
                                               wave_sum_u64((unsigned long long)__popcll(mask) * deg),
                                               wave_sum_u64(large ? deg : 0u)};
    if (lane == 0) {
        MbfsCounters* ctr = a.ctr;
        __hip_atomic_store(&ctr->n_small, (uint32_t)__popcll(sm), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ctr->n_large, (uint32_t)__popcll(lm), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < kMbfsSums; ++i)
            __hip_atomic_store(&ctr->sum[i].v, sum[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!decide) return;
    __threadfence();
    mbfs_decide(a, true, s_params);
}

constexpr uint32_t kMbfsWg = 1024, kMbfsTile = 4 * kMbfsWg;  // vertices per workgroup tile (4 chunks per wave)

// new = next & ~visited for every vertex: masks, level planes, the two active queues, counters.
// kDecide: the last workgroup to add its counters decides the next superstep (one launch less per
// superstep, 5 us).  Bound by its passes over next and frontier and the joins' plane words, and on
// few vertices by the chain of atomics on each counter, hence workgroups of 1024 threads: 256 chains
// of one add for 2^20 vertices.  Levels go into bit planes: as one byte store per joining (source,
// vertex) with the wave's other lanes masked, this kernel took 36..46 us in the five supersteps of RMAT-20
// with 64 sources that join most, and 20..24 with planes.
template <class T, bool kDecide>
__global__ __launch_bounds__(kMbfsWg) void k_mbfs_update(MbfsArgs a, int32_t level_fixed) {
    constexpr uint32_t kWaves = kMbfsWg / kWave;
    __shared__ uint32_t s_sm[kWaves], s_lg[kWaves], s_bsm[kWaves], s_blg[kWaves];
    __shared__ unsigned long long s_sum[kMbfsSums];
    __shared__ uint32_t s_last;
    __shared__ float s_params[kDecide ? kMlpWaveLds : 4];
    if (kDecide && a.ctl->done) return;
    const int32_t level = kDecide ? a.ctl->step + 1 : level_fixed;
    const uint32_t lv = level >= 255 ? 255u : (uint32_t)level;  // 255: saturated, reported as unreached
    const uint32_t n = a.n, lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    T* planes = static_cast<T*>(a.planes);
    if (threadIdx.x < kMbfsSums) s_sum[threadIdx.x] = 0;  // read behind the first tile's barriers
    uint32_t cact = 0;
    unsigned long long adeg = 0, bits = 0, redges = 0, dlg = 0;
    for (uint64_t base = (uint64_t)blockIdx.x * kMbfsTile; base < n; base += (uint64_t)gridDim.x * kMbfsTile) {
        const uint64_t v0 = base + wv * 4 * kWave + lane;
        unsigned long long raw[4], fr[4], nx[4], vis[4];
        uint32_t dg[4];
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const uint64_t v = v0 + c * kWave;
            raw[c] = v < n ? a.next[v] : 0ull;
            fr[c] = v < n ? a.frontier[v] : 0ull;
        }
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) vis[c] = raw[c] ? a.visited[v0 + c * kWave] : 0ull;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const uint64_t v = v0 + c * kWave;
            nx[c] = raw[c] & ~vis[c];
            dg[c] = nx[c] ? a.row_ptr[v + 1] - a.row_ptr[v] : 0u;
        }
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const uint64_t v = v0 + c * kWave;
            if (raw[c]) a.next[v] = 0;
            if (nx[c]) a.visited[v] = vis[c] | nx[c];
            if (fr[c] != nx[c]) a.frontier[v] = nx[c];
        }
        for (uint32_t p = 0; p < kMbfsPlanes; ++p) {  // uniform
            if (!((lv >> p) & 1u)) continue;
            T* plane = planes + (size_t)p * n;
            if (lv == 1u << p) {  // the plane's first use: every word written, none read
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c)
                    if (v0 + c * kWave < n) plane[v0 + c * kWave] = (T)nx[c];
                continue;
            }
            T x[4];
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) x[c] = nx[c] ? plane[v0 + c * kWave] : (T)0;
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c)
                if (nx[c]) plane[v0 + c * kWave] = (T)(x[c] | (T)nx[c]);
        }
        unsigned long long msm[4], mlg[4];
        uint32_t csm = 0, clg = 0;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const uint32_t deg = dg[c];
            cact += (uint32_t)__popcll(__ballot(nx[c] != 0));
            msm[c] = __ballot(deg > 0 && deg <= a.large);
            mlg[c] = __ballot(deg > a.large);
            csm += (uint32_t)__popcll(msm[c]);
            clg += (uint32_t)__popcll(mlg[c]);
            adeg += deg;
            dlg += deg > a.large ? deg : 0u;
            bits += __popcll(nx[c]);
            redges += (unsigned long long)__popcll(nx[c]) * deg;
        }
        if (lane == 0) {
            s_sm[wv] = csm;
            s_lg[wv] = clg;
        }
        __syncthreads();
        if (wv == 0) {
            const uint32_t sm = lane < kWaves ? s_sm[lane] : 0u, lg = lane < kWaves ? s_lg[lane] : 0u;
            const uint32_t ism = wave_incl_scan(sm), ilg = wave_incl_scan(lg);
            uint32_t got = 0;
            if (lane == kWave - 2 && ism) got = atomicAdd(&a.ctr->n_small, ism);
            if (lane == kWave - 1 && ilg) got = atomicAdd(&a.ctr->n_large, ilg);
            const uint32_t bsm = __builtin_amdgcn_readlane(got, kWave - 2), blg = __builtin_amdgcn_readlane(got, kWave - 1);
            if (lane < kWaves) {
                s_bsm[lane] = bsm + ism - sm;
                s_blg[lane] = blg + ilg - lg;
            }
        }
        __syncthreads();
        uint32_t osm = s_bsm[wv], olg = s_blg[wv];
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const uint32_t v = (uint32_t)(v0 + c * kWave);
            if ((msm[c] >> lane) & 1ull) a.q_small[osm + lanes_below(msm[c])] = v;
            if ((mlg[c] >> lane) & 1ull) a.q_large[olg + lanes_below(mlg[c])] = v;
            osm += (uint32_t)__popcll(msm[c]);
            olg += (uint32_t)__popcll(mlg[c]);
        }
    }
    if (cact) {  // uniform across the wave
        adeg = wave_sum_u64(adeg);
        bits = wave_sum_u64(bits);
        redges = wave_sum_u64(redges);
        dlg = wave_sum_u64(dlg);
        if (lane == 0) {
            atomicAdd(&s_sum[kMbfsActive], (unsigned long long)cact);
            atomicAdd(&s_sum[kMbfsActiveDeg], adeg);
            atomicAdd(&s_sum[kMbfsNewBits], bits);
            atomicAdd(&s_sum[kMbfsReachedEdges], redges);
            atomicAdd(&s_sum[kMbfsLargeDeg], dlg);
        }
    }
    __syncthreads();
    if (wv != 0) return;
    const unsigned long long sum = lane < kMbfsSums ? s_sum[lane] : 0ull;
    if (sum) atomicAdd(&a.ctr->sum[lane].v, sum);
    if constexpr (kDecide) {
        // the wave's atomics have been performed before its ticket is taken
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(&a.ctr->ticket, 1u);
        if ((uint32_t)__builtin_amdgcn_readfirstlane(t) == gridDim.x - 1) mbfs_decide(a, false, s_params);
    }
}

// Bit j, j + 4, .. j + 28 of four planes' words as the nibbles of a word.
__device__ __forceinline__ uint32_t mbfs_nibbles(uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3, uint32_t j) {
    constexpr uint32_t kLow = 0x11111111u;
    return ((x0 >> j) & kLow) | (((x1 >> j) & kLow) << 1) | (((x2 >> j) & kLow) << 2) | (((x3 >> j) & kLow) << 3);
}

// The planes as level bytes, one row of n per source, 0xFF where the source does not reach the
// vertex: rows [row0, row1) at `out` (by the control block of a finished run: every row, at ctl->out).
// A lane takes 4 vertices: the planes' words become nibbles, then bytes, 32 sources at a time, and 4
// words of 4 sources each are transposed into 4 stores of 4 vertices each.  Bound by the stores: a
// wave writes 256 contiguous bytes of a row at a time.  RMAT-20, 64 sources:
// 25 us for 64 MiB of levels from 40 of planes and masks.
template <class T>
__global__ __launch_bounds__(256) void k_mbfs_finish(MbfsArgs a, MbfsCtl* __restrict__ host, uint8_t* out, uint32_t row0,
                                                     uint32_t row1) {
    const MbfsCtl* ctl = a.ctl;
    if (host) {
        if (blockIdx.x == 0 && threadIdx.x < sizeof(MbfsCtl) / 8)
            reinterpret_cast<unsigned long long*>(host)[threadIdx.x] =
                reinterpret_cast<const unsigned long long*>(ctl)[threadIdx.x];
        if (!ctl->done || !ctl->out) return;
        out = ctl->out;
        row0 = 0;
        row1 = ctl->k;
    }
    const uint32_t n = a.n;
    const uint32_t last = ctl->step < 255 ? (uint32_t)ctl->step : 255u;  // the planes up to its bits were written
    const uint32_t np = 32 - __builtin_clz(last | 1u);
    const T* planes = static_cast<const T*>(a.planes);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q * 4 < n; q += stride) {
        const uint64_t v0 = q * 4;
        const uint32_t cnt = n - v0 < 4 ? (uint32_t)(n - v0) : 4u;
        T x[kMbfsPlanes][4];
        unsigned long long vis[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            vis[i] = i < cnt ? a.visited[v0 + i] : 0ull;
#pragma unroll
            for (uint32_t p = 0; p < kMbfsPlanes; ++p)
                x[p][i] = p < np && i < cnt ? planes[(size_t)p * n + v0 + i] : (T)0;
        }
#pragma unroll
        for (uint32_t h = 0; h < (sizeof(T) == 8 ? 2u : 1u); ++h) {
            auto word = [h](unsigned long long w) { return (uint32_t)(w >> (32 * h)); };
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                uint32_t lo[4], hi[4];  // nibbles of sources 32h + j + 4i
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    const uint32_t u = ~word(vis[i]);
                    lo[i] = mbfs_nibbles(word(x[0][i]) | u, word(x[1][i]) | u, word(x[2][i]) | u, word(x[3][i]) | u, j);
                    hi[i] = np > 4 ? mbfs_nibbles(word(x[4][i]) | u, word(x[5][i]) | u, word(x[6][i]) | u,
                                                  word(x[7][i]) | u, j)
                                   : ((u >> j) & 0x11111111u) * 15u;
                }
#pragma unroll
                for (uint32_t odd = 0; odd < 2; ++odd) {
                    uint32_t b[4];  // bytes of sources s0, s0 + 8, s0 + 16, s0 + 24, vertex i
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        constexpr uint32_t kNib = 0x0F0F0F0Fu;
                        b[i] = odd ? ((lo[i] >> 4) & kNib) | (hi[i] & ~kNib) : (lo[i] & kNib) | ((hi[i] & kNib) << 4);
                    }
                    const uint32_t s0 = 32 * h + j + 4 * odd;
#pragma unroll
                    for (uint32_t t = 0; t < 4; ++t) {
                        const uint32_t s = s0 + 8 * t;
                        if (8 * t + j + 4 * odd >= 8 * sizeof(T) || s < row0 || s >= row1) continue;
                        uint32_t w = 0;
#pragma unroll
                        for (uint32_t i = 0; i < 4; ++i) w |= ((b[i] >> (8 * t)) & 0xFFu) << (8 * i);
                        uint8_t* to = out + (uint64_t)(s - row0) * n + v0;
                        if (cnt == 4) {
                            __builtin_memcpy(to, &w, 4);  // rows of any alignment
                        } else {
                            for (uint32_t i = 0; i < cnt; ++i) to[i] = (uint8_t)(w >> (8 * i));
                        }
                    }
                }
            }
        }
    }
}

// Host-driven superstep: the host's decision written into the control block.
__global__ void k_mbfs_set_ctl(MbfsCtl* ctl, int32_t step, uint32_t pull, uint32_t n_small, uint32_t n_large,
                               uint32_t hub_wgs) {
    ctl->step = step;
    ctl->pull = pull;
    ctl->n_small = n_small;
    ctl->n_large = n_large;
    ctl->hub_wgs = hub_wgs;
}
__global__ void k_mbfs_zero(MbfsCounters* c) {
    if (threadIdx.x < sizeof(MbfsCounters) / 8) reinterpret_cast<unsigned long long*>(c)[threadIdx.x] = 0;
}

static uint32_t mbfs_large(const medusa_graph* g, const medusa_opts& o) {
    return o.large_degree ? o.large_degree : (g->tuned.mbfs_large ? g->tuned.mbfs_large : kMbfsLargeDefault);
}
static uint32_t mbfs_grid(const medusa_graph* g, const medusa_opts& o) {
    return o.grid ? o.grid : (g->tuned.mbfs_grid ? g->tuned.mbfs_grid : kMbfsGridDefault);
}

// Bytes of device memory for the rows of a host output on their way there.
constexpr size_t kMbfsRowBytes = 256u << 20;

template <class T>
static void mbfs_run(medusa_graph* g, const uint32_t* srcs, uint32_t k, uint8_t* out, const medusa_opts& o,
                     medusa_stats& st) {
    const uint32_t n = g->n;
    const uint64_t m = g->m;
    const uint32_t large = mbfs_large(g, o), grid = mbfs_grid(g, o);
    g->q_small.ensure(n);
    g->q_large.ensure(n);
    DBuf<unsigned long long>& masks = g->bitmap;
    masks.ensure(3 * (size_t)n);
    DBuf<uint32_t>& planes = g->stamp;  // reused as the storage of the level planes
    planes.ensure((kMbfsPlanes * sizeof(T) * (size_t)n + 3) / 4);
    MbfsCounters* C = dev_counters<MbfsCounters>(g);
    static_assert(sizeof(MbfsCtl) <= sizeof(CtlStorage), "control block storage");
    g->mbfs_ctl.ensure(1);
    MbfsCtl* ctl = reinterpret_cast<MbfsCtl*>(g->mbfs_ctl.p);
    MbfsCtl* host = reinterpret_cast<MbfsCtl*>(g->h_ctr_raw.p);
    hipStream_t s = g->stream;
    const bool host_driven = o.timing || o.trace;
    uint32_t mode = 0;
    if (o.direction == MEDUSA_DIR_PUSH) mode = 1;
    else if (o.direction == MEDUSA_DIR_PULL) mode = 2;
    else if (o.policy && policy_kind(o.policy) == MEDUSA_POLICY_DIRECTION) mode = 3;
    const float* policy = (mode == 3 && !host_driven) ? policy_device_params(o.policy) : nullptr;
    g->trace.clear();

    build_pull_layout(g);
    const PullLayout& PL = *g->pull;
    MbfsArgs a{};
    a.row_ptr = g->row_ptr.p;
    a.col = g->col.p;
    a.cptr = g->cptr.p;
    a.csrc = g->csrc.p;
    a.q_small = g->q_small.p;
    a.q_large = g->q_large.p;
    a.visited = masks.p;
    a.frontier = masks.p + n;
    a.next = masks.p + 2 * (size_t)n;
    a.runs = PL.d_runs.p;
    a.wg_run = PL.wg_run.p;
    a.perm = PL.perm.p;
    a.ell = PL.ell.p;
    a.ctr = C;
    a.ctl = ctl;
    a.policy = policy;
    a.planes = planes.p;
    a.n = n;
    a.large = large;
    a.items = PL.total_wgs;
    a.grid = grid;
    const dim3 update_grid(grid_for(n, kMbfsTile, 512)), finish_grid(grid_for(n, 1024, 8192));
    const bool direct = kernels_can_write(g, out);  // else the rows are copied out at the end

    auto expand = [&]() {
        hipLaunchKernelGGL(k_mbfs_expand, dim3(grid), dim3(256), 0, s, a);
        MDS_LAUNCHED();
    };
    // capture (once per buffers, launch shape, policy buffer and slot count) a batch of supersteps
    auto captured = [&](GraphCache& gc, uint32_t slots) -> hipGraphExec_t {
        const uintptr_t key[8] = {(uintptr_t)masks.p,   (uintptr_t)policy,
                                  ((uintptr_t)grid << 32) | large,
                                  (uintptr_t)planes.p,  (uintptr_t)host,
                                  (uintptr_t)a.q_small, (uintptr_t)a.q_large,
                                  ((uintptr_t)sizeof(T) << 32) | slots};
        if (gc.exec && std::equal(key, key + 8, gc.key)) return gc.exec;
        gc.reset();
        MDS_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        hipGraph_t graph = nullptr;
        try {
            for (uint32_t b = 0; b < slots; ++b) {
                expand();
                hipLaunchKernelGGL((k_mbfs_update<T, true>), update_grid, dim3(kMbfsWg), 0, s, a, 0);
            }
            hipLaunchKernelGGL(k_mbfs_finish<T>, finish_grid, dim3(256), 0, s, a, host, (uint8_t*)nullptr, 0u, 0u);
            MDS_LAUNCHED();
        } catch (...) {
            (void)hipStreamEndCapture(s, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        hipError_t e = hipStreamEndCapture(s, &graph);
        if (e == hipSuccess) e = hipGraphInstantiate(&gc.exec, graph, nullptr, nullptr, 0);
        if (graph) (void)hipGraphDestroy(graph);
        MDS_HIP(e);
        std::copy(key, key + 8, gc.key);
        return gc.exec;
    };
    const uint32_t head = head_slots(g->mbfs_last_steps, kMbfsBatch);
    hipGraphExec_t head_exec = nullptr;
    if (!host_driven) head_exec = captured(head == kMbfsBatch ? g->mbfs_graph : g->mbfs_head, head);

    MbfsSources sources{};
    std::copy(srcs, srcs + k, sources.v);
    MDS_HIP(hipEventRecord(g->ev_begin, s));
    hipLaunchKernelGGL(k_mbfs_fill, dim3(grid_for(3ull * n, 256, 4096)), dim3(256), 0, s, a, (unsigned long long)m, k,
                       mode, direct ? out : nullptr);
    MDS_LAUNCHED();
    hipLaunchKernelGGL(k_mbfs_start, dim3(1), dim3(kWave), 0, s, a, sources, k, host_driven ? 0u : 1u);
    MDS_LAUNCHED();

    MbfsCtl h{};
    if (!host_driven) {
        for (uint32_t batch = 0;; ++batch) {
            MDS_HIP(hipGraphLaunch(batch == 0 ? head_exec : captured(g->mbfs_graph, kMbfsBatch), s));
            MDS_HIP(hipEventRecord(g->ev_end, s));
            MDS_HIP(hipStreamSynchronize(s));
            if (host->done) break;
            MDS_CHECK(batch < (n + kMbfsBatch) / kMbfsBatch + 2, MEDUSA_ERR_INTERNAL,
                      "mbfs: superstep loop did not end");
        }
        h = *host;
        g->mbfs_last_steps = h.supersteps;
    } else {
        Sched sched(o, Sched::kMbfs);
        const bool timing = o.timing != 0;
        if (timing) ensure_events(g, 2);
        MbfsCounters c = read_counters<MbfsCounters>(g);
        Frontier f{};
        f.n = n;
        f.m = m;
        h.n_u = (uint64_t)n * k - c.sum[kMbfsNewBits].v;
        h.m_u = (uint64_t)m * k - c.sum[kMbfsReachedEdges].v;
        h.reached = c.sum[kMbfsNewBits].v;
        h.reached_edges = c.sum[kMbfsReachedEdges].v;
        bool pull = false;
        for (uint32_t t = 0; c.sum[kMbfsActive].v; ++t) {
            f.step = t;
            f.n_f = c.sum[kMbfsActive].v;
            f.m_f = c.sum[kMbfsActiveDeg].v;
            f.n_u = h.n_u;
            f.m_u = h.m_u;
            if (o.direction == MEDUSA_DIR_PUSH) pull = false;
            else if (o.direction == MEDUSA_DIR_PULL) pull = true;
            else pull = sched.bfs_pull(f, pull);
            hipLaunchKernelGGL(k_mbfs_set_ctl, dim3(1), dim3(1), 0, s, ctl, (int32_t)t, pull ? 1u : 0u, c.n_small,
                               c.n_large, mbfs_hub_wgs(grid, c.n_small, c.n_large, c.sum[kMbfsLargeDeg].v, f.m_f));
            MDS_LAUNCHED();
            hipLaunchKernelGGL(k_mbfs_zero, dim3(1), dim3(sizeof(MbfsCounters) / 8), 0, s, C);
            MDS_LAUNCHED();
            if (timing) MDS_HIP(hipEventRecord(g->events[0], s));
            expand();
            if (timing) MDS_HIP(hipEventRecord(g->events[1], s));
            hipLaunchKernelGGL((k_mbfs_update<T, false>), update_grid, dim3(kMbfsWg), 0, s, a, (int32_t)(t + 1));
            MDS_LAUNCHED();
            c = read_counters<MbfsCounters>(g);
            double kms = 0;
            if (timing) {
                float ms = 0;
                MDS_HIP(hipEventElapsedTime(&ms, g->events[0], g->events[1]));
                kms = ms;
                st.kernel_ms += ms;
                ++st.kernel_launches;
            }
            uint64_t probes = 0;
            for (const MbfsLine& l : c.probes) probes += l.v;
            const uint64_t kb = pull ? 4ull * (n + 1) + 8ull * n + 12ull * probes : 20ull * f.n_f + 20ull * f.m_f;
            const uint64_t new_bits = c.sum[kMbfsNewBits].v;
            h.kernel_bytes += kb;
            h.alg_bytes += kb + 24ull * n + new_bits;
            if (pull) ++h.pull_steps; else ++h.push_steps;
            sched.record(g, f, pull ? 1.0 : 0.0, kms);
            ++h.supersteps;
            if (t + 1 >= 255 && new_bits) h.saturated = 1;
            h.reached += new_bits;
            h.reached_edges += c.sum[kMbfsReachedEdges].v;
            h.n_u -= new_bits;
            h.m_u -= c.sum[kMbfsReachedEdges].v;
        }
        // the last update's level, for the finish
        hipLaunchKernelGGL(k_mbfs_set_ctl, dim3(1), dim3(1), 0, s, ctl, (int32_t)h.supersteps, 0u, 0u, 0u, 0u);
        MDS_LAUNCHED();
        if (direct) {
            hipLaunchKernelGGL(k_mbfs_finish<T>, finish_grid, dim3(256), 0, s, a, (MbfsCtl*)nullptr, out, 0u, k);
            MDS_LAUNCHED();
        }
        MDS_HIP(hipEventRecord(g->ev_end, s));
        MDS_HIP(hipStreamSynchronize(s));
    }
    float ms = 0;
    MDS_HIP(hipEventElapsedTime(&ms, g->ev_begin, g->ev_end));
    st.device_ms = ms;
    st.supersteps = h.supersteps;
    st.push_steps = h.push_steps;
    st.pull_steps = h.pull_steps;
    st.kernel_bytes = h.kernel_bytes;
    st.alg_bytes = h.alg_bytes + (uint64_t)k * n + 24ull * n;
    st.edges_traversed = h.reached_edges;
    st.reached = (uint32_t)std::min<uint64_t>(h.reached, 0xFFFFFFFFull);
    st.reserved[0] = h.saturated;
    if (direct) return;
    // as many rows at a time as the row buffer holds
    const uint32_t rows = (uint32_t)std::min<uint64_t>(k, std::max<uint64_t>(1, kMbfsRowBytes / n));
    g->mbfs_rows.ensure(((size_t)rows * n + 3) / 4);
    for (uint32_t r = 0; r < k; r += rows) {
        const uint32_t r1 = std::min(k, r + rows);
        uint8_t* buf = reinterpret_cast<uint8_t*>(g->mbfs_rows.p);
        hipLaunchKernelGGL(k_mbfs_finish<T>, finish_grid, dim3(256), 0, s, a, (MbfsCtl*)nullptr, buf, r, r1);
        MDS_LAUNCHED();
        copy_out(g, out + (size_t)r * n, buf, (size_t)(r1 - r) * n);
    }
}

}  // namespace medusa

using namespace medusa;

extern "C" int medusa_mbfs(medusa_graph* g, const uint32_t* sources, uint32_t k, uint8_t* levels,
                           const medusa_opts* opts, medusa_stats* stats) {
    return guard([&] {
        const auto lock = enter(g);
        MDS_CHECK(levels && sources, MEDUSA_ERR_ARG, "mbfs: null argument");
        MDS_CHECK(k >= 1 && k <= 64, MEDUSA_ERR_ARG, "mbfs: k must be in [1, 64]");
        for (uint32_t s = 0; s < k; ++s)
            MDS_CHECK(sources[s] < g->n, MEDUSA_ERR_ARG, "mbfs: source %u out of range", sources[s]);
        medusa_opts o{};
        if (opts) o = *opts;
        MDS_CHECK(o.direction >= 0 && o.direction <= 2, MEDUSA_ERR_ARG, "mbfs: bad direction %d", o.direction);
        MDS_CHECK(o.grid == 0 || (o.grid >= 2 && o.grid <= 65535), MEDUSA_ERR_ARG, "mbfs: grid must be 0 or 2..65535");
        medusa_stats st{};
        if (k <= 8) mbfs_run<uint8_t>(g, sources, k, levels, o, st);
        else if (k <= 16) mbfs_run<uint16_t>(g, sources, k, levels, o, st);
        else if (k <= 32) mbfs_run<uint32_t>(g, sources, k, levels, o, st);
        else mbfs_run<unsigned long long>(g, sources, k, levels, o, st);
        if (stats) *stats = st;
    });
}
