// Multi-source BFS: up to 64 sources advance together, one bit per source in a
// 64-bit mask per vertex (frontier, visited, next).
//
// No reference counterpart: "MBFS" in the reference is multi-GPU BFS
// (HowToBuild:13); the semantics here are those of k independent BFS runs
// (Algorithm/UserOperators.h:17-36 per source), checked against exactly that.
//
// Superstep, over vertices in the pull layout's internal order:
//   push:   active vertices (frontier mask != 0) OR their mask into next[v] of every
//           out-neighbour that still lacks some of those bits (64-bit atomicOr); vertices
//           up to `large` out-degree go through the wave-cooperative queue, hubs above it
//           are split over whole workgroups (the threshold is autotunable);
//   update: after a push: new = next & ~visited, and the queues of the next push, with ballot
//           + in-workgroup prefix scan;
//   pull:   every vertex not yet visited by all sources ORs the frontier masks of its
//           in-neighbours, stopping early once every missing bit has been found, and takes its
//           own new bits in the same pass;
//   queue:  after a pull, before a push: the queues from the frontier masks.
// New bits: visited |= new; frontier = new (in the other of two frontier arrays); the level goes
// into bit planes (plane p holds bit p of every (vertex, source) level).  After the last superstep the
// finish turns the planes into one level byte per (source, vertex) in the original order.
//
// Drivers as for BFS: device-driven (the last workgroup of each update or pull writes the
// next superstep into a control block; batches of launches, each doing what the control block says,
// are captured as hipGraphs and replayed until done, sized by the previous run on the handle, and
// each ends with the finish, which returns at once unless the run is done) and host-driven (timing or
// tracing) over the same kernels.

#include <algorithm>
#include <cstddef>
#include <vector>

#include "engine.h"
#include "sched.h"

namespace medusa {

constexpr uint32_t kMbfsBatch = 16;  // launches of a replay without a previous run
constexpr uint32_t kMbfsSplit = 8;  // minimum workgroup items per hub

// Counters of a launch, spread over kMbfsSegs lines by workgroup: same-address atomics serialise.
constexpr uint32_t kMbfsSegs = 32;
// active vertices, their out-degrees, those of the hubs among them (above `large`), queue entries and
// hubs (low and high word), in-edges examined, new (source, vertex) pairs, the pairs' out-degrees
enum {
    kMbfsActive, kMbfsActiveDeg, kMbfsLargeDeg, kMbfsQueued, kMbfsProbes, kMbfsNewBits, kMbfsReachedEdges,
    kMbfsSums
};
struct MbfsLine {
    alignas(128) uint32_t v;
};
struct MbfsCounters {
    struct {
        alignas(128) unsigned long long v[kMbfsSums];
    } sum[kMbfsSegs];
    MbfsLine queued[2][kMbfsSegs];  // queue entries per segment, by superstep parity
    MbfsLine hubs[2];
    MbfsLine sub[kMbfsSegs], top;   // tickets
};

enum : uint32_t { kMbfsPush, kMbfsUpdate, kMbfsPull, kMbfsQueue };
struct MbfsCtl {
    int32_t step;
    uint32_t phase, pull, done, n_large, hub_wgs, mode, saturated;
    uint32_t supersteps, push_steps, pull_steps, k, slots, n_small;
    unsigned long long n, m, n_f, m_f, n_u, m_u, reached, reached_edges, kernel_bytes, alg_bytes, full;
    uint8_t* out;  // where the finish of a device-driven run writes the levels, or null
};

// What a device-driven run leaves in pinned memory.
constexpr uint32_t kMbfsEnds = 1024;
struct MbfsHost {
    MbfsCtl ctl;
    unsigned long long t_begin, t_end;   // wall clock before the first kernel and after the last superstep
    unsigned long long made[kMbfsEnds];  // and when workgroups of the finish had stored their levels
};

struct MbfsArgs {
    const uint32_t *dst, *pos;
    const uint2* out;        // first out-edge, out-degree
    const uint8_t* indeg;
    const uint64_t* base;
    const uint4* hub;
    const uint32_t* src;
    uint32_t *q_small, *q_large;
    unsigned long long *visited, *next, *frontier[2];  // frontier of superstep t: [t % 2]
    MbfsCounters* ctr;
    MbfsCtl* ctl;  // two: a launch reads one and writes the other
    const float* policy;
    void* planes;  // kMbfsPlanes of n words each, of the width that holds k bits
    uint32_t n, large, nslices, nhubs, grid, span;
};
constexpr uint32_t kMbfsPlanes = 8;
constexpr uint32_t kMbfsSplitRows = 1u << 17;  // vertices below which the finish deals rows over workgroups
constexpr uint32_t kMbfsTile = 1024;  // vertices of a workgroup's round of an update or queue pass

// Queue segment span for n vertices: kMbfsSegs segments cover [0, n) in whole tiles.
static uint32_t mbfs_span(uint32_t n) {
    const uint64_t tiles = ((uint64_t)n + kMbfsTile - 1) / kMbfsTile;
    return (uint32_t)((tiles + kMbfsSegs - 1) / kMbfsSegs * kMbfsTile);
}

// ---- layout ---------------------------------------------------------------------------

// One workgroup per window: its vertices by in-degree, hubs first.  The order of vertices of one
// degree is whatever the LDS counters give: it changes no result.
__global__ __launch_bounds__(1024) void k_pull_sort(uint32_t n, const uint32_t* __restrict__ cptr,
                                                    const uint32_t* __restrict__ row_ptr, uint32_t* __restrict__ perm,
                                                    uint32_t* __restrict__ pos, uint2* __restrict__ out,
                                                    uint8_t* __restrict__ indeg, uint32_t* __restrict__ hub_count) {
    __shared__ uint32_t cnt[kWave + 2], first[kWave + 2];
    static_assert(kPullLaneMax == kWave, "one wave scans the degrees' counts");
    const uint32_t t = threadIdx.x;
    const uint64_t w0 = (uint64_t)blockIdx.x * kPullWindow;
    if (t < kWave + 2) cnt[t] = 0;
    __syncthreads();
    uint32_t deg[4], key[4], at[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        const uint64_t v = w0 + j * 1024 + t;
        if (v >= n) continue;
        deg[j] = cptr[v + 1] - cptr[v];
        key[j] = deg[j] > kPullLaneMax ? 0u : 1u + kPullLaneMax - deg[j];
        at[j] = atomicAdd(&cnt[key[j]], 1u);
    }
    __syncthreads();
    if (t < kWave) {
        const uint32_t c = cnt[t], incl = wave_incl_scan(c);
        first[t] = incl - c;
        if (t == kWave - 1) {
            first[kWave] = incl;
            first[kWave + 1] = incl + cnt[kWave];
        }
    }
    __syncthreads();
    if (t == 0 && cnt[0]) atomicAdd(hub_count, cnt[0]);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        const uint64_t v = w0 + j * 1024 + t;
        if (v >= n) continue;
        const uint32_t p = (uint32_t)w0 + first[key[j]] + at[j];
        perm[p] = (uint32_t)v;
        pos[v] = p;
        out[p] = uint2{row_ptr[v], row_ptr[v + 1] - row_ptr[v]};
        indeg[p] = deg[j] > kPullLaneMax ? kPullHub : (uint8_t)deg[j];
    }
}

// The columns of every slice and the in-edges of every hub; one wave per slice or hub.
__global__ __launch_bounds__(256) void k_pull_fill(uint32_t n, uint32_t nslices, uint32_t nhubs,
                                                   const uint32_t* __restrict__ cptr, const uint32_t* __restrict__ csrc,
                                                   const uint32_t* __restrict__ perm, const uint32_t* __restrict__ pos,
                                                   const uint8_t* __restrict__ indeg, const uint64_t* __restrict__ base,
                                                   const uint4* __restrict__ hub, uint32_t* __restrict__ src) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t nw = (uint64_t)gridDim.x * 4, total = (uint64_t)nslices + nhubs;
    for (uint64_t s = (uint64_t)blockIdx.x * 4 + threadIdx.x / kWave; s < total; s += nw) {  // uniform per wave
        if (s >= nslices) {
            const uint4 h = hub[s - nslices];
            const uint32_t b = cptr[perm[h.x]];
            uint32_t* to = src + (((uint64_t)h.w << 32) | h.z);
            for (uint32_t k = lane; k < h.y; k = advance_to(k, kWave, h.y)) to[k] = pos[csrc[b + k]];
            continue;
        }
        const uint64_t b = base[s], len = (base[s + 1] - b) / kWave, p = s * kWave + lane;
        const uint32_t d = p < n && indeg[p] != kPullHub ? indeg[p] : 0u;
        const uint32_t e = d ? cptr[perm[p]] : 0u;
        for (uint64_t k = 0; k < len; ++k) src[b + k * kWave + lane] = k < d ? pos[csrc[e + k]] : 0u;
    }
}

__global__ void k_pull_dst(uint64_t m, const uint32_t* __restrict__ col, const uint32_t* __restrict__ pos,
                           uint32_t* __restrict__ dst) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < m; e += stride) dst[e] = pos[col[e]];
}

// Sorted and filled on the GPU (RMAT-20: 1.5 ms; on the host, with the sort over all vertices and an
// upload of every slab, 130 ms); the host sums the slices' and hubs' lengths.
static void build_pull_layout(medusa_graph* g) {
    if (g->pull) return;
    const uint32_t n = g->n;
    hipStream_t s = g->stream;
    auto L = std::make_unique<PullLayout>();
    const uint32_t windows = (uint32_t)(((uint64_t)n + kPullWindow - 1) / kPullWindow);
    L->nslices = (uint32_t)(((uint64_t)n + kWave - 1) / kWave);
    L->pos.alloc(n);
    L->out.alloc(n);
    L->indeg.alloc(n);
    DBuf<uint32_t> perm, count;
    perm.alloc(n);
    count.alloc(1);
    const uint32_t zero = 0;
    MDS_HIP(hipMemcpyAsync(count.p, &zero, 4, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_pull_sort, dim3(windows), dim3(1024), 0, s, n, g->cptr.p, g->row_ptr.p, perm.p, L->pos.p,
                       L->out.p, L->indeg.p, count.p);
    MDS_LAUNCHED();
    std::vector<uint8_t> indeg(n);
    std::vector<uint32_t> order;
    MDS_HIP(hipMemcpyAsync(indeg.data(), L->indeg.p, n, hipMemcpyDeviceToHost, s));
    MDS_HIP(hipMemcpyAsync(&L->nhubs, count.p, 4, hipMemcpyDeviceToHost, s));
    MDS_HIP(hipStreamSynchronize(s));
    if (L->nhubs) {
        order.resize(n);
        MDS_HIP(hipMemcpyAsync(order.data(), perm.p, (size_t)n * 4, hipMemcpyDeviceToHost, s));
        MDS_HIP(hipStreamSynchronize(s));
    }
    // a slice is as long as its longest in-edge list that is not a hub's: in a window sorted by
    // in-degree, its first one's
    std::vector<uint64_t> base((size_t)L->nslices + 1);
    uint64_t at = 0;
    for (uint32_t i = 0; i < L->nslices; ++i) {
        base[i] = at;
        const uint64_t p1 = std::min<uint64_t>(n, (uint64_t)(i + 1) * kWave);
        for (uint64_t p = (uint64_t)i * kWave; p < p1; ++p)
            if (indeg[p] != kPullHub) {
                at += (uint64_t)indeg[p] * kWave;
                break;
            }
    }
    base[L->nslices] = at;
    std::vector<uint4> hub;
    hub.reserve(L->nhubs);
    if (L->nhubs)
        for (uint32_t p = 0; p < n; ++p)
            if (indeg[p] == kPullHub) {
                const uint32_t v = order[p], d = g->h_cptr[v + 1] - g->h_cptr[v];
                hub.push_back(uint4{p, d, (uint32_t)at, (uint32_t)(at >> 32)});
                at += d;
            }
    MDS_CHECK(hub.size() == L->nhubs, MEDUSA_ERR_INTERNAL, "mbfs: hub count");
    // longest first: a wave that starts one late would end the launch late
    std::sort(hub.begin(), hub.end(),
              [](const uint4& a, const uint4& b) { return a.y != b.y ? a.y > b.y : a.x < b.x; });
    L->base.upload(base.data(), base.size(), s);
    if (L->nhubs) L->hub.upload(hub.data(), hub.size(), s);
    L->src.alloc(std::max<uint64_t>(at, 1));
    hipLaunchKernelGGL(k_pull_fill, dim3(grid_for((uint64_t)L->nslices + L->nhubs, 4, 8192)), dim3(256), 0, s, n,
                       L->nslices, L->nhubs, g->cptr.p, g->csrc.p, (const uint32_t*)perm.p, (const uint32_t*)L->pos.p,
                       (const uint8_t*)L->indeg.p, (const uint64_t*)L->base.p, (const uint4*)L->hub.p, L->src.p);
    MDS_LAUNCHED();
    L->dst.alloc(std::max<uint64_t>(g->m, 1));
    hipLaunchKernelGGL(k_pull_dst, dim3(grid_for(g->m, 1024, 8192)), dim3(256), 0, s, g->m, g->col.p,
                       (const uint32_t*)L->pos.p, L->dst.p);
    MDS_LAUNCHED();
    MDS_HIP(hipStreamSynchronize(s));
    g->pull = std::move(L);
}

// ---- start ----------------------------------------------------------------------------

// Masks cleared, counters and control block set up.
__global__ __launch_bounds__(256) void k_mbfs_fill(MbfsArgs a, unsigned long long m, uint32_t k, uint32_t mode,
                                                   uint8_t* out, MbfsHost* host) {
    const uint64_t tid = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    // visited, next and frontier 0 follow each other; frontier 1 is written whole before it is read
    for (uint64_t i = tid; i < 3ull * a.n; i += stride) a.visited[i] = 0;
    if (blockIdx.x != 0) return;
    for (uint32_t i = threadIdx.x; i < sizeof(MbfsCounters) / 8; i += blockDim.x)
        reinterpret_cast<unsigned long long*>(a.ctr)[i] = 0;
    if (threadIdx.x == 0) {
        host->t_begin = (unsigned long long)wall_clock64();
        MbfsCtl z{};
        z.mode = mode;
        z.n = a.n;
        z.m = m;
        z.k = k;
        z.n_u = (unsigned long long)a.n * k;
        z.m_u = m * k;
        z.full = k == 64 ? ~0ull : ((1ull << k) - 1);
        z.out = out;
        a.ctl[0] = z;
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

struct MbfsPushLds {
    uint32_t beg[4][kWave], off[4][kWave];
    unsigned long long mask[4][kWave];
    uint32_t pre[kMbfsSegs + 1];
};

__device__ __forceinline__ void mbfs_offer(const MbfsArgs& a, uint32_t e, unsigned long long mask) {
    const uint32_t v = a.dst[e];
    const unsigned long long add = mask & ~a.visited[v];
    if (add && (a.next[v] & add) != add) atomicOr(&a.next[v], add);
}

// Wave-cooperative push; wave w of the nwaves taking part holds queue entries
// w, w + nwaves, ... one per lane.  Entries [pre[s], pre[s + 1]) of the queue lie in segment s.
__device__ __forceinline__ void mbfs_push_small(const MbfsArgs& a, const MbfsLine* __restrict__ queued,
                                                const unsigned long long* __restrict__ frontier, uint32_t wave0,
                                                uint32_t nwaves, MbfsPushLds& L) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    if (wv == 0) {
        const uint32_t incl = wave_incl_scan(lane < kMbfsSegs ? queued[lane].v : 0u);
        if (lane < kMbfsSegs) L.pre[lane + 1] = incl;
        if (lane == 0) L.pre[0] = 0;
    }
    __syncthreads();
    const uint32_t qn = L.pre[kMbfsSegs];
    for (uint64_t r = 0; wave0 + r * kWave * nwaves < qn; ++r) {  // uniform across the wave
        const uint64_t i = wave0 + (r * kWave + lane) * nwaves;
        uint2 edges{0, 0};
        unsigned long long fm = 0;
        if (i < qn) {
            uint32_t sg = 0;
#pragma unroll
            for (uint32_t step = kMbfsSegs / 2; step; step >>= 1)
                if (L.pre[sg + step] <= i) sg += step;
            const uint32_t u = a.q_small[(size_t)sg * a.span + (uint32_t)(i - L.pre[sg])];
            edges = a.out[u];
            fm = frontier[u];
        }
        const uint32_t incl = wave_incl_scan(edges.y);
        const uint32_t total = __builtin_amdgcn_readlane(incl, kWave - 1);
        L.beg[wv][lane] = edges.x;
        L.off[wv][lane] = incl - edges.y;
        L.mask[wv][lane] = fm;
        wave_lds_fence();
        for (uint32_t e0 = 0; e0 < total; e0 = advance_to(e0, kWave, total)) {  // uniform across the wave
            if (!lies_before(e0, lane, total)) continue;
            const uint32_t e = e0 + lane;
            uint32_t lo = 0;
#pragma unroll
            for (uint32_t step = kWave / 2; step; step >>= 1)
                if (L.off[wv][lo + step] <= e) lo += step;
            mbfs_offer(a, L.beg[wv][lo] + (e - L.off[wv][lo]), L.mask[wv][lo]);
        }
        wave_lds_fence();
    }
}

// Hubs: each queue vertex split into `split` edge ranges, one per workgroup item.
__device__ __forceinline__ void mbfs_push_large(const MbfsArgs& a, uint32_t qn,
                                                const unsigned long long* __restrict__ frontier, uint32_t wg0,
                                                uint32_t nwg) {
    uint32_t split = nwg / qn;
    split = split < kMbfsSplit ? kMbfsSplit : (split > 4096u ? 4096u : split);
    for (uint64_t w = wg0; w < (uint64_t)qn * split; w += nwg) {
        const uint32_t u = a.q_large[w / split], part = (uint32_t)(w % split);
        const uint2 edges = a.out[u];
        const unsigned long long fm = frontier[u];
        const EdgePart E = edge_part(edges.x, edges.y, part, split);
        const uint32_t cnt = E.hi - E.lo;  // an eighth of an edge array at most
        for (uint32_t k = threadIdx.x; k < cnt; k += blockDim.x) mbfs_offer(a, E.lo + k, fm);
    }
}

// A thread's share of a launch's sums.  Out-degrees and in-edges of distinct vertices add up to at
// most m, below 2^32.
struct MbfsAcc {
    uint32_t active = 0, deg = 0, large_deg = 0, small = 0, large = 0, probes = 0;
    unsigned long long bits = 0, edges = 0;
    __device__ __forceinline__ void add(const MbfsArgs& a, unsigned long long nx, uint32_t d) {
        const uint32_t b = (uint32_t)__popcll(nx);
        active += 1;
        deg += d;
        bits += b;
        edges += (unsigned long long)b * d;
        if (d > a.large) {
            large += 1;
            large_deg += d;
        } else if (d) {
            small += 1;
        }
    }
};

// What the planes hold for a level: the level, with 128 and 255 exchanged, so the levels past 254
// (saturated, reported as unreached), which a long graph has one of in every superstep, take one plane
// each and not all eight; and, above the code's eight bits, the plane that is used for the first time plus 1.
constexpr uint32_t kMbfsSaturated = 255;
__device__ __forceinline__ uint32_t mbfs_code(uint32_t level) {
    const uint32_t code = level >= kMbfsSaturated ? 128u : level == 128 ? 255u : level;
    const uint32_t first = level <= 128 && !(level & (level - 1)) ? (uint32_t)__builtin_ctz(level) + 1 : 0u;
    return code | first << 8;
}

// The new bits of a lane's kN vertices v0, v0 + 64, .. (nx = 0 past the last vertex and where the caller
// has none of its own: `mine`) at the level of `code`.  In a plane's first use every word is written and
// none read.  The others' words are read and written a plane at a time, its kN loads together: vertex by
// vertex these were up to 32 dependent accesses of a superstep.  700 x 700 lattice, 1262 supersteps of 8
// sources: 25.8 ms so, 25.4 a plane at a time, 21.1 with the codes for the saturated levels (and with the
// workgroups that find nothing to do leaving at once); two planes at a time are level, all eight at a time
// spill (29.2).
template <class T, uint32_t kN>
__device__ __forceinline__ void mbfs_set_levels(const MbfsArgs& a, uint32_t code, uint64_t v0,
                                                const unsigned long long (&nx)[kN], const bool (&mine)[kN]) {
    T* const planes = static_cast<T*>(a.planes) + v0;
    uint32_t bits = code & 0xFF;
    if (code >> 8) {
        const uint32_t p = (code >> 8) - 1;
        T* plane = planes + (size_t)p * a.n;
#pragma unroll
        for (uint32_t c = 0; c < kN; ++c)
            if (mine[c]) plane[c * kWave] = (T)nx[c];
        bits &= ~(1u << p);
    }
    unsigned long long any = 0;
#pragma unroll
    for (uint32_t c = 0; c < kN; ++c) any |= nx[c];
    if (!any) return;
#pragma unroll 1
    for (; bits; bits &= bits - 1) {  // uniform
        T* plane = planes + (size_t)__builtin_ctz(bits) * a.n;
        T old[kN];
#pragma unroll
        for (uint32_t c = 0; c < kN; ++c)
            if (nx[c]) old[c] = plane[c * kWave];
#pragma unroll
        for (uint32_t c = 0; c < kN; ++c)
            if (nx[c]) plane[c * kWave] = old[c] | (T)nx[c];
    }
}
template <class T>
__device__ __forceinline__ void mbfs_set_level(const MbfsArgs& a, uint32_t code, uint32_t p, unsigned long long nx) {
    const unsigned long long one[1] = {nx};
    const bool mine[1] = {true};
    mbfs_set_levels<T, 1>(a, code, p, one, mine);
}

constexpr uint32_t kMbfsPullGroup = 4;  // in-edges a lane probes per round
constexpr uint32_t kMbfsPullGrid = 512;
__device__ __forceinline__ uint32_t mbfs_pull_wgs(const MbfsArgs& a) { return max(a.grid, kMbfsPullGrid); }

__device__ __forceinline__ uint32_t wave_or(uint32_t x) {
    x |= dpp_or_zero<0x111>(x);
    x |= dpp_or_zero<0x112>(x);
    x |= dpp_or_zero<0x114>(x);
    x |= dpp_or_zero<0x118>(x);
    x |= dpp_or_zero<0x142, 0xa>(x);
    x |= dpp_or_zero<0x143, 0xc>(x);
    return (uint32_t)__builtin_amdgcn_readlane((int)x, kWave - 1);
}
__device__ __forceinline__ unsigned long long wave_or(unsigned long long x) {
    return ((unsigned long long)wave_or((uint32_t)(x >> 32)) << 32) | wave_or((uint32_t)x);
}

// Bottom-up: a vertex missing some sources ORs its in-neighbours' frontier masks until every missing
// bit is found, then takes the new bits: masks, level and sums, in the same pass.  A wave takes a
// slice (a vertex per lane; the k-th sources of 64 vertices are one load, kMbfsPullGroup in-edges per
// round, loads issued together, merged one by one with the same early exit and probe count as a plain
// loop) or a hub (64 in-edges per step, four steps' loads together).  Bound by the gather of
// 8-byte masks: in RMAT-20's full sweeps (17 M in-edges, 64 sources, 142 us) 35 % of 17 M requests
// miss the L2s, 770 MB of lines from the memory-side cache.  Eight in-edges per round, nontemporal
// loads of the sources and half as many registers changed nothing or lost.  In the original order over
// slabs sorted across all vertices the sweep took as long and an update of 20..24 us followed.
// `probes` counts in-edges examined up to and including the last one needed (a hub's in steps of 64).
template <class T>
__device__ __forceinline__ void mbfs_pull(const MbfsArgs& a, unsigned long long full, uint32_t lv,
                                          const unsigned long long* __restrict__ frontier,
                                          unsigned long long* __restrict__ nxt, MbfsAcc& acc) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t nw = mbfs_pull_wgs(a) * 4, w = blockIdx.x * 4 + threadIdx.x / kWave;
    for (uint32_t h = w; h < a.nhubs; h += nw) {  // uniform across the wave
        const uint4 H = a.hub[h];
        const uint32_t p = H.x, deg = H.y;
        const uint32_t* src = a.src + (((uint64_t)H.w << 32) | H.z);
        const unsigned long long vis = a.visited[p];
        unsigned long long found = 0;
        uint32_t probes = 0;
        bool all = vis == full;
        for (uint32_t k0 = 0; k0 < deg && !all; k0 = advance_to(k0, 4 * kWave, deg)) {
            uint32_t u[4];
            unsigned long long f[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t off = j * kWave + lane;
                u[j] = lies_before(k0, off, deg) ? src[k0 + off] : 0u;
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) f[j] = lies_before(k0, j * kWave + lane, deg) ? frontier[u[j]] : 0ull;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                if (all || !lies_before(k0, j * kWave, deg)) continue;
                found |= wave_or(f[j]);
                probes += min(deg - k0 - j * kWave, (uint32_t)kWave);
                all = (found | vis) == full;
            }
        }
        const unsigned long long nx = found & ~vis;
        if (lane == 0) {
            acc.probes += probes;
            nxt[p] = nx;
            mbfs_set_level<T>(a, lv, p, nx);
            if (nx) {
                a.visited[p] = vis | nx;
                acc.add(a, nx, a.out[p].y);
            }
        }
    }
    // slices are heavier towards a window's start: every second round is dealt the other way round
    uint32_t r = 0;
    for (uint64_t s0 = 0; s0 < a.nslices; s0 += nw, ++r) {
        const uint64_t s = s0 + ((r & 1u) ? nw - 1 - w : w);
        if (s >= a.nslices) continue;  // uniform across the wave
        const uint32_t p = (uint32_t)(s * kWave) + lane;
        const uint32_t ind = s * kWave + lane < a.n ? a.indeg[p] : kPullHub;
        const bool mine = ind != kPullHub;  // hubs above
        const unsigned long long vis = mine ? a.visited[p] : full;
        const uint32_t deg = vis != full ? ind : 0u;
        const uint32_t* src = a.src + a.base[s] + lane;
        unsigned long long found = 0;
        bool all = deg == 0;
        uint32_t u[kMbfsPullGroup];
#pragma unroll
        for (uint32_t j = 0; j < kMbfsPullGroup; ++j) u[j] = j < deg ? src[j * kWave] : 0u;
        for (uint32_t k0 = 0; k0 < deg && !all; k0 += kMbfsPullGroup) {
            unsigned long long f[kMbfsPullGroup];
#pragma unroll
            for (uint32_t j = 0; j < kMbfsPullGroup; ++j) f[j] = k0 + j < deg ? frontier[u[j]] : 0ull;
            // the next round's sources while the masks are on their way
#pragma unroll
            for (uint32_t j = 0; j < kMbfsPullGroup; ++j) {
                const uint32_t k = k0 + kMbfsPullGroup + j;
                u[j] = k < deg ? src[(size_t)k * kWave] : 0u;
            }
#pragma unroll
            for (uint32_t j = 0; j < kMbfsPullGroup; ++j) {
                if (all || k0 + j >= deg) continue;
                found |= f[j];
                ++acc.probes;
                all = (found | vis) == full;
            }
        }
        if (mine) {
            const unsigned long long nx = found & ~vis;
            nxt[p] = nx;
            mbfs_set_level<T>(a, lv, p, nx);
            if (nx) {
                a.visited[p] = vis | nx;
                acc.add(a, nx, a.out[p].y);
            }
        }
    }
}

struct MbfsTileLds {
    uint32_t sm[4], lg[4], base_sm, base_lg;
};

// The frontier that the next push reads, in tiles of kMbfsTile vertices: after a push (kUpdate) new =
// next & ~visited with masks, level and sums, else the frontier as it is; its vertices with out-edges
// appended to the queues.  Bound by its passes over the masks.
template <class T, bool kUpdate>
__device__ __forceinline__ void mbfs_tiles(const MbfsArgs& a, uint32_t lv, unsigned long long* __restrict__ nxt,
                                           MbfsLine* __restrict__ queued, uint32_t* __restrict__ hubs, MbfsAcc& acc,
                                           MbfsTileLds& L) {
    const uint32_t n = a.n, lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    for (uint64_t base = (uint64_t)blockIdx.x * kMbfsTile; base < n; base += (uint64_t)gridDim.x * kMbfsTile) {
        const uint64_t v0 = base + wv * 4 * kWave + lane;
        unsigned long long nx[4];
        uint32_t dg[4];
        if constexpr (kUpdate) {
            unsigned long long raw[4], vis[4];
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) raw[c] = v0 + c * kWave < n ? a.next[v0 + c * kWave] : 0ull;
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) vis[c] = raw[c] ? a.visited[v0 + c * kWave] : 0ull;
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) {
                const uint64_t v = v0 + c * kWave;
                nx[c] = raw[c] & ~vis[c];
                if (raw[c]) a.next[v] = 0;
                if (nx[c]) a.visited[v] = vis[c] | nx[c];
                if (v < n) nxt[v] = nx[c];
            }
            bool mine[4];
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) mine[c] = v0 + c * kWave < n;
            mbfs_set_levels<T, 4>(a, lv, v0, nx, mine);
        } else {
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) nx[c] = v0 + c * kWave < n ? nxt[v0 + c * kWave] : 0ull;
        }
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) dg[c] = nx[c] ? a.out[v0 + c * kWave].y : 0u;
        unsigned long long msm[4], mlg[4];
        uint32_t csm = 0, clg = 0;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            if (kUpdate && nx[c]) acc.add(a, nx[c], dg[c]);
            msm[c] = __ballot(dg[c] > 0 && dg[c] <= a.large);
            mlg[c] = __ballot(dg[c] > a.large);
            csm += (uint32_t)__popcll(msm[c]);
            clg += (uint32_t)__popcll(mlg[c]);
        }
        if (lane == 0) {
            L.sm[wv] = csm;
            L.lg[wv] = clg;
        }
        __syncthreads();
        const uint32_t sg = (uint32_t)(base / a.span);
        if (threadIdx.x == 0) {
            const uint32_t tsm = L.sm[0] + L.sm[1] + L.sm[2] + L.sm[3], tlg = L.lg[0] + L.lg[1] + L.lg[2] + L.lg[3];
            L.base_sm = tsm ? atomicAdd(&queued[sg].v, tsm) : 0u;
            L.base_lg = tlg ? atomicAdd(hubs, tlg) : 0u;
        }
        __syncthreads();
        uint32_t osm = L.base_sm, olg = L.base_lg;
        for (uint32_t x = 0; x < wv; ++x) {
            osm += L.sm[x];
            olg += L.lg[x];
        }
        uint32_t* q = a.q_small + (size_t)sg * a.span;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const uint32_t v = (uint32_t)(v0 + c * kWave);
            if ((msm[c] >> lane) & 1ull) q[osm + lanes_below(msm[c])] = v;
            if ((mlg[c] >> lane) & 1ull) a.q_large[olg + lanes_below(mlg[c])] = v;
            osm += (uint32_t)__popcll(msm[c]);
            olg += (uint32_t)__popcll(mlg[c]);
        }
        __syncthreads();
    }
}

// End of an update or pull: the workgroup's sums to its counter line and, with kDecide, its ticket of
// `wgs` that have work (two levels, so no address sees more than wgs / kMbfsSegs atomics).  True in the
// first wave of the workgroup that came last.
template <bool kDecide>
__device__ __forceinline__ bool mbfs_finish_launch(MbfsCounters* __restrict__ ctr, const MbfsAcc& acc, uint32_t wgs) {
    __shared__ unsigned long long s_sum[kMbfsSums];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    if (threadIdx.x < kMbfsSums) s_sum[threadIdx.x] = 0;
    __syncthreads();
    auto total = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(x), kWave - 1); };
    const uint32_t active = total(acc.active), probes = total(acc.probes);
    if (active | probes) {  // uniform across the wave
        const uint32_t deg = total(acc.deg), large_deg = total(acc.large_deg);
        const uint32_t small = total(acc.small), large = total(acc.large);
        const unsigned long long bits = wave_sum_u64(acc.bits), edges = wave_sum_u64(acc.edges);
        if (lane == 0) {
            atomicAdd(&s_sum[kMbfsActive], (unsigned long long)active);
            atomicAdd(&s_sum[kMbfsActiveDeg], (unsigned long long)deg);
            atomicAdd(&s_sum[kMbfsLargeDeg], (unsigned long long)large_deg);
            atomicAdd(&s_sum[kMbfsQueued], ((unsigned long long)large << 32) | small);
            atomicAdd(&s_sum[kMbfsProbes], (unsigned long long)probes);
            atomicAdd(&s_sum[kMbfsNewBits], bits);
            atomicAdd(&s_sum[kMbfsReachedEdges], edges);
        }
    }
    __syncthreads();
    if (threadIdx.x >= kWave) return false;
    const uint32_t sg = blockIdx.x % kMbfsSegs;
    const unsigned long long sum = lane < kMbfsSums ? s_sum[lane] : 0ull;
    if (sum) atomicAdd(&ctr->sum[sg].v[lane], sum);
    if constexpr (!kDecide) return false;
    // the workgroup's atomics (all by this wave or returned) have been performed before its ticket
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t last = 0;
    if (lane == 0) {
        const uint32_t members = (wgs - sg + kMbfsSegs - 1) / kMbfsSegs;  // workgroups of line sg
        const uint32_t nsegs = wgs < kMbfsSegs ? wgs : kMbfsSegs;
        if (atomicAdd(&ctr->sub[sg].v, 1u) == members - 1) last = atomicAdd(&ctr->top.v, 1u) == nsegs - 1;
    }
    return __builtin_amdgcn_readfirstlane((int)last) != 0;
}

// Direction of the next superstep, by one wave: fixed, learned, or the direction-optimising
// heuristic.
__device__ __forceinline__ bool mbfs_direction(const MbfsCtl& c, const float* __restrict__ policy, float* s_params) {
    if (c.mode == 1) return false;
    if (c.mode == 2) return true;
    const double alpha = Sched::kAlphaMbfs * c.k;
    const bool plain = c.m <= Sched::kMbfsPullEdges || (double)c.m_f > (double)c.m_u / alpha;
    if (c.mode != 3 || !policy ||
        !bfs_policy_consulted(false, (double)c.n_f, (double)c.m_f, (double)c.m_u, (double)c.n, alpha, Sched::kBeta))
        return plain;
    const double rec[MEDUSA_TRACE_FIELDS] = {(double)c.step, (double)c.n_f, (double)c.m_f, (double)c.n_u,
                                             (double)c.m_u, (double)c.n, (double)c.m, 0.0, 0.0};
    float c_push, c_pull;
    policy_direction_costs_wave(rec, policy, s_params, c_push, c_pull);
    return policy_pull(c_push, c_pull, plain);
}

// One wave, after every workgroup of an update or pull (or the start, when `first`) has added its
// counters: folds them into the control block, decides the next superstep and clears them.
__device__ __forceinline__ void mbfs_decide(const MbfsArgs& a, bool first, uint32_t slot, float* s_params) {
    MbfsCounters* ctr = a.ctr;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    unsigned long long line[kMbfsSums];
#pragma unroll
    for (int i = 0; i < kMbfsSums; ++i) line[i] = lane < kMbfsSegs ? load_now(&ctr->sum[lane].v[i]) : 0ull;
    MbfsCtl c = load_now_block(a.ctl + slot);
    auto total = [](unsigned long long x) {
        return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan((uint32_t)x), kWave - 1);
    };
    const uint32_t n_active = total(line[kMbfsActive]), active_deg = total(line[kMbfsActiveDeg]);
    const uint32_t large_deg = total(line[kMbfsLargeDeg]), probes = total(line[kMbfsProbes]);
    const uint32_t n_small = total(line[kMbfsQueued]), n_large = total(line[kMbfsQueued] >> 32);
    const unsigned long long bits = wave_sum_u64(line[kMbfsNewBits]), edges = wave_sum_u64(line[kMbfsReachedEdges]);
    const uint32_t par = (uint32_t)c.step & 1u;
    const unsigned long long n = c.n;
    if (!first) {
        // byte model of the superstep just finished: push = queue + offsets + mask per active
        // vertex, col + visited + next probe per edge; pull = offsets + visited per vertex,
        // source + frontier mask per probe; update = 24n
        const unsigned long long kb = c.pull ? 4ull * (n + 1) + 8ull * n + 12ull * probes
                                             : 20ull * c.n_f + 20ull * c.m_f;
        c.kernel_bytes += kb;
        c.alg_bytes += kb + 24ull * n + bits;
        c.supersteps += 1;
        if (c.pull) c.pull_steps += 1; else c.push_steps += 1;
        c.slots += c.pull ? 1u : 2u;
        c.step += 1;
    }
    if (c.step >= 255 && n_active) c.saturated = 1;
    c.reached += bits;
    c.reached_edges += edges;
    c.n_u -= bits;
    c.m_u -= edges;
    c.n_f = n_active;
    c.m_f = active_deg;
    c.n_small = n_small;
    c.n_large = n_large;
    c.hub_wgs = mbfs_hub_wgs(a.grid, n_small, n_large, large_deg, active_deg);
    if (n_active == 0) c.done = 1;
    const bool queued = first || !c.pull;  // by the start or the update
    c.pull = !c.done && mbfs_direction(c, a.policy, s_params) ? 1u : 0u;
    c.phase = c.pull ? kMbfsPull : queued ? kMbfsPush : kMbfsQueue;
    if (c.phase == kMbfsQueue && !c.done) c.slots += 1;
    if (lane < kMbfsSegs) {
#pragma unroll
        for (int i = 0; i < kMbfsSums; ++i) ctr->sum[lane].v[i] = 0;
        ctr->sub[lane].v = 0;
        if (!first) ctr->queued[par][lane].v = 0;  // the queue of the superstep just finished
    }
    if (lane == 0) {
        ctr->top.v = 0;
        if (!first) ctr->hubs[par].v = 0;
        a.ctl[first ? slot : slot ^ 1u] = c;
    }
}

struct MbfsSources {
    uint32_t v[64];
};

// The k sources (any of them repeated) at level 0: masks, queues and counters; one workgroup of one
// wave.  `decide`: and the first decision.
__global__ __launch_bounds__(kWave) void k_mbfs_start(MbfsArgs a, MbfsSources src, uint32_t k, uint32_t decide) {
    __shared__ float s_params[kMlpWaveLds];
    const uint32_t lane = threadIdx.x;
    const uint32_t v = lane < k ? a.pos[src.v[lane]] : 0xFFFFFFFFu;  // (vertices are below 2^32 - 1)
    unsigned long long mask = 0;
    for (uint32_t j = 0; j < k; ++j)
        if (v == (uint32_t)__builtin_amdgcn_readlane((int)v, j)) mask |= 1ull << j;
    const bool one = lane < k && (uint32_t)__builtin_ctzll(mask) == lane;  // the first of its vertex
    MbfsAcc acc;
    if (one) {
        const uint32_t deg = a.out[v].y;
        a.frontier[0][v] = mask;
        a.visited[v] = mask;
        acc.add(a, mask, deg);
    }
    const unsigned long long sm = __ballot(acc.small != 0), lm = __ballot(acc.large != 0);
    if (acc.small) a.q_small[lanes_below(sm)] = v;  // segment 0
    if (acc.large) a.q_large[lanes_below(lm)] = v;
    if (lane == 0) {
        a.ctr->queued[0][0].v = (uint32_t)__popcll(sm);
        a.ctr->hubs[0].v = (uint32_t)__popcll(lm);
    }
    mbfs_finish_launch<false>(a.ctr, acc, 1);
    if (!decide) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // its atomics have been performed
    mbfs_decide(a, true, 0, s_params);
}

// One launch of the superstep loop, doing what the control block says.  Pushes take the first a.grid
// workgroups, pulls at least kMbfsPullGrid and the other passes over the vertices all of them: a caller's
// small grid is for the expansion of a frontier.  64 sources, 64 workgroups asked for: Chung-Lu with 600 K
// vertices 2.52 ms where every pass had only those, 0.94 now; RMAT-18 1.03 and 0.34.  (Pulls of RMAT-18 are
// faster on 512 workgroups than on all 2048, 344 and 400 us a run; Erdos-Renyi's slower, 583 and 567.)
template <class T, bool kDecide>
__global__ __launch_bounds__(256, 8) void k_mbfs_super(MbfsArgs a, uint32_t slot) {
    __shared__ MbfsPushLds s_push;
    __shared__ MbfsTileLds s_tile;
    __shared__ float s_params[kDecide ? kMlpWaveLds : 4];
    const MbfsCtl* ctl = a.ctl + slot;
    // the control block with the phase that follows in the same superstep, for the next launch
    auto pass_on = [&](uint32_t phase) {
        if (!kDecide || blockIdx.x != 0 || threadIdx.x >= sizeof(MbfsCtl) / 4) return;
        uint32_t x = reinterpret_cast<const uint32_t*>(ctl)[threadIdx.x];
        if (threadIdx.x == offsetof(MbfsCtl, phase) / 4) x = phase;
        reinterpret_cast<uint32_t*>(a.ctl + (slot ^ 1u))[threadIdx.x] = x;
    };
    const uint32_t phase = ctl->phase;
    if (ctl->done) {
        pass_on(phase);
        return;
    }
    const uint32_t step = (uint32_t)ctl->step, par = step & 1u;
    const uint32_t lv = mbfs_code(step + 1);
    MbfsAcc acc;
    if (phase == kMbfsPush) {
        pass_on(kMbfsUpdate);
        const uint32_t hub = ctl->hub_wgs;
        if (blockIdx.x >= a.grid) return;
        if (blockIdx.x < hub) {
            mbfs_push_large(a, ctl->n_large, a.frontier[par], blockIdx.x, hub);
        } else {
            const uint32_t wg = blockIdx.x - hub, nwg = a.grid - hub;
            if (wg * 4 >= ctl->n_small) return;  // no entry for its waves
            mbfs_push_small(a, a.ctr->queued[par], a.frontier[par], wg * 4 + threadIdx.x / kWave, nwg * 4, s_push);
        }
        return;
    }
    if (phase == kMbfsQueue) {
        pass_on(kMbfsPush);
        mbfs_tiles<T, false>(a, lv, a.frontier[par], a.ctr->queued[par], &a.ctr->hubs[par].v, acc, s_tile);
        return;
    }
    // workgroups without a slice, hub or tile leave at once, without a ticket (RMAT-18 pushed from one source
    // 254 us before, 248 now; 25 K vertices, 16 sources 478 and 470)
    const uint32_t wgs = phase == kMbfsPull ? min(mbfs_pull_wgs(a), (max(a.nslices, a.nhubs) + 3) / 4)
                                            : min(gridDim.x, (a.n - 1) / kMbfsTile + 1);
    if (blockIdx.x >= wgs) return;
    if (phase == kMbfsPull)
        mbfs_pull<T>(a, ctl->full, lv, a.frontier[par], a.frontier[par ^ 1u], acc);
    else
        mbfs_tiles<T, true>(a, lv, a.frontier[par ^ 1u], a.ctr->queued[par ^ 1u], &a.ctr->hubs[par ^ 1u].v, acc,
                            s_tile);
    if (mbfs_finish_launch<kDecide>(a.ctr, acc, wgs)) mbfs_decide(a, false, slot, s_params);
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
// wave writes 256 contiguous bytes of a row at a time.  RMAT-20, 64 sources: 30 us for 64 MiB of levels
// from 40 of planes and masks.
template <class T>
__global__ __launch_bounds__(1024) void k_mbfs_finish(MbfsArgs a, MbfsHost* __restrict__ host, uint8_t* out,
                                                      uint32_t row0, uint32_t row1) {
    const MbfsCtl* ctl = a.ctl;  // a batch has an even number of launches
    if (host) {
        if (blockIdx.x == 0 && blockIdx.y == 0) {
            if (threadIdx.x < sizeof(MbfsCtl) / 8)
                reinterpret_cast<unsigned long long*>(&host->ctl)[threadIdx.x] =
                    reinterpret_cast<const unsigned long long*>(ctl)[threadIdx.x];
            if (threadIdx.x == 0) host->t_end = (unsigned long long)wall_clock64();
        }
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
        uint32_t at[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) at[i] = a.pos[i < cnt ? v0 + i : v0];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) vis[i] = a.visited[at[i]];
        // a vertex that no source reaches has no level to read
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
#pragma unroll
            for (uint32_t p = 0; p < kMbfsPlanes; ++p)
                x[p][i] = p < np && vis[i] ? planes[(size_t)p * n + at[i]] : (T)0;
        if (np == kMbfsPlanes) {  // uniform: codes back to levels (mbfs_code)
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                T some = 0, every = (T)~(T)0;
#pragma unroll
                for (uint32_t p = 0; p < kMbfsPlanes - 1; ++p) {
                    some |= x[p][i];
                    every &= x[p][i];
                }
                const T saturated = x[kMbfsPlanes - 1][i] & (T)~some, l128 = x[kMbfsPlanes - 1][i] & every;
#pragma unroll
                for (uint32_t p = 0; p < kMbfsPlanes - 1; ++p) x[p][i] = (T)((x[p][i] & (T)~l128) | saturated);
            }
        }
#pragma unroll
        for (uint32_t h = 0; h < (sizeof(T) == 8 ? 2u : 1u); ++h) {
            auto word = [h](unsigned long long w) { return (uint32_t)(w >> (32 * h)); };
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                if (gridDim.y > 1 && blockIdx.y != 4 * h + j) continue;
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
    if (!host) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        host->made[(blockIdx.y * gridDim.x + blockIdx.x) % kMbfsEnds] = (unsigned long long)wall_clock64();
}

// Host-driven launch: the host's decision written into the control block, and into the second one for the
// update that follows a push.  `first` of a superstep: every counter cleared except its own queue's
// (parity step % 2).
__global__ __launch_bounds__(kWave) void k_mbfs_set_ctl(MbfsCtl* ctl, MbfsCounters* c, uint32_t first, int32_t step,
                                                        uint32_t phase, uint32_t n_small, uint32_t n_large,
                                                        uint32_t hub_wgs) {
    const uint32_t lane = threadIdx.x, par = (uint32_t)step & 1u;
    if (lane == 0) {
        ctl->step = step;
        ctl->phase = phase;
        ctl->n_small = n_small;
        ctl->n_large = n_large;
        ctl->hub_wgs = hub_wgs;
        MbfsCtl c1 = *ctl;
        c1.phase = kMbfsUpdate;
        ctl[1] = c1;
    }
    if (!first) return;
    if (lane < kMbfsSegs) {
        for (int i = 0; i < kMbfsSums; ++i) c->sum[lane].v[i] = 0;
        c->queued[par ^ 1u][lane].v = 0;
    }
    if (lane == 0) c->hubs[par ^ 1u].v = 0;
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
    const uint32_t large = mbfs_large(g, o), grid = mbfs_grid(g, o), wgs = std::max(grid, kMbfsGridDefault);
    g->q_small.ensure((size_t)kMbfsSegs * mbfs_span(n));
    g->q_large.ensure(n);
    DBuf<unsigned long long>& masks = g->bitmap;
    masks.ensure(4 * (size_t)n);
    DBuf<uint32_t>& planes = g->stamp;  // reused as the storage of the level planes
    planes.ensure((kMbfsPlanes * sizeof(T) * (size_t)n + 3) / 4);
    // the two control blocks, then the counters
    static_assert(sizeof(MbfsCtl) <= sizeof(CtlStorage), "control block storage");
    static_assert(sizeof(MbfsCtl) % 8 == 0 && sizeof(CtlStorage) % 128 == 0, "control block and counter alignment");
    g->mbfs_ctl.ensure(2 + (sizeof(MbfsCounters) + sizeof(CtlStorage) - 1) / sizeof(CtlStorage));
    MbfsCtl* ctl = reinterpret_cast<MbfsCtl*>(g->mbfs_ctl.p);
    MbfsCounters* C = reinterpret_cast<MbfsCounters*>(g->mbfs_ctl.p + 2);
    static_assert(sizeof(MbfsCounters) <= kHostWords * 8, "pinned memory of a handle");
    MbfsHost* host = host_counters<MbfsHost>(g);  // (or the host-driven loop's counters)
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
    a.dst = PL.dst.p;
    a.pos = PL.pos.p;
    a.out = PL.out.p;
    a.indeg = PL.indeg.p;
    a.base = PL.base.p;
    a.hub = PL.hub.p;
    a.src = PL.src.p;
    a.q_small = g->q_small.p;
    a.q_large = g->q_large.p;
    a.visited = masks.p;
    a.next = masks.p + n;
    a.frontier[0] = masks.p + 2 * (size_t)n;
    a.frontier[1] = masks.p + 3 * (size_t)n;
    a.ctr = C;
    a.ctl = ctl;
    a.policy = policy;
    a.planes = planes.p;
    a.n = n;
    a.large = large;
    a.nslices = PL.nslices;
    a.nhubs = PL.nhubs;
    a.grid = grid;
    a.span = mbfs_span(n);
    // a workgroup per window of the layout, which fetches every line of it once, where that fills the
    // 256 CUs (RMAT-20 30 us against 35 with quarters of windows), else quarters
    const uint32_t finish_wg = n >= 256 * kPullWindow ? 1024 : 256;
    // on few vertices the rows are dealt over workgroups too: a workgroup with all 64 of them is a chain
    // of 256 stores a lane (25 K vertices, 46 sources: 11.9 us, 7.3 dealt out)
    const dim3 finish_grid(grid_for(n, 4 * finish_wg, 8192), n < kMbfsSplitRows ? 4 * ((sizeof(T) + 3) / 4) : 1);
    const bool direct = kernels_can_write(g, out, (size_t)k * n);  // else the rows are copied out at the end

    // capture (once per buffers, launch shape, policy buffer and slot count) a batch of launches
    auto captured = [&](uint32_t slots) -> hipGraphExec_t {
        static_assert(kHeadStep % 2 == 0, "a batch starts and ends with the first control block");
        GraphCache& gc = g->mbfs_heads[__builtin_ctz(sizeof(T))][slots / kHeadStep];
        const uintptr_t key[7] = {(uintptr_t)masks.p,   (uintptr_t)policy,
                                  ((uintptr_t)grid << 32) | large,
                                  (uintptr_t)planes.p,  (uintptr_t)host,
                                  (uintptr_t)a.q_small, (uintptr_t)a.q_large};
        if (gc.exec && std::equal(key, key + 7, gc.key)) return gc.exec;
        gc.reset();
        MDS_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        hipGraph_t graph = nullptr;
        try {
            for (uint32_t b = 0; b < slots; ++b)
                hipLaunchKernelGGL((k_mbfs_super<T, true>), dim3(wgs), dim3(256), 0, s, a, b & 1u);
            hipLaunchKernelGGL(k_mbfs_finish<T>, finish_grid, dim3(finish_wg), 0, s, a, host, (uint8_t*)nullptr, 0u,
                               0u);
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
        std::copy(key, key + 7, gc.key);
        return gc.exec;
    };
    uint32_t slots = next_slots(g->mbfs_last_slots, 0, kMbfsBatch);
    hipGraphExec_t exec = host_driven ? nullptr : captured(slots);

    MbfsSources sources{};
    std::copy(srcs, srcs + k, sources.v);
    if (host_driven) MDS_HIP(hipEventRecord(g->ev_begin, s));
    hipLaunchKernelGGL(k_mbfs_fill, dim3(grid_for(3ull * n, 256, 4096)), dim3(256), 0, s, a, (unsigned long long)m, k,
                       mode, direct ? out : nullptr, host);
    MDS_LAUNCHED();
    hipLaunchKernelGGL(k_mbfs_start, dim3(1), dim3(kWave), 0, s, a, sources, k, host_driven ? 0u : 1u);
    MDS_LAUNCHED();

    MbfsCtl h{};
    if (!host_driven) {
        for (uint64_t done = 0;; exec = captured(slots = next_slots(g->mbfs_last_slots, done, kMbfsBatch))) {
            MDS_HIP(hipGraphLaunch(exec, s));
            MDS_HIP(hipStreamSynchronize(s));
            if (host->ctl.done) break;
            done += slots;
            MDS_CHECK(done < 3ull * n + 16ull * kMbfsBatch, MEDUSA_ERR_INTERNAL, "mbfs: superstep loop did not end");
        }
        h = host->ctl;
        g->mbfs_last_slots = h.slots;
        unsigned long long t_end = host->t_end;
        const uint32_t ends = std::min(finish_grid.x * finish_grid.y, kMbfsEnds);
        if (direct) t_end = std::max(t_end, *std::max_element(host->made, host->made + ends));
        st.device_ms = (double)(t_end - host->t_begin) / (double)g->wall_khz;
    } else {
        Sched sched(o, Sched::kMbfs, k);
        const bool timing = o.timing != 0;
        if (timing) ensure_events(g, 2);
        unsigned long long c[kMbfsSums];
        auto read_sums = [&]() {  // waits for the stream
            MDS_HIP(hipMemcpyAsync(g->h_ctr_raw.p, C, sizeof(C->sum), hipMemcpyDeviceToHost, s));
            MDS_HIP(hipStreamSynchronize(s));
            const MbfsCounters* x = reinterpret_cast<const MbfsCounters*>(g->h_ctr_raw.p);
            for (int i = 0; i < kMbfsSums; ++i) {
                c[i] = 0;
                for (uint32_t sg = 0; sg < kMbfsSegs; ++sg) c[i] += x->sum[sg].v[i];
            }
        };
        bool first = true;  // launch of a superstep
        auto decide = [&](uint32_t t, uint32_t phase) {
            const uint32_t n_small = (uint32_t)c[kMbfsQueued], n_large = (uint32_t)(c[kMbfsQueued] >> 32);
            hipLaunchKernelGGL(k_mbfs_set_ctl, dim3(1), dim3(kWave), 0, s, ctl, C, first ? 1u : 0u, (int32_t)t, phase,
                               n_small, n_large,
                               mbfs_hub_wgs(grid, n_small, n_large, c[kMbfsLargeDeg], c[kMbfsActiveDeg]));
            MDS_LAUNCHED();
            first = false;
        };
        auto launch = [&](uint32_t slot) {
            hipLaunchKernelGGL((k_mbfs_super<T, false>), dim3(wgs), dim3(256), 0, s, a, slot);
            MDS_LAUNCHED();
        };
        read_sums();
        Frontier f{};
        f.n = n;
        f.m = m;
        h.n_u = (uint64_t)n * k - c[kMbfsNewBits];
        h.m_u = (uint64_t)m * k - c[kMbfsReachedEdges];
        h.reached = c[kMbfsNewBits];
        h.reached_edges = c[kMbfsReachedEdges];
        bool pull = false, queued = true;
        for (uint32_t t = 0; c[kMbfsActive]; ++t) {
            f.step = t;
            f.n_f = c[kMbfsActive];
            f.m_f = c[kMbfsActiveDeg];
            f.n_u = h.n_u;
            f.m_u = h.m_u;
            if (o.direction == MEDUSA_DIR_PUSH) pull = false;
            else if (o.direction == MEDUSA_DIR_PULL) pull = true;
            else pull = sched.bfs_pull(f, pull);
            first = true;
            if (!pull && !queued) {
                decide(t, kMbfsQueue);
                launch(0);
            }
            decide(t, pull ? kMbfsPull : kMbfsPush);
            if (timing) MDS_HIP(hipEventRecord(g->events[0], s));
            launch(0);
            if (!pull) launch(1);  // the update
            if (timing) MDS_HIP(hipEventRecord(g->events[1], s));
            queued = !pull;
            read_sums();
            double kms = 0;
            if (timing) {
                float ms = 0;
                MDS_HIP(hipEventElapsedTime(&ms, g->events[0], g->events[1]));
                kms = ms;
                st.kernel_ms += ms;
                ++st.kernel_launches;
            }
            const uint64_t kb = pull ? 4ull * (n + 1) + 8ull * n + 12ull * c[kMbfsProbes]
                                     : 20ull * f.n_f + 20ull * f.m_f;
            h.kernel_bytes += kb;
            h.alg_bytes += kb + 24ull * n + c[kMbfsNewBits];
            if (pull) ++h.pull_steps; else ++h.push_steps;
            sched.record(g, f, pull ? 1.0 : 0.0, kms);
            ++h.supersteps;
            if (t + 1 >= 255 && c[kMbfsNewBits]) h.saturated = 1;
            h.reached += c[kMbfsNewBits];
            h.reached_edges += c[kMbfsReachedEdges];
            h.n_u -= c[kMbfsNewBits];
            h.m_u -= c[kMbfsReachedEdges];
        }
        // the last level, for the finish
        hipLaunchKernelGGL(k_mbfs_set_ctl, dim3(1), dim3(kWave), 0, s, ctl, C, 0u, (int32_t)h.supersteps, 0u, 0u, 0u,
                           0u);
        MDS_LAUNCHED();
        if (direct) {
            hipLaunchKernelGGL(k_mbfs_finish<T>, finish_grid, dim3(finish_wg), 0, s, a, (MbfsHost*)nullptr, out, 0u, k);
            MDS_LAUNCHED();
        }
        MDS_HIP(hipEventRecord(g->ev_end, s));
        MDS_HIP(hipStreamSynchronize(s));
        float ms = 0;
        MDS_HIP(hipEventElapsedTime(&ms, g->ev_begin, g->ev_end));
        st.device_ms = ms;
    }
    st.supersteps = h.supersteps;
    st.push_steps = h.push_steps;
    st.pull_steps = h.pull_steps;
    st.kernel_bytes = h.kernel_bytes;
    st.alg_bytes = h.alg_bytes + (uint64_t)k * n + 24ull * n;
    st.edges_traversed = h.reached_edges;
    st.reached = (uint32_t)std::min<uint64_t>(h.reached, 0xFFFFFFFFull);
    st.reserved[0] = h.saturated;
    if (direct) return;
    check_device_output(g, out, (size_t)k * n);  // before the first row is written
    // as many rows at a time as the row buffer holds
    const uint32_t rows = (uint32_t)std::min<uint64_t>(k, std::max<uint64_t>(1, kMbfsRowBytes / n));
    g->mbfs_rows.ensure(((size_t)rows * n + 3) / 4);
    for (uint32_t r = 0; r < k; r += rows) {
        const uint32_t r1 = std::min(k, r + rows);
        uint8_t* buf = reinterpret_cast<uint8_t*>(g->mbfs_rows.p);
        MDS_HIP(hipEventRecord(g->ev_begin, s));
        hipLaunchKernelGGL(k_mbfs_finish<T>, finish_grid, dim3(finish_wg), 0, s, a, (MbfsHost*)nullptr, buf, r, r1);
        MDS_LAUNCHED();
        MDS_HIP(hipEventRecord(g->ev_end, s));
        copy_out(g, out + (size_t)r * n, buf, (size_t)(r1 - r) * n);  // waits for the stream
        float ms = 0;
        MDS_HIP(hipEventElapsedTime(&ms, g->ev_begin, g->ev_end));
        st.device_ms += ms;
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
