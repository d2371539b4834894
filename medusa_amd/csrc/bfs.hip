// BFS superstep engine.
//
// Reference: every superstep FunctorHolder<EDGE>::Run(UpdateLevel) sweeps all |E|
// edges (MultipleGPU/MultiAPIHoster.h:657-678, MedusaRT/APIKernelWrappers.h:34-44):
// if level[src]==step and level[dst]==-1 then level[dst]=step+1 and vote to
// continue (Algorithm/UserOperators.h:17-36, MedusaRT/SystemLibGPU.h:19-22); the
// host loop resets and reads the vote each step (Algorithm/main.cu:283-302,
// MultipleGPU/MultiUtilities.h:48-69).  Levels are int32, -1 = unreached
// (Algorithm/Message.h:9-10).
//
// Any number of sources may be given (medusa_bfs_multi): all start at level 0, which on a
// packed batch of disjoint graphs with one source per graph gives every graph's own BFS
// levels in one run.  Here a superstep is ONE kernel that only touches the frontier and
// builds the next one as it goes:
//   frontier: a queue in segments plus a queue of its hubs (out-degree above `large`), and which
//          vertices have been visited as a bitmap;
//   push:  waves take queue entries and share their out-edges through an in-wave prefix scan;
//          hubs are split over whole workgroups; a target is claimed by the lane whose 64-bit
//          atomic OR first sets its visited bit, so each joining vertex is counted exactly once
//          (large frontiers store levels instead, and a compaction finds who joined);
//   pull:  every unvisited vertex scans its in-edges for a visited vertex and stops at the first
//          hit; each wave owns some words of the next bitmap and writes them whole, no atomics;
//   counters: joined vertices, their out-degrees, hub degrees and probed in-edges, summed
//          per workgroup into two packed 64-bit atomics; joined hubs are appended to the next
//          hub queue (one atomic per wave that has any);
//   direction: Beamer's rule with thresholds measured for this GPU (Sched), or the
//          learned policy near the rule's switching point.
// In the reference every writer stores the same level, so its claim is a plain store; here the
// first setter of the bit also writes the level, which gives the same levels.
//
//   solo:  while a frontier has few out-edges one workgroup runs superstep after superstep by
//          itself, with the frontier in LDS, instead of a launch of the whole grid for each.
//
// Two drivers run the same kernel:
//   device-driven (default): the last workgroup of each superstep (by a ticket taken after
//     its counters) decides the next one (direction, hub queue split, the termination vote)
//     into a control block in HBM.  A run is one hipGraph: the reset, a starting kernel that
//     reads the run's parameters from pinned host memory, a number of superstep slots (as many as
//     the previous run on the handle used) and a closing kernel that copies the levels out and
//     the control block to pinned memory; the host launches it and waits once, and replays
//     batches of kBfsBatch slots if the control block does not say done (a handle's first run
//     launches the same kernels one by one);
//   host-driven (timing or trace requested): the host reads the counters after every
//     superstep, times it with hipEvents and logs the trace record.

#include <algorithm>
#include <cstddef>

#include "engine.h"
#include "sched.h"

namespace medusa {

// kBfsLargeDefault, the out-degree above which a frontier vertex is split over workgroups.  Below it one
// wave walks the whole list, 256 out-edges at a time, and the superstep waits for the longest.  us a run
// at thresholds of 384, 512, 768, 1024, 1280 and 2048: Chung-Lu with 2.4 M vertices (out-degrees up to 39914)
// 340, 345, 361, 378, 398 and 445; 8 M 711, 703, 719, 740, 764 and 830; 600 K 183, 185, 189, 193, 196
// and 207; RMAT-20 (up to 598) 268 at 384 and 155 from 512 on; RMAT-22 (up to 866) 491, 484 and 339..334 from
// 768 on.  So 768 or 1024 would be faster for the heuristic: it stays at 1280 for the learned direction,
// whose gain over it on the 2.4 M-vertex graph is 6.3..6.9 % at 1280, 2.6..3.2 % at 1024 and none at 768 (six
// trainings), where it has to be 2 %.  The autotuner finds the lower thresholds for a caller's graph.
constexpr uint32_t kLargeSplit = 16;  // workgroups per hub in the large-vertex push
constexpr uint32_t kBfsBatch = 8;     // supersteps per captured graph

// Control block of the device-driven loop.  There are two: launch k of a batch reads block k % 2
// and leaves the next launch's in the other, so a workgroup that starts late never sees what an
// early one of the same launch has written.
struct BfsCtl {
    int32_t step;       // superstep being run (= level of the frontier)
    uint32_t pull;      // direction of this superstep
    uint32_t done;      // the vote: no vertex joined the frontier
    uint32_t n_small, n_large;
    uint32_t supersteps, push_steps, pull_steps;
    uint32_t mode;      // 0 heuristic, 1 push, 2 pull, 3 learned policy
    uint32_t hub_wgs;   // push: workgroups of the expansion given to the hub queue
    uint32_t pending;   // a push with plain claims has run and its compaction has not
    uint32_t small;     // push with exact (atomic) claims: the frontier's out-edges fit one queue segment
    uint32_t slots;     // kernel launches the loop has used (a push with plain claims takes two)
    uint32_t vsel;      // which visited bitmap is current
    unsigned long long n, m, n_f, m_f, n_u, m_u, reached, reached_edges, kernel_bytes, alg_bytes;
    int32_t* out;              // where the closing kernel copies the levels (null: nowhere)
    unsigned long long t_begin;  // wall clock at the reset
};

// Pinned host memory of a device-driven run.
constexpr uint32_t kBfsHostSources = 4096;    // sources the starting kernel takes from here
constexpr size_t kBfsStageBytes = 1u << 20;   // levels up to which a host output goes through pinned memory
struct BfsHost {
    BfsCtl ctl;                // written by the closing kernel
    unsigned long long t_end;  // wall clock after the last superstep
    int32_t* out;              // the run's parameters, read by the starting kernel
    uint32_t count, mode;
    uint32_t src[kBfsHostSources];
};
static_assert(sizeof(BfsHost) <= kHostWords * 8, "pinned memory of a handle");

// Workgroups of a push expansion given to the hub queue: in proportion to its share of
// the frontier's out-edges, at least one for each non-empty queue.
__host__ __device__ inline uint32_t bfs_hub_wgs(uint32_t grid, uint32_t n_small, uint32_t n_large,
                                                unsigned long long deg_large, unsigned long long deg_sum) {
    if (!n_large) return 0;
    if (!n_small) return grid;
    unsigned long long h = deg_sum ? (unsigned long long)grid * deg_large / deg_sum : 1ull;
    if (h < 1) h = 1;
    if (h > grid - 1) h = grid - 1;
    return (uint32_t)h;
}

// Host-driven superstep: the host's decision written into the control block.
__global__ void k_bfs_set_ctl(BfsCtl* ctl, int32_t step, uint32_t pull, uint32_t small, uint32_t n_small,
                              uint32_t n_large, uint32_t hub_wgs, uint32_t vsel) {
    ctl->step = step;
    ctl->pull = pull;
    ctl->small = small;
    ctl->done = 0;
    ctl->n_small = n_small;
    ctl->n_large = n_large;
    ctl->hub_wgs = hub_wgs;
    ctl->pending = 0;
    ctl->vsel = vsel;
    BfsCtl c = *ctl;  // for the compaction, if one follows
    c.pending = 1;
    ctl[1] = c;
}

// Counters of one superstep.  Atomics on one address serialise (about 10 ns each on this
// GPU), so they are spread over kBfsSlots addresses, each on its own 128-byte line:
//   seg[p][s]: the frontier of parity p (superstep t's frontier has parity t % 2) is a queue
//     in kBfsSlots segments of `span` entries, filled by rounds of vertices (bfs_round_segment)
//     or by workgroups (exact claims); its counter packs the vertices appended (low half, also
//     the append offset) and the sum of their out-degrees (high half);
//   work[s]: workgroup b adds the out-degree sum of the hubs it found (low half) and the
//     in-edges it probed (high half) into slot b % kBfsSlots;
//   sub / top: two levels of tickets that find the last workgroup of a superstep.
// Every half's total is bounded by n or by m (both below 2^32), so no carry crosses into a
// high half.
constexpr uint32_t kBfsSlots = 32;
constexpr uint32_t kBfsRound = 1024;  // vertices per workgroup round of the compaction; segment spans are multiples
struct BfsLine {
    alignas(128) unsigned long long v;
};
struct BfsTicket {
    alignas(128) uint32_t v;
};
struct BfsCounters {
    BfsLine seg[2][kBfsSlots];
    BfsLine work[kBfsSlots];
    BfsTicket sub[kBfsSlots];      // workgroups of slot s that have finished the superstep
    MDS_COUNTER(uint32_t, top);    // slots whose workgroups have all finished
    MDS_COUNTER(uint32_t, n_hub);  // joined hubs, appended to the next hub queue
};

// Buffers and shape of a BFS run, passed by value to every superstep kernel.  Superstep t
// reads the frontier as queue q[t % 2] (push) and hub queue hub[t % 2] and builds the next
// frontier's in q[(t + 1) % 2] and hub[(t + 1) % 2].  A pull needs no frontier bitmap: all
// out-neighbours of the earlier frontiers have been visited, so a visited in-neighbour of an
// unvisited vertex is in the frontier.  It reads one visited bitmap and writes the other, which is
// then the current one; pushes change the current one in place.  (Three frontier bitmaps in
// rotation took a second atomic from every exact claim and a pass that cleared one in every
// superstep; a run's kernels with them and without: RMAT-20 154 and 151 us, Erdos-Renyi with 65536
// vertices 69 and 67, Chung-Lu with 2.4 M 477 and 470.)
struct BfsArgs {
    const uint32_t *row_ptr, *col, *cptr, *csrc;
    int32_t* level;
    uint32_t* q[2];    // segmented queues, kBfsSlots * span entries each
    uint32_t* hub[2];  // hub queues, n entries each
    unsigned long long* vis[2];  // one bit per vertex that has a level (n / 8 bytes, stays in L2)
    BfsCounters* ctr;
    BfsCtl* ctl;
    const float* policy;  // learned direction policy (device parameters) or null
    uint32_t n, nwords, large, grid, span;
    unsigned long long m, exact_edges;  // frontier out-edges up to which a push claims exactly
};

// Segment span for n vertices: kBfsSlots segments cover [0, n) in whole compaction rounds.
__host__ __device__ constexpr uint32_t bfs_span(uint32_t n) {
    const uint64_t per = ((uint64_t)n + kBfsSlots - 1) / kBfsSlots;
    const uint64_t span = (per + kBfsRound - 1) / kBfsRound * kBfsRound;
    return (uint32_t)(span ? span : kBfsRound);
}

// Whether a superstep is run by one workgroup (as a push, whatever the direction heuristic or the
// policy would say of the whole grid) whose LDS holds frontiers of `cap` vertices: the frontier
// and every vertex it may reach must fit, and its out-edges take at most kSoloRounds rounds of cap
// (one, unless the whole graph fits, and so its visited bitmap too).  Erdos-Renyi, 4096 vertices and
// 33 K arcs: 74 us a run with eight rounds, 84 with one (two supersteps of the whole grid then), 130
// with none and no run in one graph.
constexpr uint32_t kSoloRounds = 8;
__host__ __device__ inline bool bfs_solo_fits(uint32_t cap, unsigned long long n, unsigned long long n_f,
                                              unsigned long long m_f) {
    return n_f <= cap && (m_f <= cap || (n <= cap && m_f <= (unsigned long long)kSoloRounds * cap));
}

// A push claims exactly (an atomic OR of the visited bit, no compaction) when the frontier has at most
// `exact_edges` out-edges: 1, or 2 when it also has at most 64 vertices (every wave then reads
// all of them and takes an equal share of their out-edges).  Workgroup b appends its winners to
// segment b mod kBfsSlots of the next queue whatever their ids: exact_edges is at most a
// segment's span, so any segment could hold them all.  (With every winner in segment 0, 4096
// waves added to one counter: 94 us for a superstep of 44 K vertices and 68 K out-edges of the
// 2.4 M-vertex Chung-Lu graph, 24 us with the segments.)
__host__ __device__ inline uint32_t bfs_small(bool pull, unsigned long long n_f, unsigned long long m_f,
                                              unsigned long long exact_edges) {
    return pull || m_f > exact_edges ? 0u : (n_f <= (unsigned long long)kWave ? 2u : 1u);
}

__device__ __forceinline__ unsigned long long bfs_pack(uint32_t lo, uint32_t hi) {
    return (unsigned long long)lo | ((unsigned long long)hi << 32);
}

constexpr uint32_t kRoundChunks = kBfsRound / 256;  // 64-vertex chunks per wave per workgroup round

// Joined vertices that a wave holds in LDS before it appends them to the next queue: an append is a
// chain of three round trips to memory (place, offsets, store), which a wave's rounds share, without a
// barrier.  Compactions of the 2.4 M-vertex Chung-Lu graph, two to three rounds a wave: 16..24 us with an
// append of the workgroup per round, 13 now.
constexpr uint32_t kJoinCap = 1024, kJoinRound = 256;  // entries; most of them added per round
struct BfsJoinLds {
    unsigned long long words[4][kJoinCap / kWave];  // of a pull: joins among the listed vertices of a word
    uint32_t v[4][kJoinCap];
};
struct BfsJoins {
    uint32_t* list;  // the wave's, kJoinCap entries
    uint32_t n = 0;  // uniform
    // Every lane calls it: lanes with `joined` add v.
    __device__ __forceinline__ void put(bool joined, uint32_t v) {
        const unsigned long long m = __ballot(joined);
        if (joined) list[n + lanes_below(m)] = v;
        n += (uint32_t)__popcll(m);
    }
};

// Where a wave's joins go: a segment of the next queue and the hub queue.
struct BfsSink {
    uint32_t* q_next;
    BfsLine* seg_next;
    uint32_t* hub_next;
};

// The wave's held joins, at their place in the next queue; hubs (out-degree above `large`) also go to
// the next hub queue (one atomic per 64 vertices that have any; hubs are few) and their degrees into
// `hacc`.  `place` is called once, behind the first offsets' loads.  Returns the joins' out-degrees
// (of distinct vertices: below 2^32), in every lane.
template <class Place>
__device__ __forceinline__ uint32_t bfs_flush_list(const BfsArgs& a, const BfsJoins& J, const BfsSink& o, Place place,
                                                   unsigned long long& hacc) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t* q = nullptr;
    uint32_t dsum = 0;
    constexpr uint32_t kN = 4;
    for (uint32_t i0 = 0; i0 == 0 || i0 < J.n; i0 += kWave * kN) {
        uint32_t v[kN], b[kN], e[kN];
#pragma unroll
        for (uint32_t j = 0; j < kN; ++j) {
            const uint32_t i = i0 + j * kWave + lane;
            v[j] = i < J.n ? J.list[i] : 0xFFFFFFFFu;
            b[j] = e[j] = 0;
            if (i < J.n) {
                b[j] = a.row_ptr[v[j]];
                e[j] = a.row_ptr[v[j] + 1];
            }
        }
        if (i0 == 0) q = place();
#pragma unroll
        for (uint32_t j = 0; j < kN; ++j) {
            const uint32_t i = i0 + j * kWave + lane, deg = e[j] - b[j];
            if (i < J.n) q[i] = v[j];
            dsum += deg;
            const unsigned long long hm = __ballot(deg > a.large);
            if (hm) {
                uint32_t hb = 0;
                if (lane == 0) hb = atomicAdd(&a.ctr->n_hub, (uint32_t)__popcll(hm));
                hb = __builtin_amdgcn_readfirstlane(hb);
                if (deg > a.large) {
                    o.hub_next[hb + lanes_below(hm)] = v[j];
                    hacc += deg;
                }
            }
        }
    }
    return __builtin_amdgcn_readlane(wave_incl_scan(dsum), kWave - 1);
}

// One wave's held joins appended to segment sg of the next queue: one atomic for their place and
// number, one for their out-degrees, both performed on return.
__device__ __forceinline__ void bfs_flush_wave(const BfsArgs& a, BfsJoins& J, const BfsSink& o, uint32_t sg,
                                               unsigned long long& hacc) {
    if (!J.n) return;  // uniform across the wave
    const bool first = (threadIdx.x & (kWave - 1)) == 0;
    wave_lds_fence();
    uint32_t base = 0;
    if (first) base = (uint32_t)atomicAdd(&o.seg_next[sg].v, bfs_pack(J.n, 0));
    const uint32_t dsum = bfs_flush_list(
        a, J, o, [&] { return o.q_next + (size_t)sg * a.span + __builtin_amdgcn_readfirstlane(base); }, hacc);
    if (first) atomicAdd(&o.seg_next[sg].v, bfs_pack(0, dsum));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    J.n = 0;
    wave_lds_fence();
}

// The same for every wave of the workgroup at once (every thread calls it, all with the same sg), with
// one pair of atomics: at the end of a superstep all waves append, and 4096 pairs on kBfsSlots
// addresses took 1.5 us more than 1024.
__device__ __forceinline__ void bfs_flush(const BfsArgs& a, BfsJoins& J, const BfsSink& o, uint32_t sg,
                                          unsigned long long& hacc) {
    __shared__ uint32_t s_n[4], s_base, s_deg[4];
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    if (lane == 0) s_n[wv] = J.n;
    __syncthreads();
    const uint32_t n = s_n[0] + s_n[1] + s_n[2] + s_n[3];
    if (!n) {  // uniform
        __syncthreads();  // s_n is written again by the next call
        return;
    }
    if (threadIdx.x == 0) s_base = (uint32_t)atomicAdd(&o.seg_next[sg].v, bfs_pack(n, 0));
    const uint32_t dsum = bfs_flush_list(
        a, J, o,
        [&] {
            __syncthreads();
            uint32_t at = s_base;
            for (uint32_t w = 0; w < wv; ++w) at += s_n[w];
            return o.q_next + (size_t)sg * a.span + at;
        },
        hacc);
    if (lane == 0) s_deg[wv] = dsum;
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&o.seg_next[sg].v, bfs_pack(0, s_deg[0] + s_deg[1] + s_deg[2] + s_deg[3]));
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    J.n = 0;
}

// End of a counting kernel: the workgroup's hub degrees and probes go into its slot (one
// atomic), then, with kDecide, it draws a ticket; returns true (to every thread) in the last
// workgroup to finish.  Tickets are drawn only after the counter atomics have returned (the
// asm makes the increment depend on their results), and every wave waited for its appends
// before a barrier above, so when the last ticket is drawn every workgroup's counts have been
// performed at the device's coherence point.  Device-scope atomics and atomic loads are
// coherent across the XCDs' L2 caches without a fence (a device-scope release fence would
// write the L2 back).  Two levels of tickets (per slot, then across slots) keep the atomics on
// any one address to about grid / kBfsSlots.
template <bool kDecide>
__device__ __forceinline__ bool bfs_finish(BfsCounters* __restrict__ ctr, unsigned long long wacc) {
    __shared__ unsigned long long s_sum[4];
    __shared__ uint32_t s_last;
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    wacc = wave_sum_u64(wacc);
    if (lane == 0) s_sum[wv] = wacc;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long tw = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
        const uint32_t s = blockIdx.x % kBfsSlots;
        unsigned long long ret = 0;
        if (tw) ret = atomicAdd(&ctr->work[s].v, tw);
        if (kDecide) {
            uint32_t inc = 1;
            asm volatile("" : "+v"(inc) : "v"(ret));
            const uint32_t members = (gridDim.x - s + kBfsSlots - 1) / kBfsSlots;  // workgroups of slot s
            const uint32_t nslots = gridDim.x < kBfsSlots ? gridDim.x : kBfsSlots;
            bool last = false;
            if (atomicAdd(&ctr->sub[s].v, inc) == members - 1) {
                uint32_t inc2 = 1;
                asm volatile("" : "+v"(inc2) : "v"(members));
                last = atomicAdd(&ctr->top, inc2) == nslots - 1;
            }
            s_last = last ? 1u : 0u;
        }
    }
    if constexpr (!kDecide) return false;
    __syncthreads();
    return s_last != 0;
}

// ---- superstep bodies ---------------------------------------------------------------

// Prefix of the frontier queue's segment counts in LDS (one wave scans them): entries
// [pre[s], pre[s + 1]) of the frontier live in segment s.
__device__ __forceinline__ void bfs_queue_prefix(const BfsLine* __restrict__ seg, uint32_t* pre) {
    if (threadIdx.x < kWave) {
        const uint32_t lane = threadIdx.x;
        const uint32_t c = lane < kBfsSlots ? (uint32_t)seg[lane].v : 0u;
        const uint32_t incl = wave_incl_scan(c);
        if (lane < kBfsSlots) pre[lane + 1] = incl;
        if (lane == 0) pre[0] = 0;
    }
    __syncthreads();
}

// Queue entry i of the frontier.
__device__ __forceinline__ uint32_t bfs_queue_at(const BfsArgs& a, const uint32_t* __restrict__ q, const uint32_t* pre,
                                                 uint32_t i) {
    uint32_t s = 0;  // last segment with pre[s] <= i
#pragma unroll
    for (uint32_t step = kBfsSlots / 2; step; step >>= 1)
        if (pre[s + step] <= i) s += step;
    return q[(size_t)s * a.span + (i - pre[s])];
}

constexpr uint32_t kPushUnroll = 4;  // out-edges per lane per round of the push, loads issued together

// Claims of a round's targets v[j] (0xFFFFFFFF: none) for level `next`; a vertex whose visited bit is
// set is skipped (the bitmap is small enough to stay in L2, the level array is not).  Plain: `level[v]
// = next`, a plain store; every writer stores the same value, so the race is benign (as in the
// reference) and the compaction after the push finds the vertices that joined.
__device__ __forceinline__ void bfs_claim_plain(const BfsArgs& a, const unsigned long long* __restrict__ visited,
                                                const uint32_t (&v)[kPushUnroll], int32_t next) {
#pragma unroll
    for (uint32_t j = 0; j < kPushUnroll; ++j)
        if (v[j] != 0xFFFFFFFFu && !(visited[v[j] >> 6] & (1ull << (v[j] & 63)))) a.level[v[j]] = next;
}

// Exact: whoever sets the visited bit wins the vertex, stores its level and holds it for the next
// queue's segment `own`.  The calling wave is converged.  A wave with many out-edges goes through this
// chain of dependent accesses once per round, so the round's loads and atomics are issued together (a
// compare-and-swap on the level one after the other, then the bit: 34..36 us for 46 K and 62 K out-edges
// of that graph, 20 now).
struct BfsExact {
    unsigned long long* visited;
    BfsSink sink;
    uint32_t own;
    BfsJoins J;
};
__device__ __forceinline__ void bfs_claim_exact(const BfsArgs& a, BfsExact& x, const uint32_t (&v)[kPushUnroll],
                                                int32_t next, unsigned long long& hacc) {
    unsigned long long seen[kPushUnroll];
#pragma unroll
    for (uint32_t j = 0; j < kPushUnroll; ++j) seen[j] = v[j] != 0xFFFFFFFFu ? x.visited[v[j] >> 6] : ~0ull;
#pragma unroll
    for (uint32_t j = 0; j < kPushUnroll; ++j)
        if (!((seen[j] >> (v[j] & 63)) & 1ull)) seen[j] = atomicOr(&x.visited[v[j] >> 6], 1ull << (v[j] & 63));
#pragma unroll
    for (uint32_t j = 0; j < kPushUnroll; ++j) {
        const bool won = !((seen[j] >> (v[j] & 63)) & 1ull);
        if (won) a.level[v[j]] = next;
        x.J.put(won, v[j]);
    }
    static_assert(kJoinRound >= kWave * kPushUnroll, "a round's winners");
    if (x.J.n > kJoinCap - kJoinRound) bfs_flush_wave(a, x.J, x.sink, x.own, hacc);
}

// Wave-cooperative push over the frontier queue (hubs and vertices without out-edges are
// skipped: out-degree taken as 0).  Of the `nwaves` waves taking part (`wave0` is this wave's
// index among them), wave w holds queue entries w, w + nwaves, w + 2*nwaves, ... one per lane,
// so a run of high-degree vertices spreads over many waves instead of sharing one; the lanes
// then share the entries' out-edges through an in-wave prefix scan, kPushUnroll edges per lane
// per round.
template <bool kExact>
__device__ __forceinline__ void push_queue(const BfsArgs& a, const uint32_t* __restrict__ q, const uint32_t* pre,
                                           int32_t next, uint32_t wave0, uint32_t nwaves, uint32_t (*s_beg)[kWave],
                                           uint32_t (*s_off)[kWave], BfsExact& x, unsigned long long& hacc) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const uint32_t qn = pre[kBfsSlots];
    for (uint64_t r = 0; wave0 + r * kWave * nwaves < qn; ++r) {  // uniform across the wave
        const uint64_t i = wave0 + (r * kWave + lane) * nwaves;
        uint32_t beg = 0, deg = 0;
        if (i < qn) {
            const uint32_t u = bfs_queue_at(a, q, pre, (uint32_t)i);
            beg = a.row_ptr[u];
            deg = a.row_ptr[u + 1] - beg;
            if (deg > a.large) deg = 0;  // a hub: expanded from the hub queue
        }
        const uint32_t incl = wave_incl_scan(deg);
        const uint32_t total = __shfl(incl, kWave - 1, kWave);
        s_beg[wv][lane] = beg;
        s_off[wv][lane] = incl - deg;
        __builtin_amdgcn_wave_barrier();
        for (uint32_t e0 = 0; e0 < total; e0 = advance_to(e0, kWave * kPushUnroll, total)) {  // uniform across the wave
            uint32_t v[kPushUnroll];
#pragma unroll
            for (uint32_t j = 0; j < kPushUnroll; ++j) {
                const uint32_t e = e0 + j * kWave + lane;
                v[j] = 0xFFFFFFFFu;
                if (lies_before(e0, j * kWave + lane, total)) {
                    // owner = last lane whose exclusive offset is <= e (it has deg > 0)
                    uint32_t lo = 0;
#pragma unroll
                    for (uint32_t step = kWave / 2; step; step >>= 1)
                        if (s_off[wv][lo + step] <= e) lo += step;
                    v[j] = a.col[s_beg[wv][lo] + (e - s_off[wv][lo])];
                }
            }
            if constexpr (kExact) bfs_claim_exact(a, x, v, next, hacc);
            else bfs_claim_plain(a, x.visited, v, next);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Exact-claim push of a frontier of at most 64 vertices (hubs included): every wave reads the
// whole frontier and its out-degree prefix, and the grid's waves take the out-edges of their
// concatenation 64 * kPushUnroll at a time, wave w the w-th share and every (waves of the grid)-th
// after it, so a frontier of one high-degree vertex still spreads over many waves.  (One share a
// wave covers the default grid's frontiers up to 2^25 vertices, and fewer out-edges on a smaller grid.)
__device__ __forceinline__ void push_tiny(const BfsArgs& a, const uint32_t* __restrict__ q, const uint32_t* pre,
                                          int32_t next, uint32_t (*s_beg)[kWave], uint32_t (*s_off)[kWave],
                                          BfsExact& x, unsigned long long& hacc) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const uint32_t qn = pre[kBfsSlots];
    const uint64_t e_begin = ((uint64_t)blockIdx.x * (blockDim.x / kWave) + wv) * kWave * kPushUnroll;
    uint32_t beg = 0, deg = 0;
    if (lane < qn) {
        const uint32_t u = bfs_queue_at(a, q, pre, lane);
        beg = a.row_ptr[u];
        deg = a.row_ptr[u + 1] - beg;
    }
    const uint32_t incl = wave_incl_scan(deg);
    const uint32_t total = __shfl(incl, kWave - 1, kWave);
    if (e_begin >= total) return;  // uniform across the wave
    s_beg[wv][lane] = beg;
    s_off[wv][lane] = incl - deg;
    __builtin_amdgcn_wave_barrier();
    for (uint64_t e0 = e_begin; e0 < total; e0 += (uint64_t)gridDim.x * blockDim.x * kPushUnroll) {
        uint32_t v[kPushUnroll];
#pragma unroll
        for (uint32_t j = 0; j < kPushUnroll; ++j) {
            const uint64_t e = e0 + j * kWave + lane;
            v[j] = 0xFFFFFFFFu;
            if (e < total) {
                uint32_t lo = 0;
#pragma unroll
                for (uint32_t step = kWave / 2; step; step >>= 1)
                    if (s_off[wv][lo + step] <= e) lo += step;
                v[j] = a.col[s_beg[wv][lo] + ((uint32_t)e - s_off[wv][lo])];
            }
        }
        bfs_claim_exact(a, x, v, next, hacc);
    }
}

// Hubs: each vertex of the hub queue is split into `split` contiguous edge ranges, one per
// workgroup item; the `nwg` workgroups taking part stride over the items.
template <bool kExact>
__device__ __forceinline__ void push_hubs(const BfsArgs& a, const uint32_t* __restrict__ q, uint32_t qn, int32_t next,
                                          uint32_t wg0, uint32_t nwg, BfsExact& x,
                                          unsigned long long& hacc) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t split = nwg / qn;
    split = split < kLargeSplit ? kLargeSplit : (split > 4096u ? 4096u : split);
    for (uint64_t w = wg0; w < (uint64_t)qn * split; w += nwg) {
        const uint32_t u = q[w / split], part = (uint32_t)(w % split);
        const uint32_t b = a.row_ptr[u], deg = a.row_ptr[u + 1] - b;
        const EdgePart E = edge_part(b, deg, part, split);
        const uint32_t cnt = E.hi - E.lo;  // a sixteenth of an edge array at most
        for (uint32_t k0 = (threadIdx.x - lane) * kPushUnroll; k0 < cnt;
             k0 += blockDim.x * kPushUnroll) {  // uniform per wave
            uint32_t v[kPushUnroll];
#pragma unroll
            for (uint32_t j = 0; j < kPushUnroll; ++j) {
                const uint32_t k = k0 + j * kWave + lane;
                v[j] = k < cnt ? a.col[E.lo + k] : 0xFFFFFFFFu;
            }
            if constexpr (kExact) bfs_claim_exact(a, x, v, next, hacc);
            else bfs_claim_plain(a, x.visited, v, next);
        }
    }
}

constexpr uint32_t kPullLane = 32;  // in-degree up to which one lane scans a vertex alone
constexpr uint32_t kPullGroup = 4;  // in-edges a lane probes per round

// Segment of the next queue for the joins of a round of kBfsRound vertices from `blk`: the rounds are
// dealt over the segments, so none gets more than its span, and with a multiple of kBfsSlots
// workgroups all rounds of one have the same segment.
__device__ __forceinline__ uint32_t bfs_round_segment(uint64_t blk) { return (uint32_t)(blk / kBfsRound) % kBfsSlots; }

// A wave's round (join masks of its kRoundChunks chunks from vertex v0) held, and the held ones
// appended when the list is full or the next round has another segment.
__device__ __forceinline__ void bfs_join_round(const BfsArgs& a, BfsJoins& J, const BfsSink& o,
                                               const unsigned long long (&jm)[kRoundChunks], uint64_t v0, uint64_t blk,
                                               unsigned long long& hacc) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    static_assert(kJoinRound >= kWave * kRoundChunks, "a round's joins");
#pragma unroll
    for (uint32_t k = 0; k < kRoundChunks; ++k) J.put((jm[k] >> lane) & 1ull, (uint32_t)(v0 + k * kWave) + lane);
    if (gridDim.x % kBfsSlots || J.n > kJoinCap - kJoinRound) bfs_flush_wave(a, J, o, bfs_round_segment(blk), hacc);
}

constexpr uint32_t kPullWords = kJoinCap / kWave;          // visited words a wave takes at a time
constexpr uint32_t kPullRounds = kPullWords / kRoundChunks;  // in rounds

// Bottom-up probe of one vertex per lane and j (in-edges [b, e), none if b == e): joined[j] where a source
// is visited.  A lane scans a vertex of in-degree <= kPullLane alone, kPullGroup in-edges
// of every j per round; above that the whole wave scans it 64 in-edges at a time and stops at the
// first hit (ballot), so one high in-degree vertex does not hold its wave for hundreds of sequential
// probes.  `probes` counts in-edges examined up to and including the first hit in either case.
__device__ __forceinline__ void pull_probe(const BfsArgs& a, const unsigned long long* __restrict__ cur,
                                           const uint32_t (&b)[kRoundChunks], const uint32_t (&e)[kRoundChunks],
                                           bool (&joined)[kRoundChunks], unsigned long long& probes) {
    typedef uint32_t Sources __attribute__((ext_vector_type(kPullGroup), aligned(4)));
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t sb[kRoundChunks], se[kRoundChunks];
    bool more = false;
#pragma unroll
    for (uint32_t k = 0; k < kRoundChunks; ++k) {
        joined[k] = false;
        sb[k] = b[k];
        se[k] = e[k] - b[k] > kPullLane ? b[k] : e[k];
        more |= sb[k] < se[k];
    }
    while (__ballot(more)) {  // uniform across the wave
        // a group is one load where the array goes on that far (4-byte aligned; entries past se unused)
        Sources u[kRoundChunks];
#pragma unroll
        for (uint32_t k = 0; k < kRoundChunks; ++k) {
            u[k] = Sources{0, 0, 0, 0};
            if (sb[k] < se[k]) {
                if ((unsigned long long)sb[k] + kPullGroup <= a.m) {
                    u[k] = *reinterpret_cast<const Sources*>(a.csrc + sb[k]);
                } else {
#pragma unroll
                    for (uint32_t j = 0; j < kPullGroup; ++j)
                        if (lies_before(sb[k], j, se[k])) u[k][j] = a.csrc[sb[k] + j];
                }
            }
        }
        unsigned long long word[kRoundChunks][kPullGroup];
#pragma unroll
        for (uint32_t k = 0; k < kRoundChunks; ++k)
#pragma unroll
            for (uint32_t j = 0; j < kPullGroup; ++j)
                word[k][j] = lies_before(sb[k], j, se[k]) ? cur[u[k][j] >> 6] : 0ull;
        more = false;
#pragma unroll
        for (uint32_t k = 0; k < kRoundChunks; ++k) {
            uint32_t hit = kPullGroup;
#pragma unroll
            for (uint32_t j = kPullGroup; j-- > 0;)
                if ((word[k][j] >> (u[k][j] & 63)) & 1ull) hit = j;
            const uint32_t left = min(se[k] - sb[k], kPullGroup);
            if (hit < kPullGroup) {
                probes += hit + 1;
                joined[k] = true;
                sb[k] = se[k];
            } else {
                probes += left;
                sb[k] += left;
            }
            more |= sb[k] < se[k];
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kRoundChunks; ++k) {
        for (unsigned long long bm = __ballot(e[k] - b[k] > kPullLane); bm; bm &= bm - 1) {
            const uint32_t owner = __builtin_ctzll(bm);
            // in scalar registers, and so the loop: it is the longest chain of a superstep (RMAT-20, pulled
            // from one source: 997 us with the bounds by a lane shuffle, 827 now)
            const uint32_t vb = __builtin_amdgcn_readlane(b[k], owner), ve = __builtin_amdgcn_readlane(e[k], owner);
            unsigned long long hm = 0;
            uint32_t k0 = vb, seen = 0;
            for (; k0 < ve && !hm; k0 = advance_to(k0, kWave, ve)) {
                bool hit = false;
                if (lies_before(k0, lane, ve)) {
                    const uint32_t u = a.csrc[k0 + lane];
                    hit = (cur[u >> 6] >> (u & 63)) & 1ull;
                }
                hm = __ballot(hit);
                seen += hm ? (uint32_t)__builtin_ctzll(hm) + 1 : min(ve - k0, (uint32_t)kWave);
            }
            if (lane == owner) {
                probes += seen;
                joined[k] = hm != 0;
            }
        }
    }
}

// Pull superstep: workgroup rounds of kBfsRound consecutive vertices, of which each wave owns
// kRoundChunks visited words.  A wave lists the unvisited vertices of kPullRounds rounds, which then
// fill its lanes however few of each word they are, and probes kRoundChunks of them per lane at a time;
// the joins replace them at the front of the list and go to the next queue together, and every owned
// word of the next visited bitmap is written whole, so the pull needs no compaction.  Bound by
// the chain of dependent loads (visited word, in-offsets, sources, bitmap words), which a pass over
// the list goes through once.  Chung-Lu, 2.4 M vertices, pulls of 1.3 M to 0.5 M unvisited vertices:
// 34..26 us with a lane per vertex of the round, 25..20 now.
__device__ __forceinline__ void pull_all(const BfsArgs& a, const unsigned long long* __restrict__ cur,
                                         unsigned long long* __restrict__ nxt, const BfsSink& o, int32_t next,
                                         unsigned long long& hacc, unsigned long long& probes, BfsJoins J,
                                         unsigned long long* words) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave, grid = gridDim.x;
    // all rounds of a pass over the list have the same segment
    const uint32_t rounds = grid % kBfsSlots ? 1u : kPullRounds;
    for (uint64_t round0 = blockIdx.x; round0 * kBfsRound < a.n; round0 += (uint64_t)rounds * grid) {
        // lane l owns word l % kRoundChunks of the wave's part of round l / kRoundChunks
        const uint64_t w = (round0 + (uint64_t)(lane / kRoundChunks) * grid) * (kBfsRound / kWave) + wv * kRoundChunks +
                           lane % kRoundChunks;
        const bool owner = lane < rounds * kRoundChunks && w < a.nwords;
        const unsigned long long vis = owner ? cur[w] : 0ull;
        unsigned long long open = owner ? ~vis : 0ull;
        if (owner && (w + 1) * kWave > a.n) open &= (1ull << (a.n % kWave)) - 1;
        uint32_t cand = 0;
        const uint32_t owned = (uint32_t)__popcll(__ballot(owner));  // lanes 0, 1, .. (a round may end short)
        for (uint32_t i = 0; i < owned; ++i) {
            const unsigned long long m = bfs_pack(__builtin_amdgcn_readlane((uint32_t)open, i),
                                                  __builtin_amdgcn_readlane((uint32_t)(open >> 32), i));
            const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((uint32_t)w, i) * kWave + lane;
            if ((m >> lane) & 1ull) J.list[cand + lanes_below(m)] = v;
            cand += (uint32_t)__popcll(m);
        }
        if (lane < kPullWords) words[lane] = 0;
        wave_lds_fence();
        for (uint32_t i0 = 0; i0 < cand; i0 += kWave * kRoundChunks) {
            uint32_t v[kRoundChunks], b[kRoundChunks], e[kRoundChunks];
            bool joined[kRoundChunks];
#pragma unroll
            for (uint32_t k = 0; k < kRoundChunks; ++k) {
                const uint32_t i = i0 + k * kWave + lane;
                v[k] = i < cand ? J.list[i] : 0u;
                b[k] = e[k] = 0;
                if (i < cand) {
                    b[k] = a.cptr[v[k]];
                    e[k] = a.cptr[v[k] + 1];
                }
            }
            wave_lds_fence();
            pull_probe(a, cur, b, e, joined, probes);
#pragma unroll
            for (uint32_t k = 0; k < kRoundChunks; ++k) {
                if (joined[k]) {
                    a.level[v[k]] = next;
                    const uint32_t d = v[k] / kBfsRound - (uint32_t)round0;  // 0, grid, 2 grid or 3 grid
                    const uint32_t r = (d >= grid) + (d >= 2 * grid) + (d >= 3 * grid);
                    atomicOr(&words[r * kRoundChunks + v[k] / kWave % kRoundChunks], 1ull << (v[k] % kWave));
                }
                J.put(joined[k], v[k]);  // behind the entries read so far
            }
        }
        wave_lds_fence();
        if (owner) nxt[w] = vis | words[lane];
        bfs_flush(a, J, o, bfs_round_segment(round0 * kBfsRound), hacc);
    }
}

// Sums of the next frontier's segment counters and of the work slots (each wave reduces them
// itself, so every thread gets them without a barrier).
__device__ __forceinline__ void bfs_sum_counters(BfsCounters* __restrict__ ctr, uint32_t par_next,
                                                 unsigned long long& joined, unsigned long long& work) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const unsigned long long j = lane < kBfsSlots ? load_now(&ctr->seg[par_next][lane].v) : 0ull;
    const unsigned long long w = lane < kBfsSlots ? load_now(&ctr->work[lane].v) : 0ull;
    joined = wave_sum_u64(j);
    work = wave_sum_u64(w);
}

// Counters cleared for the next superstep (by one workgroup, after every thread has read
// them): the segment counters of parity `par_free` (a frontier already expanded), the work
// slots, the tickets and the hub count.
__device__ __forceinline__ void bfs_clear_counters(BfsCounters* __restrict__ ctr, uint32_t par_free) {
    if (threadIdx.x < kBfsSlots) {
        ctr->seg[par_free][threadIdx.x].v = 0;
        ctr->work[threadIdx.x].v = 0;
        ctr->sub[threadIdx.x].v = 0;
    }
    if (threadIdx.x == 0) {
        ctr->top = 0;
        ctr->n_hub = 0;
    }
}

// LDS frontier capacity of a superstep slot's workgroup 0, and of the starting kernel's workgroup:
// one round of kPushUnroll out-edges per thread.
constexpr uint32_t kSoloSlot = 256 * kPushUnroll;
constexpr uint32_t kSoloStart = 1024 * kPushUnroll;

// Counts of a finished superstep.
struct BfsCounts {
    uint32_t n_new, n_hub;
    unsigned long long deg_sum, deg_large, probes;
    uint32_t slots;  // launches it took
};

// The counts of the superstep just finished folded into the control block; true if another follows.
__device__ __forceinline__ bool bfs_fold(const BfsArgs& a, BfsCtl& c, const BfsCounts& k) {
    const uint32_t n = a.n, n_new = k.n_new;
    // bytes of the superstep just finished: push = queue entry and out-offsets per frontier vertex
    // (12) + target id and visited bit per out-edge (8); exact claims then add the bit OR (8), level
    // (4), out-offsets (8) and queue entry (4) per join, plain claims the store per join (4) and the
    // compaction's level pass (4n), visited bitmap (8 per word), out-offsets and queue entry per
    // join (12); pull = visited word per 64 vertices, read and written (16), and in-offsets of
    // unvisited vertices (8) + source id and bitmap word per probed in-edge (8) + level, out-offsets
    // and queue entry per join (16)
    const unsigned long long kb =
        c.pull    ? 8ull * c.n_u + 8ull * k.probes + 16ull * a.nwords + 16ull * n_new
        : c.small ? 12ull * c.n_f + 8ull * c.m_f + 24ull * n_new
                  : 12ull * c.n_f + 8ull * c.m_f + 4ull * n + 8ull * a.nwords + 16ull * n_new;
    c.kernel_bytes += kb;
    c.alg_bytes += kb;
    c.slots += k.slots;
    if (n_new == 0) {
        c.done = 1;
        return false;
    }
    c.step += 1;
    c.n_f = n_new;
    c.m_f = k.deg_sum;
    c.n_u -= n_new;
    c.m_u -= k.deg_sum;
    c.reached += n_new;
    c.reached_edges += k.deg_sum;
    c.n_small = n_new - k.n_hub;
    c.n_large = k.n_hub;
    c.hub_wgs = bfs_hub_wgs(a.grid, c.n_small, k.n_hub, k.deg_large, k.deg_sum);
    return true;
}

// The heuristic's direction of the next superstep (Beamer, Asanovic, Patterson, SC'12) after one in
// direction `pull`.
__device__ __forceinline__ bool bfs_heuristic(const BfsCtl& c, bool pull) {
    return !pull ? (double)c.m_f > (double)c.m_u / Sched::kAlphaBfs : !((double)c.n_f < (double)c.n / Sched::kBeta);
}
// Whether the learned policy is asked for it.
__device__ __forceinline__ bool bfs_asks(const BfsArgs& a, const BfsCtl& c, bool pull) {
    return c.mode == 3 && a.policy &&
           bfs_policy_consulted(pull, (double)c.n_f, (double)c.m_f, (double)c.m_u, (double)c.n, Sched::kAlphaBfs,
                                Sched::kBeta);
}
__device__ __forceinline__ void bfs_record(const BfsCtl& c, double (&rec)[MEDUSA_TRACE_FIELDS]) {
    rec[0] = (double)c.step;
    rec[1] = (double)c.n_f;
    rec[2] = (double)c.m_f;
    rec[3] = (double)c.n_u;
    rec[4] = (double)c.m_u;
    rec[5] = (double)c.n;
    rec[6] = (double)c.m;
    rec[7] = rec[8] = 0.0;
}
__device__ __forceinline__ void bfs_set_direction(const BfsArgs& a, BfsCtl& c, bool pull, bool solo) {
    c.pull = pull ? 1u : 0u;
    c.small = solo ? 3u : bfs_small(pull, c.n_f, c.m_f, a.exact_edges);
    c.supersteps += 1;
    if (pull)
        c.pull_steps += 1;
    else
        c.push_steps += 1;
}

// The decision after a superstep of the whole grid (the deciding workgroup, after every workgroup
// of the superstep has added its counters; its first wave does the work): counters folded in and
// cleared for the next superstep, direction by the heuristic or the learned policy, hub queue split
// and the termination vote, written into the control block.  The updated control block waits in
// LDS while the policy is evaluated, so it holds no registers there.
__device__ __forceinline__ void bfs_decide(const BfsArgs& a, uint32_t slot, BfsCtl* s_c, float* s_params) {
    if (threadIdx.x >= kWave) return;
    // with a policy, its parameters start for LDS now, behind the counter loads, holding no
    // registers; a decision that does not consult it only waits for them at the end
    if (a.policy) mlp_stage_wave_begin(a.policy, s_params);
    BfsCounters* ctr = a.ctr;
    const uint32_t lane = threadIdx.x;
    uint32_t par;
    bool pull = false, ask = false, plain = false, solo = false, more;
    double rec[MEDUSA_TRACE_FIELDS] = {};
    {
        BfsCtl c = load_now_block(a.ctl + slot);
        par = (uint32_t)c.step & 1u;
        unsigned long long joined, work;
        bfs_sum_counters(ctr, par ^ 1u, joined, work);
        const uint32_t n_hub = load_now(&ctr->n_hub);
        const BfsCounts k{(uint32_t)joined, n_hub, joined >> 32, (uint32_t)work, work >> 32,
                          c.pending ? 2u : 1u};
        c.vsel ^= c.pull;  // a pull wrote the other bitmap
        c.pending = 0;
        more = bfs_fold(a, c, k);
        if (more) {
            solo = c.mode != 2 && bfs_solo_fits(kSoloSlot, c.n, c.n_f, c.m_f);
            if (c.mode == 2) {
                pull = true;
            } else if (c.mode != 1 && !solo) {
                ask = bfs_asks(a, c, c.pull != 0);
                pull = bfs_heuristic(c, c.pull != 0);
                // between the margins the heuristic's choice stands, and with a policy a pull goes on
                plain = pull || c.pull != 0;
                if (ask) bfs_record(c, rec);
            }
        }
        if (lane == 0) *s_c = c;
        wave_lds_fence();
    }
    if (ask) {  // uniform across the wave
        float c_push, c_pull;
        policy_direction_costs_wave(rec, a.policy, s_params, c_push, c_pull, true);
        pull = policy_pull(c_push, c_pull, plain);
    } else if (a.policy) {
        mlp_stage_wave_wait();
    }
    bfs_clear_counters(ctr, par);  // this wave read them above
    if (lane == 0) {
        BfsCtl c = *s_c;
        if (more) bfs_set_direction(a, c, pull, solo);
        a.ctl[slot ^ 1u] = c;
    }
}

// ---- solo supersteps ------------------------------------------------------------------
// One workgroup, the others idle or not launched: a thin frontier's superstep costs two dependent
// global round trips and a few barriers (2 us, and 4 to 5 for each full round of 4096 scattered
// out-edges, which one CU issues line by line) instead of a launch, 1024 workgroups' tickets and the
// counters' round trips (8..11 us).  The supersteps of Erdos-Renyi with 65536 vertices: 105 us a run
// before, 84 now; RMAT-20 183 and 164; the 2.4 M-vertex Chung-Lu graph, whose tail of thin
// supersteps took a launch each, 500 and 481.

template <uint32_t kThreads>
struct BfsSoloLds {
    static constexpr uint32_t kCap = kThreads * kPushUnroll;
    uint32_t off[kCap], beg[kCap];            // the frontier's out-edge prefix and offsets
    uint32_t v[kCap], vbeg[kCap], deg[kCap];  // the next frontier as it is claimed
    unsigned long long vis[kCap / 64];        // the visited bitmap of a graph of at most kCap vertices
    uint32_t wsum[kThreads / kWave];
    uint32_t n, n_hub;
    unsigned long long deg_sum, deg_large;
};

template <uint32_t kThreads>
__device__ __forceinline__ void solo_reset(BfsSoloLds<kThreads>& L) {
    if (threadIdx.x == 0) {
        L.n = L.n_hub = 0;
        L.deg_sum = L.deg_large = 0;
    }
}

// Claims up to kPushUnroll vertices v[j] (0xFFFFFFFF: none) per thread for `level` and appends the
// ones this thread won to the next frontier.  No other workgroup touches the bitmap in this launch,
// so workgroup scope is enough; the targets' row offsets load beside the claims.  kLdsVis: the
// bitmap is L.vis (a small graph's few lines of global memory would take one atomic at a time:
// 33 K out-edges of 4096 vertices 80 us instead of 49).
template <bool kLdsVis, uint32_t kThreads, uint32_t kN>
__device__ __forceinline__ void solo_claim(const BfsArgs& a, unsigned long long* visited, BfsSoloLds<kThreads>& L,
                                           const uint32_t (&v)[kN], int32_t level) {
    unsigned long long old[kN];
    uint32_t b[kN], e[kN];
#pragma unroll
    for (uint32_t j = 0; j < kN; ++j) {
        b[j] = e[j] = 0;
        old[j] = ~0ull;
        if (v[j] != 0xFFFFFFFFu) {
            b[j] = a.row_ptr[v[j]];
            e[j] = a.row_ptr[v[j] + 1];
            old[j] = __hip_atomic_fetch_or(kLdsVis ? &L.vis[v[j] >> 6] : &visited[v[j] >> 6], 1ull << (v[j] & 63),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    // one LDS atomic per wave and counter: hundreds of lanes on one LDS address would serialise
    unsigned long long wm[kN];
    uint32_t cnt = 0, dsum = 0, hubs = 0, hsum = 0;  // out-degrees of distinct vertices: below 2^32 in all
#pragma unroll
    for (uint32_t j = 0; j < kN; ++j) {
        const bool won = !((old[j] >> (v[j] & 63)) & 1ull);
        wm[j] = __ballot(won);
        cnt += (uint32_t)__popcll(wm[j]);
        if (won) {
            const uint32_t d = e[j] - b[j];
            dsum += d;
            hubs += d > a.large;
            hsum += d > a.large ? d : 0u;
        }
    }
    if (!cnt) return;  // uniform across the wave
    dsum = __builtin_amdgcn_readlane(wave_incl_scan(dsum), kWave - 1);
    uint32_t i = 0;
    if (lane_id() == 0) {
        i = atomicAdd(&L.n, cnt);
        atomicAdd(&L.deg_sum, (unsigned long long)dsum);
    }
    i = __builtin_amdgcn_readfirstlane(i);
    if (hubs) {
        atomicAdd(&L.n_hub, hubs);
        atomicAdd(&L.deg_large, (unsigned long long)hsum);
    }
#pragma unroll
    for (uint32_t j = 0; j < kN; ++j) {
        if ((wm[j] >> lane_id()) & 1ull) {
            const uint32_t at = i + lanes_below(wm[j]);
            a.level[v[j]] = level;
            L.v[at] = v[j];
            L.vbeg[at] = b[j];
            L.deg[at] = e[j] - b[j];
        }
        i += (uint32_t)__popcll(wm[j]);
    }
}

// Supersteps of the frontier in L (v, vbeg, deg; L.n vertices, complete behind a barrier) and of the
// ones after it while they fit; c (the same in every thread) follows.  Ends with c.done, or with the
// first frontier that does not fit in L and no direction chosen for it.  Every thread calls it.
template <bool kLdsVis, uint32_t kThreads>
__device__ __forceinline__ void bfs_solo(const BfsArgs& a, unsigned long long* visited, BfsSoloLds<kThreads>& L,
                                         BfsCtl& c) {
    constexpr uint32_t kCap = BfsSoloLds<kThreads>::kCap, kPer = kPushUnroll;
    const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wv = t / kWave;
    for (;;) {
        // the frontier's offsets, kPer consecutive entries per thread
        const uint32_t n = L.n;
        uint32_t d[kPer], sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) {
            const uint32_t i = t * kPer + j;
            d[j] = i < n ? L.deg[i] : 0u;
            sum += d[j];
            if (i < n) L.beg[i] = L.vbeg[i];
        }
        const uint32_t incl = wave_incl_scan(sum);
        if (lane == kWave - 1) L.wsum[wv] = incl;
        __syncthreads();
        uint32_t at = incl - sum, total = 0;
#pragma unroll
        for (uint32_t w = 0; w < kThreads / kWave; ++w) {
            if (w < wv) at += L.wsum[w];
            total += L.wsum[w];
        }
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) {
            L.off[t * kPer + j] = at;  // past n: total
            at += d[j];
        }
        solo_reset(L);
        __syncthreads();
        for (uint32_t e0 = 0; e0 < total; e0 += kCap) {  // uniform
            // kPushUnroll consecutive out-edges per thread: one search for the first one's owner, the
            // last entry whose offset is at most e (it has out-edges), then steps to the next
            uint32_t v[kPushUnroll], x[kPushUnroll];
            const uint32_t first = e0 + t * kPushUnroll;
            uint32_t lo = 0;
            if (first < total) {
#pragma unroll
                for (uint32_t step = kCap / 2; step; step >>= 1)
                    if (L.off[lo + step] <= first) lo += step;
            }
#pragma unroll
            for (uint32_t j = 0; j < kPushUnroll; ++j) {
                x[j] = 0;
                if (first + j < total) {
                    while (lo + 1 < n && L.off[lo + 1] <= first + j) ++lo;
                    x[j] = L.beg[lo] + (first + j - L.off[lo]);
                }
            }
#pragma unroll
            for (uint32_t j = 0; j < kPushUnroll; ++j) v[j] = first + j < total ? a.col[x[j]] : 0xFFFFFFFFu;
            solo_claim<kLdsVis>(a, visited, L, v, c.step + 1);
        }
        __syncthreads();
        if (!bfs_fold(a, c, BfsCounts{L.n, L.n_hub, L.deg_sum, L.deg_large, 0, 0})) return;
        if (!bfs_solo_fits(kCap, c.n, c.n_f, c.m_f)) return;
        bfs_set_direction(a, c, false, true);
    }
}

// The frontier in L handed to the next launch, in queue step % 2 (segment 0,
// which may run on over the others' space), its hub queue and its counters; the control block goes
// to *ctl.  (Counters other than the queues' are zero: nobody adds to them in this launch.)
template <uint32_t kThreads>
__device__ __forceinline__ void solo_publish(const BfsArgs& a, BfsSoloLds<kThreads>& L, const BfsCtl& c,
                                             BfsCtl* ctl) {
    const uint32_t t = threadIdx.x, par = (uint32_t)c.step & 1u;
    if (!c.done) {
        const uint32_t n = L.n;
        if (t < kBfsSlots) {
            a.ctr->seg[par][t].v = t == 0 ? bfs_pack(n, (uint32_t)L.deg_sum) : 0ull;
            a.ctr->seg[par ^ 1u][t].v = 0;
        }
        __syncthreads();
        if (t == 0) L.n_hub = 0;
        __syncthreads();
        for (uint32_t i = t; i < n; i += kThreads) {
            const uint32_t v = L.v[i];
            a.q[par][i] = v;
            if (L.deg[i] > a.large) a.hub[par][atomicAdd(&L.n_hub, 1u)] = v;
        }
    }
    if (t == 0) *ctl = c;
}

// ---- kernels (both drivers) ---------------------------------------------------------

// The control block of superstep 0 from the first frontier's counts, no direction chosen yet.
__device__ __forceinline__ BfsCtl bfs_first(const BfsArgs& a, const BfsCounts& k, unsigned long long m, uint32_t mode,
                                            int32_t* out) {
    BfsCtl c{};
    c.mode = mode;
    c.n = a.n;
    c.m = m;
    c.n_f = k.n_new;
    c.m_f = k.deg_sum;
    c.n_u = a.n - c.n_f;
    c.m_u = m - c.m_f;
    c.reached = c.n_f;
    c.reached_edges = c.m_f;
    c.n_small = k.n_new - k.n_hub;
    c.n_large = k.n_hub;
    c.hub_wgs = bfs_hub_wgs(a.grid, c.n_small, c.n_large, k.deg_large, c.m_f);
    c.out = out;
    c.t_begin = a.ctl->t_begin;
    return c;
}
// Direction of a superstep after a push (or the first), by one wave.
__device__ __forceinline__ bool bfs_next_pull(const BfsArgs& a, const BfsCtl& c, float* s_params) {
    if (c.mode == 1) return false;
    if (c.mode == 2) return true;
    const bool plain = bfs_heuristic(c, false);
    if (!bfs_asks(a, c, false)) return plain;
    double rec[MEDUSA_TRACE_FIELDS];
    bfs_record(c, rec);
    float c_push, c_pull;
    policy_direction_costs_wave(rec, a.policy, s_params, c_push, c_pull);
    return policy_pull(c_push, c_pull, plain);
}

// First decision after k_bfs_mark placed the sources; one workgroup.  The work slots, tickets and
// hub count are cleared (queue 0's counters stay: superstep 0 reads them).
__global__ __launch_bounds__(kWave) void k_bfs_first_decide(BfsArgs a, unsigned long long m, uint32_t mode,
                                                            int32_t* out) {
    __shared__ float s_params[kMlpWaveLds];
    BfsCounters* ctr = a.ctr;
    unsigned long long joined, work;
    bfs_sum_counters(ctr, 0, joined, work);
    const uint32_t n_hub = load_now(&ctr->n_hub);
    BfsCtl c = bfs_first(a, BfsCounts{(uint32_t)joined, n_hub, joined >> 32, (uint32_t)work, 0, 0}, m, mode, out);
    bfs_set_direction(a, c, bfs_next_pull(a, c, s_params), false);
    if (threadIdx.x < kBfsSlots) {
        ctr->work[threadIdx.x].v = 0;
        ctr->sub[threadIdx.x].v = 0;
    }
    if (threadIdx.x == 0) {
        ctr->top = 0;
        ctr->n_hub = 0;
        *a.ctl = c;
    }
}

// Start of a device-driven run, one workgroup, after the reset: the sources (any duplicates counted
// once) at level 0 and the supersteps from there on that one workgroup runs fastest; then the
// first decision for the whole grid, and the frontier is handed to the superstep slots.
__global__ __launch_bounds__(1024) void k_bfs_start(BfsArgs a, const BfsHost* __restrict__ host, unsigned long long m) {
    __shared__ BfsSoloLds<1024> L;
    __shared__ float s_params[kMlpWaveLds];
    __shared__ uint32_t s_pull;
    static_assert(kBfsHostSources <= BfsSoloLds<1024>::kCap, "the sources fit the LDS frontier");
    const uint32_t t = threadIdx.x;
    auto param = [](const auto* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
    // one trip over the bus: the first sources with the parameters that say how many there are
    uint32_t src = param(&host->src[t]);
    const uint32_t count = param(&host->count), mode = param(&host->mode);
    int32_t* out = param(&host->out);
    solo_reset(L);
    __syncthreads();
    for (uint32_t i0 = 0; i0 < count; i0 += 1024) {
        if (i0) src = i0 + t < count ? param(&host->src[i0 + t]) : 0u;
        const uint32_t v[1] = {i0 + t < count ? src : 0xFFFFFFFFu};
        solo_claim<false>(a, a.vis[0], L, v, 0);
    }
    __syncthreads();
    BfsCtl c = bfs_first(a, BfsCounts{L.n, L.n_hub, L.deg_sum, L.deg_large, 0, 0}, m, mode, out);
    if (c.mode != 2 && bfs_solo_fits(kSoloStart, c.n, c.n_f, c.m_f)) {
        bfs_set_direction(a, c, false, true);
        if (a.n <= BfsSoloLds<1024>::kCap) {
            if (t < a.nwords) L.vis[t] = a.vis[0][t];  // behind the barrier above
            bfs_solo<true>(a, a.vis[0], L, c);
            if (t < a.nwords) a.vis[0][t] = L.vis[t];
        } else {
            bfs_solo<false>(a, a.vis[0], L, c);
        }
    }
    if (!c.done) {
        if (t < kWave) {
            const bool pull = bfs_next_pull(a, c, s_params);
            if (t == 0) s_pull = pull ? 1u : 0u;
        }
        __syncthreads();
        bfs_set_direction(a, c, s_pull != 0, false);
    }
    solo_publish(a, L, c, a.ctl);
}

// End of a batch of slots: the control block to the host, and the levels to their destination when
// the run is done.
// `odd`: the batch had an odd number of slots, so it left the control block in the second place;
// the next batch starts from the first.
__global__ __launch_bounds__(256) void k_bfs_close(BfsArgs a, BfsHost* __restrict__ host, uint32_t odd) {
    const BfsCtl* ctl = a.ctl + odd;
    if (blockIdx.x == 0) {
        if (odd && threadIdx.x < sizeof(BfsCtl) / 4)
            reinterpret_cast<uint32_t*>(a.ctl)[threadIdx.x] = reinterpret_cast<const uint32_t*>(ctl)[threadIdx.x];
        if (threadIdx.x == 0) host->t_end = (unsigned long long)wall_clock64();
        if (threadIdx.x < sizeof(BfsCtl) / 8)
            reinterpret_cast<unsigned long long*>(&host->ctl)[threadIdx.x] =
                reinterpret_cast<const unsigned long long*>(ctl)[threadIdx.x];
    }
    int32_t* out = ctl->out;
    if (!ctl->done || !out) return;
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = tid;
    if (reinterpret_cast<uintptr_t>(out) % 16 == 0) {
        const uint64_t n4 = a.n / 4;
        for (uint64_t q = tid; q < n4; q += stride)
            reinterpret_cast<int4*>(out)[q] = reinterpret_cast<const int4*>(a.level)[q];
        i = 4 * n4 + tid;
    }
    for (; i < a.n; i += stride) out[i] = a.level[i];
}

// Level reset, counters and the visited bitmap cleared; with `single` < n that
// vertex is placed at level 0, in the bitmap and in queue 0 with its counters (the host-driven loop;
// otherwise k_bfs_start or k_bfs_mark places the sources).
__global__ __launch_bounds__(256) void k_bfs_seed(BfsArgs a, uint32_t single) {
    const uint32_t n = a.n;
    const bool one = single < n;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.ctl->t_begin = (unsigned long long)wall_clock64();
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
        a.level[v] = v == single ? 0 : -1;
    for (uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; w < a.nwords; w += stride)
        a.vis[0][w] = one && w == single / kWave ? 1ull << (single & 63) : 0ull;
    if (blockIdx.x != 0) return;
    bfs_clear_counters(a.ctr, 0);
    bfs_clear_counters(a.ctr, 1);
    __syncthreads();
    if (threadIdx.x == 0 && one) {
        const uint32_t deg = a.row_ptr[single + 1] - a.row_ptr[single], sg = single / a.span;
        a.ctr->seg[0][sg].v = bfs_pack(1u, deg);
        a.q[0][(size_t)sg * a.span] = single;
        if (deg > a.large) {
            a.hub[0][0] = single;
            a.ctr->work[0].v = deg;
            a.ctr->n_hub = 1u;
        }
    }
}

// Several sources: each is placed at level 0, in the bitmap and in queue 0; a vertex given more
// than once is counted once (the lane that sets its bit).  One queue atomic per source.
__global__ __launch_bounds__(256) void k_bfs_mark(BfsArgs a, const uint32_t* __restrict__ src, uint32_t count) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    unsigned long long hacc = 0;
    for (uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x - lane); i0 < count;
         i0 += (uint64_t)gridDim.x * blockDim.x) {  // uniform per wave
        const uint64_t i = i0 + lane;
        bool won = false;
        uint32_t v = 0, deg = 0;
        if (i < count) {
            v = src[i];
            const unsigned long long bit = 1ull << (v & 63);
            won = !(atomicOr(&a.vis[0][v >> 6], bit) & bit);
        }
        if (won) {
            a.level[v] = 0;
            deg = a.row_ptr[v + 1] - a.row_ptr[v];
            const uint32_t sg = v / a.span;
            const uint32_t off = (uint32_t)atomicAdd(&a.ctr->seg[0][sg].v, bfs_pack(1u, deg));
            a.q[0][(size_t)sg * a.span + off] = v;
        }
        const bool hub = won && deg > a.large;
        const unsigned long long hm = __ballot(hub);
        if (hm) {
            uint32_t hb = 0;
            if (lane == 0) hb = atomicAdd(&a.ctr->n_hub, (uint32_t)__popcll(hm));
            hb = __shfl(hb, 0, kWave);
            if (hub) {
                a.hub[0][hb + lanes_below(hm)] = v;
                hacc += deg;
            }
        }
    }
    bfs_finish<false>(a.ctr, hacc);
}

// Host-driven superstep t: counters cleared except the frontier's queue segments (parity t % 2).
__global__ __launch_bounds__(64) void k_zero_counters(BfsCounters* c, uint32_t par_free) {
    bfs_clear_counters(c, par_free);
}

// After a push with plain claims: the next frontier = {v : level[v] == step + 1}, as its
// queue, hub queue and counters, and the visited bitmap (one ballot per 64 vertices) rebuilt from the
// levels, in workgroup rounds of kBfsRound consecutive vertices (wave w the chunks w * kRoundChunks + k),
// whose level loads are issued together.
__device__ __forceinline__ void compact_level(const BfsArgs& a, unsigned long long* visited, int32_t next,
                                              const BfsSink& o, unsigned long long& hacc, BfsJoins J) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    uint64_t blk = (uint64_t)blockIdx.x * kBfsRound;
    for (; blk < a.n; blk += (uint64_t)gridDim.x * kBfsRound) {
        const uint64_t c0 = blk / kWave + wv * kRoundChunks;  // first chunk of this wave
        int32_t lv[kRoundChunks];
#pragma unroll
        for (uint32_t k = 0; k < kRoundChunks; ++k) {
            const uint64_t v = (c0 + k) * kWave + lane;
            lv[k] = v < a.n ? a.level[v] : -1;
        }
        unsigned long long jm[kRoundChunks];
#pragma unroll
        for (uint32_t k = 0; k < kRoundChunks; ++k) {
            jm[k] = __ballot(lv[k] == next);
            const unsigned long long vm = __ballot(lv[k] >= 0);
            if (lane == 0 && c0 + k < a.nwords) visited[c0 + k] = vm;
        }
        bfs_join_round(a, J, o, jm, c0 * kWave, blk, hacc);
    }
    bfs_flush(a, J, o, bfs_round_segment(blk), hacc);
}

// One launch of the superstep loop, doing what the control block says:
//   pending: the compaction after a push with plain claims;
//   pull:    every unvisited vertex; the next frontier's queue, hub queue, visited bitmap and
//            counters come out of the same pass;
//   small:   3: workgroup 0 runs this superstep and the ones after it solo; else push with exact
//            claims (the frontier's out-edges fit one queue segment); the
//            winners are recorded as they are claimed; with at most 64 frontier vertices every
//            wave takes an equal share of their out-edges (hubs included);
//   else:    push with plain claims; it leaves `pending` set, so the next launch compacts.
// The first hub_wgs workgroups of a push take the hub queue, the rest the frontier queue.  With
// kDecide the last workgroup to finish a counting phase decides the next superstep; otherwise the host
// reads the counters.
template <bool kDecide>
__global__ __launch_bounds__(256) void k_bfs_super(BfsArgs a, uint32_t slot) {
    __shared__ uint32_t s_beg[4][kWave], s_off[4][kWave];
    __shared__ uint32_t s_pre[kBfsSlots + 1];
    // the joins of the whole grid's supersteps, or the solo supersteps' frontier
    union Work {
        BfsJoinLds joins;
        BfsSoloLds<256> solo;
    };
    __shared__ alignas(16) unsigned char s_work[kDecide ? sizeof(Work) : sizeof(BfsJoinLds)];
    __shared__ BfsCtl s_c;
    __shared__ float s_params[kDecide ? kMlpWaveLds : 4];
    const BfsCtl* ctl = a.ctl + slot;
    // the control block as it is, with `pending` set or not, for the next launch
    auto pass_on = [&](uint32_t pending) {
        if (!kDecide || blockIdx.x != 0) return;
        if (threadIdx.x < sizeof(BfsCtl) / 4) {
            uint32_t x = reinterpret_cast<const uint32_t*>(ctl)[threadIdx.x];
            if (threadIdx.x == offsetof(BfsCtl, pending) / 4) x = pending;
            reinterpret_cast<uint32_t*>(a.ctl + (slot ^ 1u))[threadIdx.x] = x;
        }
    };
    if (ctl->done) {
        pass_on(0);
        return;
    }
    const int32_t step = ctl->step, next = step + 1;
    const uint32_t par = (uint32_t)step & 1u, vsel = ctl->vsel;
    unsigned long long *visited = vsel ? a.vis[1] : a.vis[0], *other = vsel ? a.vis[0] : a.vis[1];
    const BfsSink sink{a.q[par ^ 1u], a.ctr->seg[par ^ 1u], a.hub[par ^ 1u]};
    const BfsJoins joins{reinterpret_cast<BfsJoinLds*>(s_work)->v[threadIdx.x / kWave]};
    unsigned long long hacc = 0;
    if (ctl->pending) {
        compact_level(a, visited, next, sink, hacc, joins);
        if (bfs_finish<kDecide>(a.ctr, hacc)) bfs_decide(a, slot, &s_c, s_params);
        return;
    }
    if (ctl->pull) {
        unsigned long long probes = 0;
        pull_all(a, visited, other, sink, next, hacc, probes, joins,
                 reinterpret_cast<BfsJoinLds*>(s_work)->words[threadIdx.x / kWave]);
        if (bfs_finish<kDecide>(a.ctr, hacc + (probes << 32))) bfs_decide(a, slot, &s_c, s_params);
        return;
    }
    BfsExact x{visited, sink, blockIdx.x % kBfsSlots, joins};
    const uint32_t hub = ctl->hub_wgs, small = ctl->small;
    if constexpr (kDecide) {
        if (small == 3) {
            if (blockIdx.x != 0) return;
            BfsSoloLds<256>& L = *reinterpret_cast<BfsSoloLds<256>*>(s_work);
            bfs_queue_prefix(a.ctr->seg[par], s_pre);
            const uint32_t qn = s_pre[kBfsSlots];
            for (uint32_t i = threadIdx.x; i < qn; i += 256) {
                const uint32_t u = bfs_queue_at(a, a.q[par], s_pre, i);
                const uint32_t b = a.row_ptr[u];
                L.vbeg[i] = b;
                L.deg[i] = a.row_ptr[u + 1] - b;
            }
            if (threadIdx.x == 0) L.n = qn;
            BfsCtl c = *ctl;
            __syncthreads();
            bfs_solo<false>(a, visited, L, c);
            c.slots += 1;
            c.out = ctl->out;  // again, rather than kept (on the stack) through the supersteps
            c.t_begin = ctl->t_begin;
            if (!c.done) {
                if (threadIdx.x < kWave) {
                    const bool pull = bfs_next_pull(a, c, s_params);
                    if (threadIdx.x == 0) s_pre[0] = pull ? 1u : 0u;
                }
                __syncthreads();
                bfs_set_direction(a, c, s_pre[0] != 0, false);
            }
            solo_publish(a, L, c, a.ctl + (slot ^ 1u));
            return;
        }
    }
    if (!small) pass_on(1);
    if (small == 2) {
        bfs_queue_prefix(a.ctr->seg[par], s_pre);
        push_tiny(a, a.q[par], s_pre, next, s_beg, s_off, x, hacc);
    } else if (blockIdx.x < hub) {
        if (small)
            push_hubs<true>(a, a.hub[par], ctl->n_large, next, blockIdx.x, hub, x, hacc);
        else
            push_hubs<false>(a, a.hub[par], ctl->n_large, next, blockIdx.x, hub, x, hacc);
    } else {
        bfs_queue_prefix(a.ctr->seg[par], s_pre);
        const uint32_t wg = blockIdx.x - hub, nwg = gridDim.x - hub, w0 = wg * 4 + threadIdx.x / kWave;
        if (small)
            push_queue<true>(a, a.q[par], s_pre, next, w0, nwg * 4, s_beg, s_off, x, hacc);
        else
            push_queue<false>(a, a.q[par], s_pre, next, w0, nwg * 4, s_beg, s_off, x, hacc);
    }
    if (small) bfs_flush(a, x.J, x.sink, x.own, hacc);
    if (small && bfs_finish<kDecide>(a.ctr, hacc)) bfs_decide(a, slot, &s_c, s_params);
}

// Degree threshold of the hub queue and workgroups of the expansion: the caller's value,
// else the handle's autotuned one, else the default.
static uint32_t bfs_large(const medusa_graph* g, const medusa_opts& o) {
    return o.large_degree ? o.large_degree : (g->tuned.bfs_large ? g->tuned.bfs_large : kBfsLargeDefault);
}
static uint32_t bfs_grid(const medusa_graph* g, const medusa_opts& o) {
    return o.grid ? o.grid : (g->tuned.bfs_grid ? g->tuned.bfs_grid : kBfsGridDefault);
}

static uint32_t bfs_mode(const medusa_opts& o) {
    if (o.direction == MEDUSA_DIR_PUSH) return 1;
    if (o.direction == MEDUSA_DIR_PULL) return 2;
    if (o.policy && policy_kind(o.policy) == MEDUSA_POLICY_DIRECTION) return 3;
    return 0;
}

// Work buffers of one BFS run: the handle's own (allocated on its first BFS), or, for
// medusa_bfs_noalloc, the caller's level array and the library's static scratch.
struct BfsBufs {
    int32_t* level;
    uint32_t* q[2];                 // frontier queues, kBfsSlots * bfs_span(n) entries each
    uint32_t* hub[2];               // hub queues, n entries each
    unsigned long long* vis[2];     // visited bitmaps, (n + 63) / 64 words each
    const uint32_t* sources;        // several sources (device), or null
    BfsCtl* ctl;
    BfsCounters* ctr;
};
static size_t bfs_queue_cap(uint32_t n) { return (size_t)kBfsSlots * bfs_span(n); }
// Control blocks and counters share one allocation: the control blocks, then the counters.
constexpr size_t kBfsCtlUnits = 2 + (sizeof(BfsCounters) + sizeof(CtlStorage) - 1) / sizeof(CtlStorage);
static BfsBufs handle_bufs(medusa_graph* g) {
    g->bfs_ctl.ensure(kBfsCtlUnits);
    static_assert(sizeof(BfsCtl) <= sizeof(CtlStorage), "control block storage");
    const size_t nwords = ((size_t)g->n + 63) / 64;
    const size_t qcap = bfs_queue_cap(g->n);
    return {g->level.p,
            {g->q_small.p, g->q_small.p + qcap},
            {g->q_large.p, g->q_large.p + g->n},
            {g->bitmap.p, g->bitmap.p + nwords},
            g->q_aux.p,
            reinterpret_cast<BfsCtl*>(g->bfs_ctl.p),
            reinterpret_cast<BfsCounters*>(g->bfs_ctl.p + 2)};
}

// Frontier out-edges up to which a push claims exactly instead of compacting after it.
static unsigned long long bfs_exact_edges(uint32_t n) { return bfs_span(n); }

static BfsArgs bfs_args(medusa_graph* g, const BfsBufs& B, uint32_t large, uint32_t grid, const float* policy) {
    BfsArgs a{};
    a.row_ptr = g->row_ptr.p;
    a.col = g->col.p;
    a.cptr = g->cptr.p;
    a.csrc = g->csrc.p;
    a.level = B.level;
    a.q[0] = B.q[0];
    a.q[1] = B.q[1];
    a.hub[0] = B.hub[0];
    a.hub[1] = B.hub[1];
    a.vis[0] = B.vis[0];
    a.vis[1] = B.vis[1];
    a.ctr = B.ctr;
    a.ctl = B.ctl;
    a.policy = policy;
    a.n = g->n;
    a.nwords = (g->n + 63) / 64;
    a.large = large;
    a.grid = grid;
    a.span = bfs_span(g->n);
    a.m = g->m;
    a.exact_edges = bfs_exact_edges(g->n);
    return a;
}

// Seeding of the host-driven loop, and of a device-driven run of more sources than the starting
// kernel takes: every source at level 0 and in the bitmap (one source by value, several from
// B.sources), the first queue, hub queue and counters.
static void bfs_seed(medusa_graph* g, const BfsBufs& B, const BfsArgs& a, uint32_t nsrc, uint32_t single) {
    hipStream_t s = g->stream;
    hipLaunchKernelGGL(k_bfs_seed, dim3(grid_for(g->n, 256, 4096)), dim3(256), 0, s, a,
                       nsrc == 1 ? single : 0xFFFFFFFFu);
    MDS_LAUNCHED();
    if (nsrc > 1) {
        hipLaunchKernelGGL(k_bfs_mark, dim3(grid_for(nsrc, 256, 1024)), dim3(256), 0, s, a, B.sources, nsrc);
        MDS_LAUNCHED();
    }
}

// One device-driven slot: one launch of the superstep kernel (a push with plain claims takes two
// slots, its expansion and its compaction; every other superstep one).
static void bfs_enqueue_slot(medusa_graph* g, const BfsArgs& a, uint32_t parity) {
    hipLaunchKernelGGL(k_bfs_super<true>, dim3(a.grid), dim3(256), 0, g->stream, a, parity);
}

// Bytes of the seeding: the level reset (4 per vertex), the visited bitmap (8 per word) and the sources
// (16 each: id, level, bit OR).
static uint64_t bfs_seed_bytes(uint32_t n, uint32_t nwords, uint32_t nsrc) {
    return 4ull * n + 8ull * nwords + 16ull * nsrc;
}

// Device-driven run: reset, start, superstep slots and close, then batches of slots and a close until
// the control block says done.  capture: each sequence is captured once as a hipGraph and replayed
// (but for a handle's first, see below); without it (medusa_bfs_noalloc, which may not allocate) the
// same kernels are launched one by one.
static void bfs_run_device(medusa_graph* g, const BfsBufs& B, uint32_t nsrc, const uint32_t* sources, int32_t* out,
                           const medusa_opts& o, medusa_stats& st, bool capture = true) {
    const uint32_t n = g->n;
    const unsigned long long m = g->m;
    const uint32_t nwords = (n + 63) / 64;
    const uint32_t large = bfs_large(g, o), grid = bfs_grid(g, o);
    hipStream_t s = g->stream;
    const uint32_t mode = bfs_mode(o);
    const float* policy = mode == 3 ? policy_device_params(o.policy) : nullptr;
    const BfsArgs a = bfs_args(g, B, large, grid, policy);
    BfsHost* host = host_counters<BfsHost>(g);

    // where the closing kernel puts the levels: the output itself, or pinned memory for a small host
    // output; larger host outputs are copied afterwards
    const bool in_place = out == B.level, direct = !in_place && kernels_can_write(g, out, (size_t)n * 4);
    const bool staged = !in_place && !direct && (size_t)n * 4 <= kBfsStageBytes && !is_device_memory(out);
    if (staged) g->h_levels.ensure(n);
    int32_t* target = direct ? out : staged ? g->h_levels.p : nullptr;

    const bool by_start = nsrc <= kBfsHostSources;
    auto launch = [&](bool start, uint32_t slots) {
        if (start) {
            hipLaunchKernelGGL(k_bfs_seed, dim3(grid_for(n, 256, 4096)), dim3(256), 0, s, a, 0xFFFFFFFFu);
            hipLaunchKernelGGL(k_bfs_start, dim3(1), dim3(1024), 0, s, a, (const BfsHost*)host, m);
        }
        for (uint32_t k = 0; k < slots; ++k) bfs_enqueue_slot(g, a, k & 1u);
        hipLaunchKernelGGL(k_bfs_close, dim3(grid_for(n, 1024, 1024)), dim3(256), 0, s, a, host, slots & 1u);
        MDS_LAUNCHED();
    };
    // capture (once per graph, threshold, policy buffer and slot count) a run's kernels
    auto captured = [&](GraphCache& gc, bool start, uint32_t slots) -> hipGraphExec_t {
        const uintptr_t key[6] = {(uintptr_t)B.level, (uintptr_t)B.hub[0], (uintptr_t)policy,
                                  ((uintptr_t)grid << 32) | large, (uintptr_t)B.vis[0], (uintptr_t)B.q[0]};
        if (gc.exec && std::equal(key, key + 6, gc.key)) return gc.exec;
        gc.reset();
        MDS_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        hipGraph_t graph = nullptr;
        hipError_t e = hipSuccess;
        try {
            launch(start, slots);
        } catch (...) {
            (void)hipStreamEndCapture(s, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        e = hipStreamEndCapture(s, &graph);
        if (e == hipSuccess) e = hipGraphInstantiate(&gc.exec, graph, nullptr, nullptr, 0);
        if (graph) (void)hipGraphDestroy(graph);
        MDS_HIP(e);
        std::copy(key, key + 6, gc.key);
        return gc.exec;
    };
    // a handle's first run launches its first sequence: what it would capture has a slot count that the
    // next run, which knows how many it takes, rarely wants again (first run on ER with 80 K vertices
    // 280 us with the capture, 149 without; with 8.7 K 210 and 124; RMAT-20 704 and 678)
    const bool known = g->bfs_next_head != kNoHead;
    const uint32_t head = known ? g->bfs_next_head : kBfsBatch;
    hipGraphExec_t exec = nullptr;
    if (capture && !by_start) exec = captured(g->bfs_graph, false, kBfsBatch);
    else if (capture && known) exec = captured(g->bfs_heads[head], true, head);

    host->out = target;
    host->count = nsrc;
    host->mode = mode;
    host->ctl.done = 0;
    if (by_start) {
        std::copy(sources, sources + nsrc, host->src);
    } else {
        bfs_seed(g, B, a, nsrc, sources[0]);
        hipLaunchKernelGGL(k_bfs_first_decide, dim3(1), dim3(kWave), 0, s, a, m, mode, target);
        MDS_LAUNCHED();
    }
    for (uint32_t batch = 0;; ++batch) {
        if (capture && batch > 0) exec = captured(g->bfs_graph, false, kBfsBatch);
        if (exec) MDS_HIP(hipGraphLaunch(exec, s));
        else launch(by_start && batch == 0, kBfsBatch);
        MDS_HIP(hipStreamSynchronize(s));
        if (host->ctl.done) break;
        MDS_CHECK(batch < (2ull * n + 2) / kBfsBatch + 2, MEDUSA_ERR_INTERNAL, "bfs: superstep loop did not end");
    }
    const BfsCtl h = host->ctl;
    if (capture) g->bfs_next_head = std::min(h.slots, kMaxHeadSlots);
    st.device_ms = (double)(host->t_end - h.t_begin) / (double)g->wall_khz;
    st.supersteps = h.supersteps;
    st.push_steps = h.push_steps;
    st.pull_steps = h.pull_steps;
    st.edges_traversed = h.reached_edges;
    st.reached = (uint32_t)h.reached;
    st.kernel_bytes = h.kernel_bytes;
    st.alg_bytes = h.alg_bytes + bfs_seed_bytes(n, nwords, nsrc);
    if (staged) std::memcpy(out, g->h_levels.p, (size_t)n * 4);
    else if (!in_place && !direct) copy_out(g, out, B.level, (size_t)n * 4);
}

// Sums of the counter slots, read back to the host (waits for the stream).
struct BfsSums {
    uint32_t n_new = 0, n_hub = 0;
    unsigned long long deg_sum = 0, deg_large = 0, probes = 0;
};
static BfsSums read_bfs_counters(medusa_graph* g, const BfsCounters* ctr, uint32_t par_next) {
    static_assert(sizeof(BfsCounters) <= kHostWords * 8, "pinned memory of a handle");
    MDS_HIP(hipMemcpyAsync(g->h_ctr_raw.p, ctr, sizeof(BfsCounters), hipMemcpyDeviceToHost, g->stream));
    MDS_HIP(hipStreamSynchronize(g->stream));
    BfsCounters h;
    std::memcpy(&h, g->h_ctr_raw.p, sizeof(BfsCounters));
    unsigned long long joined = 0, work = 0;
    for (uint32_t i = 0; i < kBfsSlots; ++i) {
        joined += h.seg[par_next][i].v;
        work += h.work[i].v;
    }
    BfsSums r;
    r.n_new = (uint32_t)joined;
    r.deg_sum = joined >> 32;
    r.deg_large = (uint32_t)work;
    r.probes = work >> 32;
    r.n_hub = h.n_hub;
    return r;
}

// Host-driven run: the same kernels, with the host deciding each superstep from the counters
// read back after it (timing and tracing); a superstep's time covers its expansion and, after
// a push, the compaction.
static void bfs_run_host(medusa_graph* g, uint32_t nsrc, uint32_t single, int32_t* out, const medusa_opts& o,
                         medusa_stats& st) {
    const uint32_t n = g->n;
    const uint64_t m = g->m;
    const uint32_t nwords = (n + 63) / 64;
    const uint32_t large = bfs_large(g, o), grid = bfs_grid(g, o);
    hipStream_t s = g->stream;
    const bool timing = o.timing != 0;
    const BfsBufs B = handle_bufs(g);
    const BfsArgs a = bfs_args(g, B, large, grid, nullptr);
    g->trace.clear();

    MDS_HIP(hipEventRecord(g->ev_begin, s));
    bfs_seed(g, B, a, nsrc, single);
    BfsSums c = read_bfs_counters(g, B.ctr, 0);

    Frontier f{};
    f.n = n;
    f.m = m;
    f.n_f = c.n_new;
    f.m_f = c.deg_sum;
    f.n_u = n - f.n_f;
    f.m_u = m - f.m_f;
    uint64_t reached_edges = f.m_f, reached = f.n_f, bytes = bfs_seed_bytes(n, nwords, nsrc);
    bool pull = false;
    uint32_t vsel = 0;
    uint32_t solo_cap = nsrc <= kBfsHostSources ? kSoloStart : kSoloSlot;
    Sched sched(o, Sched::kBfs);
    if (timing) ensure_events(g, 2);
    for (uint32_t t = 0;; ++t) {
        f.step = t;
        // the device-driven loop's solo supersteps are pushes, here of the whole grid
        if (o.direction != MEDUSA_DIR_PULL && !bfs_solo_fits(solo_cap, n, f.n_f, f.m_f)) solo_cap = kSoloSlot;
        if (o.direction == MEDUSA_DIR_PUSH) pull = false;
        else if (o.direction == MEDUSA_DIR_PULL) pull = true;
        else pull = bfs_solo_fits(solo_cap, n, f.n_f, f.m_f) ? false : sched.bfs_pull(f, pull);
        const uint32_t n_small = c.n_new - c.n_hub;
        const uint32_t hub = bfs_hub_wgs(grid, n_small, c.n_hub, c.deg_large, c.deg_sum);
        const uint32_t small = bfs_small(pull, f.n_f, f.m_f, a.exact_edges);
        hipLaunchKernelGGL(k_bfs_set_ctl, dim3(1), dim3(1), 0, s, B.ctl, (int32_t)t, pull ? 1u : 0u, small, n_small,
                           c.n_hub, hub, vsel);
        MDS_LAUNCHED();
        hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(kWave), 0, s, a.ctr, (t & 1u) ^ 1u);
        MDS_LAUNCHED();
        if (timing) MDS_HIP(hipEventRecord(g->events[0], s));
        hipLaunchKernelGGL(k_bfs_super<false>, dim3(grid), dim3(256), 0, s, a, 0u);
        MDS_LAUNCHED();
        if (!pull && !small) {  // the compaction
            hipLaunchKernelGGL(k_bfs_super<false>, dim3(grid), dim3(256), 0, s, a, 1u);
            MDS_LAUNCHED();
        }
        if (timing) MDS_HIP(hipEventRecord(g->events[1], s));
        c = read_bfs_counters(g, B.ctr, (t & 1u) ^ 1u);
        double kms = 0;
        if (timing) {
            float ms = 0;
            MDS_HIP(hipEventElapsedTime(&ms, g->events[0], g->events[1]));
            kms = ms;
            st.kernel_ms += ms;
            ++st.kernel_launches;
        }
        // the byte model of the device-driven loop's decision
        uint64_t kb;
        if (pull) {
            kb = 8ull * f.n_u + 8ull * c.probes + 16ull * nwords + 16ull * c.n_new;
            ++st.pull_steps;
            vsel ^= 1u;
        } else if (small) {
            kb = 12ull * f.n_f + 8ull * f.m_f + 24ull * c.n_new;
            ++st.push_steps;
        } else {
            kb = 12ull * f.n_f + 8ull * f.m_f + 4ull * n + 8ull * nwords + 16ull * c.n_new;
            ++st.push_steps;
        }
        st.kernel_bytes += kb;
        bytes += kb;
        sched.record(g, f, pull ? 1.0 : 0.0, kms);
        ++st.supersteps;
        if (c.n_new == 0) break;
        f.n_f = c.n_new;
        f.m_f = c.deg_sum;
        f.n_u -= c.n_new;
        f.m_u -= c.deg_sum;
        reached += c.n_new;
        reached_edges += c.deg_sum;
    }
    MDS_HIP(hipEventRecord(g->ev_end, s));
    MDS_HIP(hipStreamSynchronize(s));
    float ms = 0;
    MDS_HIP(hipEventElapsedTime(&ms, g->ev_begin, g->ev_end));
    st.device_ms = ms;
    st.edges_traversed = reached_edges;
    st.reached = (uint32_t)reached;
    st.alg_bytes = bytes;
    copy_out(g, out, g->level.p, (size_t)n * 4);
}

static void bfs_entry(medusa_graph* g, const uint32_t* sources, uint32_t count, int32_t* levels,
                      const medusa_opts* opts, medusa_stats* stats) {
    const auto lock = enter(g);
    MDS_CHECK(levels, MEDUSA_ERR_ARG, "bfs: null output");
    MDS_CHECK(sources && count >= 1, MEDUSA_ERR_ARG, "bfs: need at least one source");
    const uint32_t n = g->n;
    for (uint32_t i = 0; i < count; ++i)
        MDS_CHECK(sources[i] < n, MEDUSA_ERR_ARG, "bfs: source %u out of range (n=%u)", sources[i], n);
    medusa_opts o{};
    if (opts) o = *opts;
    MDS_CHECK(o.direction >= 0 && o.direction <= 2, MEDUSA_ERR_ARG, "bfs: bad direction %d", o.direction);
    MDS_CHECK(o.grid == 0 || (o.grid >= 2 && o.grid <= 65535), MEDUSA_ERR_ARG, "bfs: grid must be 0 or 2..65535");
    g->level.ensure(n);
    g->q_small.ensure(2 * bfs_queue_cap(n));
    g->q_large.ensure(2 * (size_t)n);
    g->q_aux.ensure(std::max(n, count));
    g->bitmap.ensure(2 * (((size_t)n + 63) / 64));
    if (count > (o.timing || o.trace ? 1u : kBfsHostSources))
        MDS_HIP(hipMemcpyAsync(g->q_aux.p, sources, (size_t)count * 4, hipMemcpyHostToDevice, g->stream));
    medusa_stats st{};
    if (o.timing || o.trace) bfs_run_host(g, count, sources[0], levels, o, st);
    else bfs_run_device(g, handle_bufs(g), count, sources, levels, o, st);
    if (stats) *stats = st;
}

// ---- BFS with no device allocation ------------------------------------------------
// Work buffers of medusa_bfs_noalloc: two frontier queues and two hub queues of
// kNoAllocMaxVertices entries each, two visited bitmaps, the control
// blocks and the counters, in one array per GPU that lives as long as the process.  Host code
// must not pass `scratch` itself to a kernel (in host code the name is a stand-in, not a device
// address): the device address is looked up once per device with hipGetSymbolAddress and kept
// in s_scratch.
constexpr uint32_t kNoAllocMaxVertices = MEDUSA_NOALLOC_MAX_VERTICES;
constexpr size_t kNoAllocQueueBytes = (size_t)kNoAllocMaxVertices * 4;
constexpr size_t kNoAllocBitmapBytes = (size_t)kNoAllocMaxVertices / 8;
static_assert((size_t)kBfsSlots * bfs_span(kNoAllocMaxVertices) == kNoAllocMaxVertices,
              "the segmented queue of the largest graph fills kNoAllocMaxVertices entries exactly");
constexpr size_t kNoAllocBytes = 4 * kNoAllocQueueBytes + 2 * kNoAllocBitmapBytes + kBfsCtlUnits * sizeof(CtlStorage);
static_assert(kNoAllocMaxVertices % 2048 == 0, "queue and bitmap regions stay 256-byte aligned");
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
static std::mutex s_scratch_mu;
static unsigned char* s_scratch[kMaxDevices] = {};

static unsigned char* scratch_on(int device) {
    MDS_CHECK(device >= 0 && device < kMaxDevices, MEDUSA_ERR_ARG, "bfs_noalloc: device %d out of range", device);
    const std::lock_guard<std::mutex> lock(s_scratch_mu);
    if (!s_scratch[device]) {
        void* p = nullptr;
        MDS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));  // the calling thread has `device` current
        MDS_CHECK(p != nullptr, MEDUSA_ERR_HIP, "bfs_noalloc: no address for the scratch array");
        s_scratch[device] = static_cast<unsigned char*>(p);
    }
    return s_scratch[device];
}

static void bfs_noalloc(medusa_graph* g, uint32_t source, int32_t* levels, medusa_stats* stats) {
    const auto lock = enter(g);  // makes the graph's device current
    const uint32_t n = g->n;
    MDS_CHECK(levels, MEDUSA_ERR_ARG, "bfs_noalloc: null output");
    MDS_CHECK(source < n, MEDUSA_ERR_ARG, "bfs_noalloc: source %u out of range (n=%u)", source, n);
    MDS_CHECK(n <= kNoAllocMaxVertices, MEDUSA_ERR_ARG,
              "bfs_noalloc: %u vertices exceed the scratch limit of %u (MEDUSA_NOALLOC_MAX_VERTICES)", n,
              kNoAllocMaxVertices);
    hipPointerAttribute_t attr{};
    const hipError_t e = hipPointerGetAttributes(&attr, levels);
    (void)hipGetLastError();
    MDS_CHECK(e == hipSuccess && attr.type == hipMemoryTypeDevice && attr.device == g->device, MEDUSA_ERR_ARG,
              "bfs_noalloc: levels must be device memory of the graph's GPU");
    unsigned char* base = scratch_on(g->device);
    BfsBufs B{};
    B.level = levels;
    // a graph of n <= kNoAllocMaxVertices vertices needs at most kNoAllocMaxVertices entries per queue
    MDS_CHECK(bfs_queue_cap(n) <= kNoAllocMaxVertices, MEDUSA_ERR_INTERNAL, "bfs_noalloc: queue layout");
    for (int i = 0; i < 2; ++i) {
        B.q[i] = reinterpret_cast<uint32_t*>(base + i * kNoAllocQueueBytes);
        B.hub[i] = reinterpret_cast<uint32_t*>(base + (2 + i) * kNoAllocQueueBytes);
    }
    for (int i = 0; i < 2; ++i)
        B.vis[i] = reinterpret_cast<unsigned long long*>(base + 4 * kNoAllocQueueBytes + i * kNoAllocBitmapBytes);
    CtlStorage* ctl = reinterpret_cast<CtlStorage*>(base + 4 * kNoAllocQueueBytes + 2 * kNoAllocBitmapBytes);
    B.ctl = reinterpret_cast<BfsCtl*>(ctl);
    B.ctr = reinterpret_cast<BfsCounters*>(ctl + 2);
    B.sources = nullptr;  // one source: not used
    medusa_opts o{};  // heuristic direction, default or tuned launch shape
    medusa_stats st{};
    bfs_run_device(g, B, 1, &source, levels, o, st, /*capture=*/false);
    if (stats) *stats = st;
}

}  // namespace medusa

using namespace medusa;

extern "C" int medusa_bfs(medusa_graph* g, uint32_t source, int32_t* levels, const medusa_opts* opts,
                          medusa_stats* stats) {
    return guard([&] { bfs_entry(g, &source, 1, levels, opts, stats); });
}

extern "C" int medusa_bfs_multi(medusa_graph* g, const uint32_t* sources, uint32_t count, int32_t* levels,
                                const medusa_opts* opts, medusa_stats* stats) {
    return guard([&] { bfs_entry(g, sources, count, levels, opts, stats); });
}

extern "C" int medusa_bfs_noalloc(medusa_graph* g, uint32_t source, int32_t* levels, medusa_stats* stats) {
    return guard([&] { bfs_noalloc(g, source, levels, stats); });
}
