// PageRank superstep engine (FP32, compensated combine in a fixed order).
//
// Reference: MPG/UserOperators.h:175-270 runs per superstep InitMessageBuffer(0.0)
// (MPG/InitMessage.h), SendMsg* scatter of rank/outdeg into per-in-edge message
// slots (MPG/UserOperators.h:29-163), a CUDPP segmented ADD scan (MPG/MsgCombiner.h:68-117)
// and UpdateVertex rank = 0.15 + 0.85*sum (MPG/UserOperators.h:16-26); fixed 100
// supersteps (MPG/main.cu:166).  Here the formula is the normalised one with
// dangling mass redistributed:
//     r_0 = 1/n,  r_{t+1}(v) = (1-d)/n + d*(S_t(v) + D_t/n)
//     S_t(v) = sum over in-edges u->v of c_t(u),  c_t(u) = r_t(u)/outdeg(u)
//     D_t = sum of r_t(u) over outdeg(u) == 0.
//
// A packed batch of disjoint graphs runs in the same launches: graph g uses its own
// vertex count n_g for r_0, (1-d)/n_g and D_t/n_g, and D_t sums its own dangling vertices,
// so every graph's ranks are bit-identical to a run on that graph alone.
//
// Canonical combine order (identical for every kernel variant and lane mapping,
// so push/pull and every binning give bit-identical ranks):
//   a segment of values x_0..x_{L-1} (in-edges in ascending original source id,
//   or dangling vertices in internal order) is cut into blocks of 4096; in a
//   block, lane j (0..63) Kahan-adds x_{j}, x_{j+64}, ... in order starting from
//   (0,0); lanes are then merged by kahan_combine down a tree with offsets
//   32,16,8,4,2,1 (lane i absorbs lane i+off); block results are merged left to
//   right with kahan_combine; the value is s - c.
// Scalars: d_f = (float)d, tele = (float)((1-d)/n), base_t = fmaf(d_f, D_t/(float)n, tele),
// r_0 = (float)(1/n),
// r_{t+1}(v) = fmaf(d_f, S_t(v), base_t), c = r/(float)outdeg (IEEE division).

#include <cmath>

#include "engine.h"
#include "sched.h"

namespace medusa {

constexpr uint32_t kBlock = 4096;  // elements per canonical block (64 lanes x 64 rounds)

// Lane exchanges of the canonical tree, in vector registers (v_permlane32_swap, v_permlane16_swap
// and row shifts) instead of through the LDS crossbar.
//
// swap32 turns a, b into (a's lanes 0..31 | b's lanes 0..31) and (a's 32..63 | b's 32..63);
// swap16 does the same with the 16-lane rows of each half: a = (a0 b0 a2 b2), b = (a1 b1 a3 b3).
__device__ __forceinline__ void swap32(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    const uint32_t lo = r[0], hi = r[1];  // a bit_cast of a vector element takes element 0
    a = __builtin_bit_cast(float, lo);
    b = __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ void swap16(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    const uint32_t lo = r[0], hi = r[1];  // a bit_cast of a vector element takes element 0
    a = __builtin_bit_cast(float, lo);
    b = __builtin_bit_cast(float, hi);
}
// x of the lane kOff above in the same 16-lane row (0 past the row's end).
template <int kOff>
__device__ __forceinline__ float row_above(float x) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x100 | kOff, 0xf, 0xf, true));
}

// Two lanes' pairs as the tree's offset 32 (16) merges them, for two vertices at once: the lower
// half (the even rows) of the result holds (s, c)'s vertex, the other half (the odd rows)
// (s2, c2)'s.  With one vertex in both arguments both halves (both rows) end the same.
__device__ __forceinline__ void merge32(float& s, float& c, float s2, float c2) {
    swap32(s, s2);
    swap32(c, c2);
    kahan_combine(s, c, s2, c2);
}
__device__ __forceinline__ void merge16(float& s, float& c, float s2, float c2) {
    swap16(s, s2);
    swap16(c, c2);
    kahan_combine(s, c, s2, c2);
}
// Offsets 8, 4, 2, 1 inside every 16-lane row; the row's lane 0 ends with its result.
__device__ __forceinline__ void row_tree(float& s, float& c) {
    kahan_combine(s, c, row_above<8>(s), row_above<8>(c));
    kahan_combine(s, c, row_above<4>(s), row_above<4>(c));
    kahan_combine(s, c, row_above<2>(s), row_above<2>(c));
    kahan_combine(s, c, row_above<1>(s), row_above<1>(c));
}
// The whole 64-lane tree of one vertex; lane 0 ends with the result.
__device__ __forceinline__ void wave_tree(float& s, float& c) {
    merge32(s, c, s, c);
    merge16(s, c, s, c);
    row_tree(s, c);
}

// Canonical sum of `len` values x(k), computed by one whole wave; every lane
// returns the same (s - c).  Each lane keeps 16 loads in flight and adds them
// in ascending order.
template <class Load>
__device__ __forceinline__ float wave_segment_sum(uint32_t len, Load load) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    float as = 0.f, ac = 0.f;
    for (uint32_t b0 = 0; b0 < len; b0 = advance_to(b0, kBlock, len)) {
        const uint32_t lim = min(len - b0, kBlock);
        float s = 0.f, c = 0.f;
        for (uint32_t r0 = 0; r0 * kWave < lim; r0 += 16) {
            float x[16];
#pragma unroll
            for (uint32_t j = 0; j < 16; ++j) {
                const uint32_t k = lane + (r0 + j) * kWave;
                x[j] = k < lim ? load(b0 + k) : 0.f;
            }
#pragma unroll
            for (uint32_t j = 0; j < 16; ++j)
                if (lane + (r0 + j) * kWave < lim) kahan_add(s, c, x[j]);
        }
        wave_tree(s, c);
        s = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, s)));
        c = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, c)));
        if (b0 == 0) {
            as = s;
            ac = c;
        } else {
            kahan_combine(as, ac, s, c);
        }
    }
    return as - ac;
}

// 16-leaf canonical subtree in registers: slot j absorbs slot j+off for
// off = 8, 4, 2, 1.  Absent leaves are (0,0), an exact identity.
__device__ __forceinline__ void tree16(float (&s)[16], float (&c)[16]) {
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1)
#pragma unroll
        for (int j = 0; j < off; ++j) kahan_combine(s[j], c[j], s[j + off], c[j + off]);
}

// Leaves r, r+st, ..., r+15*st of a vertex of in-degree `deg` (one lane), reduced
// by tree16.  Element i of the vertex sits at col[i*stride] (ELL slab, pull) or at
// vals[seg + i] (message slots, push).
template <bool kFromMsg>
__device__ __forceinline__ void lane_subtree(float& S, float& C, uint32_t r, uint32_t st, uint32_t deg,
                                             const uint32_t* __restrict__ col, uint32_t stride,
                                             const float* __restrict__ vals, uint32_t seg) {
    uint32_t idx[16];
    float s[16], c[16];
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) {
        const uint32_t i = r + st * j;
        idx[j] = (i < deg) ? (kFromMsg ? seg + i : col[(size_t)i * stride]) : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) {
        s[j] = (r + st * j < deg) ? vals[idx[j]] : 0.f;
        c[j] = 0.f;
    }
    tree16(s, c);
    S = s[0];
    C = c[0];
}

// Binned variant: the sums of one lane item (planned by pr_bins.h), whose lane l holds slots
// at[64 j + l], j = 0, 1, ...: with `per` = pr_lane_group(deg) vertices the item's slots are
// column-major, so that is element r + st j of vertex l mod per, with st = 64 / per and
// r = l / per.  A lane reduces its (at most 16) elements by the tree's offsets down to st, then
// the st lanes of a vertex merge by the offsets below it, and lane i < per ends with vertex i's
// sum.  Slots past a vertex's own in-degree hold +0.0 and are not distinguished from elements:
// (0, 0) pairs merge as the exact identity that the canonical tree uses for absent elements.
template <uint32_t L>
__device__ __forceinline__ void lane_item_leaves(float& S, float& C, uint32_t st, uint32_t deg, const float* at) {
    const uint32_t r = st == 1 ? 0u : st == 2 ? lane_id() >> 5 : lane_id() >> 4;
    float s[L], c[L];
#pragma unroll
    for (uint32_t j = 0; j < L; ++j) {
        s[j] = r + st * j < deg ? at[64 * j] : 0.f;
        c[j] = 0.f;
    }
#pragma unroll
    for (uint32_t off = L / 2; off >= 1; off >>= 1)
#pragma unroll
        for (uint32_t j = 0; j < off; ++j) kahan_combine(s[j], c[j], s[j + off], c[j + off]);
    S = s[0];
    C = c[0];
}
__device__ __forceinline__ float lane_item_sum(uint32_t deg, const float* at) {
    float s, c;
    if (deg <= 1) {
        lane_item_leaves<1>(s, c, 1, deg, at);
    } else if (deg <= 2) {
        lane_item_leaves<2>(s, c, 1, deg, at);
    } else if (deg <= 4) {
        lane_item_leaves<4>(s, c, 1, deg, at);
    } else if (deg <= 8) {
        lane_item_leaves<8>(s, c, 1, deg, at);
    } else {
        const uint32_t st = 64 / pr_lane_group(deg);
        lane_item_leaves<16>(s, c, st, deg, at);
        if (st >= 2) merge32(s, c, s, c);
        if (st == 4) merge16(s, c, s, c);
    }
    return s - c;
}

// Canonical (s, c) pair of one dangling block, computed by one wave (lane 0 holds it).
__device__ __forceinline__ void dangle_block_sum(const float* __restrict__ rank, const PrBlock B, float& s, float& c) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const float* x = rank + B.begin;
    s = 0.f;
    c = 0.f;
    for (uint32_t r0 = 0; r0 * kWave < B.len; r0 += 16) {
        float v[16];
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j) {
            const uint32_t k = lane + (r0 + j) * kWave;
            v[j] = k < B.len ? x[k] : 0.f;
        }
#pragma unroll
        for (uint32_t j = 0; j < 16; ++j)
            if (lane + (r0 + j) * kWave < B.len) kahan_add(s, c, v[j]);
    }
    wave_tree(s, c);
}

// base = fmaf(d, D / (float)n_g, (float)((1 - d) / n_g)) for dangling mass D.
__device__ __forceinline__ float pr_base_value(float D, float d, uint32_t n_g) {
    const float tele = (float)((1.0 - (double)d) / (double)n_g);
    return fmaf(d, D / (float)n_g, tele);
}

// A single graph with at most this many dangling vertices (one block) can have every wave of the
// pull or push superstep sum them itself, 16 loads a lane and round, instead of a launch of one workgroup
// doing it before.  The launch costs 5 us, a round about 1.3 us for every 2048 workgroups, which
// run at once: own_base where that is at most kOwnBaseRounds.  Pull superstep with the launch and
// without: RMAT-14 (1781 dangling) 7.5 and 5.9 us, RMAT-16, 8 edges a vertex (2593) 8.9 and 7.5, RMAT-17
// (1263) 13.9 and 12.5, RMAT-18 (3034) 26.5 and 26.7, RMAT-19, 24 edges a vertex (2539) 62 and 75.
constexpr uint32_t kOwnBaseVertices = 4096, kOwnBaseRounds = 4;

// One superstep for every vertex.  kFromMsg: values come from the message
// array in slot order (push variant) instead of contrib[src] (pull variant).  kOwnBase: every
// wave sums the dangling block `dangling` of rank_in itself; otherwise base_p was written before.
template <bool kFromMsg, bool kOwnBase>
__global__ __launch_bounds__(256) void k_pr_main(const PrRun* __restrict__ runs, const uint32_t* __restrict__ wg_run,
                                                 const uint32_t* __restrict__ ell, const uint32_t* __restrict__ cptr,
                                                 const uint32_t* __restrict__ crow,
                                                 const float* __restrict__ vals,
                                                 const uint32_t* __restrict__ outdeg,
                                                 const float* __restrict__ base_p,
                                                 const float* __restrict__ rank_in, PrBlock dangling, uint32_t n,
                                                 float d, float* __restrict__ rank_out,
                                                 float* __restrict__ contrib_out) {
    const uint32_t wg = blockIdx.x;
    const PrRun R = runs[wg_run[wg]];  // a table lookup, not a search at every workgroup's start
    const uint32_t local = wg - R.wg_begin;
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    float base;
    if constexpr (kOwnBase) {
        float s, c;
        dangle_block_sum(rank_in, dangling, s, c);
        const float D = s - c;
        base = pr_base_value(
            __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, D))), d, n);
    } else {
        base = base_p[R.part];
    }

    auto finish = [&](uint32_t p, float S) {
        const float r = fmaf(d, S, base);
        rank_out[p] = r;
        const uint32_t od = outdeg[p];
        if (od) contrib_out[p] = r / (float)od;
    };

    if (R.kind == kPrWave) {
        const uint32_t p = R.begin + local * 4 + wave;
        if (p >= R.begin + R.count) return;  // uniform across the wave
        const uint32_t b = cptr[p], len = cptr[p + 1] - b;
        const float S = wave_segment_sum(len, [&](uint32_t k) {
            return kFromMsg ? vals[b + k] : vals[crow[b + k]];
        });
        if (lane == 0) finish(p, S);
        return;
    }
    // kPrLane (and kPrZero, whose deg is 0): a wave takes `per` vertices, 64 / per lanes each, so
    // no lane gathers more than 16 values, in one round of loads.  With one lane per vertex
    // whatever the in-degree, a vertex of 33..64 in-edges was four rounds of index loads and
    // gathers in one lane: pull superstep of
    // RMAT-16 9.2 -> 7.5 us, RMAT-18 32 -> 27 us (41 registers instead of 94).
    const uint32_t per = pr_lane_group(R.deg), st = kWave / per;
    const uint32_t i = local * 4 * per + wave * per + (lane & (per - 1));
    const bool in = i < R.count;  // the lanes of a vertex agree
    const uint32_t p = R.begin + (in ? i : 0u);
    float S, C;
    lane_subtree<kFromMsg>(S, C, lane / per, st, in ? R.deg : 0u, ell + R.ell_base + (in ? i : 0u), R.ell_stride, vals,
                           kFromMsg ? cptr[p] : 0u);
    if (st >= 2) merge32(S, C, S, C);
    if (st == 4) merge16(S, C, S, C);
    if (in && lane < per) finish(p, S - C);
}

// Dangling mass, step 1: one wave per canonical block of a graph's dangling tail
// writes the block's (s, c) pair.
__global__ __launch_bounds__(256) void k_pr_dangle(const float* __restrict__ rank, const PrBlock* __restrict__ blocks,
                                                   uint32_t nblk, float* __restrict__ partials) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const uint32_t b = blockIdx.x * 4 + wave;
    if (b >= nblk) return;  // uniform across the wave
    float s, c;
    dangle_block_sum(rank, blocks[b], s, c);
    if (lane == 0) {
        partials[2 * b] = s;
        partials[2 * b + 1] = c;
    }
}

// base = fmaf(d, D / (float)n_g, (float)((1 - d) / n_g)) of a graph whose `nblocks` block pairs
// start at partials[2 * first]: the pairs merge left to right.  Called by a whole wave; every
// lane returns the value.
__device__ __forceinline__ float pr_base_fold(const float* __restrict__ partials, uint32_t first, uint32_t nblocks,
                                              uint32_t n_g, float d) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    float as = 0.f, ac = 0.f;
    for (uint32_t c0 = 0; c0 < nblocks; c0 += kWave) {
        const uint32_t i = c0 + lane;
        const float ps = i < nblocks ? partials[2 * (first + i)] : 0.f;
        const float pc = i < nblocks ? partials[2 * (first + i) + 1] : 0.f;
        const uint32_t lim = min(nblocks - c0, (uint32_t)kWave);
        for (uint32_t j = 0; j < lim; ++j) {
            const float s2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ps), j));
            const float c2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pc), j));
            if (c0 + j == 0) {
                as = s2;
                ac = c2;
            } else {
                kahan_combine(as, ac, s2, c2);
            }
        }
    }
    return pr_base_value(as - ac, d, n_g);
}

// Dangling mass, step 2 (after the block kernel, so its partials are visible): one wave
// per graph merges the graph's block pairs and writes its base.
__global__ __launch_bounds__(256) void k_pr_base(const float* __restrict__ partials, const PrPart* __restrict__ parts,
                                                 uint32_t nparts, float d, float* __restrict__ base_out) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t w = blockIdx.x * 4 + threadIdx.x / kWave;
    if (w >= nparts) return;  // uniform across the wave
    const PrPart P = parts[w];
    const float base = pr_base_fold(partials, P.first_block, P.nblocks, P.n, d);
    if (lane == 0) base_out[w] = base;
}

// Dangling mass of several graphs (or of one with many blocks) inside the binned send: every
// block's wave publishes its pair and takes a ticket, and the wave with the last ticket merges
// the pairs of all graphs into their bases, so the combine needs no launch in between (4.5 us of
// the 30 us superstep of a batch of 64 graphs, 8 M arcs).  The exchanges' results are waited for
// before the ticket is drawn, and the merging wave reads the pairs with device-scope loads, so
// no fence is needed.
constexpr uint32_t kFoldParts = 256;      // graphs a single wave merges, one lane each
constexpr uint32_t kFoldPartBlocks = 32;  // blocks per graph up to which one lane merges them

// Whether the send merges the bases itself (above the limits a launch of k_pr_base does, one wave
// per graph; nothing dangling leaves no wave to take a ticket).
static bool pr_send_folds(const PrLayout& L) {
    if (L.blocks.empty()) return false;
    if (L.parts.size() == 1) return true;
    uint32_t most = 0;
    for (const PrPart& P : L.parts) most = std::max(most, P.nblocks);
    return L.parts.size() <= kFoldParts && most <= kFoldPartBlocks;
}

// Bases of every graph from the published pairs, by one wave; graph order and merge order as in
// k_pr_base.
__device__ __forceinline__ void pr_fold_published(const float* __restrict__ partials, uint32_t nblk,
                                                  const PrPart* __restrict__ parts, uint32_t nparts, float d,
                                                  float* __restrict__ base_out) {
    const uint32_t lane = lane_id();
    float as = 0.f, ac = 0.f;
    if (nparts == 1) {
        for (uint32_t c0 = 0; c0 < nblk; c0 += kWave) {
            const uint32_t i = c0 + lane;
            const float ps = i < nblk ? load_now(partials + 2 * i) : 0.f;
            const float pc = i < nblk ? load_now(partials + 2 * i + 1) : 0.f;
            const uint32_t lim = min(nblk - c0, (uint32_t)kWave);
            for (uint32_t j = 0; j < lim; ++j) {
                const float s2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ps), j));
                const float c2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pc), j));
                if (c0 + j == 0) {
                    as = s2;
                    ac = c2;
                } else {
                    kahan_combine(as, ac, s2, c2);
                }
            }
        }
        if (lane == 0) base_out[0] = pr_base_value(as - ac, d, parts[0].n);
        return;
    }
    for (uint32_t g = lane; g < nparts; g += kWave) {
        const PrPart P = parts[g];
        as = ac = 0.f;
        for (uint32_t i0 = 0; i0 < P.nblocks; i0 += 8) {
            float s2[8], c2[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                const bool in = i0 + j < P.nblocks;
                s2[j] = in ? load_now(partials + 2 * (P.first_block + i0 + j)) : 0.f;
                c2[j] = in ? load_now(partials + 2 * (P.first_block + i0 + j) + 1) : 0.f;
            }
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                if (i0 + j >= P.nblocks) continue;
                if (i0 + j == 0) {
                    as = s2[j];
                    ac = c2[j];
                } else {
                    kahan_combine(as, ac, s2[j], c2[j]);
                }
            }
        }
        base_out[g] = pr_base_value(as - ac, d, P.n);
    }
}

constexpr uint32_t kSmallBlocks = 64;  // dangling blocks up to which one workgroup does both steps

// Both dangling-mass steps in one workgroup when there are at most kSmallBlocks blocks:
// wave w sums blocks w, w+4, ... into LDS, then wave w merges graphs w, w+4, ... in block
// order.  Same operations and order as k_pr_dangle followed by k_pr_base.
__global__ __launch_bounds__(256) void k_pr_dangle_base(const float* __restrict__ rank,
                                                        const PrBlock* __restrict__ blocks, uint32_t nblk,
                                                        const PrPart* __restrict__ parts, uint32_t nparts, float d,
                                                        float* __restrict__ base_out) {
    __shared__ float s_s[kSmallBlocks], s_c[kSmallBlocks];
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    for (uint32_t b = wave; b < nblk; b += 4) {
        float s, c;
        dangle_block_sum(rank, blocks[b], s, c);
        if (lane == 0) {
            s_s[b] = s;
            s_c[b] = c;
        }
    }
    __syncthreads();
    if (lane != 0) return;
    for (uint32_t g = wave; g < nparts; g += 4) {
        const PrPart P = parts[g];
        float as = 0.f, ac = 0.f;
        for (uint32_t i = 0; i < P.nblocks; ++i) {
            if (i == 0) {
                as = s_s[P.first_block];
                ac = s_c[P.first_block];
            } else {
                kahan_combine(as, ac, s_s[P.first_block + i], s_c[P.first_block + i]);
            }
        }
        base_out[g] = pr_base_value(as - ac, d, P.n);
    }
}

// Workgroups of a launch are dispatched round-robin over the 8 XCDs (each with its own L2):
// item b of a launch of `count` maps to XCD (b mod 8)'s contiguous share of the items, so
// consecutive items run on one XCD.
__device__ __forceinline__ uint32_t xcd_major(uint32_t b, uint32_t count) {
    const uint32_t q = count / 8, r = count % 8, x = b % 8, j = b / 8;
    return x * q + min(x, r) + j;
}

// Workgroup b of a launch of `count` (dispatched to XCD b mod 8) takes item
// ((j / kXcdGroup) 8 + x) kXcdGroup + j mod kXcdGroup, b = 8 j + x: blocks of kXcdGroup
// consecutive items run on one XCD at once, and the blocks go round-robin over the XCDs, so
// consecutive items share an L2 while every XCD gets a mix of the items; the tail past the
// last whole round of blocks maps to itself.  A bijection on [0, count).
constexpr uint32_t kXcdGroup = 8;
__device__ __forceinline__ uint32_t xcd_grouped(uint32_t b, uint32_t count) {
    const uint32_t full = count / (8 * kXcdGroup) * (8 * kXcdGroup);
    if (b >= full) return b;
    const uint32_t x = b % 8, j = b / 8;
    return ((j / kXcdGroup) * 8 + x) * kXcdGroup + j % kXcdGroup;
}

constexpr uint32_t kSendThreads = 512;
constexpr uint32_t kSendWaves = kSendThreads / kWave;

// Binned send (one launch per superstep).  Workgroups [0, ntiles) each compute their chunk's
// contributions c = r / outdeg into LDS and write one tile of the message array (contiguous;
// runs are padded to 4 entries, so every access is 16-byte aligned).  Tiles of one chunk run on
// one XCD, so the chunk's ranks are read from HBM once per XCD.
// The first `dwg` workgroups write the (s, c) pairs of the dangling blocks of `rank` (one block
// per wave), which the combine of the same superstep merges into its base; with base_out (see
// pr_send_folds) the last of those waves merges them here.  They come first so that the merge is
// over before the tiles are.
__global__ __launch_bounds__(kSendThreads) void k_pr_send(const PrTile* __restrict__ tiles, uint32_t ntiles,
                                                 const uint16_t* __restrict__ srcloc, const float* __restrict__ rank,
                                                 const uint32_t* __restrict__ outdeg, float* __restrict__ msg,
                                                 const PrBlock* __restrict__ blocks,
                                                 uint32_t nblk, uint32_t dwg, float* __restrict__ partials,
                                                 const PrPart* __restrict__ parts, uint32_t nparts, float d,
                                                 float* __restrict__ base_out, uint32_t* __restrict__ ticket) {
    __shared__ float s_c[kPrChunkSources];
    using u16x4 = unsigned short __attribute__((ext_vector_type(4)));
    using f32x4 = float __attribute__((ext_vector_type(4)));
    using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
    if (blockIdx.x < dwg) {
        const uint32_t lane = threadIdx.x & (kWave - 1);
        const uint32_t b = blockIdx.x * kSendWaves + threadIdx.x / kWave;
        if (b >= nblk) return;  // uniform across the wave
        float bs, bc;
        dangle_block_sum(rank, blocks[b], bs, bc);
        if (!base_out) {
            if (lane == 0) {
                partials[2 * b] = bs;
                partials[2 * b + 1] = bc;
            }
            return;
        }
        uint32_t t = 0;
        if (lane == 0) {
            const float r0 = atomicExch(&partials[2 * b], bs), r1 = atomicExch(&partials[2 * b + 1], bc);
            uint32_t inc = 1;
            asm volatile("" : "+v"(inc) : "v"(r0), "v"(r1));
            t = atomicAdd(ticket, inc);
        }
        t = __builtin_amdgcn_readfirstlane(t);
        if (t != nblk - 1) return;
        pr_fold_published(partials, nblk, parts, nparts, d, base_out);
        if (lane == 0) *ticket = 0;  // for the next superstep's send
        return;
    }
    const PrTile T = tiles[xcd_major(blockIdx.x - dwg, ntiles)];
    const u16x4* __restrict__ sl = reinterpret_cast<const u16x4*>(srcloc + T.msg_begin);
    f32x4* __restrict__ out = reinterpret_cast<f32x4*>(msg + T.msg_begin);
    const uint32_t nq = (T.msg_end - T.msg_begin) / 4;
    auto fetch = [&](uint32_t q0, u16x4(&a)[4]) {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t q = q0 + u * kSendThreads + threadIdx.x;
            a[u] = q < nq ? sl[q] : u16x4{0, 0, 0, 0};
        }
    };
    u16x4 a[4];
    fetch(0, a);  // in flight while the chunk's contributions are computed
    {  // chunks start on multiples of kPrChunkSources, so the slice is 16-byte aligned
        auto contrib = [](float r, uint32_t od) { return od ? r / (float)od : 0.f; };
        const f32x4* r4 = reinterpret_cast<const f32x4*>(rank + T.src_begin);
        const u32x4* o4 = reinterpret_cast<const u32x4*>(outdeg + T.src_begin);
        f32x4* s4 = reinterpret_cast<f32x4*>(s_c);
        const uint32_t n4 = T.src_count / 4;
        for (uint32_t i = threadIdx.x; i < n4; i += kSendThreads) {
            const f32x4 r = r4[i];
            const u32x4 o = o4[i];
            s4[i] = f32x4{contrib(r.x, o.x), contrib(r.y, o.y), contrib(r.z, o.z), contrib(r.w, o.w)};
        }
        for (uint32_t i = 4 * n4 + threadIdx.x; i < T.src_count; i += kSendThreads)
            s_c[i] = contrib(rank[T.src_begin + i], outdeg[T.src_begin + i]);
    }
    __syncthreads();
    for (uint32_t q0 = 0; q0 < nq; q0 += 4 * kSendThreads) {
        u16x4 nxt[4];
        fetch(q0 + 4 * kSendThreads, nxt);  // the next round's offsets fly while this round writes
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t q = q0 + u * kSendThreads + threadIdx.x;
            if (q < nq) out[q] = f32x4{s_c[a[u].x], s_c[a[u].y], s_c[a[u].z], s_c[a[u].w]};
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) a[u] = nxt[u];
    }
}

uint32_t pr_send_tile_slots(const medusa_graph* g, uint32_t nblk) {
    int cus = 0, per_cu = 0;
    MDS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device));
    MDS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k_pr_send),
                                                         (int)kSendThreads, 0));
    const uint64_t slots = (uint64_t)std::max(cus, 0) * (uint64_t)std::max(per_cu, 0);
    const uint64_t dwg = (nblk + kSendWaves - 1) / kSendWaves;
    return slots > dwg ? (uint32_t)std::min<uint64_t>(slots - dwg, 1u << 20) : 0u;
}

constexpr uint32_t kCombineThreads = 512;
constexpr uint32_t kCombineWaves = kCombineThreads / kWave;
constexpr uint32_t kCombineUnroll = 4;  // groups of four entries per thread in flight

// Binned combine (one launch per superstep).  Workgroup b < nbins takes bin xcd_grouped(b):
//   1. zeroes its LDS slots while every wave loads the records of its items (items w, w+8, ...
//      for wave w, one per lane) into registers;
//   2. reads its entries four at a time: a group's message-array position (qmsg, planned on
//      the host; a group never straddles two runs) and its four slots (8 bytes) load together,
//      then its four messages (16 bytes); each message goes to its LDS slot (padding entries to
//      a dummy slot);
//   3. after the barrier, wave w sums its items from LDS in the canonical order: lane items
//      (lane_item_sum; at most 16 slots per lane) and wave vertices, four at a time.  A wave
//      vertex alone spent most of its time in the tree's twelve dependent exchanges, and the bins
//      of the heaviest destinations (about 90 wave vertices, or two 64-vertex lane items) ran
//      long after the others; four trees now share seven merges in vector registers.  Combine
//      of RMAT-16 (141 bins, one round) 18.8 -> 8.8 us, of RMAT-20 29.6 -> 25.1 us (5.3 TB/s).
// Workgroups from nbins on sum the hub destinations (one wave each) by gathering r / outdeg of
// their sources over the CSC, with the same division the send does.  kFold: a single graph with at most 64
// dangling blocks, whose base every wave merges here from the send's block pairs; otherwise
// base[part] was written by k_pr_base.  kContrib: also write r / outdeg (the next superstep
// runs another variant, which reads it).
template <bool kFold, bool kContrib>
__global__ __launch_bounds__(kCombineThreads) void k_pr_combine(
    const PrBin* __restrict__ bins, uint32_t nbins, const PrItem* __restrict__ items,
    const PrItem* __restrict__ hubs, uint32_t nhubs, const uint32_t* __restrict__ qmsg,
    const float* __restrict__ msg, const uint16_t* __restrict__ slot, const uint32_t* __restrict__ cptr,
    const uint32_t* __restrict__ crow, const float* __restrict__ rank_in, const uint32_t* __restrict__ outdeg,
    const float* __restrict__ base_p, const float* __restrict__ partials, uint32_t nblk, uint32_t n, float d,
    float* __restrict__ rank_out, float* __restrict__ contrib_out) {
    __shared__ float lds[kPrBinValues + 4];  // + the dummy slot of padding entries
    using u16x4 = unsigned short __attribute__((ext_vector_type(4)));
    using f32x4 = float __attribute__((ext_vector_type(4)));
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    auto finish = [&](uint32_t p, float S, float base) {
        const float r = fmaf(d, S, base);
        rank_out[p] = r;
        if (kContrib) {
            const uint32_t od = outdeg[p];
            if (od) contrib_out[p] = r / (float)od;
        }
    };
    if (blockIdx.x >= nbins) {
        const uint32_t h = (blockIdx.x - nbins) * kCombineWaves + wave;
        if (h >= nhubs) return;  // uniform across the wave
        const PrItem I = hubs[h];
        const float base = kFold ? pr_base_fold(partials, 0, nblk, n, d) : base_p[I.part];
        const uint32_t b = cptr[I.v], len = cptr[I.v + 1] - b;
        const float S = wave_segment_sum(len, [&](uint32_t k) {
            const uint32_t u = crow[b + k];
            return rank_in[u] / (float)outdeg[u];  // u has an out-edge
        });
        if (lane == 0) finish(I.v, S, base);
        return;
    }
    // neighbouring bins' runs share their end lines in the message array: grouped on one XCD,
    // the second fetch of such a line hits its L2 (RMAT-20: 29 MB less fetched per superstep)
    const PrBin B = bins[xcd_grouped(blockIdx.x, nbins)];
    // 1. this wave's items, one record per lane (a bin has at most 64 items per wave)
    const uint32_t my_item = B.item_begin + wave + kCombineWaves * lane;
    uint32_t iv = 0, icount = 0, ikind = 0, ilds = 0, ipart = 0, ideg = 0;
    if (my_item < B.item_end) {
        const PrItem I = items[my_item];
        iv = I.v;
        icount = I.count;
        ikind = I.kind;
        ilds = I.lds;
        ipart = I.part;
        ideg = I.deg;
    }
    float ps = 0.f, pc = 0.f;  // kFold: this lane's dangling block pair
    if (kFold && lane < nblk) {
        ps = partials[2 * lane];
        pc = partials[2 * lane + 1];
    }
    // 2. entries into their slots: the first round's loads are issued before the slots are
    // zeroed, so they fly during the zeroing and its barrier
    const u16x4* __restrict__ s4 = reinterpret_cast<const u16x4*>(slot + B.slot_begin);
    const uint32_t* __restrict__ g4 = qmsg + B.slot_begin / 4;
    const f32x4* __restrict__ m4 = reinterpret_cast<const f32x4*>(msg);
    const uint32_t nq = B.entries / 4;
    f32x4 x[kCombineUnroll];
    u16x4 t[kCombineUnroll];
    auto fetch = [&](uint32_t q0) {
        uint32_t at[kCombineUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kCombineUnroll; ++u) {
            const uint32_t q = q0 + u * kCombineThreads + threadIdx.x;
            if (q >= nq) continue;
            at[u] = g4[q];
            t[u] = s4[q];
        }
#pragma unroll
        for (uint32_t u = 0; u < kCombineUnroll; ++u)
            if (q0 + u * kCombineThreads + threadIdx.x < nq) x[u] = m4[at[u]];
    };
    auto drop = [&](uint32_t q0) {
#pragma unroll
        for (uint32_t u = 0; u < kCombineUnroll; ++u) {
            if (q0 + u * kCombineThreads + threadIdx.x >= nq) continue;
            lds[t[u].x] = x[u].x;
            lds[t[u].y] = x[u].y;
            lds[t[u].z] = x[u].z;
            lds[t[u].w] = x[u].w;
        }
    };
    fetch(0);
    {
        f32x4* z = reinterpret_cast<f32x4*>(lds);
        for (uint32_t i = threadIdx.x; i < kPrBinValues / 4; i += kCombineThreads) z[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();
    drop(0);
    for (uint32_t q0 = kCombineThreads * kCombineUnroll; q0 < nq; q0 += kCombineThreads * kCombineUnroll) {
        fetch(q0);
        drop(q0);
    }
    __syncthreads();
    // 3. sums
    float base_all = 0.f;
    if (kFold) {
        float as = 0.f, ac = 0.f;
        for (uint32_t j = 0; j < nblk; ++j) {
            const float s2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ps), j));
            const float c2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pc), j));
            if (j == 0) {
                as = s2;
                ac = c2;
            } else {
                kahan_combine(as, ac, s2, c2);
            }
        }
        base_all = pr_base_value(as - ac, d, n);
    }
    const uint32_t mine = B.item_end > B.item_begin + wave
                              ? (B.item_end - B.item_begin - wave + kCombineWaves - 1) / kCombineWaves
                              : 0u;
    for (uint32_t j = 0; j < mine;) {
        const uint32_t kind = __builtin_amdgcn_readlane(ikind, j);
        if (kind == kPrWave) {
            // up to four wave vertices at once: their Kahan chains overlap, and the tree's offsets
            // 32 and 16 merge two and four of them per exchange
            uint32_t at[4], deg[4], v[4], part[4], top = 0, cnt = 0;
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                at[q] = deg[q] = v[q] = part[q] = 0;
                if (cnt == q && j + q < mine && __builtin_amdgcn_readlane(ikind, j + q) == kPrWave) {
                    at[q] = __builtin_amdgcn_readlane(ilds, j + q);
                    deg[q] = __builtin_amdgcn_readlane(ideg, j + q);
                    v[q] = __builtin_amdgcn_readlane(iv, j + q);
                    part[q] = __builtin_amdgcn_readlane(ipart, j + q);
                    top = max(top, deg[q]);
                    ++cnt;
                }
            }
            float s[4] = {0.f, 0.f, 0.f, 0.f}, c[4] = {0.f, 0.f, 0.f, 0.f};
            for (uint32_t k = lane; k - lane < top; k += kWave) {  // uniform across the wave
                float x[4];
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) x[q] = k < deg[q] ? lds[at[q] + k] : 0.f;
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q)
                    if (k < deg[q]) kahan_add(s[q], c[q], x[q]);
            }
            merge32(s[0], c[0], s[1], c[1]);
            merge32(s[2], c[2], s[3], c[3]);
            merge16(s[0], c[0], s[2], c[2]);  // rows: vertices 0, 2, 1, 3
            row_tree(s[0], c[0]);
            const uint32_t row = lane / 16;
            const uint32_t mv = row == 0 ? v[0] : row == 1 ? v[2] : row == 2 ? v[1] : v[3];
            const uint32_t mp = row == 0 ? part[0] : row == 1 ? part[2] : row == 2 ? part[1] : part[3];
            const uint32_t mq = row == 1 ? 2u : row == 2 ? 1u : row;
            if (lane % 16 == 0 && mq < cnt) finish(mv, s[0] - c[0], kFold ? base_all : base_p[mp]);
            j += cnt;
            continue;
        }
        const uint32_t v = __builtin_amdgcn_readlane(iv, j), cnt = __builtin_amdgcn_readlane(icount, j);
        const uint32_t at = __builtin_amdgcn_readlane(ilds, j), deg = __builtin_amdgcn_readlane(ideg, j);
        const float base = kFold ? base_all : base_p[__builtin_amdgcn_readlane(ipart, j)];
        const float S = kind == kPrZero ? 0.f : lane_item_sum(deg, lds + at + lane);
        if (lane < cnt) finish(v + lane, S, base);
        ++j;
    }
}

uint32_t pr_combine_slots(const medusa_graph* g) {
    int cus = 0, per_cu = 0;
    MDS_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, g->device));
    MDS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, reinterpret_cast<const void*>(k_pr_combine<true, false>), (int)kCombineThreads, 0));
    return (uint32_t)std::min<uint64_t>((uint64_t)std::max(cus, 0) * (uint64_t)std::max(per_cu, 0), 1u << 20);
}

// r_0 = (float)(1 / n_g) for every vertex of graph g (graph found by binary search
// over the range starts, which internal ids keep), its contribution when the first superstep
// reads one (contrib not null), and the send's ticket.
__global__ void k_pr_init(uint32_t n, const uint32_t* __restrict__ part_begin, uint32_t nparts,
                          const uint32_t* __restrict__ outdeg, float* __restrict__ rank, float* __restrict__ contrib,
                          uint32_t* __restrict__ ticket) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *ticket = 0;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = nparts;  // last graph with begin <= p
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (part_begin[mid] <= p) lo = mid;
            else hi = mid;
        }
        const float r0 = (float)(1.0 / (double)(part_begin[lo + 1] - part_begin[lo]));
        rank[p] = r0;
        if (!contrib) continue;
        const uint32_t od = outdeg[p];
        if (od) contrib[p] = r0 / (float)od;
    }
}

// Push variant: every out-edge (internal CSR order) writes its source's
// contribution into its destination's in-edge slot.
__global__ void k_pr_scatter(uint32_t n, const uint32_t* __restrict__ optr, const uint32_t* __restrict__ oslot,
                             const float* __restrict__ contrib, float* __restrict__ msg) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    for (uint32_t p = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; p < n; p += waves) {
        const uint32_t b = optr[p], e = optr[p + 1];
        if (b == e) continue;
        const float x = contrib[p];
        if (!lies_before(b, lane, e)) continue;
        for (uint32_t k = b + lane;; k += kWave) {
            msg[oslot[k]] = x;
            if (!lies_before(k, kWave, e)) break;
        }
    }
}

// End of a run: the ranks in original vertex order, and the L1 distance of the last two iterates
// as one FP64 sum per workgroup, which the host adds up in order (512 atomics on one address took
// as long as the rest of the pass).
constexpr uint32_t kFinishWgs = 1024;
__global__ __launch_bounds__(256) void k_pr_finish(uint32_t n, const uint32_t* __restrict__ iperm,
                                                   const float* __restrict__ rank, const float* __restrict__ prev,
                                                   float* __restrict__ out, double* __restrict__ resid) {
    __shared__ double s_part[4];
    double acc = 0.0;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        out[v] = rank[iperm[v]];
        acc += fabs((double)rank[v] - (double)prev[v]);
    }
#pragma unroll
    for (int off = kWave / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) s_part[threadIdx.x / kWave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) resid[blockIdx.x] = s_part[0] + s_part[1] + s_part[2] + s_part[3];
}

// A single graph with at most this many dangling blocks merges its base inside the binned
// combine (every wave merges the block pairs itself) instead of in a launch of its own.
constexpr uint32_t kFoldBlocks = 64;

// In-edges up to which the default variant is the pull, when its superstep is one launch
// (own_base); us per superstep, pull against binned: R-MAT 12 (66 K arcs) 4.7 and 8.0,
// 14 (262 K) 5.2 and 8.3, 15 (524 K) 5.6 and 9.1, 16 (1.05 M) 7.3 and 10.9, 17 (2.1 M) 12.5 and
// 17.7, 18 (4.2 M) 26.7 and 24.4; 14 with 65 K arcs (1781 dangling) 5.9 and 7.9; Chung-Lu, 4200
// vertices (2490 dangling) 6.1 and 7.2.  From here to about 3 M in-edges the pull is still the faster,
// but what decides there (dangling share, in-degree spread) is what the variant policy learns,
// and its measured gain is defined against the fixed binned variant.
constexpr uint64_t kPullDefaultEdges = 1u << 19;

static void pr_run(medusa_graph* g, float damping, uint32_t steps, float* out, const medusa_opts& o,
                   medusa_stats& st) {
    build_pr_layout(g);
    PrLayout& L = *g->pr;
    const uint32_t n = g->n;
    const uint64_t m = g->m;
    const uint32_t nd = L.n_dangling;
    const uint32_t nblk = (uint32_t)L.blocks.size();
    const uint32_t nparts = (uint32_t)L.parts.size();
    MDS_CHECK(o.variant == MEDUSA_PR_DEFAULT || o.variant == MEDUSA_PR_PULL || o.variant == MEDUSA_PR_PUSH ||
                  o.variant == MEDUSA_PR_BINNED,
              MEDUSA_ERR_ARG, "pagerank: unknown variant %d", o.variant);
    // the engine's default: the pull on small graphs, else the binned exchange wherever its layout
    // can be planned
    const bool own_base = L.parts.size() == 1 && nd <= kOwnBaseVertices &&
                          ((nd + 1023) / 1024) * ((L.total_wgs + 2047) / 2048) <= kOwnBaseRounds;
    const int dflt = o.variant != MEDUSA_PR_DEFAULT             ? o.variant
                     : own_base && m <= kPullDefaultEdges       ? MEDUSA_PR_PULL
                     : build_pr_bins(g, /*required=*/false)     ? MEDUSA_PR_BINNED
                                                                : MEDUSA_PR_PULL;
    // kernel variant of every superstep: the caller's, or the learned policy's per superstep
    // (it keeps the caller's unless it predicts a clear gain); the ranks are the same bits
    uint64_t wave_vertices = 0, lane_vertices = 0;
    for (const PrRun& r : L.runs) {
        if (r.kind == kPrWave) wave_vertices += r.count;
        if (r.kind == kPrLane) lane_vertices += r.count;
    }
    Sched sched(o, Sched::kBfs);
    const bool binned_ok = dflt == MEDUSA_PR_BINNED || (o.policy && build_pr_bins(g, /*required=*/false));
    std::vector<uint8_t> var(steps);
    uint64_t sig = 1469598103934665603ull;  // FNV-1a over the sequence, keys the captured graph
    for (uint32_t t = 0; t < steps; ++t) {
        const double rec[MEDUSA_TRACE_FIELDS] = {(double)t, (double)nd, (double)wave_vertices, (double)lane_vertices,
                                                 0.0, (double)n, (double)m, 0.0, 0.0};
        var[t] = (uint8_t)sched.pr_variant(rec, dflt, binned_ok);
        sig = (sig ^ var[t]) * 1099511628211ull;
    }
    const bool push = std::find(var.begin(), var.end(), (uint8_t)MEDUSA_PR_PUSH) != var.end();
    const bool binned = std::find(var.begin(), var.end(), (uint8_t)MEDUSA_PR_BINNED) != var.end();
    if (binned) build_pr_bins(g, /*required=*/true);
    PrBins* Bn = L.bins.get();
    const bool fold = nparts == 1 && nblk <= kFoldBlocks;
    L.rank.ensure(n);
    L.contrib0.ensure(n);
    L.contrib1.ensure(n);
    L.base.ensure(nparts);
    L.partials.ensure(2 * (size_t)std::max(nblk, 1u));
    L.resid.ensure(kFinishWgs);
    L.h_resid.ensure(kFinishWgs);
    L.ticket.ensure(1);
    L.rank_prev.ensure(n);
    if (push) L.msg.ensure(m);
    hipStream_t s = g->stream;
    // an output the kernels can write is written by the last one itself
    const bool direct = kernels_can_write(g, out, (size_t)n * 4);
    if (!direct) L.unperm.ensure(n);
    const bool send_folds = !fold && pr_send_folds(L);

    const float d_f = damping;
    const uint32_t dangle_wgs = (nblk + 3) / 4, base_wgs = (nparts + 3) / 4;
    // base of the next superstep from the ranks in `r`
    auto enqueue_base = [&](const float* r) {
        if (nblk <= kSmallBlocks) {
            hipLaunchKernelGGL(k_pr_dangle_base, dim3(1), dim3(256), 0, s, r, (const PrBlock*)L.d_blocks.p, nblk,
                               (const PrPart*)L.d_parts.p, nparts, d_f, L.base.p);
            MDS_LAUNCHED();
            return;
        }
        if (nblk) {
            hipLaunchKernelGGL(k_pr_dangle, dim3(dangle_wgs), dim3(256), 0, s, r, (const PrBlock*)L.d_blocks.p, nblk,
                               L.partials.p);
            MDS_LAUNCHED();
        }
        hipLaunchKernelGGL(k_pr_base, dim3(base_wgs), dim3(256), 0, s, (const float*)L.partials.p,
                           (const PrPart*)L.d_parts.p, nparts, d_f, L.base.p);
        MDS_LAUNCHED();
    };

    hipLaunchKernelGGL(k_pr_init, dim3(grid_for(n, 256)), dim3(256), 0, s, n, (const uint32_t*)L.d_part_begin.p,
                       nparts, L.outdeg.p, L.rank.p,
                       steps > 0 && var[0] == MEDUSA_PR_BINNED ? nullptr : L.contrib0.p, L.ticket.p);
    MDS_LAUNCHED();

    const bool timing = o.timing != 0 || o.trace != 0;
    // per superstep: [3t] superstep start, [3t+1] main kernel start where launches come before it (an
    // event between two others takes 3 us, half of a small graph's superstep), [3t+2] main kernel end
    if (timing) ensure_events(g, 3 * (size_t)steps);
    g->trace.clear();
    float* rk[2] = {L.rank.p, L.rank_prev.p};
    float* ct[2] = {L.contrib0.p, L.contrib1.p};

    auto launches_before = [&](uint32_t t) {
        return var[t] != MEDUSA_PR_BINNED && (!own_base || var[t] == MEDUSA_PR_PUSH);
    };
    auto enqueue_steps = [&](bool with_events) {
        for (uint32_t t = 0; t < steps; ++t) {
            const float* r_in = rk[t & 1];
            float* r_out = rk[(t + 1) & 1];
            const float* c_in = ct[t & 1];
            float* c_out = ct[(t + 1) & 1];
            const bool step_push = var[t] == MEDUSA_PR_PUSH;
            if (with_events) MDS_HIP(hipEventRecord(g->events[3 * t], s));
            if (var[t] == MEDUSA_PR_BINNED) {
                // send: the contributions of r_t as messages, and the dangling block pairs of r_t;
                // combine: r_{t+1} (and c_{t+1} when the next superstep runs another variant)
                const uint32_t dwg = (nblk + kSendWaves - 1) / kSendWaves;
                if (dwg + Bn->ntiles) {  // none when nothing dangles and every in-edge goes to a hub
                    hipLaunchKernelGGL(k_pr_send, dim3(Bn->ntiles + dwg), dim3(kSendThreads), 0, s,
                                       (const PrTile*)Bn->tiles.p, Bn->ntiles, (const uint16_t*)Bn->srcloc.p, r_in,
                                       (const uint32_t*)L.outdeg.p, Bn->msg.p, (const PrBlock*)L.d_blocks.p, nblk, dwg,
                                       L.partials.p, (const PrPart*)L.d_parts.p, nparts, d_f,
                                       send_folds ? L.base.p : nullptr, L.ticket.p);
                    MDS_LAUNCHED();
                }
                if (!fold && !send_folds) {
                    hipLaunchKernelGGL(k_pr_base, dim3(base_wgs), dim3(256), 0, s, (const float*)L.partials.p,
                                       (const PrPart*)L.d_parts.p, nparts, d_f, L.base.p);
                    MDS_LAUNCHED();
                }
                const bool keep = t + 1 < steps && var[t + 1] != MEDUSA_PR_BINNED;
                const uint32_t cwg = Bn->nbins + (Bn->nhubs + kCombineWaves - 1) / kCombineWaves;
                const PrItem* hubs = Bn->items.p + (Bn->items.n - Bn->nhubs);
                auto kern = fold ? (keep ? k_pr_combine<true, true> : k_pr_combine<true, false>)
                                 : (keep ? k_pr_combine<false, true> : k_pr_combine<false, false>);
                hipLaunchKernelGGL(kern, dim3(cwg), dim3(kCombineThreads), 0, s, (const PrBin*)Bn->bins.p,
                                   Bn->nbins, (const PrItem*)Bn->items.p, hubs, Bn->nhubs,
                                   (const uint32_t*)Bn->qmsg.p, (const float*)Bn->msg.p,
                                   (const uint16_t*)Bn->slot.p, L.cptr.p, L.crow.p, r_in, L.outdeg.p,
                                   (const float*)L.base.p, (const float*)L.partials.p, nblk, n, d_f, r_out, c_out);
                MDS_LAUNCHED();
                if (with_events) MDS_HIP(hipEventRecord(g->events[3 * t + 2], s));
                continue;
            }
            if (!own_base) enqueue_base(r_in);
            if (step_push) {
                hipLaunchKernelGGL(k_pr_scatter, dim3(grid_for(n, 4, 16384)), dim3(256), 0, s, n, L.optr.p,
                                   L.oslot.p, c_in, L.msg.p);
                MDS_LAUNCHED();
            }
            if (with_events && launches_before(t)) MDS_HIP(hipEventRecord(g->events[3 * t + 1], s));
            auto kern = step_push ? (own_base ? k_pr_main<true, true> : k_pr_main<true, false>)
                                  : (own_base ? k_pr_main<false, true> : k_pr_main<false, false>);
            hipLaunchKernelGGL(kern, dim3(L.total_wgs), dim3(256), 0, s, (const PrRun*)L.d_runs.p,
                               (const uint32_t*)L.d_wg_run.p, (const uint32_t*)L.ell.p, L.cptr.p, L.crow.p,
                               step_push ? (const float*)L.msg.p : c_in, L.outdeg.p, (const float*)L.base.p, r_in,
                               nblk ? L.blocks[0] : PrBlock{0, 0}, n, d_f, r_out, c_out);
            MDS_LAUNCHED();
            if (with_events) MDS_HIP(hipEventRecord(g->events[3 * t + 2], s));
        }
    };

    MDS_HIP(hipEventRecord(g->ev_begin, s));
    if (o.use_graph && !timing && steps > 0) {
        // the captured sequence only depends on (steps, variants, damping): buffers are fixed per layout
        if (!L.exec || L.exec_steps != steps || L.exec_sig != sig || L.exec_damping != damping) {
            if (L.exec) (void)hipGraphExecDestroy(L.exec);
            L.exec = nullptr;
            L.exec_sig = 0;
            // capture must not include the event record issued above
            MDS_HIP(hipStreamSynchronize(s));
            hipGraph_t graph = nullptr;
            MDS_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            try {
                enqueue_steps(false);
            } catch (...) {
                hipGraph_t dummy = nullptr;
                (void)hipStreamEndCapture(s, &dummy);
                if (dummy) (void)hipGraphDestroy(dummy);
                throw;
            }
            MDS_HIP(hipStreamEndCapture(s, &graph));
            hipError_t e = hipGraphInstantiate(&L.exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            MDS_HIP(e);
            L.exec_steps = steps;
            L.exec_sig = sig;
            L.exec_damping = damping;
        }
        MDS_HIP(hipGraphLaunch(L.exec, s));
    } else {
        enqueue_steps(timing);
    }
    MDS_HIP(hipEventRecord(g->ev_end, s));
    float* final_rank = rk[steps & 1];
    const float* prev_rank = rk[(steps + 1) & 1];
    // without a superstep there is no previous iterate: the distance to itself is 0
    const uint32_t fin = grid_for(n, 256, kFinishWgs);
    hipLaunchKernelGGL(k_pr_finish, dim3(fin), dim3(256), 0, s, n, L.iperm.p, (const float*)final_rank,
                       steps > 0 ? prev_rank : (const float*)final_rank, direct ? out : L.unperm.p, L.resid.p);
    MDS_LAUNCHED();
    MDS_HIP(hipMemcpyAsync(L.h_resid.p, L.resid.p, fin * sizeof(double), hipMemcpyDeviceToHost, s));
    if (!direct) copy_out(g, out, L.unperm.p, (size_t)n * 4);
    else MDS_HIP(hipStreamSynchronize(s));
    for (uint32_t i = 0; i < fin; ++i) st.residual_l1 += L.h_resid.p[i];
    float ms = 0;
    MDS_HIP(hipEventElapsedTime(&ms, g->ev_begin, g->ev_end));
    st.device_ms = ms;
    // byte model per superstep (pull over CSC): 4(n+1) offsets + 8m (source id and gathered
    // contribution per in-edge) + 16n (rank write, contribution write, out-degree read,
    // dangling read); the push variant reads message slots instead of gathering
    // contributions and adds its scatter
    const uint64_t pull_bytes = 4ull * (n + 1) + 8ull * m + 16ull * n;
    const uint64_t push_bytes = 4ull * m + 8ull * n + 8ull * n + 4ull * (n - nd);
    const uint64_t scatter_bytes = 4ull * (n + 1) + 8ull * m + 4ull * n;
    for (uint32_t t = 0; t < steps; ++t) {
        // the binned variant computes the same superstep as the pull and is costed by the same model
        const bool p = var[t] == MEDUSA_PR_PUSH;
        st.kernel_bytes += p ? push_bytes : pull_bytes;
        st.alg_bytes += (p ? push_bytes + scatter_bytes : pull_bytes) + 4ull * nd;
        if (p) ++st.push_steps;
        else if (var[t] == MEDUSA_PR_PULL) ++st.pull_steps;
        if (timing) {
            float k_ms = 0, s_ms = 0;
            MDS_HIP(hipEventElapsedTime(&k_ms, g->events[3 * t + (launches_before(t) ? 1 : 0)], g->events[3 * t + 2]));
            MDS_HIP(hipEventElapsedTime(&s_ms, g->events[3 * t], g->events[3 * t + 2]));
            st.kernel_ms += k_ms;
            if (o.trace) {
                TraceRec r;
                const double rec[MEDUSA_TRACE_FIELDS] = {(double)t, (double)nd, (double)wave_vertices,
                                                         (double)lane_vertices, 0.0, (double)n, (double)m,
                                                         (double)var[t], (double)s_ms};
                std::copy(rec, rec + MEDUSA_TRACE_FIELDS, r.f);
                g->trace.push_back(r);
            }
        }
    }
    st.kernel_launches = steps;
    st.edges_traversed = (uint64_t)steps * m;
    st.supersteps = steps;
    st.reached = n;
}

}  // namespace medusa

using namespace medusa;

extern "C" int medusa_pagerank(medusa_graph* g, float damping, uint32_t steps, float* rank, const medusa_opts* opts,
                               medusa_stats* stats) {
    return guard([&] {
        const auto lock = enter(g);
        MDS_CHECK(rank, MEDUSA_ERR_ARG, "pagerank: null output");
        MDS_CHECK(damping >= 0.f && damping < 1.f, MEDUSA_ERR_ARG, "pagerank: damping must be in [0,1)");
        medusa_opts o{};
        if (opts) o = *opts;
        medusa_stats st{};
        pr_run(g, damping, steps, rank, o, st);
        if (stats) *stats = st;
    });
}
