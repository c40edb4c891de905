// Tree-vs-tree candidate search: the set the reference's simultaneous DFS emits
// (src/axisalignedboundingboxtree.h:54-95 via src/solidboolean.cpp:94-101),
// i.e. every (a, b) whose FP64 triangle boxes closed-overlap.
//
// Breadth-first over node pairs: each level's kernel reads the frontier written
// by the previous one.  A thread loads the two nodes of its pair (64 B each,
// both child boxes inside), tests the up-to-4 child combinations with the FP32
// outward-rounded boxes (a superset test), and appends the surviving pairs to
// the next frontier.  A pair of leaves met there is rechecked with the exact
// FP64 closed box test on the 96-B FP64 records and becomes a candidate (one
// test per lane; tested where the pair was found, a lane waited for the loads
// of up to four in turn).  Appends take one atomic per wave or workgroup and
// queue, offsets from ballots.  Queues past capacity raise `overflow`; the
// host grows them and repeats the search, so nothing is ever dropped.
#include "sbg_device.h"
#include "sbg_internal.h"

#pragma clang fp contract(off)

namespace sbg {

struct FBox {
    float lx, ly, lz, hx, hy, hz;
};

__device__ __forceinline__ bool fbox_overlap(const FBox &a, const FBox &b)
{
    return a.lx <= b.hx && a.hx >= b.lx && a.ly <= b.hy && a.hy >= b.ly && a.lz <= b.hz && a.hz >= b.lz;
}

__device__ __forceinline__ FBox leaf_box(const float *__restrict__ box32, uint32_t tri)
{
    const float4 *p = reinterpret_cast<const float4 *>(box32 + (size_t)kBox32Stride * tri);
    const float4 lo = p[0], hi = p[1];
    return {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
}

__device__ __forceinline__ Box64 record_box(const double *__restrict__ tri64, uint32_t t)
{
    const double2 *p = reinterpret_cast<const double2 *>(tri64 + (size_t)kTri64Stride * t);
    const double2 r0 = p[0], r1 = p[1], r2 = p[2], r3 = p[3], r4 = p[4], r5 = p[5];
    return tri_box64({r0.x, r0.y, r1.x}, {r2.x, r2.y, r3.x}, {r4.x, r4.y, r5.x});
}

// Children of a node reference: one (a leaf) or two, with their FP32 boxes.
struct Kids {
    uint32_t c0, c1;
    FBox b0, b1;
    bool two;
};

__device__ __forceinline__ Kids kids_of(const BNode *__restrict__ nodes, const float *__restrict__ box32, uint32_t ref)
{
    Kids k;
    if (ref & kLeafBit) {
        k.c0 = k.c1 = ref;
        k.b0 = k.b1 = leaf_box(box32, ref & ~kLeafBit);
        k.two = false;
        return k;
    }
    const BNode *nd = nodes + ref;
    const float4 a = nd->a, b = nd->b, cc = nd->c;
    const int4 d = nd->d;
    k.c0 = (uint32_t)d.x;
    k.c1 = (uint32_t)d.y;
    k.b0 = {a.x, a.y, a.z, a.w, b.x, b.y};
    k.b1 = {b.z, b.w, cc.x, cc.y, cc.z, cc.w};
    k.two = true;
    return k;
}

__device__ __forceinline__ bool both_leaves(uint2 pr) { return (pr.x & pr.y & kLeafBit) != 0u; }

// whether a pair of leaves is a candidate: the exact FP64 closed box test
__device__ __forceinline__ bool leaves_overlap(const TraverseArgs &t, uint2 pr)
{
    return box64_overlap(record_box(t.tri64A, pr.x & ~kLeafBit), record_box(t.tri64B, pr.y & ~kLeafBit));
}

__device__ __forceinline__ uint64_t cand_key(uint2 pr)
{
    return ((uint64_t)(pr.x & ~kLeafBit) << 32) | (pr.y & ~kLeafBit);
}

// Expansion of one node pair: child pair s = 2u + v (u over A's children, v
// over B's) goes on when its FP32 boxes overlap (bit s of next).  A pair of
// leaves has no children: cand says whether it is a candidate.  Every field is
// a named register, so nothing lands in scratch memory.
struct Expansion {
    uint32_t a0, a1, b0, b1;
    uint32_t next;
    bool cand;
};

__device__ __forceinline__ void expand_nodes(const TraverseArgs &t, uint2 pr, Expansion &x)
{
    const Kids ka = kids_of(t.nodesA, t.boxA, pr.x);
    const Kids kb = kids_of(t.nodesB, t.boxB, pr.y);
    x.a0 = ka.c0;
    x.a1 = ka.c1;
    x.b0 = kb.c0;
    x.b1 = kb.c1;
    x.next = (fbox_overlap(ka.b0, kb.b0) ? 1u : 0u) | (kb.two && fbox_overlap(ka.b0, kb.b1) ? 2u : 0u) |
             (ka.two && fbox_overlap(ka.b1, kb.b0) ? 4u : 0u) |
             (ka.two && kb.two && fbox_overlap(ka.b1, kb.b1) ? 8u : 0u);
}

__device__ __forceinline__ Expansion expand_pair(const TraverseArgs &t, uint2 pr, bool valid)
{
    Expansion x = {0, 0, 0, 0, 0, false};
    if (!valid)
        return x;
    if (both_leaves(pr))
        x.cand = leaves_overlap(t, pr);
    else
        expand_nodes(t, pr, x);
    return x;
}

// child pair of slot s (a compile-time constant at every use)
__device__ __forceinline__ uint2 slot_pair(const Expansion &x, int s)
{
    return make_uint2(s < 2 ? x.a0 : x.a1, (s & 1) ? x.b1 : x.b0);
}

// The wave's child pairs in slot order, lane by lane within a slot: one ballot
// per slot (counts by shuffled prefix sums took six dependent LDS permutes).
struct SlotMasks {
    unsigned long long m[4];
    __device__ __forceinline__ uint32_t total() const
    {
        return (uint32_t)(__popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]) + __popcll(m[3]));
    }
};

__device__ __forceinline__ SlotMasks slot_masks(uint32_t next)
{
    return {{__ballot(next & 1u), __ballot(next & 2u), __ballot(next & 4u), __ballot(next & 8u)}};
}

__device__ __forceinline__ unsigned long long lanes_below()
{
    return (1ull << (threadIdx.x & 63)) - 1ull;
}

// writes the wave's child pairs of `next` to out[base ...), those below cap
__device__ __forceinline__ void put_slots(const Expansion &x, uint32_t next, const SlotMasks &sm, uint2 *out,
                                          uint32_t base, uint32_t cap)
{
    const unsigned long long below = lanes_below();
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) {
        const uint32_t pos = base + (uint32_t)__popcll(sm.m[sl] & below);
        if ((next >> sl & 1u) && pos < cap)
            out[pos] = slot_pair(x, sl);
        base += (uint32_t)__popcll(sm.m[sl]);
    }
}

// first of `total` slots of a queue, taken by one lane of the wave (every lane
// gets it); past the capacity the overflow flag is raised
__device__ __forceinline__ uint32_t wave_take(uint32_t total, uint32_t *counter, uint32_t cap, uint32_t *overflow)
{
    uint32_t base = 0;
    if ((threadIdx.x & 63) == 0 && total) {
        base = atomicAdd(counter, total);
        if (base + total > cap)
            atomicOr(overflow, 1u);
    }
    return __shfl(base, 0, 64);
}

// Workgroup size of the grid-wide breadth-first levels (the launches' grids
// are given in units of 256 lanes).
constexpr int kExpandThreads = 256;
constexpr int kExpandWaves = kExpandThreads / 64;

// One breadth-first level over the whole grid: frontier `in` (inCount pairs)
// to `out`, candidates appended.  Workgroups of kExpandThreads lanes, which
// take one atomic per queue.
__device__ __forceinline__ void expand_level(const TraverseArgs &t, const uint2 *__restrict__ in,
                                             const uint32_t *__restrict__ inCount, uint2 *__restrict__ out,
                                             uint32_t *outCount, uint32_t outCap, uint64_t *__restrict__ cand,
                                             uint32_t *candCount, uint32_t candCap, uint32_t *overflow)
{
    __shared__ uint32_t s_count[2][kExpandWaves], s_at[2][kExpandWaves];  // next pairs, candidates
    const int wave = threadIdx.x >> 6;
    // both frontier buffers hold outCap pairs; a count past it has already
    // raised `overflow` and the whole search is repeated with larger queues
    const uint32_t n = *inCount < outCap ? *inCount : outCap;
    const uint32_t stride = gridDim.x * kExpandThreads;
    for (uint32_t base = blockIdx.x * kExpandThreads; base < n; base += stride) {  // uniform over the workgroup
        const uint32_t i = base + threadIdx.x;
        const bool valid = i < n;
        const uint2 pr = valid ? in[i] : make_uint2(0, 0);
        const Expansion x = expand_pair(t, pr, valid);
        const SlotMasks sm = slot_masks(x.next);
        const unsigned long long cm = __ballot(x.cand);
        if ((threadIdx.x & 63) == 0) {
            s_count[0][wave] = sm.total();
            s_count[1][wave] = (uint32_t)__popcll(cm);
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            const uint32_t *cnt = s_count[threadIdx.x];
            uint32_t total = 0;
            for (int w = 0; w < kExpandWaves; ++w)
                total += cnt[w];
            uint32_t at = total ? atomicAdd(threadIdx.x ? candCount : outCount, total) : 0u;
            if (total && at + total > (threadIdx.x ? candCap : outCap))
                atomicOr(overflow, 1u);
            for (int w = 0; w < kExpandWaves; ++w) {
                s_at[threadIdx.x][w] = at;
                at += cnt[w];
            }
        }
        __syncthreads();
        const uint32_t on = s_at[0][wave];
        uint32_t oc = s_at[1][wave];
        put_slots(x, x.next, sm, out, on, outCap);
        oc += (uint32_t)__popcll(cm & lanes_below());
        if (x.cand && oc < candCap)
            cand[oc] = cand_key(pr);
    }
}

__global__ __launch_bounds__(kExpandThreads) void k_expand(TraverseArgs t, const uint2 *__restrict__ in,
                                                const uint32_t *__restrict__ inCount, uint2 *__restrict__ out,
                                                uint32_t *outCount, uint32_t outCap, uint64_t *__restrict__ cand,
                                                uint32_t *candCount, uint32_t candCap, uint32_t *overflow)
{
    expand_level(t, in, inCount, out, outCount, outCap, cand, candCount, candCap, overflow);
}

// ---- first frontier from the trees' tiles --------------------------------------
// The levels from two roots down to subtrees of a tile's size hold few pairs
// and cost a launch or a workgroup's round each.  Instead every pair of tiles
// is tested by its boxes at once (1,280 x 1,280 at the 1,310,720-triangle
// pair), one workgroup per tile of A and 256 tiles of B, and the pieces of the
// tiles that overlap give the frontier, some tens of tests per pair of tiles.
// A pass from the roots took 730 us against 637 at the 81,920-triangle pair,
// 973 against 879 at two 393,132-triangle cubes, 1,706 against 1,681 at
// 1,310,720 triangles.
constexpr int kSearchOut = 1024;  // frontier pairs a workgroup gathers before it takes slots

__global__ __launch_bounds__(256) void k_search_tiles(TileSet a, TileSet b, uint2 *__restrict__ frontier,
                                                      uint32_t *count, uint32_t cap, uint32_t *overflow)
{
    __shared__ uint32_t s_tile[256], s_ntile, s_nout, s_base;
    __shared__ float4 s_piece[2 * kTilePieces];
    __shared__ uint2 s_out[kSearchOut];
    const uint32_t ta = blockIdx.x, tb0 = blockIdx.y * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0)
        s_ntile = s_nout = 0;
    __syncthreads();
    if (tb0 < b.ntiles) {
        const float *p = a.box + 6 * (size_t)ta, *q = b.box + 6 * (size_t)tb0;
        if (fbox_overlap({p[0], p[1], p[2], p[3], p[4], p[5]}, {q[0], q[1], q[2], q[3], q[4], q[5]}))
            s_tile[atomicAdd(&s_ntile, 1u)] = tb0;
    }
    __syncthreads();
    const uint32_t ntile = s_ntile;
    if (ntile == 0)
        return;
    const uint32_t na = a.pieces.count[ta];
    for (uint32_t k = threadIdx.x; k < 2 * na; k += 256)
        s_piece[k] = a.pieces.piece[2 * (size_t)ta * kTilePieces + k];
    __syncthreads();
    for (uint32_t k = wave; k < ntile; k += 4) {
        const uint32_t tb = s_tile[k], nb = b.pieces.count[tb];
        const float4 *pb = b.pieces.piece + 2 * (size_t)tb * kTilePieces;
        for (uint32_t j0 = 0; j0 < na * nb; j0 += 64) {
            const uint32_t j = j0 + lane, ia = j / nb, ib = j - ia * nb;
            bool hit = false;
            uint2 pr = make_uint2(0, 0);
            if (ia < na) {
                const float4 al = s_piece[2 * ia], ah = s_piece[2 * ia + 1], bl = pb[2 * ib], bh = pb[2 * ib + 1];
                hit = fbox_overlap({al.x, al.y, al.z, ah.x, ah.y, ah.z}, {bl.x, bl.y, bl.z, bh.x, bh.y, bh.z});
                pr = make_uint2(__float_as_uint(al.w), __float_as_uint(bl.w));
            }
            const unsigned long long m = __ballot(hit);
            if (!m)
                continue;
            uint32_t at = 0;
            if (lane == 0)
                at = atomicAdd(&s_nout, (uint32_t)__popcll(m));
            at = __shfl(at, 0, 64) + (uint32_t)__popcll(m & lanes_below());
            if (hit && at < (uint32_t)kSearchOut) {
                s_out[at] = pr;
            } else if (hit) {  // more than a workgroup gathers: a slot of its own
                const uint32_t slot = atomicAdd(count, 1u);
                if (slot < cap)
                    frontier[slot] = pr;
                else
                    atomicOr(overflow, 1u);
            }
        }
    }
    __syncthreads();
    const uint32_t n = s_nout < (uint32_t)kSearchOut ? s_nout : (uint32_t)kSearchOut;
    if (threadIdx.x == 0 && n) {
        s_base = atomicAdd(count, n);
        if (s_base + n > cap)
            atomicOr(overflow, 1u);
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < n; k += 256)
        if (s_base + k < cap)
            frontier[s_base + k] = s_out[k];
}

void launch_search_tiles(const TileSet &a, const TileSet &b, uint2 *frontier, uint32_t *count, uint32_t cap,
                         uint32_t *overflow, hipStream_t s)
{
    hipLaunchKernelGGL(k_search_tiles, dim3(a.ntiles, (b.ntiles + 255) / 256), dim3(256), 0, s, a, b, frontier, count,
                       cap, overflow);
}

// ---- top of the search in one workgroup -------------------------------------
// The first levels of a tree-vs-tree search hold a handful of node pairs, and a
// grid-wide launch per level costs a launch's latency for a few lanes of work
// (and waits for free slots behind any kernel that fills the chip).  One
// workgroup of 1024 lanes expands level after level instead, frontier in the
// two global frontier buffers, next-frontier slots handed out from LDS, until
// a level holds more than topMax pairs, the level cap is reached or the
// frontier empties.  cnt[l] gets every level's size as the grid-wide kernel
// would leave it; *levelOut gets the first level not expanded here.
__global__ __launch_bounds__(1024) void k_search_top(TraverseArgs t, uint2 *__restrict__ front0,
                                                     uint2 *__restrict__ front1, uint32_t *__restrict__ cnt,
                                                     uint32_t fcap, uint64_t *__restrict__ cand, uint32_t *candCount,
                                                     uint32_t candCap, uint32_t *overflow, int maxLevels,
                                                     uint32_t topMax, uint32_t *levelOut)
{
    __shared__ uint32_t s_next;
    const int lane = threadIdx.x & 63;
    uint32_t nIn = cnt[0];
    int level = 0;
    while (level < maxLevels && nIn > 0 && nIn <= topMax) {
        const uint2 *in = (level & 1) ? front1 : front0;
        uint2 *out = (level & 1) ? front0 : front1;
        if (threadIdx.x == 0)
            s_next = 0;
        __syncthreads();
        for (uint32_t b = 0; b < nIn; b += 1024) {
            const uint32_t i = b + threadIdx.x;
            const bool valid = i < nIn;
            const uint2 pr = valid ? in[i] : make_uint2(0, 0);
            const Expansion x = expand_pair(t, pr, valid);
            // next-frontier slots: one LDS atomic per wave
            const SlotMasks sm = slot_masks(x.next);
            const uint32_t total = sm.total();
            uint32_t on = 0;
            if (lane == 0 && total)
                on = atomicAdd(&s_next, total);
            on = __shfl(on, 0, 64);
            if (total && on + total > fcap && lane == 0)
                atomicOr(overflow, 1u);
            put_slots(x, x.next, sm, out, on, fcap);
            const unsigned long long cm = __ballot(x.cand);
            if (cm) {
                const uint32_t oc = wave_take((uint32_t)__popcll(cm), candCount, candCap, overflow) +
                                    (uint32_t)__popcll(cm & lanes_below());
                if (x.cand && oc < candCap)
                    cand[oc] = cand_key(pr);
            }
        }
        // the next level reads this one's output: workgroup-scope ordering of
        // the global frontier writes, and the count from LDS
        __syncthreads();
        nIn = s_next;
        if (threadIdx.x == 0)
            cnt[level + 1] = nIn;
        ++level;
        __syncthreads();
    }
    if (threadIdx.x == 0)
        *levelOut = (uint32_t)level;
}

// Persistent depth-first stage.  One wave per workgroup keeps a stack of node
// pairs in LDS (spilling to a per-wave region of global memory when full).
// Each step pops up to 64 pairs (one per lane), expands them and pushes the
// surviving child pairs back.  Pairs of leaves are set aside in LDS until 64 of
// them fill a wave for the exact test, so a step waits for two 64-B node loads
// and nothing else; candidates are set aside too and leave 64 or more at a time
// with one atomic (47 us at the 1,310,720-triangle pair, 100 with the tests and
// the atomic inside the step).  An empty wave claims
// the next few seed pairs (the breadth-first frontier) from a shared counter.
// Waves never wait for each other: a wave leaves when its own lists are empty
// and no seed is left.  Spill overflow or the iteration cap raise `overflow`
// (the host then repeats the search breadth-first), so nothing is dropped
// silently.
constexpr int kDfsLds = 1024;
constexpr int kDfsLeaves = 64 + 4 * 64;  // one step adds at most 256 to fewer than 64
constexpr int kDfsCands = 128;           // one test adds at most 64 to fewer than 64
constexpr uint32_t kDfsMaxIter = 1u << 24;

// With levelBase, the seeds are the frontier of level *levelBase: `seeds` /
// `seedsAlt` are the even / odd levels' frontier buffers and seedCount the
// per-level counts.
__global__ __launch_bounds__(64) void k_traverse_dfs(TraverseArgs t, const uint2 *__restrict__ seeds,
                                                     const uint2 *__restrict__ seedsAlt,
                                                     const uint32_t *__restrict__ seedCount, uint32_t seedCap,
                                                     const uint32_t *__restrict__ levelBase, uint32_t *head,
                                                     uint2 *__restrict__ spill,
                                                     uint32_t spillPerWave, uint64_t *__restrict__ cand,
                                                     uint32_t *candCount, uint32_t candCap, uint32_t *overflow)
{
    __shared__ uint2 s_stack[kDfsLds], s_leaf[kDfsLeaves];
    __shared__ uint64_t s_cand[kDfsCands];
    const int lane = threadIdx.x;
    if (levelBase) {
        const uint32_t level = *levelBase;
        seeds = (level & 1) ? seedsAlt : seeds;
        seedCount += level;
    }
    const uint32_t nseed = *seedCount < seedCap ? *seedCount : seedCap;
    // seeds per claim: enough for every wave to start busy, at most one per lane
    uint32_t grab = nseed / gridDim.x;
    grab = grab < 1u ? 1u : (grab > 64u ? 64u : grab);
    uint2 *gstack = spill + (size_t)blockIdx.x * spillPerWave;
    int sp = 0;          // LDS entries (same value in every lane, as the rest)
    uint32_t gsp = 0;    // spilled entries
    uint32_t nleaf = 0, ncand = 0;
    bool seeds_left = true;
    const unsigned long long below = lanes_below();
    auto flush = [&]() {
        const uint32_t base = wave_take(ncand, candCount, candCap, overflow);
        for (uint32_t k = lane; k < ncand; k += 64)
            if (base + k < candCap)
                cand[base + k] = s_cand[k];
        ncand = 0;
        __syncthreads();
    };
    auto test_leaves = [&]() {  // up to 64 of them
        const uint32_t m = nleaf < 64u ? nleaf : 64u;
        nleaf -= m;
        bool hit = false;
        uint2 pr = make_uint2(0, 0);
        if ((uint32_t)lane < m) {
            pr = s_leaf[nleaf + lane];
            hit = leaves_overlap(t, pr);
        }
        const unsigned long long hm = __ballot(hit);
        if (hit)
            s_cand[ncand + (uint32_t)__popcll(hm & below)] = cand_key(pr);
        ncand += (uint32_t)__popcll(hm);
        __syncthreads();
        if (ncand >= 64u)
            flush();
    };
    uint32_t iter = 0;
    for (; iter < kDfsMaxIter; ++iter) {
        if (nleaf >= 64u) {
            test_leaves();
            continue;
        }
        if (sp == 0 && gsp > 0) {
            const uint32_t m = gsp < (uint32_t)(kDfsLds / 2) ? gsp : (uint32_t)(kDfsLds / 2);
            for (uint32_t k = lane; k < m; k += 64)
                s_stack[k] = gstack[gsp - m + k];
            gsp -= m;
            sp = (int)m;
            __syncthreads();
        }
        if (sp == 0 && seeds_left) {
            uint32_t start = 0;
            if (lane == 0)
                start = atomicAdd(head, grab);
            start = __shfl(start, 0, 64);
            seeds_left = start < nseed;
            if (seeds_left) {
                const uint32_t m = nseed - start < grab ? nseed - start : grab;
                if ((uint32_t)lane < m)
                    s_stack[lane] = seeds[start + lane];
                sp = (int)m;
                __syncthreads();
            }
        }
        if (sp == 0) {
            if (nleaf == 0)
                break;
            test_leaves();
            continue;
        }
        const int take = sp < 64 ? sp : 64;
        const bool valid = lane < take;
        uint2 pr = make_uint2(0, 0);
        if (valid)
            pr = s_stack[sp - take + lane];
        sp -= take;
        __syncthreads();
        Expansion x = {0, 0, 0, 0, 0, false};
        if (valid) {
            if (both_leaves(pr)) {  // a seed of two leaves: on to the tests
                x.a0 = pr.x;
                x.b0 = pr.y;
                x.next = 1u;
            } else {
                expand_nodes(t, pr, x);
            }
        }
        // pairs of leaves apart from the others
        const uint32_t la0 = x.a0 >> 31, la1 = x.a1 >> 31, lb0 = x.b0 >> 31, lb1 = x.b1 >> 31;
        const uint32_t leaves = x.next & (la0 & lb0 | (la0 & lb1) << 1 | (la1 & lb0) << 2 | (la1 & lb1) << 3);
        const uint32_t inner = x.next & ~leaves;
        const SlotMasks lm = slot_masks(leaves);
        put_slots(x, leaves, lm, s_leaf, nleaf, (uint32_t)kDfsLeaves);
        nleaf += lm.total();
        // push the others: LDS when they fit, else the wave's spill region
        const SlotMasks im = slot_masks(inner);
        const uint32_t total = im.total();
        if (sp + (int)total <= kDfsLds) {
            put_slots(x, inner, im, s_stack, (uint32_t)sp, (uint32_t)kDfsLds);
            sp += (int)total;
        } else if (gsp + total <= spillPerWave) {
            put_slots(x, inner, im, gstack, gsp, spillPerWave);
            gsp += total;
        } else {
            if (lane == 0)
                atomicOr(overflow, 4u);
            break;
        }
        __syncthreads();
    }
    if (ncand)
        flush();
    if (iter == kDfsMaxIter && lane == 0)
        atomicOr(overflow, 8u);
}

void launch_traverse_dfs(const TraverseArgs &t, const uint2 *seeds, const uint32_t *seedCount, uint32_t seedCap,
                         uint32_t *head, uint2 *spill, uint32_t spillPerWave, int waves, uint64_t *cand,
                         uint32_t *candCount, uint32_t candCap, uint32_t *overflow, hipStream_t s)
{
    hipLaunchKernelGGL(k_traverse_dfs, dim3(waves), dim3(64), 0, s, t, seeds, seeds, seedCount, seedCap,
                       (const uint32_t *)nullptr, head, spill, spillPerWave, cand, candCount, candCap, overflow);
}

// The single-pair search after its first frontier: the one-workgroup levels,
// then the depth-first stage from the level reached.  Up to 8 grid-wide levels
// between the two cost a launch and a grid's start each and no longer pay now
// that the depth-first steps are short: 734 us a pass with 8, 714 with 4, 637
// with none at the 81,920-triangle pair, 1,700 / 1,683 / 1,681 at 1,310,720.
// levelWord: one u32 of scratch.
void launch_search_levels(const TraverseArgs &t, uint2 *front0, uint2 *front1, uint32_t *cnt, uint32_t fcap,
                          uint32_t topMax, int lastLevel, uint32_t *levelWord, uint32_t *head, uint2 *spill,
                          uint32_t spillPerWave, int waves, uint64_t *cand, uint32_t *candCount, uint32_t candCap,
                          uint32_t *overflow, hipStream_t s)
{
    hipLaunchKernelGGL(k_search_top, dim3(1), dim3(1024), 0, s, t, front0, front1, cnt, fcap, cand, candCount,
                       candCap, overflow, lastLevel, topMax, levelWord);
    hipLaunchKernelGGL(k_traverse_dfs, dim3(waves), dim3(64), 0, s, t, (const uint2 *)front0, (const uint2 *)front1,
                       (const uint32_t *)cnt, fcap, (const uint32_t *)levelWord, head, spill, spillPerWave, cand,
                       candCount, candCap, overflow);
}

// root pair: both meshes non-empty; a root may itself be a leaf (1 triangle)
__global__ void k_seed(TraverseArgs t, uint32_t rootA, uint32_t rootB, const float *__restrict__ rootBoxA,
                       const float *__restrict__ rootBoxB, uint2 *frontier, uint32_t *count, uint64_t *cand,
                       uint32_t *candCount)
{
    if (threadIdx.x != 0)
        return;
    FBox a = {rootBoxA[0], rootBoxA[1], rootBoxA[2], rootBoxA[3], rootBoxA[4], rootBoxA[5]};
    FBox b = {rootBoxB[0], rootBoxB[1], rootBoxB[2], rootBoxB[3], rootBoxB[4], rootBoxB[5]};
    if (!fbox_overlap(a, b))
        return;
    if ((rootA & kLeafBit) && (rootB & kLeafBit)) {
        const uint32_t ta = rootA & ~kLeafBit, tb = rootB & ~kLeafBit;
        if (box64_overlap(record_box(t.tri64A, ta), record_box(t.tri64B, tb))) {
            cand[0] = ((uint64_t)ta << 32) | tb;
            *candCount = 1;
        }
        return;
    }
    frontier[0] = make_uint2(rootA, rootB);
    *count = 1;
}

void launch_expand(const TraverseArgs &t, const uint2 *in, const uint32_t *inCount, uint2 *out,
                   uint32_t *outCount, uint32_t outCap, uint64_t *cand, uint32_t *candCount,
                   uint32_t candCap, uint32_t *overflow, int grid, hipStream_t s)
{
    hipLaunchKernelGGL(k_expand, dim3(grid * 256 / kExpandThreads), dim3(kExpandThreads), 0, s, t, in, inCount,
                       out, outCount, outCap, cand, candCount, candCap, overflow);
}

void launch_seed(const TraverseArgs &t, uint32_t rootA, uint32_t rootB, const float *rootBoxA,
                 const float *rootBoxB, uint2 *frontier, uint32_t *count, uint64_t *cand,
                 uint32_t *candCount, hipStream_t s)
{
    hipLaunchKernelGGL(k_seed, dim3(1), dim3(64), 0, s, t, rootA, rootB, rootBoxA, rootBoxB, frontier, count,
                       cand, candCount);
}

}  // namespace sbg
