// Linear BVH over Morton-sorted triangles (Karras, "Maximizing Parallelism in
// the Construction of BVHs, Octrees, and k-d Trees", HPG 2012), replacing the
// reference's recursive top-down tree (src/axisalignedboundingboxtree.cpp:27-141).
// The pair set found against it is the same: every node box contains its
// members' boxes in both trees, and leaf pairs are rechecked with the exact FP64
// closed test (src/axisalignedboundingboxtree.h:62-67).
//
// Node i (0 <= i < n-1) is internal; node 0 is the root.  Leaves are referenced
// as kLeafBit | triangle, so traversal never needs a leaf -> triangle lookup.
// Each child's FP32 box is stored inside its parent, so one 64-B node load
// yields both child boxes.
#include "sbg_internal.h"

namespace sbg {

// common-prefix length of sorted keys i and j, ties broken by index
__device__ __forceinline__ int delta(const uint32_t *__restrict__ codes, int n, int i, int j)
{
    if (j < 0 || j >= n)
        return -1;
    const uint32_t a = codes[i], b = codes[j];
    if (a == b)
        return 32 + __clz((uint32_t)(i ^ j));
    return __clz(a ^ b);
}

// 64-bit keys (mesh id above the Morton code, for the combined tree of a batch)
__device__ __forceinline__ int delta(const uint64_t *__restrict__ codes, int n, int i, int j)
{
    if (j < 0 || j >= n)
        return -1;
    const uint64_t a = codes[i], b = codes[j];
    if (a == b)
        return 64 + __clz((uint32_t)(i ^ j));
    return __clzll(a ^ b);
}

// The tree is built and refit bottom-up in tiles of kTreeTile sorted leaves, one
// workgroup each; a node whose leaf range crosses a tile boundary is a "top"
// node, made by k_top_nodes.
constexpr uint16_t kNoSplit = 0xffffu;

__device__ __forceinline__ void write_root(float *rootBox, float4 lo, float4 hi)
{
    rootBox[0] = lo.x;
    rootBox[1] = lo.y;
    rootBox[2] = lo.z;
    rootBox[3] = hi.x;
    rootBox[4] = hi.y;
    rootBox[5] = hi.z;
}

__device__ __forceinline__ void put6(float *dst, const float v[6])
{
#pragma unroll
    for (int k = 0; k < 6; ++k)
        dst[k] = v[k];
}

// one more piece of the workgroup's tile in the list for the pair search
__device__ __forceinline__ void list_piece(const TreePieces &out, uint32_t *n, uint32_t ref, const float b[6])
{
    if (!out.count)
        return;
    const uint32_t k = atomicAdd(n, 1u);
    float4 *dst = out.piece + 2 * ((size_t)blockIdx.x * kTilePieces + k);
    dst[0] = make_float4(b[0], b[1], b[2], __uint_as_float(ref));
    dst[1] = make_float4(b[3], b[4], b[5], 0.0f);
}

// Stage 1: the radix tree of a tile's leaves, bottom-up.  The tree is fixed by
// the common-prefix lengths of neighbouring keys alone: the parent of a node
// over leaves [lo, hi] splits at hi or at lo - 1, whichever neighbour shares
// the longer prefix (Apetrei, "Fast and Simple Agglomerative LBVH
// Construction", 2014), so a walk from every leaf needs no search in the keys.
// At a split inside the tile the first child to arrive leaves its box,
// reference and far end in LDS and stops, the second merges and goes on.  All
// hand-offs stay inside the workgroup, so no lane waits and no device-wide
// fence is needed.  Karras' numbering is kept: a node that is its parent's left
// child is node hi, a right child node lo, the root node 0, so a node inside
// the tile has its index inside the tile too.
//
// A split that only one child reached belongs to a top node; that child (a
// "piece" of the tile, like one whose parent splits on the tile's border) goes
// to piece[lo] as a box, and the union of the tile's leaves from lo on (suffix)
// and up to hi (prefix) is kept for the top nodes that start or end there.  Box
// unions are exact (min / max), so stage 2 can assemble any top node's box
// from these in any order.  Indices inside the tile that no node took are top
// nodes; they are listed.
//
// Bound by the latency of the walk's LDS steps (and the 64-B node stores).  In
// the pair step at 1,310,720 leaves (another mesh's kernels beside) it takes
// 114 us and the top nodes 35; searching every node's range and split in the
// global keys (about 60 dependent loads each) took 116 us before a refit of
// 119 + 15.  The batch's 3.0 M leaves: 176 + 37 us, before 188 + 162 + 8.
template <typename K>
__global__ __launch_bounds__(kTreeTile) void k_tree_tiles(const K *__restrict__ codes,
                                                          const uint32_t *__restrict__ ids,
                                                          const float *__restrict__ box32, int n,
                                                          BNode *__restrict__ nodes, uint32_t *__restrict__ topList,
                                                          uint32_t *topCount, float *__restrict__ prefix,
                                                          float *__restrict__ suffix, float *__restrict__ piece,
                                                          float *__restrict__ tileBox, TreePieces out, float *rootBox)
{
    __shared__ float s_box[kTreeTile][2][6];        // per split: the children's boxes,
    __shared__ uint32_t s_ref[kTreeTile][2];        // references,
    __shared__ uint16_t s_far[kTreeTile][2];        // far ends (offset in the tile)
    __shared__ uint16_t s_child[kTreeTile][2];      // and own splits (kNoSplit: a leaf)
    __shared__ uint32_t s_flag[kTreeTile];          // arrivals: 1, + kRightCame for a right child
    __shared__ uint16_t s_idx[kTreeTile], s_end[kTreeTile];  // per split: its node's index and other end
    __shared__ uint16_t s_parent[kTreeTile];        // and its parent's index (kNoSplit: none in the tile)
    __shared__ int8_t s_delta[kTreeTile + 1];       // prefix length of (pos - 1, pos)
    __shared__ uint8_t s_taken[kTreeTile], s_start[kTreeTile], s_stop[kTreeTile];
    __shared__ float s_wave[kTreeTile / 64][6];
    __shared__ uint32_t s_ntop, s_top0, s_npiece;
    constexpr uint32_t kRightCame = 0x100u;
    const int tile0 = blockIdx.x * kTreeTile;
    const int tile1 = min(tile0 + kTreeTile, n);
    const int me = threadIdx.x, pos = tile0 + me;
    const bool valid = pos < tile1;
    if (me == 0)
        s_ntop = s_npiece = 0;
    s_flag[me] = 0;
    s_taken[me] = s_start[me] = s_stop[me] = 0;
    if (valid)
        s_delta[me] = (int8_t)delta(codes, n, pos, pos - 1);
    if (pos == tile1 - 1)
        s_delta[me + 1] = (int8_t)delta(codes, n, pos, pos + 1);
    __syncthreads();
    float4 lo4 = make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.0f);
    float4 hi4 = make_float4(-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), 0.0f);
    if (valid) {
        const uint32_t tri = ids[pos];
        lo4 = reinterpret_cast<const float4 *>(box32 + (size_t)kBox32Stride * tri)[0];
        hi4 = reinterpret_cast<const float4 *>(box32 + (size_t)kBox32Stride * tri)[1];
        float4 wl = lo4, wh = hi4;
        uint32_t ref = kLeafBit | tri;
        int lo = me, hi = me;  // offsets in the tile
        uint16_t mine = kNoSplit;
        // each step moves to a strictly larger range, so a walk ends within
        // the tile's depth; the bound only guards malformed input
        for (int step = 0; step <= kTreeTile; ++step) {
            const int dl = s_delta[lo], dr = s_delta[hi + 1];
            const bool left = dr > dl;  // a left child: its parent splits behind hi
            if (mine != kNoSplit) {
                const int idx = left ? hi : lo;
                s_idx[mine] = (uint16_t)idx;
                s_end[mine] = (uint16_t)(left ? lo : hi);
                s_taken[idx] = 1;
                s_parent[mine] = kNoSplit;  // until its parent is met
                for (int c = 0; c < 2; ++c)
                    if (s_child[mine][c] != kNoSplit)
                        s_parent[s_child[mine][c]] = (uint16_t)idx;
                ref = (uint32_t)(tile0 + idx);
            }
            if (dl < 0 && dr < 0) {  // the whole tree
                write_root(rootBox, wl, wh);
                break;
            }
            const int split = left ? hi : lo - 1;
            if (split < 0 || tile0 + split + 1 >= tile1) {  // its sibling lies in the next tile
                const float b[6] = {wl.x, wl.y, wl.z, wh.x, wh.y, wh.z};
                put6(piece + 6 * (size_t)(tile0 + lo), b);
                list_piece(out, &s_npiece, ref, b);
                s_start[lo] = 1;
                s_stop[hi] = 1;
                break;
            }
            const int side = left ? 0 : 1;
            float *slot = s_box[split][side];
            slot[0] = wl.x;
            slot[1] = wl.y;
            slot[2] = wl.z;
            slot[3] = wh.x;
            slot[4] = wh.y;
            slot[5] = wh.z;
            s_ref[split][side] = ref;
            s_far[split][side] = (uint16_t)(left ? lo : hi);
            s_child[split][side] = mine;
            __threadfence_block();
            if (atomicAdd(&s_flag[split], left ? 1u : 1u + kRightCame) == 0)
                break;
            __threadfence_block();
            const float *o = s_box[split][1 - side];
            wl = make_float4(fminf(wl.x, o[0]), fminf(wl.y, o[1]), fminf(wl.z, o[2]), 0.0f);
            wh = make_float4(fmaxf(wh.x, o[3]), fmaxf(wh.y, o[4]), fmaxf(wh.z, o[5]), 0.0f);
            if (left)
                hi = s_far[split][1];
            else
                lo = s_far[split][0];
            mine = (uint16_t)split;
        }
    }
    __syncthreads();
    const uint32_t came = s_flag[me];
    if ((came & 255u) == 2u) {
        // a node of the tile, whole
        const float *b0 = s_box[me][0], *b1 = s_box[me][1];
        BNode *nd = nodes + tile0 + s_idx[me];
        nd->a = make_float4(b0[0], b0[1], b0[2], b0[3]);
        nd->b = make_float4(b0[4], b0[5], b1[0], b1[1]);
        nd->c = make_float4(b1[2], b1[3], b1[4], b1[5]);
        // a parent outside the tile writes its children's links itself
        const int parent = s_parent[me] == kNoSplit ? -1 : tile0 + s_parent[me];
        nd->d = make_int4((int)s_ref[me][0], (int)s_ref[me][1], parent, tile0 + s_end[me]);
    } else if (came) {
        // one child of a top node
        const int side = came & kRightCame ? 1 : 0;
        const int lo = side ? me + 1 : s_far[me][0], hi = side ? s_far[me][1] : me;
        put6(piece + 6 * (size_t)(tile0 + lo), s_box[me][side]);
        list_piece(out, &s_npiece, s_ref[me][side], s_box[me][side]);
        s_start[lo] = 1;
        s_stop[hi] = 1;
    }
    if (gridDim.x == 1)  // one tile: no top node, and a search starts from the root
        return;
    // indices no node of the tile took: slots from LDS, one global reservation
    // per tile (one per wave held the kernel to the rate of one counter: 215
    // us at 3.0 M leaves)
    const int lane = me & 63, wave = me >> 6;
    const bool top = pos < n - 1 && valid && !s_taken[me];
    const unsigned long long tops = __ballot(top);
    uint32_t slot = 0;
    if (lane == 0 && tops)
        slot = atomicAdd(&s_ntop, (uint32_t)__popcll(tops));
    slot = __shfl(slot, 0, 64) + (uint32_t)__popcll(tops & ((1ull << lane) - 1ull));
    __syncthreads();
    if (me == 0)
        s_top0 = s_ntop ? atomicAdd(topCount, s_ntop) : 0u;
    // prefix / suffix unions over the tile's positions: wave scans, then the
    // waves' totals
    float pv[6] = {lo4.x, lo4.y, lo4.z, hi4.x, hi4.y, hi4.z}, sv[6] = {lo4.x, lo4.y, lo4.z, hi4.x, hi4.y, hi4.z};
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const float up = __shfl_up(pv[k], off, 64), dn = __shfl_down(sv[k], off, 64);
            if (lane >= off)
                pv[k] = k < 3 ? fminf(pv[k], up) : fmaxf(pv[k], up);
            if (lane + off < 64)
                sv[k] = k < 3 ? fminf(sv[k], dn) : fmaxf(sv[k], dn);
        }
    }
    if (lane == 63)
        put6(s_wave[wave], pv);
    __syncthreads();
    if (top)
        topList[s_top0 + slot] = (uint32_t)pos;
    if (me == 0 && out.count)
        out.count[blockIdx.x] = s_npiece;
    for (int w = 0; w < kTreeTile / 64; ++w) {
        if (w < wave)
#pragma unroll
            for (int k = 0; k < 6; ++k)
                pv[k] = k < 3 ? fminf(pv[k], s_wave[w][k]) : fmaxf(pv[k], s_wave[w][k]);
        if (w > wave)
#pragma unroll
            for (int k = 0; k < 6; ++k)
                sv[k] = k < 3 ? fminf(sv[k], s_wave[w][k]) : fmaxf(sv[k], s_wave[w][k]);
    }
    if (valid) {
        if (s_stop[me])
            put6(prefix + 6 * (size_t)pos, pv);
        if (s_start[me])
            put6(suffix + 6 * (size_t)pos, sv);
    }
    if (me == kTreeTile - 1)
        put6(tileBox + 6 * (size_t)blockIdx.x, pv);
}

// Sparse table over tile boxes: level j holds the union of tiles [t, t + 2^j).
// One workgroup.  Up to kLdsTiles tiles the levels are built in place in LDS
// (read, barrier, write, barrier) and copied out as they complete; beyond that
// each level is a pass over global memory.  The LDS is sized to the tiles at
// launch (24 B per tile): a workgroup asking for the whole 144 KB waits for a
// CU with nothing else resident, which the ray-grid build beside it delays.
constexpr uint32_t kLdsTiles = 6144;  // 144 KB of LDS (gfx950 gives a workgroup 160 KB)
constexpr int kLdsTileRounds = kLdsTiles / 1024;

__global__ __launch_bounds__(1024) void k_tile_table(float *__restrict__ table, uint32_t ntiles, int levels)
{
    extern __shared__ float s_tiles[];  // 6 x ntiles when ntiles <= kLdsTiles
    auto s_t = [&](int k, uint32_t t) -> float & { return s_tiles[(size_t)k * ntiles + t]; };
    if (ntiles <= kLdsTiles) {
        for (uint32_t t = threadIdx.x; t < ntiles; t += 1024)
            for (int k = 0; k < 6; ++k)
                s_t(k, t) = table[6 * (size_t)t + k];
        __syncthreads();
        for (int j = 1; j < levels; ++j) {
            const uint32_t half = 1u << (j - 1);
            float v[kLdsTileRounds][6];
#pragma unroll
            for (int r = 0; r < kLdsTileRounds; ++r) {
                const uint32_t t = threadIdx.x + 1024u * r;
                if (t + 2 * half <= ntiles)
#pragma unroll
                    for (int k = 0; k < 6; ++k)
                        v[r][k] = k < 3 ? fminf(s_t(k, t), s_t(k, t + half)) : fmaxf(s_t(k, t), s_t(k, t + half));
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kLdsTileRounds; ++r) {
                const uint32_t t = threadIdx.x + 1024u * r;
                if (t + 2 * half <= ntiles)
#pragma unroll
                    for (int k = 0; k < 6; ++k) {
                        s_t(k, t) = v[r][k];
                        table[6 * ((size_t)j * ntiles + t) + k] = v[r][k];
                    }
            }
            __syncthreads();
        }
        return;
    }
    for (int j = 1; j < levels; ++j) {
        const uint32_t half = 1u << (j - 1);
        const float *src = table + 6 * (size_t)(j - 1) * ntiles;
        float *dst = table + 6 * (size_t)j * ntiles;
        for (uint32_t t = threadIdx.x; t + 2 * half <= ntiles; t += 1024)
            for (int k = 0; k < 6; ++k) {
                const float a = src[6 * (size_t)t + k], b = src[6 * (size_t)(t + half) + k];
                dst[6 * (size_t)t + k] = k < 3 ? fminf(a, b) : fmaxf(a, b);
            }
        __syncthreads();
    }
}

// Box of the leaves [lo, hi], a child of a top node: a piece of one tile, or
// the suffix of lo's tile, the prefix of hi's and (with whole tiles between)
// two sparse-table entries.
__device__ __forceinline__ void range_box(uint32_t lo, uint32_t hi, const float *__restrict__ prefix,
                                          const float *__restrict__ suffix, const float *__restrict__ piece,
                                          const float *__restrict__ table, uint32_t ntiles, float v[6])
{
    const uint32_t tl = lo / kTreeTile, th = hi / kTreeTile;
    const float *a = tl == th ? piece + 6 * (size_t)lo : suffix + 6 * (size_t)lo;
    const float *b = tl == th ? a : prefix + 6 * (size_t)hi;
#pragma unroll
    for (int c = 0; c < 6; ++c)
        v[c] = c < 3 ? fminf(a[c], b[c]) : fmaxf(a[c], b[c]);
    if (th > tl + 1) {
        const uint32_t first = tl + 1, len = th - first;
        const int j = 31 - __clz(len);
        const float *x = table + 6 * ((size_t)j * ntiles + first);
        const float *y = table + 6 * ((size_t)j * ntiles + th - (1u << j));
#pragma unroll
        for (int c = 0; c < 6; ++c)
            v[c] = c < 3 ? fminf(v[c], fminf(x[c], y[c])) : fmaxf(v[c], fmaxf(x[c], y[c]));
    }
}

// Stage 2: every top node at once, a few per tile: its range and split from the
// keys by Karras' searches, its children's boxes from the tiles' pieces.  It
// writes its children's parent links, so nothing waits on anything.
template <typename K>
__global__ __launch_bounds__(256) void k_top_nodes(const K *__restrict__ codes, const uint32_t *__restrict__ ids, int n,
                                                   BNode *__restrict__ nodes, const uint32_t *__restrict__ topList,
                                                   const uint32_t *__restrict__ topCount,
                                                   const float *__restrict__ prefix, const float *__restrict__ suffix,
                                                   const float *__restrict__ piece, const float *__restrict__ table,
                                                   uint32_t ntiles, float *rootBox)
{
    const uint32_t ntop = *topCount;
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < ntop; k += gridDim.x * 256) {
        const int i = (int)topList[k];
        const int d = (delta(codes, n, i, i + 1) - delta(codes, n, i, i - 1)) >= 0 ? 1 : -1;
        const int dmin = delta(codes, n, i, i - d);
        int lmax = 2;
        while (delta(codes, n, i, i + lmax * d) > dmin)
            lmax <<= 1;
        int l = 0;
        for (int t = lmax >> 1; t >= 1; t >>= 1)
            if (delta(codes, n, i, i + (l + t) * d) > dmin)
                l += t;
        const int j = i + l * d;
        const int dnode = delta(codes, n, i, j);
        int s = 0;
        int t = l;
        do {
            t = (t + 1) >> 1;
            if (delta(codes, n, i, i + (s + t) * d) > dnode)
                s += t;
        } while (t > 1);
        const int gamma = i + s * d + (d < 0 ? d : 0);
        const int lo = i < j ? i : j;
        const int hi = i < j ? j : i;
        float b0[6], b1[6];
        range_box((uint32_t)lo, (uint32_t)gamma, prefix, suffix, piece, table, ntiles, b0);
        range_box((uint32_t)gamma + 1, (uint32_t)hi, prefix, suffix, piece, table, ntiles, b1);
        BNode *nd = nodes + i;
        nd->a = make_float4(b0[0], b0[1], b0[2], b0[3]);
        nd->b = make_float4(b0[4], b0[5], b1[0], b1[1]);
        nd->c = make_float4(b1[2], b1[3], b1[4], b1[5]);
        nd->d.x = lo == gamma ? (int)(kLeafBit | ids[gamma]) : gamma;
        nd->d.y = hi == gamma + 1 ? (int)(kLeafBit | ids[gamma + 1]) : gamma + 1;
        nd->d.w = j;  // the node covers sorted leaves [min(i, j), max(i, j)]
        if (lo != gamma)
            nodes[gamma].d.z = i;
        if (hi != gamma + 1)
            nodes[gamma + 1].d.z = i;
        if (i == 0) {
            nd->d.z = -1;
            write_root(rootBox,
                       make_float4(fminf(b0[0], b1[0]), fminf(b0[1], b1[1]), fminf(b0[2], b1[2]), 0.0f),
                       make_float4(fmaxf(b0[3], b1[3]), fmaxf(b0[4], b1[4]), fmaxf(b0[5], b1[5]), 0.0f));
        }
    }
}

__global__ void k_fill_u32(uint32_t *p, uint32_t v, size_t n)
{
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        p[i] = v;
}

// plain streaming copy, 16 B per lane per iteration (counter calibration)
__global__ __launch_bounds__(256) void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16)
{
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride)
        dst[i] = src[i];
}

void launch_copy16(const void *src, void *dst, size_t n16, hipStream_t s)
{
    if (n16 == 0)
        return;
    hipLaunchKernelGGL(k_copy16, dim3(4096), dim3(256), 0, s, (const uint4 *)src, (uint4 *)dst, n16);
}

void launch_fill_u32(uint32_t *p, uint32_t value, size_t n, hipStream_t s)
{
    if (n == 0)
        return;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, value, n);
}

static int table_levels(uint32_t ntiles)
{
    int L = 1;
    while ((1u << L) <= ntiles)
        ++L;
    return L;
}

uint32_t tree_tiles(uint32_t n) { return (n + kTreeTile - 1) / kTreeTile; }

float *tree_tile_boxes(float *scratch, uint32_t n) { return scratch + 18 * (size_t)n; }

size_t tree_scratch_floats(uint32_t n)
{
    const uint32_t ntiles = tree_tiles(n);
    return 18 * (size_t)n + 6 * (size_t)ntiles * table_levels(ntiles) + 6;
}

// work: n + 1 u32 (the top-node count, zero on entry, then the top-node list);
// scratch: tree_scratch_floats(n) floats (prefix, suffix, pieces, tile table)
template <typename K>
static void tree(const K *codes, const uint32_t *ids, const float *box32, uint32_t n, BNode *nodes, uint32_t *work,
                 float *scratch, TreePieces pieces, float *rootBox, hipStream_t s)
{
    if (n < 2)
        return;
    const uint32_t ntiles = tree_tiles(n);
    float *prefix = scratch, *suffix = prefix + 6 * (size_t)n, *piece = suffix + 6 * (size_t)n;
    float *table = tree_tile_boxes(scratch, n);
    hipLaunchKernelGGL(k_tree_tiles<K>, dim3(ntiles), dim3(kTreeTile), 0, s, codes, ids, box32, (int)n, nodes, work + 1,
                       work, prefix, suffix, piece, table, pieces, rootBox);
    if (ntiles < 2)
        return;
    const size_t lds = ntiles <= kLdsTiles ? sizeof(float) * 6 * ntiles : 0;
    if (lds > 65536)  // past the default cap on dynamic LDS (the error, if any, surfaces at the launch check)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_tile_table),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k_tile_table, dim3(1), dim3(1024), lds, s, table, ntiles, table_levels(ntiles));
    hipLaunchKernelGGL(k_top_nodes<K>, dim3(256), dim3(256), 0, s, codes, ids, (int)n, nodes,
                       (const uint32_t *)(work + 1), (const uint32_t *)work, prefix, suffix, piece, table, ntiles,
                       rootBox);
}

void launch_tree(const uint32_t *codes, const uint32_t *ids, const float *box32, uint32_t n, BNode *nodes,
                 uint32_t *work, float *scratch, TreePieces pieces, float *rootBox, hipStream_t s)
{
    tree(codes, ids, box32, n, nodes, work, scratch, pieces, rootBox, s);
}

void launch_tree64(const uint64_t *codes, const uint32_t *ids, const float *box32, uint32_t n, BNode *nodes,
                   uint32_t *work, float *scratch, float *rootBox, hipStream_t s)
{
    launch_fill_u32(work, 0u, 1, s);
    tree(codes, ids, box32, n, nodes, work, scratch, TreePieces{nullptr, nullptr}, rootBox, s);
}

}  // namespace sbg
