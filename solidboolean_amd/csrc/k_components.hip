// Connected components of a mesh's triangles across opposite half-edges: the
// groups that buildFaceGroups (src/solidboolean.cpp:167-239) forms for
// triangles no intersection loop touches (its leftover pass, :230-238, starts a
// group at each unvisited triangle in index order and floods it with a
// breadth-first search across half-edges, :203-226).  Triangle t's edge i -> j
// leads to the triangle that owns the half-edge j -> i.  Only unblocked
// triangles enter the half-edge table, as only untouched triangles enter the
// reference's map (addUnintersectedTriangles, :250-285), and a directed edge
// that two of them share is the reference's "repeated halfedge" failure
// (:271-282): the table flags it and the call fails.  Without repeats the
// relation is symmetric, so the flood fill's groups are exactly the
// connected components.
//
// The two half-edges of an edge meet in an LDS table (or, past the tiles that
// the triangle list is taken in, in a list sorted by a hash of the edge) and a
// concurrent union-find unites their triangles, always hooking the larger root under the smaller, so
// a component's root is its smallest triangle index, where the leftover pass
// starts that group.
#include "sbg_internal.h"

namespace sbg {

constexpr unsigned long long kEmptyKey = ~0ull;
constexpr int kComponentBlock = 256;

__device__ __forceinline__ uint32_t he_slot(unsigned long long key, uint32_t mask)
{
    return (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> 32) & mask;
}

// every half-edge of every triangle; owners start at ~0u and become the
// smallest triangle that holds the key
__global__ __launch_bounds__(kComponentBlock) void k_he_insert(const uint32_t *__restrict__ T, uint32_t nt,
                                                               unsigned long long *__restrict__ keys,
                                                               uint32_t *__restrict__ owners, uint32_t mask)
{
    const uint32_t e = blockIdx.x * kComponentBlock + threadIdx.x;
    if (e >= 3u * nt)
        return;
    const uint32_t t = e / 3, k = e - 3 * t;
    const uint32_t from = T[3 * (size_t)t + k], to = T[3 * (size_t)t + (k + 1) % 3];
    const unsigned long long key = (unsigned long long)from << 32 | to;
    uint32_t s = he_slot(key, mask);
    // the table holds at least twice as many slots as half-edges, so a free
    // slot is always found
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        const unsigned long long cur = atomicCAS(&keys[s], kEmptyKey, key);
        if (cur == kEmptyKey || cur == key) {
            atomicMin(&owners[s], t);
            return;
        }
        s = (s + 1) & mask;
    }
}

// owner of half-edge `key`, or ~0u
__device__ __forceinline__ uint32_t he_owner(const unsigned long long *__restrict__ keys,
                                             const uint32_t *__restrict__ owners, uint32_t mask,
                                             unsigned long long key)
{
    uint32_t s = he_slot(key, mask);
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        const unsigned long long cur = keys[s];
        if (cur == key)
            return owners[s];
        if (cur == kEmptyKey)
            return ~0u;
        s = (s + 1) & mask;
    }
    return ~0u;
}

// raises the repeated-half-edge flag; once it stands it is only read
__device__ __forceinline__ bool repeat_known(const uint32_t *repeated)
{
    return __hip_atomic_load(repeated, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
}
__device__ __forceinline__ void raise_repeat(uint32_t *repeated)
{
    if (!repeat_known(repeated))
        atomicOr(repeated, 1u);
}

__device__ __forceinline__ uint32_t cc_find(uint32_t *parent, uint32_t x)
{
    uint32_t p = __hip_atomic_load(&parent[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (p != x) {
        const uint32_t gp = __hip_atomic_load(&parent[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (gp != p)  // path halving; a lost race only leaves a longer path
            __hip_atomic_store(&parent[x], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = p;
        p = gp;
    }
    return x;
}

// Union of a's and b's sets: the larger root is hooked under the smaller,
// unless it stopped being a root meanwhile.
__device__ __forceinline__ void cc_unite(uint32_t *parent, uint32_t t, uint32_t o)
{
    uint32_t a = cc_find(parent, t), b = cc_find(parent, o);
    while (a != b) {
        if (a > b) {
            const uint32_t x = a;
            a = b;
            b = x;
        }
        const uint32_t old = atomicCAS(&parent[b], b, a);
        if (old == b)
            break;
        b = cc_find(parent, old);
        a = cc_find(parent, a);
    }
}

// ---- components in tiles ----------------------------------------------------
// A mesh's triangle list is local: most edges lie inside a run of a thousand
// triangles.  So a workgroup takes a tile of kCcTile consecutive triangles,
// pairs the half-edges of each edge in an LDS table and unites their triangles
// in LDS.  An edge is settled there when every unblocked triangle at one of
// its ends lies in the tile (the tile's count of that vertex equals the mesh's,
// counted by a first pass): then no triangle elsewhere holds the edge, and a
// repeated directed edge shows up in the LDS table.  The half-edges of all
// other edges are listed, sorted by a hash of their edge (k_sort.hip, so the
// memory traffic is streams) and paired in LDS run by run of equal hashes.
//
// What bounded the former table in global memory was device-wide atomics: two
// per half-edge (claim a key, lower its owner), about 6 G/s whatever the order.
// Measured figures stand at launch_components.
//
// A table entry is an edge's first half-edge e as (e + 1) << 1, and bit 0 once
// the opposite one has come.  A half-edge that meets one of its own direction,
// or an opposite place already taken, repeats a directed edge.
constexpr int kCcTile = 1024;
constexpr int kCcVertSlots = 4096, kCcEdgeSlots = 4096;  // at most 3 * kCcTile entries each
constexpr uint32_t kNoVertex = ~0u;

__device__ __forceinline__ uint32_t vert_hash(uint32_t v) { return (v * 2654435761u) >> 20; }
static_assert(kCcVertSlots == 1 << 12 && kCcEdgeSlots == 1 << 12, "hashes give 12 bits");

// the tile's corners counted per vertex in an LDS table; the slot of a vertex
// is where its key is found.  The vertex kNoVertex (the empty mark) is left out.
__device__ __forceinline__ void count_vertex(uint32_t *keys, uint32_t *counts, uint32_t v)
{
    if (v == kNoVertex)
        return;
    uint32_t h = vert_hash(v);
    for (int probe = 0; probe < kCcVertSlots; ++probe) {
        uint32_t cur = __hip_atomic_load(&keys[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (cur == kNoVertex)
            cur = atomicCAS(&keys[h], kNoVertex, v);
        if (cur == kNoVertex || cur == v) {
            atomicAdd(&counts[h], 1u);
            return;
        }
        h = (h + 1) & (kCcVertSlots - 1);
    }
}

__device__ __forceinline__ void tile_vertices(const uint32_t *__restrict__ T, uint32_t nt,
                                              const uint8_t *__restrict__ blocked, uint32_t *keys, uint32_t *counts,
                                              uint32_t v[3], bool &live)
{
    for (int k = threadIdx.x; k < kCcVertSlots; k += kCcTile) {
        keys[k] = kNoVertex;
        counts[k] = 0;
    }
    __syncthreads();
    const uint32_t t = blockIdx.x * kCcTile + threadIdx.x;
    live = t < nt && !(blocked && blocked[t]);
    if (live) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            v[k] = T[3 * (size_t)t + k];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            count_vertex(keys, counts, v[k]);
    }
    __syncthreads();
}

// corners of unblocked triangles at every vertex (valence: zero on entry)
__global__ __launch_bounds__(kCcTile) void k_cc_valence(const uint32_t *__restrict__ T, uint32_t nt,
                                                        const uint8_t *__restrict__ blocked,
                                                        uint32_t *__restrict__ valence)
{
    __shared__ uint32_t s_key[kCcVertSlots], s_count[kCcVertSlots];
    uint32_t v[3];
    bool live;
    tile_vertices(T, nt, blocked, s_key, s_count, v, live);
    for (int k = threadIdx.x; k < kCcVertSlots; k += kCcTile)
        if (s_key[k] != kNoVertex)
            atomicAdd(&valence[s_key[k]], s_count[k]);
}

// whether the tile holds every corner at v (counts[] then reads 1)
__device__ __forceinline__ bool vertex_whole(const uint32_t *keys, const uint32_t *whole, uint32_t v)
{
    if (v == kNoVertex)
        return false;
    uint32_t h = vert_hash(v);
    for (int probe = 0; probe < kCcVertSlots; ++probe) {
        if (keys[h] == v)
            return whole[h] != 0;
        h = (h + 1) & (kCcVertSlots - 1);
    }
    return false;
}

// hash of the edge {lo, hi}, well mixed in its top bits
__device__ __forceinline__ uint32_t edge_hash(uint32_t lo, uint32_t hi)
{
    uint32_t h = lo * 2654435761u ^ hi * 2246822519u;
    h ^= h >> 15;
    h *= 0x85ebca6bu;
    h ^= h >> 13;
    return h * 0xc2b2ae35u;
}

// sort keys of the listed half-edges: hash bits above the half-edge's index
constexpr int kOpenShift = 40;

// Pairs the tile's half-edges and unites their triangles; parent[t] = the
// smallest triangle of t's set within the tile.  The half-edges of edges the
// tile does not settle go to list (*count of them, in no order; room for
// all), keyed by the top hashBits of their edge's hash.
__global__ __launch_bounds__(kCcTile) void k_cc_tiles(const uint32_t *__restrict__ T, uint32_t nt,
                                                      const uint8_t *__restrict__ blocked,
                                                      const uint32_t *__restrict__ valence, int hashBits,
                                                      uint32_t *__restrict__ parent, uint64_t *__restrict__ list,
                                                      uint32_t *__restrict__ count, uint32_t *__restrict__ repeated)
{
    __shared__ uint32_t s_key[kCcVertSlots], s_count[kCcVertSlots];
    __shared__ uint32_t s_edge[kCcEdgeSlots];
    __shared__ uint32_t s_vert[3 * kCcTile];
    __shared__ uint32_t s_parent[kCcTile];
    const uint32_t tile0 = blockIdx.x * kCcTile, t = tile0 + threadIdx.x;
    uint32_t v[3] = {0, 0, 0};
    bool live;
    tile_vertices(T, nt, blocked, s_key, s_count, v, live);
    for (int k = threadIdx.x; k < kCcVertSlots; k += kCcTile)
        s_count[k] = s_key[k] != kNoVertex && s_count[k] == valence[s_key[k]] ? 1u : 0u;
    for (int k = threadIdx.x; k < kCcEdgeSlots; k += kCcTile)
        s_edge[k] = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        s_vert[3 * threadIdx.x + k] = v[k];
    s_parent[threadIdx.x] = threadIdx.x;
    __syncthreads();
    uint32_t open = 0;  // bits of the triangle's half-edges to list
    if (live) {
        bool whole[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            whole[k] = vertex_whole(s_key, s_count, v[k]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t from = v[k], to = v[(k + 1) % 3];
            if (!whole[k] && !whole[(k + 1) % 3])
                open |= 1u << k;
            const uint32_t lo = min(from, to), hi = max(from, to);
            const uint32_t mine = (3 * threadIdx.x + k + 1) << 1;
            uint32_t s = edge_hash(lo, hi) >> 20;
            for (int probe = 0; probe < kCcEdgeSlots; ++probe) {
                const uint32_t cur = atomicCAS(&s_edge[s], 0u, mine);
                if (cur == 0u)
                    break;
                const uint32_t e = (cur >> 1) - 1, ot = e / 3, ok = e - 3 * ot;
                const uint32_t of = s_vert[e], oto = s_vert[3 * ot + (ok == 2 ? 0 : ok + 1)];
                if (min(of, oto) == lo && max(of, oto) == hi) {
                    if (of == from || (cur & 1u) || atomicOr(&s_edge[s], 1u) & 1u)
                        raise_repeat(repeated);
                    else
                        cc_unite(s_parent, threadIdx.x, ot);
                    break;
                }
                s = (s + 1) & (kCcEdgeSlots - 1);
            }
        }
    }
    __syncthreads();
    if (t < nt)
        parent[t] = live ? tile0 + cc_find(s_parent, threadIdx.x) : t;
    // list slots: a wave prefix, one LDS add per wave, one global add per tile
    uint32_t *s_sum = s_key;  // the vertex table is done with
    const int lane = threadIdx.x & 63;
    const uint32_t mine = (uint32_t)__popc(open);
    uint32_t incl = mine;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_up(incl, off, 64);
        if (lane >= off)
            incl += u;
    }
    if (threadIdx.x == 0)
        s_sum[0] = 0;
    __syncthreads();
    uint32_t base = 0;
    if (lane == 63 && incl)
        base = atomicAdd(&s_sum[0], incl);
    base = __shfl(base, 63, 64);
    __syncthreads();
    if (threadIdx.x == 0)
        s_sum[1] = s_sum[0] ? atomicAdd(count, s_sum[0]) : 0u;
    __syncthreads();
    uint64_t *out = list + s_sum[1] + base + incl - mine;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (open >> k & 1u) {
            const uint32_t from = v[k], to = v[(k + 1) % 3];
            const uint32_t h = edge_hash(min(from, to), max(from, to)) >> (32 - hashBits);
            *out++ = (uint64_t)h << kOpenShift | (3ull * t + k);
        }
}

// The listed half-edges, sorted by hash, so that both of an edge lie in one run
// of equal hashes: a workgroup takes the runs that start in its kCcTile
// entries and pairs them in an LDS table as k_cc_tiles does.  mate[e] (~0u on
// entry) gets the triangle across half-edge e for one of the two, unless both
// lie in one tile, which has united them.
constexpr int kCcAhead = 512;  // entries past its own that a workgroup holds
constexpr int kCcHeld = kCcTile + kCcAhead;

// the half-edge's ends, from << 32 | to
__device__ __forceinline__ uint64_t half_of(const uint32_t *__restrict__ T, uint32_t e)
{
    return (uint64_t)T[e] << 32 | T[e % 3u == 2u ? e - 2u : e + 1u];
}

// the halves a and b of one edge
__device__ __forceinline__ void pair_halves(uint64_t a, uint32_t ea, uint64_t b, uint32_t eb,
                                            uint32_t *__restrict__ mate, uint32_t *repeated)
{
    if (a == b)
        raise_repeat(repeated);
    else if (ea / (3u * kCcTile) != eb / (3u * kCcTile))
        mate[ea] = eb / 3u;
}

// A run longer than a workgroup holds, list[first, last): thousands of triangles
// on one edge, which three half-edges prove to be repeated, or as many edges
// of one hash.  The same pairing in an open-addressed table in global memory, a
// slot of `table` per entry, so it takes one insertion per entry however long the
// run is; it ends as soon as a repeat is known.  A million triangles collapsed to
// a point are refused in 0.47 ms a call; 2,600 two-triangle shells with an edge of
// one hash each, a run of 5,200, take 1.3 ms.  An entry of the table is an
// edge's first half-edge e as (e + 1) << 1, and bit 0 once the opposite one has come.
__device__ void match_long_run(const uint32_t *__restrict__ T, const uint64_t *__restrict__ list, uint64_t first,
                               uint64_t last, unsigned long long *table, uint32_t *__restrict__ mate,
                               uint32_t *repeated)
{
    const uint64_t slots = last - first;
    for (uint64_t k = threadIdx.x; k < slots; k += kCcTile)
        __hip_atomic_store(&table[k], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence();
    __syncthreads();
    for (uint64_t i = first + threadIdx.x; i < last && !repeat_known(repeated); i += kCcTile) {
        const uint32_t e = (uint32_t)list[i];
        const uint64_t half = half_of(T, e), back = half << 32 | half >> 32;
        // MurmurHash3's 64-bit finalizer, whose last step leaves the top half as
        // it is: the run's entries share edge_hash
        uint64_t h = half < back ? half : back;
        h ^= h >> 33;
        h *= 0xff51afd7ed558ccdull;
        h ^= h >> 33;
        h *= 0xc4ceb9fe1a85ec53ull;
        uint64_t s = (h >> 32) * slots >> 32;  // slots fit 32 bits
        for (uint64_t probe = 0; probe < slots; ++probe) {
            const unsigned long long cur = atomicCAS(&table[s], 0ull, (unsigned long long)(e + 1ull) << 1);
            if (cur == 0ull)
                break;
            const uint32_t o = (uint32_t)((cur >> 1) - 1ull);
            const uint64_t other = half_of(T, o);
            if (other == half || other == back) {
                if ((cur & 1ull) || atomicOr(&table[s], 1ull) & 1ull)
                    raise_repeat(repeated);
                else
                    pair_halves(half, e, other, o, mate, repeated);
                break;
            }
            s = s + 1 < slots ? s + 1 : 0;
        }
    }
}

// spare: as many entries as list (the sort's other buffer)
__global__ __launch_bounds__(kCcTile) void k_cc_match(const uint32_t *__restrict__ T,
                                                      const uint64_t *__restrict__ list,
                                                      const uint32_t *__restrict__ count, uint64_t *__restrict__ spare,
                                                      uint32_t *__restrict__ mate, uint32_t *repeated)
{
    __shared__ uint64_t s_half[kCcHeld];  // from << 32 | to
    __shared__ uint32_t s_hash[kCcHeld], s_e[kCcHeld];
    __shared__ uint32_t s_edge[kCcEdgeSlots];
    __shared__ uint32_t s_end, s_last0, s_known;
    const uint64_t n = *count, first = (uint64_t)blockIdx.x * kCcTile;
    if (first >= n)
        return;
    if (threadIdx.x == 0)
        s_known = repeat_known(repeated);
    __syncthreads();
    if (s_known)  // the call fails whatever else is found
        return;
    const uint32_t held = (uint32_t)(n - first < (uint64_t)kCcHeld ? n - first : (uint64_t)kCcHeld);
    const uint32_t own = held < (uint32_t)kCcTile ? held : (uint32_t)kCcTile;
    auto hash_at = [&](uint64_t i) -> uint32_t { return (uint32_t)(list[i] >> kOpenShift); };
    // the hash of the run that came in from the workgroup before, which takes it
    const uint32_t before = first ? hash_at(first - 1) : ~0u;  // no hash has 32 bits
    for (uint32_t j = threadIdx.x; j < held; j += kCcTile) {
        const uint64_t key = list[first + j];
        s_hash[j] = (uint32_t)(key >> kOpenShift);
        s_e[j] = (uint32_t)key;
        s_half[j] = half_of(T, s_e[j]);
    }
    for (int k = threadIdx.x; k < kCcEdgeSlots; k += kCcTile)
        s_edge[k] = 0;
    if (threadIdx.x == 0) {
        s_end = held;
        s_last0 = own - 1;
    }
    __syncthreads();
    // its last run is the entries [s_last0, s_end), as far as held
    const uint32_t last = s_hash[own - 1];
    for (uint32_t j = threadIdx.x; j < held; j += kCcTile) {
        if (j < own && s_hash[j] == last)
            atomicMin(&s_last0, j);
        else if (j >= own && s_hash[j] != last)
            atomicMin(&s_end, j);
    }
    __syncthreads();
    const bool longRun = s_end == held && first + held < n && hash_at(first + held) == last;
    const uint32_t end = longRun ? s_last0 : s_end;
    for (uint32_t j = threadIdx.x; j < end; j += kCcTile) {
        if (s_hash[j] == before)
            continue;
        const uint64_t half = s_half[j], back = half << 32 | half >> 32;
        const uint32_t lo = min((uint32_t)half, (uint32_t)back), hi = max((uint32_t)half, (uint32_t)back);
        uint32_t s = (edge_hash(lo, hi) * 0x9E3779B1u) >> 20;
        for (int probe = 0; probe < kCcEdgeSlots; ++probe) {
            const uint32_t cur = atomicCAS(&s_edge[s], 0u, (j + 1) << 1);
            if (cur == 0u)
                break;
            const uint32_t o = (cur >> 1) - 1;
            if (s_half[o] == half || s_half[o] == back) {
                if ((cur & 1u) || atomicOr(&s_edge[s], 1u) & 1u)
                    raise_repeat(repeated);
                else
                    pair_halves(half, s_e[j], s_half[o], s_e[o], mate, repeated);
                break;
            }
            s = (s + 1) & (kCcEdgeSlots - 1);
        }
    }
    if (longRun && last != before) {
        uint64_t a = first + held, b = n;  // the run's end: the first entry of another hash
        while (a < b) {
            const uint64_t m = a + (b - a) / 2;
            if (hash_at(m) == last)
                a = m + 1;
            else
                b = m;
        }
        const uint64_t run = first + s_last0;
        match_long_run(T, list, run, a, reinterpret_cast<unsigned long long *>(spare + run), mate, repeated);
    }
}

// Unites the triangles of mated half-edges.  A tile's border meets few others
// thousands of times over: each pair of roots is united once per tile (an LDS
// set of pairs), or the few roots' words would take every union of the mesh
// (550 us with a union per half-edge).
constexpr int kCcPairSlots = 4096;

__global__ __launch_bounds__(kCcTile) void k_cc_unite(const uint32_t *__restrict__ mate, uint32_t nt, uint32_t *parent)
{
    __shared__ unsigned long long s_pair[kCcPairSlots];
    for (int k = threadIdx.x; k < kCcPairSlots; k += kCcTile)
        s_pair[k] = kEmptyKey;
    __syncthreads();
    const uint32_t t = blockIdx.x * kCcTile + threadIdx.x;
    if (t >= nt)
        return;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint32_t o = mate[3 * (size_t)t + k];
        if (o == ~0u)
            continue;
        // ancestors at some moment, which is all the set needs
        const uint32_t a = parent[t], b = parent[o];
        if (a == b)
            continue;
        const unsigned long long key = (unsigned long long)a << 32 | b;
        uint32_t s = edge_hash(a, b) >> 20;
        bool seen = false;
        for (int probe = 0; probe < 16; ++probe) {
            const unsigned long long cur = atomicCAS(&s_pair[s], kEmptyKey, key);
            seen = cur == key;
            if (seen || cur == kEmptyKey)
                break;
            s = (s + 1) & (kCcPairSlots - 1);
        }
        if (!seen)
            cc_unite(parent, a, b);
    }
}

__global__ __launch_bounds__(kComponentBlock) void k_cc_labels(const uint8_t *__restrict__ blocked, uint32_t nt,
                                                               uint32_t *parent, uint32_t *__restrict__ labels)
{
    const uint32_t t = blockIdx.x * kComponentBlock + threadIdx.x;
    if (t >= nt)
        return;
    labels[t] = (blocked && blocked[t]) ? ~0u : cc_find(parent, t);
}

// Half-edge table queries for the host's face grouping.  repeat: triangle t
// repeats a directed edge when an earlier triangle owns one of its half-edges
// or two of its own are equal (where inserting its half-edges in order would
// first fail); *firstRepeat = the smallest such t.
__global__ __launch_bounds__(kComponentBlock) void k_he_opposite(const uint32_t *__restrict__ T, uint32_t nt,
                                                                 const unsigned long long *__restrict__ keys,
                                                                 const uint32_t *__restrict__ owners, uint32_t mask,
                                                                 uint32_t *__restrict__ opposite,
                                                                 uint32_t *__restrict__ firstRepeat)
{
    const uint32_t e = blockIdx.x * kComponentBlock + threadIdx.x;
    if (e >= 3u * nt)
        return;
    const uint32_t t = e / 3, k = e - 3 * t;
    const uint32_t from = T[3 * (size_t)t + k], to = T[3 * (size_t)t + (k + 1) % 3];
    opposite[e] = he_owner(keys, owners, mask, (unsigned long long)to << 32 | from);
    bool repeat = he_owner(keys, owners, mask, (unsigned long long)from << 32 | to) < t;
    for (uint32_t j = 0; j < k; ++j)
        repeat |= T[3 * (size_t)t + j] == from && T[3 * (size_t)t + (j + 1) % 3] == to;
    if (repeat)
        atomicMin(firstRepeat, t);
}

__global__ __launch_bounds__(kComponentBlock) void k_he_query(const unsigned long long *__restrict__ queries,
                                                              uint32_t nq,
                                                              const unsigned long long *__restrict__ keys,
                                                              const uint32_t *__restrict__ owners, uint32_t mask,
                                                              uint32_t *__restrict__ out)
{
    const uint32_t i = blockIdx.x * kComponentBlock + threadIdx.x;
    if (i < nq)
        out[i] = he_owner(keys, owners, mask, queries[i]);
}

size_t component_table_slots(uint32_t nt)
{
    size_t cap = 1024;
    while (cap < 6 * (size_t)nt)
        cap <<= 1;
    return cap;
}

// Hash bits so that some tens of listed half-edges share a hash: whole 8-bit
// sort passes.
static int open_bits(size_t halfEdges)
{
    return halfEdges <= (1u << 14) ? 8 : (halfEdges <= (1u << 22) ? 16 : 24);
}

// At 1,314,540 triangles (a torus in ring order, a ring longer than a tile, so
// that every edge is listed) the kernels take 0.39 ms: fills 14 us, valence 56,
// tiles 68, the two sort passes 82, match 78, unite 72, labels 17.  One table
// and one forest in global memory for all half-edges took 3.86 ms.
// list, listAlt: 3 nt u64; hist: sort_hist_entries(3 nt); valence: nv + 2 (the
// last words are the list's length and the repeated-half-edge flag); mate: 3 nt;
// parent, labels: nt
void launch_components(const uint32_t *T, uint32_t nt, size_t nv, const uint8_t *blocked, uint64_t *list,
                       uint64_t *listAlt, uint32_t *hist, uint32_t *valence, uint32_t *mate, uint32_t *parent,
                       uint32_t *labels, hipStream_t s)
{
    if (nt == 0)
        return;
    const size_t he = 3 * (size_t)nt;
    const dim3 tiles((nt + kCcTile - 1) / kCcTile);
    uint32_t *count = valence + nv, *repeated = valence + nv + 1;
    launch_fill_u32(valence, 0u, nv + 2, s);
    launch_fill_u32(mate, ~0u, he, s);
    hipLaunchKernelGGL(k_cc_valence, tiles, dim3(kCcTile), 0, s, T, nt, blocked, valence);
    hipLaunchKernelGGL(k_cc_tiles, tiles, dim3(kCcTile), 0, s, T, nt, blocked, valence, open_bits(he), parent, list,
                       count, repeated);
    const int bits[2] = {kOpenShift, kOpenShift + open_bits(he)};
    const bool alt = radix_sort_u64(list, listAlt, he, bits, 1, hist, s, count) != 0;
    hipLaunchKernelGGL(k_cc_match, dim3((unsigned)((he + kCcTile - 1) / kCcTile)), dim3(kCcTile), 0, s, T,
                       alt ? listAlt : list, count, alt ? list : listAlt, mate, repeated);
    hipLaunchKernelGGL(k_cc_unite, tiles, dim3(kCcTile), 0, s, mate, nt, parent);
    hipLaunchKernelGGL(k_cc_labels, dim3((nt + kComponentBlock - 1) / kComponentBlock), dim3(kComponentBlock), 0, s,
                       blocked, nt, parent, labels);
}

}  // namespace sbg

namespace sbg {

// keys, owners: component_table_slots(nt) entries; opposite: 3 nt;
// firstRepeat: 1 word; queries / queryOwner: nq
void launch_half_edges(const uint32_t *T, uint32_t nt, const unsigned long long *queries, uint32_t nq,
                       unsigned long long *keys, uint32_t *owners, uint32_t *opposite, uint32_t *queryOwner,
                       uint32_t *firstRepeat, hipStream_t s)
{
    const size_t slots = component_table_slots(nt);
    const uint32_t mask = (uint32_t)(slots - 1);
    launch_fill_u32(firstRepeat, ~0u, 1, s);
    if (nt) {
        launch_fill_u32(reinterpret_cast<uint32_t *>(keys), ~0u, 2 * slots, s);
        launch_fill_u32(owners, ~0u, slots, s);
        const uint32_t he = 3u * nt;
        hipLaunchKernelGGL(k_he_insert, dim3((he + kComponentBlock - 1) / kComponentBlock), dim3(kComponentBlock), 0,
                           s, T, nt, keys, owners, mask);
        hipLaunchKernelGGL(k_he_opposite, dim3((he + kComponentBlock - 1) / kComponentBlock), dim3(kComponentBlock),
                           0, s, T, nt, keys, owners, mask, opposite, firstRepeat);
    } else {
        launch_fill_u32(reinterpret_cast<uint32_t *>(keys), ~0u, 2 * slots, s);
    }
    if (nq)
        hipLaunchKernelGGL(k_he_query, dim3((nq + kComponentBlock - 1) / kComponentBlock), dim3(kComponentBlock), 0, s,
                           queries, nq, keys, owners, mask, queryOwner);
}

}  // namespace sbg
