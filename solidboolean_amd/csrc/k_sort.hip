// Stable LSD radix sort, 8-bit digits, for u32 keys (+ u32 values) and u64 keys.
//
// Per pass: (1) every block counts the digits of its tile (256 x ITEMS keys)
// into LDS and writes a 256 x nblocks histogram column; (2) one block per digit
// turns the histogram (digit-major) into exclusive offsets; (3) every block
// loads its whole tile into registers, then ranks it in order, 256 keys per
// round, each key among equal digits with a 64-lane ballot match (stable within
// the wave), adds the counts of earlier waves and earlier rounds kept in LDS,
// and scatters.  ITEMS shrinks with n so that short sorts still spread over
// many workgroups.  Per key and pass: read 4 (8) B key (+4 B value) twice,
// write once.
#include "sbg_device.h"
#include "sbg_internal.h"

namespace sbg {

constexpr int kSortBlock = 256;
constexpr int kWaves = kSortBlock / 64;

// up to this many blocks the scatter kernel sums the histogram itself, and the
// pass needs no scan kernel (a launch of 3 us and its gap)
constexpr int kScanInScatter = 64;

// keys per thread for a sort of n keys
static int sort_items(size_t n) { return n >= ((size_t)1 << 20) ? 16 : (n >= ((size_t)1 << 17) ? 8 : 4); }

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K key, int shift, uint32_t mask)
{
    return (uint32_t)(key >> shift) & mask;
}

// count (may be null): the keys are the first min(n, *count) of the n the
// launch covers (a list whose length is known on the device only); the rest
// are neither read nor moved
__device__ __forceinline__ size_t sort_len(size_t n, const uint32_t *count)
{
    return count && *count < n ? *count : n;
}

template <typename K, int ITEMS>
__global__ __launch_bounds__(kSortBlock) void k_hist(const K *__restrict__ keys, size_t n,
                                                     const uint32_t *__restrict__ count, int shift, uint32_t mask,
                                                     uint32_t *__restrict__ hist, int nblocks)
{
    n = sort_len(n, count);
    __shared__ uint32_t s_cnt[256];
    s_cnt[threadIdx.x] = 0;
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * (kSortBlock * ITEMS);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        size_t idx = base + (size_t)r * kSortBlock + threadIdx.x;
        if (idx < n)
            atomicAdd(&s_cnt[digit_of(keys[idx], shift, mask)], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * nblocks + blockIdx.x] = s_cnt[threadIdx.x];
}

// exclusive scan of m entries in place, one block of 1024 threads
__global__ __launch_bounds__(1024) void k_scan(uint32_t *__restrict__ data, size_t m)
{
    __shared__ uint32_t s_part[1024];
    const size_t per = (m + 1023) / 1024;
    const size_t lo = (size_t)threadIdx.x * per;
    const size_t hi = lo + per < m ? lo + per : m;
    uint32_t sum = 0;
    for (size_t i = lo; i < hi; ++i)
        sum += data[i];
    s_part[threadIdx.x] = sum;
    __syncthreads();
    // Hillis-Steele inclusive scan of the 1024 partials
    for (int off = 1; off < 1024; off <<= 1) {
        uint32_t v = threadIdx.x >= (unsigned)off ? s_part[threadIdx.x - off] : 0;
        __syncthreads();
        s_part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = threadIdx.x ? s_part[threadIdx.x - 1] : 0;
    for (size_t i = lo; i < hi; ++i) {
        uint32_t v = data[i];
        data[i] = run;
        run += v;
    }
}

// ---- exclusive scan of a long u32 array, three launches --------------------
// Tiles of 4096 entries (16 per thread): tile sums, a one-block scan of the
// sums, then each tile rescans its entries from its base.
constexpr int kScanTile = 4096;
// up to this many entries one workgroup scans alone (a launch for three)
constexpr size_t kScanOneBlock = 16384;

__global__ __launch_bounds__(256) void k_scan_tile_sum(const uint32_t *__restrict__ data, size_t m,
                                                       uint32_t *__restrict__ tileSum)
{
    __shared__ uint32_t s[256];
    const size_t base = (size_t)blockIdx.x * kScanTile;
    uint32_t sum = 0;
    for (int k = 0; k < kScanTile / 256; ++k) {
        const size_t i = base + (size_t)k * 256 + threadIdx.x;
        if (i < m)
            sum += data[i];
    }
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            s[threadIdx.x] += s[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        tileSum[blockIdx.x] = s[0];
}

__global__ __launch_bounds__(256) void k_scan_tile_apply(uint32_t *__restrict__ data, size_t m,
                                                         const uint32_t *__restrict__ tileBase)
{
    __shared__ uint32_t s[256];
    constexpr int per = kScanTile / 256;
    const size_t lo = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * per;
    uint32_t v[per];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < per; ++k) {
        v[k] = lo + k < m ? data[lo + k] : 0u;
        sum += v[k];
    }
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t t = threadIdx.x >= (unsigned)off ? s[threadIdx.x - off] : 0;
        __syncthreads();
        s[threadIdx.x] += t;
        __syncthreads();
    }
    uint32_t run = tileBase[blockIdx.x] + (threadIdx.x ? s[threadIdx.x - 1] : 0u);
#pragma unroll
    for (int k = 0; k < per; ++k) {
        if (lo + k < m)
            data[lo + k] = run;
        run += v[k];
    }
}

size_t scan_large_temp(size_t m) { return (m + kScanTile - 1) / kScanTile + 1; }

void launch_scan_large(uint32_t *data, size_t m, uint32_t *temp, hipStream_t s)
{
    if (m == 0)
        return;
    if (m <= kScanOneBlock) {
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, data, m);
        return;
    }
    const size_t tiles = (m + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_scan_tile_sum, dim3((unsigned)tiles), dim3(256), 0, s, data, m, temp);
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, temp, tiles);
    hipLaunchKernelGGL(k_scan_tile_apply, dim3((unsigned)tiles), dim3(256), 0, s, data, m, temp);
}

// exclusive scan of each digit's row of the histogram (one workgroup per
// digit); the row's total goes to rowTotal[digit]
__global__ __launch_bounds__(256) void k_scan_rows(uint32_t *__restrict__ hist, int nblocks,
                                                   uint32_t *__restrict__ rowTotal)
{
    __shared__ uint32_t s[256];
    uint32_t *row = hist + (size_t)blockIdx.x * nblocks;
    const int per = (nblocks + 255) / 256;
    const int lo = threadIdx.x * per;
    const int hi = lo + per < nblocks ? lo + per : nblocks;
    uint32_t sum = 0;
    for (int i = lo; i < hi; ++i)
        sum += row[i];
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t v = threadIdx.x >= (unsigned)off ? s[threadIdx.x - off] : 0;
        __syncthreads();
        s[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = threadIdx.x ? s[threadIdx.x - 1] : 0;
    for (int i = lo; i < hi; ++i) {
        const uint32_t v = row[i];
        row[i] = run;
        run += v;
    }
    if (threadIdx.x == 255)
        rowTotal[blockIdx.x] = s[255];
}

// rowTotal null: `offsets` still holds the blocks' digit counts (at most
// kScanInScatter blocks), and every block sums up the ones it needs itself.
template <typename K, bool HAS_VAL, int ITEMS>
__global__ __launch_bounds__(kSortBlock) void k_scatter(const K *__restrict__ keys, const uint32_t *__restrict__ vals,
                                                        K *__restrict__ keysOut, uint32_t *__restrict__ valsOut,
                                                        size_t n, const uint32_t *__restrict__ count, int shift,
                                                        uint32_t mask, const uint32_t *__restrict__ offsets,
                                                        int nblocks, const uint32_t *__restrict__ rowTotal)
{
    n = sort_len(n, count);
    __shared__ uint32_t s_base[256];
    __shared__ uint32_t s_wcnt[kWaves][256];
    // the tile first, so that its loads overlap the offset set-up
    const size_t base = (size_t)blockIdx.x * (kSortBlock * ITEMS);
    K kreg[ITEMS];
    uint32_t vreg[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const size_t idx = base + (size_t)r * kSortBlock + threadIdx.x;
        kreg[r] = idx < n ? keys[idx] : (K)0;
        vreg[r] = (HAS_VAL && idx < n) ? vals[idx] : 0u;
    }
    // digit bases: exclusive scan of the 256 row totals
    uint32_t total = 0, earlier = 0;
    if (rowTotal) {
        total = rowTotal[threadIdx.x];
        earlier = offsets[(size_t)threadIdx.x * nblocks + blockIdx.x];
    } else {
        const uint32_t *row = offsets + (size_t)threadIdx.x * nblocks;
#pragma unroll 8
        for (int b = 0; b < nblocks; ++b) {
            const uint32_t v = row[b];
            total += v;
            earlier += b < (int)blockIdx.x ? v : 0u;
        }
    }
    s_base[threadIdx.x] = total;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t v = threadIdx.x >= (unsigned)off ? s_base[threadIdx.x - off] : 0;
        __syncthreads();
        s_base[threadIdx.x] += v;
        __syncthreads();
    }
    const uint32_t digitBase = s_base[threadIdx.x] - total;
    __syncthreads();
    s_base[threadIdx.x] = digitBase + earlier;
    for (int w = 0; w < kWaves; ++w)
        s_wcnt[w][threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const unsigned long long ltmask = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const size_t idx = base + (size_t)r * kSortBlock + threadIdx.x;
        const bool valid = idx < n;
        const K key = kreg[r];
        const uint32_t val = vreg[r];
        const uint32_t d = digit_of(key, shift, mask);
        // lanes of this wave holding the same digit
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const unsigned long long bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t rank = __popcll(peers & ltmask);
        if (valid && rank == 0)
            s_wcnt[wave][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        uint32_t pos = 0;
        if (valid) {
            pos = s_base[d] + rank;
            for (int w = 0; w < wave; ++w)
                pos += s_wcnt[w][d];
        }
        __syncthreads();
        {
            uint32_t tot = 0;
            for (int w = 0; w < kWaves; ++w) {
                tot += s_wcnt[w][threadIdx.x];
                s_wcnt[w][threadIdx.x] = 0;
            }
            s_base[threadIdx.x] += tot;
        }
        __syncthreads();
        if (valid) {
            keysOut[pos] = key;
            if (HAS_VAL)
                valsOut[pos] = val;
        }
    }
}

// A list of (first << 32 | second) keys already sorted by their high word, each run
// of equal high words put in order of the low word: every lane counts the keys of
// its run that come before its own and stores its key at that place of out.  A run
// longer than maxRun goes over as it is and raises *flag (the caller then sorts
// the whole list by both words); so do ~0 keys (padding), without the flag.
// out is a permutation of keys whatever the runs are.
//
// One lane per run, sorting in place, waited for each load in turn: 22 us for the
// candidates of two 655 k-triangle spheres, 9 now, and it was slower than
// radix passes for a batch's longer runs (38 us now).
__global__ __launch_bounds__(256) void k_sort_runs(const uint64_t *__restrict__ keys, uint64_t *__restrict__ out,
                                                   uint32_t n, const uint32_t *__restrict__ count, uint32_t maxRun,
                                                   uint32_t *flag)
{
    n = (uint32_t)sort_len(n, count);
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    const uint64_t k = keys[i];
    const uint32_t hi = (uint32_t)(k >> 32);
    uint32_t back = 0, len = 1, less = 0;
    if (k != ~0ull) {
        // four neighbours at a time, their loads in flight together
        bool more = true;
        while (more && back <= maxRun) {
            uint64_t v[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                v[j] = keys[i > back + j ? i - back - j - 1 : 0];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                more = more && i > back && (uint32_t)(v[j] >> 32) == hi;
                back += more;
                less += more && v[j] < k;
            }
        }
        len += back;
        more = true;
        for (uint32_t x = i + 1; more && len <= maxRun; x += 4) {
            uint64_t v[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                v[j] = keys[x + j < n ? x + j : n - 1];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                more = more && x + j < n && (uint32_t)(v[j] >> 32) == hi;
                len += more;
                less += more && v[j] < k;
            }
        }
    }
    if (len > maxRun) {
        atomicOr(flag, 1u);
        out[i] = k;
        return;
    }
    out[i - back + less] = k;
}

void launch_sort_runs(const uint64_t *keys, uint64_t *out, size_t n, const uint32_t *count, uint32_t maxRun,
                      uint32_t *flag, hipStream_t s)
{
    if (n)
        hipLaunchKernelGGL(k_sort_runs, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, keys, out, (uint32_t)n,
                           count, maxRun, flag);
}

// ---- sorts of one workgroup ---------------------------------------------------
// Short lists: a launch per pass and kernel (3 to 4 us of work each, as much
// again of host time) cost more than the sort.  One workgroup of 16 waves keeps
// the keys in LDS.  Per pass each wave counts the digits of its own run of
// consecutive keys, 256 lanes turn the counts into offsets, and each wave then
// places its run in order, 64 keys a round (ranks by ballots), with no barrier
// between rounds.  A step with / without them, us: 231 / 310 at two 80-triangle
// meshes (the order kernel 9.1 us for 11 launches of 2 to 4.4, the candidates'
// 8.9 for four), 315 / 387 at 1,280, 357 / 436 at 5,120, 360 / 431 at 8,366;
// the limit is what LDS holds.
constexpr int kOneSortWaves = 16;
constexpr uint32_t kOneSortMax = 8192;

// one stable pass over n keys by digit_at(i) from src order to dst order:
// place(i, slot) moves the i-th key.  s_cnt: [kOneSortWaves][256]
template <typename DigitAt, typename Place>
__device__ __forceinline__ void one_sort_pass(uint32_t n, uint32_t (*s_cnt)[256], uint32_t *s_scan,
                                              const DigitAt &digit_at, const Place &place)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t k = tid; k < kOneSortWaves * 256u; k += 64 * kOneSortWaves)
        s_cnt[k >> 8][k & 255] = 0;
    __syncthreads();
    const uint32_t per = ((n + kOneSortWaves - 1) / kOneSortWaves + 63u) & ~63u;  // a wave's run
    const uint32_t first = min(wave * per, n), last = min(first + per, n);
    for (uint32_t i = first + lane; i < last; i += 64)
        atomicAdd(&s_cnt[wave][digit_at(i)], 1u);
    __syncthreads();
    uint32_t total = 0;
    if (tid < 256) {
        for (int w = 0; w < kOneSortWaves; ++w) {
            const uint32_t v = s_cnt[w][tid];
            s_cnt[w][tid] = total;
            total += v;
        }
        s_scan[tid] = total;
    }
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t v = tid < 256 && tid >= (uint32_t)off ? s_scan[tid - off] : 0u;
        __syncthreads();
        if (tid < 256)
            s_scan[tid] += v;
        __syncthreads();
    }
    if (tid < 256) {
        const uint32_t base = s_scan[tid] - total;
        for (int w = 0; w < kOneSortWaves; ++w)
            s_cnt[w][tid] += base;
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    for (uint32_t i0 = first; i0 < last; i0 += 64) {  // uniform over the wave
        const uint32_t i = i0 + lane;
        const bool valid = i < last;
        const uint32_t d = valid ? digit_at(i) : 0u;
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < 8; ++b) {
            const unsigned long long bal = __ballot((d >> b) & 1u);
            peers &= (d >> b) & 1u ? bal : ~bal;
        }
        if (valid) {
            const uint32_t slot = s_cnt[wave][d] + (uint32_t)__popcll(peers & below);
            place(i, slot);
            // the last of the equal ones moves the wave's offset on
            if ((peers >> lane) == 1ull)
                s_cnt[wave][d] = slot + 1u;
        }
        // the next round's lanes read the offsets this round's moved on
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
}

// The tree order of a small mesh in one launch: the centroids' bounds from the
// records kernel's blocks, Morton keys, and their sort; *zero is cleared for
// the tree kernel.
__global__ __launch_bounds__(64 * kOneSortWaves) void k_small_order(const float *__restrict__ box32,
                                                                    const float *__restrict__ blockBounds, int nblocks,
                                                                    uint32_t n, int keyBits, uint32_t *__restrict__ keys,
                                                                    uint32_t *__restrict__ vals,
                                                                    uint32_t *__restrict__ zero)
{
    __shared__ uint32_t s_key[2][kOneSortMax];
    __shared__ uint16_t s_val[2][kOneSortMax];
    __shared__ uint32_t s_cnt[kOneSortWaves][256], s_scan[256];
    __shared__ float s_bounds[6];
    const uint32_t tid = threadIdx.x;
    if (tid < 64) {
        float v[6] = {__builtin_inff(), __builtin_inff(), __builtin_inff(),
                      -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
        for (int b = tid; b < nblocks; b += 64)
            for (int k = 0; k < 6; ++k)
                v[k] = k < 3 ? fminf(v[k], blockBounds[6 * b + k]) : fmaxf(v[k], blockBounds[6 * b + k]);
        for (int off = 32; off > 0; off >>= 1)
            for (int k = 0; k < 6; ++k)
                v[k] = k < 3 ? fminf(v[k], __shfl_xor(v[k], off)) : fmaxf(v[k], __shfl_xor(v[k], off));
        if (tid == 0) {
            for (int k = 0; k < 6; ++k)
                s_bounds[k] = v[k];
            *zero = 0u;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += 64 * kOneSortWaves) {
        s_key[0][i] = morton30(box_centre(box32, i), s_bounds) >> (30 - keyBits);
        s_val[0][i] = (uint16_t)i;
    }
    __syncthreads();
    int from = 0;
    for (int shift = 0; shift < keyBits; shift += 8, from ^= 1)
        one_sort_pass(
            n, s_cnt, s_scan, [&](uint32_t i) { return s_key[from][i] >> shift & 255u; },
            [&](uint32_t i, uint32_t slot) {
                s_key[from ^ 1][slot] = s_key[from][i];
                s_val[from ^ 1][slot] = s_val[from][i];
            });
    for (uint32_t i = tid; i < n; i += 64 * kOneSortWaves) {
        keys[i] = s_key[from][i];
        vals[i] = s_val[from][i];
    }
}

bool small_order(size_t n) { return n <= kOneSortMax; }

void launch_small_order(const float *box32, const float *blockBounds, int nblocks, uint32_t n, uint32_t *keys,
                        uint32_t *vals, uint32_t *zero, hipStream_t s)
{
    if (n)
        hipLaunchKernelGGL(k_small_order, dim3(1), dim3(64 * kOneSortWaves), 0, s, box32, blockBounds, nblocks, n,
                           kMortonBits, keys, vals, zero);
}

// A short candidate list in place, by the first triangle (passes over bits
// [32, 32 + firstBits)) and then each run of equal first triangles by the
// second, as k_sort_runs does.
__global__ __launch_bounds__(64 * kOneSortWaves) void k_small_pairs(uint64_t *keys, uint32_t n,
                                                                    const uint32_t *__restrict__ count, int firstBits,
                                                                    uint32_t maxRun, uint32_t *flag)
{
    __shared__ uint64_t s_key[2][kOneSortMax];
    __shared__ uint32_t s_cnt[kOneSortWaves][256], s_scan[256];
    n = (uint32_t)sort_len(n, count);
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < n; i += 64 * kOneSortWaves)
        s_key[0][i] = keys[i];
    __syncthreads();
    int from = 0;
    for (int shift = 32; shift < 32 + firstBits; shift += 8, from ^= 1)
        one_sort_pass(
            n, s_cnt, s_scan, [&](uint32_t i) { return (uint32_t)(s_key[from][i] >> shift) & 255u; },
            [&](uint32_t i, uint32_t slot) { s_key[from ^ 1][slot] = s_key[from][i]; });
    uint64_t *k = s_key[from];
    for (uint32_t i = tid; i < n; i += 64 * kOneSortWaves) {
        const uint32_t hi = (uint32_t)(k[i] >> 32);
        if (i > 0 && (uint32_t)(k[i - 1] >> 32) == hi)
            continue;
        uint32_t j = i + 1;
        while (j < n && j - i <= maxRun && (uint32_t)(k[j] >> 32) == hi)
            ++j;  // to one past the longest run sorted here
        if (j - i > maxRun) {
            atomicOr(flag, 1u);
            continue;
        }
        for (uint32_t x = i + 1; x < j; ++x) {
            const uint64_t v = k[x];
            uint32_t y = x;
            for (; y > i && k[y - 1] > v; --y)
                k[y] = k[y - 1];
            k[y] = v;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += 64 * kOneSortWaves)
        keys[i] = k[i];
}

void launch_small_pairs(uint64_t *keys, size_t n, const uint32_t *count, int firstBits, uint32_t maxRun,
                        uint32_t *flag, hipStream_t s)
{
    if (n)
        hipLaunchKernelGGL(k_small_pairs, dim3(1), dim3(64 * kOneSortWaves), 0, s, keys, (uint32_t)n, count, firstBits,
                           maxRun, flag);
}

bool small_pairs(size_t n) { return n <= kOneSortMax; }

void launch_exclusive_scan(uint32_t *data, size_t m, hipStream_t s)
{
    if (m == 0)
        return;
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, data, m);
}

int sort_blocks(size_t n)
{
    const size_t tile = (size_t)kSortBlock * sort_items(n);
    return (int)((n + tile - 1) / tile);
}
// 256 x nblocks histogram + 256 row totals
size_t sort_hist_entries(size_t n) { return (size_t)256 * (size_t)(sort_blocks(n) > 0 ? sort_blocks(n) : 1) + 256; }

template <typename K, bool HAS_VAL>
static void one_pass(const K *kin, const uint32_t *vin, K *kout, uint32_t *vout, size_t n, const uint32_t *count,
                     int shift, int bits, uint32_t *hist, hipStream_t s)
{
    const int nb = sort_blocks(n);
    const uint32_t mask = (1u << bits) - 1u;
    uint32_t *rowTotal = hist + (size_t)256 * nb;
    const int items = sort_items(n);
    if (items == 16)
        hipLaunchKernelGGL((k_hist<K, 16>), dim3(nb), dim3(kSortBlock), 0, s, kin, n, count, shift, mask, hist, nb);
    else if (items == 8)
        hipLaunchKernelGGL((k_hist<K, 8>), dim3(nb), dim3(kSortBlock), 0, s, kin, n, count, shift, mask, hist, nb);
    else
        hipLaunchKernelGGL((k_hist<K, 4>), dim3(nb), dim3(kSortBlock), 0, s, kin, n, count, shift, mask, hist, nb);
    if (nb <= kScanInScatter)
        rowTotal = nullptr;
    else
        hipLaunchKernelGGL(k_scan_rows, dim3(256), dim3(256), 0, s, hist, nb, rowTotal);
    if (items == 16)
        hipLaunchKernelGGL((k_scatter<K, HAS_VAL, 16>), dim3(nb), dim3(kSortBlock), 0, s, kin, vin, kout, vout, n,
                           count, shift, mask, hist, nb, rowTotal);
    else if (items == 8)
        hipLaunchKernelGGL((k_scatter<K, HAS_VAL, 8>), dim3(nb), dim3(kSortBlock), 0, s, kin, vin, kout, vout, n,
                           count, shift, mask, hist, nb, rowTotal);
    else
        hipLaunchKernelGGL((k_scatter<K, HAS_VAL, 4>), dim3(nb), dim3(kSortBlock), 0, s, kin, vin, kout, vout, n,
                           count, shift, mask, hist, nb, rowTotal);
}

int radix_sort_u32(uint32_t *keys, uint32_t *vals, uint32_t *keysAlt, uint32_t *valsAlt, size_t n,
                   int beginBit, int endBit, uint32_t *hist, hipStream_t s)
{
    if (n <= 1)
        return 0;
    int flip = 0;
    for (int shift = beginBit; shift < endBit; shift += 8) {
        const int bits = endBit - shift < 8 ? endBit - shift : 8;
        uint32_t *ki = flip ? keysAlt : keys, *ko = flip ? keys : keysAlt;
        uint32_t *vi = flip ? valsAlt : vals, *vo = flip ? vals : valsAlt;
        if (vals)
            one_pass<uint32_t, true>(ki, vi, ko, vo, n, nullptr, shift, bits, hist, s);
        else
            one_pass<uint32_t, false>(ki, nullptr, ko, nullptr, n, nullptr, shift, bits, hist, s);
        flip ^= 1;
    }
    return flip;
}

int radix_sort_u64(uint64_t *keys, uint64_t *keysAlt, size_t n, const int *bitRanges, int nRanges,
                   uint32_t *hist, hipStream_t s, const uint32_t *count)
{
    if (n <= 1)
        return 0;
    int flip = 0;
    for (int r = 0; r < nRanges; ++r) {
        const int beginBit = bitRanges[2 * r], endBit = bitRanges[2 * r + 1];
        for (int shift = beginBit; shift < endBit; shift += 8) {
            const int bits = endBit - shift < 8 ? endBit - shift : 8;
            uint64_t *ki = flip ? keysAlt : keys, *ko = flip ? keys : keysAlt;
            one_pass<uint64_t, false>(ki, nullptr, ko, nullptr, n, count, shift, bits, hist, s);
            flip ^= 1;
        }
    }
    return flip;
}

}  // namespace sbg
