// Lookup permutation pair (permuted input, permuted table) on the device,
// behind the reference's entry point cuda/src/commitment/permute_expression_pair.cu
// (culib.rs:127-141); the result matches permute_expression_pair_seq of
// src/plonk/lookup/prover.rs byte for byte:
//   permuted_input = sort(input[0, U)) under Fr's order (canonical value);
//   at the first row of each run of equal inputs, permuted_table = that value
//   (one table occurrence consumed); the leftover table multiset, ascending,
//   fills the remaining rows from the last one backwards; rows [U, n) are zero.
//
// Sorting: 256-bit canonical keys, merge sort — a tile of 8192 keys is sorted
// in LDS by 51-bit windows of the keys (tile_sort_kernel), then
// global merge passes, each work-group merging one 2048-key output tile found
// by a merge-path split. Both arrays (input, table) are sorted by the same
// launches (grid y). Then: not-head flags over the sorted input, leftover flags
// over the sorted table (a table run head whose value occurs in the input is
// consumed), two scans, and one output pass that pairs the r-th repeated row
// with leftover m - 1 - r.
#include "common.h"
#include "field.h"
#include "scan_u32.h"

using namespace h2;

namespace {

constexpr unsigned kThreads = 256; // element-wise kernels
constexpr unsigned kTile = 2048; // keys per merge work-group, 64 KB of LDS
constexpr unsigned kSortTile = 8192; // keys per sorted tile: 64 KB of windows, 16 KB of indices

struct Key {
    uint64_t w[4]; // canonical value, little-endian 64-bit words
};

__device__ __forceinline__ Key key_load(const Key* p)
{
    const uint4* q = (const uint4*)p;
    const uint4 a = q[0], b = q[1];
    Key k;
    k.w[0] = ((uint64_t)a.y << 32) | a.x;
    k.w[1] = ((uint64_t)a.w << 32) | a.z;
    k.w[2] = ((uint64_t)b.y << 32) | b.x;
    k.w[3] = ((uint64_t)b.w << 32) | b.z;
    return k;
}

__device__ __forceinline__ void key_store(Key* p, const Key& k)
{
    uint4* q = (uint4*)p;
    q[0] = make_uint4((uint32_t)k.w[0], (uint32_t)(k.w[0] >> 32), (uint32_t)k.w[1], (uint32_t)(k.w[1] >> 32));
    q[1] = make_uint4((uint32_t)k.w[2], (uint32_t)(k.w[2] >> 32), (uint32_t)k.w[3], (uint32_t)(k.w[3] >> 32));
}

// a < b as 256-bit integers (most significant word first)
__device__ __forceinline__ bool key_lt(const Key& a, const Key& b)
{
    if (a.w[3] != b.w[3])
        return a.w[3] < b.w[3];
    if (a.w[2] != b.w[2])
        return a.w[2] < b.w[2];
    if (a.w[1] != b.w[1])
        return a.w[1] < b.w[1];
    return a.w[0] < b.w[0];
}

__device__ __forceinline__ bool key_eq(const Key& a, const Key& b)
{
    return ((a.w[0] ^ b.w[0]) | (a.w[1] ^ b.w[1]) | (a.w[2] ^ b.w[2]) | (a.w[3] ^ b.w[3])) == 0;
}

__device__ __forceinline__ Key key_max()
{
    Key k;
    k.w[0] = k.w[1] = k.w[2] = k.w[3] = ~0ull; // above every canonical value (< r < 2^254)
    return k;
}

__device__ __forceinline__ Key key_from_fr(const Fr& v)
{
    Key k;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        k.w[i] = ((uint64_t)v.v[2 * i + 1] << 32) | v.v[2 * i];
    return k;
}

__device__ __forceinline__ Fr fr_from_key(const Key& k)
{
    Fr v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v.v[2 * i] = (uint32_t)k.w[i];
        v.v[2 * i + 1] = (uint32_t)(k.w[i] >> 32);
    }
    return v;
}

// Number of elements taken from A among the first `diag` outputs of the
// stable merge of A (length na) and B (length nb); ties go to A.
template <class GetA, class GetB>
__device__ __forceinline__ uint64_t merge_path(uint64_t na, uint64_t nb, uint64_t diag, GetA getA, GetB getB)
{
    uint64_t lo = diag > nb ? diag - nb : 0;
    uint64_t hi = diag < na ? diag : na;
    while (lo < hi) {
        const uint64_t mid = (lo + hi) >> 1;
        if (!key_lt(getB(diag - 1 - mid), getA(mid)))
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// Merges up to P outputs starting at diagonal `diag` of A|B held in LDS.
template <unsigned P>
__device__ __forceinline__ void merge_run(const Key* A, uint32_t na, const Key* B, uint32_t nb, uint32_t diag,
    Key* out)
{
    const uint32_t i0 = (uint32_t)merge_path(na, nb, diag, [A](uint64_t k) { return A[k]; },
        [B](uint64_t k) { return B[k]; });
    uint32_t i = i0, j = diag - i0;
    const uint32_t total = na + nb;
#pragma unroll
    for (unsigned k = 0; k < P; ++k) {
        if (diag + k < total) {
            const bool takeA = j >= nb || (i < na && !key_lt(B[j], A[i]));
            out[k] = takeA ? A[i] : B[j];
            if (takeA)
                ++i;
            else
                ++j;
        }
    }
}

// Sorts each 8192-key tile of keys[y * stride + (0, U)) into out.
//
// What is sorted is not the 32-byte keys but 64-bit words of 51 key bits and the key's 13-bit
// place in the tile, four times less to move through LDS and registers; the keys themselves
// are read where they lie and written once, in order. Which 51 bits:
//  - the tile's keys differ in 51 bits at most: those, and the order is complete;
//  - otherwise the window below the highest bit in which they differ. Neighbours that agree in it
//    are then compared; for uniform keys they are equal but for 2^-26 a tile;
//  - if a look at neighbouring keys before the sort shows a window that ties (signed small numbers:
//    m - x and x share all of it), the bits that tell keys apart. The highest bit in which two
//    keys differ, for every two neighbours of a sorted order, is enough to compare any two keys;
//    neighbours of an unsorted order give most of these bits, and the ones right below them, as
//    far as 51 reach, the rest. The order is checked as the keys are written;
//  - if there are too many such bits, the keys' lengths vary (powers of two, say): the length and
//    the 43 bits below the highest one.
// Keys that a window or a length leaves tied go through further rounds of their rank so far and 38
// of the bits in which tied keys differ.
// Words are sorted 8 per thread in registers, then in ten merge rounds.
// 2^20 rows of two columns: 213 us with keys as the words and 2048 a tile, now 88, and two
// merge passes of 38 us less. The whole call for signed numbers, 2^10, 2^16 and 2^20 rows: 92,
// 188, 713 us with keys as the words, now 75, 158, 639 (263, 360, 754 if a tile that ties in its
// window goes through all of them); for powers of two 91, 183, 678 and now 73, 164, 528. Keys that
// need a second round (40 lengths with more than 43 bits below) take longer on few rows: 88, 175,
// 669 and now 120, 218, 595.
constexpr unsigned kSortThreads = 1024;
constexpr unsigned kSortPer = kSortTile / kSortThreads;
constexpr unsigned kIndexBits = 13;
constexpr unsigned kWindow = 64 - kIndexBits;
constexpr uint32_t kIndexMask = kSortTile - 1;

// bits [shift, shift + 51) of a key in memory
__device__ __forceinline__ uint64_t key_window(const Key* p, uint32_t shift)
{
    const uint32_t q = shift >> 6, sh = shift & 63;
    uint64_t v = p->w[q] >> sh;
    if (sh && q < 3)
        v |= p->w[q + 1] << (64 - sh);
    return v & ((1ull << kWindow) - 1);
}

// sorts sh[0, kSortTile): all the words are different
__device__ __forceinline__ void sort_words(uint64_t* sh)
{
    const uint32_t d = threadIdx.x * kSortPer;
    uint64_t r[kSortPer];
    __syncthreads();
#pragma unroll
    for (unsigned k = 0; k < kSortPer; ++k)
        r[k] = sh[d + k];
    // odd-even transposition sort of the thread's words in registers
#pragma unroll
    for (unsigned phase = 0; phase < kSortPer; ++phase) {
#pragma unroll
        for (unsigned k = phase & 1; k + 1 < kSortPer; k += 2) {
            const uint64_t a = r[k], b = r[k + 1];
            r[k] = a < b ? a : b;
            r[k + 1] = a < b ? b : a;
        }
    }
    for (uint32_t w = kSortPer; w < kSortTile; w <<= 1) {
        __syncthreads();
#pragma unroll
        for (unsigned k = 0; k < kSortPer; ++k)
            sh[d + k] = r[k];
        __syncthreads();
        const uint32_t p = d & ~(2 * w - 1), diag = d - p;
        const uint64_t* A = sh + p;
        const uint64_t* B = A + w;
        uint32_t lo = diag > w ? diag - w : 0, hi = diag < w ? diag : w;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (A[mid] < B[diag - 1 - mid])
                lo = mid + 1;
            else
                hi = mid;
        }
        uint32_t i = lo, j = diag - lo;
        uint64_t a = i < w ? A[i] : ~0ull, b = j < w ? B[j] : ~0ull;
#pragma unroll
        for (unsigned k = 0; k < kSortPer; ++k) {
            const bool takeA = j >= w || (i < w && a < b);
            r[k] = takeA ? a : b;
            if (takeA) {
                ++i;
                a = i < w ? A[i] : ~0ull;
            } else {
                ++j;
                b = j < w ? B[j] : ~0ull;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (unsigned k = 0; k < kSortPer; ++k)
        sh[d + k] = r[k];
    __syncthreads();
}

// A choice of at most 51 key bits as runs within the key's words, highest first:
// word << 16 | lowest bit << 8 | bits
struct BitRuns {
    uint32_t count;
    uint32_t run[kWindow];
};

__device__ inline void set_runs(BitRuns& runs, const uint64_t (&mask)[4])
{
    uint32_t n = 0;
    for (int q = 3; q >= 0; --q) {
        uint64_t m = mask[q];
        while (m) {
            const uint32_t top = 63 - __builtin_clzll(m);
            const uint64_t holes = ~(m << (63 - top));
            const uint32_t bits = holes ? __builtin_clzll(holes) : 64;
            const uint32_t low = top + 1 - bits;
            runs.run[n++] = (uint32_t)q << 16 | low << 8 | bits;
            m &= (1ull << low) - 1;
        }
    }
    runs.count = n;
}

// m |= m >> n, 0 < n < 64
__device__ __forceinline__ void or_shifted(uint64_t (&m)[4], uint32_t n)
{
#pragma unroll
    for (int q = 0; q < 3; ++q)
        m[q] |= m[q] >> n | m[q + 1] << (64 - n);
    m[3] |= m[3] >> n;
}

__device__ __forceinline__ uint32_t bits_set(const uint64_t (&m)[4])
{
    return __popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]) + __popcll(m[3]);
}

// a place 1 to 8 after k, by turns of no regular period (columns often interleave a few sequences)
__device__ __forceinline__ uint32_t near_to(uint32_t k, uint32_t count)
{
    const uint32_t other = k + 1 + ((k * 0x9e3779b1u) >> 29);
    return other < count ? other : count - 1;
}

// the words of the tile's keys by a choice of bits, below their ranks (if any)
__device__ __forceinline__ void words_by_runs(uint64_t* sh, const Key* __restrict__ src, uint32_t count,
    const BitRuns& runs, const uint16_t* rank = nullptr)
{
    uint64_t v[kSortPer];
#pragma unroll
    for (unsigned k = 0; k < kSortPer; ++k)
        v[k] = rank ? rank[threadIdx.x + k * kSortThreads] : 0;
    const uint32_t n = runs.count;
    for (uint32_t i = 0; i < n;) {
        const uint32_t q = __builtin_amdgcn_readfirstlane(runs.run[i]) >> 16;
        uint64_t w[kSortPer];
#pragma unroll
        for (unsigned k = 0; k < kSortPer; ++k) {
            const uint32_t at = threadIdx.x + k * kSortThreads;
            w[k] = at < count ? src[at].w[q] : 0;
        }
        for (; i < n; ++i) { // the runs within word q
            const uint32_t e = __builtin_amdgcn_readfirstlane(runs.run[i]);
            if (e >> 16 != q)
                break;
            const uint32_t low = (e >> 8) & 255, bits = e & 255;
#pragma unroll
            for (unsigned k = 0; k < kSortPer; ++k)
                v[k] = v[k] << bits | ((w[k] >> low) & ((1ull << bits) - 1));
        }
    }
#pragma unroll
    for (unsigned k = 0; k < kSortPer; ++k) {
        const uint32_t at = threadIdx.x + k * kSortThreads;
        sh[at] = (at < count ? v[k] : (1ull << kWindow) - 1) << kIndexBits | at;
    }
}

// the words by the window from bit `shift` up
__device__ __forceinline__ void words_by_window(uint64_t* sh, const Key* __restrict__ src, uint32_t count, uint32_t shift)
{
    for (uint32_t k = threadIdx.x; k < kSortTile; k += kSortThreads)
        sh[k] = (k < count ? key_window(src + k, shift) : (1ull << kWindow) - 1) << kIndexBits | k;
}

// the words by length (8 bits) and the 43 bits below the highest set one
__device__ __forceinline__ void words_by_length(uint64_t* sh, const Key* __restrict__ src, uint32_t count)
{
    for (uint32_t k = threadIdx.x; k < kSortTile; k += kSortThreads) {
        uint64_t v = (1ull << kWindow) - 1;
        if (k < count) {
            const Key x = key_load(src + k);
            uint64_t top = x.w[0], below = 0, words = 0;
#pragma unroll
            for (int q = 1; q < 4; ++q)
                if (x.w[q]) {
                    top = x.w[q];
                    below = x.w[q - 1];
                    words = q;
                }
            const uint32_t zeros = top ? __builtin_clzll(top) : 64;
            if (zeros < 64 && zeros)
                top = top << zeros | below >> (64 - zeros);
            v = (64 * (words + 1) - zeros) << 43 | (top << 1) >> 21;
        }
        sh[k] = v << kIndexBits | k;
    }
}

__global__ void __launch_bounds__(kSortThreads) tile_sort_kernel(const Key* __restrict__ keys,
    Key* __restrict__ out, uint64_t U, uint64_t stride)
{
    __shared__ uint64_t sh[kSortTile];
    __shared__ uint16_t rank[kSortTile];
    __shared__ unsigned long long differ[4]; // bits in which the keys differ
    __shared__ unsigned long long tell[4]; // highest differing bits of neighbours; bits in which tied keys differ
    __shared__ uint32_t last_head[kSortThreads / 64];
    __shared__ uint32_t ties, misplaced;
    __shared__ BitRuns runs;
    const uint64_t base = (uint64_t)blockIdx.x * kSortTile;
    const Key* src = keys + blockIdx.y * stride + base;
    Key* dst = out + blockIdx.y * stride + base;
    const uint32_t count = U - base < kSortTile ? (uint32_t)(U - base) : kSortTile;
    const uint32_t t = threadIdx.x, lane = t & 63;
    if (t < 4) {
        differ[t] = 0;
        tell[t] = 0;
    }
    if (t == 0)
        ties = misplaced = 0;
    __syncthreads();
    // into[q] |= x[q] of all threads
    auto gather = [lane](unsigned long long* into, uint64_t (&x)[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            for (int d = 32; d; d >>= 1)
                x[q] |= __shfl_xor(x[q], d, 64);
            if (lane == 0 && x[q])
                atomicOr(&into[q], (unsigned long long)x[q]);
        }
    };
    const Key first = key_load(src);
    uint64_t x[4] = { 0, 0, 0, 0 };
    for (uint32_t k = t; k < count; k += kSortThreads) {
        const Key v = key_load(src + k);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            x[q] |= v.w[q] ^ first.w[q];
    }
    gather(differ, x);
    __syncthreads();
    uint32_t bits = 0; // the keys differ in bits below this one only
    for (int q = 3; q >= 0 && !bits; --q)
        if (differ[q])
            bits = 64 * q + 64 - __builtin_clzll(differ[q]);
    const uint32_t shift = bits > kWindow ? bits - kWindow : 0;
    const uint64_t all[4] = { differ[0], differ[1], differ[2], differ[3] };
    const bool few = bits_set(all) <= kWindow;

    // Chooses the bits that tell neighbouring keys apart and the ones below them; false if they
    // are too many.
    auto choose = [&]() -> bool {
        uint64_t y[4] = { 0, 0, 0, 0 };
        for (uint32_t k = t; k + 1 < count; k += kSortThreads) {
            const Key a = key_load(src + k);
#pragma unroll
            for (uint32_t pair = 0; pair < 3; ++pair) { // the next one, the one after it, one near
                const uint32_t other = pair == 0 ? k + 1 : pair == 1 ? k + 2 : near_to(k, count);
                if (other >= count)
                    break;
                const Key b = key_load(src + other);
                bool above = false;
#pragma unroll
                for (int q = 3; q >= 0; --q) {
                    const uint64_t e = above ? 0 : a.w[q] ^ b.w[q];
                    y[q] |= e ? 1ull << (63 - __builtin_clzll(e)) : 0;
                    above = above || e;
                }
            }
        }
        gather(tell, y);
        __syncthreads();
        uint64_t m[4] = { tell[0], tell[1], tell[2], tell[3] };
        const bool fits = bits_set(m) <= kWindow - 13; // leaves some to the bits below them
        if (fits && t < 64) { // lane e: the bits and the e below each; the most that fit are taken
            uint32_t w = 1;
            for (; 2 * w <= t + 1; w *= 2)
                or_shifted(m, w);
            if (w < t + 1)
                or_shifted(m, t + 1 - w);
            if (63u - __builtin_clzll(__ballot(bits_set(m) <= kWindow)) == t)
                set_runs(runs, m);
        }
        __syncthreads();
        if (t < 4)
            tell[t] = 0;
        return fits;
    };

    // The tile's keys in the words' order; with `check` a key below the one before it sets `misplaced`.
    auto write = [&](bool check) {
        for (uint32_t k = t; k < kSortTile; k += kSortThreads) {
            Key v {}, before {};
            if (k < count)
                v = key_load(src + (sh[k] & kIndexMask));
            if (check) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    before.w[q] = __shfl_up(v.w[q], 1, 64);
                if (lane == 0 && k && k < count)
                    before = key_load(src + (sh[k - 1] & kIndexMask));
                if (k && k < count && key_lt(v, before))
                    misplaced = 1;
            }
            if (k < count)
                key_store(dst + k, v);
        }
    };

    // padding sorts last: its words have every window bit set, and its places are past the keys'
    if (shift && few) {
        if (t == 0)
            set_runs(runs, all);
        __syncthreads();
        words_by_runs(sh, src, count, runs);
    } else {
        words_by_window(sh, src, count, shift);
    }
    if (shift && !few) {
        __syncthreads();
        for (uint32_t k = t; k + 1 < count; k += kSortThreads) {
            const uint32_t other = near_to(k, count);
            if ((sh[k] ^ sh[other]) >> kIndexBits == 0 && !key_eq(key_load(src + k), key_load(src + other)))
                ties = 1;
        }
        __syncthreads();
        if (ties) { // the same for the whole work-group
            if (choose()) {
                words_by_runs(sh, src, count, runs);
                sort_words(sh);
                write(true);
                __syncthreads();
                if (!misplaced)
                    return;
                words_by_window(sh, src, count, shift);
            } else {
                words_by_length(sh, src, count);
            }
        }
    }
    sort_words(sh);
    // The words' bits are in the keys' order now, but keys may share them: the words of the next round
    // are the place of the first key of each such group and the highest 38 bits in which keys of
    // a group differ.
    for (bool exact = few || shift == 0; !exact;) {
        uint64_t y[4] = { 0, 0, 0, 0 };
        for (uint32_t k = t; k + 1 < count; k += kSortThreads) {
            const uint64_t a = sh[k], b = sh[k + 1];
            if ((a ^ b) >> kIndexBits)
                continue;
            const Key ka = key_load(src + (a & kIndexMask)), kb = key_load(src + (b & kIndexMask));
#pragma unroll
            for (int q = 0; q < 4; ++q)
                y[q] |= ka.w[q] ^ kb.w[q];
        }
        if (__any((y[0] | y[1] | y[2] | y[3]) != 0))
            gather(tell, y);
        __syncthreads();
        uint64_t m[4] = { tell[0], tell[1], tell[2], tell[3] };
        if (bits_set(m) == 0)
            break;
        exact = bits_set(m) <= kWindow - kIndexBits;
        uint32_t head = 0; // of the group that the thread's 8 words end in, then of all before them
#pragma unroll
        for (unsigned k = 0; k < kSortPer; ++k) {
            const uint32_t at = t * kSortPer + k;
            if (at && (sh[at] ^ sh[at - 1]) >> kIndexBits)
                head = at;
        }
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t h = __shfl_up(head, d, 64);
            head = lane >= (uint32_t)d && h > head ? h : head;
        }
        if (lane == 63)
            last_head[t >> 6] = head;
        head = __shfl_up(head, 1, 64);
        if (lane == 0)
            head = 0;
        __syncthreads();
        for (uint32_t w = 0; w < t >> 6; ++w)
            head = last_head[w] > head ? last_head[w] : head;
#pragma unroll
        for (unsigned k = 0; k < kSortPer; ++k) {
            const uint32_t at = t * kSortPer + k;
            if (at && (sh[at] ^ sh[at - 1]) >> kIndexBits)
                head = at;
            rank[sh[at] & kIndexMask] = (uint16_t)head;
        }
        if (t == 0) {
            for (int q = 0; q < 4; ++q) // the lowest bits go
                while (m[q] && bits_set(m) > kWindow - kIndexBits)
                    m[q] &= m[q] - 1;
            set_runs(runs, m);
        }
        __syncthreads();
        if (t < 4)
            tell[t] = 0;
        words_by_runs(sh, src, count, runs, rank);
        sort_words(sh);
    }
    write(false);
}

// Geometry of output tile `tile` in a merge pass over runs of length w: the
// pair of runs it falls in (A at `pair`, B after it) and its diagonal range.
struct TileSpan {
    uint64_t pair, na, nb, d0, d1;
};

__device__ __forceinline__ TileSpan tile_span(uint64_t tile, uint64_t U, uint64_t w)
{
    TileSpan t;
    const uint64_t g0 = tile * kTile;
    t.pair = g0 / (2 * w) * (2 * w);
    const uint64_t rest = U - t.pair;
    t.na = rest < w ? rest : w;
    t.nb = rest > w ? (rest - w < w ? rest - w : w) : 0;
    t.d0 = g0 - t.pair;
    t.d1 = t.d0 + kTile < t.na + t.nb ? t.d0 + kTile : t.na + t.nb;
    return t;
}

// Merge-path split: the number of keys that the first d outputs of a pair of runs take from run
// A. The wave narrows the range with 64 probes per round (a 64-ary search), so a run of 2^21
// keys takes four rounds of dependent loads instead of 21.
__device__ __forceinline__ uint64_t wave_split(const Key* A, const Key* B, uint64_t na, uint64_t nb, uint64_t d,
    uint32_t lane)
{
    // first i in [lo, hi) with B[d - 1 - i] < A[i] (ties go to A), else hi
    uint64_t lo = d > nb ? d - nb : 0;
    uint64_t hi = d < na ? d : na;
    while (lo < hi) {
        const uint64_t step = (hi - lo + 63) >> 6;
        const uint64_t i = lo + lane * step;
        const bool p = i < hi && !key_lt(key_load(B + (d - 1 - i)), key_load(A + i));
        const uint32_t c = (uint32_t)__popcll(__ballot(p)); // the predicate holds on a prefix of the probes
        if (c == 0) {
            hi = lo;
        } else {
            const uint64_t first_false = lo + c * step;
            lo = lo + (c - 1) * step + 1;
            if (first_false < hi)
                hi = first_false;
        }
    }
    return lo;
}

// One merge pass: runs of length w (sorted) merged pairwise into runs of 2w,
// 2048 outputs per work-group of 1024 threads (two each). Two waves find the tile's splits
// while the other work-group of the compute unit loads or merges: a launch of its own for
// the splits took 8 us a pass beside 31 for the merge at 2^20 keys, the two together take 36.
constexpr unsigned kMergeThreads = 1024;
constexpr unsigned kMergePer = kTile / kMergeThreads;

__global__ void __launch_bounds__(kMergeThreads) merge_pass_kernel(const Key* __restrict__ keys,
    Key* __restrict__ out, uint64_t U, uint64_t stride, uint64_t w)
{
    __shared__ Key sh[kTile];
    const Key* src = keys + blockIdx.y * stride;
    Key* dst = out + blockIdx.y * stride;
    const TileSpan ts = tile_span(blockIdx.x, U, w);
    const Key* A = src + ts.pair;
    const Key* B = A + ts.na;
    __shared__ uint64_t sp[2];
    if (threadIdx.x < 128) { // wave 0: first output, wave 1: one past the last
        const uint64_t i = wave_split(A, B, ts.na, ts.nb, threadIdx.x < 64 ? ts.d0 : ts.d1, threadIdx.x & 63u);
        if ((threadIdx.x & 63u) == 0)
            sp[threadIdx.x >> 6] = i;
    }
    __syncthreads();
    const uint64_t a0 = sp[0], a1 = sp[1];
    const uint64_t b0 = ts.d0 - a0, b1 = ts.d1 - a1;
    const uint32_t ta = (uint32_t)(a1 - a0), tb = (uint32_t)(b1 - b0);
    const uint32_t t = threadIdx.x;
    for (uint32_t k = t; k < ta + tb; k += kMergeThreads)
        sh[k] = k < ta ? key_load(A + a0 + k) : key_load(B + b0 + (k - ta));
    __syncthreads();
    Key r[kMergePer];
#pragma unroll
    for (unsigned k = 0; k < kMergePer; ++k)
        r[k] = key_max();
    const uint32_t d = t * kMergePer;
    const uint32_t total = ta + tb;
    merge_run<kMergePer>(sh, ta, sh + ta, tb, d < total ? d : total, r);
    __syncthreads();
#pragma unroll
    for (unsigned k = 0; k < kMergePer; ++k)
        if (d + k < total)
            sh[d + k] = r[k];
    __syncthreads();
    const uint64_t g0 = (uint64_t)blockIdx.x * kTile;
    for (uint32_t k = t; k < ta + tb; k += kMergeThreads)
        key_store(dst + g0 + k, sh[k]);
}

// keys[i] = canonical(input[i]), keys[stride + i] = canonical(table[i]), i < U
__global__ void canonical_keys_kernel(const Fr* __restrict__ input, const Fr* __restrict__ table, Key* __restrict__ keys,
    uint64_t U, uint64_t stride)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= U)
        return;
    key_store(keys + i, key_from_fr(Fr::from_mont(Fr::load(input + i))));
    key_store(keys + stride + i, key_from_fr(Fr::from_mont(Fr::load(table + i))));
}

__device__ bool sorted_contains(const Key* __restrict__ sorted, uint64_t n, const Key& x)
{
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
        const uint64_t mid = (lo + hi) >> 1;
        if (key_lt(key_load(sorted + mid), x))
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo < n && key_eq(key_load(sorted + lo), x);
}

// repeat[i] = 1 when sorted input row i repeats row i - 1; leftover[j] = 0 when
// sorted table row j starts a run whose value occurs in the input
__global__ void flags_kernel(const Key* __restrict__ sin, const Key* __restrict__ stab, uint32_t* __restrict__ repeat,
    uint32_t* __restrict__ leftover, uint64_t U)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= U)
        return;
    repeat[i] = (i > 0 && key_eq(key_load(sin + i), key_load(sin + i - 1))) ? 1u : 0u;
    const Key v = key_load(stab + i);
    const bool head = i == 0 || !key_eq(v, key_load(stab + i - 1));
    leftover[i] = (head && sorted_contains(sin, U, v)) ? 0u : 1u;
}

__global__ void leftover_compact_kernel(const Key* __restrict__ stab, const uint32_t* __restrict__ leftover,
    const uint32_t* __restrict__ lpos, Key* __restrict__ out, uint64_t U)
{
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < U && leftover[j])
        key_store(out + lpos[j], key_load(stab + j));
}

__global__ void permute_output_kernel(const Key* __restrict__ sin, const uint32_t* __restrict__ repeat,
    const uint32_t* __restrict__ rpos, const Key* __restrict__ left, const uint32_t* __restrict__ lpos_total,
    Fr* __restrict__ pin, Fr* __restrict__ ptab, uint64_t U, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    if (i >= U) {
        Fr::zero().store(pin + i);
        Fr::zero().store(ptab + i);
        return;
    }
    const Fr v = Fr::to_mont(fr_from_key(key_load(sin + i)));
    v.store(pin + i);
    if (!repeat[i]) {
        v.store(ptab + i);
        return;
    }
    // the r-th repeated row (r = rpos[i]) takes leftover m - 1 - r; with an input
    // that is not a sub-multiset of the table the counts differ and rows without a
    // leftover stay zero
    const int64_t idx = (int64_t)*lpos_total - 1 - (int64_t)rpos[i];
    (idx >= 0 ? Fr::to_mont(fr_from_key(key_load(left + idx))) : Fr::zero()).store(ptab + i);
}

struct PermBufs {
    Key* keys[2];
    uint32_t* repeat;
    uint32_t* leftover;
    uint32_t* rpos;
    uint32_t* lpos;
    void* scan;
};

template <class WS>
PermBufs perm_carve(WS& ws, uint64_t U)
{
    PermBufs b;
    b.keys[0] = (Key*)ws.take(2 * 32 * U);
    b.keys[1] = (Key*)ws.take(2 * 32 * U);
    b.repeat = (uint32_t*)ws.take(4 * U);
    b.leftover = (uint32_t*)ws.take(4 * U);
    b.rpos = (uint32_t*)ws.take(4 * (U + 1));
    b.lpos = (uint32_t*)ws.take(4 * (U + 1));
    b.scan = ws.take(scan_u32_scratch(U));
    return b;
}

struct PermSizer {
    WorkspaceSizer s;
    void* take(uint64_t n)
    {
        s.take(n);
        return nullptr;
    }
};

unsigned blocks_for(uint64_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

} // namespace

extern "C" {

uint64_t _halo2_permute_expression_pair_workspace_size(uint64_t n, uint64_t usable_rows)
{
    (void)n;
    if (usable_rows == 0)
        return 0;
    PermSizer z;
    perm_carve(z, usable_rows);
    return z.s.bytes + 256;
}

RustError _halo2_permute_expression_pair(const void* d_compressed_input, const void* d_compressed_table,
    void* d_permuted_input, void* d_permuted_table, uint64_t n, uint64_t usable_rows, void* scratch,
    uint64_t scratch_bytes, void* stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    if (n == 0)
        return ok();
    const uint64_t U = usable_rows;
    H2_CHECK_ARG(U <= n, "_halo2_permute_expression_pair: usable_rows %lu > n %lu", (unsigned long)U,
        (unsigned long)n);
    H2_CHECK_ARG(U < (1ull << 32), "_halo2_permute_expression_pair: usable_rows must fit 32 bits");
    Workspace ws(scratch, scratch_bytes);
    PermBufs b {};
    if (U) {
        b = perm_carve(ws, U);
        if (ws.overflow)
            return fail((int)hipErrorInvalidValue, "_halo2_permute_expression_pair: workspace of %lu bytes is too small",
                (unsigned long)scratch_bytes);
    }
    if (U) {
        canonical_keys_kernel<<<blocks_for(U, kThreads), kThreads, 0, stream>>>((const Fr*)d_compressed_input,
            (const Fr*)d_compressed_table, b.keys[0], U, U);
        H2_LAUNCH_CHECK();
        const unsigned tiles = blocks_for(U, kTile);
        tile_sort_kernel<<<dim3(blocks_for(U, kSortTile), 2), kSortThreads, 0, stream>>>(b.keys[0], b.keys[1], U, U);
        H2_LAUNCH_CHECK();
        int cur = 1;
        for (uint64_t w = kSortTile; w < U; w <<= 1) {
            merge_pass_kernel<<<dim3(tiles, 2), kMergeThreads, 0, stream>>>(b.keys[cur], b.keys[cur ^ 1], U, U, w);
            H2_LAUNCH_CHECK();
            cur ^= 1;
        }
        const Key* sin = b.keys[cur];
        const Key* stab = b.keys[cur] + U;
        Key* left = b.keys[cur ^ 1];
        flags_kernel<<<blocks_for(U, kThreads), kThreads, 0, stream>>>(sin, stab, b.repeat, b.leftover, U);
        H2_LAUNCH_CHECK();
        RustError e = scan_u32_exclusive(b.repeat, b.rpos, U, b.scan, stream);
        if (e.code)
            return e;
        e = scan_u32_exclusive(b.leftover, b.lpos, U, b.scan, stream);
        if (e.code)
            return e;
        leftover_compact_kernel<<<blocks_for(U, kThreads), kThreads, 0, stream>>>(stab, b.leftover, b.lpos, left, U);
        H2_LAUNCH_CHECK();
        permute_output_kernel<<<blocks_for(n, kThreads), kThreads, 0, stream>>>(sin, b.repeat, b.rpos, left,
            b.lpos + U, (Fr*)d_permuted_input, (Fr*)d_permuted_table, U, n);
        H2_LAUNCH_CHECK();
    } else {
        permute_output_kernel<<<blocks_for(n, kThreads), kThreads, 0, stream>>>(nullptr, nullptr, nullptr, nullptr,
            nullptr, (Fr*)d_permuted_input, (Fr*)d_permuted_table, 0, n);
        H2_LAUNCH_CHECK();
    }
    return ok();
}

} // extern "C"
