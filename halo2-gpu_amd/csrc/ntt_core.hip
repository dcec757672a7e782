// Fr NTT engine: table generation and the LDS-staged Stockham pass kernel.
// See ntt_core.h for the decomposition.
//
// Inside a pass the transform runs in radix-16 and radix-8 steps on the matrix cores
// (ntt_mfma.h), each closed by one Montgomery product with the position's twiddle.
// Elements stay in the boundary's 2^256 Montgomery scale, 32 bytes each; the constants of
// those products are held in the 2^290 scale, the coset powers and zeta that multiply the
// input (9 x 29-bit products, field29.h) in the 2^261 scale.
#include <atomic>
#include <mutex>
#include <vector>

#include "field29.h"
#include "ntt_core.h"
#include "ntt_mfma.h"
#include "profile.h"

namespace h2 {

// zeta (a primitive cube root of unity, halo2's g_coset) and zeta^2 times
// 2^261 mod r, in 29-bit limbs. The reference hard-codes zeta and zeta^2 in
// 2^256 Montgomery form at cuda/include/kernel/zeta.h:19-30; these are the
// same field elements rescaled.
__device__ __forceinline__ Fr29 zeta261(uint32_t m)
{
    constexpr uint32_t z1[9] = { 0x0f9aca5du, 0x06c39377u, 0x03fb9328u, 0x0dd12516u, 0x19b77045u, 0x1b53b497u,
        0x086e5ab0u, 0x0b729bf7u, 0x00226320u };
    constexpr uint32_t z2[9] = { 0x1065364du, 0x19a50e73u, 0x05348a9cu, 0x02af1c94u, 0x11265ae2u, 0x0a454b5au,
        0x06633a88u, 0x1dbec294u, 0x000038f7u };
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i)
        r.l[i] = m == 1 ? z1[i] : z2[i];
    return r;
}

// a b / 2^256 mod r on the host (CIOS over 32-bit words), canonical
static void host_mont_mul(const uint32_t* a, const uint32_t* b, uint32_t (&w)[8])
{
    const uint32_t* m = FrParams::M;
    uint32_t t[10] = { 0 };
    for (int i = 0; i < 8; ++i) {
        uint64_t c = 0;
        for (int j = 0; j < 8; ++j) {
            c += (uint64_t)t[j] + (uint64_t)a[j] * b[i];
            t[j] = (uint32_t)c;
            c >>= 32;
        }
        c += t[8];
        t[8] = (uint32_t)c;
        t[9] = (uint32_t)(c >> 32);
        const uint32_t q = t[0] * FrParams::INV;
        c = ((uint64_t)t[0] + (uint64_t)q * m[0]) >> 32;
        for (int j = 1; j < 8; ++j) {
            c += (uint64_t)t[j] + (uint64_t)q * m[j];
            t[j - 1] = (uint32_t)c;
            c >>= 32;
        }
        c += t[8];
        t[7] = (uint32_t)c;
        t[8] = t[9] + (uint32_t)(c >> 32);
    }
    // t < 2m: reduce once
    uint32_t d[8];
    int64_t br = 0;
    for (int j = 0; j < 8; ++j) {
        const int64_t v = (int64_t)t[j] - m[j] + br;
        d[j] = (uint32_t)v;
        br = v >> 32;
    }
    const bool ge = t[8] != 0 || br == 0;
    for (int j = 0; j < 8; ++j)
        w[j] = ge ? d[j] : t[j];
}

// 2^290 mod r, and zeta, zeta^2 times 2^256 mod r
static constexpr uint32_t kTo290[8] = { 0x56e2e768u, 0x4f9e2194u, 0xc17a8552u, 0x5b7c909au, 0xc0aae0e4u, 0x49c6dd0cu,
    0xb1b089b8u, 0x1af00dfbu };
static constexpr uint32_t kZeta256[2][8] = { { 0x55fcd653u, 0x0363f299u, 0x5fc1e200u, 0x73e7950bu, 0x576d9d24u,
                                                 0xc5fce83eu, 0xa1c3a4d4u, 0x059c805du },
    { 0x4a0329b3u, 0x93e7cedeu, 0x7a96c167u, 0x7d4fdca7u, 0xb19a750au, 0x8be4ba08u, 0xa5661c25u, 0x1cbd5653u } };

// words of a value < 2^256 -> 29-bit limbs
static void host_limbs(const uint32_t (&w)[8], uint32_t (&l)[9])
{
    for (int i = 0; i < 8; ++i) {
        const int wi = (29 * i) >> 5, sh = (29 * i) & 31;
        const uint64_t two = ((uint64_t)w[wi + 1] << 32) | w[wi];
        l[i] = (uint32_t)(two >> sh) & 0x1fffffffu;
    }
    l[8] = w[7] >> 8;
}

// Output scale s (one for POST_NONE): s 2^290 mod r
static void host_scale290(NttPost post, const Fr& scale, uint32_t (&s)[8])
{
    host_mont_mul(post == POST_NONE ? FrParams::ONE : scale.v, kTo290, s);
}

// 2^29 s 8 K mod r, K = sum_b 128 2^(8b): the part of a radix-8 last step's y_0 that the shift of
// the data bytes takes away (ntt_mfma.h; a radix-16 step's is twice that)
static void host_bias8(NttPost post, const Fr& scale, uint32_t (&limbs)[9])
{
    static constexpr uint32_t k8k[8] = { 0x20202020u, 0x20202020u, 0x20202020u, 0x20202020u, 0x20202020u, 0x20202020u,
        0x20202020u, 0x20202020u }; // 8 K / 2^5
    uint32_t s[8], b[8];
    host_scale290(post, scale, s);
    host_mont_mul(s, k8k, b);
    host_limbs(b, limbs);
}

// The direct DFT's last factors for output index i mod 3: s zeta^-(i mod 3)
// (POST_SCALE_ZETA_INV), s (POST_SCALE) or 1, in the 2^261 scale.
static void host_post(NttPost post, const Fr& scale, uint32_t (&pc)[3][9])
{
    uint32_t s[8];
    host_mont_mul(post == POST_NONE ? FrParams::ONE : scale.v, Fr29Params::TO261, s);
    for (int k = 0; k < 3; ++k) {
        uint32_t w[8];
        if (k && post == POST_SCALE_ZETA_INV)
            host_mont_mul(s, kZeta256[2 - k], w); // zeta^-1 = zeta^2
        else
            memcpy(w, s, sizeof(w));
        host_limbs(w, pc[k]);
    }
}

// Tuned work-group tile sizes: log2 of the elements per work-group for
// transforms of 2^log_n (0 = the default rule). Set with h2amd_ntt_set_tiles.
// Atomic entries: a setter on one host thread may race planners on others.
static std::atomic<uint8_t> g_tile_table[NTT_MAX_LOG + 1] = {};

NttPlan ntt_plan(uint32_t log_n)
{
    NttPlan p {};
    p.P = log_n <= NTT_MAX_LOG_R ? 1 : log_n <= 2 * NTT_MAX_LOG_R ? 2 : 3;
    // A pass of 2^8 rows takes two matrix steps (16 x 16), one of 2^9 to 2^12 three: where the first
    // pass can hold the rest, all later ones are of 2^8 (2^17 .. 2^20: 5 steps; 2^25 .. 2^28: 7).
    // Even splits take 6 and up to 9: 2^20 153 -> 147 us, 2^27 24.5 -> 23.5 ms, twelve of 2^18 in an
    // uneven batch 380 -> 349 us. Else (2^13 .. 2^16: 4 steps, 2^21 .. 2^24: 6) passes are about even.
    const uint32_t rest = log_n > 8u * (p.P - 1) ? log_n - 8u * (p.P - 1) : 0;
    if (p.P > 1 && rest >= 9 && rest <= NTT_MAX_LOG_R) {
        p.log_r[0] = rest;
        for (int i = 1; i < p.P; ++i)
            p.log_r[i] = 8;
    } else if (p.P == 2) {
        p.log_r[0] = (log_n + 1) / 2;
        p.log_r[1] = log_n - p.log_r[0];
    } else {
        p.log_r[0] = log_n;
    }
    for (int i = 0; i < p.P; ++i) {
        // aim for >= 256 work-groups per transform, 512 to 4096 elements per work-group (a
        // matrix step takes 512: 16 rows of 32 vectors)
        int g = (int)log_n - (int)p.log_r[i] - 8;
        const int gmax = (int)(p.log_r[i] < 8 ? NTT_MAX_LOG_R - 1 : NTT_MAX_LOG_R) - (int)p.log_r[i]; // LDS: kMaxPassLds
        const int gmin = (int)p.log_r[i] < 9 ? 9 - (int)p.log_r[i] : 0;
        if (g > gmax)
            g = gmax;
        if (g < gmin)
            g = gmin;
        const uint8_t tuned = log_n <= NTT_MAX_LOG ? g_tile_table[log_n].load(std::memory_order_relaxed) : 0;
        if (tuned) {
            g = (int)tuned - (int)p.log_r[i];
            if (g > gmax)
                g = gmax;
            if (g > (int)log_n - (int)p.log_r[i])
                g = (int)log_n - (int)p.log_r[i];
            if (g < gmin)
                g = gmin;
        }
        if (p.P == 1)
            g = 0;
        p.log_g[i] = (uint32_t)g;
    }
    return p;
}

bool ntt_needs_scratch(uint32_t log_n, bool aliased)
{
    NttPlan p = ntt_plan(log_n);
    return p.P == 3 || (p.P == 2 && aliased);
}

static inline uint32_t split_h(uint32_t log_n) { return (log_n + 1) / 2; }

// log2 radices of a pass of 2^log_r rows, 6 <= log_r <= 12: 16s as far as 8s can fill the rest
static uint32_t radix_steps(uint32_t log_r)
{
    uint32_t steps = 0;
    for (int i = 0; log_r; ++i) {
        const uint32_t l = log_r % 3 == 0 && log_r != 12 ? 3 : 4;
        steps |= l << (8 * i);
        log_r -= l;
    }
    return steps;
}

static constexpr uint32_t kMatrixWords = 1024; // matrices of 16 powers of a root, in 16-byte words

// entries of a pass's step tables: one per element for every step but the last
static uint64_t step_entries(uint32_t log_r)
{
    uint64_t n = 0;
    uint32_t log_rs = log_r;
    for (uint32_t steps = radix_steps(log_r); steps >> 8; steps >>= 8) {
        n += 1ull << log_rs;
        log_rs -= steps & 255;
    }
    return n;
}

void ntt_tables_size(WorkspaceSizer& ws, uint32_t log_n, bool powers_twist)
{
    NttPlan p = ntt_plan(log_n);
    uint32_t h = split_h(log_n);
    ws.take(32ull << h);
    ws.take(32ull << (log_n - h));
    for (int i = 0; i < p.P; ++i)
        ws.take(32 * (log_n < NTT_MATRIX_LOG ? 1ull << log_n : step_entries(p.log_r[i])));
    ws.take(4);
    ws.take(16 * kMatrixWords);
    if (powers_twist) {
        ws.take(32ull << p.log_r[0]);
        ws.take(32ull << (log_n - p.log_r[0]));
    }
}

enum TableKind : uint8_t {
    TABLE_261 = 0, // out[i] = (base^(2^shift))^x in the 2^261 scale
    TABLE_290 = 1, // the same in the 2^290 scale
    TABLE_UNIT = 2, // the exponent u < 16 (odd) for which omega^(2^shift) = kG16^u: by it the
                    // matrix steps permute their constants
    TABLE_MATRICES = 3, // the matrices (ntt_mfma.h) of 2^29 s w^e, w = omega^(2^shift), e < 16, for the
                        // last step: s is the output's scale, and 2^29 is the one Montgomery
                        // step that then makes its result an element
};

// One table of `count` threads' work. x = i, or for a step's table (row > 0) x = j b with
// i = j 2^row + b: output j of the step at position b, so the lanes of a wave, which are
// consecutive b, read consecutive entries.
struct TableJob {
    Fr* out;
    uint32_t shift;
    uint32_t count;
    uint8_t kind, use_c, row;
};
// The tables of one transform: at most 2 + 3 * 2 + 2 + 2
struct TableSet {
    TableJob j[12];
    uint32_t nj, log_n;
    const Fr* omega;
    Fr c;
    uint32_t scale290[9]; // s 2^290
};
constexpr int kTableSets = 6;
struct TableSets {
    TableSet s[kTableSets];
};

__global__ void __launch_bounds__(64) ntt_tables_kernel(TableSets sets)
{
    const TableSet& ts = sets.s[blockIdx.z];
    if (blockIdx.y >= ts.nj)
        return;
    const TableJob job = ts.j[blockIdx.y];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= job.count)
        return;
    const uint32_t x = job.kind == TABLE_MATRICES ? i >> 5
        : job.kind == TABLE_UNIT                  ? 1
        : job.row                                 ? (i >> job.row) * (i & ((1u << job.row) - 1))
                                                  : i;
    Fr to;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        to.v[k] = Fr29Params::TO261[k];
    // square and multiply from the low bits, so that a round's two products do not wait for
    // each other: the log n squarings are the kernel's time
    Fr29 b = Fr29::from_fp((job.use_c ? ts.c : Fr::load(ts.omega)) * to);
    for (uint32_t s = 0; s < job.shift; ++s)
        b = Fr29::sqr(b);
    Fr29 r = Fr29::one();
    for (uint32_t s = 0; s < 28 && __any((x >> s) != 0); ++s) {
        const Fr29 m = Fr29::mul(r, b);
        b = Fr29::sqr(b);
#pragma unroll
        for (int k = 0; k < 9; ++k)
            r.l[k] = (x >> s) & 1 ? m.l[k] : r.l[k];
    }
    if (job.kind == TABLE_UNIT) {
        const Fr29 one256 = Fr29::from_fp(Fr::one()); // 2^256 mod m: back from the 2^261 scale
        uint32_t w[8];
        Fr29::reduce_full(Fr29::mul(r, one256)).to32(w);
        bool same = true;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            same = same && w[k] == kFrRoots16.mont[i & 7][k];
        const uint64_t m = __ballot(same) & 255u;
        if (i == 0)
            *(uint32_t*)job.out = m ? 2u * (uint32_t)__builtin_ctzll(m) + 1u : 1u;
        return;
    }
    if (job.kind == TABLE_MATRICES) {
        const uint32_t e = i >> 5, byte = i & 31;
        Fr29 scale, p = Fr29::zero(); // p = 2^(8 byte)
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            scale.l[k] = ts.scale290[k];
            p.l[k] = 8 * byte / 29 == (uint32_t)k ? 1u << (8 * byte % 29) : 0u;
        }
        // (w 2^261) (s 2^290) / 2^261 2^(8 byte) / 2^261 = 2^29 s w 2^(8 byte)
        const Fr29 v = Fr29::reduce_full(Fr29::mul(Fr29::mul(r, scale), p));
        store_matrix_column((uint8_t*)job.out, e, byte, v);
        return;
    }
    if (job.kind == TABLE_290) {
        Fr29 c;
        constexpr uint32_t one290[9] = { 0x16e2e768u, 0x1cf10ca2u, 0x1ea15493u, 0x19213582u, 0x0e0e45b7u, 0x0e866055u,
            0x06e1271bu, 0x1f763611u, 0x001af00du };
#pragma unroll
        for (int k = 0; k < 9; ++k)
            c.l[k] = one290[k];
        r = Fr29::mul(r, c);
    }
    r.store32(job.out + i);
}

RustError ntt_tables_plan(Workspace& ws, NttTables& t, uint32_t log_n, const Fr* d_omega, bool powers_twist,
    const Fr& c, NttPost post, const Fr& scale, TableSet& ts)
{
    NttPlan p = ntt_plan(log_n);
    uint32_t h = split_h(log_n);
    const bool direct = log_n < NTT_MATRIX_LOG;
    ts.nj = 0;
    ts.log_n = log_n;
    ts.omega = d_omega;
    ts.c = c;
    uint32_t scale290[8];
    host_scale290(post, scale, scale290);
    host_limbs(scale290, ts.scale290);
    auto job = [&](void* out, uint32_t count, uint32_t shift, bool use_c, TableKind kind, uint32_t row) {
        ts.j[ts.nj++] = TableJob { (Fr*)out, shift, count, kind, use_c, (uint8_t)row };
    };
    auto add = [&](uint32_t log_count, uint32_t shift, bool use_c, TableKind kind) -> Fr* {
        Fr* out = (Fr*)ws.take(32ull << log_count);
        job(out, 1u << log_count, shift, use_c, kind, 0);
        return out;
    };
    t.h = h;
    if (p.P > 1) {
        t.tw_lo = add(h, 0, false, TABLE_290);
        t.tw_hi = add(log_n - h, h, false, TABLE_261);
    }
    for (int i = 0; i < p.P; ++i) {
        if (direct) {
            t.twr[i] = add(log_n, 0, false, TABLE_261);
            continue;
        }
        Fr* out = (Fr*)ws.take(32 * step_entries(p.log_r[i]));
        t.twr[i] = out;
        uint32_t log_rs = p.log_r[i];
        for (uint32_t steps = radix_steps(p.log_r[i]); steps >> 8; steps >>= 8) {
            job(out, 1u << log_rs, log_n - log_rs, false, TABLE_290, log_rs - (steps & 255));
            out += 1ull << log_rs;
            log_rs -= steps & 255;
        }
    }
    if (!direct) {
        uint32_t* unit = (uint32_t*)ws.take(4);
        uint4* matrices = (uint4*)ws.take(16 * kMatrixWords);
        t.unit = unit;
        t.last_matrices = matrices;
        job(unit, 64, log_n - 4, false, TABLE_UNIT, 0);
        job(matrices, 512, log_n - 4, false, TABLE_MATRICES, 0);
    }
    if (powers_twist) { // c^(n1 stride + column): rows and columns of the first pass
        t.c_rows = add(p.log_r[0], log_n - p.log_r[0], true, TABLE_261);
        t.c_cols = add(log_n - p.log_r[0], 0, true, TABLE_261);
    }
    if (ws.overflow)
        return fail((int)hipErrorInvalidValue, "NTT workspace too small for the twiddle tables (log_n=%u)", log_n);
    return ok();
}

static RustError launch_tables(const TableSets& sets, int count, hipStream_t stream)
{
    uint32_t maxc = 64, nj = 1;
    for (int k = 0; k < count; ++k) {
        nj = sets.s[k].nj > nj ? sets.s[k].nj : nj;
        for (uint32_t i = 0; i < sets.s[k].nj; ++i)
            maxc = sets.s[k].j[i].count > maxc ? sets.s[k].j[i].count : maxc;
    }
    ntt_tables_kernel<<<dim3((maxc + 63) / 64, nj, count), 64, 0, stream>>>(sets);
    H2_LAUNCH_CHECK();
    return ok();
}

RustError ntt_tables_build(const NttTableSpec* specs, NttTables* const* tables, int count, Workspace& ws,
    hipStream_t stream)
{
    for (int base = 0; base < count; base += kTableSets) {
        TableSets sets {};
        const int n = count - base < kTableSets ? count - base : kTableSets;
        for (int k = 0; k < n; ++k) {
            const NttTableSpec& sp = specs[base + k];
            RustError e = ntt_tables_plan(ws, *tables[base + k], sp.log_n, sp.d_omega, sp.powers_twist, sp.c, sp.post,
                sp.scale, sets.s[k]);
            if (e.code)
                return e;
        }
        RustError e = launch_tables(sets, n, stream);
        if (e.code)
            return e;
    }
    return ok();
}

struct PassBatch {
    const Fr* in[NTT_MAX_BATCH];
    Fr* out[NTT_MAX_BATCH];
};

struct PassParams {
    uint32_t log_n, log_r, log_g, log_l;
    uint64_t in_len;
    const Fr* tw_lo;
    const Fr* tw_hi;
    const Fr* twr;
    const Fr* c_rows;
    const Fr* c_cols;
    const uint32_t* unit; // u of the transform's 16th root kG16^u
    const uint4* last_matrices; // of the last pass's last step
    uint32_t h;
    uint32_t steps; // log2 of the matrix steps' radices (4 or 3; 0 = no step), a byte each, first step lowest
    int twist;
    int post;
    int last;
    uint32_t xcd_remap;
    uint32_t bias8[9]; // of the last step's y_0 (host_bias8)
    uint32_t pc[3][9]; // constants of the direct DFT's last product (host_post)
};

// LDS: the matrices of the 16 powers of the root (16 KiB), then the tile, 32 bytes an element,
// then in every pass but the last the columns' inter-pass twiddles (pass_twiddles).
// Slot i of the tile is element lds_slot(i): the low 3 bits of i XOR a function of the higher
// ones, a permutation inside every block of 8 (256 bytes). The accesses of 16 or 32 bytes per
// lane at a power-of-two stride (the loads and stores of the last steps, the digit-reversed
// read of the store) then spread over the banks instead of sharing a few.

// Inter-pass twiddle of frequency k1 of a column: (entry k1 mod 2^l) (entry k1 >> l), two
// tables of about sqrt(R) entries per column, l = twiddle_split(log_r)
__host__ __device__ constexpr uint32_t twiddle_split(uint32_t log_r) { return (log_r + 1) / 2; }
__host__ __device__ constexpr uint32_t twiddle_entries(uint32_t log_r)
{
    return (1u << twiddle_split(log_r)) + (1u << (log_r - twiddle_split(log_r)));
}
static uint32_t pass_lds_bytes(uint32_t log_r, uint32_t log_g, bool last)
{
    return 16 * kMatrixWords + (32u << (log_r + log_g)) + (last ? 0 : (32 * twiddle_entries(log_r)) << log_g);
}
static constexpr uint32_t kMaxPassLds = 160 << 10; // a column of 4096: 16 + 128 + 4 KiB; 16 of 256: 16 + 128 + 16

__device__ __forceinline__ uint32_t lds_slot(uint32_t i) { return i ^ (((i >> 3) ^ (i >> 6) ^ (i >> 9)) & 7u); }

__device__ __forceinline__ void lds_store(uint4* X, uint32_t slot, const Fr29& x)
{
    uint32_t v[8];
    x.to32(v);
    uint4* p = X + 2 * lds_slot(slot);
    p[0] = make_uint4(v[0], v[1], v[2], v[3]);
    p[1] = make_uint4(v[4], v[5], v[6], v[7]);
}

// Frequency of position q of a column after the steps (digits reversed), and back.
__device__ __forceinline__ uint32_t step_frequency(const PassParams& pp, uint32_t q)
{
    const uint32_t l1 = pp.steps & 255, l2 = (pp.steps >> 8) & 255, l3 = pp.steps >> 16;
    return (q >> (l2 + l3)) | (((q >> l3) & ((1u << l2) - 1)) << l1) | ((q & ((1u << l3) - 1)) << (l1 + l2));
}
__device__ __forceinline__ uint32_t step_position(const PassParams& pp, uint32_t k)
{
    const uint32_t l1 = pp.steps & 255, l2 = (pp.steps >> 8) & 255, l3 = pp.steps >> 16;
    return ((k & ((1u << l1) - 1)) << (l2 + l3)) | (((k >> l1) & ((1u << l2) - 1)) << l3) | (k >> (l1 + l2));
}

__device__ __forceinline__ Fr29 post_constant(const PassParams& pp, uint32_t m)
{
    Fr29 w;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const uint32_t c0 = pp.pc[0][i], c1 = pp.pc[1][i], c2 = pp.pc[2][i];
        w.l[i] = m == 0 ? c0 : m == 1 ? c1 : c2;
    }
    return w;
}

enum StepEnd : int {
    END_TWIDDLE = 0, // not the pass's last step: the position's twiddle of the pass
    END_PASS = 1, // the inter-pass twiddle
    END_LAST = 2, // the canonical form (the matrices hold the output's scale)
};

// One radix-2^LR step (decimation in frequency) of every column of the tile in place:
// the blocks of 2^log_rs positions become 2^LR blocks of 2^(log_rs - LR). A unit of work is
// 32 vectors (position b of block blk, 2^LR elements each); the work-group's waves share the
// units, or split a unit's outputs among them when they are more, and then wait for each
// other between reading a unit and writing it.
template <int LR>
__device__ __forceinline__ void matrix_step(const PassParams& pp, uint4* lds, uint32_t j0, uint32_t log_rs, StepEnd end,
    const Fr* __restrict__ tw)
{
    constexpr uint32_t r = 1u << LR, H = r / 2;
    uint4* X = lds + kMatrixWords;
    const uint32_t lane = threadIdx.x & 63, half = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const uint32_t log_s = log_rs - LR;
    const uint32_t vectors = 1u << (pp.log_r + pp.log_g - LR);
    const uint32_t units = (vectors + 31) >> 5;
    uint32_t per = units >= waves ? 1 : waves / units; // waves per unit
    if (per > H)
        per = H;
    const uint32_t stride = waves / per;
    const uint32_t part = wave & (per - 1);
    const uint32_t j_lo = part * (H / per), j_hi = j_lo + H / per;
    uint32_t unit = wave / per;
    do {
        const uint32_t t = unit * 32 + (lane & 31);
        const bool act = t < vectors;
        const uint32_t b = act ? t & ((1u << log_s) - 1) : 0;
        const uint32_t base = act ? ((t >> log_s) << log_rs) + b : 0;
        mfma_v4 x[r];
        if (unit < units) {
#pragma unroll
            for (uint32_t a = 0; a < r; ++a) {
                const uint4 w = X[2 * lds_slot(base + (a << log_s)) + half];
                x[a] = mfma_v4 { (int)(w.x ^ 0x80808080u), (int)(w.y ^ 0x80808080u), (int)(w.z ^ 0x80808080u),
                    (int)(w.w ^ 0x80808080u) };
            }
        }
        if (per > 1)
            __syncthreads();
        if (unit < units) {
            // the next outputs' matrices are read while the vector unit works on the last ones'
            mfma_v4 m[r];
            auto read_matrices = [&](uint32_t j) {
#pragma unroll
                for (uint32_t a = 0; a < r; ++a) {
                    const uint4 w = lds[(((a * j * (16 / r)) & 15) << 6) + lane];
                    m[a] = mfma_v4 { (int)w.x, (int)w.y, (int)w.z, (int)w.w };
                }
            };
            read_matrices(j_lo);
            for (uint32_t j = j_lo; j < j_hi; ++j) {
                const uint32_t jj = j + half * H;
                const uint32_t slot = base + (jj << log_s);
                uint4 w0, w1;
                if (end == END_TWIDDLE) {
                    const uint4* p = (const uint4*)(tw + ((jj << log_s) + b));
                    w0 = p[0];
                    w1 = p[1];
                }
                mfma_v16 E = {}, O = {};
#pragma unroll
                for (uint32_t a = 0; a < H; ++a) {
                    E = __builtin_amdgcn_mfma_i32_32x32x32_i8(m[2 * a], x[2 * a], E, 0, 0, 0);
                    O = __builtin_amdgcn_mfma_i32_32x32x32_i8(m[2 * a + 1], x[2 * a + 1], O, 0, 0, 0);
                }
                read_matrices(j + 1 < j_hi ? j + 1 : j);
                __builtin_amdgcn_sched_barrier(0);
                Fr29 w;
                if (end == END_TWIDDLE) {
                    const uint32_t words[8] = { w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w };
                    w = Fr29::from32(words);
                }
                uint32_t v[10];
                mfma_limbs(E, O, j == 0 && end != END_LAST ? (int)(128 * r * 257) : 0, v);
                if (end == END_PASS) {
                    const uint32_t k1 = step_frequency(pp, slot & ((1u << pp.log_r) - 1));
                    const uint32_t l = twiddle_split(pp.log_r);
                    const uint4* T = X + (2u << (pp.log_r + pp.log_g))
                        + 2 * twiddle_entries(pp.log_r) * (slot >> pp.log_r);
                    w = Fr29::mul(Fr29::load32(T + 2 * (k1 & ((1u << l) - 1))),
                        Fr29::load32(T + 2 * ((1u << l) + (k1 >> l))));
                }
                Fr29 y;
                if (end == END_LAST) {
                    if (jj == 0) {
#pragma unroll
                        for (int i = 0; i < 9; ++i)
                            v[i] += pp.bias8[i] * (r / 8);
                    }
                    y = mont_step(v);
                    if (pp.post == POST_SCALE_ZETA_INV) {
                        const uint32_t k1 = step_frequency(pp, slot & ((1u << pp.log_r) - 1));
                        const uint32_t col = j0 + (slot >> pp.log_r);
                        const uint32_t i = (uint32_t)((col + ((uint64_t)k1 << pp.log_l)) % 3u);
                        if (i)
                            y = canonical_3m(Fr29::mul(y, zeta261(3u - i)));
                    }
                } else {
                    y = mul_10x9(v, w);
                }
                if (act)
                    lds_store(X, slot, y);
            }
        }
        unit += stride;
    } while (per == 1 && unit < units);
}

// x times its twist (x < 2^256: the product is < 1.25 m): zeta^(i mod 3) for index i, or
// row n1's part of c^i (the column's part rides in the inter-pass twiddles)
__device__ __forceinline__ Fr29 twisted(const PassParams& pp, const Fr29& x, uint64_t gi, uint32_t n1)
{
    if (pp.twist == TWIST_ZETA) {
        const uint32_t m = (uint32_t)(gi % 3u);
        return m ? Fr29::mul(x, zeta261(m)) : x;
    }
    return Fr29::mul(x, Fr29::load32(pp.c_rows + n1));
}

// The inter-pass twiddles of the tile's columns: for column j0 + g (n2 = its part of the index)
// the powers x = 0, 1, ... and 2^l, 2 2^l, ... of omega^(n2 2^log_l), the first ones in the
// 2^290 scale and times c^column (first pass with TWIST_POWERS), the others in the 2^261
// scale. Read from LDS they cost the last step one product an element; from the two
// tables of omega's powers a step's lanes would read 128 cache lines.
__device__ __forceinline__ void pass_twiddles(const PassParams& pp, uint4* T, uint32_t j0)
{
    constexpr uint32_t k232[9] = { 0, 0, 0, 0, 0, 0, 0, 0, 1 }; // 2^232: 2^290 scale -> 2^261
    const uint32_t n = twiddle_entries(pp.log_r), l = twiddle_split(pp.log_r);
    for (uint32_t i = threadIdx.x; i < n << pp.log_g; i += blockDim.x) {
        const uint32_t g = i / n, k = i % n;
        const bool low = k < (1u << l);
        const uint32_t col = j0 + g;
        const uint32_t e = ((col >> pp.log_l) * (low ? k : (k - (1u << l)) << l)) << pp.log_l;
        Fr29 w = Fr29::load32(pp.tw_lo + (e & ((1u << pp.h) - 1)));
        const uint32_t hi = e >> pp.h;
        if (hi)
            w = Fr29::mul(w, Fr29::load32(pp.tw_hi + hi));
        if (!low)
            w = Fr29::mul(w, Fr29::from_limbs(k232));
        else if (pp.twist == TWIST_POWERS)
            w = Fr29::mul(w, Fr29::load32(pp.c_cols + col));
        w.store32(T + 2 * i);
    }
}

// A transform of fewer points than a matrix step takes (2 to 32): y_k = sum_i x_i w^(ik) by
// definition. Eight threads per output take every eighth term, at most 4 products deep (one
// thread per output was 32 deep: a call of 2^5 points 36 us, now 29, the host's part).
__device__ __forceinline__ void ntt_direct(const Fr* __restrict__ in, Fr* __restrict__ out, const PassParams& pp,
    uint4* lds)
{
    constexpr uint32_t kParts = 8; // 8 N <= 256 threads
    const uint32_t N = 1u << pp.log_n, k = threadIdx.x & (N - 1), part = threadIdx.x >> pp.log_n;
    uint4* sums = lds + 2 * N;
    if (part == 0) {
        Fr29 x = Fr29::zero();
        if (k < pp.in_len) {
            x = Fr29::load32(in + k);
            if (pp.twist != TWIST_NONE)
                x = twisted(pp, x, k, k);
        }
        lds_store(lds, k, x);
    }
    __syncthreads();
    if (part < kParts) {
        Fr29 y = Fr29::zero();
        for (uint32_t i = part; i < N; i += kParts) {
            const uint4* p = lds + 2 * lds_slot(i);
            // x < 5.3 m (2^256): each product < 1.04 m, the sum < 4.2 m < 2^256
            y = Fr29::normalize(Fr29::add(y, Fr29::mul(Fr29::load32(p), Fr29::load32(pp.twr + ((i * k) & (N - 1))))));
        }
        lds_store(sums, part * N + k, y);
    }
    __syncthreads();
    if (part)
        return;
    Fr29 y = Fr29::zero();
#pragma unroll
    for (uint32_t i = 0; i < kParts; ++i) // limbs < 8 2^29
        y = Fr29::add(y, Fr29::load32(sums + 2 * lds_slot(i * N + k)));
    const Fr29 w = post_constant(pp, pp.post == POST_SCALE_ZETA_INV ? k % 3u : 0u);
    canonical_3m(Fr29::mul(Fr29::normalize(y), w)).store32(out + k); // < 1.25 m before
}

// Work-group `b` (of nwg) of one pass of one transform. Every value in LDS is < 2.1 m, or
// the input itself (any 256-bit word).
__device__ __forceinline__ void ntt_pass_tile(
    const Fr* __restrict__ in, Fr* __restrict__ out, const PassParams& pp, uint32_t b, uint4* lds)
{
    if (pp.log_n < NTT_MATRIX_LOG) {
        ntt_direct(in, out, pp, lds);
        return;
    }
    const uint32_t log_r = pp.log_r, log_g = pp.log_g, log_l = pp.log_l;
    const uint32_t R = 1u << log_r;
    const uint32_t G = 1u << log_g;
    const uint32_t RG = R << log_g;
    const uint32_t T = blockDim.x;
    const uint32_t nwg = (uint32_t)((1ull << pp.log_n) >> (log_r + log_g));
    if (pp.xcd_remap) // blocks are dealt to the 8 XCDs round robin: keep neighbouring columns on one L2
        b = (b & 7u) * (nwg >> 3) + (b >> 3);
    const uint32_t j0 = b << log_g;
    const uint64_t stride = (1ull << pp.log_n) >> log_r;
    uint4* X = lds + kMatrixWords;

    const uint32_t u = *pp.unit;
    const uint4* roots = (const uint4*)kFrRoots16.a;
    for (uint32_t i = threadIdx.x; i < kMatrixWords; i += T)
        lds[i] = roots[(((u * (i >> 6)) & 15) << 6) + (i & 63)];
    // the tile as it is, 8 elements per thread in flight; then, where there is a twist, each
    // thread multiplies the elements it brought
    constexpr uint32_t kLoads = 8;
    for (uint32_t f0 = threadIdx.x; f0 < RG; f0 += kLoads * T) {
        uint4 v[kLoads][2];
#pragma unroll
        for (uint32_t k = 0; k < kLoads; ++k) {
            const uint32_t f = f0 + k * T;
            const uint64_t gi = (uint64_t)(j0 + (f & (G - 1))) + (uint64_t)(f >> log_g) * stride;
            v[k][0] = v[k][1] = make_uint4(0, 0, 0, 0);
            if (f < RG && gi < pp.in_len) {
                const uint4* q = (const uint4*)(in + gi);
                v[k][0] = q[0];
                v[k][1] = q[1];
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kLoads; ++k) {
            const uint32_t f = f0 + k * T;
            if (f < RG) {
                uint4* p = X + 2 * lds_slot(((f & (G - 1)) << log_r) + (f >> log_g));
                p[0] = v[k][0];
                p[1] = v[k][1];
            }
        }
    }
    if (!pp.last)
        pass_twiddles(pp, X + 2 * RG, j0);
    if (pp.twist != TWIST_NONE) {
        for (uint32_t f = threadIdx.x; f < RG; f += T) {
            const uint64_t gi = (uint64_t)(j0 + (f & (G - 1))) + (uint64_t)(f >> log_g) * stride;
            const uint32_t slot = ((f & (G - 1)) << log_r) + (f >> log_g);
            if (gi < pp.in_len)
                lds_store(X, slot, twisted(pp, Fr29::load32(X + 2 * lds_slot(slot)), gi, f >> log_g));
        }
    }
    uint32_t log_rs = log_r;
    const Fr* tw = pp.twr;
    for (int s = 0; log_rs; ++s) {
        __syncthreads();
        const uint32_t lr = (pp.steps >> (8 * s)) & 255;
        const StepEnd end = lr < log_rs ? END_TWIDDLE : pp.last ? END_LAST : END_PASS;
        if (end == END_LAST) {
            for (uint32_t i = threadIdx.x; i < kMatrixWords; i += T)
                lds[i] = pp.last_matrices[i];
            __syncthreads();
        }
        if (lr == 4)
            matrix_step<4>(pp, lds, j0, log_rs, end, tw);
        else
            matrix_step<3>(pp, lds, j0, log_rs, end, tw);
        tw += 1u << log_rs;
        log_rs -= lr;
    }
    __syncthreads();

    const bool mapA = (G > 1) && (log_l > 0);
    const uint32_t lmask = (1u << log_l) - 1;
    for (uint32_t f = threadIdx.x; f < RG; f += T) {
        uint32_t g, k1;
        if (mapA) {
            g = f & (G - 1);
            k1 = f >> log_g;
        } else {
            k1 = f & (R - 1);
            g = f >> log_r;
        }
        const uint4* p = X + 2 * lds_slot((g << log_r) + step_position(pp, k1));
        const uint32_t j = j0 + g;
        const uint32_t K = j & lmask;
        const uint32_t n2 = j >> log_l;
        const uint64_t o = ((uint64_t)n2 << (log_l + log_r)) + K + ((uint64_t)k1 << log_l);
        uint4* q = (uint4*)(out + o);
        q[0] = p[0];
        q[1] = p[1];
    }
}

__global__ void __launch_bounds__(512) ntt_pass_kernel(PassBatch pb, PassParams pp)
{
    extern __shared__ uint4 lds[];
    ntt_pass_tile(pb.in[blockIdx.y], pb.out[blockIdx.y], pp, blockIdx.x, lds);
}

// One pass of many transforms of different sizes: work-groups
// [block0, block0 + nwg) of the launch belong to the transform.
struct BatchPass {
    const Fr* in;
    Fr* out;
    uint32_t block0, nwg;
    PassParams pp;
};

__global__ void __launch_bounds__(512) ntt_pass_batch_kernel(const BatchPass* __restrict__ jobs, uint32_t njobs)
{
    extern __shared__ uint4 lds[];
    uint32_t lo = 0, hi = njobs; // last job with block0 <= blockIdx.x (uniform)
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].block0 <= blockIdx.x)
            lo = mid;
        else
            hi = mid;
    }
    const BatchPass& jb = jobs[lo];
    const PassParams pp = jb.pp;
    ntt_pass_tile(jb.in, jb.out, pp, blockIdx.x - jb.block0, lds);
}

// The dynamic-LDS limit of the pass kernels, raised once per process (std::call_once:
// concurrent first calls from several host threads are safe).
static hipError_t raise_lds_limits()
{
    static std::once_flag once;
    static hipError_t status = hipSuccess;
    std::call_once(once, [] {
        status = hipFuncSetAttribute((const void*)ntt_pass_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
            (int)kMaxPassLds);
        if (status == hipSuccess)
            status = hipFuncSetAttribute((const void*)ntt_pass_batch_kernel,
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxPassLds);
    });
    return status;
}

// Threads per work-group: 8 waves where a compute unit gets one work-group (its tile takes more
// than half of the LDS, or there are no more work-groups than compute units) or a tile has work
// for them (a unit of a matrix step is 512 elements); 4 otherwise, so that two work-groups share a
// compute unit and one's memory phases overlap the other's products. With 4 waves for 256
// work-groups and for tiles of 2048 in 84 KiB a single 2^19 took 111 us, now 97, eight of them
// 594, now 518 (2^18: 72, 66; 2^17: 52.2, 49.7); with 8 waves everywhere eight of 2^17 take 213
// instead of 161.
static uint32_t pass_threads(uint32_t rg, uint64_t groups, uint32_t lds_bytes)
{
    return rg >= 4096 || groups <= 256 || 2 * lds_bytes > kMaxPassLds ? 512 : 256;
}

RustError ntt_run(const NttTables& t, uint32_t log_n, const NttJob* jobs, int count, uint64_t in_len,
    Fr* scratch, uint64_t scratch_slots, NttTwist twist, NttPost post, const Fr& scale, hipStream_t stream)
{
    if (count <= 0)
        return ok();
    H2_CHECK_ARG(log_n >= 1 && log_n <= NTT_MAX_LOG, "NTT log_n=%u out of range [1, %u]", log_n, NTT_MAX_LOG);
    H2_TRY(raise_lds_limits());
    const NttPlan p = ntt_plan(log_n);
    const uint64_t N = 1ull << log_n;
    bool aliased = false;
    for (int i = 0; i < count; ++i)
        aliased |= (const void*)jobs[i].in == (const void*)jobs[i].out;
    const bool need_scratch = p.P == 3 || (p.P == 2 && aliased);
    H2_CHECK_ARG(!need_scratch || (scratch != nullptr && scratch_slots > 0), "NTT of 2^%u needs a scratch buffer",
        log_n);
    int max_batch = NTT_MAX_BATCH;
    if (need_scratch && scratch_slots < (uint64_t)max_batch)
        max_batch = (int)scratch_slots;
    uint32_t pc[3][9], bias8[9];
    host_post(post, scale, pc);
    host_bias8(post, scale, bias8);

    for (int base = 0; base < count; base += max_batch) {
        const int nb = count - base < max_batch ? count - base : max_batch;
        for (int pass = 0; pass < p.P; ++pass) {
            PassBatch pb {};
            for (int i = 0; i < nb; ++i) {
                const NttJob& jb = jobs[base + i];
                Fr* s = scratch ? scratch + (uint64_t)i * N : nullptr;
                const Fr* src;
                Fr* dst;
                if (p.P == 1) {
                    src = jb.in;
                    dst = jb.out;
                } else if (p.P == 2) {
                    Fr* mid = need_scratch ? s : jb.out;
                    src = pass == 0 ? jb.in : mid;
                    dst = pass == 0 ? mid : jb.out;
                } else {
                    src = pass == 0 ? jb.in : (pass == 1 ? s : jb.out);
                    dst = pass == 0 ? s : jb.out;
                }
                pb.in[i] = src;
                pb.out[i] = dst;
            }
            PassParams pp {};
            pp.log_n = log_n;
            pp.log_r = p.log_r[pass];
            pp.log_g = p.log_g[pass];
            uint32_t log_l = 0;
            for (int q = 0; q < pass; ++q)
                log_l += p.log_r[q];
            pp.log_l = log_l;
            pp.in_len = pass == 0 ? in_len : N;
            pp.tw_lo = t.tw_lo;
            pp.tw_hi = t.tw_hi;
            pp.h = t.h;
            pp.twr = t.twr[pass];
            pp.c_rows = t.c_rows;
            pp.c_cols = t.c_cols;
            pp.twist = pass == 0 ? (int)twist : TWIST_NONE;
            pp.last = pass == p.P - 1;
            pp.post = pp.last ? (int)post : POST_NONE;
            memcpy(pp.pc, pc, sizeof(pc));
            memcpy(pp.bias8, bias8, sizeof(bias8));
            pp.unit = t.unit;
            pp.last_matrices = t.last_matrices;
            if (log_n >= NTT_MATRIX_LOG)
                pp.steps = radix_steps(pp.log_r);
            const uint32_t RG = 1u << (pp.log_r + pp.log_g);
            const uint32_t nwg = (uint32_t)(N >> (pp.log_r + pp.log_g));
            pp.xcd_remap = (nwg % 8 == 0 && nwg >= 64) ? 1u : 0u;
            dim3 grid(nwg, nb);
            {
                ProfScope prof("ntt_pass", stream);
                const uint32_t lds = pass_lds_bytes(pp.log_r, pp.log_g, pp.last);
                ntt_pass_kernel<<<grid, pass_threads(RG, (uint64_t)nwg * nb, lds), lds, stream>>>(pb, pp);
            }
            H2_LAUNCH_CHECK();
        }
    }
    return ok();
}

// ---------------------------------------------------------- uneven batches

uint64_t ntt_batch_pass_bytes(int count) { return 3ull * (uint64_t)count * sizeof(BatchPass); }

RustError ntt_run_batch(const NttBatchJob* jobs, int count, NttTwist twist, NttPost post, void* d_pass,
    hipStream_t stream)
{
    if (count <= 0)
        return ok();
    H2_TRY(raise_lds_limits());
    std::vector<BatchPass> host(3ull * count);
    uint32_t nlaunch[3] = { 0, 0, 0 }, grid[3] = { 0, 0, 0 }, rgmax[3] = { 0, 0, 0 }, lds[3] = { 0, 0, 0 }; // rgmax: log2
    for (int i = 0; i < count; ++i) {
        const NttBatchJob& jb = jobs[i];
        H2_CHECK_ARG(jb.log_n >= 1 && jb.log_n <= NTT_MAX_LOG, "NTT batch: log_n=%u out of range [1, %u]", jb.log_n,
            NTT_MAX_LOG);
        NttPlan p = ntt_plan(jb.log_n);
        if (p.P > 1) // whole 4096-element tiles: a batch fills the chip with many transforms, not wide ones
            for (int q = 0; q < p.P; ++q) {
                const uint32_t g = (p.log_r[q] < 8 ? NTT_MAX_LOG_R - 1 : NTT_MAX_LOG_R) - p.log_r[q];
                p.log_g[q] = g < jb.log_n - p.log_r[q] ? g : jb.log_n - p.log_r[q];
            }
        H2_CHECK_ARG(p.P < 3 || jb.scratch, "NTT batch: 2^%u needs a scratch buffer", jb.log_n);
        H2_CHECK_ARG(p.P != 2 || (const void*)jb.in != (const void*)jb.out, "NTT batch: in-place 2^%u transform",
            jb.log_n);
        uint32_t pc[3][9], bias8[9];
        host_post(post, jb.scale, pc);
        host_bias8(post, jb.scale, bias8);
        for (int pass = 0; pass < p.P; ++pass) {
            BatchPass bp {};
            if (p.P == 1) {
                bp.in = jb.in;
                bp.out = jb.out;
            } else if (p.P == 2) {
                bp.in = pass == 0 ? jb.in : jb.out;
                bp.out = jb.out;
            } else {
                bp.in = pass == 0 ? jb.in : (pass == 1 ? jb.scratch : jb.out);
                bp.out = pass == 0 ? jb.scratch : jb.out;
            }
            PassParams& pp = bp.pp;
            pp.log_n = jb.log_n;
            pp.log_r = p.log_r[pass];
            pp.log_g = p.log_g[pass];
            uint32_t log_l = 0;
            for (int q = 0; q < pass; ++q)
                log_l += p.log_r[q];
            pp.log_l = log_l;
            pp.in_len = pass == 0 ? jb.in_len : (1ull << jb.log_n);
            pp.tw_lo = jb.tables->tw_lo;
            pp.tw_hi = jb.tables->tw_hi;
            pp.h = jb.tables->h;
            pp.twr = jb.tables->twr[pass];
            pp.c_rows = jb.tables->c_rows;
            pp.c_cols = jb.tables->c_cols;
            pp.twist = pass == 0 ? (int)twist : TWIST_NONE;
            pp.last = pass == p.P - 1;
            pp.post = pp.last ? (int)post : POST_NONE;
            memcpy(pp.pc, pc, sizeof(pc));
            memcpy(pp.bias8, bias8, sizeof(bias8));
            pp.unit = jb.tables->unit;
            pp.last_matrices = jb.tables->last_matrices;
            if (jb.log_n >= NTT_MATRIX_LOG)
                pp.steps = radix_steps(pp.log_r);
            const uint32_t rg = pp.log_r + pp.log_g;
            bp.nwg = (uint32_t)((1ull << jb.log_n) >> (pp.log_r + pp.log_g));
            // as ntt_run (two of 2^22 1046 -> 1001 us); the transform's first block only rotates the XCDs
            pp.xcd_remap = (bp.nwg % 8 == 0 && bp.nwg >= 64) ? 1u : 0u;
            bp.block0 = grid[pass];
            grid[pass] += bp.nwg;
            if (rg > rgmax[pass])
                rgmax[pass] = rg;
            const uint32_t bytes = pass_lds_bytes(pp.log_r, pp.log_g, pp.last);
            if (bytes > lds[pass])
                lds[pass] = bytes;
            host[(uint64_t)pass * count + nlaunch[pass]++] = bp;
        }
    }
    // pinned staging: the host table may go away on return without draining the stream
    {
        RustError e = stage_upload(d_pass, host.data(), sizeof(BatchPass) * host.size(), nullptr, nullptr, 0, stream);
        if (e.code)
            return e;
    }
    const BatchPass* dp = (const BatchPass*)d_pass;
    for (int pass = 0; pass < 3; ++pass) {
        if (!nlaunch[pass])
            continue;
        ProfScope prof("ntt_pass_batch", stream);
        ntt_pass_batch_kernel<<<grid[pass], pass_threads(1u << rgmax[pass], grid[pass], lds[pass]), lds[pass],
            stream>>>(dp + (uint64_t)pass * count, nlaunch[pass]);
        H2_LAUNCH_CHECK();
    }
    return ok();
}

RustError ntt_set_tiles(const uint8_t* tiles, uint32_t count)
{
    H2_CHECK_ARG(count <= NTT_MAX_LOG + 1, "h2amd_ntt_set_tiles: %u entries exceed %u", count, NTT_MAX_LOG + 1);
    for (uint32_t i = 0; i < count; ++i)
        H2_CHECK_ARG(tiles[i] == 0 || (tiles[i] >= 6 && tiles[i] <= NTT_MAX_LOG_R),
            "h2amd_ntt_set_tiles: tile 2^%u for 2^%u outside [2^6, 2^%u]", tiles[i], i, NTT_MAX_LOG_R);
    for (uint32_t i = 0; i <= NTT_MAX_LOG; ++i)
        g_tile_table[i].store(i < count ? tiles[i] : 0, std::memory_order_relaxed);
    return ok();
}

} // namespace h2
