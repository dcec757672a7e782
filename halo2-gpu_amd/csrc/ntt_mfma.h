// Radix-16 and radix-8 DFT steps of Fr vectors on the matrix cores.
//
// A radix-r DFT is a contraction: y_j = sum_a w^(aj) x_a with r-th roots w^e. An element is
// 32 bytes, and multiplying by a constant is linear in them: byte b of x contributes
// x_b (w^e 2^(8b) mod m). So w^e is a 32 x 32 matrix of 8-bit digits (column b = the digits
// of w^e 2^(8b) mod m) and y_j is a sum of r matrix-vector products over bytes: one
// v_mfma_i32_32x32x32_i8 per (a, j) for 32 vectors at once, every position of the transform
// that takes the same step being a vector. The 32-bit column sums are then carried into
// limbs and reduced, together with the multiplication by the position's twiddle, by one
// Montgomery product. Per element and 4 levels that is one product and ~160 instructions
// around it, where radix-4 butterflies in the vector unit took two products and the reduced
// additions, ~790 instructions. The matrix cores run beside the vector unit (16 products of
// 32 cycles per 64 outputs, after the even/odd split below; leaving them out of a 2^24
// transform saves 3% of its time). What bounds a step now is the vector unit's issue: ~430
// instructions per element at ~4 cycles per wave. Coset transforms, against the radix-4 form:
// 2^16 x 9 125 -> 103 us, 2^20 0.165 -> 0.147 ms, 2^22 0.60 -> 0.55 ms, 2^24 2.60 -> 2.40 ms
// (0.78 ms of it the loads and stores of columns 128 KiB apart).
//
// Digits: the matrix columns are the centred residues (|v| <= m/2) in balanced digits
// [-128, 127], the data bytes x_b - 128 (one XOR). The shift by 128 drops out: its
// contribution to y_j is -K sum_a w^(aj), K = sum_b 128 2^(8b), which is 0 mod m but for
// j = 0, where r K is added back. The value of y_j that the column sums spell is signed,
// |y_j| <= 32 * 128 * r * m / 2 = 2^11 r m.
// A column sum (32-bit) is below 2^21.91 in absolute value, r * 128 included (worst row
// over all j of the exact digits, r = 16), so a pair c0 + 2^8 c1 fits an int32. The last step's
// matrices carry the output's scale s (2^29 s w^e): for an arbitrary s their sums are those of
// 512 digits that nobody chooses, 2^22 on average and 39 standard deviations from 2^23.
//
// Even / odd split: w^(r/2) = -1, so with E_j and O_j the sums over even and odd a,
// y_j = E_j + O_j and y_(j + r/2) = E_j - O_j: half the matrix products.
//
// The roots: every primitive 16th root is g^u (g = kG16, u odd), so the matrices are the
// constants of g^e, and the transform's own root only permutes them (e -> u e mod 16).
#pragma once

#include "field29.h"

namespace h2 {

typedef int mfma_v4 __attribute__((ext_vector_type(4)));
typedef int mfma_v16 __attribute__((ext_vector_type(16)));

struct FrRoots16 {
    uint32_t a[4096]; // [e][lane][4 words]: lane l holds row l & 31, input bytes 16 (l >> 5) ..+15 of g^e's matrix
    uint32_t mont[8][8]; // g^(2i + 1) 2^256 mod m, canonical
};

namespace fr_roots {

struct U256 {
    uint64_t v[4];
};
constexpr U256 kM { { 0x43e1f593f0000001ull, 0x2833e84879b97091ull, 0xb85045b68181585dull, 0x30644e72e131a029ull } };
constexpr U256 kG16 { { 0xb11509c6e306460bull, 0x996dfbe1174efb98ull, 0x1c6e4f4594dd508cull,
    0x21082ca216cbbf4eull } }; // 7^((m - 1) / 16)

constexpr bool geq(const U256& a, const U256& b)
{
    for (int i = 3; i >= 0; --i)
        if (a.v[i] != b.v[i])
            return a.v[i] > b.v[i];
    return true;
}
constexpr U256 sub(const U256& a, const U256& b)
{
    U256 r {};
    uint64_t br = 0;
    for (int i = 0; i < 4; ++i) {
        r.v[i] = a.v[i] - b.v[i] - br;
        br = (a.v[i] < b.v[i] || (a.v[i] == b.v[i] && br)) ? 1 : 0;
    }
    return r;
}
constexpr U256 dbl(const U256& a) // 2 a mod m, a < m < 2^254
{
    U256 r {};
    for (int i = 0; i < 4; ++i)
        r.v[i] = (a.v[i] << 1) | (i ? a.v[i - 1] >> 63 : 0);
    return geq(r, kM) ? sub(r, kM) : r;
}
constexpr U256 addm(const U256& a, const U256& b)
{
    U256 r {};
    uint64_t c = 0;
    for (int i = 0; i < 4; ++i) {
        const uint64_t s = a.v[i] + b.v[i];
        r.v[i] = s + c;
        c = (s < a.v[i] || r.v[i] < s) ? 1 : 0;
    }
    return geq(r, kM) ? sub(r, kM) : r;
}
constexpr U256 mulm(const U256& a, const U256& b)
{
    U256 r {};
    for (int i = 255; i >= 0; --i) {
        r = dbl(r);
        if ((b.v[i >> 6] >> (i & 63)) & 1)
            r = addm(r, a);
    }
    return r;
}

constexpr FrRoots16 make()
{
    FrRoots16 t {};
    U256 w { { 1, 0, 0, 0 } };
    for (int e = 0; e < 16; ++e) {
        U256 v = w;
        for (int b = 0; b < 32; ++b) {
            // centred: v or v - m (two's complement), whichever is the smaller
            const U256 neg = sub(kM, v);
            const U256 c = geq(neg, v) ? v : sub(U256 {}, neg);
            uint32_t carry = 0;
            for (int row = 0; row < 32; ++row) {
                const uint32_t s = (uint32_t)((c.v[row >> 3] >> (8 * (row & 7))) & 255) + carry;
                carry = s >= 128 ? 1 : 0; // the digit is s or s - 256
                const int lane = row + 32 * (b >> 4);
                t.a[(e * 64 + lane) * 4 + ((b & 15) >> 2)] |= (s & 255) << (8 * (b & 3));
            }
            for (int k = 0; k < 8; ++k)
                v = dbl(v);
        }
        if (e & 1) {
            U256 x = w;
            for (int k = 0; k < 256; ++k)
                x = dbl(x);
            for (int i = 0; i < 8; ++i)
                t.mont[e >> 1][i] = (uint32_t)(x.v[i >> 1] >> (32 * (i & 1)));
        }
        w = mulm(w, kG16);
    }
    return t;
}

} // namespace fr_roots

__device__ constexpr FrRoots16 kFrRoots16 = fr_roots::make();

// acc + a b of signed 32-bit factors (one v_mad_i64_i32; as C the compiler takes the sign
// extension and the shift apart)
__device__ __forceinline__ int64_t mad_i64(int32_t a, int32_t b, int64_t acc)
{
    uint64_t carry;
    asm("v_mad_i64_i32 %0, %1, %2, %3, %0" : "+v"(acc), "=s"(carry) : "v"(a), "s"(b));
    return acc;
}

// Column (e, byte) of a matrix table (FrRoots16::a's layout) from a canonical value
__device__ __forceinline__ void store_matrix_column(uint8_t* a, uint32_t e, uint32_t byte, const Fr29& v)
{
    // centred: v or v - m as two's complement over 256 bits
    uint32_t w[8], n[8], twice[8];
    v.to32(w);
    int64_t br = 0, cmp = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        br += (int64_t)w[k] - FrParams::M[k];
        n[k] = (uint32_t)br;
        br >>= 32;
        twice[k] = (w[k] << 1) | (k ? w[k - 1] >> 31 : 0u); // 2 v < 2^255
        cmp += (int64_t)FrParams::M[k] - twice[k];
        cmp >>= 32;
    }
    uint32_t carry = 0;
#pragma unroll
    for (int row = 0; row < 32; ++row) {
        const uint32_t word = cmp < 0 ? n[row >> 2] : w[row >> 2]; // 2 v > m: v - m
        const uint32_t s = ((word >> (8 * (row & 3))) & 255) + carry;
        carry = s >= 128 ? 1 : 0;
        a[(e * 64 + row + 32 * (byte >> 4)) * 16 + (byte & 15)] = (uint8_t)s;
    }
}

// Montgomery product of a 10-limb value a, |a| < 2^271 (limbs 0..8 in [0, 2^29), limb 9
// signed), and b (9 normalised limbs, < m), radix 2^290, plus m: a b / 2^290 mod m as
// normalised limbs of a value in (m - 2^-19 m, 2m + 2^-19 m). Columns hold at most 18
// products of < 2^58 (the last quotient, which adds the m, is < 2^30).
__device__ __forceinline__ Fr29 mul_10x9(const uint32_t (&a)[10], const Fr29& b)
{
    using P = Fr29P;
    constexpr uint32_t MASK = Fr29::MASK;
    uint32_t q[10];
    uint64_t acc = 0;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
#pragma unroll
        for (int i = 0; i <= k; ++i)
            acc += (uint64_t)a[i] * b.l[k - i];
#pragma unroll
        for (int i = 0; i < k; ++i)
            acc += (uint64_t)q[i] * P::M[k - i];
        q[k] = ((uint32_t)acc * P::PINV) & MASK;
        acc += (uint64_t)q[k] * P::M[0];
        acc >>= 29;
    }
    Fr29 r;
    int64_t s = (int64_t)acc;
#pragma unroll
    for (int k = 9; k < 18; ++k) {
#pragma unroll
        for (int i = k - 8; i <= 8; ++i) {
            s += (int64_t)((uint64_t)a[i] * b.l[k - i]);
            s += (int64_t)((uint64_t)q[i] * P::M[k - i]);
        }
        s += (int64_t)(int32_t)a[9] * (int64_t)(int32_t)b.l[k - 9];
        if (k == 9)
            q[9] = (((uint32_t)s * P::PINV) & MASK) + (MASK + 1);
        s += (int64_t)((uint64_t)q[9] * P::M[k - 9]);
        if (k > 9)
            r.l[k - 10] = (uint32_t)s & MASK;
        s >>= 29;
    }
    r.l[8] = (uint32_t)s;
    return r;
}

// (v + q m) / 2^29 for the q < 2^29 that makes it whole (limbs 0..8 < 2^31): |v| <= 2^15 m + 2^259 gives a value in
// (-2^-13 m, m + 2^-13 m), nearly always canonical; the other two cases sit behind a branch.
__device__ __forceinline__ Fr29 mont_step(const uint32_t (&v)[10])
{
    using P = Fr29P;
    const uint32_t q = (v[0] * P::PINV) & Fr29::MASK;
    uint64_t acc = ((uint64_t)q * P::M[0] + v[0]) >> 29;
    Fr29 r;
#pragma unroll
    for (int k = 1; k < 9; ++k) {
        acc += (uint64_t)q * P::M[k] + v[k];
        r.l[k - 1] = (uint32_t)acc & Fr29::MASK;
        acc >>= 29;
    }
    const int32_t top = (int32_t)((uint32_t)acc + v[9]);
    r.l[8] = (uint32_t)top;
    if (top < 0 || (uint32_t)top >= P::M[8]) {
        const int32_t sign = top < 0 ? 1 : -1; // + m, or - m if that is not negative
        Fr29 t;
        int32_t c = 0;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int32_t d = (int32_t)r.l[k] + sign * (int32_t)P::M[k] + c;
            t.l[k] = (uint32_t)d & Fr29::MASK;
            c = d >> 29;
            if (k == 8)
                t.l[8] = (uint32_t)d;
        }
        if ((int32_t)t.l[8] >= 0)
            r = t;
    }
    return r;
}

// normalised r < 3m -> canonical
__device__ __forceinline__ Fr29 canonical_3m(Fr29 r)
{
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        Fr29 t;
        int32_t b = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int32_t d = (int32_t)r.l[i] - (int32_t)Fr29P::M[i] + b;
            t.l[i] = (uint32_t)d & Fr29::MASK;
            b = d >> 29;
        }
#pragma unroll
        for (int i = 0; i < 9; ++i)
            r.l[i] = b < 0 ? r.l[i] : t.l[i];
    }
    return r;
}

// The sums S = E + O (y_j, lower lanes) and D = E - O (y_(j + r/2), upper lanes) of 32
// vectors, from the accumulators, as 10 limbs per lane (the last one signed): lane l < 32
// gets vector l's y_j, lane l + 32 the same vector's y_(j + r/2). An accumulator has 16 of
// the 32 digits of its vector's value (register i is digit 8 (i / 4) + 4 (l / 32) + i % 4,
// the other half-wave has the rest): neighbouring digits pair up, the half-waves exchange S
// pairs for D pairs, and the 16 pairs (2^16 apart) are carried into 29-bit limbs. `bias` is
// added to every S pair.
__device__ __forceinline__ void mfma_limbs(const mfma_v16& E, const mfma_v16& O, int bias, uint32_t (&a)[10])
{
    int P[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = E[2 * i] + 256 * E[2 * i + 1], o = O[2 * i] + 256 * O[2 * i + 1];
        const auto w = __builtin_amdgcn_permlane32_swap((unsigned)(e + o + bias), (unsigned)(e - o), false, false);
        P[4 * (i / 2) + i % 2] = (int)w[0];
        P[4 * (i / 2) + i % 2 + 2] = (int)w[1];
    }
    int64_t acc = P[0];
    int p = 1;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (p < 16 && 16 * p < 29 * (k + 1)) {
                acc = mad_i64(P[p], 1 << (16 * p - 29 * k), acc);
                ++p;
            }
        a[k] = (uint32_t)acc & Fr29::MASK;
        acc >>= 29;
    }
    a[9] = (uint32_t)acc;
}

} // namespace h2
