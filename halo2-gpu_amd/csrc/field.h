// BN254 prime-field arithmetic for gfx950 (CDNA4).
//
// Storage format (the boundary format of the reference's FFI, halo2curves'
// in-memory repr): 32 bytes, little-endian, Montgomery form a * 2^256 mod m,
// fully reduced. In registers an element is 8 x 32-bit limbs.
//
// Multiplication is Montgomery product scanning with interleaved reduction
// (FIPS, Koc-Acar-Kaliski 1996): every 32x32 partial product goes through one
// `v_mad_u64_u32` into a 64-bit column accumulator whose carry-out feeds a
// third accumulator word through `v_addc_co_u32`. This keeps the integer
// multiply-add unit (64 lanes/clk/CU on gfx950) the only hot resource.
// (Products by the constants of a DFT run on the matrix cores: ntt_mfma.h.)
//
// Constants (moduli, -m^-1 mod 2^32, R mod m, R^2 mod m) are BN254's; the
// reference keeps the same values at cuda/include/field/alt_bn128.hpp:19-47.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace h2 {

struct FrParams {
    static constexpr uint32_t M[8] = { 0xf0000001u, 0x43e1f593u, 0x79b97091u, 0x2833e848u,
        0x8181585du, 0xb85045b6u, 0xe131a029u, 0x30644e72u };
    static constexpr uint32_t INV = 0xefffffffu;
    static constexpr uint32_t ONE[8] = { 0x4ffffffbu, 0xac96341cu, 0x9f60cd29u, 0x36fc7695u,
        0x7879462eu, 0x666ea36fu, 0x9a07df2fu, 0x0e0a77c1u };
    static constexpr uint32_t R2[8] = { 0xae216da7u, 0x1bb8e645u, 0xe35c59e3u, 0x53fe3ab1u,
        0x53bb8085u, 0x8c49833du, 0x7f4e44a5u, 0x0216d0b1u };
    static constexpr uint32_t R3[8] = { 0xb4bf0040u, 0x5e94d8e1u, 0x1cfbb6b8u, 0x2a489cbeu, 0xa19fcfedu,
        0x893cc664u, 0x7fcc657cu, 0x0cf8594bu }; // 2^768 mod m
};

struct FqParams {
    static constexpr uint32_t M[8] = { 0xd87cfd47u, 0x3c208c16u, 0x6871ca8du, 0x97816a91u,
        0x8181585du, 0xb85045b6u, 0xe131a029u, 0x30644e72u };
    static constexpr uint32_t INV = 0xe4866389u;
    static constexpr uint32_t ONE[8] = { 0xc58f0d9du, 0xd35d438du, 0xf5c70b3du, 0x0a78eb28u,
        0x7879462cu, 0x666ea36fu, 0x9a07df2fu, 0x0e0a77c1u };
    static constexpr uint32_t R2[8] = { 0x538afa89u, 0xf32cfc5bu, 0xd44501fbu, 0xb5e71911u,
        0x0a417ff6u, 0x47ab1effu, 0xcab8351fu, 0x06d89f71u };
    static constexpr uint32_t R3[8] = { 0xda1530dfu, 0xb1cd6dafu, 0xa7283db6u, 0x62f210e6u, 0x0ada0afbu,
        0xef7f0b0cu, 0x2d592544u, 0x20fd6e90u }; // 2^768 mod m
};

// acc(64) + x*y -> acc, carry-out of the 64-bit sum added into c2.
__device__ __forceinline__ void mac96(uint64_t& acc, uint32_t& c2, uint32_t x, uint32_t y)
{
    uint64_t cm;
    asm("v_mad_u64_u32 %0, %1, %3, %4, %0\n\t"
        "v_addc_co_u32_e64 %2, %1, %2, 0, %1"
        : "+v"(acc), "=&s"(cm), "+v"(c2)
        : "v"(x), "v"(y));
}

// m (P::M) in 30-bit limbs
template <class P>
__host__ __device__ constexpr int32_t modulus30(int i)
{
    const int q = 30 * i / 32, s = 30 * i % 32;
    const uint64_t w = (uint64_t)(q < 8 ? P::M[q < 8 ? q : 7] : 0u)
        | (uint64_t)(q + 1 < 8 ? P::M[q + 1 < 8 ? q + 1 : 7] : 0u) << 32;
    return (int32_t)((w >> s) & 0x3fffffffu);
}

// x^-1 mod m (P::M, odd, < 2^254) for 0 < x < m, both as 8 little-endian 32-bit limbs, by
// division steps (Bernstein and Yang, "Fast constant-time gcd computation and modular
// inversion", 2019, in the form that starts at delta = 1/2). One step on (delta, f, g), f odd:
//   delta > 0 and g odd: (1 - delta, g, (g - f) / 2)
//   otherwise:           (1 + delta, f, (g + (g mod 2) f) / 2)
// It looks at parities only, so 30 steps depend on the low 32 bits of f and g; they are
// collected in a matrix (u v; q r), |u| + |v| and |q| + |r| <= 2^30, and (f, g) <- matrix (f, g)
// / 2^30 (exact) and (d, e) <- matrix (d, e) / 2^30 mod m (a multiple of m below 2^29 m in
// magnitude makes it exact) keep f = d x and g = e x (mod m). At g = 0, f = +-1 and
// x^-1 = +-d. 590 steps (20 rounds) reach it for inputs below 2^256; the loop's own limit of 25 is
// what bounds it. |d|, |e| grow by at most m / 2 a round.
//
// Within a round several steps are taken at once, in the way that P. Wuille's note "The safegcd
// implementation in libsecp256k1 explained" (2021) describes for public data: with theta = delta - 1/2, the trailing zeros
// of g are that many steps at once, and as long as theta < 0 the steps only add f to g, so
// w = -g / f mod 2^k clears k <= -theta bits by one multiple of f. When theta >= 0 and g is
// odd, f and g are exchanged (g' = -f, theta' = -theta - 1), and the step is one of adding.
// Variable time: the data is public.
//
// ONE: a single lane of the wave is active, so that the steps are held in scalar registers and
// their branches are scalar ones. What bounds that use is the chain of one lane: ~5 scalar
// instructions a step in the rounds and ~90 multiply-adds after each. Against 31 plain steps of
// the binary gcd on 64-bit images a round, the inversion of 128 totals (products.hip) takes
// 67 us instead of 127.
template <class P, bool ONE = false>
__host__ __device__ inline void inv_mod_plain(const uint32_t (&x)[8], uint32_t (&out)[8])
{
    constexpr int32_t M30 = 0x3fffffff;
    auto uniform = [](uint32_t t) -> uint32_t {
#ifdef __HIP_DEVICE_COMPILE__
        if constexpr (ONE)
            return (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
#endif
        return t;
    };
    int32_t f[9], g[9], d[9], e[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int q = 30 * i / 32, s = 30 * i % 32;
        const uint64_t w = (uint64_t)x[q] | (uint64_t)(q + 1 < 8 ? x[q + 1 < 8 ? q + 1 : 7] : 0u) << 32;
        f[i] = modulus30<P>(i);
        g[i] = (int32_t)((w >> s) & M30);
        d[i] = 0;
        e[i] = i == 0 ? 1 : 0;
#ifdef __HIP_DEVICE_COMPILE__
        if constexpr (ONE) { // in vector registers: v_mad_i64_i32 is one instruction, scalar four
            asm("" : "+v"(f[i]), "+v"(g[i]));
            asm("" : "+v"(d[i]), "+v"(e[i]));
        }
#endif
    }
    int theta = 0;
    for (int round = 0; round < 25; ++round) {
        int32_t any = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i)
            any |= g[i];
        if (uniform((uint32_t)any) == 0)
            break;
        uint32_t fl = uniform((uint32_t)f[0] | (uint32_t)f[1] << 30);
        uint32_t gl = uniform((uint32_t)g[0] | (uint32_t)g[1] << 30);
        uint32_t u = 1, v = 0, q = 0, r = 1; // two's complement, |.| <= 2^30
        int left = 30;
        for (;;) {
            const int z = __builtin_ctz(gl | 1u << left);
            gl >>= z;
            u <<= z;
            v <<= z;
            theta += z;
            left -= z;
            if (left == 0)
                break;
            if (theta >= 0) {
                uint32_t t = fl;
                fl = gl;
                gl = 0u - t;
                t = u;
                u = q;
                q = 0u - t;
                t = v;
                v = r;
                r = 0u - t;
                theta = -theta - 1;
            }
            int k = left < 6 ? left : 6;
#ifdef __HIP_DEVICE_COMPILE__
            if constexpr (ONE)
                asm("" : "+s"(k)); // not a three-way minimum, which only the vector unit has
#endif
            k = -theta < k ? -theta : k;
            // f (2 - f^2) = 1 / f mod 2^6 (f is its own inverse mod 2^3)
            const uint32_t w = (gl * fl * (fl * fl - 2u)) & ((1u << k) - 1u);
            gl += fl * w;
            q += u * w;
            r += v * w;
        }
        const int32_t ui = (int32_t)u, vi = (int32_t)v, qi = (int32_t)q, ri = (int32_t)r;
        int64_t cf = (int64_t)ui * f[0] + (int64_t)vi * g[0];
        int64_t cg = (int64_t)qi * f[0] + (int64_t)ri * g[0];
        int64_t cd = (int64_t)ui * d[0] + (int64_t)vi * e[0];
        int64_t ce = (int64_t)qi * d[0] + (int64_t)ri * e[0];
        // P::INV = -1 / m mod 2^32: the multiples of m that clear the low 30 bits, in [-2^29, 2^29)
        const int32_t md = (int32_t)((uint32_t)cd * P::INV << 2) >> 2;
        const int32_t me = (int32_t)((uint32_t)ce * P::INV << 2) >> 2;
        cd += (int64_t)md * modulus30<P>(0);
        ce += (int64_t)me * modulus30<P>(0);
        cf >>= 30;
        cg >>= 30;
        cd >>= 30;
        ce >>= 30;
#pragma unroll
        for (int i = 1; i < 9; ++i) {
            cf += (int64_t)ui * f[i] + (int64_t)vi * g[i];
            cg += (int64_t)qi * f[i] + (int64_t)ri * g[i];
            cd += (int64_t)ui * d[i] + (int64_t)vi * e[i] + (int64_t)md * modulus30<P>(i);
            ce += (int64_t)qi * d[i] + (int64_t)ri * e[i] + (int64_t)me * modulus30<P>(i);
            f[i - 1] = (int32_t)cf & M30;
            g[i - 1] = (int32_t)cg & M30;
            d[i - 1] = (int32_t)cd & M30;
            e[i - 1] = (int32_t)ce & M30;
            cf >>= 30;
            cg >>= 30;
            cd >>= 30;
            ce >>= 30;
        }
        f[8] = (int32_t)cf; // the sign is the top limb's
        g[8] = (int32_t)cg;
        d[8] = (int32_t)cd;
        e[8] = (int32_t)ce;
    }
    // d <- d * f (f = +-1), then into [0, m): |d| < 14 m
    const bool neg = f[8] < 0;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int32_t t = (neg ? -d[i] : d[i]) + c;
        d[i] = i < 8 ? t & M30 : t;
        c = t >> 30;
    }
    for (int k = 0; k < 14 && d[8] < 0; ++k) {
        c = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int32_t t = d[i] + modulus30<P>(i) + c;
            d[i] = i < 8 ? t & M30 : t;
            c = t >> 30;
        }
    }
    for (int k = 0; k < 14; ++k) {
        int32_t s[9];
        c = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int32_t t = d[i] - modulus30<P>(i) + c;
            s[i] = i < 8 ? t & M30 : t;
            c = t >> 30;
        }
        if (s[8] < 0)
            break;
#pragma unroll
        for (int i = 0; i < 9; ++i)
            d[i] = s[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = 32 * i / 30, s = 32 * i % 30;
        const uint64_t w = (uint64_t)(uint32_t)d[q] | (uint64_t)(uint32_t)d[q + 1] << 30;
        out[i] = (uint32_t)(w >> s);
    }
}

template <class P>
struct Fp256 {
    uint32_t v[8];

    __host__ __device__ __forceinline__ static Fp256 zero()
    {
        Fp256 r;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            r.v[i] = 0;
        return r;
    }
    __host__ __device__ __forceinline__ static Fp256 one()
    {
        Fp256 r;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            r.v[i] = P::ONE[i];
        return r;
    }
    __host__ __device__ __forceinline__ static Fp256 r2()
    {
        Fp256 r;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            r.v[i] = P::R2[i];
        return r;
    }
    __device__ __forceinline__ static Fp256 load(const void* p)
    {
        const uint4* q = (const uint4*)p;
        uint4 a = q[0], b = q[1];
        Fp256 r;
        r.v[0] = a.x; r.v[1] = a.y; r.v[2] = a.z; r.v[3] = a.w;
        r.v[4] = b.x; r.v[5] = b.y; r.v[6] = b.z; r.v[7] = b.w;
        return r;
    }
    __device__ __forceinline__ void store(void* p) const
    {
        uint4* q = (uint4*)p;
        q[0] = make_uint4(v[0], v[1], v[2], v[3]);
        q[1] = make_uint4(v[4], v[5], v[6], v[7]);
    }
    __device__ __forceinline__ bool is_zero() const
    {
        uint32_t o = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            o |= v[i];
        return o == 0;
    }
    __device__ __forceinline__ bool operator==(const Fp256& b) const
    {
        uint32_t o = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            o |= v[i] ^ b.v[i];
        return o == 0;
    }
    __device__ __forceinline__ bool operator!=(const Fp256& b) const { return !(*this == b); }

    // r = t - M if t >= M else t   (t < 2M)
    __device__ __forceinline__ static Fp256 reduce_once(const uint32_t* t)
    {
        uint32_t d[8];
        uint32_t borrow = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint64_t x = (uint64_t)t[j] - P::M[j] - borrow;
            d[j] = (uint32_t)x;
            borrow = (uint32_t)(x >> 32) & 1u;
        }
        Fp256 r;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            r.v[j] = borrow ? t[j] : d[j];
        return r;
    }

    __device__ __forceinline__ static Fp256 add(const Fp256& a, const Fp256& b)
    {
        uint32_t t[8];
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            c = (uint64_t)a.v[j] + b.v[j] + (c >> 32);
            t[j] = (uint32_t)c;
        }
        // a, b < M < 2^254: the sum never leaves 256 bits
        return reduce_once(t);
    }

    __device__ __forceinline__ static Fp256 sub(const Fp256& a, const Fp256& b)
    {
        uint32_t t[8];
        uint32_t borrow = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint64_t x = (uint64_t)a.v[j] - b.v[j] - borrow;
            t[j] = (uint32_t)x;
            borrow = (uint32_t)(x >> 32) & 1u;
        }
        uint32_t mask = 0u - borrow;
        Fp256 r;
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            c = (uint64_t)t[j] + (P::M[j] & mask) + (c >> 32);
            r.v[j] = (uint32_t)c;
        }
        return r;
    }

    __device__ __forceinline__ static Fp256 neg(const Fp256& a)
    {
        return sub(zero(), a);
    }

    __device__ __forceinline__ static Fp256 mul(const Fp256& a, const Fp256& b)
    {
        uint32_t m[8];
        uint32_t t[8];
        uint64_t acc = 0;
        uint32_t c2 = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int j = k - i;
                if (j >= 0 && j < 8)
                    mac96(acc, c2, a.v[i], b.v[j]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int j = k - i;
                if (i < k && j >= 1 && j < 8)
                    mac96(acc, c2, m[i], P::M[j]);
            }
            if (k < 8) {
                m[k] = (uint32_t)acc * P::INV;
                mac96(acc, c2, m[k], P::M[0]);
            } else {
                t[k - 8] = (uint32_t)acc;
            }
            acc = (acc >> 32) | ((uint64_t)c2 << 32);
            c2 = 0;
        }
        // M < 2^254 < R/4 keeps the FIPS output below 2M
        return reduce_once(t);
    }

    __device__ __forceinline__ static Fp256 sqr(const Fp256& a) { return mul(a, a); }

    __device__ __forceinline__ static Fp256 dbl(const Fp256& a) { return add(a, a); }

    // a^e for a small exponent (square-and-multiply, msb first)
    __device__ __forceinline__ static Fp256 pow_u64(const Fp256& a, uint64_t e)
    {
        Fp256 r = one();
        if (e == 0)
            return r;
        int top = 63 - __clzll(e);
        for (int i = top; i >= 0; --i) {
            r = sqr(r);
            if ((e >> i) & 1ull)
                r = mul(r, a);
        }
        return r;
    }

    // a^-1 by division steps (inv_mod_plain): plain inverse of the
    // stored word A = a R, times R^3 with one Montgomery product (A^-1 R^2 = a^-1 R);
    // inverse_vt(0) = 0
    __device__ static Fp256 inverse_vt(const Fp256& a)
    {
        if (a.is_zero())
            return zero();
        Fp256 ri, r3;
        inv_mod_plain<P>(a.v, ri.v);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            r3.v[i] = P::R3[i];
        return mul(ri, r3);
    }

    // a^(M-2) with 4-bit fixed windows; inverse(0) = 0
    __device__ static Fp256 inverse(const Fp256& a)
    {
        Fp256 tbl[16];
        tbl[0] = one();
        tbl[1] = a;
#pragma unroll
        for (int i = 2; i < 16; ++i)
            tbl[i] = mul(tbl[i - 1], a);
        uint32_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            e[i] = P::M[i];
        e[0] -= 2u; // M is odd and > 2, no borrow
        Fp256 r = one();
        bool started = false;
        for (int w = 63; w >= 0; --w) {
            uint32_t nib = (e[w >> 3] >> ((w & 7) * 4)) & 0xfu;
            if (started) {
                r = sqr(r);
                r = sqr(r);
                r = sqr(r);
                r = sqr(r);
            }
            if (nib) {
                // select without dynamic register indexing
                Fp256 s = tbl[0];
#pragma unroll
                for (int i = 1; i < 16; ++i)
                    if ((uint32_t)i == nib)
                        s = tbl[i];
                r = started ? mul(r, s) : s;
                started = true;
            }
        }
        return r;
    }

    __device__ __forceinline__ static Fp256 from_mont(const Fp256& a)
    {
        Fp256 o = zero();
        o.v[0] = 1;
        return mul(a, o);
    }
    __device__ __forceinline__ static Fp256 to_mont(const Fp256& a) { return mul(a, r2()); }
};

template <class P>
__device__ __forceinline__ Fp256<P> operator*(const Fp256<P>& a, const Fp256<P>& b) { return Fp256<P>::mul(a, b); }
template <class P>
__device__ __forceinline__ Fp256<P> operator+(const Fp256<P>& a, const Fp256<P>& b) { return Fp256<P>::add(a, b); }
template <class P>
__device__ __forceinline__ Fp256<P> operator-(const Fp256<P>& a, const Fp256<P>& b) { return Fp256<P>::sub(a, b); }

using Fr = Fp256<FrParams>;
using Fq = Fp256<FqParams>;

} // namespace h2
