// BN254 G1 bucket arithmetic on the 29-bit-limb field form (field29.h).
//
// Same formulas as curve.h (EFD, short Weierstrass a = 0, XYZZ coordinates:
// madd-2008-s, add-2008-s, dbl-2008-s, mdbl-2008-s) with lazy reduction.
// Every coordinate lives in the 2^261 Montgomery scale; the MSM converts the
// bases into it once per call and converts the result back.
//
// State invariant: the four coordinates of a G1X29 are normalised; X < 5.2m, the others
// < 2m (X is a square plus 4m minus three products, left as it is: 5.2m < 2^256 still fits a
// 32-byte word, and every product below has room for it, (5.2m)^2 < 2^261 m; Y is a sum of
// two products under one reduction, mul_sum, < 1.2m; ZZ and ZZZ are products). Affine inputs
// are canonical (< m). A product of values a and b (in units of m) is < 1 + a b / 169; the
// comments give the bounds in units of m.
//
// The formulas carry as little as they can: a difference that only enters mul_sum's wide
// operand is left with limbs up to 1.5 2^30, and P = 0 (the doubling / identity case) is read
// off P^2, whose zero has two representatives, so P itself needs no reduction. Against the
// form with X and P reduced below 2m and every difference normalised, the bucket
// accumulation of five 2^20-row table commitments took 4.33 instead of 4.67 ms, that of a
// 3 000 001 point MSM 3.34 instead of 3.60 ms (it is bound by the 1548 multiply-adds of an
// addition: 18.2 G additions/s is 28 T multiply-adds/s of the ~33 T/s a loop of nothing
// else reaches).
#pragma once

#include "curve.h"
#include "field29.h"

namespace h2 {

using Fq29 = F29<Fq29P>;

__device__ __forceinline__ Fq29 nsub2(const Fq29& a, const Fq29& b) { return Fq29::normalize(Fq29::sub2(a, b)); }
// 4m - b with limbs < 2^30 (b normalised, < 4m): the negation mul_sum takes as its last operand
__device__ __forceinline__ Fq29 neg4(const Fq29& b) { return Fq29::sub4(Fq29::zero(), b); }

struct G1A29 {
    Fq29 x, y;

    __device__ __forceinline__ static G1A29 load(const void* p)
    {
        const uint8_t* b = (const uint8_t*)p;
        return G1A29 { Fq29::load32(b), Fq29::load32(b + 32) };
    }
    __device__ __forceinline__ bool is_inf() const { return x.is_zero() && y.is_zero(); }
    // -(x, y) = (x, 2m - y): y stays < 2m, normalised (G1 has no 2-torsion, y != 0)
    __device__ __forceinline__ G1A29 neg() const { return is_inf() ? *this : G1A29 { x, nsub2(Fq29::zero(), y) }; }
};

struct G1X29 {
    Fq29 X, Y, ZZ, ZZZ;

    __device__ __forceinline__ static G1X29 inf()
    {
        return G1X29 { Fq29::one(), Fq29::one(), Fq29::zero(), Fq29::zero() };
    }
    __device__ __forceinline__ bool is_inf() const { return ZZ.is_zero(); }

    __device__ __forceinline__ static G1X29 from_affine(const G1A29& a)
    {
        if (a.is_inf())
            return inf();
        return G1X29 { a.x, a.y, Fq29::one(), Fq29::one() };
    }

    // 128 bytes: four coordinates in the 32-byte word layout (values < 2m < 2^256)
    __device__ __forceinline__ static G1X29 load(const void* p)
    {
        const uint8_t* b = (const uint8_t*)p;
        return G1X29 { Fq29::load32(b), Fq29::load32(b + 32), Fq29::load32(b + 64), Fq29::load32(b + 96) };
    }
    __device__ __forceinline__ void store(void* p) const
    {
        uint8_t* b = (uint8_t*)p;
        X.store32(b);
        Y.store32(b + 32);
        ZZ.store32(b + 64);
        ZZZ.store32(b + 96);
    }

    // mdbl-2008-s: 2 (x, y), affine non-identity input
    __device__ __forceinline__ static G1X29 dbl_affine(const G1A29& a)
    {
        const Fq29 U = Fq29::add(a.y, a.y); // < 4, limbs < 2^30
        const Fq29 V = Fq29::sqr(U); // < 1.1
        const Fq29 W = Fq29::mul(U, V);
        const Fq29 S = Fq29::mul(a.x, V);
        const Fq29 x2 = Fq29::sqr(a.x);
        const Fq29 M = Fq29::normalize(Fq29::add(Fq29::add(x2, x2), x2)); // < 3.5
        G1X29 r;
        r.X = Fq29::normalize(Fq29::sub4_wide(Fq29::sqr(M), Fq29::add(S, S))); // < 5.1
        // M (S - X3) - W y with one reduction: < 1 + (3.5 * 7.1 + 1.1 * 4) / 169 < 1.2
        r.Y = Fq29::mul_sum(M, Fq29::sub6(S, r.X), W, neg4(a.y));
        r.ZZ = V;
        r.ZZZ = W;
        return r;
    }

    // dbl-2008-s (out of line: it is the rare branch of add)
    __device__ __noinline__ static G1X29 dbl(const G1X29& p) { return dbl_inline(p); }

    __device__ __forceinline__ static G1X29 dbl_inline(const G1X29& p)
    {
        if (p.is_inf())
            return p;
        const Fq29 U = Fq29::add(p.Y, p.Y); // < 4, limbs < 2^30
        const Fq29 V = Fq29::sqr(U);
        const Fq29 W = Fq29::mul(U, V);
        const Fq29 S = Fq29::mul(p.X, V);
        const Fq29 x2 = Fq29::sqr(p.X);
        const Fq29 M = Fq29::normalize(Fq29::add(Fq29::add(x2, x2), x2));
        G1X29 r;
        r.X = Fq29::normalize(Fq29::sub4_wide(Fq29::sqr(M), Fq29::add(S, S)));
        r.Y = Fq29::mul_sum(M, Fq29::sub6(S, r.X), W, neg4(p.Y)); // < 1.2, as in dbl_affine
        r.ZZ = Fq29::mul(V, p.ZZ);
        r.ZZZ = Fq29::mul(W, p.ZZZ);
        return r;
    }

    // madd-2008-s with the exceptional cases: p + q (q affine) or, with `neg`, p - q. The
    // sign goes into S2 = y ZZZ, whose difference with Y is normalised anyway.
    __device__ static G1X29 add_affine(const G1X29& p, const G1A29& q, bool neg = false)
    {
        if (q.is_inf())
            return p;
        if (p.is_inf())
            return from_affine(neg ? q.neg() : q);
        const Fq29 U2 = Fq29::mul(q.x, p.ZZ);
        Fq29 S2 = Fq29::mul(q.y, p.ZZZ); // < 1.02
#pragma unroll
        for (int i = 0; i < 9; ++i)
            S2.l[i] = neg ? Fq29P::K2M[i] - S2.l[i] : S2.l[i]; // 2 - S2, limbs < 2^30
        const Fq29 P = Fq29::normalize(Fq29::sub6(U2, p.X)); // < 7.1
        const Fq29 R = nsub2(S2, p.Y); // < 4
        const Fq29 PP = Fq29::sqr(P); // < 1.3
        if (Fq29::is_zero_mod_rare(PP)) {
            if (Fq29::is_zero_mod(Fq29::reduce_2m(R)))
                return dbl_affine(neg ? q.neg() : q);
            return inf();
        }
        const Fq29 PPP = Fq29::mul(P, PP);
        const Fq29 Q = Fq29::mul(p.X, PP);
        G1X29 r;
        r.X = Fq29::normalize(Fq29::sub4_wide(Fq29::sqr(R), Fq29::add(PPP, Fq29::add(Q, Q)))); // < 5.2
        // R (Q - X3) - Y1 PPP with one reduction: < 1 + (4 * 7.1 + 2 * 4) / 169 < 1.3
        r.Y = Fq29::mul_sum(R, Fq29::sub6(Q, r.X), p.Y, neg4(PPP));
        r.ZZ = Fq29::mul(p.ZZ, PP);
        r.ZZZ = Fq29::mul(p.ZZZ, PPP);
        return r;
    }

    // add-2008-s with the exceptional cases
    __device__ static G1X29 add(const G1X29& p, const G1X29& q)
    {
        if (q.is_inf())
            return p;
        if (p.is_inf())
            return q;
        const Fq29 U1 = Fq29::mul(p.X, q.ZZ); // < 1.1
        const Fq29 U2 = Fq29::mul(q.X, p.ZZ);
        const Fq29 S1 = Fq29::mul(p.Y, q.ZZZ);
        const Fq29 S2 = Fq29::mul(q.Y, p.ZZZ);
        const Fq29 P = nsub2(U2, U1); // < 3.1
        const Fq29 R = nsub2(S2, S1);
        const Fq29 PP = Fq29::sqr(P);
        if (Fq29::is_zero_mod_rare(PP)) {
            if (Fq29::is_zero_mod(Fq29::reduce_2m(R)))
                return dbl_inline(p);
            return inf();
        }
        const Fq29 PPP = Fq29::mul(P, PP);
        const Fq29 Q = Fq29::mul(U1, PP);
        G1X29 r;
        r.X = Fq29::normalize(Fq29::sub4_wide(Fq29::sqr(R), Fq29::add(PPP, Fq29::add(Q, Q)))); // < 5.2
        r.Y = Fq29::mul_sum(R, Fq29::sub6(Q, r.X), S1, neg4(PPP)); // < 1.2, as in add_affine
        r.ZZ = Fq29::mul(Fq29::mul(p.ZZ, q.ZZ), PP);
        r.ZZZ = Fq29::mul(Fq29::mul(p.ZZZ, q.ZZZ), PPP);
        return r;
    }

    // XYZZ -> Jacobian (X ZZ^2, Y ZZZ^2, ZZZ): x = X ZZ^2 / ZZZ^2 = X / ZZ and
    // y = Y ZZZ^2 / ZZZ^3 because ZZ^3 = ZZZ^2; the identity keeps Z = 0
    __device__ __forceinline__ void to_jacobian(Fq29& jx, Fq29& jy, Fq29& jz) const
    {
        jx = Fq29::mul(X, Fq29::sqr(ZZ));
        jy = Fq29::mul(Y, Fq29::sqr(ZZZ));
        jz = ZZZ;
    }
    __device__ __forceinline__ static G1X29 from_jacobian(const Fq29& jx, const Fq29& jy, const Fq29& jz)
    {
        const Fq29 zz = Fq29::sqr(jz);
        return G1X29 { jx, jy, zz, Fq29::mul(zz, jz) };
    }
};

} // namespace h2
