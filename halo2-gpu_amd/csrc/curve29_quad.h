// One G1 point on four lanes: lane r of a quad holds coordinate r (X, Y, ZZ, ZZZ) of an
// XYZZ point, so the independent products of a point addition run side by side.
//
// Where a chain of dependent additions is what takes the time (the bucket reduction, the
// pieces of a split bucket), a lane that adds on its own spends 14 products one after the
// other; a quad spends 4, plus the exchanges between its lanes (DPP quad permutations,
// no LDS). It costs about 1.6 times the lane-instructions, so kernels with
// enough independent additions to fill the chip keep one lane per addition (G1X29::add).
//
// Same formulas and bounds as curve29.h; a quad's four lanes must take the same branches.
#pragma once

#include "curve29.h"

namespace h2 {

// value of lane (p_r) of the quad on lane r, p given as four 2-bit selectors. The moves stay
// moves: folded into a subtraction with the same register as the other operand
// (v_subrev_u32_dpp v, x, x) the compiler's form gave the negated difference.
template <int P0, int P1, int P2, int P3>
__device__ __forceinline__ Fq29 quad_perm(const Fq29& a)
{
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i)
        r.l[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)a.l[i], P0 | (P1 << 2) | (P2 << 4) | (P3 << 6), 0xf, 0xf,
            true);
#pragma unroll
    for (int i = 0; i < 9; ++i)
        asm("" : "+v"(r.l[i]));
    return r;
}
template <int P>
__device__ __forceinline__ bool quad_flag(bool f) // lane P's flag on all four lanes
{
    return __builtin_amdgcn_mov_dpp(f ? 1 : 0, P * 0x55, 0xf, 0xf, true) != 0;
}

__device__ __forceinline__ Fq29 fq_select(bool c, const Fq29& a, const Fq29& b)
{
    Fq29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i)
        r.l[i] = c ? a.l[i] : b.l[i];
    return r;
}

// lane r's coordinate of the identity (1, 1, 0, 0)
__device__ __forceinline__ Fq29 quad_inf(uint32_t r) { return fq_select(r < 2, Fq29::one(), Fq29::zero()); }

__device__ __forceinline__ bool quad_is_inf(const Fq29& p) { return quad_flag<2>(p.is_zero()); }

// lane r's 32 bytes of a 128-byte point slot
__device__ __forceinline__ Fq29 quad_load(const void* slot, uint32_t r)
{
    return Fq29::load32((const uint8_t*)slot + 32 * r);
}
__device__ __forceinline__ void quad_store(const Fq29& p, void* slot, uint32_t r)
{
    p.store32((uint8_t*)slot + 32 * r);
}

// dbl-2008-s
__device__ __forceinline__ Fq29 quad_dbl(const Fq29& p, uint32_t r)
{
    if (quad_is_inf(p))
        return p;
    // X^2 on lane 0, V = (2 Y)^2 on lane 1
    Fq29 a = p;
#pragma unroll
    for (int i = 0; i < 9; ++i)
        a.l[i] <<= r == 1 ? 1 : 0; // U = 2 Y, limbs < 2^30
    const Fq29 m1 = Fq29::sqr(a);
    const Fq29 V = quad_perm<1, 1, 1, 1>(m1);
    // S = X V on lane 0, W = U V on lane 1, ZZ3 = ZZ V on lane 2
    const Fq29 m2 = Fq29::mul(a, V);
    const Fq29 W = quad_perm<1, 1, 1, 1>(m2);
    const Fq29 M = Fq29::normalize(Fq29::add(Fq29::add(m1, m1), m1)); // lane 0: 3 X^2
    // M^2 on lane 0, W Y on lane 1, ZZZ3 = W ZZZ on lane 3
    const Fq29 m3 = Fq29::mul(fq_select(r == 0, M, p), fq_select(r == 0, M, W));
    const Fq29 X3 = Fq29::normalize(Fq29::sub4_wide(m3, Fq29::add(m2, m2))); // lane 0
    const Fq29 m4 = Fq29::mul(M, Fq29::sub6(m2, X3)); // lane 0: M (S - X3)
    // lane 1: M (S - X3) - W Y
    const Fq29 Y3 = Fq29::reduce_2m(nsub2(quad_perm<0, 0, 0, 0>(m4), m3));
    return fq_select(r < 2, fq_select(r == 0, X3, Y3), fq_select(r == 2, m2, m3));
}

// add-2008-s with the exceptional cases: p + q
__device__ __forceinline__ Fq29 quad_add(const Fq29& p, const Fq29& q, uint32_t r)
{
    if (quad_is_inf(q))
        return p;
    if (quad_is_inf(p))
        return q;
    // U1 = X1 ZZ2, S1 = Y1 ZZZ2, U2 = ZZ1 X2, S2 = ZZZ1 Y2 on lanes 0..3
    const Fq29 m1 = Fq29::mul(p, quad_perm<2, 3, 0, 1>(q));
    // P = U2 - U1 on lane 0, R = S2 - S1 on lane 1
    const Fq29 D = nsub2(quad_perm<2, 3, 0, 1>(m1), m1);
    // PP = P^2, R^2, ZZ1 ZZ2, ZZZ1 ZZZ2
    const Fq29 m2 = Fq29::mul(fq_select(r < 2, D, p), fq_select(r < 2, D, q));
    const Fq29 PP = quad_perm<0, 0, 0, 0>(m2);
    if (Fq29::is_zero_mod_rare(PP)) { // the same on the quad's four lanes
        if (quad_flag<1>(Fq29::is_zero_mod(Fq29::reduce_2m(D))))
            return quad_dbl(p, r);
        return quad_inf(r);
    }
    // PPP = P PP, Q = U1 PP, ZZ3 = ZZ1 ZZ2 PP on lanes 0..2
    const Fq29 m3 = Fq29::mul(fq_select(r < 2, fq_select(r == 0, D, quad_perm<0, 0, 0, 0>(m1)), m2), PP);
    const Fq29 PPP = quad_perm<0, 0, 0, 0>(m3);
    // lane 1: X3 = R^2 - PPP - 2 Q
    const Fq29 X3 = Fq29::normalize(Fq29::sub4_wide(m2, Fq29::add(PPP, Fq29::add(m3, m3))));
    // S1 PPP on lane 0, R (Q - X3) on lane 1, ZZZ3 = ZZZ1 ZZZ2 PPP on lane 3
    const Fq29 m4 = Fq29::mul(fq_select(r < 2, fq_select(r == 0, quad_perm<1, 1, 1, 1>(m1), D), m2),
        fq_select(r == 1, Fq29::sub6(m3, X3), PPP));
    // lane 1: Y3 = R (Q - X3) - S1 PPP
    const Fq29 Y3 = Fq29::reduce_2m(nsub2(m4, quad_perm<0, 0, 0, 0>(m4)));
    return fq_select(r < 2, fq_select(r == 0, quad_perm<1, 1, 1, 1>(X3), Y3), fq_select(r == 2, m3, m4));
}

} // namespace h2
