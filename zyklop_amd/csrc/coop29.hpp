// XYZZ additions of the 29-bit form (field29.hpp) by a group of lanes: the
// bucket reduction's point operations, where the length of a dependent chain
// and not the number of additions sets the time.
//
// A thread that adds two points alone runs 14 field products one after the
// other (28 or more for G2), about 6.3 us (G2 16 us) for a lone wave. Four of
// those products are independent at every step of the formula, so a group of
// four lanes, each holding one coordinate (X, Y, ZZ, ZZZ) of both points,
// does the addition in four products: every lane multiplies its coordinates,
// and the values the next step needs move inside the group by DPP (quad_perm),
// which costs a VALU move and no LDS round trip. G2 takes two quads, one per
// Fp2 component; each component of a product is one sum of two Fp products
// with one reduction (f29_mulsum<2>), the other component's operands coming
// across by DPP. The work per addition is about 1.6 times that of one thread,
// the latency a third (G1) to a fifth (G2).
//
// All lanes of a group must be active and in step. Lane roles: bits 0..1 of
// the lane give the coordinate, bit 2 (G2) the component.
#pragma once
#include "field29.hpp"

namespace zk {

template <int A, int B, int C, int D>
ZK_DEV F29 f29_quad(const F29& a) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++)
        r.l[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a.l[i], A | B << 2 | C << 4 | D << 6, 0xf, 0xf, true);
    return r;
}
template <int A, int B, int C, int D>
ZK_DEV uint32_t u32_quad(uint32_t a) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a, A | B << 2 | C << 4 | D << 6, 0xf, 0xf, true);
}
// value of lane ^ 4: half-row mirror (lane ^ 7), then the quad reversed
ZK_DEV uint32_t u32_xor4(uint32_t a) {
    return u32_quad<3, 2, 1, 0>((uint32_t)__builtin_amdgcn_update_dpp(0, (int)a, 0x141, 0xf, 0xf, true));
}
ZK_DEV F29 f29_xor4(const F29& a) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = u32_xor4(a.l[i]);
    return r;
}
// m ? x : y for lane masks m of all ones or zeros
ZK_DEV F29 f29_sel(uint32_t m, const F29& x, const F29& y) {
    F29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = (x.l[i] & m) | (y.l[i] & ~m);
    return r;
}
ZK_DEV uint32_t f29_or(const F29& a) {
    uint32_t d = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) d |= a.l[i];
    return d;
}

// What differs between the curves. mul: the lane's component of x*y, x and y
// normalized, y < 8p; the result is below p + (x*y + 8x*p)/169p (G1: without
// the 8x*p). all: whether a lane flag holds in every component.
template <class T> struct Coop;
template <>
struct Coop<Fp> {
    static constexpr int LANES = 4;
    uint32_t m1, m2, ml1;   // masks: coordinate odd (Y, ZZZ), coordinate >= 2 (ZZ, ZZZ), coordinate Y
    ZK_DEV explicit Coop(uint32_t lane)
        : m1(0u - (lane & 1u)), m2(0u - (lane >> 1 & 1u)), ml1(m1 & ~m2) {}
    ZK_DEV F29 mul(const F29& x, const F29& y) const { return f29_mul(x, y); }
    ZK_DEV uint32_t any(uint32_t f) const { return f; }
    ZK_DEV uint32_t all(uint32_t f) const { return f; }
};
template <>
struct Coop<Fq2> {
    static constexpr int LANES = 8;
    uint32_t m1, m2, ml1, mc;   // mc: component c1
    ZK_DEV explicit Coop(uint32_t lane)
        : m1(0u - (lane & 1u)), m2(0u - (lane >> 1 & 1u)), ml1(m1 & ~m2), mc(0u - (lane >> 2 & 1u)) {}
    // c0: x0*y0 + x1*(8p - y1), c1: x1*y0 + x0*y1; the columns stay below
    // (9 + 36 + 9) * 2^58 plus the carry
    ZK_DEV F29 mul(const F29& x, const F29& y) const {
        const F29 yp = f29_xor4(y);
        F29 neg;
#pragma unroll
        for (int i = 0; i < 9; i++) neg.l[i] = f29c::P8[i] - yp.l[i];
        const F29 a[2] = {x, f29_xor4(x)}, b[2] = {f29_sel(mc, yp, y), f29_sel(mc, y, neg)};
        return f29_mulsum<2>(a, b);
    }
    ZK_DEV uint32_t any(uint32_t f) const { return f | u32_xor4(f); }
    ZK_DEV uint32_t all(uint32_t f) const { return f & u32_xor4(f); }
};

// Bounds kept by both operations, in units of p (mul's bound, worst cases of
// G2): X < 7.4, Y < 2.8, ZZ and ZZZ < 2, limbs normalized; points of the
// accumulation (all below 2) are inside.

// dbl-2008-s-1: U = 2Y, V = U^2, XX = X^2 | W = U*V, S = X*V, ZZ3 = V*ZZ,
// MM = (3XX)^2 | X3 = MM - 2S, Y3 = M*(S - X3) - W*Y, ZZZ3 = W*ZZZ.
// U < 5.6, V < 1.5, M < 5; S < 1.5, W < 1.4, MM < 1.4; X3 in (3, 7.4); Y3 < 2.7.
template <class T>
ZK_DEV F29 coop_dbl(const Coop<T>& k, const F29& a) {
    using namespace f29c;
    const F29 u = f29_sel(k.m1, f29_norm(f29_add(a, a)), a);   // X, U, -, -
    const F29 r1 = k.mul(u, u);                                // XX, V, -, -
    const F29 xx = f29_quad<0, 0, 0, 0>(r1);
    const F29 M = f29_norm(f29_add(f29_add(xx, xx), xx));
    const uint32_t m3 = k.m1 & k.m2;
    F29 x2 = f29_sel(k.m2, a, u);                              // X, U, ZZ, M
    x2 = f29_sel(m3, M, x2);
    const F29 r2 = k.mul(x2, f29_sel(m3, M, f29_quad<1, 1, 1, 1>(r1)));   // S, W, ZZ3, MM
    const F29 S = f29_quad<0, 0, 0, 0>(r2), W = f29_quad<1, 1, 1, 1>(r2), MM = f29_quad<3, 3, 3, 3>(r2);
    F29 X3, x3, y3;
#pragma unroll
    for (int i = 0; i < 9; i++) X3.l[i] = P6[i] - 2 * S.l[i] + MM.l[i];
    X3 = f29_norm(X3);
    F29 t, nw;
#pragma unroll
    for (int i = 0; i < 9; i++) {
        t.l[i] = S.l[i] + P8[i] - X3.l[i];
        nw.l[i] = P2[i] - W.l[i];
    }
    x3 = f29_norm(f29_sel(k.m1, nw, t));                       // T, -W, -, ZZZ
    x3 = f29_sel(k.m2, a, x3);
    y3 = f29_sel(k.m2, W, f29_sel(k.m1, a, M));                // M, Y, -, W
    const F29 r3 = k.mul(x3, y3);
    const F29 Y3 = f29_norm(f29_add(r3, f29_quad<0, 0, 0, 0>(r3)));
    return f29_sel(k.m2, f29_sel(k.m1, r3, r2), f29_sel(k.m1, Y3, X3));
}

// add-2008-s, a + b, either of which may be infinity (ZZ = 0); equal points
// go through the doubling, opposite points give infinity (all zero).
// U, S < 1.45; P, R = second - first + 2p in (0.5, 3.5); PP, RR < 1.3;
// PPP < 1.2, Q < 1.1; X3 = RR - PPP - 2Q + 6p in (2.6, 7.3); T = Q - X3 + 8p
// in (0.7, 6.5); Y3 = T*R + (2p - S1)*PPP < 2.6; ZZ3, ZZZ3 < 1.1.
template <class T>
ZK_DEV F29 coop_add(const Coop<T>& k, const F29& a, const F29& b) {
    using namespace f29c;
    const uint32_t afin = u32_quad<2, 2, 2, 2>(k.any(f29_or(a))), bfin = u32_quad<2, 2, 2, 2>(k.any(f29_or(b)));
    const F29 r1 = k.mul(a, f29_quad<2, 3, 0, 1>(b));          // U1, S1, U2, S2
    const F29 r1x = f29_quad<2, 3, 0, 1>(r1);
    F29 d;
#pragma unroll
    for (int i = 0; i < 9; i++) d.l[i] = r1x.l[i] + P2[i] - r1.l[i];
    const F29 D = f29_norm(d);                                 // P, R, -P, -R
    const F29 r2 = k.mul(f29_sel(k.m2, a, D), f29_sel(k.m2, b, D));   // PP, RR, ZZ1*ZZ2, ZZZ1*ZZZ2
    const uint32_t zero = k.all(f29_zero_mod(r2) ? 1u : 0u);
    const F29 PP = f29_quad<0, 0, 0, 0>(r2);
    const F29 r3 = k.mul(f29_sel(k.m2, r2, f29_sel(k.m1, f29_quad<0, 0, 0, 0>(r1), D)), PP);   // PPP, Q, ZZ3, -
    const F29 PPP = f29_quad<0, 0, 0, 0>(r3), Q = f29_quad<1, 1, 1, 1>(r3), RR = f29_quad<1, 1, 1, 1>(r2);
    F29 X3;
#pragma unroll
    for (int i = 0; i < 9; i++) X3.l[i] = (P6[i] - PPP.l[i] - 2 * Q.l[i]) + RR.l[i];
    X3 = f29_norm(X3);
    const F29 S1 = f29_quad<1, 1, 1, 1>(r1);
    F29 t, ns;
#pragma unroll
    for (int i = 0; i < 9; i++) {
        t.l[i] = Q.l[i] + P8[i] - X3.l[i];
        ns.l[i] = P2[i] - S1.l[i];
    }
    const F29 x4 = f29_norm(f29_sel(k.m1, t, ns));             // -S1, T, ZZ.., ZZZ1*ZZZ2
    const F29 r4 = k.mul(f29_sel(k.m2, r2, x4), f29_sel(k.ml1, D, PPP));   // -S1*PPP, T*R, -, ZZZ3
    const F29 Y3 = f29_norm(f29_add(r4, f29_quad<0, 0, 0, 0>(r4)));
    F29 r = f29_sel(k.m2, f29_sel(k.m1, r4, r3), f29_sel(k.m1, Y3, X3));
    r = f29_sel(afin ? 0u : ~0u, b, r);
    r = f29_sel(bfin ? 0u : ~0u, a, r);
    const uint32_t eqx = u32_quad<0, 0, 0, 0>(zero), eqy = u32_quad<1, 1, 1, 1>(zero);
    if (eqx && afin && bfin) {
        if (eqy) r = coop_dbl<T>(k, a);
        else r = F29{};
    }
    return r;
}

}  // namespace zk
