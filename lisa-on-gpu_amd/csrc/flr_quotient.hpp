// flr_quotient.hpp -- the exact stencils' quotients in two operations each.
//
// Written for host and device: the host build (the bit-for-bit test against a / b) defines
// FLR_HOST_DEVICE empty and FLR_RCP_SEED as an approximate reciprocal.
#pragma once

#ifndef FLR_HOST_DEVICE
#define FLR_HOST_DEVICE __host__ __device__
#endif
#ifndef FLR_RCP_SEED
#define FLR_RCP_SEED(x) __builtin_amdgcn_rcp(x)
#endif

namespace flr {

// The smallest sample position from which div_recip is proven for half point count h.
constexpr int exact2_min_position(int h) { return h <= 16 ? 256 : 512; }

// The reciprocal of b as an unevaluated sum: 1/b = y + l up to ~2^-103 of itself.
struct Recip {
    double y, l;
};

// a / b, correctly rounded, as y a + l a rounded once, from b's two-part reciprocal. Why the bits
// are those of a / b for the stencils' denominators, b = j + e or j + 1 - e, at most h (u = 2^-53): at a
// position cf >= 2^c (in samples) the fraction e is a multiple of ulp(cf) >= 2^(c-52); so are j + e and
// j + (1 - e), which are exact, and b = B 2^(c-52) with B <= h 2^(52-c). The quotient of such a b and a
// 53-bit a is never a midpoint M of two doubles (M < 2^54 odd), and is at least 1 / (B M) >
// 2^(c-106) / h of itself away from each. recip_pair's y is off by at most e1 = 3 u (the roundings of
// F G, of its reciprocal and of the product by the other factor), 1 - b y = e1 comes out exactly, and
// l = e1 y leaves e1^2 = 9 u^2 and its own rounding, 3 u^2; the product l a adds 3 u^2. Together
// 15 u^2 = 15 2^-106, below that distance when h <= 2^c / 15: c = 8 for h <= 16, 9 up to
// kMaxHalf (exact2_min_position). That is for a of 2^-967 or more, whose l a is a normal number; smaller
// ones are off by units of the smallest double, and an infinite a gives an infinity or NaN where
// div_rcp gives NaN. Two operations per quotient instead of div_rcp's three, and one
// v_rcp_f64 (4 issue slots) per tap pair instead of two: 58 issue slots instead of 72 per tap pair of
// six units with one fraction, 30 instead of 36 of a complex stencil, 23 instead of 27 of one unit.
// The exact forms are bound by these FP64 operations: 1-yr FP64 drop-in (3,153,600 samples) 1.125 ->
// 0.961 ms with equal arms, 2.002 -> 1.769 ms with unequal ones, order 31 with a custom table
// (262,145 samples) 0.135 -> 0.119 ms (interleaved A/B).
FLR_HOST_DEVICE inline double div_recip(double a, const Recip &r)
{
    return __builtin_fma(a, r.y, a * r.l);
}

// The same quotient from y alone: with y off by at most e1, q = y a by at most e1 + u, the residual
// a - b q comes out exactly (a multiple of ulp(b) ulp(q) below 8 b of them) and the last operation rounds
// a / b off by e1 (e1 + u): 12 u^2 with recip_pair's e1 = 3 u, 30 u^2 with recip_quad's 5 u, less than
// div_recip's from the same y.
FLR_HOST_DEVICE inline double div_recip_y(double a, double b, const Recip &r)
{
    const double q = a * r.y;
    return __builtin_fma(__builtin_fma(-b, q, a), r.y, q);
}

// The two denominators of a tap pair, F = j + e and G = j + (1 - e): one hardware reciprocal of
// their product (relative error below 2^-22), refined to third order, gives both.
FLR_HOST_DEVICE inline void recip_pair(double F, double G, Recip &rF, Recip &rG)
{
    const double p = F * G;
    double r = FLR_RCP_SEED(p);
    const double e = __builtin_fma(-p, r, 1.0);
    r = __builtin_fma(r, __builtin_fma(e, e, e), r);
    rF.y = G * r;
    rG.y = F * r;
    rF.l = __builtin_fma(-F, rF.y, 1.0) * rF.y;
    rG.l = __builtin_fma(-G, rG.y, 1.0) * rG.y;
}

// Two tap pairs at once: one hardware reciprocal of p1 p2 for all four denominators (14 issue slots
// per pair, with the two sums j + e and j + (1 - e), instead of 16). Their y is off by up to e1 = 5 u
// (p1, p1 p2, its reciprocal, the product by p2, the product by the other factor; p2's rounding cancels),
// so a quotient by div_recip is a / b up to 25 u^2 + 5 u^2 + 5 u^2 = 35 u^2, by div_recip_y up to 30 u^2: below
// the least distance from a midpoint, 2^c u^2 / h, from position 2^9 on for h <= 14 and h <= 17, from 2^10
// on for h <= 29 and h <= 34 (exact4_min_position; kernels for any order use div_recip_y). With the six undelayed
// units of unequal arms sharing theirs, 13,744 instead of 15,791 issue slots per sample of unequal-arm
// TDI: 1,048,577 samples, 2nd generation, 453 -> 410 us (equal arms 225 -> 221).
constexpr int exact4_min_position(int h) { return h <= 17 ? 512 : 1024; }

FLR_HOST_DEVICE inline void recip_quad(double F1, double G1, double F2, double G2, Recip &rF1,
                                       Recip &rG1, Recip &rF2, Recip &rG2)
{
    const double p1 = F1 * G1, p2 = F2 * G2, p = p1 * p2;
    double r = FLR_RCP_SEED(p);
    const double e = __builtin_fma(-p, r, 1.0);
    r = __builtin_fma(r, __builtin_fma(e, e, e), r);
    const double r1 = r * p2, r2 = r * p1;
    rF1.y = G1 * r1;
    rG1.y = F1 * r1;
    rF2.y = G2 * r2;
    rG2.y = F2 * r2;
    rF1.l = __builtin_fma(-F1, rF1.y, 1.0) * rF1.y;
    rG1.l = __builtin_fma(-G1, rG1.y, 1.0) * rG1.y;
    rF2.l = __builtin_fma(-F2, rF2.y, 1.0) * rF2.y;
    rG2.l = __builtin_fma(-G2, rG2.y, 1.0) * rG2.y;
}

}  // namespace flr
