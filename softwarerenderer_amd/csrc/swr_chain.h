// swr_chain.h — the result of a chain of fp32 additions of one constant, without running it.
//
// The reference steps every interpolant along a span by repeated addition
// (PixelData::stepX, PixelData.h:104-118; PixelShaderBase::drawSpan, PixelShaderBase.h:96-112):
// the value at pixel x of a span starting at xl is init followed by (x - xl) additions of the
// plane's a, each rounded to fp32.  Replaying that chain costs one addition per pixel of the
// span before x.  chain_add gives the same bits in a number of steps that grows with the
// number of binades the chain crosses (logarithmic in its length), not with its length.
//
// Why a run of additions inside one binade is one multiplication.  Let v lie in the binade
// [2^e, 2^(e+1)) (or its negative), so v = m*u with u = 2^(e-23) and m an integer, and let
// a = q*u (q real, exact in double).  While the exact sum v + a stays in the binade, fp32
// spacing there is u, so round-to-nearest-even gives fl(v + a) = RNE(m + q)*u.  If q is not
// a half-integer, RNE(m + q) = m + RNE(q) for every m: each addition adds d = RNE(q)*u, and
// k additions add k*d exactly.  If q is a half-integer (a tie), RNE(m + q) = m + RNE(q) when
// m is even, and the result is then even again: after one addition inside the binade (which
// leaves m even whatever it was), every later one adds d.  The closed form is used only while
// every intermediate result stays at least u inside the binade (so each exact sum is within
// u/2 of it and cannot round across an edge); each edge crossing is one explicit addition.
// Zero, the subnormals and the lowest normal binade share the spacing 2^-149, so they are one
// binade here, [0, 2^-125).  An infinity or NaN takes explicit additions until one changes
// nothing: every later one gives the same then.  So no start and no step makes the cost grow
// with the length.  A line is walked in pieces that each start with a chain of their own: one
// addition per step wherever |v| < 2^-100 made a constant zero cost the square of the line's
// length (20,000 screen-long lines, zero z and one colour: 8290 us, now 1043; with random
// values 1112 and 1050), and a Span primitive's zero planes one addition per pixel (200k
// triangles at 1280x720, Span, hash program: 4727 us, now 752).
#pragma once

#include <stdint.h>

namespace swr {

// 1 / x approximately (the hardware reciprocal on the GPU, a rounded division on the host);
// chain_add corrects what the estimate gets wrong.
__host__ __device__ inline double approx_rcp(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return 1.0 / x;
#endif
}

// The exponent field of a finite float's magnitude bits, 1 for the subnormals: the binade of
// spacing 2^(field - 150).  Field 1 stands for all of [0, 2^-125).
__host__ __device__ inline int chain_field(uint32_t magnitude)
{
    const int field = (int)(magnitude >> 23);
    return field > 0 ? field : 1;
}

// fp32 value after n sequential additions of a: `for (k = 0; k < n; ++k) v = v + a;`
// (round to nearest even, subnormals kept, no contraction).
__host__ __device__ inline float chain_add(float v, float a, int n)
{
    if (n <= 16) {  // short chains: the additions themselves are cheaper
        for (int k = 0; k < n; ++k)
            v = v + a;
        return v;
    }
    int binade = 0;     // the binade the evenness below refers to (0: none)
    bool even = false;  // m is known to be even (a tie's additions are regular)
    while (n > 0) {
        const uint32_t vb = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
        const uint32_t ab = __builtin_bit_cast(uint32_t, a) & 0x7fffffffu;
        if (n <= 2 || vb >= 0x7f800000u || ab >= 0x7f800000u) {
            const float nv = v + a;
            if (__builtin_bit_cast(uint32_t, nv) == __builtin_bit_cast(uint32_t, v))
                return v;
            v = nv;
            --n;
            continue;
        }
        // in units of u from here on: |v| = m, the change of |v| per addition q
        const int f = chain_field(vb);
        if (f != binade) {
            binade = f;
            even = false;
        }
        const int lo = f > 1 ? 0x800000 : 0;  // the binade's lower edge; the upper is 2^24
        const int m = (int)(vb & 0x7fffffu) + ((vb >> 23) != 0 ? 0x800000 : 0);
        const bool neg = v < 0.0f;
        const double qa = __builtin_ldexp((double)a, 150 - f);  // exact: a power-of-two scaling
        const double q = neg ? -qa : qa;
        const double r = __builtin_rint(q);  // to even where q is a tie
        const double off = q - r;
        const bool tie = off == 0.5 || off == -0.5;
        if (tie && !even) {  // one addition inside the binade makes m even
            v = v + a;
            --n;
            const uint32_t nb = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
            even = nb < 0x7f800000u && chain_field(nb) == f;
            continue;
        }
        if (r == 0.0) {
            // |a| <= u/2: every addition rounds back to v (or, for v = -0 and a = +0, to the
            // +0 of the first), unless v sits on the binade's lower edge and a points to
            // zero and is not too small for the spacing below it, u/2
            const float nv = v + a;
            if (!(q < 0.0 && m == lo) || nv == v)
                return nv;
            v = nv;
            --n;
            continue;
        }
        // the largest k with every m + j*r (1 <= j <= k) inside [lo + 1, 2^24 - 1]
        const double room = (double)(r > 0.0 ? 0xffffff - m : m - lo - 1);
        const double step = r > 0.0 ? r : -r;
        // floor(room / step) is below 2^24: estimated from a reciprocal, then made exact by
        // the two loops
        double k = room < 0.0 ? 0.0 : __builtin_floor(room * approx_rcp(step));
        while (k > 0.0 && k * step > room)
            k -= 1.0;
        while ((k + 1.0) * step <= room)
            k += 1.0;
        if (k > (double)n)
            k = (double)n;
        const float nm = __builtin_ldexpf((float)((double)m + k * r), f - 150);  // exact
        v = neg ? -nm : nm;
        n -= (int)k;
        if (n > 0) {  // the addition that reaches or crosses the binade's edge
            v = v + a;
            --n;
        }
    }
    return v;
}

}  // namespace swr
