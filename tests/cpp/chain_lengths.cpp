// chain_add (softwarerenderer_amd/csrc/swr_chain.h) over lengths and magnitudes, on the host.
//   chain_lengths values   against the addition loop, bit for bit: zeros of both signs,
//                          subnormals, the edges of the lowest and highest binades, infinities
//                          and NaN at up to 2^20 additions, random floats of every exponent
//   chain_lengths cost     2^30 additions from the same starts (a loop would take hours)
// Prints the number of cases and mismatches; exits 1 on a mismatch.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "swr_chain.h"

static float from_bits(uint32_t b)
{
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}

static uint32_t to_bits(float f)
{
    uint32_t b;
    std::memcpy(&b, &f, 4);
    return b;
}

static float loop_add(float v, float a, int n)
{
    for (int k = 0; k < n; ++k)
        v = v + a;
    return v;
}

static bool same(float x, float y)
{
    return to_bits(x) == to_bits(y) || (std::isnan(x) && std::isnan(y));
}

int main(int argc, char **argv)
{
    const bool cost = argc > 1 && std::strcmp(argv[1], "cost") == 0;
    std::vector<float> special;
    for (uint32_t b : {0x00000000u, 0x00000001u, 0x00000002u, 0x00000123u, 0x007fffffu,
                       0x00800000u, 0x00800001u, 0x00ffffffu, 0x01000000u, 0x01000001u,
                       0x0d800000u, 0x3f800000u, 0x3f7fffffu, 0x42c80001u, 0x7e800000u,
                       0x7f000000u, 0x7f7fffffu, 0x7f800000u, 0x7fc00000u, 0x7fc01234u}) {
        special.push_back(from_bits(b));
        special.push_back(from_bits(b | 0x80000000u));
    }
    std::mt19937 rng(7);
    long bad = 0, done = 0;
    float sink = 0.0f;
    const auto check = [&](float v, float a, int n) {
        const float x = swr::chain_add(v, a, n);
        ++done;
        if (cost) {
            sink = x;
            return;
        }
        const float y = loop_add(v, a, n);
        if (!same(x, y)) {
            if (bad < 10)
                std::printf("mismatch v=%a a=%a n=%d: %a vs loop %a\n", v, a, n, x, y);
            ++bad;
        }
    };
    // every pair of the special values, and each of them with steps small against it
    for (float v : special)
        for (float a : special)
            for (int n : {17, 18, 100, 4097})
                check(v, a, cost ? 1 << 30 : n);
    for (float v : special)
        for (uint32_t a : {0x00000000u, 0x80000000u, 0x00000001u, 0x80000001u, 0x00000007u,
                           0x73000000u, 0xf3000000u, 0x72ffffffu, 0x74000000u})
            check(v, from_bits(a), cost ? 1 << 30 : 1 << 20);
    // random floats of every exponent; steps near the start's magnitude and below it
    for (long i = 0; i < (cost ? 100000 : 300000); ++i) {
        const uint32_t vb = rng();
        uint32_t ab = rng();
        if (i % 4) {  // a step 0 to 31 binades below the start
            const int f = (int)((vb >> 23) & 255u) - (int)(rng() % 32u);
            ab = (ab & 0x807fffffu) | (uint32_t)(f > 0 ? f : 0) << 23;
            if (i % 4 == 2)
                ab &= 0xfff00000u;  // few bits: ties
        }
        check(from_bits(vb), from_bits(ab), cost ? 1 << 30 : (int)(rng() % 3000u));
    }
    // the lowest two binades and the subnormals, both signs, steps of a few units
    for (long i = 0; i < (cost ? 20000 : 100000); ++i)
        check(from_bits((rng() % 0x01800000u) | (rng() & 0x80000000u)),
              from_bits((rng() % 0x00010000u << (rng() % 8u)) | (rng() & 0x80000000u)),
              cost ? 1 << 30 : (int)(rng() % 3000u));
    std::printf("cases %ld mismatches %ld%s\n", done, bad, sink == 12345.0f ? " " : "");
    return bad ? 1 : 0;
}
