// The binning sort's buckets (softwarerenderer_amd/csrc/swr_buckets.h) on the host: the mapping
// is a bijection that bucket_tile inverts, and no bucket holds many times its share of a column,
// strip, diagonal or block of tiles.  Prints the worst excess; exits 1 above the limit given.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "swr_buckets.h"

int main(int argc, char **argv)
{
    const double limit = argc > 1 ? std::atof(argv[1]) : 0.0;
    const swr::TileDigit digit = {0, true};
    for (uint32_t tile = 0; tile < (1u << 18); ++tile) {
        const uint32_t b = digit.of(tile);
        if (b > 255u || swr::bucket_tile(b, tile >> 8) != tile) {
            std::printf("tile %u: bucket %u does not lead back\n", tile, b);
            return 1;
        }
    }
    double worst = 0.0;
    long shapes = 0;
    for (int w = 16; w <= 1024; ++w) {
        const int h = (1 << 18) / w < 512 ? (1 << 18) / w : 512;
        // tiles (x(y) .. x(y) + n - 1, y) for y in [y0, y1): x = x0 + slope * y
        const auto shape = [&](int x0, int slope, int n, int y0, int y1) {
            std::vector<int> count(256, 0);
            int total = 0, most = 0;
            for (int y = y0; y < y1 && y < h; ++y)
                for (int x = x0 + slope * y; x < x0 + slope * y + n; ++x)
                    if (x >= 0 && x < w) {
                        ++total;
                        const int c = ++count[digit.of((uint32_t)(y * w + x))];
                        most = c > most ? c : most;
                    }
            if (total < 64)
                return;
            const double excess = (double)most / (double)((total + 255) / 256);
            worst = excess > worst ? excess : worst;
            ++shapes;
        };
        for (int x0 : {0, w / 3, w / 2, w - 1})
            for (int slope : {0, 1, -1, 2, -2})
                shape(x0, slope, 1, 0, h);
        for (int n : {2, 4, 8, 16})
            shape(w / 3, 0, n, 0, h);
        for (int n : {16, 32, 64})
            shape(w / 3, 0, n, 10, 10 + n);
    }
    std::printf("shapes %ld worst excess %.2f\n", shapes, worst);
    return worst <= limit ? 0 : 1;
}
