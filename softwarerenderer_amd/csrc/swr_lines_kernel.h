// swr_lines_kernel.h — the raster stage of points and lines: one wave64 per 8x8 tile, lane =
// pixel, the tile's fragment records in draw order through the pixel program.  A template
// over the program, like the triangle kernel (swr_raster_kernel.h), so that programs compiled
// outside the library (include/swr/pixel_program.h) instantiate it too.
#pragma once

#include "swr_common.h"
#include "swr_programs.h"

namespace swr {

// fragment record words: pixel x, y (int), key, source primitive, z, w, varyings
constexpr int FR_X = 0, FR_Y = 1, FR_KEY = 2, FR_SRC = 3, FR_Z = 4, FR_W = 5, FR_VAR = 6;

// A pixel of a point or line step: PixelData as pixelDataFromVertex fills it
// (Rasterizer.h:160-173): w = v.w, invw = 1/v.w, pvar = v.pvar (no perspective divide).
template <class L>
struct VertexPixel {
    static constexpr bool SPANS = true;  // (no primitive records to replay)
    float zv, wv;
    float av[L::NA > 0 ? L::NA : 1];
    float pv[L::NP > 0 ? L::NP : 1];
    __device__ float z() const { return zv; }
    __device__ float invw() const { return 1.0f / wv; }
    __device__ float w() const { return wv; }
    __device__ float avar(int k) const { return av[k]; }
    __device__ float pvar(int k, float) const { return pv[k]; }
    __device__ float w_raw() const { return wv; }
    __device__ float p_raw(int k) const { return pv[k]; }
    __device__ static float w_of(float raw) { return raw; }
    __device__ static float pvar_of(float raw, float) { return raw; }
    static constexpr bool REPLAY = false;  // no planes: programs keep the values
    uint32_t prim = 0;
};

// One wave64 per 8x8 tile, lane = pixel: the tile's fragments, 64 at a time.  Lane k loads
// the round's fragment k into LDS and marks bit k in its pixel's word; every pixel then takes
// its own fragments, lowest bit first (draw order), so the pixels of a tile shade side by side
// and a round takes as many steps as its busiest pixel has fragments.  Bound by those steps
// where many lines meet in a pixel: a 48k-edge wireframe sphere at 1280x720 (its poles) takes
// 40 us; 64 us with each step's record read from memory, 214 us with the fragments
// taken one by one, a lane at a time.
template <template <class> class ProgT, int NZ, int NW, int NA, int NP>
__global__ void __launch_bounds__(256) k_lines_raster(RasterArgs a)
{
    using L = Layout<NZ, NW, NA, NP>;
    using Prog = ProgT<L>;
    __shared__ unsigned long long s_mask[4][64];  // per wave: a pixel's fragments of the round
    constexpr int RW = FR_VAR + L::NA + L::NP, RS = RW | 1;  // odd: records spread over banks
    __shared__ float s_rec[4][64 * RS];           // the round's fragment records
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int tile = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6)) + wv);
    if (tile >= a.tiles)
        return;
    if (a.status[ST_OVERFLOW] | a.status[ST_ERROR])
        return;
    const uint32_t beg = a.ranges[2 * tile], end = a.ranges[2 * tile + 1];
    if (beg >= end)
        return;
    const int bx = (tile % a.tiles_x) * TILE, by = (tile / a.tiles_x) * TILE;
    const int px = bx + (lane & 7), py = by + (lane >> 3);
    const bool inside = px < a.width && py < a.height;
    const size_t o = (size_t)py * (size_t)a.pitch + (size_t)px;
    const int kw = Prog::KEY_WORD == REC_SRC ? FR_SRC : FR_KEY;

    typename Prog::State st;
    if (inside)
        Prog::load(st, a, o);
    for (uint32_t c = beg; c < end; c += 64) {
        s_mask[wv][lane] = 0ull;
        lds_sync();
        if (c + (uint32_t)lane < end) {
            const float *r = a.prims + (size_t)a.vals[c + lane] * (size_t)a.stride;
            float w[RW];
#pragma unroll
            for (int k = 0; k < RW; ++k)
                w[k] = r[k];
            const int fx = (int)__float_as_uint(w[FR_X]), fy = (int)__float_as_uint(w[FR_Y]);
#pragma unroll
            for (int k = 2; k < RW; ++k)
                s_rec[wv][lane * RS + k] = w[k];
            // fragments lie on the target and in this tile: a pixel index below 64
            atomicOr(&s_mask[wv][((fy - by) * TILE + (fx - bx)) & 63], 1ull << lane);
        }
        lds_sync();
        unsigned long long m = s_mask[wv][lane];
        while (m) {
            const int j = __builtin_ctzll(m);
            m &= m - 1ull;
            const float *r = s_rec[wv] + j * RS;
            VertexPixel<L> p;
            p.zv = r[FR_Z];
            p.wv = r[FR_W];
#pragma unroll
            for (int k = 0; k < L::NA; ++k)
                p.av[k] = r[FR_VAR + k];
#pragma unroll
            for (int k = 0; k < L::NP; ++k)
                p.pv[k] = r[FR_VAR + L::NA + k];
            Prog::shade(st, a, p, __float_as_uint(r[kw]), px, py);
        }
        lds_sync();  // the next round clears the words
    }
    if (inside)
        Prog::template store<VertexPixel<L>>(st, a, o, px, py);
}

template <template <class> class ProgT, int NZ, int NW, int NA, int NP>
inline hipError_t launch_lr(const RasterArgs &a, hipStream_t s)
{
    const uint32_t blocks = ((uint32_t)a.tiles + 3) / 4;
    hipLaunchKernelGGL((k_lines_raster<ProgT, NZ, NW, NA, NP>), dim3(blocks > 0 ? blocks : 1),
                       dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace swr
