// swr_common.h — definitions shared by the gfx950 kernels and the host orchestration.
//
// Float arithmetic in every kernel follows the reference's evaluation order operation by
// operation (one rounding each, no contraction: the library is built with
// -ffp-contract=off and the pragma below), so the device reproduces the reference's bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <limits.h>

#include "../../include/swr_hip.h"

#pragma clang fp contract(off)

namespace swr {

// ---- primitive record: one per primitive that reaches the rasterizer, in draw order ----
// words (u32 / f32):
//   0 key   1 flags   2..5 tile rect tx0 ty0 tx1 ty1 (inclusive)
//   8..16  edge equations e0.abc e1.abc e2.abc (EdgeEquation.h:37-43)
//   17..22 bottom-flat part: ox oy is1 is2 row_lo row_hi   (rows lo <= y < hi)
//   23..28 top-flat part:    ox oy is1 is2 row_lo row_hi   (rows lo < y <= hi)
//   17..20 Block primitives instead: the 8x8 blocks of the reference's block grid,
//          bx0 by0 bx1 by1 (inclusive, in blocks; clamped to the target)
//   32..   parameter planes a,b,c: [z][invw][avar 0..na)[pvar 0..np)
constexpr int REC_KEY = 0;
constexpr int REC_FLAGS = 1;
constexpr int REC_TILES = 2;
constexpr int REC_EDGE = 8;
constexpr int REC_BOT = 17;
constexpr int REC_BLOCKS = 17;
constexpr int REC_TOP = 23;
constexpr int REC_PARAM = 32;

constexpr uint32_t FLAG_BLOCK = 1u;
constexpr uint32_t FLAG_TIE0 = 2u;
constexpr uint32_t FLAG_TIE1 = 4u;
constexpr uint32_t FLAG_TIE2 = 8u;
constexpr uint32_t FLAG_BOTTOM = 16u;
constexpr uint32_t FLAG_TOP = 32u;

constexpr int TILE = SWR_BLOCK_SIZE;   // one 8x8 tile = one reference block = one wave64
constexpr int BATCH = SWR_BATCH_PRIMITIVES;
constexpr int MAX_CLIP = SWR_MAX_CLIP_VERTS;

// status word indices (device u64 array, copied to the host after a draw)
constexpr int ST_PRIMS = 0;        // primitives emitted
constexpr int ST_PAIRS = 1;        // (primitive, tile) pairs emitted
constexpr int ST_OVERFLOW = 2;     // bit 0: prim arena, bit 1: pair arena
constexpr int ST_ERROR = 3;        // bit 0: index range, bit 1: clip overflow
constexpr int ST_BIG = 4;          // primitives queued for cooperative pair expansion
constexpr int ST_KEPT = 5;         // pairs left after dropping rejected blocks / tiles
constexpr int ST_CLIPQ = 6;        // triangles queued for the clipper
constexpr int ST_LIVE = 8;         // triangles the emit pass walks (the live list)
constexpr int ST_STICKY = 7;       // failures of asynchronous draws not yet reported: bit 0
                                   // overflow, bits 1.. the ST_ERROR bits; never cleared by
                                   // a draw, only by the host once it has reported them
constexpr int ST_WORDS = 16;       // a draw clears every word but ST_STICKY

// Counters a triangle draw's begin kernel clears, in one small buffer: the clip queue's 64
// regions (16 words apart), then the persistent raster's RASTER_QUEUES bin queues (32 words,
// 128 bytes, apart: one cache line each), RASTER_QUEUES / 8 per XCD.
constexpr uint32_t CLIPQ_COUNTERS = 64 * 16;
constexpr uint32_t RASTER_QUEUES = 64;
constexpr uint32_t RASTER_QUEUE_STRIDE = 32;
constexpr uint32_t DRAW_COUNTER_WORDS = CLIPQ_COUNTERS + RASTER_QUEUES * RASTER_QUEUE_STRIDE;

// record word 6: index of the primitive's first (tile, primitive) pair
constexpr int REC_PAIRBASE = 6;
// record word 7: the input triangle the primitive comes from (scene-local index)
constexpr int REC_SRC = 7;
// record word 29: the scene of a batched draw (0 otherwise)
constexpr int REC_SCENE = 29;

// Which plane equations the rasterizer interpolates (chosen by the pixel program).
struct ParamLayout {
    int nz;        // 1: z plane
    int nw;        // 1: invw plane (InterpolateW or PVarCount > 0)
    int na, np;    // avar / pvar planes stored (program class)
    int set_na, set_np;  // planes actually set up (declared counts, <= na / np)
    int count;     // nz + nw + na + np
    int stride;    // record stride in words
};

// ---- float -> int as x86-64 cvttss2si (out of range or NaN -> INT_MIN) ----------------
__host__ __device__ inline int f2i(float f)
{
    return (f > -2147483904.0f && f < 2147483648.0f) ? (int)f : INT_MIN;
}

// std::min / std::max argument order (matters for NaN)
__host__ __device__ inline float ref_min(float a, float b) { return (b < a) ? b : a; }
__host__ __device__ inline float ref_max(float a, float b) { return (a < b) ? b : a; }
__host__ __device__ inline int imin(int a, int b) { return (b < a) ? b : a; }
__host__ __device__ inline int imax(int a, int b) { return (a < b) ? b : a; }

// Orders one wave's LDS traffic: LDS operations of a wave complete in issue order, so
// keeping the compiler from moving them across this point and waiting for the wave's own
// LDS traffic makes its earlier LDS writes visible to its later reads (a barrier for data
// that only the calling wave shares).
__device__ inline void lds_sync()
{
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    __asm__ volatile("" ::: "memory");
}

// Wave-wide inclusive scan of 64 lanes: DPP steps inside the rows of 16 lanes, then the rows'
// totals handed on (a shuffle per step waits for the LDS six times over).  Every lane calls it.
__device__ inline uint32_t wave_incl(uint32_t v)
{
#define SWR_SCAN_STEP(CTRL, ROWS) \
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false)
    SWR_SCAN_STEP(0x111, 0xF);  // row_shr 1, 2, 4, 8
    SWR_SCAN_STEP(0x112, 0xF);
    SWR_SCAN_STEP(0x114, 0xF);
    SWR_SCAN_STEP(0x118, 0xF);
    SWR_SCAN_STEP(0x142, 0xA);  // row_bcast 15, 31
    SWR_SCAN_STEP(0x143, 0xC);
#undef SWR_SCAN_STEP
    return v;
}

// EdgeEquation::test (EdgeEquation.h:53-61): v > 0 || (v == 0 && tie), as one compare:
// v >= 0 with the tie, v >= the smallest denormal without it (the kernels keep fp32
// denormals, so nothing lies strictly between 0 and it; NaN fails both forms).
__device__ inline bool edge_pass(float v, bool tie)
{
    return v >= (tie ? 0.0f : __uint_as_float(1u));
}

// Block classification from the four corners, Rasterizer.h:270-304: 0 skip,
// 1 drawBlock<true> (per-pixel edge tests), 2 drawBlock<false> (all 64 pixels).
// e[9] = e0.abc e1.abc e2.abc; corners use v + a*7 / v + b*7 (EdgeData::stepX/Y(eqn, s)).
__device__ inline int classify_block(const float *e, uint32_t flags, int x, int y)
{
    const float xf = (float)x + 0.5f, yf = (float)y + 0.5f, s = 7.0f;
    bool p[4][3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float a = e[3 * k], b = e[3 * k + 1], c = e[3 * k + 2];
        const bool tie = (flags >> (1 + k)) & 1u;
        float v00 = a * xf + b * yf + c;
        float v01 = v00 + b * s;
        float v10 = v00 + a * s;
        float v11 = v01 + a * s;
        p[0][k] = edge_pass(v00, tie);
        p[1][k] = edge_pass(v01, tie);
        p[2][k] = edge_pass(v10, tie);
        p[3][k] = edge_pass(v11, tie);
    }
    int result = 0;
    bool same = true;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        result += (p[q][0] && p[q][1] && p[q][2]) ? 1 : 0;
        // `a == b == c` parses as (a == b) == c: true iff an odd number of edges pass
        same = same && ((p[q][0] == p[q][1]) == p[q][2]);
    }
    if (result == 0)
        return same ? 0 : 1;
    return result == 4 ? 2 : 1;
}

// True unless some edge is negative at every pixel centre of the block by more than the
// rounding the per-pixel chain can accumulate, i.e. unless no pixel of drawBlock<true>
// (PixelShaderBase.h:55-94) can pass all three edge tests.  The chained value of pixel
// (i, j) is init = (a*xf + b*yf) + c followed by j additions of b and i of a: at most 18
// roundings, each at most 2^-24 of a partial sum bounded by M = |a xf| + |b yf| + |c| +
// 7|a| + 7|b|, so below 2^-19.8 M in all.  The edge's maximum over the block (a corner: the
// function is linear) is evaluated in fp32, with at most 9 roundings of terms bounded by M
// (below 2^-20.8 M), and the block is dropped only when that evaluation is below -2^-18 M:
// the exact maximum is then below -2^-18 M + 2^-20.8 M, more negative than any chain's
// rounding can lift.  A coefficient or bound that is not finite keeps the block.  ext = 7 is
// one 8x8 block; a larger ext tests a square of (ext + 1)^2 pixels (a bin of blocks: the
// bound then covers every block's chain, which starts inside the square).
__device__ inline bool block_may_cover(const float *e, int x, int y, int ext = 7)
{
    const float xf = (float)x + 0.5f, yf = (float)y + 0.5f, s = (float)ext;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float a = e[3 * k], b = e[3 * k + 1], c = e[3 * k + 2];
        const float m = fabsf(a * xf) + fabsf(b * yf) + fabsf(c) + s * (fabsf(a) + fabsf(b));
        const float mx = a * xf + b * yf + c + fmaxf(0.0f, s * a) + fmaxf(0.0f, s * b);
        if (mx < -m * 3.814697265625e-06f)  // 2^-18; false for NaN and infinite bounds
            return false;
    }
    return true;
}

// classify_block's class from which corners pass which edges, in lane masks alone.
__device__ inline int corners_class(const bool (&p)[4][3])
{
    bool any = false, all = true, same = true;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool in = p[q][0] & p[q][1] & p[q][2];
        any = any | in;
        all = all & in;
        same = same & ((p[q][0] == p[q][1]) == p[q][2]);
    }
    return any ? (all ? 2 : 1) : (same ? 0 : 1);
}

// The classes of the 2x2 blocks of the 16-pixel bin at (bx, by), two bits each in row-major
// order: classify_block of each block of the primitive's block grid, 0 where block_may_cover
// drops it.  The same operations on the same values, all four blocks and edges without branches,
// so that the products of a column or row of blocks are taken once and the corners' tests
// combine in scalar registers (expansion of 1M triangles: 45 -> 29 us; one block at a time is
// faster the branching way: 244 us against 282 on 12.7M pairs of 8-pixel bins).
__device__ inline uint32_t classify_blocks4(const float *rec, uint32_t flags, int bx, int by)
{
    const uint32_t *ru = reinterpret_cast<const uint32_t *>(rec);
    const float xf[2] = {(float)bx + 0.5f, (float)(bx + TILE) + 0.5f};
    const float yf[2] = {(float)by + 0.5f, (float)(by + TILE) + 0.5f}, s = 7.0f;
    bool p[4][4][3], may[4] = {true, true, true, true};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float a = rec[REC_EDGE + 3 * k], b = rec[REC_EDGE + 3 * k + 1],
                    c = rec[REC_EDGE + 3 * k + 2];
        const float ax[2] = {a * xf[0], a * xf[1]}, by2[2] = {b * yf[0], b * yf[1]};
        const float as = a * s, bs = b * s, span = s * (fabsf(a) + fabsf(b));
        const float up = fmaxf(0.0f, s * a), vp = fmaxf(0.0f, s * b);
        const bool tie = (flags >> (1 + k)) & 1u;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float x = ax[q & 1], y = by2[q >> 1];
            const float v00 = x + y + c, v01 = v00 + bs;
            p[q][0][k] = edge_pass(v00, tie);
            p[q][1][k] = edge_pass(v01, tie);
            p[q][2][k] = edge_pass(v00 + as, tie);
            p[q][3][k] = edge_pass(v01 + as, tie);
            const float m = fabsf(x) + fabsf(y) + fabsf(c) + span;
            may[q] = may[q] & !(v00 + up + vp < -m * 3.814697265625e-06f);
        }
    }
    const int kx = bx >> 3, ky = by >> 3;
    uint32_t packed = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int x = kx + (q & 1), y = ky + (q >> 1);
        const bool in = (x >= (int)ru[REC_BLOCKS]) & (x <= (int)ru[REC_BLOCKS + 2]) &
                        (y >= (int)ru[REC_BLOCKS + 1]) & (y <= (int)ru[REC_BLOCKS + 3]);
        const int cls = corners_class(p[q]);
        packed |= in & ((cls == 2) | may[q]) ? (uint32_t)cls << (2 * q) : 0u;
    }
    return packed;
}

// Span: a primitive's two flat parts, in registers for walks over several scanlines.
struct SpanRec {
    float ox[2], oy[2], is1[2], is2[2];  // bottom-flat, top-flat
    int lo[2], hi[2];
};

__device__ inline SpanRec load_span(const float *rec)
{
    SpanRec s;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const float *p = rec + (q == 0 ? REC_BOT : REC_TOP);
        s.ox[q] = p[0];
        s.oy[q] = p[1];
        s.is1[q] = p[2];
        s.is2[q] = p[3];
        s.lo[q] = (int)__float_as_uint(p[4]);
        s.hi[q] = (int)__float_as_uint(p[5]);
    }
    return s;
}

// Span: the flat part owning scanline y and its pixel range [xl, xr)
// (Rasterizer.h:370-380 bottom-flat, :397-407 top-flat).  Returns false when no part owns y.
__device__ inline bool span_row_extent(const SpanRec &s, uint32_t flags, int y, int sc_minx,
                                       int sc_maxx, int &xl, int &xr)
{
    const bool inb = (flags & FLAG_BOTTOM) && s.lo[0] <= y && y < s.hi[0];
    const bool intop = (flags & FLAG_TOP) && s.lo[1] < y && y <= s.hi[1];
    const float ox = inb ? s.ox[0] : s.ox[1], oy = inb ? s.oy[0] : s.oy[1];
    const float is1 = inb ? s.is1[0] : s.is1[1], is2 = inb ? s.is2[0] : s.is2[1];
    const float dy = ((float)y - oy) + 0.5f;
    const float cx1 = ox + is1 * dy + 0.5f;
    const float cx2 = ox + is2 * dy + 0.5f;
    xl = imax(sc_minx, f2i(cx1));
    xr = imin(sc_maxx, f2i(cx2));
    return inb || intop;
}

__device__ inline bool span_row_extent(const float *rec, uint32_t flags, int y, int sc_minx,
                                       int sc_maxx, int &xl, int &xr)
{
    return span_row_extent(load_span(rec), flags, y, sc_minx, sc_maxx, xl, xr);
}

// Span: true when some scanline of the square block of `size` pixels at (bx, by) has pixels of
// the primitive inside the block's columns (the ranges the rasterizer computes,
// Rasterizer.h:370-380, 397-407).
__device__ inline bool span_block_any(const SpanRec &s, uint32_t flags, int bx, int by,
                                      int sc_minx, int sc_maxx, int size = TILE)
{
    bool any = false;
    for (int r = 0; r < size && !any; ++r) {
        int xl, xr;
        const bool rowv = span_row_extent(s, flags, by + r, sc_minx, sc_maxx, xl, xr);
        any = rowv && imax(xl, bx) < imin(xr, bx + size);
    }
    return any;
}

// pair value: primitive index | classification << 30 (Block primitives)
constexpr uint32_t PAIR_PRIM_MASK = 0x3FFFFFFFu;
// 16x16 bins whose pair values carry the classes of the bin's four 8x8 blocks: primitive
// index (24 bits) | class of block b << (24 + 2 b), blocks in row-major order (Block: the
// corner classification of Rasterizer.h:270-304 after block_may_cover; Span: 1 when some
// scanline of the block has pixels of the primitive)
constexpr int PAIR_CLS4_SHIFT = 24;
constexpr uint32_t PAIR_CLS4_PRIM_MASK = 0x00FFFFFFu;

// ---- batched draws ------------------------------------------------------------------
// One scene of a batched draw: its inputs, its VertexProcessor / Rasterizer state and its
// render targets.  Scene s owns the virtual triangles [batch0 * 1024, batch0 * 1024 + tris)
// (each scene starts on a fresh 1024-triangle batch, so its draw order is exactly that of
// a draw of its own) and, for each bin size 8 << L (L = 0, 1, 2), the global bins
// [bin0[L], bin0[L] + bins_x[L] * bins_y[L]).
struct SceneDev {
    const int32_t *indices;
    const uint8_t *attr0;
    uint64_t attr0_bytes;
    void *t0, *t1, *t2;
    float mvp[16];
    float vp_px, vp_py, vp_ox, vp_oy, dz_scale, dz_bias;
    int stride0, cull_mode, raster_mode;
    int sc_minx, sc_maxx, sc_miny, sc_maxy;
    int width, height, pitch;
    int bins_x[3], bins_y[3];
    uint32_t bin0[3];
    uint32_t tris, batch0;
};

// Flags of an input triangle's counts: the main pass emits it (not the clip queue); clipping
// appended fan triangles to its batch.
constexpr uint32_t COUNT_LIVE = 1u, COUNT_APPENDS = 2u;

// ---- launch arguments ---------------------------------------------------------------
struct GeomArgs {
    // input
    const int32_t *indices;
    const uint8_t *attr0;
    int stride0;
    uint64_t attr0_bytes;       // 0: unknown
    uint64_t attr0_need;        // bytes the vertex program reads per vertex
    float mvp[16];
    int vs_program, vs_na, vs_np;
    uint32_t tris;              // input triangles (complete triples)
    uint32_t batches;
    // state
    int raster_mode, cull_mode;
    int sc_minx, sc_maxx, sc_miny, sc_maxy;   // scissor as Rasterizer.h:83-86 stores it
    float vp_px, vp_py, vp_ox, vp_oy;         // VertexProcessor.cpp:50-53
    float dz_scale, dz_bias;                  // 0.5f*(f-n), 0.5f*(n+f)
    int width, height, tiles_x, tiles_y;  // tiles_x, tiles_y, tiles: bins of 1 << bin_shift px
    int bin_shift;              // 3, 4 or 5: screen bins of 8, 16 or 32 pixels
    int cls4;                   // 16x16 bins: pair values carry the four block classes
    ParamLayout lay;
    int window_input;           // 1: vertices are window-space RasterizerVertex (IRasterizer seam)
    const swr_rasterizer_vertex *wverts;
    uint64_t wvert_count;
    // scan buffers
    uint32_t *cnt;              // [batches*1024] pairs of each input triangle's first fan
                                // triangle, 0 when it draws nothing
    uint8_t *cflag;             // [batches*1024] COUNT_LIVE, COUNT_APPENDS
    uint2 *app;                 // [batches*1024] {fan triangles appended | drawn ones << 16, their
                                // pairs}, valid where COUNT_APPENDS is set
    const uint2 *ex;            // [batches*1024] (primitives, pairs) before the first fan
                                // triangle, valid where cnt is not 0
    const uint4 *app_ex;        // [tris] {primitives, pairs before the appended ones, fans the
                                // batch has appended before}, valid where COUNT_APPENDS is set
    uint32_t *live;             // [tris] the live triangles in order (nullptr: emit walks all)
    // outputs
    float *prims;               // records
    uint64_t prim_cap;
    uint32_t *pair_keys;        // tile id
    uint32_t *pair_vals;        // primitive index
    uint64_t pair_cap;
    unsigned long long *status;
    uint32_t *ranges;           // [tiles*2] cleared by the count pass
    uint32_t tiles;
    uint32_t sentinel;          // pair key of a tile the primitive cannot shade (dropped)
    uint32_t *prim_pb;          // [prim_cap] index of each primitive's first pair
    uint32_t *chunk_kept;       // [pair_cap / expansion chunk] kept pairs per chunk (or null)
    uint32_t *clipq;            // [tris + 64*256] triangles that straddle a clip plane
    uint32_t *clipq_cnt;        // [DRAW_COUNTER_WORDS]: clip queue regions, raster queues
    // post-transform vertices (the vertex pass; vwin == nullptr: off): window-space
    // (x, y, z, clip w) and the clip mask of each vertex [0, nverts) of attribute 0
    float4 *vwin;
    uint8_t *vmask;
    uint32_t nverts;
    // batched draw: per-scene state replaces the fields above (nscenes == 0: single draw)
    const SceneDev *scenes;
    const uint32_t *batch_scene;  // [batches] scene of each virtual batch
    uint32_t nscenes;
};

// A texture and its mip chain in device memory (swr_texture_create): level k is
// w[k] x h[k] texels 0x00RRGGBB at texels + off[k].
constexpr int TEX_MAX_LEVELS = 32;
struct TexDev {
    const uint32_t *texels;
    int levels, max_aniso;
    int w[TEX_MAX_LEVELS], h[TEX_MAX_LEVELS];
    uint64_t off[TEX_MAX_LEVELS];
};

struct RasterArgs {
    const float *prims;
    int stride;
    const uint32_t *ranges;     // [tiles*2] begin, end into vals
    const uint32_t *vals;       // primitive index per sorted pair
    const unsigned long long *status;
    int tiles, tiles_x;         // bins of 1 << bin_shift pixels
    int bin_shift;
    int cls4;                   // 16x16 bins: pair values carry the four block classes
    int waves_per_bin;          // bins larger than 8x8: waves sharing one bin's blocks
    int width, height, pitch;
    int sc_minx, sc_maxx;       // Span x clipping (Rasterizer.h:377-378, 404-405)
    int na_set, np_set;         // declared counts (hash / log programs)
    int iz, iw;
    void *t0, *t1, *t2;
    uint32_t *log;
    uint64_t log_cap;
    unsigned long long *log_count;
    float checker_cells;
    const SceneDev *scenes;     // batched draw (nscenes == 0: single draw)
    uint32_t nscenes;
    int xcd;                    // 1: tile blocks grouped per XCD
    const TexDev *tex;          // SWR_PS_TEXTURE
    int fold;                   // 0 (modules built earlier read it; the sort folds failures)
    const void *user;           // SWR_PS_MODULE: the program's uniforms (device memory)
    int spans;                  // 0: every primitive is a Block primitive (raster mode Block)
    uint32_t *queue;            // persistent raster: RASTER_QUEUES bin-queue heads, zeroed by the
                                // draw's begin kernel (nullptr: one workgroup per bin)
};

// An asynchronous draw's failures, kept for the next swr_synchronize: once every earlier
// kernel of the draw has finished (stream order), its overflow and error words are final.
// Returns the sticky word.
__device__ inline unsigned long long fold_status(unsigned long long *st)
{
    const unsigned long long f = (st[ST_OVERFLOW] ? 1ull : 0ull) | (st[ST_ERROR] << 1);
    return f ? atomicOr(&st[ST_STICKY], f) | f : st[ST_STICKY];
}

// The last kernel before the raster stage hands the status words, final by then, to the host:
// called by the first wave of one workgroup, a word per lane.  `host` is pinned memory the GPU
// writes in place; a copy after the raster stage would cost a launch of its own (4 us of a
// small frame's 81).
struct StatusOut {
    unsigned long long *host;  // nullptr: nothing to hand over
    int fold;                  // 1: an asynchronous draw; its failures go to ST_STICKY first
};
__device__ inline void hand_over_status(unsigned long long *st, const StatusOut &o)
{
    if (!o.host)
        return;
    const uint32_t lane = threadIdx.x;
    if (lane < (uint32_t)ST_WORDS) {
        const unsigned long long v = lane == ST_STICKY && o.fold ? fold_status(st) : st[lane];
        __hip_atomic_store(&o.host[lane], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Scene-local state of a batched draw over the single-draw arguments.
__device__ inline void apply_scene(GeomArgs &a, const SceneDev &s)
{
    a.indices = s.indices;
    a.attr0 = s.attr0;
    a.attr0_bytes = s.attr0_bytes;
    a.stride0 = s.stride0;
#pragma unroll
    for (int i = 0; i < 16; ++i)
        a.mvp[i] = s.mvp[i];
    a.vp_px = s.vp_px;
    a.vp_py = s.vp_py;
    a.vp_ox = s.vp_ox;
    a.vp_oy = s.vp_oy;
    a.dz_scale = s.dz_scale;
    a.dz_bias = s.dz_bias;
    a.cull_mode = s.cull_mode;
    a.raster_mode = s.raster_mode;
    a.sc_minx = s.sc_minx;
    a.sc_maxx = s.sc_maxx;
    a.sc_miny = s.sc_miny;
    a.sc_maxy = s.sc_maxy;
    a.width = s.width;
    a.height = s.height;
    a.tiles_x = s.bins_x[a.bin_shift - 3];
    a.tiles_y = s.bins_y[a.bin_shift - 3];
}

// The scene owning global bin `tile` of bin level lvl (scenes sorted by bin0[lvl]).
__device__ inline uint32_t scene_of_tile(const SceneDev *sc, uint32_t n, uint32_t tile, int lvl)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (sc[mid].bin0[lvl] <= tile)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

}  // namespace swr
