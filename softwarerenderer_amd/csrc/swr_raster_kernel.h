// swr_raster_kernel.h — the raster stage's kernel: one wave64 per 8x8 block.
//
// A block is exactly one of the reference's 8x8 blocks (Rasterizer.h:247-250 aligns blocks
// to multiples of 8 in window space).  Screen bins of 8x8, 16x16 or 32x32 pixels hold their
// primitives in draw order; the wave walks its block's primitives in that order and every
// pixel's target values (colour/depth, hash/count, ...) stay in registers for the whole
// walk, written back once, coalesced.
//
// Interpolants are reproduced bit for bit by replaying the reference's incremental chains:
//   Block (PixelShaderBase.h:55-94): row start R_j = init(x+.5, y+.5) with +b repeated j
//     times (PixelData::stepY per row), then +a per pixel along the row (stepX); edge
//     values alike.  The corner classification (Rasterizer.h:270-304) was done at binning
//     and rides in the pair value.
//   Span (PixelShaderBase.h:96-112): value(x) = init(xl+.5, y+.5) then +a per pixel from
//     xl, with [xl, xr) from the flat-part edge walk (Rasterizer.h:370-405); the additions
//     before the tile's first column are fast-forwarded (chain_add, swr_chain.h), so a
//     tile's cost does not grow with its distance from the span's start.
//   w = 1/invw and pvar = pvarTemp * w at the pixel (PixelData.h:84-103).
//
// Work split.  The chains are independent of draw order, only shading is not.  So the
// wave takes GS primitives at a time.  Phase A: lane = (slot, row) walks one 8-pixel row
// of one plane of one primitive — 7 adds produce the row — and the rows go through LDS
// into pixel-per-lane layout; with fewer than 8 primitives per group (9 planes or more, for
// the registers' sake) the 8 slots hold several planes of each.  Phase B: lane = pixel shades
// the GS primitives in draw order.
//
// What bounds it: vector issue and the wait for loads, about evenly.  On the 1080p soup of 1M
// triangles it issues 609 G wave instructions/s (plain additions reach 1020 here, compares, fp64
// and 32-bit products 575), and a wave spends 41% of its time waiting for results, 31% ready and
// waiting for issue, 28% issuing; the hash program's longest lists leave the CUs busy for 58% of
// the launch.  Per group of 8 primitives the row starts cost 7 DPP additions per chain (14
// instructions as additions and selects), programs that only test z take no coverage masks (NaN
// rows), coverage of every kind is three stepped compares without branches, a group's record
// loads leave together, and larger bins drop hidden primitives of long lists for programs that
// only test z.  1080p soup of 1M triangles, Block, 16-pixel bins: 109 -> 75 us; 150k triangles,
// Adaptive, 1003x701: 87 -> 69 us; 10-plane hash program on 12.7M pairs: 4699 us with half
// the slots idle, 3239 us with two planes per primitive in them.
//
// The kernel is a template over the pixel program, so that programs compiled outside the
// library (include/swr/pixel_program.h) instantiate it the same way the built-in ones do.
#pragma once

#include <atomic>
#include <type_traits>

#include "swr_common.h"
#include "swr_programs.h"

namespace swr {

// ---- the tile kernel ----------------------------------------------------------------------
// Workgroups are handed to the 8 XCDs round-robin (workgroup b runs on XCD b % 8), and
// each XCD has its own L2.  Renumber so that XCD x works through one contiguous run of
// tile blocks (a band of tile rows): primitive records shared by neighbouring tiles are
// then fetched into one L2 instead of up to eight.  A bijection on [0, n).
constexpr unsigned XCDS = 8;

__device__ inline unsigned xcd_block(unsigned b, unsigned n)
{
    const unsigned q = n / XCDS, r = n % XCDS;
    const unsigned x = b % XCDS, i = b / XCDS;
    return x * q + (x < r ? x : r) + i;
}

// Planes phase A chains for a program: all of them, unless the program declares CHAINED
// (it reads only the first CHAINED per fragment and chains the others itself later).
template <class P, int N, class = void>
struct chained_planes {
    static constexpr int value = N;
};
template <class P, int N>
struct chained_planes<P, N, decltype((void)P::CHAINED)> {
    static constexpr int value = P::CHAINED < N ? P::CHAINED : N;
};

// Programs in which a pixel's last fragment alone decides its targets (LAST_WINS): a block
// walks its list from the end and stops once every pixel has been reached, so its time is
// bound by the layers above the first covering ones instead of by the list (40,960 large
// triangles at 640x480, 240 M fragments, Span, RGB: 1987 us in draw order, 64 us this way;
// one layer, a 1280x720 textured floor: 64 us both ways).
template <class P, class = void>
struct last_wins {
    static constexpr bool value = false;
};
template <class P>
struct last_wins<P, decltype((void)P::LAST_WINS)> {
    static constexpr bool value = P::LAST_WINS;
};

// Programs that only test z (NEAREST): shade reads nothing but v.z(), under `z < x`, which is
// false for NaN.  Phase A then writes NaN where the primitive does not cover the pixel, and
// phase B needs no coverage masks.
template <class P, class = void>
struct nearest_only {
    static constexpr bool value = false;
};
template <class P>
struct nearest_only<P, decltype((void)P::NEAREST)> {
    static constexpr bool value = P::NEAREST;
};

// The largest of the wave's values (NaN left out), in every lane's view the same.
__device__ __forceinline__ float wave_max(float v)
{
#define SWR_MAX_STEP(CTRL, ROWS)                                                                \
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(                                    \
                     __float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xF, false)))
    SWR_MAX_STEP(0x111, 0xF);  // row_shr 1, 2, 4, 8: lane 15 of each row holds its row's
    SWR_MAX_STEP(0x112, 0xF);
    SWR_MAX_STEP(0x114, 0xF);
    SWR_MAX_STEP(0x118, 0xF);
    SWR_MAX_STEP(0x142, 0xA);  // row_bcast 15, 31: lane 63 holds the wave's
    SWR_MAX_STEP(0x143, 0xC);
#undef SWR_MAX_STEP
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// True when no pixel of the 8x8 block at (bx, by) can pass `z < depth` for any depth up to
// zmax, under any rounding of the z chain.  The plane's least value over the block's pixel
// centres is at a corner; it is evaluated in fp32 with at most 9 roundings of terms bounded by
// m = |a xf| + |b yf| + |c| + 7|a| + 7|b| (below 2^-20.8 m).  A Block chain adds 18 roundings of
// partial sums bounded by m (below 2^-19.8 m), so 2^-18 m covers both twice over.  A Span chain
// starts at the span's first pixel, at the scissor's edge at the earliest: n additions of
// partial sums bounded by M, the plane's terms at the farthest pixel of it, so (n + 4) 2^-24 M;
// twice that is taken.  Coefficients or bounds that are not finite keep the primitive.
template <bool SPANS>
__device__ inline bool block_behind(const float *rec, int bx, int by, int sc_minx, float zmax)
{
    const float a = rec[REC_PARAM], b = rec[REC_PARAM + 1], c = rec[REC_PARAM + 2];
    const float xf = (float)bx + 0.5f, yf = (float)by + 0.5f;
    const float lo = a * xf + b * yf + c + fminf(0.0f, 7.0f * a) + fminf(0.0f, 7.0f * b);
    const float m = fabsf(a * xf) + fabsf(b * yf) + fabsf(c) + 7.0f * (fabsf(a) + fabsf(b));
    float err = m * 3.814697265625e-06f;  // 2^-18
    if constexpr (SPANS) {
        if (!(__float_as_uint(rec[REC_FLAGS]) & FLAG_BLOCK)) {
            const float far = fmaxf(fabsf((float)sc_minx), xf + 8.0f);
            const float M = m + fabsf(a) * far;
            err += M * (xf - (float)sc_minx + 32.0f) * 1.1920928955078125e-07f;  // 2^-23
        }
    }
    return lo - err > zmax && m < 1e37f;
}

// Row starts of a block's chains: lane (slot, row) holds K chains' first-row values v and
// steps them `row` times by b.  Rows of a slot are two lanes apart (slot_of / row_of below),
// so a DPP shift by two lanes hands every lane the value of the row above; the lanes of row 0
// have no source inside their 16 lanes and keep theirs.  After step k lane `row` holds the
// chain's value after min(row, k) additions: 7 additions per chain instead of 7 additions and
// 7 selects.  The chains take turns, so a value is read at least two instructions after it is
// written (the DPP read hazard); the leading s_nop covers the values' producers and a change
// of the execution mask.  Every lane of a slot is active or none is.
#define SWR_ROW_STEP(V, B) \
    "v_add_f32_dpp " V ", " V ", " B " row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
#define SWR_ROW_STEPS(X) X X X X X X X
__device__ __forceinline__ void row_starts(float (&v)[1], const float (&b)[1])
{
    __asm__ volatile("s_nop 4\n\t" SWR_ROW_STEPS(SWR_ROW_STEP("%0", "%1") "s_nop 1\n\t")
            : "+&v"(v[0])
            : "v"(b[0]));
}
__device__ __forceinline__ void row_starts(float (&v)[2], const float (&b)[2])
{
    __asm__ volatile("s_nop 4\n\t" SWR_ROW_STEPS(SWR_ROW_STEP("%0", "%2") SWR_ROW_STEP("%1", "%3")
                                                     "s_nop 0\n\t")
                     : "+&v"(v[0]), "+&v"(v[1])
                     : "v"(b[0]), "v"(b[1]));
}
__device__ __forceinline__ void row_starts(float (&v)[3], const float (&b)[3])
{
    __asm__ volatile("s_nop 4\n\t" SWR_ROW_STEPS(SWR_ROW_STEP("%0", "%3") SWR_ROW_STEP("%1", "%4")
                                            SWR_ROW_STEP("%2", "%5"))
            : "+&v"(v[0]), "+&v"(v[1]), "+&v"(v[2])
            : "v"(b[0]), "v"(b[1]), "v"(b[2]));
}
#undef SWR_ROW_STEP
#undef SWR_ROW_STEPS

// Phase A's lanes: slots 2q and 2q + 1 share 16 lanes, rows two lanes apart.
__device__ inline int slot_of(int lane) { return ((lane >> 4) << 1) | (lane & 1); }
__device__ inline int row_of(int lane) { return (lane >> 1) & 7; }
constexpr int slot_lane(int slot) { return ((slot >> 1) << 4) | (slot & 1); }
// a slot's 64 row values in LDS, 4 words apart from the next slot's: the two slots of 16 lanes
// write different banks
constexpr int SLOT_WORDS = 68;

// The next work item of a persistent raster workgroup: the first unclaimed item of queue
// home, home + 1, ... (mod RASTER_QUEUES); queues found empty are not asked again.  `items`
// items are dealt into the queues as contiguous runs.  NO_ITEM once every queue is empty.
constexpr uint32_t NO_ITEM = 0xFFFFFFFFu;

// Called by a whole wave (lane 0 claims; the values stay wave-uniform, in scalar registers).
__device__ inline uint32_t take_item(uint32_t *queue, uint32_t items, uint32_t home,
                                     uint32_t &tried, int lane)
{
    const uint32_t q = items / RASTER_QUEUES, r = items % RASTER_QUEUES;
    while (tried < RASTER_QUEUES) {
        const uint32_t x = (home + tried) % RASTER_QUEUES;
        const uint32_t first = x * q + (x < r ? x : r), len = q + (x < r ? 1u : 0u);
        uint32_t i = 0;
        if (lane == 0)
            i = atomicAdd(&queue[x * RASTER_QUEUE_STRIDE], 1u);
        i = __builtin_amdgcn_readlane(i, 0);
        if (i < len)
            return first + i;
        ++tried;
    }
    return NO_ITEM;
}

// The raster kernel.  A workgroup takes either raster_waves bins of 8x8 pixels (one wave per
// bin: the bin is one block and its list carries each primitive's block class), or one bin of
// 16x16 or 32x32 pixels whose 4 or 16 blocks its waves share (wave w takes blocks w, w + W,
// ...): each wave reads the bin's list and keeps, in a per-wave ring in LDS, the primitives
// its block classifies as drawn (Rasterizer.h:270-304 with block_may_cover, or the Span
// rows), in list order.
// MODE 0: 8x8 bins; 1: 16x16 bins whose pair values carry the block classes; 2: larger bins
// whose blocks the kernel classifies.
// SPANS = false: every primitive of the draw is a Block primitive (raster mode Block), so the
// kernel carries no Span code and its registers.
template <template <class> class ProgT, int NZ, int NW, int NA, int NP, int GSX, int MODE,
          bool QUEUE, bool SPANS>
__global__ void __launch_bounds__(512) k_raster(RasterArgs a0)
{
    constexpr bool FILT = MODE != 0;
    using L = Layout<NZ, NW, NA, NP>;
    using Prog = ProgT<L>;
    constexpr int N = L::N;
    constexpr int NS = N > 0 ? N : 1;
    constexpr int NC = chained_planes<Prog, N>::value;  // planes phase A chains
    constexpr bool LAST = last_wins<Prog>::value;
    // primitives per group: the program's default, or the tuned value
    constexpr int GS = GSX > 0 ? GSX : (N <= 8 ? 8 : (N <= 16 ? 4 : (N <= 32 ? 2 : 1)));
    static_assert(GS >= 1 && GS <= 8 && (GS & (GS - 1)) == 0, "at most 8 primitives a group");
    constexpr int PP = 8 / GS;  // planes phase A chains side by side: its 8 slots hold GS
                                // primitives times PP planes
    constexpr bool NEAREST = nearest_only<Prog>::value;
    static_assert(!NEAREST || NC == 1, "a program that only tests z chains z alone");
    constexpr int MAXW = MODE == 0 ? 8 : 4;  // waves per workgroup: blockDim.x / 64 at most
    constexpr uint32_t RING = 128;  // per-wave ring of a larger bin's drawn primitives
    constexpr int RW = FILT ? MAXW : 1;
    constexpr int ROWS = NC > 0 ? 8 * SLOT_WORDS : 4;
    __shared__ __align__(16) float s_rows[MAXW][ROWS];
    __shared__ unsigned long long s_cov[NEAREST ? 1 : MAXW][GS];
    __shared__ uint32_t s_ring[RW][RING];

    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wpb = (int)(blockDim.x >> 6);
    // 8x8 blocks per bin side: 1 for 8x8 bins (FILT = false), else 2 or 4
    const int S = FILT ? 1 << (a0.bin_shift - 3) : 1;
    if (a0.status[ST_OVERFLOW] | a0.status[ST_ERROR])
        return;
    // phase B: lane = pixel (pi, pj); phase A: lane = (slot, row)
    const int pi = lane & 7, pj = lane >> 3;
    const int lslot = slot_of(lane), row = row_of(lane);
    const int slot = lslot & (GS - 1), sub = lslot / GS;  // primitive of the group, plane of PP
    float *rows = s_rows[wv];
    unsigned char *covb = reinterpret_cast<unsigned char *>(s_cov[NEAREST ? 0 : wv]);
    uint32_t *ring = s_ring[FILT ? wv : 0];
    const unsigned long long below = (1ull << lane) - 1ull;

    // The work items are the workgroups of the launch: wpb 8x8 bins (one per wave), or one
    // larger bin whose blocks the waves share.  With QUEUE, persistent workgroups take items
    // from RASTER_QUEUES queues, each a contiguous run of items (queues QPX x .. QPX x + QPX - 1
    // a band of bin rows for XCD x; workgroup b runs on XCD b % 8), their own queue first, then
    // the next ones (stealing), and leave once all queues are past their ends.  A workgroup
    // keeps its waves on one item at a time, so they share its pair lists and primitive
    // records in the CU's cache as the waves of a launched workgroup do.  Without QUEUE, each
    // workgroup draws the item of its launch index.  An item's bits do not depend on the
    // workgroup that draws it.
    constexpr uint32_t QPX = RASTER_QUEUES / XCDS;  // queues per XCD
    static_assert(QPX >= 1 && QPX * XCDS == RASTER_QUEUES, "whole queues per XCD");
    __shared__ uint32_t s_item;
    const uint32_t items = S == 1 ? ((uint32_t)a0.tiles + (uint32_t)wpb - 1) / (uint32_t)wpb
                                  : (uint32_t)a0.tiles;
    const uint32_t home = (blockIdx.x % XCDS) * QPX + (blockIdx.x / XCDS) % QPX;
    // wave 0 takes the next item while the waves draw the current one
    uint32_t tried = 0, next = 0;  // (wave 0) queues found empty, the item taken
    if (QUEUE && wv == 0)
        next = take_item(a0.queue, items, home, tried, lane);
    bool taken = false;
    for (;;) {
        uint32_t item;
        if constexpr (!QUEUE) {
            if (taken)
                break;
            taken = true;
            item = a0.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
        } else {
            if (threadIdx.x == 0)
                s_item = next;
            __syncthreads();
            item = __builtin_amdgcn_readfirstlane(s_item);
            if (item == NO_ITEM)
                break;
            __syncthreads();  // every wave has read the item before wave 0 writes the next
            if (wv == 0)
                next = take_item(a0.queue, items, home, tried, lane);
        }
        const int tile =
            __builtin_amdgcn_readfirstlane(S == 1 ? (int)item * wpb + wv : (int)item);
        if (tile >= a0.tiles)
            continue;
        const uint32_t beg = a0.ranges[2 * tile], end = a0.ranges[2 * tile + 1];
        if (beg >= end)
            continue;
        RasterArgs a = a0;
        int lt = tile;  // bin index within its target
        if (a0.nscenes) {
            const int lvl = a0.bin_shift - 3;
            const SceneDev &Sc =
                a0.scenes[scene_of_tile(a0.scenes, a0.nscenes, (uint32_t)tile, lvl)];
            a.width = Sc.width;
            a.height = Sc.height;
            a.pitch = Sc.pitch;
            a.tiles_x = Sc.bins_x[lvl];
            a.sc_minx = Sc.sc_minx;
            a.sc_maxx = Sc.sc_maxx;
            a.t0 = Sc.t0;
            a.t1 = Sc.t1;
            a.t2 = Sc.t2;
            lt = tile - (int)Sc.bin0[lvl];
        }
        const int tx = lt % a.tiles_x, ty = lt / a.tiles_x;
        for (int bi = S == 1 ? 0 : wv; bi < S * S; bi += S == 1 ? 1 : wpb) {
            const int bx = (tx << a.bin_shift) + (bi % S) * TILE;
            const int by = (ty << a.bin_shift) + (bi / S) * TILE;
            if (bx >= a.width || by >= a.height)
                continue;
            const int px = bx + pi, py = by + pj;
            const bool inside = px < a.width && py < a.height;
            const size_t o = (size_t)py * (size_t)a.pitch + (size_t)px;
            const int ry = by + row;
            const float ryf = (float)ry;
            const float xf = (float)bx + 0.5f, yf = (float)by + 0.5f;

            typename Prog::State st;
            if (inside)
                Prog::load(st, a, o);
            bool drew = false;  // a larger bin's block may keep no primitive: nothing to store

            // next list entry to read, counted in walking order (LAST: from the list's end)
            uint32_t pos = 0;
            const uint32_t num = end - beg;
            const auto entry = [&](uint32_t k) { return LAST ? end - 1u - k : beg + k; };
            uint32_t head = 0, tail = 0;   // ring of the block's drawn primitives (S > 1)
            for (;;) {
                int cnt;
                if (!FILT) {
                    if (pos >= num)
                        break;
                    cnt = (int)((num - pos) < (uint32_t)GS ? (num - pos) : (uint32_t)GS);
                } else {
                    while (tail - head < (uint32_t)GS && pos < num) {
                        const uint32_t i = pos + (uint32_t)lane;
                        uint32_t pv = 0;
                        bool keep = false;
                        if (i < num && MODE == 1) {
                            pv = a.vals[entry(i)];
                            const uint32_t cls = (pv >> (PAIR_CLS4_SHIFT + 2 * bi)) & 3u;
                            keep = cls != 0;
                            pv = (pv & PAIR_CLS4_PRIM_MASK) | cls << 30;
                        } else if (i < num) {
                            pv = a.vals[entry(i)] & PAIR_PRIM_MASK;
                            const float *rec = a.prims + (size_t)pv * (size_t)a.stride;
                            const uint32_t flags = __float_as_uint(rec[REC_FLAGS]);
                            if (!SPANS || (flags & FLAG_BLOCK)) {
                                // a block of the primitive's block grid (the scissor clamps the
                                // grid, Rasterizer.h:240-250, not the triangle), then its class
                                const uint32_t *ru = reinterpret_cast<const uint32_t *>(rec);
                                const int kx = bx >> 3, ky = by >> 3;
                                int cls = 0;
                                if (kx >= (int)ru[REC_BLOCKS] && kx <= (int)ru[REC_BLOCKS + 2] &&
                                    ky >= (int)ru[REC_BLOCKS + 1] &&
                                    ky <= (int)ru[REC_BLOCKS + 3]) {
                                    cls = classify_block(rec + REC_EDGE, flags, bx, by);
                                    if (cls == 1 && !block_may_cover(rec + REC_EDGE, bx, by))
                                        cls = 0;
                                }
                                keep = cls != 0;
                                pv |= (uint32_t)cls << 30;
                            } else {
                                keep = span_block_any(load_span(rec), flags, bx, by, a.sc_minx,
                                                      a.sc_maxx);
                            }
                        }
                        // Past a list's first 64 entries, programs that only test z drop what
                        // lies behind the block's farthest pixel so far: a record read and some
                        // 25 instructions for 64 entries instead of a group's for 8 (soup of 1M
                        // triangles, 1920x1080, 16-pixel bins: 82 -> 74 us).  8x8 bins' lists
                        // are a quarter as long and have no ring.
                        if constexpr (NEAREST)
                            if (pos > 0) {
                                const float zmax =
                                    wave_max(inside ? st.depth : -__builtin_inff());
                                if (keep)
                                    keep = !block_behind<SPANS>(
                                        a.prims + (size_t)(pv & PAIR_PRIM_MASK) *
                                                      (size_t)a.stride,
                                        bx, by, a.sc_minx, zmax);
                            }
                        const unsigned long long m = __ballot(keep);
                        if (keep)
                            ring[(tail + (uint32_t)__popcll(m & below)) & (RING - 1)] = pv;
                        tail += (uint32_t)__popcll(m);
                        pos += 64;
                    }
                    lds_sync();
                    if (tail == head)
                        break;
                    cnt = (int)((tail - head) < (uint32_t)GS ? (tail - head) : (uint32_t)GS);
                }
                drew = true;
                const bool act = slot < cnt;
                uint32_t pv = 0u;
                if (act)
                    pv = !FILT ? a.vals[entry(pos + (uint32_t)slot)]
                               : ring[(head + (uint32_t)slot) & (RING - 1)];
                if (!FILT)
                    pos += (uint32_t)cnt;
                else
                    head += (uint32_t)cnt;
                // idle slots (slot >= cnt) read record 0: the loads need no branch
                const float *__restrict__ rec =
                    a.prims + (size_t)(pv & PAIR_PRIM_MASK) * (size_t)a.stride;
                const int cls = (int)(pv >> 30);
                const uint32_t flags = __float_as_uint(rec[REC_FLAGS]);
                const uint32_t key = __float_as_uint(rec[Prog::KEY_WORD]);
                const bool blk = !SPANS || (flags & FLAG_BLOCK) != 0;
                float zp[3] = {0.0f, 0.0f, 0.0f};
                if constexpr (NEAREST) {
                    zp[0] = rec[REC_PARAM];
                    zp[1] = rec[REC_PARAM + 1];
                    zp[2] = rec[REC_PARAM + 2];
                }

                // Coverage of this lane's row as three functions stepped along its columns: a
                // pixel is in when each value is at least its limit (edge_pass).  Block: the
                // edges; a full block, all zero with limit 0; an idle slot or a row without
                // pixels, an infinite limit.
                float ev[3] = {0.0f, 0.0f, 0.0f}, ea[3] = {0.0f, 0.0f, 0.0f};
                float lim[3] = {0.0f, 0.0f, 0.0f};
                const bool part = act && blk && cls != 2;
                if (__ballot(part) != 0ull) {
                    float eb[3];
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        ea[e] = rec[REC_EDGE + 3 * e];
                        eb[e] = rec[REC_EDGE + 3 * e + 1];
                        ev[e] = ea[e] * xf + eb[e] * yf + rec[REC_EDGE + 3 * e + 2];
                    }
                    row_starts(ev, eb);
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        ev[e] = part ? ev[e] : 0.0f;
                        ea[e] = part ? ea[e] : 0.0f;
                        lim[e] = part && !((flags >> (1 + e)) & 1u) ? __uint_as_float(1u) : 0.0f;
                    }
                }
                // Span: this row's part and [xl, xr) (Rasterizer.h:370-380, 397-407), as
                // i - dl >= 0 and dr - 1 - i >= 0
                int xl = 0, dl = 0;
                if constexpr (SPANS) {
                    if (act && !blk) {
                        int xr = 0;
                        const bool rowv =
                            span_row_extent(rec, flags, ry, a.sc_minx, a.sc_maxx, xl, xr);
                        dl = xl <= bx ? 0 : (xl - bx < 8 ? xl - bx : 8);
                        const int dr = xr <= bx ? 0 : (xr - bx < 8 ? xr - bx : 8);
                        ev[0] = -(float)dl;
                        ea[0] = 1.0f;
                        ev[1] = (float)(dr - 1);
                        ea[1] = -1.0f;
                        lim[2] = rowv ? 0.0f : __builtin_inff();
                    }
                }
                if (!act)
                    lim[2] = __builtin_inff();
                const float xs = (float)xl + 0.5f, ys = ryf + 0.5f;
                const int pre = bx - xl;  // Span: chain steps from xl to the block's first column
                // whether column i of this lane's row is covered, for i = 0 .. 7 in turn
                const auto column = [&]() {
                    const bool in = ev[0] >= lim[0] && ev[1] >= lim[1] && ev[2] >= lim[2];
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        ev[e] = ev[e] + ea[e];
                    return in;
                };
                // the first column's value of plane (pa, pb, pc) on this lane's row
                // (K planes at once: pa, pb, pc; the value replaces pc)
                const auto first = [&](const auto &pa, const auto &pb, auto &pc) {
                    constexpr int K = (int)(sizeof(pc) / sizeof(float));
                    float r[K];
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        r[k] = pa[k] * xf + pb[k] * yf + pc[k];
                    if (!SPANS || __ballot(act && blk) != 0ull)
                        row_starts(r, pb);
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        if constexpr (SPANS)
                            if (act && !blk)  // init at xl, then the additions to column 0
                                r[k] = chain_add(pa[k] * xs + pb[k] * ys + pc[k], pa[k], pre);
                        pc[k] = r[k];
                    }
                };

                float val[GS][NS];
                float *to = rows + lslot * SLOT_WORDS + row * 8;
                if constexpr (NEAREST) {
                    // the z row with NaN where the primitive does not cover the pixel
                    const float pa[1] = {zp[0]}, pb[1] = {zp[1]};
                    float z[1] = {zp[2]};
                    first(pa, pb, z);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        float q[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            q[i] = column() ? z[0] : __uint_as_float(0x7FC00000u);
                            if (!SPANS || 4 * h + i >= dl)
                                z[0] = z[0] + pa[0];
                        }
                        *reinterpret_cast<float4 *>(to + 4 * h) =
                            make_float4(q[0], q[1], q[2], q[3]);
                    }
                    lds_sync();
#pragma unroll
                    for (int s2 = 0; s2 < GS; ++s2)
                        val[s2][0] = rows[s2 * SLOT_WORDS + lane];
                } else {
                    uint32_t rowmask = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        rowmask |= column() ? (1u << i) : 0u;
                    if (act && (GS == 8 || sub == 0))
                        covb[slot * 8 + row] = (unsigned char)rowmask;
                    // chained values: phase A row walk, then transpose to pixel-per-lane; pass
                    // t takes planes PP t .. PP t + PP - 1 of every primitive of the group
                    constexpr int PASSES = (NC + PP - 1) / PP;
                    const float *pl = rec + REC_PARAM + 3 * sub;
                    const auto passes = [&](auto kc, int t0) {
                        constexpr int K = decltype(kc)::value;  // passes whose starts go together
                        float pa[K], pb[K], v[K];
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            const int p = PP * (t0 + k);
                            // lanes past the last plane read it again
                            const float *q = p + PP <= NC || sub < NC - p
                                                 ? pl + 3 * p
                                                 : rec + REC_PARAM + 3 * (NC - 1);
                            pa[k] = q[0];
                            pb[k] = q[1];
                            v[k] = q[2];
                        }
                        first(pa, pb, v);
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            float out[8];
#pragma unroll
                            for (int i = 0; i < 8; ++i) {
                                out[i] = v[k];
                                if (!SPANS || i >= dl)
                                    v[k] = v[k] + pa[k];
                            }
                            *reinterpret_cast<float4 *>(to) =
                                make_float4(out[0], out[1], out[2], out[3]);
                            *reinterpret_cast<float4 *>(to + 4) =
                                make_float4(out[4], out[5], out[6], out[7]);
                            lds_sync();
#pragma unroll
                            for (int u = 0; u < PP; ++u) {
                                const int p = PP * (t0 + k) + u;
                                if (p < NC)
#pragma unroll
                                    for (int s2 = 0; s2 < GS; ++s2)
                                        val[s2][p] = rows[(u * GS + s2) * SLOT_WORDS + lane];
                            }
                            lds_sync();
                        }
                    };
#pragma unroll
                    for (int t = 0; t + 3 <= PASSES; t += 3)
                        passes(std::integral_constant<int, 3>{}, t);
                    if constexpr (PASSES % 3 == 2)
                        passes(std::integral_constant<int, 2>{}, PASSES - 2);
                    else if constexpr (PASSES % 3 == 1)
                        passes(std::integral_constant<int, 1>{}, PASSES - 1);
                    if (NC == 0)
                        lds_sync();
                }

                // phase B: shade the group's primitives in walking order: draw order, or with
                // LAST the reverse, where only a pixel's first fragment is shaded
#pragma unroll
                for (int s2 = 0; s2 < GS; ++s2) {
                    if constexpr (NEAREST) {  // slots beyond cnt hold NaN
                        const uint32_t k2 = __builtin_amdgcn_readlane(key, slot_lane(s2));
                        const uint32_t prim2 =
                            Prog::PLANES ? __builtin_amdgcn_readlane(pv, slot_lane(s2)) &
                                               PAIR_PRIM_MASK
                                         : 0u;
                        Prog::shade(st, a, ChainPixel<L, SPANS>{val[s2], prim2}, k2, px, py);
                    } else if (s2 < cnt) {
                        const unsigned long long m = s_cov[wv][s2];
                        const uint32_t k2 = __builtin_amdgcn_readlane(key, slot_lane(s2));
                        const uint32_t prim2 =
                            Prog::PLANES ? __builtin_amdgcn_readlane(pv, slot_lane(s2)) &
                                               PAIR_PRIM_MASK
                                         : 0u;
                        bool shaded = ((m >> lane) & 1ull) && inside;
                        if constexpr (LAST)
                            shaded = shaded && !st.hit;
                        if (shaded)
                            Prog::shade(st, a, ChainPixel<L, SPANS>{val[s2], prim2}, k2, px,
                                        py);
                    }
                }
                lds_sync();
                if constexpr (LAST)
                    if (__ballot(inside && !st.hit) == 0ull)
                        break;  // the rest of the list lies under what is drawn
            }
            if (inside && drew)
                Prog::template store<ChainPixel<L, SPANS>>(st, a, o, px, py);
        }
    }
}

// Workgroups of `threads` threads of `kernel` that the GPU holds at once (its CUs times the
// kernel's occupancy per CU), kept in `known` per device and workgroup size (each kernel
// keeps its own); 0 when the runtime cannot tell.
inline uint32_t resident_groups(const void *kernel, uint32_t threads,
                                std::atomic<uint32_t> (&known)[16][9])
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16 || threads / 64 > 8)
        return 0;
    std::atomic<uint32_t> &slot = known[dev][threads / 64];
    uint32_t v = slot.load(std::memory_order_relaxed);
    if (v)
        return v;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, (int)threads, 0) !=
            hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    v = (uint32_t)(cus > 0 ? cus : 0) * (uint32_t)(per > 0 ? per : 0);
    slot.store(v, std::memory_order_relaxed);
    return v;
}

// One raster launch of `blocks` workgroups of `w` waves; with a queue, as many persistent
// workgroups as the GPU holds at once (at most `blocks`).
template <template <class> class ProgT, int NZ, int NW, int NA, int NP, int GSX, int MODE,
          bool SPANS>
inline hipError_t launch_mode(const RasterArgs &a, uint32_t blocks, uint32_t w, hipStream_t s)
{
    if (a.queue) {
        static std::atomic<uint32_t> known[16][9];  // [device][threads / 64]
        const uint32_t res = resident_groups(
            reinterpret_cast<const void *>(
                &k_raster<ProgT, NZ, NW, NA, NP, GSX, MODE, true, SPANS>),
            64 * w, known);
        if (res) {
            hipLaunchKernelGGL((k_raster<ProgT, NZ, NW, NA, NP, GSX, MODE, true, SPANS>),
                               dim3(blocks < res ? blocks : res), dim3(64 * w), 0, s, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_raster<ProgT, NZ, NW, NA, NP, GSX, MODE, false, SPANS>),
                       dim3(blocks), dim3(64 * w), 0, s, a);
    return hipGetLastError();
}

// 8x8 bins: `waves` bins per workgroup, one wave each; larger bins: one bin per workgroup
// of a.waves_per_bin waves.
template <template <class> class ProgT, int NZ, int NW, int NA, int NP, int GSX = 0>
inline hipError_t launch(const RasterArgs &a, hipStream_t s, int waves)
{
    uint32_t w = (uint32_t)waves, blocks = (uint32_t)((a.tiles + w - 1) / w);
    if (a.bin_shift > 3) {
        w = (uint32_t)a.waves_per_bin;
        blocks = (uint32_t)a.tiles;
    }
    if (!blocks)
        return hipSuccess;
    const int mode = a.bin_shift > 3 ? (a.cls4 ? 1 : 2) : 0;
    if (a.spans) {
        if (mode == 1)
            return launch_mode<ProgT, NZ, NW, NA, NP, GSX, 1, true>(a, blocks, w, s);
        if (mode == 2)
            return launch_mode<ProgT, NZ, NW, NA, NP, GSX, 2, true>(a, blocks, w, s);
        return launch_mode<ProgT, NZ, NW, NA, NP, GSX, 0, true>(a, blocks, w, s);
    }
    if (mode == 1)
        return launch_mode<ProgT, NZ, NW, NA, NP, GSX, 1, false>(a, blocks, w, s);
    if (mode == 2)
        return launch_mode<ProgT, NZ, NW, NA, NP, GSX, 2, false>(a, blocks, w, s);
    return launch_mode<ProgT, NZ, NW, NA, NP, GSX, 0, false>(a, blocks, w, s);
}

}  // namespace swr
