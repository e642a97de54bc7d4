// swr_lines.hip — points and lines on gfx950.
//
// The reference draws a line as a DDA (Rasterizer.h:175-222): steps = max(|dx|, |dy|) of the
// truncated endpoints, one per-step increment per value, each step's vertex handed to the
// pixel shader as it is (pixelDataFromVertex, Rasterizer.h:160-173) when it passes the
// scissor test.  The vertex of step k is a chain of k float additions: a line is walked in
// pieces of LINE_PIECE steps, each started with the chain's value there (chain_add) and taken
// by a lane of its own.  A point is a line of one step with no increment (drawPointTemplate,
// Rasterizer.h:149-158).
//
// Draw sequence:
//   count   per primitive: vertex program, LineClipper / clipPoints, viewport transform and
//           a walk of the x/y chain counting the fragments that pass the scissor test and
//           land on the target; each workgroup's totals
//   scan    exclusive scan of the counts: each primitive's first fragment, in draw order; the
//           totals into the status words
//   emit    the same walk with every value: fragment records and (tile, fragment) pairs
//   sort    stable radix sort of the pairs by tile (the triangle path's sort)
//   raster  one wave64 per 8x8 tile: lane = pixel, the tile's fragments in draw order
//           through the pixel program (the triangle path's programs)
// Fragment order within a pixel is the reference's invocation order: fragments are numbered
// in (primitive, step) order and the sort is stable.
#include "swr_chain.h"
#include "swr_common.h"
#include "swr_internal.h"
#include "swr_lines_kernel.h"
#include "swr_programs.h"
#include "swr_vertex.h"

namespace swr {

int fragment_stride(const ParamLayout &L) { return FR_VAR + emit_class(L.na + L.np); }

template <int NV>
struct LVert {
    float x, y, z, w;
    float v[NV > 0 ? NV : 1];
};

// LineClipper::clipToPlane, LineClipper.cpp:30-56, plane p of VertexProcessor.cpp:197-202
__device__ inline void clip_line_plane(int p, const Pos4 &v0, const Pos4 &v1, float &t0, float &t1,
                                       bool &clipped)
{
    if (clipped)
        return;
    const float dp0 = plane_dot(p, v0), dp1 = plane_dot(p, v1);
    const bool n0 = dp0 < 0, n1 = dp1 < 0;
    if (n0 && n1) {
        clipped = true;
        return;
    }
    if (n0) {
        const float t = -dp0 / (dp1 - dp0);
        t0 = ref_max(t0, t);
    } else {
        const float t = dp0 / (dp0 - dp1);
        t1 = ref_min(t1, t);
    }
}

// Window-space vertices of primitive i.  False when the primitive draws nothing (skipped,
// clipped, or an index error, which is flagged in the status words).
//   drawElements: VertexProcessor.cpp:78-120 (batches of 1024 primitives) -> clipLines
//     (:167-215) or clipPoints (:152-165) -> transformVertices (:347-377) -> the list entry.
//   IRasterizer seam: drawLineList / drawPointList (Rasterizer.h:116-132).
template <int NV>
__device__ bool prepare_primitive(const LineArgs &A, uint64_t i, LVert<NV> *V)
{
    const GeomArgs &a = A.g;
    const int nv = A.mode == SWR_DRAW_LINE ? 2 : 1;
    const uint64_t ib = (uint64_t)nv * i;
    int32_t ids[2];
    ids[0] = a.indices[ib];
    ids[1] = nv == 2 ? a.indices[ib + 1] : ids[0];
    if (a.window_input) {
        if (ids[0] == -1)
            return false;  // Rasterizer.h:119, 128
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (q < nv && (ids[q] < 0 || (uint64_t)ids[q] >= a.wvert_count)) {
                atomicOr(&a.status[ST_ERROR], 1ull);
                return false;
            }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const swr_rasterizer_vertex &s = a.wverts[ids[q]];
            V[q].x = s.x;
            V[q].y = s.y;
            V[q].z = s.z;
            V[q].w = s.w;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int k2 = k - a.lay.na;
                V[q].v[k] = k < a.lay.na ? s.avar[k & 15] : (k2 < a.lay.np ? s.pvar[k2 & 15] : 0.0f);
            }
        }
        return true;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (q < nv && (ids[q] < 0 || (a.attr0_bytes && (uint64_t)ids[q] * (uint64_t)a.stride0 +
                                                            a.attr0_need > a.attr0_bytes))) {
            atomicOr(&a.status[ST_ERROR], 1ull);
            return false;
        }
    Pos4 P[2];
    float var[2][NV > 0 ? NV : 1];
#pragma unroll
    for (int q = 0; q < 2; ++q)
        fetch_vertex<NV>(a, ids[q], P[q], var[q]);  // a point fetches its vertex twice
    if (nv == 1) {
        if (clip_mask(P[0]))
            return false;
    } else {
        const int m0 = clip_mask(P[0]), m1 = clip_mask(P[1]);
        const int cm = m0 | m1;
        float t0 = 0.0f, t1 = 1.0f;
        bool clipped = false;
#pragma unroll
        for (int p = 0; p < 6; ++p)
            if (cm & (1 << p))
                clip_line_plane(p, P[0], P[1], t0, t1, clipped);
        if (clipped)
            return false;
        // Helper::interpolateVertex (PolyClipper.h:34-48) from the unclipped endpoints
        const Pos4 A0 = P[0], A1 = P[1];
        float var0[NV > 0 ? NV : 1], var1[NV > 0 ? NV : 1];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            var0[k] = var[0][k];
            var1[k] = var[1][k];
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (!(q == 0 ? m0 : m1))
                continue;
            const float t = q == 0 ? t0 : t1;
            P[q].x = lerp1(A0.x, A1.x, t);
            P[q].y = lerp1(A0.y, A1.y, t);
            P[q].z = lerp1(A0.z, A1.z, t);
            P[q].w = lerp1(A0.w, A1.w, t);
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const bool lerped = k < a.lay.na ? (k < a.vs_na) : ((k - a.lay.na) < a.vs_np);
                var[q][k] = lerped ? lerp1(var0[k], var1[k], t) : 0.0f;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const WinV w = to_window(a, P[q]);
        V[q].x = w.x;
        V[q].y = w.y;
        V[q].z = w.z;
        V[q].w = w.w;
#pragma unroll
        for (int k = 0; k < NV; ++k)
            V[q].v[k] = var[q][k];
    }
    return true;
}

// Rasterizer::scissorTest, Rasterizer.h:143-147
__device__ inline bool scissor_pass(const GeomArgs &a, float x, float y)
{
    return x >= (float)a.sc_minx && x < (float)a.sc_maxx && y >= (float)a.sc_miny &&
           y < (float)a.sc_maxy;
}

// The pixel a step lands on, when the shader would touch the target there.
__device__ inline bool on_target(const GeomArgs &a, float x, float y, int &px, int &py)
{
    if (!scissor_pass(a, x, y))
        return false;
    px = f2i(x);
    py = f2i(y);
    return px >= 0 && py >= 0 && px < a.width && py < a.height;
}

__device__ inline unsigned long long wave_sum(unsigned long long v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

// One fragment record and its (tile, fragment) pair.
template <int NV>
__device__ inline void write_fragment(const LineArgs &A, uint64_t f, uint64_t i, int px, int py,
                                      const LVert<NV> &v)
{
    const GeomArgs &a = A.g;
    float *r = A.frags + f * (uint64_t)A.fstride;
    r[FR_X] = __uint_as_float((uint32_t)px);
    r[FR_Y] = __uint_as_float((uint32_t)py);
    r[FR_KEY] = __uint_as_float(a.window_input ? (uint32_t)i
                                               : ((uint32_t)(i >> 10) << 15) + (uint32_t)(i & 1023u));
    r[FR_SRC] = __uint_as_float((uint32_t)i);
    r[FR_Z] = v.z;
    r[FR_W] = v.w;
#pragma unroll
    for (int k = 0; k < NV; ++k)
        r[FR_VAR + k] = v.v[k];
    A.keys[f] = (uint32_t)(py >> 3) * (uint32_t)a.tiles_x + (uint32_t)(px >> 3);
    A.vals[f] = (uint32_t)f;
}

// A wave takes LINES primitives, a lane each for their setup; the lines' steps are then dealt to
// all lanes in pieces, line by line, so that a wave takes as long as its lines together and not
// as its longest.  Bound by the serial steps of a piece (and in the emit pass by its scattered
// record stores): 60,000 lines, a fifth of them across a 1920x1080 screen, took 269 us to count
// and 656 us to emit with a thread per line, now 117 and 374 us (195 and 453 us with 64 lines per
// wave, which leaves too few waves); 60,000 points 48 us to count with the totals as atomics on
// two words, now 6 us.
constexpr uint32_t LINE_PIECE = 32, LINES = 16;

// FAR: a launch of later workgroups, from A.group0 on (launch_walk).
template <int NV, bool EMIT, bool FAR>
__global__ void __launch_bounds__(64) k_lines_walk(LineArgs A)
{
    constexpr int W = 4 + NV, ST = 2 * W + 1;  // start and step; odd: lines spread over banks
    __shared__ float s_line[LINES * ST];
    __shared__ uint32_t s_steps[LINES], s_first[LINES], s_done[LINES];
    const GeomArgs &a = A.g;
    const uint32_t lane = threadIdx.x, group = (FAR ? A.group0 : 0u) + blockIdx.x;
    const uint64_t base = (uint64_t)group * LINES, i = base + lane;
    LVert<NV> V[2];
    const bool mine = lane < LINES && i < A.prims;
    bool live = mine && (!EMIT || A.count[i].y != 0u) && prepare_primitive<NV>(A, i, V);
    uint32_t n = 0, steps = 0;
    int px, py;
    if (live && A.mode == SWR_DRAW_POINT) {
        if (on_target(a, V[0].x, V[0].y, px, py)) {
            if (EMIT)
                write_fragment<NV>(A, A.first[i].y, i, px, py, V[0]);
            n = 1;
        }
    } else if (live) {
        // Rasterizer::drawLineTemplate / computeVertexStep / stepVertex, Rasterizer.h:175-222
        int64_t adx = (int64_t)f2i(V[1].x) - (int64_t)f2i(V[0].x);
        int64_t ady = (int64_t)f2i(V[1].y) - (int64_t)f2i(V[0].y);
        adx = adx < 0 ? -adx : adx;
        ady = ady < 0 ? -ady : ady;
        const int64_t most = adx > ady ? adx : ady;
        if (most > SWR_MAX_LINE_STEPS) {
            atomicOr(&a.status[ST_ERROR], 4ull);
            live = false;
        } else {
            steps = (uint32_t)most;
            const float fs = (float)most;
            float *l = s_line + lane * ST;
            l[0] = V[0].x;
            l[1] = V[0].y;
            l[2] = V[0].z;
            l[3] = V[0].w;
            l[W + 0] = (V[1].x - V[0].x) / fs;
            l[W + 1] = (V[1].y - V[0].y) / fs;
            l[W + 2] = (V[1].z - V[0].z) / fs;
            l[W + 3] = (V[1].w - V[0].w) / fs;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                l[4 + k] = V[0].v[k];
                l[W + 4 + k] = (V[1].v[k] - V[0].v[k]) / fs;
            }
        }
    }
    const uint32_t pieces = (steps + LINE_PIECE - 1) / LINE_PIECE;
    const uint32_t incl = wave_incl(pieces);
    if (lane < LINES) {
        s_steps[lane] = steps;
        s_first[lane] = incl - pieces;
        s_done[lane] = 0u;  // fragments of the line's earlier pieces
    }
    const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);
    lds_sync();
    for (uint32_t p0 = 0; p0 < total; p0 += 64) {
        const uint32_t p = p0 + lane;
        const bool has = p < total;
        uint32_t lo = 0, hi = LINES;  // the last line with s_first <= p (it has pieces)
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_first[mid] <= p)
                lo = mid;
            else
                hi = mid;
        }
        const float *l = s_line + lo * ST;
        const uint32_t at = has ? (p - s_first[lo]) * LINE_PIECE : 0u;
        const uint32_t left = has ? s_steps[lo] - at : 0u;
        const uint32_t len = left < LINE_PIECE ? left : LINE_PIECE;
        const float sx = l[W + 0], sy = l[W + 1];
        const float x0 = has ? chain_add(l[0], sx, (int)at) : 0.0f;
        const float y0 = has ? chain_add(l[1], sy, (int)at) : 0.0f;
        uint32_t cnt = 0;
        {
            float x = x0, y = y0;
            for (uint32_t s = 0; s < len; ++s) {
                cnt += on_target(a, x, y, px, py) ? 1u : 0u;
                x += sx;
                y += sy;
            }
        }
        if (!EMIT) {
            if (cnt)
                atomicAdd(&s_done[lo], cnt);
            continue;
        }
        // the piece's first fragment: the line's, plus its earlier pieces' (in this round: the
        // lanes below with the same line)
        const uint32_t ex = wave_incl(cnt);
        const uint32_t head = s_first[lo] > p0 ? s_first[lo] - p0 : 0u;  // the line's first lane
        const uint32_t before = (uint32_t)__shfl((int)(ex - cnt), (int)head, 64);
        const uint32_t done = s_done[lo];
        lds_sync();  // every lane has read its line's count
        if (cnt)
            atomicAdd(&s_done[lo], cnt);
        lds_sync();
        if (!cnt)
            continue;
        const uint64_t li = base + lo;
        uint64_t f = (uint64_t)A.first[li].y + done + (ex - cnt - before);
        LVert<NV> v;
        v.x = x0;
        v.y = y0;
        v.z = A.iz ? chain_add(l[2], l[W + 2], (int)at) : l[2];
        v.w = A.iw ? chain_add(l[3], l[W + 3], (int)at) : l[3];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const bool stepped =
                k < a.lay.na ? (k < a.lay.set_na) : ((k - a.lay.na) < a.lay.set_np);
            v.v[k] = stepped ? chain_add(l[4 + k], l[W + 4 + k], (int)at) : l[4 + k];
        }
        for (uint32_t s = 0; s < len; ++s) {
            if (on_target(a, v.x, v.y, px, py)) {
                write_fragment<NV>(A, f, li, px, py, v);
                ++f;
            }
            v.x += sx;
            v.y += sy;
            if (A.iz)
                v.z += l[W + 2];
            if (A.iw)
                v.w += l[W + 3];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const bool stepped =
                    k < a.lay.na ? (k < a.lay.set_na) : ((k - a.lay.na) < a.lay.set_np);
                if (stepped)
                    v.v[k] += l[W + 4 + k];
            }
        }
    }
    if (!EMIT) {
        lds_sync();
        if (mine)
            n += s_done[lane];
        if (mine)
            A.count[i] = make_uint2(live ? 1u : 0u, n);
        // 64-bit totals per workgroup: the scan adds them up (a workgroup's
        // fit 32 bits, all of them need not)
        const unsigned long long frags = wave_sum(n);
        if (lane == 0)
            A.parts[group] = frags;
    }
}

__global__ void __launch_bounds__(256) k_lines_begin(LineArgs A)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ST_WORDS && i != ST_STICKY)
        A.g.status[i] = 0ull;
    for (uint64_t k = i; k < 2ull * A.g.tiles; k += (uint64_t)gridDim.x * blockDim.x)
        A.g.ranges[k] = 0u;
}

// ---- launchers ------------------------------------------------------------------------------
uint32_t lines_groups(uint64_t prims) { return (uint32_t)((prims + LINES - 1) / LINES); }

// A launch holds fewer than 2^32 threads, which 2^30 primitives, the most a draw takes, reach
// with 4 threads each: a second launch takes the workgroups from 2^25 on (an offset in every
// launch costs long lines 2%).
template <int NV, bool EMIT>
static void launch_walk(LineArgs A, hipStream_t s)
{
    const uint32_t n = lines_groups(A.prims), most = 1u << 25, first = n < most ? n : most;
    if (first)
        hipLaunchKernelGGL((k_lines_walk<NV, EMIT, false>), dim3(first), dim3(64), 0, s, A);
    A.group0 = first;
    if (n > first)
        hipLaunchKernelGGL((k_lines_walk<NV, EMIT, true>), dim3(n - first), dim3(64), 0, s, A);
}

hipError_t launch_lines_count(const LineArgs &A, hipStream_t s)
{
    const uint64_t clear = A.g.tiles * 2ull > ST_WORDS ? A.g.tiles * 2ull : ST_WORDS;
    const uint64_t cb = (clear + 255) / 256 < 4096 ? (clear + 255) / 256 : 4096;
    hipLaunchKernelGGL(k_lines_begin, dim3((uint32_t)cb), dim3(256), 0, s, A);
    launch_walk<0, false>(A, s);
    return hipGetLastError();
}

hipError_t launch_lines_emit(const LineArgs &A, hipStream_t s)
{
    switch (emit_class(A.g.lay.na + A.g.lay.np)) {
    case 0: launch_walk<0, true>(A, s); break;
    case 3: launch_walk<3, true>(A, s); break;
    case 5: launch_walk<5, true>(A, s); break;
    case 8: launch_walk<8, true>(A, s); break;
    default: launch_walk<32, true>(A, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_lines_raster(const swr_pixel_shader_desc &ps, const ParamLayout &L,
                               const RasterArgs &a, hipStream_t s)
{
    switch (ps.program) {
    case SWR_PS_COVERAGE: return launch_lr<ProgCoverage, 0, 0, 0, 0>(a, s);
    case SWR_PS_RGB: return launch_lr<ProgRGB, 0, 0, 3, 0>(a, s);
    case SWR_PS_DEPTH_CHECKER: return launch_lr<ProgDepthChecker, 1, 1, 3, 2>(a, s);
    case SWR_PS_VISIBILITY: return launch_lr<ProgVisibility, 1, 0, 0, 0>(a, s);
    case SWR_PS_HASH:
        return L.na == 4 ? launch_lr<ProgHash, 1, 1, 4, 4>(a, s)
                         : launch_lr<ProgHash, 1, 1, 16, 16>(a, s);
    case SWR_PS_LOG:
        return L.na == 4 ? launch_lr<ProgLog, 1, 1, 4, 4>(a, s)
                         : launch_lr<ProgLog, 1, 1, 16, 16>(a, s);
    case SWR_PS_MODULE:
        return (hipError_t)ps.module->launch_fragments(&a, s);
    default: return hipSuccess;
    }
}

}  // namespace swr
