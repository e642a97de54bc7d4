// swr_diff.hip — differentiable shading over a visibility buffer, forward and backward.
//
// The visibility draw (SWR_PS_VISIBILITY, one batched draw over every view) leaves per
// pixel the nearest input triangle and its depth.  Everything else is recomputed from it:
//
//   barycentrics   r = (X, Y, 1), the pixel centre in NDC; h_i = (x_i, y_i, w_i) the clip
//                  coordinates of the triangle's vertices.  D_i = r . (h_j x h_k) over the
//                  cyclic (i, j, k); b_i = D_i / (D_0 + D_1 + D_2): the perspective-correct
//                  weights (sum_i b_i h_i is parallel to r).
//   colour         C = sum_i b_i A_i (per channel), 0 on the background.
//   edge antialiasing
//                  for every pair of 4-neighbour pixels (p, q) showing different triangles:
//                  the front pixel f is the one with the smaller depth (background is
//                  farthest; ties go to the lower pixel index) and T its triangle.  Among
//                  T's edges that separate the two pixel centres (edge function >= 0 at f,
//                  < 0 at the other pixel o) take the first one crossed from f, at
//                  t = E(f) / (E(f) - E(o)) in [0, 1], and walk on across interior edges
//                  to the first silhouette edge the segment crosses (no neighbouring
//                  triangle across it, or the neighbour faces the other way).  The pixel
//                  whose half of the segment holds the crossing is blended with the other:
//                    t < 1/2: f += a (1/2 - t) (C_o - C_f);  else o += a (t - 1/2) (E - C_o)
//                  where E is the silhouette triangle's colour at the crossing point,
//                  with the axis weight a = ey^2 / (ex^2 + ey^2) for horizontal pairs and
//                  ex^2 / (ex^2 + ey^2) for vertical pairs, (ex, ey) the edge's direction on
//                  screen.  Each axis alone keeps the image continuous as an edge sweeps
//                  over a pixel centre, and the weights sum to one, so the sum does too.
//                  Blends use the colours before antialiasing and add up.
//
// Passes.  Forward: k_diff_interp (barycentrics, colour, image = colour, and the cheap part
// of every pair's decision; pairs that need the silhouette walk go to a queue),
// k_diff_march (one lane per queued pair: the walk, the stored decision, per-tile flags),
// k_diff_blend (only tiles with an active pair: the antialiasing added to the image).
// Backward: k_diff_bwd_interior (every pixel: its own triangle's interpolation under
// dL/dimage) and k_diff_bwd_edges (the active pairs: what the antialiasing adds),
// both reading the stored decisions; gradients reach the vertex attributes through b_i,
// the clip coordinates through D_i (barycentrics) and through t (the silhouette crossing),
// gathered in lists in LDS, summed and flushed with float atomics.  A backward whose buffers are
// not those of the last forward on the context takes decisions again itself
// (k_diff_backward).  The walk is queued because few pairs need it (about 1% on a
// 41k-vertex sphere at 512 x 512) and a wave that holds one waits on its chain of dependent
// loads with all 64 lanes.
//
// Precision.  D_i is a cancellation-prone quantity: for a small or grazing triangle the
// three clip vectors are nearly parallel, and fp32 loses up to 1e-4 of D.  The values
// (D, b, t and every derivative) are therefore evaluated in fp64 from the fp32 inputs.  That
// arithmetic with its loads is about half of the interior backward (136 of 240 us on 64 views of
// 512x512) and little of the other kernels, which wait on dependent loads.  The discrete choices
// of the antialiasing pass use fp32, so they are reproducible by a CPU restatement.
#include <cstring>
#include <vector>

#include "swr_common.h"
#include "swr_internal.h"

namespace swr {

struct DiffArgs {
    int V, W, H, N, T;
    int culled;    // every visible triangle faces the same way (the visibility draw culled)
    int tiles_x, tiles_per_view;  // 16x16-pixel tiles, one per workgroup
    float sx, sy;  // W/2, H/2: NDC -> window scale (viewport (0, 0, W, H))
    const float4 *clip;
    const int32_t *tris;
    const int32_t *adj;
    const float *attr;
    const uint32_t *ids;
    const float *depth;
    float *bary;
    float *color;
    float *image;
    const float *gimage;  // dL/dimage, or the target image T when l2_target
    int l2_target;        // dL/dimage = image - T
    float *gclip;
    float *gattr;  // per-view partial attribute gradients [V][N][C], summed afterwards
    float *gattr_out;
    // antialiasing decisions of the forward pass, two pairs per pixel (to the right, below):
    // flags (PairLds::flags | edge << 4) and {crossing t, triangle}; reused by the backward
    uint8_t *pflag;
    int2 *pdata;
    uint32_t *tflag;   // per (view, tile): bit 0 some pair of the tile's pixels is active,
                       // bit 1 some pair to the right of its last column, bit 2 some pair
                       // below its last row
    // per (view, tile) b: the pairs that need the silhouette walk (pair index 2 * pixel +
    // dir) at queue[b * 512 ..) with qcnt[b] entries; and per region of `region_tiles`
    // consecutive tiles r: its active pairs (the blend pass appends them) at
    // elist[r * region_tiles * 512 ..) with ecnt[r] entries
    uint32_t *queue, *qcnt;
    uint32_t *elist, *ecnt;
    uint32_t region_tiles;
    int row_keys;  // 1: clip rows fit the int keys of the edge backward's table
    int pairs;     // 1: store the decisions, 2: load the stored ones, 0: take them again
    // several meshes (null for one): per view, the clip row of global vertex g is
    // vrow[view] + g and visibility id k names triangle vtri[view].x + k - 1 (k <= .y);
    // per scene (S of them), its first vertex, first view and first row
    const long long *vrow;
    const int2 *vtri;
    const int *svert, *sview;
    int S;
};

// dL/d(image channel c of pixel i): the caller's image gradient, or image - target for the
// fused L2 loss (SWR_DIFF_L2_TARGET), formed in the same fp32 operation torch would use.
__device__ inline float grad_image(const DiffArgs &d, size_t i, int C, int c)
{
    const float g = d.gimage[i * C + c];
    return d.l2_target ? d.image[i * C + c] - g : g;
}

// Clip / gradient row of vertex v (global number) as seen by `view`.
__device__ inline size_t crow(const DiffArgs &d, int view, int v)
{
    return d.vrow ? (size_t)(d.vrow[view] + v) : (size_t)view * d.N + v;
}

// Triangle named by visibility id `id` in `view`; -1 for the background (0) or an id past
// the view's triangles.
__device__ inline int id_tri(const DiffArgs &d, int view, uint32_t id)
{
    if (!d.vtri)
        return (id == 0 || id > (uint32_t)d.T) ? -1 : (int)id - 1;
    const int2 t = d.vtri[view];
    return (id == 0 || id > (uint32_t)t.y) ? -1 : t.x + (int)id - 1;
}

// Pixel of this thread: a workgroup of 256 threads covers one 16x16 tile of one view, so a
// wave (16x4 pixels) reads its neighbours, triangles and vertices from a small area.
struct PixelIdx {
    int view, px, py;
    int tile;  // (view, tile) index of the workgroup
    size_t i;
};

// Workgroup b runs on XCD b % 8 (round-robin dispatch).  Renumber so that each XCD works
// through one contiguous run of (view, tile) blocks: the views an XCD is working on at any
// moment have their vertex data and gradient slices in that XCD's L2, where the float
// atomics of the backward pass resolve.
__device__ inline int xcd_order(unsigned b, unsigned n)
{
    const unsigned q = n / 8u, r = n % 8u, x = b % 8u, i = b / 8u;
    return (int)(x * q + (x < r ? x : r) + i);
}

__device__ inline bool pixel_of_thread(const DiffArgs &d, PixelIdx &q)
{
    const int b = xcd_order(blockIdx.x, gridDim.x);
    q.tile = b;
    q.view = b / d.tiles_per_view;
    const int t = b - q.view * d.tiles_per_view;
    const int ty = t / d.tiles_x, tx = t - ty * d.tiles_x;
    q.px = tx * 16 + (int)(threadIdx.x & 15);
    q.py = ty * 16 + (int)(threadIdx.x >> 4);
    if (q.px >= d.W || q.py >= d.H)
        return false;
    q.i = ((size_t)q.view * d.H + q.py) * d.W + q.px;
    return true;
}

// clip (x, y, w) of a vertex, in fp64
struct H3 {
    double x, y, w;
};

__device__ inline H3 cross3(const H3 &a, const H3 &b)
{
    return {a.y * b.w - a.w * b.y, a.w * b.x - a.x * b.w, a.x * b.y - a.y * b.x};
}

__device__ inline double dot3(const H3 &a, const H3 &b) { return a.x * b.x + a.y * b.y + a.w * b.w; }

__device__ inline H3 load_h(const DiffArgs &d, int view, int v)
{
    const float4 c = d.clip[crow(d, view, v)];
    return {(double)c.x, (double)c.y, (double)c.w};
}

__device__ inline H3 pixel_ray(const DiffArgs &d, int px, int py)
{
    const double X = 2.0 * ((double)px + 0.5) / (double)d.W - 1.0;
    const double Y = 1.0 - 2.0 * ((double)py + 0.5) / (double)d.H;
    return {X, Y, 1.0};
}

// Window position of a clip-space vertex (w > 0): fp32 for decisions (tri_win), fp64 for
// values.

__device__ inline double2 to_win_d(const DiffArgs &d, const H3 &h)
{
    const double sx = 0.5 * d.W, sy = 0.5 * d.H;
    return make_double2(sx * (h.x / h.w) + sx, -sy * (h.y / h.w) + sy);
}

__device__ inline float edge_fn(float2 j, float2 k, float2 p)
{
    return (k.x - j.x) * (p.y - j.y) - (k.y - j.y) * (p.x - j.x);
}

__device__ inline double edge_d(double2 j, double2 k, double2 p)
{
    return (k.x - j.x) * (p.y - j.y) - (k.y - j.y) * (p.x - j.x);
}

// The active pairs' lists: one per EDGE_REGIONS-th of the tiles (a counter each: one for all
// tiles would serialise their atomics).
constexpr uint32_t EDGE_REGIONS = 256;

// One neighbour pair as the antialiasing pass sees it.
struct Pair {
    bool active;      // a silhouette edge crosses the segment between the centres
    bool p_blended;   // the blended pixel is p (else q)
    bool horiz;       // horizontal pair
    float tf, s;      // fp32 crossing (decisions), orientation of the triangle
    int tri, vj, vk;  // triangle and the edge's vertices
    int edge;         // the edge's index in the triangle (opposite vertex)
    int front_is_p;
};

// Values of an active pair in fp64: the crossing t and the axis weight a, with their
// derivatives with respect to the window positions of the edge's vertices j and k.
struct PairVal {
    double t, a;
    double2 tj, tk, aj, ak;
};

__device__ inline PairVal pair_val(const DiffArgs &d, int view, const Pair &pr, int px, int py,
                                   int qx, int qy)
{
    PairVal r;
    const double2 j = to_win_d(d, load_h(d, view, pr.vj)), k = to_win_d(d, load_h(d, view, pr.vk));
    const double2 P = make_double2(px + 0.5, py + 0.5), Qp = make_double2(qx + 0.5, qy + 0.5);
    const double2 F = pr.front_is_p ? P : Qp, Q = pr.front_is_p ? Qp : P;
    const double s = pr.s;
    const double ef = s * edge_d(j, k, F), eq = s * edge_d(j, k, Q);
    const double den = ef - eq;
    r.t = ef / den;
    const double dtf = -eq / (den * den), dtq = ef / (den * den);
    // edge(j, k, P) partials: d/dj = (k.y - P.y, P.x - k.x), d/dk = (P.y - j.y, j.x - P.x)
    r.tj = make_double2(s * (dtf * (k.y - F.y) + dtq * (k.y - Q.y)),
                        s * (dtf * (F.x - k.x) + dtq * (Q.x - k.x)));
    r.tk = make_double2(s * (dtf * (F.y - j.y) + dtq * (Q.y - j.y)),
                        s * (dtf * (j.x - F.x) + dtq * (j.x - Q.x)));
    // a = ey^2 / L2 (horizontal pair) or ex^2 / L2, L2 = ex^2 + ey^2, (ex, ey) = k - j
    const double ex = k.x - j.x, ey = k.y - j.y, L2 = ex * ex + ey * ey;
    const double wx = ey * ey / L2;
    const double dex = -2.0 * ex * ey * ey / (L2 * L2), dey = 2.0 * ey * ex * ex / (L2 * L2);
    const double sg = pr.horiz ? 1.0 : -1.0;  // d(1 - wx) = -d(wx)
    r.a = pr.horiz ? wx : 1.0 - wx;
    r.ak = make_double2(sg * dex, sg * dey);
    r.aj = make_double2(-sg * dex, -sg * dey);
    return r;
}

// Window positions of triangle t's vertices (fp32); false when a vertex has w <= 0.
__device__ inline bool tri_win(const DiffArgs &d, int view, int t, float2 *v, int *vid)
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
        vid[i] = d.tris[3 * t + i];
    bool front = true;  // the three vertices' loads leave together
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float4 h = d.clip[crow(d, view, vid[i])];
        front = front && h.w > 0.0f;
        v[i] = make_float2(d.sx * (h.x / h.w) + d.sx, -d.sy * (h.y / h.w) + d.sy);
    }
    return front;
}

constexpr int MARCH_STEPS = 8;

// The pair (p, q): start in the front pixel's triangle and walk along the segment from the
// front centre F to the other centre Q across interior edges (adjacent triangles facing the
// same way) until the segment leaves the mesh through a silhouette edge, ends inside a
// triangle (no crossing: inactive), or MARCH_STEPS triangles were visited (inactive).  The
// exit edge of a triangle is the one the segment crosses first while leaving its half-plane
// (edge value < 0 at Q and falling from F to Q).
// The cheap part of a pair's decision: false when no silhouette can separate p and q (same
// triangle, no front triangle, or two visible triangles of a culled draw sharing a vertex);
// otherwise the front pixel and its triangle, where the walk starts.
__device__ inline bool pair_start(const DiffArgs &d, int view, int px, int py, int qx, int qy,
                                  bool &pf_out, int &cur_out)
{
    const size_t base = (size_t)view * d.W * d.H;
    const size_t ip = base + (size_t)py * d.W + px, iq = base + (size_t)qy * d.W + qx;
    const uint32_t a = d.ids[ip], b = d.ids[iq];
    if (a == b)
        return false;
    bool pf;
    if (a == 0)
        pf = false;
    else if (b == 0)
        pf = true;
    else {
        const float dp = d.depth[ip], dq = d.depth[iq];
        pf = dp < dq || (dp == dq && ip < iq);
    }
    const int cur = id_tri(d, view, pf ? a : b);
    if (cur < 0)
        return false;
    if (d.culled && a != 0 && b != 0) {
        // two visible triangles of a culled draw that share a vertex both face the viewer:
        // no silhouette is taken to separate their pixels
        const int other = id_tri(d, view, pf ? b : a);
        if (other >= 0) {
            const int c0 = d.tris[3 * cur], c1 = d.tris[3 * cur + 1], c2 = d.tris[3 * cur + 2];
            const int o0 = d.tris[3 * other], o1 = d.tris[3 * other + 1],
                      o2 = d.tris[3 * other + 2];
            const bool share = c0 == o0 || c0 == o1 || c0 == o2 || c1 == o0 || c1 == o1 ||
                               c1 == o2 || c2 == o0 || c2 == o1 || c2 == o2;
            if (share)
                return false;
        }
    }
    pf_out = pf;
    cur_out = cur;
    return true;
}

__device__ inline Pair eval_pair(const DiffArgs &d, int view, int px, int py, int qx, int qy)
{
    Pair r;
    r.active = r.p_blended = r.horiz = false;
    r.tf = 0.0f;
    r.s = 1.0f;
    r.tri = r.vj = r.vk = r.edge = r.front_is_p = 0;
    bool pf;
    int cur;
    if (!pair_start(d, view, px, py, qx, qy, pf, cur))
        return r;
    const bool horiz = py == qy;
    const float2 F = pf ? make_float2(px + 0.5f, py + 0.5f) : make_float2(qx + 0.5f, qy + 0.5f);
    const float2 Q = pf ? make_float2(qx + 0.5f, qy + 0.5f) : make_float2(px + 0.5f, py + 0.5f);
    float2 v[3];
    int vid[3];
    if (!tri_win(d, view, cur, v, vid))
        return r;
    float area = edge_fn(v[0], v[1], v[2]);
    if (!(area != 0.0f))
        return r;
    int from = -1;
    int ad[3];  // the triangle's neighbours, loaded beside its vertex numbers: a step then waits
                // for one load of these and one of the vertices
#pragma unroll
    for (int e = 0; e < 3; ++e)
        ad[e] = d.adj[3 * cur + e];
    for (int step = 0; step < MARCH_STEPS; ++step) {
        const float s = area > 0.0f ? 1.0f : -1.0f;
        float best = 2.0f;
        int be = -1;
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            if (e == from)
                continue;
            const int j = (e + 1) % 3, k = (e + 2) % 3;
            const float ef = s * edge_fn(v[j], v[k], F), eq = s * edge_fn(v[j], v[k], Q);
            if (eq < 0.0f && ef > eq) {
                const float tt = ef / (ef - eq);
                if (tt < best) {
                    best = tt;
                    be = e;
                }
            }
        }
        if (be < 0)
            return r;  // the segment ends inside this triangle
        const int n = be == 0 ? ad[0] : (be == 1 ? ad[1] : ad[2]);
        float2 nv[3];
        int nvid[3], nad[3] = {-1, -1, -1};
        float an = 0.0f;
        bool interior = false;
        if (n >= 0 && n < d.T) {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                nad[e] = d.adj[3 * n + e];
        }
        if (n >= 0 && n < d.T && tri_win(d, view, n, nv, nvid)) {
            an = edge_fn(nv[0], nv[1], nv[2]);
            interior = an != 0.0f && ((an > 0.0f) == (area > 0.0f));
        }
        if (!interior) {
            // vertices j = be + 1 and k = be + 2 of the triangle, by selects (a runtime index
            // would put the arrays in memory)
            const float2 vj = be == 0 ? v[1] : (be == 1 ? v[2] : v[0]);
            const float2 vk = be == 0 ? v[2] : (be == 1 ? v[0] : v[1]);
            if (vk.x == vj.x && vk.y == vj.y)
                return r;  // a degenerate edge has no direction
            r.active = true;
            r.horiz = horiz;
            r.tf = best;
            r.s = s;
            r.tri = cur;
            r.edge = be;
            r.vj = be == 0 ? vid[1] : (be == 1 ? vid[2] : vid[0]);
            r.vk = be == 0 ? vid[2] : (be == 1 ? vid[0] : vid[1]);
            r.front_is_p = pf;
            r.p_blended = (best < 0.5f) == pf;
            return r;
        }
        int fe = -1;
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (nad[e] == cur)
                fe = e;
        if (fe < 0)
            return r;
        cur = n;
        from = fe;
        area = an;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            v[i] = nv[i];
            vid[i] = nvid[i];
            ad[i] = nad[i];
        }
    }
    return r;
}

// Perspective-correct barycentrics of triangle t at the centre of pixel (px, py), in fp64
// (the pixel may lie outside the triangle: the antialiasing extrapolates).  False when the
// three clip vectors are linearly dependent there (S == 0).
struct Bary {
    int v[3];
    H3 h[3];
    H3 r;
    double b[3], S, inv;  // inv = 1 / S: one fp64 division per pixel, products after it
};

__device__ inline bool bary_at_ray(const DiffArgs &d, int view, int t, const H3 &r, Bary &B)
{
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        B.v[m] = d.tris[3 * t + m];
        B.h[m] = load_h(d, view, B.v[m]);
    }
    B.r = r;
    const double D0 = dot3(B.r, cross3(B.h[1], B.h[2])), D1 = dot3(B.r, cross3(B.h[2], B.h[0])),
                 D2 = dot3(B.r, cross3(B.h[0], B.h[1]));
    B.S = D0 + D1 + D2;
    if (B.S == 0.0)
        return false;
    B.inv = 1.0 / B.S;
    B.b[0] = D0 * B.inv;
    B.b[1] = D1 * B.inv;
    B.b[2] = D2 * B.inv;
    return true;
}

__device__ inline bool bary_at(const DiffArgs &d, int view, int t, int px, int py, Bary &B)
{
    return bary_at_ray(d, view, t, pixel_ray(d, px, py), B);
}

// The point where the pair's segment crosses the silhouette edge, as a ray (NDC, 1), and
// its derivative with respect to t.
__device__ inline H3 crossing_ray(const DiffArgs &d, const Pair &pr, double t, int px, int py,
                                  int qx, int qy, H3 &drdt)
{
    const double fx = (pr.front_is_p ? px : qx) + 0.5, fy = (pr.front_is_p ? py : qy) + 0.5;
    const double ox = (pr.front_is_p ? qx : px) + 0.5, oy = (pr.front_is_p ? qy : py) + 0.5;
    const double wx = fx + t * (ox - fx), wy = fy + t * (oy - fy);
    drdt = {2.0 * (ox - fx) / d.W, -2.0 * (oy - fy) / d.H, 0.0};
    return {2.0 * wx / d.W - 1.0, 1.0 - 2.0 * wy / d.H, 1.0};
}

// d(colour at ray r)/d(r) . dr, per channel, for barycentrics B: b_m = D_m / S with
// dD_m/dr = h_j x h_k.
template <int C>
__device__ inline void bary_color_dr(const DiffArgs &d, const Bary &B, const H3 &dr, double *out)
{
    const H3 c0 = cross3(B.h[1], B.h[2]), c1 = cross3(B.h[2], B.h[0]), c2 = cross3(B.h[0], B.h[1]);
    const double e0 = dot3(c0, dr), e1 = dot3(c1, dr), e2 = dot3(c2, dr);
    const double es = e0 + e1 + e2;
    const double db[3] = {(e0 - B.b[0] * es) * B.inv, (e1 - B.b[1] * es) * B.inv,
                          (e2 - B.b[2] * es) * B.inv};
#pragma unroll
    for (int c = 0; c < C; ++c)
        out[c] = db[0] * d.attr[(size_t)B.v[0] * C + c] + db[1] * d.attr[(size_t)B.v[1] * C + c] +
                 db[2] * d.attr[(size_t)B.v[2] * C + c];
}

template <int C>
__device__ inline void bary_color(const DiffArgs &d, const Bary &B, double *col)
{
#pragma unroll
    for (int c = 0; c < C; ++c)
        col[c] = B.b[0] * d.attr[(size_t)B.v[0] * C + c] + B.b[1] * d.attr[(size_t)B.v[1] * C + c] +
                 B.b[2] * d.attr[(size_t)B.v[2] * C + c];
}

// The colour interp_pixel gives pixel (px, py) of `view` before antialiasing (the attributes
// at its barycentrics, 0 on the background, rounded to fp32): read from the colour buffer
// when the caller keeps one, else computed again by the same operations (same bits).
template <int C>
__device__ inline void pixel_color(const DiffArgs &d, int view, size_t i, int px, int py,
                                   double *out)
{
    if (d.color) {
#pragma unroll
        for (int c = 0; c < C; ++c)
            out[c] = d.color[i * C + c];
        return;
    }
    double col[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        col[c] = 0.0;
    Bary B;
    const int tri = id_tri(d, view, d.ids[i]);
    if (tri >= 0 && bary_at(d, view, tri, px, py, B))
        bary_color<C>(d, B, col);
#pragma unroll
    for (int c = 0; c < C; ++c)
        out[c] = (double)(float)col[c];
}

// Gradient accumulation of one workgroup (one 16x16 tile of one view): an open-addressing
// table in LDS keyed by vertex, flushed to global memory once per distinct vertex.  The
// pixels of a tile touch a few dozen vertices, so this replaces most global float atomics
// (which serialise on shared vertices) by LDS atomics.  A vertex that finds no slot after
// ACC_PROBES probes goes straight to global memory.  Slots are never freed, so a vertex that
// got a slot is found again within the same probes.
constexpr int ACC_SLOTS = 256;   // power of two
constexpr int ACC_PROBES = 32;   // one 16x16 tile: a few dozen vertices, the table never fills
constexpr int ACC_VALS = 8;      // at most: clip x, y, w, attributes 0..4
// values per slot with C attribute channels: clip x, y, w and the C attributes
template <int C> constexpr int acc_vals() { return 3 + C; }
// words of a slot: odd, so that the slots' values spread over the LDS banks
template <int C> constexpr int acc_stride() { return acc_vals<C>() * 4 + 1; }
// Each value is kept in four copies, picked by the pixel's (x, y) parity: the pixels of one
// triangle are neighbours, and four copies cut the lanes of a wave that add into the same
// LDS word (which serialise) about four times.  The flush sums the copies.
constexpr int ACC_COPIES = 4;  // (acc_stride counts on it)

__device__ inline int acc_copy() { return (int)((threadIdx.x & 1u) | ((threadIdx.x >> 3) & 2u)); }

struct VertexAcc {
    int *key;
    float *val;
};

__device__ inline int acc_slot(const VertexAcc &A, int v)
{
    const unsigned h = ((unsigned)v * 2654435761u) >> 24;  // 8 bits: ACC_SLOTS
#pragma unroll 1
    for (int probe = 0; probe < ACC_PROBES; ++probe) {
        const int sl = (int)((h + (unsigned)probe) & (ACC_SLOTS - 1));
        const int k = __atomic_load_n(&A.key[sl], __ATOMIC_RELAXED);
        if (k == v)
            return sl;
        if (k == -1) {
            const int old = atomicCAS(&A.key[sl], -1, v);
            if (old == -1 || old == v)
                return sl;
        }
    }
    return -1;
}

template <int C>
__device__ inline void acc_clip(const DiffArgs &d, const VertexAcc &A, int view, int v, float gx,
                                float gy, float gw)
{
    const int sl = acc_slot(A, v);
    if (sl >= 0) {
        float *x = &A.val[sl * acc_stride<C>() + acc_copy()];
        atomicAdd(x + 0 * ACC_COPIES, gx);
        atomicAdd(x + 1 * ACC_COPIES, gy);
        atomicAdd(x + 2 * ACC_COPIES, gw);
    } else {
        float *g = d.gclip + crow(d, view, v) * 4;
        atomicAdd(g + 0, gx);
        atomicAdd(g + 1, gy);
        atomicAdd(g + 3, gw);
    }
}

// clip and attribute gradients of one vertex with a single table lookup
template <int C>
__device__ inline void acc_vertex(const DiffArgs &d, const VertexAcc &A, int view, int v,
                                  float gx, float gy, float gw, const float *ga)
{
    const int sl = acc_slot(A, v);
    if (sl >= 0) {
        float *x = &A.val[sl * acc_stride<C>() + acc_copy()];
        atomicAdd(x + 0 * ACC_COPIES, gx);
        atomicAdd(x + 1 * ACC_COPIES, gy);
        atomicAdd(x + 2 * ACC_COPIES, gw);
#pragma unroll
        for (int c = 0; c < C; ++c)
            atomicAdd(x + (3 + c) * ACC_COPIES, ga[c]);
    } else {
        float *g = d.gclip + crow(d, view, v) * 4;
        atomicAdd(g + 0, gx);
        atomicAdd(g + 1, gy);
        atomicAdd(g + 3, gw);
#pragma unroll
        for (int c = 0; c < C; ++c)
            atomicAdd(d.gattr + crow(d, view, v) * C + c, ga[c]);
    }
}

// The slots of the three vertices of one pixel's triangle: the first probes of the three
// lookups are issued together (one LDS round trip instead of three in the common case that
// the vertex already has its slot), the rest probe on.
__device__ inline void acc_find3(const VertexAcc &A, const int (&v)[3], int (&sl)[3])
{
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const int h = (int)((((unsigned)v[m] * 2654435761u) >> 24) & (ACC_SLOTS - 1));
        sl[m] = __atomic_load_n(&A.key[h], __ATOMIC_RELAXED) == v[m] ? h : -1;
    }
#pragma unroll
    for (int m = 0; m < 3; ++m)
        if (sl[m] < 0)
            sl[m] = acc_slot(A, v[m]);
}

template <int C>
__device__ inline void acc_flush(const DiffArgs &d, const VertexAcc &A, int view)
{
    for (int sl = threadIdx.x; sl < ACC_SLOTS; sl += blockDim.x) {
        const int v = A.key[sl];
        if (v < 0)
            continue;
        float x[ACC_VALS];
#pragma unroll
        for (int k = 0; k < acc_vals<C>(); ++k) {
            const float *q = &A.val[sl * acc_stride<C>() + k * ACC_COPIES];
            x[k] = (q[0] + q[1]) + (q[2] + q[3]);
        }
        float *g = d.gclip + crow(d, view, v) * 4;
        if (x[0] != 0.0f) atomicAdd(g + 0, x[0]);
        if (x[1] != 0.0f) atomicAdd(g + 1, x[1]);
        if (x[2] != 0.0f) atomicAdd(g + 3, x[2]);
#pragma unroll
        for (int c = 0; c < C; ++c)
            if (x[3 + c] != 0.0f)
                atomicAdd(d.gattr + crow(d, view, v) * C + c, x[3 + c]);
    }
}

// Backward of col = sum_m b_m A_m given dL/dcol: adds to the attributes and, through
// b_m = D_m / S with D_m = r . (h_j x h_k), to the clip coordinates of the three vertices.
// The gradients bary_backward accumulates, per vertex m: {clip x, y, w, attribute 0..C).
template <int C>
__device__ inline void bary_grads(const DiffArgs &d, const Bary &B, const double *gcol,
                                  float (&out)[3][3 + C])
{
    double u[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        u[m] = 0.0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            u[m] += gcol[c] * d.attr[(size_t)B.v[m] * C + c];
            out[m][3 + c] = (float)(B.b[m] * gcol[c]);
        }
    }
    const double ub = u[0] * B.b[0] + u[1] * B.b[1] + u[2] * B.b[2];
    H3 g[3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const double gD = (u[m] - ub) * B.inv;
        const int j = (m + 1) % 3, k = (m + 2) % 3;
        // dD_m/dh_j = h_k x r, dD_m/dh_k = r x h_j
        const H3 dj = cross3(B.h[k], B.r), dk = cross3(B.r, B.h[j]);
        g[j].x += gD * dj.x;
        g[j].y += gD * dj.y;
        g[j].w += gD * dj.w;
        g[k].x += gD * dk.x;
        g[k].y += gD * dk.y;
        g[k].w += gD * dk.w;
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        out[m][0] = (float)g[m].x;
        out[m][1] = (float)g[m].y;
        out[m][2] = (float)g[m].w;
    }
}

template <int C>
__device__ inline void bary_backward(const DiffArgs &d, const VertexAcc &A, int view,
                                     const Bary &B, const double *gcol)
{
    float g[3][3 + C];
    bary_grads<C>(d, B, gcol, g);
#pragma unroll
    for (int m = 0; m < 3; ++m)
        acc_vertex<C>(d, A, view, B.v[m], g[m][0], g[m][1], g[m][2], &g[m][3]);
}

// Up to two values per thread into the workgroup's own segment `seg`; thread 0 writes the
// segment's length to *cnt.  Every thread of the workgroup calls it.  (A list shared by all
// workgroups needs a global counter, whose atomics serialise.)
__device__ inline void tile_append2(uint32_t *seg, uint32_t *cnt, bool t0, uint32_t v0, bool t1,
                                    uint32_t v1)
{
    __shared__ uint32_t s_n;
    const unsigned lane = threadIdx.x & 63u;
    if (threadIdx.x == 0)
        s_n = 0;
    __syncthreads();
    const unsigned long long m0 = __ballot(t0), m1 = __ballot(t1);
    const uint32_t n = (uint32_t)(__popcll(m0) + __popcll(m1));
    uint32_t base = 0;
    if (lane == 0 && n)
        base = atomicAdd(&s_n, n);
    base = __shfl(base, 0, 64);
    const unsigned long long below = (1ull << lane) - 1ull;
    if (t0)
        seg[base + (uint32_t)__popcll(m0 & below)] = v0;
    if (t1)
        seg[base + (uint32_t)__popcll(m0) + (uint32_t)__popcll(m1 & below)] = v1;
    __syncthreads();
    if (threadIdx.x == 0)
        *cnt = s_n;
}

template <int C>
__device__ inline void interp_pixel(const DiffArgs &d, const PixelIdx &pi, bool *walk)
{
    const size_t i = pi.i;
    const int view = pi.view, px = pi.px, py = pi.py;
    const uint32_t id = d.ids[i];
    double col[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        col[c] = 0.0;
    float2 bb = make_float2(0.0f, 0.0f);
    Bary B;
    const int tri = id_tri(d, view, id);
    if (tri >= 0 && bary_at(d, view, tri, px, py, B)) {
        bary_color<C>(d, B, col);
        bb = make_float2((float)B.b[0], (float)B.b[1]);
    }
    reinterpret_cast<float2 *>(d.bary)[i] = bb;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if (d.color)
            d.color[i * C + c] = (float)col[c];
        d.image[i * C + c] = (float)col[c];  // the blend pass adds the antialiasing
    }
    if (threadIdx.x == 0) {
        d.tflag[pi.tile] = 0u;
        if (pi.tile < (int)EDGE_REGIONS)
            d.ecnt[pi.tile] = 0u;  // the blend pass adds to it
    }
    // this pixel's two pairs (to the right, below): decided here unless a silhouette walk
    // is needed
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
        const int qx = px + (dir == 0), qy = py + (dir == 1);
        bool pf;
        int cur;
        walk[dir] = qx < d.W && qy < d.H && pair_start(d, view, px, py, qx, qy, pf, cur);
    }
    reinterpret_cast<uint16_t *>(d.pflag)[i] = 0;
}

template <int C>
__global__ void __launch_bounds__(256) k_diff_interp(DiffArgs d)
{
    PixelIdx pi;
    bool walk[2] = {false, false};
    if (pixel_of_thread(d, pi))
        interp_pixel<C>(d, pi, walk);
    // the pairs that need a silhouette walk, queued for k_diff_march
    const uint32_t k0 = (walk[0] || walk[1]) ? (uint32_t)(2 * pi.i) : 0u;
    tile_append2(d.queue + (size_t)pi.tile * 512, d.qcnt + pi.tile, walk[0], k0, walk[1], k0 + 1u);
}


__device__ inline bool neighbour(const DiffArgs &d, int px, int py, int k, int &qx, int &qy)
{
    qx = px + (k == 0 ? 1 : (k == 1 ? -1 : 0));
    qy = py + (k == 2 ? 1 : (k == 3 ? -1 : 0));
    return qx >= 0 && qx < d.W && qy >= 0 && qy < d.H;
}

// ---- pair decisions shared by a tile -------------------------------------------------------
// Each pair of neighbouring pixels is evaluated once per 16x16 tile: thread (lx, ly) takes the
// pair to its right and the pair below it, the tile's first column and row also the pairs
// across the tile's left and top border.  h[ly][lx + 1] holds the pair (lx, ly)-(lx + 1, ly),
// v[ly + 1][lx] the pair (lx, ly)-(lx, ly + 1), both seen from the left / upper pixel; the
// other pixel reads it with the roles swapped.
struct PairLds {
    int flags;  // 1 active, 2 first pixel blended, 4 first pixel in front, 8 s < 0,
                // bits 4-5 the edge index
    float tf;
    int tri, vj, vk;
};

// Stored form of a pair: the flags byte, and {t, triangle} when active; the edge's vertices
// are re-read from the triangle on load.
__device__ inline void store_pair(const DiffArgs &d, size_t k, const PairLds &x)
{
    d.pflag[k] = (uint8_t)x.flags;
    if (x.flags & 1)
        d.pdata[k] = make_int2(__float_as_int(x.tf), x.tri);
}

__device__ inline PairLds load_pair(const DiffArgs &d, size_t k)
{
    PairLds x;
    const int f = d.pflag[k];
    x.flags = f;
    if (f & 1) {
        const int2 q = d.pdata[k];
        const int e = f >> 4;
        x.tf = __int_as_float(q.x);
        x.tri = q.y;
        x.vj = d.tris[3 * x.tri + (e + 1) % 3];
        x.vk = d.tris[3 * x.tri + (e + 2) % 3];
    }
    return x;
}

__device__ inline PairLds pack_pair(const Pair &p)
{
    PairLds x;
    x.flags = (p.active ? 1 | (p.edge << 4) : 0) | (p.p_blended ? 2 : 0) |
              (p.front_is_p ? 4 : 0) | (p.s < 0.0f ? 8 : 0);
    x.tf = p.tf;
    x.tri = p.tri;
    x.vj = p.vj;
    x.vk = p.vk;
    return x;
}

__device__ inline Pair unpack_pair(const PairLds &x, bool swap, bool horiz)
{
    Pair p;
    p.active = x.flags & 1;
    p.p_blended = ((x.flags & 2) != 0) != swap;
    p.front_is_p = ((x.flags & 4) != 0) != swap;
    p.s = (x.flags & 8) ? -1.0f : 1.0f;
    p.tf = x.tf;
    p.tri = x.tri;
    p.vj = x.vj;
    p.vk = x.vk;
    p.horiz = horiz;
    return p;
}



// A workgroup's share of per-tile segments: TILES consecutive tiles, their lengths scanned
// into s_off (s_off[k] = entries before tile k, s_off[TILES] = all), so the workgroup's threads
// take the entries densely, one each.
template <int TILES>
__device__ inline void group_segments(const uint32_t *cnt, uint32_t tiles, uint32_t t0,
                                      uint32_t *s_off)
{
    static_assert(TILES <= 64, "a tile per lane of the first wave");
    if (threadIdx.x < 64) {
        const uint32_t lane = threadIdx.x;
        const uint32_t v =
            wave_incl(lane < TILES && t0 + lane < tiles ? cnt[t0 + lane] : 0u);
        if (lane < TILES)
            s_off[lane + 1] = v;
        if (lane == 0)
            s_off[0] = 0;
    }
    __syncthreads();
}

// The tile (within the group) of entry j: the largest k with s_off[k] <= j.
template <int TILES>
__device__ inline uint32_t group_tile(const uint32_t *s_off, uint32_t j)
{
    uint32_t lo = 0, hi = TILES;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_off[mid] <= j)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// The queued pairs, one lane each: the silhouette walk, the stored decision, and the tile
// flags of active pairs.  A walk is a chain of dependent loads (adjacency, then the next
// triangle's vertices), so the kernel is latency-bound and wants every queued pair in flight
// at once: a silhouette fills a tile's queue, so 256 lanes take 8 tiles.  64 views of 512x512:
// 183 us with 1024 lanes per 64 tiles (a compute unit holds one such workgroup), 351 us with
// 64 lanes per 8 tiles (several passes), 109 us now; one 256x256 view 30 -> 17 us.
constexpr int MARCH_TILES = 8, MARCH_THREADS = 256;

__global__ void __launch_bounds__(MARCH_THREADS) k_diff_march(DiffArgs d)
{
    __shared__ uint32_t s_off[MARCH_TILES + 1];
    const uint32_t tiles = (uint32_t)(d.tiles_per_view * d.V), t0 = blockIdx.x * MARCH_TILES;
    group_segments<MARCH_TILES>(d.qcnt, tiles, t0, s_off);
    const uint32_t n = s_off[MARCH_TILES];
    const size_t HW = (size_t)d.W * d.H;
    for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) {
        const uint32_t t = group_tile<MARCH_TILES>(s_off, j);
        const uint32_t k = d.queue[(size_t)(t0 + t) * 512 + (j - s_off[t])];
        const size_t i = k >> 1;
        const int dir = (int)(k & 1u);
        const int view = (int)(i / HW);
        const size_t rem = i - (size_t)view * HW;
        const int py = (int)(rem / (size_t)d.W), px = (int)(rem - (size_t)py * d.W);
        const Pair pr = eval_pair(d, view, px, py, px + (dir == 0), py + (dir == 1));
        store_pair(d, k, pack_pair(pr));
        if (pr.active) {
            const int tx = px >> 4, ty = py >> 4;
            const uint32_t bits = 1u | (dir == 0 && (px & 15) == 15 ? 2u : 0u) |
                                  (dir == 1 && (py & 15) == 15 ? 4u : 0u);
            atomicOr(&d.tflag[(size_t)view * d.tiles_per_view + ty * d.tiles_x + tx], bits);
        }
    }
}

// Whether (view, tile) b has an active pair: one of its pixels' own pairs, or a pair across
// its left or top border (owned by the neighbouring tile's last column or row).
__device__ inline bool tile_has_pairs(const DiffArgs &d, int b)
{
    const int t = b % d.tiles_per_view;
    const int tx = t % d.tiles_x, ty = t / d.tiles_x;
    uint32_t f = d.tflag[b] & 1u;
    if (tx > 0)
        f |= d.tflag[b - 1] & 2u;
    if (ty > 0)
        f |= d.tflag[b - d.tiles_x] & 4u;
    return f != 0;
}

constexpr int TP_H = 16 * 17, TP_V = 17 * 16;

__device__ inline PairLds eval_packed(const DiffArgs &d, int view, int ax, int ay, int bx, int by)
{
    if (ax < 0 || ay < 0 || bx >= d.W || by >= d.H || ax >= d.W || ay >= d.H) {
        PairLds x;
        x.flags = 0;
        return x;
    }
    return pack_pair(eval_pair(d, view, ax, ay, bx, by));
}

// Fills the tile's pair table; every thread of the workgroup calls it, then a barrier.
__device__ inline void tile_pairs(const DiffArgs &d, const PixelIdx &pi, PairLds *h, PairLds *v)
{
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int px = pi.px, py = pi.py, view = pi.view;
    h[ly * 17 + lx + 1] = eval_packed(d, view, px, py, px + 1, py);
    v[(ly + 1) * 16 + lx] = eval_packed(d, view, px, py, px, py + 1);
    if (lx == 0)
        h[ly * 17] = eval_packed(d, view, px - 1, py, px, py);
    if (ly == 0)
        v[lx] = eval_packed(d, view, px, py - 1, px, py);
}

// The pair between this thread's pixel and neighbour k (0 right, 1 left, 2 below, 3 above).
__device__ inline Pair tile_pair(const PairLds *h, const PairLds *v, int k);

// A pixel's four pairs from the workgroup's LDS table.
struct TilePairs {
    const PairLds *h, *v;
    __device__ Pair get(int k) const { return tile_pair(h, v, k); }
};
__device__ inline Pair tile_pair(const PairLds *h, const PairLds *v, int k)
{
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    switch (k) {
    case 0: return unpack_pair(h[ly * 17 + lx + 1], false, true);
    case 1: return unpack_pair(h[ly * 17 + lx], true, true);
    case 2: return unpack_pair(v[(ly + 1) * 16 + lx], false, false);
    default: return unpack_pair(v[ly * 16 + lx], true, false);
    }
}

// The blend a pixel receives from one active pair where it is the blended pixel:
//   front pixel (t < 1/2):  + a (1/2 - t) (C_q - C_p)
//   other pixel (t >= 1/2): + a (t - 1/2) (E - C_p), E = the silhouette triangle's colour
//                           where the segment crosses the edge.  As the edge sweeps onto
//                           this pixel's centre E becomes the colour the pixel then shows,
//                           so the image stays continuous; on the edge, E is a convex mix of
//                           the edge's endpoint colours, so it stays bounded.
// One lane per (blended pixel, pair), packed over the tile: about one pixel in ten of a tile on a
// silhouette receives a blend, so a lane per pixel going through its four pairs leaves most lanes
// waiting for a chain of fp64 work and dependent loads.  Both kinds of source colour go through
// the same instructions (a triangle at a ray).  The values reach their pixel through LDS, which
// adds them in the order of its pairs.  8 heightfields in 2 views of 768x768: 217 -> 94 us;
// 64 views of a sphere at 512x512: 78 -> 54 us.
template <int C>
__global__ void __launch_bounds__(256) k_diff_blend(DiffArgs d)
{
    __shared__ uint32_t s_items[4], s_own[4], s_base;
    __shared__ uint16_t s_item[4 * 256];
    __shared__ double s_add[C * 256];
    const int b = xcd_order(blockIdx.x, gridDim.x);
    if (!tile_has_pairs(d, b))
        return;  // the image is the colour here (uniform over the workgroup)
    const size_t HW = (size_t)d.W * d.H;
    PixelIdx pi;
    const bool valid = pixel_of_thread(d, pi);
    const size_t i = pi.i;
    const int view = pi.view;
    // the flags of the pixel's pairs as neighbour() numbers them
    uint32_t f[4] = {0u, 0u, 0u, 0u};
    if (valid) {
        const uint32_t own = reinterpret_cast<const uint16_t *>(d.pflag)[i];
        f[0] = own & 0xFFu;
        f[2] = own >> 8;
        if (pi.px > 0)
            f[1] = d.pflag[2 * (i - 1)];
        if (pi.py > 0)
            f[3] = d.pflag[2 * (i - d.W) + 1];
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    uint32_t before = 0, total = 0;  // items of the wave's lower lanes, of the wave
    bool mine[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        // flag 2 names the pair's left / upper pixel, the pair's second one for k = 1, 3
        mine[k] = (f[k] & 1u) && ((f[k] & 2u) != 0u) != ((k & 1) != 0);
        const unsigned long long m = __ballot(mine[k]);
        before += (uint32_t)__popcll(m & below);
        total += (uint32_t)__popcll(m);
    }
    const bool right = f[0] & 1u, down = f[2] & 1u;
    const unsigned long long mr = __ballot(right), md = __ballot(down);
    if (lane == 0) {
        s_items[wave] = total;
        s_own[wave] = (uint32_t)(__popcll(mr) + __popcll(md));
    }
    __syncthreads();
    uint32_t n = 0, nown = 0, own_at = 0;
    for (uint32_t w = 0; w < 4; ++w) {
        if (w == wave) {
            before += n;
            own_at = nown;
        }
        n += s_items[w];
        nown += s_own[w];
    }
    // the backward pass's antialiasing work is per active pair: list the pixels' own two, with
    // one global append per tile, spread over EDGE_REGIONS counters
    const uint32_t region = (uint32_t)b / d.region_tiles;
    if (threadIdx.x == 0 && nown)
        s_base = atomicAdd(d.ecnt + region, nown);
    uint32_t mycount = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (mine[k])
            s_item[before + mycount++] = (uint16_t)(threadIdx.x << 2 | k);
    __syncthreads();
    if (right || down) {
        uint32_t *to = d.elist + (size_t)region * d.region_tiles * 512 + s_base + own_at;
        if (right)
            to[__popcll(mr & below)] = (uint32_t)(2 * i);
        if (down)
            to[__popcll(mr) + __popcll(md & below)] = (uint32_t)(2 * i) + 1u;
    }
    double out[C];
    if (mycount)
#pragma unroll
        for (int c = 0; c < C; ++c)
            out[c] = d.image[i * C + c];  // the colour, until this thread stores the blend
    for (uint32_t r = 0; r < n; r += 256) {
        if (r)
            __syncthreads();  // the values of the items before are added
        if (r + threadIdx.x < n) {
            const uint32_t it = s_item[r + threadIdx.x];
            const int k = (int)(it & 3u), lx = (int)(it >> 2) & 15, ly = (int)(it >> 6);
            const int px = pi.px - (int)(threadIdx.x & 15) + lx;
            const int py = pi.py - (int)(threadIdx.x >> 4) + ly;
            int qx, qy;
            neighbour(d, px, py, k, qx, qy);
            const size_t ip = (size_t)view * HW + (size_t)py * d.W + px;
            const size_t iq = (size_t)view * HW + (size_t)qy * d.W + qx;
            const size_t at = 2 * ((k & 1) ? iq : ip) + (size_t)(k >> 1);
            const Pair pr = unpack_pair(load_pair(d, at), k & 1, k < 2);
            const PairVal pv = pair_val(d, view, pr, px, py, qx, qy);
            double src[C];
            bool known = true;
            if (pr.front_is_p && d.color) {
                pixel_color<C>(d, view, iq, qx, qy, src);
            } else {
                // the other pixel's colour before antialiasing, or the triangle's at the crossing
                int tri = pr.tri;
                H3 ray;
                if (pr.front_is_p) {
                    tri = id_tri(d, view, d.ids[iq]);
                    ray = pixel_ray(d, qx, qy);
                } else {
                    H3 drdt;
                    ray = crossing_ray(d, pr, pv.t, px, py, qx, qy, drdt);
                }
#pragma unroll
                for (int c = 0; c < C; ++c)
                    src[c] = 0.0;
                Bary B;
                if (tri >= 0 && bary_at_ray(d, view, tri, ray, B))
                    bary_color<C>(d, B, src);
                else
                    known = pr.front_is_p;  // the background's colour is 0
                if (pr.front_is_p)
#pragma unroll
                    for (int c = 0; c < C; ++c)
                        src[c] = (double)(float)src[c];
            }
            const double w = pv.a * (pr.front_is_p ? 0.5 - pv.t : pv.t - 0.5);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const double cp = d.image[ip * C + c];
                s_add[c * 256 + threadIdx.x] = known ? w * (src[c] - cp) : -0.0;
            }
        }
        __syncthreads();
        for (uint32_t j = 0; j < mycount; ++j) {
            const uint32_t at = before + j - r;  // past this round's items: a large number
            if (at < 256u)
#pragma unroll
                for (int c = 0; c < C; ++c)
                    out[c] += s_add[c * 256 + at];
        }
    }
    if (mycount)
#pragma unroll
        for (int c = 0; c < C; ++c)
            d.image[i * C + c] = (float)out[c];
}

// d(window x, y) of a clip-space vertex -> d(clip x, y, w), accumulated.
template <int C>
__device__ inline void scatter_window_grad(const DiffArgs &d, const VertexAcc &A, int view, int v,
                                           double gx, double gy)
{
    const H3 h = load_h(d, view, v);
    const double iw = 1.0 / h.w, sx = 0.5 * d.W, sy = 0.5 * d.H;
    acc_clip<C>(d, A, view, v, (float)(gx * sx * iw), (float)(-gy * sy * iw),
             (float)((-gx * sx * h.x + gy * sy * h.y) * iw * iw));
}

// A pixel's whole gradient: the interpolation of its own triangle and the antialiasing.
template <int C, class PS>
__device__ inline void backward_pixel(const DiffArgs &d, const VertexAcc &A, const PixelIdx &pi,
                                      const PS &pairs)
{
    const size_t HW = (size_t)d.W * d.H;
    const size_t i = pi.i;
    const int view = pi.view, px = pi.px, py = pi.py;
    double gp[C], gc[C], cp[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        gp[c] = grad_image(d, i, C, c);
        gc[c] = gp[c];
        cp[c] = 0.0;
    }
    pixel_color<C>(d, view, i, px, py, cp);

    // antialiasing: colour gradients (gather) and silhouette crossings (scatter)
    for (int k = 0; k < 4; ++k) {
        int qx, qy;
        if (!neighbour(d, px, py, k, qx, qy))
            continue;
        const Pair pr = pairs.get(k);
        if (!pr.active)
            continue;
        const size_t iq = (size_t)view * HW + (size_t)qy * d.W + qx;
        const bool t_low = pr.tf < 0.5f;  // the front pixel is the blended one
        if (!pr.p_blended) {
            // q is blended; its blend reads C_p only when q is the front pixel
            if (t_low) {
                const PairVal pv = pair_val(d, view, pr, px, py, qx, qy);
                const double w = pv.a * (0.5 - pv.t);
#pragma unroll
                for (int c = 0; c < C; ++c)
                    gc[c] += w * grad_image(d, iq, C, c);
            }
            continue;
        }
        const PairVal pv = pair_val(d, view, pr, px, py, qx, qy);
        const double wt = t_low ? 0.5 - pv.t : pv.t - 0.5;
        const double w = pv.a * wt;
        double src[C];
        double dedt = 0.0;  // d(w gp . E)/dt through the crossing point
        Bary B;
        if (t_low) {
            pixel_color<C>(d, view, iq, qx, qy, src);
        } else {
            H3 drdt;
            if (!bary_at_ray(d, view, pr.tri, crossing_ray(d, pr, pv.t, px, py, qx, qy, drdt), B))
                continue;
            bary_color<C>(d, B, src);
            double gsrc[C], de[C];
#pragma unroll
            for (int c = 0; c < C; ++c)
                gsrc[c] = w * gp[c];
            bary_backward<C>(d, A, view, B, gsrc);
            bary_color_dr<C>(d, B, drdt, de);
#pragma unroll
            for (int c = 0; c < C; ++c)
                dedt += gsrc[c] * de[c];
        }
        double dot = 0.0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            gc[c] -= w * gp[c];
            dot += gp[c] * (src[c] - cp[c]);
        }
        const double dldt = pv.a * (t_low ? -dot : dot) + dedt, dlda = wt * dot;
        scatter_window_grad<C>(d, A, view, pr.vj, dldt * pv.tj.x + dlda * pv.aj.x,
                            dldt * pv.tj.y + dlda * pv.aj.y);
        scatter_window_grad<C>(d, A, view, pr.vk, dldt * pv.tk.x + dlda * pv.ak.x,
                            dldt * pv.tk.y + dlda * pv.ak.y);
    }

    // barycentric interpolation of the pixel's own triangle
    const uint32_t id = d.ids[i];
    Bary B;
    const int tri = id_tri(d, view, id);
    if (tri < 0 || !bary_at(d, view, tri, px, py, B))
        return;
    bary_backward<C>(d, A, view, B, gc);
}

// The whole backward of one 16x16 tile, for a backward whose buffers the last forward did
// not store decisions for: pair decisions evaluated into LDS, vertex gradients accumulated
// in LDS and flushed once per vertex.
template <int C>
__global__ void __launch_bounds__(256) k_diff_backward(DiffArgs d)
{
    __shared__ int s_key[ACC_SLOTS];
    __shared__ __align__(16) float s_val[ACC_SLOTS * acc_stride<C>()];
    __shared__ PairLds s_h[TP_H], s_v[TP_V];
    for (int sl = threadIdx.x; sl < ACC_SLOTS; sl += blockDim.x)
        s_key[sl] = -1;
    for (int k = threadIdx.x; k < ACC_SLOTS * acc_stride<C>() / 4; k += blockDim.x)
        reinterpret_cast<float4 *>(s_val)[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    PixelIdx pi;
    const bool valid = pixel_of_thread(d, pi);
    tile_pairs(d, pi, s_h, s_v);
    __syncthreads();
    const VertexAcc A{s_key, s_val};
    if (valid)  // every thread reaches the barrier below
        backward_pixel<C>(d, A, pi, TilePairs{s_h, s_v});
    __syncthreads();
    acc_flush<C>(d, A, pi.view);
}

// DPP lane shifts inside rows of 16 lanes (one pixel row of the 16x16 tile): lane i reads
// lane i + n; a read past the row end yields `edge`.
template <int N>
__device__ inline int row_next(int v, int edge)
{
    return __builtin_amdgcn_update_dpp(edge, v, 0x100 + N, 0xF, 0xF, false);
}
template <int N>
__device__ inline float row_next(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + N, 0xF, 0xF,
                                                      false));
}
template <int N>
__device__ inline int row_prev(int v, int edge)
{
    return __builtin_amdgcn_update_dpp(edge, v, 0x110 + N, 0xF, 0xF, false);
}

// Every pixel's interpolation under dL/dimage.  Neighbouring pixels mostly show the same
// triangle (82% of horizontal pairs on the 41k-vertex sphere), so the lanes of a pixel row
// first merge their gradient values pairwise, then in fours and eights (a lane keeps its values
// when its partner shows another triangle).  The sums per vertex of the tile then go through
// lists, not through LDS float atomics, which take about two cycles per lane whatever the
// banks: a lane stores its merged values (3 corners of NV) with plain LDS writes, links each
// corner into its vertex's list with one exchange (3 atomics instead of 3 NV), and after a
// barrier a thread per (vertex, value) walks the vertex's two lists (of even and odd waves, so
// that the chains of reads overlap), adds in fp64 and flushes: neighbouring lanes add to
// neighbouring words of a gradient row, a third of the memory requests of a lane per vertex.
// Tiles of background alone leave at once.  64 views of 512x512 (41k vertices): 485 us with LDS
// float atomics and a flush of one lane per vertex, 427 us with lists and that flush, 240 us
// now (136 us without any accumulation); 16 terrain views of 768x768: 189 us.
constexpr uint32_t LIST_END = 0xFFFFu;

template <int C>
__global__ void __launch_bounds__(256) k_diff_bwd_interior(DiffArgs d)
{
    constexpr int NV = 3 + C;
    __shared__ int s_key[ACC_SLOTS];
    __shared__ uint32_t s_head[2][ACC_SLOTS];
    __shared__ uint16_t s_next[3 * 256];
    constexpr int ST = NV | 1;               // odd: lanes' entries spread over the banks
    __shared__ float s_val[3 * 256 * ST];    // entry m * 256 + thread: corner m of a lane
    __shared__ uint8_t s_used[ACC_SLOTS];    // the occupied slots, packed
    __shared__ uint32_t s_cnt[4];
    PixelIdx pi;
    const bool valid = pixel_of_thread(d, pi);
    const int t0 = valid ? id_tri(d, pi.view, d.ids[pi.i]) : -1;
    if (!__syncthreads_or(t0 >= 0))
        return;  // background: nothing to add
    static_assert(ACC_SLOTS == 256, "a slot per thread");
    s_key[threadIdx.x] = -1;
    s_head[0][threadIdx.x] = s_head[1][threadIdx.x] = LIST_END;
    int tri = -1, vid[3] = {0, 0, 0};
    float g[3][NV];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int k = 0; k < NV; ++k)
            g[m][k] = 0.0f;
    if (t0 >= 0) {
        Bary B;
        if (bary_at(d, pi.view, t0, pi.px, pi.py, B)) {
            double gc[C];
#pragma unroll
            for (int c = 0; c < C; ++c)
                gc[c] = grad_image(d, pi.i, C, c);
            bary_grads<C>(d, B, gc, g);
            tri = t0;
#pragma unroll
            for (int m = 0; m < 3; ++m)
                vid[m] = B.v[m];
        }
    }
    // merge along the row: at stride s, lane i (i % 2s == 0) takes lane i + s's sums when
    // both show the same triangle and lane i + s still holds its own (it merged nothing away)
    const int lx = (int)(threadIdx.x & 15u);
    bool keep = tri >= 0;
#define SWR_MERGE(S)                                                                            \
    {                                                                                          \
        const int t_n = row_next<S>(keep ? tri : -2, -3);                                      \
        const int t_p = row_prev<S>(keep ? tri : -2, -3);                                      \
        const bool take = keep && (lx % (2 * S)) == 0 && t_n == tri;                           \
        const bool give = keep && (lx % (2 * S)) == S && t_p == tri;                           \
        _Pragma("unroll") for (int m = 0; m < 3; ++m)                                          \
            _Pragma("unroll") for (int k = 0; k < NV; ++k)                                     \
        {                                                                                      \
            const float o = row_next<S>(g[m][k]);                                              \
            g[m][k] = take ? g[m][k] + o : g[m][k];                                            \
        }                                                                                      \
        keep = keep && !give;                                                                  \
    }
    if (__ballot(keep) != 0ull) {
        SWR_MERGE(1)
        SWR_MERGE(2)
        SWR_MERGE(4)
    }
#undef SWR_MERGE
    __syncthreads();
    const VertexAcc A{s_key, nullptr};
    if (keep) {
        int sl[3];
        acc_find3(A, vid, sl);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const uint32_t e = (uint32_t)m * 256u + threadIdx.x;
            if (sl[m] >= 0) {
#pragma unroll
                for (int k = 0; k < NV; ++k)
                    s_val[e * ST + k] = g[m][k];
                s_next[e] = (uint16_t)atomicExch(&s_head[(threadIdx.x >> 6) & 1u][sl[m]], e);
            } else {  // no slot for this vertex
                float *gc = d.gclip + crow(d, pi.view, vid[m]) * 4;
                atomicAdd(gc + 0, g[m][0]);
                atomicAdd(gc + 1, g[m][1]);
                atomicAdd(gc + 3, g[m][2]);
#pragma unroll
                for (int c = 0; c < C; ++c)
                    atomicAdd(d.gattr + crow(d, pi.view, vid[m]) * C + c, g[m][3 + c]);
            }
        }
    }
    __syncthreads();
    const bool used = s_key[threadIdx.x] >= 0;
    const unsigned long long mu = __ballot(used);
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    if (lane == 0)
        s_cnt[w] = (uint32_t)__popcll(mu);
    __syncthreads();
    uint32_t before = 0, n = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
        before += q < w ? s_cnt[q] : 0u;
        n += s_cnt[q];
    }
    if (used)
        s_used[before + (uint32_t)__popcll(mu & ((1ull << lane) - 1ull))] = (uint8_t)threadIdx.x;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n * NV; i += 256) {
        const uint32_t sl = s_used[i / NV], k = i % NV;
        uint32_t e0 = s_head[0][sl], e1 = s_head[1][sl];
        double x = 0.0;
        while (e0 != LIST_END || e1 != LIST_END) {
            const bool h0 = e0 != LIST_END, h1 = e1 != LIST_END;
            const uint32_t a0 = h0 ? e0 : 0u, a1 = h1 ? e1 : 0u;
            const float v0 = s_val[a0 * ST + k], v1 = s_val[a1 * ST + k];
            e0 = h0 ? s_next[a0] : LIST_END;
            e1 = h1 ? s_next[a1] : LIST_END;
            x += (double)(h0 ? v0 : 0.0f) + (double)(h1 ? v1 : 0.0f);
        }
        const size_t row = crow(d, pi.view, s_key[sl]);
        float *to = k < 3 ? d.gclip + row * 4 + (k == 2 ? 3 : k) : d.gattr + row * C + (k - 3);
        if (x != 0.0)
            atomicAdd(to, (float)x);
    }
}

// ---- what the antialiasing adds to the gradients ---------------------------------------------
// One lane per active pair (the blend pass listed them; the decisions come from the forward's
// store).  A pair blends one pixel B with a source colour: when the crossing lies in the front
// pixel's half, B is the front pixel and the source the other pixel's colour, else B is the
// other pixel and the source the silhouette triangle's colour at the crossing.  Either way the
// source is a triangle's interpolation along a ray, so all lanes run the same code: B's and
// the source's interpolation, forward and backward, and the crossing's derivatives.  Bound by the
// latency of that chain (dependent loads, fp64 divisions), so it is kept short and every wave
// gets 64 pairs: pairs cluster on silhouettes, and a wave per 16 tiles left most waves idle
// behind a few long ones.
// One 256x256 view / 64 views of 512x512 / 16 terrain views of 768x768: 79 / 553 / 1007 us with a
// lane per pixel and its four pairs in turn, 31 / 67 / 347 us with a lane per pair and a wave per
// 16 tiles, 20 / 56 / 146 us with the even split (the larger ones beside the interior kernel),
// 20 / 30 / 82 us in turn with it.
//
// Neighbouring silhouette pairs share vertices: a wave takes 64 pairs at a time, a pair stores
// its 8 entries (two triangles' corners, the window gradients of the edge's ends), each rounded
// to fp32 by itself, with plain LDS writes and links each into its clip row's list; a lane per
// (row, value) then adds the list in fp64 and flushes, as in the interior kernel (LDS float
// atomics took 309 us instead of 242 us on the terrain, alone and before the even split).  A
// row that finds no slot goes to global memory.
constexpr int EDGE_SLOTS = 256;  // power of two
constexpr int EDGE_PROBES = 8;
constexpr int EDGE_ENTRIES = 8;  // per pair

template <int C>
struct EdgeLists {
    static constexpr int NV = 3 + C, ST = NV | 1;  // odd: entries spread over the banks
    int key[EDGE_SLOTS];
    uint32_t head[EDGE_SLOTS];
    uint16_t next[EDGE_ENTRIES * 64];
    uint8_t used[EDGE_SLOTS];
    float val[EDGE_ENTRIES * 64 * ST];
};

// Entry `n` of this lane's pair: {clip x, y, w, attributes} of clip row `row`.
template <int C>
__device__ inline void edge_add(const DiffArgs &d, EdgeLists<C> &A, int n, size_t row,
                                const float (&g)[3 + C])
{
    constexpr int NV = 3 + C;
    int slot = -1;
    if (d.row_keys) {
        const unsigned h = ((unsigned)row * 2654435761u) >> 24;  // 8 bits: EDGE_SLOTS
#pragma unroll 1
        for (int probe = 0; probe < EDGE_PROBES && slot < 0; ++probe) {
            const int sl = (int)((h + (unsigned)probe) & (EDGE_SLOTS - 1));
            int old = __atomic_load_n(&A.key[sl], __ATOMIC_RELAXED);
            if (old == -1)
                old = atomicCAS(&A.key[sl], -1, (int)row);
            if (old == -1 || old == (int)row)
                slot = sl;
        }
    }
    if (slot >= 0) {
        const uint32_t e = (uint32_t)n * 64u + threadIdx.x;
#pragma unroll
        for (int k = 0; k < NV; ++k)
            A.val[e * EdgeLists<C>::ST + k] = g[k];
        A.next[e] = (uint16_t)atomicExch(&A.head[slot], e);
        return;
    }
    atomicAdd(d.gclip + row * 4 + 0, g[0]);
    atomicAdd(d.gclip + row * 4 + 1, g[1]);
    atomicAdd(d.gclip + row * 4 + 3, g[2]);
#pragma unroll
    for (int c = 0; c < C; ++c)
        atomicAdd(d.gattr + row * C + c, g[3 + c]);
}

// Adds every list to the gradients: a lane per (row, value), neighbouring lanes to
// neighbouring words of a gradient row.
template <int C>
__device__ inline void edge_flush(const DiffArgs &d, EdgeLists<C> &A)
{
    constexpr uint32_t NV = 3 + C;
    const uint32_t lane = threadIdx.x;
    uint32_t n = 0;
#pragma unroll
    for (uint32_t q = 0; q < EDGE_SLOTS / 64; ++q) {
        const bool used = A.key[q * 64 + lane] >= 0;
        const unsigned long long m = __ballot(used);
        if (used)
            A.used[n + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint8_t)(q * 64 + lane);
        n += (uint32_t)__popcll(m);
    }
    lds_sync();
    for (uint32_t i = lane; i < n * NV; i += 64) {
        const uint32_t sl = A.used[i / NV], k = i % NV;
        double x = 0.0;
        for (uint32_t e = A.head[sl]; e != LIST_END; e = A.next[e])
            x += (double)A.val[e * EdgeLists<C>::ST + k];
        const size_t row = (size_t)A.key[sl];
        float *to = k < 3 ? d.gclip + row * 4 + (k == 2 ? 3 : k) : d.gattr + row * C + (k - 3);
        if (x != 0.0)
            atomicAdd(to, (float)x);
    }
}

// d(window x, y) of a clip-space vertex -> d(clip x, y, w).
__device__ inline void window_grad(const DiffArgs &d, const H3 &h, double gx, double gy,
                                   float (&out)[3])
{
    const double iw = 1.0 / h.w, sx = 0.5 * d.W, sy = 0.5 * d.H;
    out[0] = (float)(gx * sx * iw);
    out[1] = (float)(-gy * sy * iw);
    out[2] = (float)((-gx * sx * h.x + gy * sy * h.y) * iw * iw);
}

template <int C>
__device__ inline void backward_pair(const DiffArgs &d, EdgeLists<C> &A, uint32_t k)
{
    const size_t HW = (size_t)d.W * d.H;
    const size_t i = k >> 1;
    const int dir = (int)(k & 1u);
    const int view = (int)(i / HW);
    const size_t rem = i - (size_t)view * HW;
    const int py = (int)(rem / (size_t)d.W), px = (int)(rem - (size_t)py * d.W);
    const int qx = px + (dir == 0), qy = py + (dir == 1);
    const PairLds x = load_pair(d, k);
    const Pair pr = unpack_pair(x, false, dir == 0);
    const size_t iq = i + (dir == 0 ? (size_t)1 : (size_t)d.W);
    const size_t ib = pr.p_blended ? i : iq, io = pr.p_blended ? iq : i;
    const int bx = pr.p_blended ? px : qx, by = pr.p_blended ? py : qy;
    const int ox = pr.p_blended ? qx : px, oy = pr.p_blended ? qy : py;
    const bool t_low = pr.tf < 0.5f;  // B is the front pixel

    const PairVal pv = pair_val(d, view, pr, px, py, qx, qy);
    const double wt = t_low ? 0.5 - pv.t : pv.t - 0.5, w = pv.a * wt;
    double g[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        g[c] = grad_image(d, ib, C, c);

    // the source: the other pixel's triangle at its centre, or the silhouette's at the crossing
    Bary S, B;
    H3 drdt;
    const int tri_s = t_low ? id_tri(d, view, d.ids[io]) : pr.tri;
    H3 ray = crossing_ray(d, pr, pv.t, px, py, qx, qy, drdt);
    if (t_low)
        ray = pixel_ray(d, ox, oy);
    const bool has_s = tri_s >= 0 && bary_at_ray(d, view, tri_s, ray, S);
    if (!t_low && !has_s)
        return;  // the blend skipped it too
    const int tri_b = id_tri(d, view, d.ids[ib]);
    const bool has_b = tri_b >= 0 && bary_at(d, view, tri_b, bx, by, B);
    double src[C], cp[C], de[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        src[c] = cp[c] = de[c] = 0.0;
    if (has_s) {
        bary_color<C>(d, S, src);
        if (!t_low)
            bary_color_dr<C>(d, S, drdt, de);
    }
    if (has_b)
        bary_color<C>(d, B, cp);
    double dot = 0.0, dedt = 0.0, gs[C], gb[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        // a pixel's colour is an fp32 image value
        const double s = t_low ? (double)(float)src[c] : src[c];
        dot += g[c] * (s - (double)(float)cp[c]);
        gs[c] = w * g[c];
        gb[c] = -gs[c];
        dedt += gs[c] * de[c];
    }
    // the crossing: its edge's vertices j and k
    const double dldt = pv.a * (t_low ? -dot : dot) + dedt, dlda = wt * dot;
    float wj[3], wk[3];
    window_grad(d, load_h(d, view, pr.vj), dldt * pv.tj.x + dlda * pv.aj.x,
                dldt * pv.tj.y + dlda * pv.aj.y, wj);
    window_grad(d, load_h(d, view, pr.vk), dldt * pv.tk.x + dlda * pv.ak.x,
                dldt * pv.tk.y + dlda * pv.ak.y, wk);
    const auto triangle = [&](const Bary &T, const double *gc, int n0) {
        float out[3][3 + C];
        bary_grads<C>(d, T, gc, out);
#pragma unroll
        for (int m = 0; m < 3; ++m)
            edge_add<C>(d, A, n0 + m, crow(d, view, T.v[m]), out[m]);
    };
    if (has_s)
        triangle(S, gs, 0);
    if (has_b)
        triangle(B, gb, 3);
    // two entries without attributes
    float out[3 + C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        out[3 + c] = 0.0f;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
#pragma unroll
        for (int n = 0; n < 3; ++n)
            out[n] = v == 0 ? wj[n] : wk[n];
        edge_add<C>(d, A, 6 + v, crow(d, view, v == 0 ? pr.vj : pr.vk), out);
    }
}

template <int C>
__global__ void __launch_bounds__(64) k_diff_bwd_edges(DiffArgs d, uint32_t regions)
{
    __shared__ EdgeLists<C> A;
    __shared__ uint32_t s_off[EDGE_REGIONS + 1];  // pairs before region r
    const uint32_t lane = threadIdx.x;
    uint32_t n = 0;
#pragma unroll
    for (uint32_t q = 0; q < EDGE_REGIONS / 64; ++q) {
        const uint32_t r = q * 64 + lane;
        const uint32_t c = r < regions ? d.ecnt[r] : 0u, v = wave_incl(c);
        s_off[r] = n + v - c;
        n += __shfl(v, 63, 64);
    }
    if (lane == 0)
        s_off[EDGE_REGIONS] = n;
    lds_sync();
    for (uint32_t j0 = blockIdx.x * 64; j0 < n; j0 += gridDim.x * 64) {
#pragma unroll
        for (int q = 0; q < EDGE_SLOTS / 64; ++q) {
            A.key[q * 64 + lane] = -1;
            A.head[q * 64 + lane] = LIST_END;
        }
        lds_sync();
        const uint32_t j = j0 + lane;
        if (j < n) {
            uint32_t lo = 0, hi = EDGE_REGIONS;  // the last region with s_off <= j
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (s_off[mid] <= j)
                    lo = mid;
                else
                    hi = mid;
            }
            backward_pair<C>(d, A, d.elist[(size_t)lo * d.region_tiles * 512 + (j - s_off[lo])]);
        }
        lds_sync();
        edge_flush<C>(d, A);
        lds_sync();  // the lists are cleared for the next 64 pairs
    }
}

// grad_attributes += sum over the views that see the vertex (in view order) of the
// partials; the partials are cleared for the next call (they start at zero when the buffer
// is created).
__global__ void __launch_bounds__(256) k_diff_reduce_attr(DiffArgs d, int C)
{
    const size_t n = (size_t)d.N * C;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (size_t)gridDim.x * blockDim.x) {
        const int g = (int)(k / (size_t)C), c = (int)(k - (size_t)g * C);
        int v0 = 0, v1 = d.V;
        if (d.svert) {
            // the scene owning vertex g: the last s with svert[s] <= g (svert[S] = N > g)
            int lo = 0, hi = d.S - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (d.svert[mid] <= g)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            v0 = d.sview[lo];
            v1 = d.sview[lo + 1];
        }
        float s = 0.0f;
        for (int v = v0; v < v1; ++v) {
            float *p = d.gattr + crow(d, v, g) * C + c;
            s += *p;
            *p = 0.0f;
        }
        d.gattr_out[k] += s;
    }
}

constexpr uint32_t EDGE_WAVES = 2048;

template <int C>
static hipError_t launch_diff(const DiffArgs &d, int which, hipStream_t s)
{
    const uint32_t blocks = (uint32_t)((size_t)d.tiles_per_view * d.V);
    if (!blocks)
        return hipSuccess;
    if (which == 0) {
        hipLaunchKernelGGL(k_diff_interp<C>, dim3(blocks), dim3(256), 0, s, d);
        hipLaunchKernelGGL(k_diff_march, dim3((blocks + MARCH_TILES - 1) / MARCH_TILES),
                           dim3(MARCH_THREADS), 0, s, d);
        hipLaunchKernelGGL(k_diff_blend<C>, dim3(blocks), dim3(256), 0, s, d);
    } else {
        if (d.pairs == 2) {
            // Both kernels add into the same gradients and neither reads what the other writes,
            // but side by side on two streams they are no faster: each fills the GPU, so 64 views
            // of 512x512 take 1178 us forked and 1173 in turn, 8 views 280 and 266 us.
            // as many waves as the GPU holds (two per SIMD), or a wave per 64 possible pairs
            const uint32_t waves = blocks < EDGE_WAVES / 8 ? blocks * 8 : EDGE_WAVES;
            hipLaunchKernelGGL(k_diff_bwd_edges<C>, dim3(waves), dim3(64), 0, s, d,
                               (blocks + d.region_tiles - 1) / d.region_tiles);
            hipLaunchKernelGGL(k_diff_bwd_interior<C>, dim3(blocks), dim3(256), 0, s, d);
        } else {
            hipLaunchKernelGGL(k_diff_backward<C>, dim3(blocks), dim3(256), 0, s, d);
        }
        const size_t n = (size_t)d.N * C;
        const uint32_t rb = (uint32_t)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
        if (rb)
            hipLaunchKernelGGL(k_diff_reduce_attr, dim3(rb), dim3(256), 0, s, d, C);
    }
    return hipGetLastError();
}

static int diff_run(swr_context *c, const swr_diff_desc *dd, const float *gimage, float *gclip,
                    float *gattr, int which)
{
    if (!c || !dd)
        return SWR_ERR_INVALID_ARG;
    const swr_diff_desc &q = *dd;
    if (q.views < 0 || q.width < 0 || q.height < 0 || q.vertex_count < 0 || q.triangle_count < 0)
        return context_fail(c, SWR_ERR_INVALID_ARG, "negative size in swr_diff_desc");
    if (q.channels < 1 || q.channels > 4)
        return context_fail(c, SWR_ERR_UNSUPPORTED, "channels must be 1..4");
    const size_t px = (size_t)q.views * q.width * q.height;
    if (px == 0)
        return SWR_OK;
    const void *need[] = {q.clip, q.triangles, q.adjacency, q.attributes, q.ids, q.depth, q.bary};
    for (const void *p : need)
        if (!p || !context_is_device_ptr(p))
            return context_fail(c, SWR_ERR_INVALID_ARG, "swr_diff buffers must be device memory");
    if (q.color && !context_is_device_ptr(q.color))
        return context_fail(c, SWR_ERR_INVALID_ARG, "swr_diff buffers must be device memory");
    if (which == 0 && (!q.image || !context_is_device_ptr(q.image)))
        return context_fail(c, SWR_ERR_INVALID_ARG, "swr_diff_forward needs image");
    if (which == 1 && (!gimage || !gclip || !gattr || !context_is_device_ptr(gimage) ||
                       !context_is_device_ptr(gclip) || !context_is_device_ptr(gattr)))
        return context_fail(c, SWR_ERR_INVALID_ARG, "swr_diff_backward needs device gradients");
    DiffArgs d;
    d.V = q.views;
    d.W = q.width;
    d.H = q.height;
    d.N = q.vertex_count;
    d.T = q.triangle_count;
    d.culled = (q.flags & SWR_DIFF_CULLED) ? 1 : 0;
    d.tiles_x = (q.width + 15) / 16;
    d.tiles_per_view = d.tiles_x * ((q.height + 15) / 16);
    if ((size_t)d.tiles_per_view * d.V > 0x7FFFFFFFull)
        return context_fail(c, SWR_ERR_CAPACITY, "too many pixels for one swr_diff call");
    d.sx = (float)q.width / 2.0f;
    d.sy = (float)q.height / 2.0f;
    d.clip = reinterpret_cast<const float4 *>(q.clip);
    d.tris = q.triangles;
    d.adj = q.adjacency;
    d.attr = q.attributes;
    d.ids = q.ids;
    d.depth = q.depth;
    d.bary = q.bary;
    d.color = q.color;
    d.image = q.image;
    d.gimage = gimage;
    d.l2_target = (q.flags & SWR_DIFF_L2_TARGET) ? 1 : 0;
    if (which == 1 && d.l2_target && (!q.image || !context_is_device_ptr(q.image)))
        return context_fail(c, SWR_ERR_INVALID_ARG, "SWR_DIFF_L2_TARGET needs the forward's image");
    d.gclip = gclip;
    d.gattr = nullptr;
    d.gattr_out = gattr;
    d.vrow = nullptr;
    d.vtri = nullptr;
    d.svert = d.sview = nullptr;
    d.S = 1;
    size_t rows = (size_t)d.V * d.N;  // clip / gradient rows
    uint64_t table_gen = 0;
    if (q.scenes > 1) {
        const int S = q.scenes;
        const int32_t *pv = q.scene_views, *pn = q.scene_vertices, *pt = q.scene_triangles;
        if (!pv || !pn || !pt)
            return context_fail(c, SWR_ERR_INVALID_ARG, "swr_diff scenes > 1 needs the scene tables");
        if (pv[0] != 0 || pn[0] != 0 || pt[0] != 0 || pv[S] != q.views || pn[S] != q.vertex_count ||
            pt[S] != q.triangle_count)
            return context_fail(c, SWR_ERR_INVALID_ARG,
                                "swr_diff scene tables must run from 0 to views / vertex_count / "
                                "triangle_count");
        for (int k = 0; k < S; ++k)
            if (pv[k + 1] < pv[k] || pn[k + 1] < pn[k] || pt[k + 1] < pt[k])
                return context_fail(c, SWR_ERR_INVALID_ARG, "swr_diff scene tables must not decrease");
        // table: vrow [V] i64, vtri [V] int2, svert [S + 1] i32, sview [S + 1] i32
        std::vector<unsigned char> tab((size_t)16 * d.V + (size_t)8 * (S + 1));
        long long *vrow = reinterpret_cast<long long *>(tab.data());
        int2 *vtri = reinterpret_cast<int2 *>(tab.data() + (size_t)8 * d.V);
        int32_t *svert = reinterpret_cast<int32_t *>(tab.data() + (size_t)16 * d.V);
        int32_t *sview = svert + (S + 1);
        long long base = 0;
        for (int k = 0; k < S; ++k) {
            const long long nk = pn[k + 1] - pn[k];
            for (int v = pv[k]; v < pv[k + 1]; ++v) {
                vrow[v] = base + (long long)(v - pv[k]) * nk - pn[k];
                vtri[v] = make_int2(pt[k], pt[k + 1] - pt[k]);
            }
            base += (long long)(pv[k + 1] - pv[k]) * nk;
        }
        std::memcpy(svert, pn, sizeof(int32_t) * (S + 1));
        std::memcpy(sview, pv, sizeof(int32_t) * (S + 1));
        rows = (size_t)base;
        const unsigned char *dev =
            static_cast<const unsigned char *>(context_diff_table(c, tab.data(), tab.size(), &table_gen));
        if (!dev)
            return context_last_code(c);
        d.vrow = reinterpret_cast<const long long *>(dev);
        d.vtri = reinterpret_cast<const int2 *>(dev + (size_t)8 * d.V);
        d.svert = reinterpret_cast<const int *>(dev + (size_t)16 * d.V);
        d.sview = d.svert + (S + 1);
        d.S = S;
    }
    if (which == 1) {
        // per-view partials: views do not contend on one vertex's attribute gradient
        d.gattr = (float *)context_zeroed_scratch(c, 0, rows * q.channels * 4);
        if (!d.gattr)
            return context_last_code(c);
    }
    // The forward stores its pair decisions; a backward over the same buffers and sizes
    // reuses them instead of walking the silhouettes again.
    // layout: flags [2 px] u8, data [2 px] int2, per tile: flags, queue and list lengths
    // u32, queue [tiles][512] u32, which the active pairs' lists take over: the blend pass
    // writes them once the march pass has read the queue
    const size_t tiles = (size_t)d.tiles_per_view * d.V, off_f = 0,
                 off_d = (off_f + px * 2 + 15) & ~(size_t)15, off_t = off_d + px * 2 * sizeof(int2),
                 off_q = (off_t + tiles * 12 + 15) & ~(size_t)15;
    d.region_tiles = (uint32_t)((tiles + EDGE_REGIONS - 1) / EDGE_REGIONS);
    d.row_keys = rows <= 0x7FFFFFFFull ? 1 : 0;
    if (px * 2 > 0xFFFFFFFFull)
        return context_fail(c, SWR_ERR_CAPACITY, "too many pixels for one swr_diff call");
    uint8_t *pbuf = (uint8_t *)context_zeroed_scratch(c, 1, off_q + tiles * 512 * 4);
    if (!pbuf)
        return context_last_code(c);
    d.qcnt = reinterpret_cast<uint32_t *>(pbuf + off_t) + tiles;
    d.ecnt = reinterpret_cast<uint32_t *>(pbuf + off_t) + 2 * tiles;
    d.pflag = pbuf + off_f;
    d.pdata = reinterpret_cast<int2 *>(pbuf + off_d);
    d.tflag = reinterpret_cast<uint32_t *>(pbuf + off_t);
    d.queue = reinterpret_cast<uint32_t *>(pbuf + off_q);
    d.elist = d.queue;
    const uint64_t tag[9] = {(uint64_t)(uintptr_t)q.clip,      (uint64_t)(uintptr_t)q.triangles,
                             (uint64_t)(uintptr_t)q.adjacency, (uint64_t)(uintptr_t)q.ids,
                             (uint64_t)(uintptr_t)q.depth,     (uint64_t)(uintptr_t)pbuf,
                             ((uint64_t)q.views << 32) | (uint32_t)q.width,
                             ((uint64_t)q.height << 40) | ((uint64_t)(q.flags & SWR_DIFF_CULLED) << 32) |
                                 (uint32_t)q.triangle_count,
                             q.scenes > 1 ? table_gen : 0};
    uint64_t *held = context_diff_tag(c);
    if (which == 0) {
        d.pairs = 1;
        std::memcpy(held, tag, sizeof tag);
    } else {
        d.pairs = std::memcmp(held, tag, sizeof tag) == 0 ? 2 : 0;
    }
    hipStream_t s = context_stream(c);
    hipError_t e;
    switch (q.channels) {
    case 1: e = launch_diff<1>(d, which, s); break;
    case 2: e = launch_diff<2>(d, which, s); break;
    case 3: e = launch_diff<3>(d, which, s); break;
    default: e = launch_diff<4>(d, which, s); break;
    }
    if (e != hipSuccess)
        return context_fail(c, SWR_ERR_HIP, hipGetErrorString(e));
    return SWR_OK;
}

}  // namespace swr

extern "C" {

int swr_diff_forward(swr_context *c, const swr_diff_desc *d)
{
    return swr::diff_run(c, d, nullptr, nullptr, nullptr, 0);
}

int swr_diff_backward(swr_context *c, const swr_diff_desc *d, const float *grad_image,
                      float *grad_clip, float *grad_attributes)
{
    return swr::diff_run(c, d, grad_image, grad_clip, grad_attributes, 1);
}

}  // extern "C"
