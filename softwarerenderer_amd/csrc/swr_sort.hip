// swr_sort.hip — exclusive scans and the stable (tile, primitive) radix sort.
//
// Binning needs, per 8x8 tile, the primitives touching it in draw order.  The emit pass
// writes (tile, primitive) pairs grouped by primitive in draw order; a stable radix sort on
// the tile id regroups them by tile while keeping draw order inside each tile.  Only each
// tile's own order matters, not the order of the tiles, so one scatter deals the ids to 256
// buckets (swr_buckets.h), and one workgroup per bucket regroups its pairs by the ids' remaining
// bits and writes its tiles' ranges (k_bucket; up to 2^18 tiles).  More tiles take least
// significant digit passes of 8 bits each, then k_ranges.  Ranks inside a block are made
// stable with wave ballots: the lanes of a wave holding the same digit are found with a
// ballot per bit, and a lane's rank is the number of such lanes below it.
//
// A pass is bound by launches and by its scattered writes rather than by bytes (964k pairs:
// 12 bytes each way, 4 us at 6 TB/s): two digit passes of four launches and the ranges' took
// 67 us on the 1080p soup's 964k pairs, the scatter and the buckets take 45 us (964k pairs in
// 8160 bins) and 20 instead of 34 us on a small frame (7.5k pairs in 4800 bins).
#include <utility>

#include "swr_buckets.h"
#include "swr_common.h"
#include "swr_internal.h"

namespace swr {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ inline uint32_t sadd(uint32_t a, uint32_t b) { return a + b; }
__device__ inline uint2 sadd(uint2 a, uint2 b) { return make_uint2(a.x + b.x, a.y + b.y); }
__device__ inline uint4 sadd(uint4 a, uint4 b)
{
    return make_uint4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
template <typename T> __device__ inline T szero();
template <> __device__ inline uint32_t szero<uint32_t>() { return 0u; }
template <> __device__ inline uint2 szero<uint2>() { return make_uint2(0u, 0u); }
template <> __device__ inline uint4 szero<uint4>() { return make_uint4(0u, 0u, 0u, 0u); }

__device__ inline uint2 wave_incl(uint2 v) { return make_uint2(wave_incl(v.x), wave_incl(v.y)); }
__device__ inline uint4 wave_incl(uint4 v)
{
    return make_uint4(wave_incl(v.x), wave_incl(v.y), wave_incl(v.z), wave_incl(v.w));
}
__device__ inline uint32_t ssub(uint32_t a, uint32_t b) { return a - b; }
__device__ inline uint2 ssub(uint2 a, uint2 b) { return make_uint2(a.x - b.x, a.y - b.y); }
__device__ inline uint4 ssub(uint4 a, uint4 b)
{
    return make_uint4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w);
}

// Block-wide exclusive scan of one value per thread; returns the block total in *total.
template <typename T>
__device__ T block_exclusive(T v, T *total)
{
    constexpr int NW = SCAN_THREADS / 64;
    __shared__ T s_w[NW];
    const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
    const T inc = wave_incl(v);
    if (lane == 63)
        s_w[w] = inc;
    __syncthreads();
    T pre = szero<T>(), tot = szero<T>();
#pragma unroll
    for (int k = 0; k < NW; ++k) {
        const T x = s_w[k];
        if (k < w)
            pre = sadd(pre, x);
        tot = sadd(tot, x);
    }
    __syncthreads();  // s_w is reused by the next call
    *total = tot;
    return sadd(pre, ssub(inc, v));
}

// SCAN_ITEMS consecutive elements from `base`: 16-byte loads when the run is whole and
// aligned, element by element (zero past n) otherwise.
template <typename T>
__device__ inline void load_items(const T *in, uint64_t base, uint64_t n, T (&v)[SCAN_ITEMS])
{
    const T *p = in + base;
    if (base + SCAN_ITEMS <= n && ((uintptr_t)p & 15u) == 0) {
        constexpr int Q = SCAN_ITEMS * (int)sizeof(T) / 16;
        uint4 q[Q];
#pragma unroll
        for (int k = 0; k < Q; ++k)
            q[k] = reinterpret_cast<const uint4 *>(p)[k];
        __builtin_memcpy(v, q, sizeof v);
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i)
            v[i] = base + i < n ? p[i] : szero<T>();
    }
}

template <typename T>
__device__ inline void store_items(T *out, uint64_t base, uint64_t n, const T (&v)[SCAN_ITEMS])
{
    T *p = out + base;
    if (base + SCAN_ITEMS <= n && ((uintptr_t)p & 15u) == 0) {
        constexpr int Q = SCAN_ITEMS * (int)sizeof(T) / 16;
        uint4 q[Q];
        __builtin_memcpy(q, v, sizeof q);
#pragma unroll
        for (int k = 0; k < Q; ++k)
            reinterpret_cast<uint4 *>(p)[k] = q[k];
    } else {
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i)
            if (base + i < n)
                p[i] = v[i];
    }
}

// Sum of scan tile b (SCAN_TILE elements) into sums[b].
template <typename T>
__device__ void reduce_tile(const T *in, uint64_t n, T *sums, uint32_t b)
{
    const uint64_t base = (uint64_t)b * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    T v[SCAN_ITEMS];
    load_items<T>(in, base, n, v);
    T acc = szero<T>();
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
        acc = sadd(acc, v[i]);
    T total;
    block_exclusive<T>(acc, &total);
    if (threadIdx.x == 0)
        sums[b] = total;
}

template <typename T>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_reduce(const T *in, uint64_t n, T *sums)
{
    reduce_tile<T>(in, n, sums, blockIdx.x);
}

// One block scans the block sums in place (exclusive), SCAN_TILE sums per step.
template <typename T>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_sums(T *sums, uint32_t nblocks)
{
    T carry = szero<T>();
    for (uint64_t c0 = 0; c0 < nblocks; c0 += SCAN_TILE) {
        const uint64_t base = c0 + (uint64_t)threadIdx.x * SCAN_ITEMS;
        T v[SCAN_ITEMS];
        load_items<T>(sums, base, nblocks, v);
        T acc = szero<T>();
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i)
            acc = sadd(acc, v[i]);
        T total;
        T run = sadd(block_exclusive<T>(acc, &total), carry);
#pragma unroll
        for (int i = 0; i < SCAN_ITEMS; ++i) {
            const T x = v[i];
            v[i] = run;
            run = sadd(run, x);
        }
        store_items<T>(sums, base, nblocks, v);
        carry = sadd(carry, total);
    }
}

// The totals of the (prims, pairs) scan, published by the thread that owns the last element,
// with arena overflow against the capacities.
__device__ inline void publish_totals(uint2 t, unsigned long long *status, uint64_t cap_x,
                                      uint64_t cap_y)
{
    status[ST_PRIMS] = t.x;
    status[ST_PAIRS] = t.y;
    unsigned long long of = 0;
    if (t.x > cap_x) of |= 1ull;
    if (t.y > cap_y) of |= 2ull;
    status[ST_OVERFLOW] = of;
}

// Sum of sums[0 .. b) over the block (the carry into block b when no pass has scanned the
// block sums): b / SCAN_THREADS loads per thread, for scans of few blocks.
template <typename T>
__device__ T block_carry(const T *sums, uint32_t b)
{
    T acc = szero<T>();
    for (uint32_t k = threadIdx.x; k < b; k += SCAN_THREADS)
        acc = sadd(acc, sums[k]);
    T total;
    block_exclusive<T>(acc, &total);
    __syncthreads();  // block_exclusive's LDS is used again by the caller
    return total;
}

// Writes the exclusive scan.  CARRY: the block adds up the block sums before it (the
// two-kernel scan); else sums[] holds their exclusive scan.  With `status` set the thread
// that owns the last element publishes the total (publish_totals).
template <typename T, bool CARRY>
__device__ void down_tile(const T *in, uint64_t n, const T *sums, T *out,
                          unsigned long long *status, uint64_t cap_x, uint64_t cap_y,
                          uint32_t b)
{
    const T carry = CARRY ? block_carry<T>(sums, b) : sums[b];
    const uint64_t base = (uint64_t)b * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    T vals[SCAN_ITEMS];
    load_items<T>(in, base, n, vals);
    T acc = szero<T>();
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
        acc = sadd(acc, vals[i]);
    T total;
    T run = sadd(block_exclusive<T>(acc, &total), carry);
    T o[SCAN_ITEMS];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        o[i] = run;
        if (status && base + i == n - 1)
            publish_totals(sadd(run, vals[i]), status, cap_x, cap_y);
        run = sadd(run, vals[i]);
    }
    store_items<T>(out, base, n, o);
}

template <typename T, bool CARRY>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_down(const T *in, uint64_t n,
                                                          const T *sums, T *out,
                                                          unsigned long long *status,
                                                          uint64_t cap_x, uint64_t cap_y)
{
    down_tile<T, CARRY>(in, n, sums, out, status, cap_x, cap_y, blockIdx.x);
}

// Scans of up to this many blocks skip the pass over the block sums: each block of the
// down pass adds up the sums before it (at most SCAN_CARRY_BLOCKS / SCAN_THREADS loads per
// thread, one round of independent L2 loads).
constexpr uint32_t SCAN_CARRY_BLOCKS = 8192;

template <typename T>
hipError_t scan_impl(const T *in, T *out, uint64_t n, T *tmp, unsigned long long *status,
                     uint64_t cap_x, uint64_t cap_y, hipStream_t s)
{
    if (!n)
        return hipSuccess;
    uint32_t nb = (uint32_t)((n + SCAN_TILE - 1) / SCAN_TILE);
    hipLaunchKernelGGL(k_scan_reduce<T>, dim3(nb), dim3(SCAN_THREADS), 0, s, in, n, tmp);
    if (nb <= SCAN_CARRY_BLOCKS) {
        hipLaunchKernelGGL((k_scan_down<T, true>), dim3(nb), dim3(SCAN_THREADS), 0, s, in, n,
                           tmp, out, status, cap_x, cap_y);
    } else {
        hipLaunchKernelGGL(k_scan_sums<T>, dim3(1), dim3(SCAN_THREADS), 0, s, tmp, nb);
        hipLaunchKernelGGL((k_scan_down<T, false>), dim3(nb), dim3(SCAN_THREADS), 0, s, in, n,
                           tmp, out, status, cap_x, cap_y);
    }
    return hipGetLastError();
}

uint64_t scan_tmp_elems(uint64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }

__global__ void __launch_bounds__(SCAN_THREADS) k_sum_parts(const unsigned long long *parts,
                                                            uint32_t n,
                                                            unsigned long long *status)
{
    __shared__ unsigned long long s_w[SCAN_THREADS / 64];
    unsigned long long x = 0;
    for (uint32_t k = threadIdx.x; k < n; k += SCAN_THREADS)
        x += parts[k];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1)
        x += __shfl_xor(x, o, 64);
    if ((threadIdx.x & 63u) == 0)
        s_w[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SCAN_THREADS / 64; ++w)
            x += s_w[w];
        status[ST_PAIRS] = x;
    }
}

hipError_t scan_lines(const uint2 *in, uint2 *out, uint64_t n, uint2 *tmp,
                      const unsigned long long *parts, uint32_t nparts,
                      unsigned long long *status, hipStream_t s)
{
    // (the capacities of lines and points are the host's business: no overflow here)
    hipError_t e = scan_impl<uint2>(in, out, n, tmp, status, ~0ull, ~0ull, s);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(SCAN_THREADS), 0, s, parts, nparts, status);
    return hipGetLastError();
}

// ---- the draw-order places of a draw's primitives -------------------------------------------
// A wave takes a batch of 1024 input triangles, a workgroup FAN_BATCHES batches.  Bound by the
// bytes: a triangle's counts are 5 bytes here (a word of pairs and a byte of flags), 8 bytes of
// places are written where it draws, and the appended fans' counts are read only where clipping
// made some.  As one element per triangle for the live list and two per triangle for the
// places, 8 bytes each, read twice and written once, the scans of 5.2M triangles (64 views of
// 82k) took 80 us and now take 18; of 1M, 30% of them clipped, 21 and now 11 us; with few
// workgroups both are a chain of loads and scans (150k triangles: 10 us both ways).
constexpr uint32_t FAN_BATCHES = SCAN_THREADS / 64;
static_assert(BATCH == 1024, "16 triangles per lane");
static_assert(BATCH * (MAX_CLIP - 3) < 65536, "a batch's appended fans count in 16 bits");

// The lane's 16 triangles of batch b: words w and flag bytes f of triangles
// 256 r + 4 lane .. + 3 for r = 0 .. 3.
__device__ inline void fan_load(const uint32_t *cnt, const uint8_t *cflag, uint32_t b,
                                uint32_t lane, uint4 (&w)[4], uint32_t (&f)[4])
{
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
        w[r] = reinterpret_cast<const uint4 *>(cnt)[(size_t)b * 256 + r * 64 + lane];
        f[r] = reinterpret_cast<const uint32_t *>(cflag)[(size_t)b * 256 + r * 64 + lane];
    }
}

__device__ inline uint32_t item(const uint4 &w, int i)
{
    return i == 0 ? w.x : (i == 1 ? w.y : (i == 2 ? w.z : w.w));
}

// The appended counts of the same triangles, two to a uint4; the loads leave together.
__device__ inline void fan_load_appended(const uint2 *app, uint32_t b, uint32_t lane,
                                         uint4 (&q)[4][2])
{
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 2; ++k)
            q[r][k] = reinterpret_cast<const uint4 *>(
                app + (size_t)b * BATCH + r * 256 + 4 * lane)[k];
}

// Triangle i's appended counts, 0 where there are none.
__device__ inline uint2 appended(const uint4 (&q)[2], uint32_t f, int i)
{
    const bool has = (f >> (8 * i)) & COUNT_APPENDS;
    const uint4 &h = q[i >> 1];
    return make_uint2(has ? (i & 1 ? h.z : h.x) : 0u, has ? (i & 1 ? h.w : h.y) : 0u);
}

__device__ inline bool fan_appends(const uint32_t (&f)[4])
{
    return __ballot((f[0] | f[1] | f[2] | f[3]) & (COUNT_APPENDS * 0x01010101u)) != 0ull;
}

// {primitives, pairs, live} of the lane's triangles, appended ones (any) included.
__device__ inline uint4 fan_sum(const uint4 (&w)[4], const uint32_t (&f)[4], bool any,
                                const uint4 (&q)[4][2])
{
    uint4 t = szero<uint4>();
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t c = item(w[r], i);
            t.x += c ? 1u : 0u;
            t.y += c;
            t.z += (f[r] >> (8 * i)) & COUNT_LIVE ? 1u : 0u;
        }
    if (any) {
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint2 x = appended(q[r], f[r], i);
                t.x += x.x >> 16;
                t.y += x.y;
            }
    }
    return t;
}

// The lane's share of batch b's sum.
__device__ inline uint4 batch_sum(const uint32_t *cnt, const uint8_t *cflag, const uint2 *app,
                                  uint32_t b, uint32_t lane)
{
    uint4 w[4], q[4][2];
    uint32_t f[4];
    fan_load(cnt, cflag, b, lane, w, f);
    const bool any = fan_appends(f);
    if (any)
        fan_load_appended(app, b, lane, q);
    return fan_sum(w, f, any, q);
}

__device__ inline uint32_t wave_sum(uint32_t v)
{
    return __builtin_amdgcn_readlane(wave_incl(v), 63);
}
__device__ inline uint4 wave_sum(uint4 v)
{
    return make_uint4(wave_sum(v.x), wave_sum(v.y), wave_sum(v.z), 0u);
}

__global__ void __launch_bounds__(SCAN_THREADS) k_fan_reduce(const uint32_t *cnt,
                                                           const uint8_t *cflag,
                                                           const uint2 *app, uint32_t batches,
                                                           uint4 *sums)
{
    __shared__ uint4 s_w[FAN_BATCHES];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t b = blockIdx.x * FAN_BATCHES + wv;
    uint4 t = wave_sum(b < batches ? batch_sum(cnt, cflag, app, b, lane) : szero<uint4>());
    if (lane == 0)
        s_w[wv] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < FAN_BATCHES; ++k)
            t = sadd(t, s_w[k]);
        sums[blockIdx.x] = t;
    }
}

// CARRY: what lies before the workgroup is FAN_COUNTS: added up here from the counts
// themselves, FAN_SUMS: from the workgroups' sums, FAN_SCANNED: already scanned.
constexpr int FAN_COUNTS = 0, FAN_SUMS = 1, FAN_SCANNED = 2;

template <int CARRY>
__global__ void __launch_bounds__(SCAN_THREADS) k_fan_down(
    const uint32_t *cnt, const uint8_t *cflag, const uint2 *app, uint32_t batches,
    const uint4 *sums, uint2 *ex, uint4 *app_ex, uint32_t *live, unsigned long long *status,
    uint64_t cap_prims, uint64_t cap_pairs)
{
    __shared__ uint4 s_own[FAN_BATCHES], s_carry[FAN_BATCHES];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t b = blockIdx.x * FAN_BATCHES + wv;
    uint4 w[4];
    uint32_t f[4];
    uint4 carry = szero<uint4>(), own = szero<uint4>();
    uint4 xq[4][2];
    bool any = false;
    const bool mine = b < batches;
    if (mine) {
        fan_load(cnt, cflag, b, lane, w, f);
        any = fan_appends(f);
        if (any)
            fan_load_appended(app, b, lane, xq);
        own = fan_sum(w, f, any, xq);
    }
    if (CARRY == FAN_COUNTS) {
        for (uint32_t k = wv; k < blockIdx.x * FAN_BATCHES; k += FAN_BATCHES)
            carry = sadd(carry, batch_sum(cnt, cflag, app, k, lane));
    } else if (CARRY == FAN_SUMS) {
        for (uint32_t k = threadIdx.x; k < blockIdx.x; k += SCAN_THREADS)
            carry = sadd(carry, sums[k]);
    } else if (threadIdx.x == 0) {
        carry = sums[blockIdx.x];
    }
    carry = wave_sum(carry);
    own = wave_sum(own);
    if (lane == 0) {
        s_carry[wv] = carry;
        s_own[wv] = own;
    }
    __syncthreads();
    if (!mine)
        return;
    uint4 run = szero<uint4>();
#pragma unroll
    for (uint32_t k = 0; k < FAN_BATCHES; ++k) {
        run = sadd(run, s_carry[k]);
        if (k < wv)
            run = sadd(run, s_own[k]);
    }
    if (b + 1 == batches && lane == 0) {
        const uint4 t = sadd(run, own);
        publish_totals(make_uint2(t.x, t.y), status, cap_prims, cap_pairs);
        if (live)
            status[ST_LIVE] = t.z;
    }
    // the first fan triangles and the live list
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
        const uint32_t t0 = b * (uint32_t)BATCH + r * 256 + 4 * lane;
        uint2 s = make_uint2(0u, 0u);  // {primitives | live << 16, pairs}
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t c = item(w[r], i), g = f[r] >> (8 * i);
            s.x += (c ? 1u : 0u) | (g & COUNT_LIVE ? 0x10000u : 0u);
            s.y += c;
        }
        const uint2 inc = wave_incl(s);
        uint32_t p = run.x + ((inc.x - s.x) & 0xFFFFu), q = run.y + (inc.y - s.y),
                 l = run.z + ((inc.x - s.x) >> 16);
        uint2 o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t c = item(w[r], i), g = f[r] >> (8 * i);
            o[i] = make_uint2(p, q);
            p += c ? 1u : 0u;
            q += c;
            if (live && (g & COUNT_LIVE))
                live[l++] = t0 + i;
        }
        if (s.y) {  // some of the four draw
            uint4 *to = reinterpret_cast<uint4 *>(ex + t0);
            to[0] = make_uint4(o[0].x, o[0].y, o[1].x, o[1].y);
            to[1] = make_uint4(o[2].x, o[2].y, o[3].x, o[3].y);
        }
        const uint32_t tx = __builtin_amdgcn_readlane(inc.x, 63);
        run.x += tx & 0xFFFFu;
        run.y += __builtin_amdgcn_readlane(inc.y, 63);
        run.z += tx >> 16;
    }
    // the appended ones
    if (!any)
        return;
    uint32_t before = 0;  // fans the batch has appended
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
        const uint32_t t0 = b * (uint32_t)BATCH + r * 256 + 4 * lane;
        const uint32_t fr = f[r];
        uint2 x[4], s = make_uint2(0u, 0u);  // {fans | drawn ones << 16, pairs}
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = appended(xq[r], fr, i);
            s = sadd(s, x[i]);
        }
        const uint2 inc = wave_incl(s);
        uint2 at = ssub(inc, s);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if ((fr >> (8 * i)) & COUNT_APPENDS)
                app_ex[t0 + i] = make_uint4(run.x + (at.x >> 16), run.y + at.y,
                                            before + (at.x & 0xFFFFu), 0u);
            at = sadd(at, x[i]);
        }
        const uint32_t tx = __builtin_amdgcn_readlane(inc.x, 63);
        run.x += tx >> 16;
        run.y += __builtin_amdgcn_readlane(inc.y, 63);
        before += tx & 0xFFFFu;
    }
}

static uint32_t fan_blocks(uint64_t batches)
{
    return (uint32_t)((batches + FAN_BATCHES - 1) / FAN_BATCHES);
}

size_t fan_scan_bytes(uint64_t batches) { return ((size_t)fan_blocks(batches) + 1) * 16; }

// Draws of up to this many workgroups (16k triangles) take one launch: adding up what lies
// before costs the last workgroup 60 KB of reads that hit the L2 (5 bytes for each of 12,288
// triangles; at most 96 KB more where clipping appends fans), a launch some 5 us.
constexpr uint32_t FAN_ONE_PASS = 4;

hipError_t scan_fans(const uint32_t *cnt, const uint8_t *cflag, const uint2 *app, uint2 *ex,
                     uint4 *app_ex, uint32_t *live, uint64_t batches, void *tmp,
                     unsigned long long *status, uint64_t cap_prims, uint64_t cap_pairs,
                     hipStream_t s)
{
    if (!batches)
        return hipSuccess;
    uint4 *sums = static_cast<uint4 *>(tmp);
    const uint32_t nb = fan_blocks(batches), n = (uint32_t)batches;
    const dim3 g(nb), t(SCAN_THREADS);
    if (nb <= FAN_ONE_PASS) {
        hipLaunchKernelGGL(k_fan_down<FAN_COUNTS>, g, t, 0, s, cnt, cflag, app, n, sums, ex,
                           app_ex, live, status, cap_prims, cap_pairs);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_fan_reduce, g, t, 0, s, cnt, cflag, app, n, sums);
    if (nb <= SCAN_CARRY_BLOCKS) {
        hipLaunchKernelGGL(k_fan_down<FAN_SUMS>, g, t, 0, s, cnt, cflag, app, n, sums, ex,
                           app_ex, live, status, cap_prims, cap_pairs);
    } else {
        hipLaunchKernelGGL(k_scan_sums<uint4>, dim3(1), t, 0, s, sums, nb);
        hipLaunchKernelGGL(k_fan_down<FAN_SCANNED>, g, t, 0, s, cnt, cflag, app, n, sums, ex,
                           app_ex, live, status, cap_prims, cap_pairs);
    }
    return hipGetLastError();
}

// ---- radix sort of (tile, primitive) pairs ---------------------------------------------
constexpr int RADIX_THREADS = 256;

// Pass 0 reads the emitted pairs (ST_PAIRS slots: compacted per expansion chunk, or one run
// with rejected pairs keyed >= tiles, which it drops); later passes and the ranges read the
// kept ones (ST_KEPT).
__device__ inline uint64_t pair_count(const unsigned long long *status, int word)
{
    return (status[ST_OVERFLOW] | status[ST_ERROR]) ? 0 : status[word];
}

__device__ inline void chunk_of(const unsigned long long *status, int word, uint32_t G, uint32_t b,
                                uint64_t &beg, uint64_t &end)
{
    uint64_t m = pair_count(status, word);
    uint64_t ch = (m + G - 1) / G;
    beg = (uint64_t)b * ch;
    end = beg + ch;
    if (beg > m) beg = m;
    if (end > m) end = m;
}

// The expansion's output: chunk c of `size` slots holds its kept[c] pairs at its start
// (the tiles a primitive cannot shade are already dropped).  Radix block b of G owns the
// chunks [k0, k1) and reads their pairs in order as one run, RADIX_THREADS chunks at a
// time: s_off holds the group's exclusive prefix of kept counts, a run position maps to its
// chunk by a binary search.
struct Chunks {
    const uint32_t *kept;  // nullptr: the pairs are one contiguous run (chunk_of)
    uint32_t size;
};

__device__ inline void chunks_of(const unsigned long long *status, uint32_t size, uint32_t G,
                                 uint32_t b, uint64_t &k0, uint64_t &k1)
{
    const uint64_t m = pair_count(status, ST_PAIRS);
    const uint64_t n = (m + size - 1) / size, per = (n + G - 1) / G;
    k0 = (uint64_t)b * per;
    k1 = k0 + per;
    if (k0 > n) k0 = n;
    if (k1 > n) k1 = n;
}

// Loads the kept counts of chunks [g0, g0 + RADIX_THREADS) ∩ [., k1) and their exclusive
// prefix into s_off[0 .. RADIX_THREADS]; returns the group's chunk count.
__device__ inline uint32_t load_chunk_group(const Chunks &ch, uint64_t g0, uint64_t k1,
                                            uint32_t *s_off)
{
    const uint32_t nk = (uint32_t)(k1 - g0 < RADIX_THREADS ? k1 - g0 : RADIX_THREADS);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    __shared__ uint32_t s_w[RADIX_THREADS / 64];
    const uint32_t c = tid < nk ? ch.kept[g0 + tid] : 0u;
    const uint32_t inc = wave_incl(c);
    if (lane == 63)
        s_w[w] = inc;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < RADIX_THREADS / 64; ++k) {
        pre += k < (int)w ? s_w[k] : 0u;
        tot += s_w[k];
    }
    s_off[tid] = pre + inc - c;
    if (tid == 0)
        s_off[RADIX_THREADS] = tot;
    __syncthreads();
    return nk;
}

// The slot of run position v of the group (v < s_off[nk]).
__device__ inline uint64_t chunk_slot(const Chunks &ch, uint64_t g0, uint32_t nk,
                                      const uint32_t *s_off, uint32_t v)
{
    uint32_t lo = 0, hi = nk;  // last chunk with s_off <= v
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_off[mid] <= v)
            lo = mid;
        else
            hi = mid;
    }
    return (g0 + lo) * (uint64_t)ch.size + (v - s_off[lo]);
}

__global__ void __launch_bounds__(RADIX_THREADS) k_radix_hist(const uint32_t *keys,
                                                            const unsigned long long *status,
                                                            int word, TileDigit digit,
                                                            uint32_t tiles, uint32_t *hist,
                                                            Chunks ch, int rows)
{
    __shared__ uint32_t h[256];
    __shared__ uint32_t s_off[RADIX_THREADS + 1];
    const uint32_t G = gridDim.x, b = blockIdx.x;
    h[threadIdx.x] = 0;
    __syncthreads();
    if (ch.kept) {
        uint64_t k0, k1;
        chunks_of(status, ch.size, G, b, k0, k1);
        for (uint64_t g0 = k0; g0 < k1; g0 += RADIX_THREADS) {
            const uint32_t nk = load_chunk_group(ch, g0, k1, s_off);
            const uint32_t tot = s_off[RADIX_THREADS];
            for (uint32_t v = threadIdx.x; v < tot; v += RADIX_THREADS) {
                const uint32_t k = keys[chunk_slot(ch, g0, nk, s_off, v)];
                if (k < tiles)
                    atomicAdd(&h[digit.of(k)], 1u);
            }
            __syncthreads();  // s_off is reloaded by the next group
        }
    } else {
        uint64_t beg, end;
        chunk_of(status, word, G, b, beg, end);
        for (uint64_t i = beg + threadIdx.x; i < end; i += RADIX_THREADS) {
            uint32_t k = keys[i];
            if (k < tiles)
                atomicAdd(&h[digit.of(k)], 1u);
        }
    }
    __syncthreads();
    // rows: a row of 256 per block (the scatter adds them up), else a row of G per digit
    hist[rows ? (size_t)b * 256 + threadIdx.x : (size_t)threadIdx.x * G + b] = h[threadIdx.x];
}

// Digit d's counts over the G blocks (at most 1024), scanned in place (exclusive); the
// digit's total goes to tot[d].
__global__ void __launch_bounds__(RADIX_THREADS) k_radix_scan(uint32_t *hist, uint32_t G,
                                                              uint32_t *tot)
{
    uint32_t *row = hist + (size_t)blockIdx.x * G;
    const uint32_t t = threadIdx.x;
    uint32_t v[4], acc = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        v[k] = t * 4 + k < G ? row[t * 4 + k] : 0u;
        acc += v[k];
    }
    uint32_t total;
    uint32_t run = block_exclusive<uint32_t>(acc, &total);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (t * 4 + k < G)
            row[t * 4 + k] = run;
        run += v[k];
    }
    if (t == 0)
        tot[blockIdx.x] = total;
}

// Stable scatter of one pass: RADIX_ITEMS chunks of RADIX_THREADS pairs per round, chunk j
// element tid at base + j * RADIX_THREADS + tid.  A pair's position is the digit's running
// offset plus the count of its digit in earlier chunks, in earlier waves of its chunk, and
// in lower lanes of its wave (eight ballots find the lanes with the same digit).
constexpr int RADIX_ITEMS = 4;

// One round of RADIX_ITEMS * RADIX_THREADS pairs: run positions [base, end), position i at
// slot slot_of(i); run[] carries each digit's next output position between rounds.
template <class SlotOf>
__device__ inline void scatter_round(const uint32_t *keys, const uint32_t *vals, uint32_t *okeys,
                                     uint32_t *ovals, TileDigit digit, uint32_t tiles,
                                     uint64_t cap, uint64_t base, uint64_t end, SlotOf slot_of, uint32_t *run,
                                     uint32_t (*wcnt)[RADIX_THREADS / 64][256],
                                     uint32_t (*off)[RADIX_THREADS / 64][256])
{
    constexpr int NW = RADIX_THREADS / 64;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    {
        uint32_t k[RADIX_ITEMS], v[RADIX_ITEMS], d[RADIX_ITEMS], rank[RADIX_ITEMS];
        bool valid[RADIX_ITEMS];
#pragma unroll
        for (int j = 0; j < RADIX_ITEMS; ++j) {
            const uint64_t i = base + (uint64_t)j * RADIX_THREADS + tid;
            const uint64_t slot = i < end ? slot_of(i) : 0;
            k[j] = i < end ? keys[slot] : 0u;
            valid[j] = i < end && k[j] < tiles;
            v[j] = valid[j] ? vals[slot] : 0u;
            d[j] = digit.of(k[j]);
        }
#pragma unroll
        for (int j = 0; j < RADIX_ITEMS; ++j) {
            unsigned long long m = __ballot(valid[j]);
#pragma unroll
            for (int bit = 0; bit < 8; ++bit) {
                const unsigned long long bb = __ballot((d[j] >> bit) & 1u);
                m &= ((d[j] >> bit) & 1u) ? bb : ~bb;
            }
            rank[j] = (uint32_t)__popcll(m & below);
            if (valid[j] && rank[j] == 0)
                wcnt[j][w][d[j]] = (uint32_t)__popcll(m);
        }
        __syncthreads();
        {
            uint32_t acc = run[tid];
#pragma unroll
            for (int j = 0; j < RADIX_ITEMS; ++j)
#pragma unroll
                for (int q = 0; q < NW; ++q) {
                    off[j][q][tid] = acc;
                    acc += wcnt[j][q][tid];
                    wcnt[j][q][tid] = 0;
                }
            run[tid] = acc;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < RADIX_ITEMS; ++j) {
            if (!valid[j])
                continue;
            const uint32_t pos = off[j][w][d[j]] + rank[j];
            if (pos < cap) {
                okeys[pos] = k[j];
                ovals[pos] = v[j];
            }
        }
    }
}

__global__ void __launch_bounds__(RADIX_THREADS) k_radix_scatter(
    const uint32_t *keys, const uint32_t *vals, uint32_t *okeys, uint32_t *ovals,
    unsigned long long *status, int word, TileDigit digit, uint32_t tiles, const uint32_t *hist,
    uint32_t *tot, Chunks ch, int rows)
{
    constexpr int NW = RADIX_THREADS / 64;
    __shared__ uint32_t run[256];
    __shared__ uint32_t wcnt[RADIX_ITEMS][NW][256];  // per (chunk, wave, digit) counts
    __shared__ uint32_t off[RADIX_ITEMS][NW][256];   // their exclusive prefix from run
    const uint32_t G = gridDim.x, b = blockIdx.x;
    const int tid = threadIdx.x;
    // digit tid's first position in this block: the totals of the digits below it, and its
    // counts in the blocks before (rows: added up here, else scanned by k_radix_scan)
    uint32_t mine = 0, total = 0;
    if (rows) {
        for (uint32_t r0 = 0; r0 < G; r0 += 8) {
            uint32_t c[8];  // eight rows' loads in flight
#pragma unroll
            for (uint32_t r = 0; r < 8; ++r)
                c[r] = r0 + r < G ? hist[(size_t)(r0 + r) * 256 + tid] : 0u;
#pragma unroll
            for (uint32_t r = 0; r < 8; ++r) {
                mine += r0 + r < b ? c[r] : 0u;
                total += c[r];
            }
        }
    } else {
        mine = hist[(size_t)tid * G + b];
        total = tot[tid];
    }
    uint32_t kept;
    run[tid] = block_exclusive<uint32_t>(total, &kept) + mine;
    if (b == 0) {
        if (rows)
            tot[tid] = total;
        if (tid == 0 && word == ST_PAIRS)  // the first pass drops the rejected pairs
            status[ST_KEPT] = kept;
    }
#pragma unroll
    for (int j = 0; j < RADIX_ITEMS; ++j)
#pragma unroll
        for (int q = 0; q < NW; ++q)
            wcnt[j][q][tid] = 0;
    __syncthreads();
    const uint64_t cap = pair_count(status, ST_PAIRS);
    if (ch.kept) {
        __shared__ uint32_t s_off[RADIX_THREADS + 1];
        uint64_t k0, k1;
        chunks_of(status, ch.size, G, b, k0, k1);
        for (uint64_t g0 = k0; g0 < k1; g0 += RADIX_THREADS) {
            const uint32_t nk = load_chunk_group(ch, g0, k1, s_off);
            const uint32_t tot = s_off[RADIX_THREADS];
            for (uint64_t base = 0; base < tot; base += (uint64_t)RADIX_THREADS * RADIX_ITEMS)
                scatter_round(keys, vals, okeys, ovals, digit, tiles, cap, base, tot,
                              [&](uint64_t i) { return chunk_slot(ch, g0, nk, s_off, (uint32_t)i); },
                              run, wcnt, off);
            __syncthreads();  // s_off is reloaded by the next group
        }
    } else {
        uint64_t beg, end;
        chunk_of(status, word, G, b, beg, end);
        for (uint64_t base = beg; base < end; base += (uint64_t)RADIX_THREADS * RADIX_ITEMS)
            scatter_round(keys, vals, okeys, ovals, digit, tiles, cap, base, end,
                          [](uint64_t i) { return i; }, run, wcnt, off);
    }
}

// One bucket: the pairs of the tiles that swr_buckets.h deals to bucket blockIdx.x, a run of the
// scatter's output (tot: the buckets' lengths).  Each wave owns a contiguous piece of the run: it
// counts its pairs per tile (the id's bits above the low 8: `bits` of them), the counts of all
// waves scanned tile by tile give every (wave, tile) its first position, and the wave walks its
// piece again, placing its pairs in order.  The tiles' ranges are written whether they hold
// pairs or not.  A bucket's time grows with its run, so the runs must not differ much: tiles
// that lie together on the screen lie in different buckets.
__global__ void __launch_bounds__(1024) k_bucket(const uint32_t *keys, const uint32_t *vals,
                                                 uint32_t *ovals, unsigned long long *status,
                                                 const uint32_t *tot, int bits, uint32_t tiles,
                                                 uint32_t *ranges, StatusOut out)
{
    extern __shared__ uint32_t s_cnt[];  // [waves][1 << bits]
    __shared__ uint32_t s_w[16];
    if (blockIdx.x == 0 && threadIdx.x < 64)
        hand_over_status(status, out);
    if (status[ST_OVERFLOW] | status[ST_ERROR])
        return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6, W = blockDim.x >> 6;
    const uint32_t nv = 1u << bits, bucket = blockIdx.x;
    const auto block_excl = [&](uint32_t v, uint32_t *total) {
        const uint32_t inc = wave_incl(v);
        if (lane == 63)
            s_w[w] = inc;
        __syncthreads();
        uint32_t pre = 0, all = 0;
        for (uint32_t k = 0; k < W; ++k) {
            const uint32_t x = s_w[k];
            pre += k < w ? x : 0u;
            all += x;
        }
        __syncthreads();
        *total = all;
        return pre + inc - v;
    };
    uint32_t beg;
    (void)block_excl(tid < 256 && tid < bucket ? tot[tid] : 0u, &beg);
    const uint32_t n = tot[bucket];
    uint32_t *cnt = s_cnt + (w << bits);
    for (uint32_t v = lane; v < nv; v += 64)
        cnt[v] = 0u;
    lds_sync();
    const uint32_t per = ((n + W - 1) / W + 63u) & ~63u;
    const uint32_t p0 = w * per < n ? w * per : n, p1 = p0 + per < n ? p0 + per : n;
    constexpr uint32_t U = 4;  // loads in flight
    for (uint32_t i0 = p0; i0 < p1; i0 += 64 * U) {
        uint32_t k[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = i0 + 64 * u + lane;
            k[u] = i < p1 ? keys[beg + i] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (i0 + 64 * u + lane < p1)
                atomicAdd(&cnt[k[u] >> 8], 1u);
    }
    __syncthreads();
    uint32_t base = beg;
    for (uint32_t v0 = 0; v0 < nv; v0 += blockDim.x) {
        const uint32_t v = v0 + tid;
        uint32_t sum = 0, all;
        if (v < nv)
            for (uint32_t q = 0; q < W; ++q)
                sum += s_cnt[(q << bits) + v];
        uint32_t at = base + block_excl(sum, &all);
        if (v < nv) {
            const uint32_t tile = bucket_tile(bucket, v);
            if (tile < tiles) {
                ranges[2 * (size_t)tile] = at;
                ranges[2 * (size_t)tile + 1] = at + sum;
            }
            for (uint32_t q = 0; q < W; ++q) {
                const uint32_t c = s_cnt[(q << bits) + v];
                s_cnt[(q << bits) + v] = at;
                at += c;
            }
        }
        base += all;
    }
    __syncthreads();
    for (uint32_t i0 = p0; i0 < p1; i0 += 64 * U) {
        uint32_t k[U], x[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = i0 + 64 * u + lane;
            k[u] = i < p1 ? keys[beg + i] >> 8 : 0u;
            x[u] = i < p1 ? vals[beg + i] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const bool valid = i0 + 64 * u + lane < p1;
            unsigned long long m = __ballot(valid);
            if (m == 0ull)
                break;
            for (int bit = 0; bit < bits; ++bit) {
                const bool one = (k[u] >> bit) & 1u;
                const unsigned long long bb = __ballot(one);
                m &= one ? bb : ~bb;
            }
            const uint32_t rank = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            const uint32_t at = valid ? cnt[k[u]] : 0u;
            lds_sync();  // every lane has read its tile's position
            if (valid) {
                if (rank == 0)
                    cnt[k[u]] = at + (uint32_t)__popcll(m);
                ovals[at + rank] = x[u];
            }
            lds_sync();
        }
    }
}

// Per-tile [begin, end) into the sorted kept pairs; tiles without pairs keep the zeros the
// begin kernel wrote.
__global__ void __launch_bounds__(256) k_ranges(const uint32_t *keys, unsigned long long *status,
                                              uint32_t *ranges, StatusOut out)
{
    if (blockIdx.x == 0 && threadIdx.x < 64)
        hand_over_status(status, out);
    uint64_t m = pair_count(status, ST_KEPT);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
         i += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t k = keys[i];
        if (i == 0 || keys[i - 1] != k)
            ranges[2 * (size_t)k] = (uint32_t)i;
        if (i == m - 1 || keys[i + 1] != k)
            ranges[2 * (size_t)k + 1] = (uint32_t)(i + 1);
    }
}

// Bits that tell `tiles` tile ids apart, at least 1.
static int radix_bits(uint32_t tiles)
{
    int bits = 1;
    while (bits < 32 && (1ull << bits) < (unsigned long long)tiles)
        ++bits;
    return bits;
}

// Rejected pairs carry a key >= tiles; every key below `tiles` sorts within the passes.
uint32_t pair_sentinel(uint32_t) { return 0xFFFFFFFFu; }

// Bits of a tile id above the low 8 that k_bucket regroups at most: its counters take
// 4 bytes per wave and value, 64 KB of LDS in all.
constexpr int BUCKET_BITS = 10;
// Blocks up to which the scatter adds up the histogram rows itself (64 rows are 64 KB per
// block from L2, less than a launch costs); beyond it k_radix_scan does.
constexpr uint32_t SCAN_ROWS = 64;

hipError_t sort_pairs(SortBuffers &sb, unsigned long long *status, uint32_t tiles, hipStream_t s)
{
    const int bits = radix_bits(tiles);
    const bool bucket = bits > 8 && bits <= 8 + BUCKET_BITS;
    const int passes = bucket ? 1 : (bits + 7) / 8;
    uint32_t *ka = sb.keys_a, *va = sb.vals_a, *kb = sb.keys_b, *vb = sb.vals_b;
    const int rows = sb.blocks <= SCAN_ROWS ? 1 : 0;
    for (int p = 0; p < passes; ++p) {
        const TileDigit digit = {8 * p, bucket};
        const int word = p == 0 ? ST_PAIRS : ST_KEPT;
        // pass 0 reads the expansion's chunks (when it compacted them), later passes one run
        Chunks ch{p == 0 ? sb.chunk_kept : nullptr, sb.chunk};
        hipLaunchKernelGGL(k_radix_hist, dim3(sb.blocks), dim3(RADIX_THREADS), 0, s, ka, status,
                           word, digit, tiles, sb.hist, ch, rows);
        if (!rows)
            hipLaunchKernelGGL(k_radix_scan, dim3(256), dim3(RADIX_THREADS), 0, s, sb.hist,
                               sb.blocks, sb.tot);
        hipLaunchKernelGGL(k_radix_scatter, dim3(sb.blocks), dim3(RADIX_THREADS), 0, s, ka, va, kb,
                           vb, status, word, digit, tiles, sb.hist, sb.tot, ch, rows);
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    sb.ranged = bucket;
    if (bucket) {
        // a wave per 64 pairs or so of an average bucket, 4 to 16 waves that fit the LDS
        const int high = bits - 8;
        const uint32_t most = (64u << 10) / (4u << high);
        uint32_t waves = sb.blocks > SCAN_ROWS ? 16 : 4;
        waves = waves < most ? waves : most;
        hipLaunchKernelGGL(k_bucket, dim3(256), dim3(64 * waves), (4u * waves) << high, s, ka, va,
                           vb, status, sb.tot, high, tiles, sb.ranges, sb.out);
        std::swap(va, vb);
    }
    sb.sorted_keys = ka;
    sb.sorted_vals = va;
    return hipGetLastError();
}

hipError_t launch_ranges(const SortBuffers &sb, unsigned long long *status, uint32_t tiles,
                         hipStream_t s)
{
    (void)tiles;
    if (sb.ranged)
        return hipSuccess;
    hipLaunchKernelGGL(k_ranges, dim3(1024), dim3(256), 0, s, sb.sorted_keys, status, sb.ranges,
                       sb.out);
    return hipGetLastError();
}

}  // namespace swr
