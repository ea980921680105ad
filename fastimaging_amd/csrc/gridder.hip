// Convolutional gridding for gfx950: the scatter-add of convolve_to_grid
// (src/stp/gridder/gridder.h:240-997) as a tile-binned gather.
//
//  1. grid_count   : per visibility, the reference's pre-processing (half-plane
//                    conversion gridder.cpp:11-37, rint centre/fraction
//                    gridder.h:377-386, bounds check gridder.cpp:202-217, uv shift
//                    gridder.h:399-413, oversampled index gridder.cpp:219-241);
//                    counts the (visibility pass, grid tile) pairs it touches and
//                    sums the good weights in the canonical order.
//  2. tile_scan    : exclusive scan of the per-tile counts.
//  3. grid_scatter : writes one 40-byte entry per (pass, tile) pair, binned by tile.
//  4. grid_tiles   : one workgroup per TILE_R x TILE_C tile sums every entry's
//                    taps that fall inside it on the FP64 matrix cores, then
//                    writes the whole tile once: no atomics, no memset.
// Per tap the arithmetic is the reference's: kval = K * w, grid += vis * kval,
// beam += kval (gridder.h:854-858); the oversampled kernel is the separable
// product ky[row] * kx[col] of normalised 1-D kernels (gridder.h:84-102).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "gridder.h"
#include "fft.h"
#include "kernel_tables.h"
#include "reduce.h"

namespace stp_hip {
namespace {

constexpr int TILE_R = 64;  // grid rows (v) per tile: 64 contiguous complex per column
static_assert(TILE_R == OCC_ROWS, "rows of TileOcc");
constexpr int W_TILE_C = 64; // with W-projection: its wide footprints touch fewer tiles
constexpr int TILE_C = 32;  // default grid columns (u) per tile; GridderArgs::tile_cols overrides
constexpr int GWG = 256;

struct GridGeom {
    int N, rows, half, s, ks, os;
    int halfplane, shift, exact, beam;
    int bpack = 0; // beam grid packed real (rows x N/2 complex: columns 2u', 2u'+1)
    int skip = 0;  // cells of tiles without entries are not written
    int tiles_r, tiles_c;
    int tc;       // tile width in grid columns (TILE_R rows per tile)
    double scale;
    long long n;
    int kfunc;
    double kparam, kwg, kws;
    // W-projection: the inputs are in |w| order, visibility k lies in plane[k]
    int wproj = 0;
    const uint16_t* plane = nullptr;
    const int* psup = nullptr; // truncated support of each plane (null: s)
    int planes = 0;            // truncated planes, where the tile sums may take phases; they do
    double phase_taps = 0.0;   // from this many taps of one kernel of each plane, added up
};

struct Entry {
    int gx, gy;   // kernel centre on the (shifted) grid for this pass
    int cp;       // cp_x | cp_y << 16 (oversampled kernel indices); W-projection: the support, bit 31 = conjugate
                  // kernel, bits 30 and 29 = rows and columns of the sub-kernel mirrored
    int idx;      // visibility index << 1 | pass; W-projection: the W sub-kernel (plane, |y| offset, |x| offset)
    double vr, vi, w; // W-projection: vr, vi are the visibility times w
};
static_assert(sizeof(Entry) == 40, "entry layout");

struct Prep {
    int good, dup;
    int gx, gy, cpx, cpy;
    double fx, fy;
    double vr, vi, w;
    double wl;   // w (wavelengths) after the half-plane conversion (W-projection)
};

// The inputs of one visibility (loads only, so that several can be in flight).
struct VisIn {
    double u, v, vr, vi, w, wl;
};

__device__ __forceinline__ VisIn load_vis(const GridGeom& g, const double* uv, const double* vis, const double* wts, long long k)
{
    VisIn r;
    r.u = uv[k];
    r.v = uv[g.n + k];
    r.vr = vis[2 * k];
    r.vi = vis[2 * k + 1];
    r.w = wts[k];
    r.wl = g.wproj ? uv[2 * g.n + k] : 0.0;
    return r;
}

__device__ __forceinline__ Prep prep_in(const GridGeom& g, const VisIn& r)
{
    Prep p;
    double u = r.u * g.scale;
    double v = r.v * g.scale;
    p.vr = r.vr;
    p.vi = r.vi;
    p.w = r.w;
    p.dup = 0;
    p.wl = r.wl;
    p.good = (fabs(u) < 1.0e9 && fabs(v) < 1.0e9) ? 1 : 0; // also rejects NaN
    if (!p.good)
        u = v = 0.0;
    if (g.halfplane) {
        if (v < 0.0) {
            p.dup = (v > -(g.s + 1)) ? 1 : 0;
            u = -u;
            v = -v;
            p.vi = -p.vi;
            p.wl = -p.wl; // gridder.cpp:39-66
        } else {
            p.dup = (v < (g.s + 1)) ? 1 : 0;
        }
    }
    const int ku = int(rint(u)), kv = int(rint(v));
    p.fx = u - ku;
    p.fy = v - kv;
    int kx = ku + g.half, ky = kv + g.half;
    if ((kx - g.s) <= 0 || (ky - g.s) <= 0 || (kx + g.s) >= g.N || (ky + g.s) >= g.N)
        p.good = 0;
    if (g.shift) {
        kx = (kx < g.half) ? kx + g.half : kx - g.half;
        ky = (ky < g.half) ? ky + g.half : ky - g.half;
    }
    p.gx = kx;
    p.gy = ky;
    const int rmax = g.os / 2;
    int cx = int(rint(p.fx * g.os)), cy = int(rint(p.fy * g.os));
    cx = cx > rmax ? rmax : (cx < -rmax ? -rmax : cx);
    cy = cy > rmax ? rmax : (cy < -rmax ? -rmax : cy);
    p.cpx = cx + rmax;
    p.cpy = cy + rmax;
    return p;
}

__device__ __forceinline__ Prep prep_vis(const GridGeom& g, const double* uv, const double* vis, const double* wts, long long k)
{
    return prep_in(g, load_vis(g, uv, vis, wts, k));
}

// Centre / kernel indices of pass `pass` (1 = conjugate copy, gridder.h:794-805).
__device__ __forceinline__ void pass_geom(const GridGeom& g, const Prep& p, int pass, int& gx, int& gy, int& cpx, int& cpy)
{
    gx = p.gx;
    gy = p.gy;
    cpx = p.cpx;
    cpy = p.cpy;
    if (pass) {
        gx = g.N - p.gx;
        gy = g.N - p.gy;
        if (g.os > 1) {
            cpx = g.os - p.cpx;
            cpy = g.os - p.cpy;
        }
    }
}

// Support of visibility position k's kernel.
__device__ __forceinline__ int plane_support(const GridGeom& g, long long k) { return g.psup ? g.psup[g.plane[k]] : g.s; }

// Entry of visibility position k, pass `pass`.  The conjugate pass conjugates the
// visibility and negates w (gridder.h:794-805); a negative w selects the
// conjugate W-kernel (gridder.h:826-843).
__device__ __forceinline__ Entry make_entry(const GridGeom& g, const Prep& p, int pass, long long k)
{
    int gx, gy, cpx, cpy;
    pass_geom(g, p, pass, gx, gy, cpx, cpy);
    Entry e;
    e.gx = gx;
    e.gy = gy;
    e.cp = cpx | (cpy << 16);
    e.vr = p.vr;
    e.vi = pass ? -p.vi : p.vi;
    e.w = p.w;
    if (g.wproj) {
        const double wl = pass ? -p.wl : p.wl;
        // the W tile kernel takes the sub-kernel index and the visibility times its weight;
        // the plane's kernel is even, so the offset -y is offset y read backwards
        const int op = g.os / 2;
        const int y = min(cpy, 2 * op - cpy), x = min(cpx, 2 * op - cpx);
        e.idx = (int(g.plane[k]) * (op + 1) + y) * (op + 1) + x;
        e.cp = int(uint32_t(plane_support(g, k)) | (wl < 0.0 ? 0x80000000u : 0u) | (cpy > op ? 0x40000000u : 0u) |
            (cpx > op ? 0x20000000u : 0u));
        e.vr = e.vr * p.w;
        e.vi = e.vi * p.w;
    } else {
        e.idx = int((k << 1) | pass);
    }
    return e;
}

// Grid row of kernel row i, or -1 if dropped.  Oversampled path: rows < 0 skipped,
// rows >= N wrapped (gridder.h:847-853); exact path wraps both ways (:977-983).
__device__ __forceinline__ int tap_row(const GridGeom& g, int gy, int i)
{
    int r = gy - g.s + i;
    if (r < 0) {
        if (!g.exact)
            return -1;
        r += g.N;
    }
    if (r >= g.N)
        r -= g.N;
    return r < g.rows ? r : -1;
}

// Grid column of kernel column j: (gx + j - s) mod N (gridder.h:807-930, :970-974).
__device__ __forceinline__ int tap_col(const GridGeom& g, int gx, int j)
{
    int c = gx - g.s + j;
    if (c < 0)
        c += g.N;
    if (c >= g.N)
        c -= g.N;
    return c;
}

// The tiles of one axis that hold kept taps of a footprint: three intervals of
// tile indices [lo[k], hi[k]] (empty when lo > hi), one per contiguous piece of
// the raw range [centre - s, centre - s + ks - 1]: below 0, inside, at or above N.
// Pieces of a small grid can share tiles; visit_tiles skips the repeats.
struct TileSpan {
    int lo[3], hi[3];
};

__host__ __device__ __forceinline__ void span_set(TileSpan& sp, int k, int lo, int hi, int w)
{
    const bool on = lo <= hi;
    sp.lo[k] = on ? lo / w : 1;
    sp.hi[k] = on ? hi / w : 0;
}

// Rows: the oversampled path skips rows < 0 and wraps rows >= N, the exact path
// also wraps rows < 0; rows beyond `last` (the half plane) are dropped.
// Columns wrap both ways (the same sets as tap_row / tap_col over every tap).
__host__ __device__ __forceinline__ void footprint_spans(int N, int last, int s, int ks, int exact, int tile_r, int tile_c,
    int gx, int gy, TileSpan& rs, TileSpan& cs)
{
    int a = gy - s, b = a + ks - 1;
    span_set(rs, 0, a + N, (a < 0 && exact) ? min(min(b, -1) + N, last) : -1, tile_r);
    span_set(rs, 1, max(a, 0), min(min(b, N - 1), last), tile_r);
    span_set(rs, 2, max(a, N) - N, (b >= N) ? min(b - N, last) : -1, tile_r);
    a = gx - s;
    b = a + ks - 1;
    span_set(cs, 0, a + N, (a < 0) ? min(b, -1) + N : -1, tile_c);
    span_set(cs, 1, max(a, 0), min(b, N - 1), tile_c);
    span_set(cs, 2, max(a, N) - N, (b >= N) ? b - N : -1, tile_c);
}

// Whether tile t lies in one of the intervals before k.
__host__ __device__ __forceinline__ bool span_seen(const TileSpan& sp, int k, int t)
{
    bool seen = false;
#pragma unroll
    for (int q = 0; q < 2; q++)
        seen = seen || (q < k && t >= sp.lo[q] && t <= sp.hi[q]);
    return seen;
}

// Calls f(tile column, tile row) once for every distinct tile of a footprint of support s.
template <typename F>
__device__ __forceinline__ void visit_tiles(const GridGeom& g, int gx, int gy, int s, F f)
{
    TileSpan rs, cs;
    footprint_spans(g.N, g.rows - 1, s, 2 * s + 1, g.exact, TILE_R, g.tc, gx, gy, rs, cs);
#pragma unroll
    for (int a = 0; a < 3; a++) {
        for (int ct = cs.lo[a]; ct <= cs.hi[a]; ct++) {
            if (span_seen(cs, a, ct))
                continue;
#pragma unroll
            for (int b = 0; b < 3; b++) {
                for (int rt = rs.lo[b]; rt <= rs.hi[b]; rt++)
                    if (!span_seen(rs, b, rt))
                        f(ct, rt);
            }
        }
    }
}

// Largest number of distinct tiles one footprint can touch along an axis of
// length N (kept indices 0..last), over every centre the gridder can produce.
int max_span_tiles(int N, int last, int s, int ks, int exact, int w, bool rows)
{
    int best = 1;
    for (int c = -1; c <= N + 1; c++) {
        TileSpan rs, cs;
        footprint_spans(N, last, s, ks, exact, w, w, rows ? 0 : c, rows ? c : 0, rs, cs);
        const TileSpan& sp = rows ? rs : cs;
        int cnt = 0;
        for (int k = 0; k < 3; k++)
            for (int t = sp.lo[k]; t <= sp.hi[k]; t++)
                if (!span_seen(sp, k, t))
                    cnt++;
        best = std::max(best, cnt);
    }
    return best;
}

// Memoised per geometry: the scan over every centre takes tens of microseconds
// of host time per call at N = 4096.
size_t footprint_tiles_max(const GridGeom& g)
{
    static std::mutex mu;
    static std::map<std::tuple<int, int, int, int, int, int>, size_t> memo;
    const auto key = std::make_tuple(g.N, g.rows, g.s, g.ks, g.exact, g.tc);
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = memo.find(key);
        if (it != memo.end())
            return it->second;
    }
    const size_t v = size_t(max_span_tiles(g.N, g.rows - 1, g.s, g.ks, g.exact, TILE_R, true)) *
        size_t(max_span_tiles(g.N, g.rows - 1, g.s, g.ks, g.exact, g.tc, false));
    std::lock_guard<std::mutex> lk(mu);
    memo[key] = v;
    return v;
}

// wpart: per block the canonical sum of the good weights and the good count.
__global__ __launch_bounds__(GWG) void grid_count_kernel(GridGeom g, const double* uv, const double* vis,
    const double* wts, uint32_t* counts, double* wpart)
{
#pragma clang fp contract(off)
    __shared__ double lds[2 * CANON_LANES];
    const long long base = (long long)blockIdx.x * CANON_BLOCK;
    double wsum = 0.0, nsum = 0.0;  // good weights, good count (exact in double)
    for (int j = 0; j < CANON_PER_LANE; j++) {
        const long long i = base + (long long)j * CANON_LANES + threadIdx.x;
        if (i >= g.n)
            break;
        const Prep p = prep_vis(g, uv, vis, wts, i);
        if (!p.good)
            continue;
        wsum = wsum + p.w;
        nsum = nsum + 1.0;
        const int sup = plane_support(g, i);
        for (int pass = 0; pass <= p.dup; pass++) {
            int gx, gy, cpx, cpy;
            pass_geom(g, p, pass, gx, gy, cpx, cpy);
            visit_tiles(g, gx, gy, sup, [&](int ct, int rt) { atomicAdd(&counts[ct * g.tiles_r + rt], 1u); });
        }
    }
    canon_tree(wsum, nsum, lds);
    if (threadIdx.x == 0) {
        wpart[2 * blockIdx.x] = wsum;
        wpart[2 * blockIdx.x + 1] = nsum;
    }
}

// Kernel functors on the device (exact gridding only; conv_func.cpp:10-202).
// Spheroidal function of the PSWF functor (conv_func.cpp:112-182): F. Schwab's
// rational approximation (Indirect Imaging, 1984), M = 6, alpha = 1; the same
// coefficients and evaluation order as the host table (kernel_tables.cpp).
__device__ double dev_spheroidal(double nu)
{
    constexpr double p0[5] = { 8.203343e-2, -3.644705e-1, 6.278660e-1, -5.335581e-1, 2.312756e-1 };
    constexpr double p1[5] = { 4.028559e-3, -3.697768e-2, 1.021332e-1, -1.201436e-1, 6.412774e-2 };
    constexpr double q0[3] = { 1.0, 8.212018e-1, 2.078043e-1 };
    constexpr double q1[3] = { 1.0, 9.599102e-1, 2.918724e-1 };
    nu = fabs(nu);
    const bool part = nu >= 0.75 && nu <= 1.0;
    const double nuend = (nu >= 0.0 && nu < 0.75) ? 0.75 : ((nu <= 1.0) ? 1.0 : 0.0);
    const double d = nu * nu - nuend * nuend;
    double top = part ? p1[0] : p0[0], bot = part ? q1[0] : q0[0];
    double dk = d; // powers by products: a library pow() per term cost most of the exact path
#pragma unroll
    for (int k = 1; k < 5; k++) {
        top += (part ? p1[k] : p0[k]) * dk;
        if (k < 3)
            bot += (part ? q1[k] : q0[k]) * dk;
        dk *= d;
    }
    return bot > 0.0 ? top / bot : 0.0;
}

__device__ double dev_kernel(const GridGeom& g, double r)
{
    double v;
    switch (g.kfunc) {
    case STP_KERNEL_TOPHAT:
        return (fabs(r) < g.kparam) ? 1.0 : 0.0;
    case STP_KERNEL_TRIANGLE:
        return fmax(1.0 - fabs(r) / g.kparam, 0.0);
    case STP_KERNEL_SINC: {
        double x = r * (M_PI / g.kws);
        if (x == 0.0)
            x = 1.0e-20;
        v = sin(x) / x;
        break;
    }
    case STP_KERNEL_GAUSSIAN:
        v = exp((-1.0 / (g.kwg * g.kwg)) * (r * r));
        break;
    case STP_KERNEL_PSWF: { // conv_func.cpp:185-196
        const double nu = r / g.kparam;
        v = dev_spheroidal(nu) * (1.0 - nu * nu);
        break;
    }
    default: { // GaussianSinc
        double x = r * (M_PI / g.kws);
        if (x == 0.0)
            x = 1.0e-20;
        v = exp((-1.0 / (g.kwg * g.kwg)) * (r * r)) * (sin(x) / x);
        break;
    }
    }
    if (g.kparam > 0.0 && fabs(r) > g.kparam)
        v = 0.0;
    return v;
}

__global__ __launch_bounds__(GWG) void grid_scatter_kernel(GridGeom g, const double* uv, const double* vis,
    const double* wts, uint32_t* cursor, Entry* entries, uint32_t cap)
{
    const long long i = (long long)blockIdx.x * GWG + threadIdx.x;
    if (i >= g.n)
        return;
    const Prep p = prep_vis(g, uv, vis, wts, i);
    if (!p.good)
        return;
    const int sup = plane_support(g, i);
    for (int pass = 0; pass <= p.dup; pass++) {
        const Entry e = make_entry(g, p, pass, i);
        visit_tiles(g, e.gx, e.gy, sup, [&](int ct, int rt) {
            const uint32_t slot = atomicAdd(&cursor[ct * g.tiles_r + rt], 1u);
            if (slot < cap)
                entries[slot] = e;
        });
    }
}

// ---------------------------------------------------------------------------
// Binning by per-block LDS counting sort (no global atomics): block b takes
// visibilities [4096 b, 4096 b + 4096) and writes its entry count of every tile
// to counts[b * ntiles + tile] (one contiguous row per block).  A column scan over
// the blocks turns each row into the block's cursor inside every tile and gives
// the tile totals, whose exclusive scan is the per-tile entry ranges.
constexpr int BWG = 1024;
constexpr int VPB = CANON_BLOCK; // visibilities per binning block (also the canonical sum block)
constexpr int MAX_LDS_TILES = 24576;

__device__ __forceinline__ void bin_count_body(const GridGeom& g, const double* uv, const double* vis, const double* wts,
    uint32_t* counts, double* wpart, int bid)
{
#pragma clang fp contract(off)
    extern __shared__ uint32_t hist[];
    __shared__ double wl[VPB];
    __shared__ unsigned long long wng[BWG / 64];
    const int ntiles = g.tiles_r * g.tiles_c;
    for (int t = threadIdx.x; t < ntiles; t += BWG)
        hist[t] = 0;
    __syncthreads();
    const long long base = (long long)bid * VPB;
    unsigned long long ng = 0;
    VisIn in[VPB / BWG];
#pragma unroll
    for (int j = 0; j < VPB / BWG; j++) {
        const long long i = base + threadIdx.x + j * BWG;
        if (i < g.n)
            in[j] = load_vis(g, uv, vis, wts, i);
    }
#pragma unroll
    for (int j = 0; j < VPB / BWG; j++) {
        const int local = threadIdx.x + j * BWG;
        const long long i = base + local;
        double wgood = 0.0;
        if (i < g.n) {
            const Prep p = prep_in(g, in[j]);
            if (p.good) {
                wgood = p.w;
                ng++;
                const int sup = plane_support(g, i);
                for (int pass = 0; pass <= p.dup; pass++) {
                    int gx, gy, cpx, cpy;
                    pass_geom(g, p, pass, gx, gy, cpx, cpy);
                    visit_tiles(g, gx, gy, sup, [&](int ct, int rt) { atomicAdd(&hist[ct * g.tiles_r + rt], 1u); });
                }
            }
        }
        wl[local] = wgood;
    }
    __syncthreads();
    // canonical sum of the good weights: lane t adds elements t, t+256, ..., t+15*256
    double a = 0.0;
    if (threadIdx.x < CANON_LANES)
        for (int j = 0; j < CANON_PER_LANE; j++)
            a = a + wl[threadIdx.x + j * CANON_LANES];
    __syncthreads();
    if (threadIdx.x < CANON_LANES)
        wl[threadIdx.x] = a;
    for (int off = CANON_LANES / 2; off >= 1; off >>= 1) {
        __syncthreads();
        if (threadIdx.x < off)
            wl[threadIdx.x] = wl[threadIdx.x] + wl[threadIdx.x + off];
    }
    // the block's good count (exact in double) beside its weight sum
    for (int off = 32; off >= 1; off >>= 1)
        ng += __shfl_down(ng, off, 64);
    if ((threadIdx.x & 63) == 0)
        wng[threadIdx.x >> 6] = ng;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long c = 0;
        for (int k = 0; k < BWG / 64; k++)
            c += wng[k];
        wpart[2 * bid] = wl[0];
        wpart[2 * bid + 1] = double(c);
    }
    for (int t = threadIdx.x; t < ntiles; t += BWG)
        counts[size_t(bid) * ntiles + t] = hist[t];
}

__global__ __launch_bounds__(BWG) void grid_bin_count_kernel(GridGeom g, const double* uv, const double* vis,
    const double* wts, uint32_t* counts, double* wpart)
{
    bin_count_body(g, uv, vis, wts, counts, wpart, int(blockIdx.x));
}

// Per tile t: counts[b][t] -> entries of tile t in blocks before b (in place); totals[t].
// A workgroup takes 64 tiles (lanes) x 16 slices of the blocks (waves).
__device__ __forceinline__ void colscan_body(uint32_t* counts, int nblk, int ntiles, uint32_t* totals, int bid)
{
    __shared__ uint32_t part[16][64];
    const int lane = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const int t = bid * 64 + lane;
    const int per = (nblk + 15) / 16, b0 = min(nblk, sl * per), b1 = min(nblk, b0 + per);
    uint32_t s = 0;
    if (t < ntiles)
        for (int b = b0; b < b1; b++)
            s += counts[size_t(b) * ntiles + t];
    part[sl][lane] = s;
    __syncthreads();
    if (sl == 0) {
        uint32_t run = 0;
        for (int k = 0; k < 16; k++) {
            const uint32_t v = part[k][lane];
            part[k][lane] = run;
            run += v;
        }
        if (t < ntiles)
            totals[t] = run;
    }
    __syncthreads();
    if (t >= ntiles)
        return;
    uint32_t run = part[sl][lane];
    for (int bb = b0; bb < b1; bb += 16) {
        uint32_t v[16];
#pragma unroll
        for (int k = 0; k < 16; k++)
            v[k] = bb + k < b1 ? counts[size_t(bb + k) * ntiles + t] : 0u;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            if (bb + k < b1)
                counts[size_t(bb + k) * ntiles + t] = run;
            run += v[k];
        }
    }
}

__global__ __launch_bounds__(1024) void bin_colscan_kernel(uint32_t* counts, int nblk, int ntiles, uint32_t* totals)
{
    colscan_body(counts, nblk, ntiles, totals, int(blockIdx.x));
}

// Exclusive scan of the tile totals into out[0..ntiles) (LDS) by the BWG threads of a
// block, each taking a run of at most TSCAN_PER tiles; returns the total.
constexpr int TSCAN_PER = (MAX_LDS_TILES + BWG - 1) / BWG;
__device__ uint32_t scan_tile_totals(const uint32_t* totals, int ntiles, uint32_t* out, uint32_t* wsum)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int per = (ntiles + BWG - 1) / BWG;
    const int i0 = min(ntiles, t * per), i1 = min(ntiles, i0 + per);
    uint32_t v[TSCAN_PER];
#pragma unroll
    for (int j = 0; j < TSCAN_PER; j++)
        v[j] = i0 + j < i1 ? totals[i0 + j] : 0u;
    uint32_t s = 0;
#pragma unroll
    for (int j = 0; j < TSCAN_PER; j++)
        s += v[j];
    uint32_t x = s;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off)
            x += y;
    }
    if (lane == 63)
        wsum[w] = x;
    __syncthreads();
    uint32_t total = 0;
    for (int k = 0; k < BWG / 64; k++) {
        total += wsum[k];
        if (k < w)
            x += wsum[k];
    }
    uint32_t run = x - s;
#pragma unroll
    for (int j = 0; j < TSCAN_PER; j++) {
        if (i0 + j < i1) {
            out[i0 + j] = run;
            run += v[j];
        }
    }
    return total;
}

// Splitting of heavy tiles.  Interferometers crowd the origin of the uv plane, so a
// few tiles can hold most of the entries, and one workgroup per tile then leaves the
// rest of the chip idle.  A tile of more than ch entries is summed in chunks of ch by
// several workgroups: chunk 0 by the tile's own, chunks 1.. by extra workgroups.  Every
// chunk of a split tile stores its FP64 sums in a slot, and merge workgroups add the
// slots in chunk order.  ch = max(split_min, entries / ext_max), so at most ext_max
// extra chunks, as many split tiles and 2 ext_max slots exist.  Below split_min entries
// a tile's sums take less than a merge costs; SPLIT_EXTRA_MAX gives every CU two chunks.
//
// The plan and the slots lie in the unused end of the entry buffer, which is sized for
// the most tiles that footprints can touch (eight entries for each visibility at 7 x 7
// taps; 1.2 to 1.6 are used): every kernel derives the same view from the entry count,
// and where the end is short there are fewer chunks or none.
constexpr uint32_t SPLIT_MIN = 1024;
// A grid of few tiles leaves the chip idle whatever its tiles hold, and where the entries
// crowd into a block or two, one wave sums them: smaller chunks there, but no more than a
// heavy tile's merge can take.  3000 visibilities of a condensed array: 141 -> 91 us at 128 x
// 128, 105 -> 82 us at 256 x 256; 100 k at 256 x 256 132 us at 1024, 141 at 256 entries.  The plan
// costs 4 us where nothing is split, so not below SPLIT_FEW_VIS (128 x 128, 1000: 47 or 51 us).
constexpr int SPLIT_FEW_TILES = 64;
constexpr long long SPLIT_FEW_VIS = 2048;
__host__ __device__ constexpr uint32_t split_min(int ntiles, long long n)
{
    return ntiles > SPLIT_FEW_TILES || n < SPLIT_FEW_VIS || n >= 64ll * SPLIT_MIN ? SPLIT_MIN
        : n <= 64 * 256                                                         ? 256u
                                                                                : uint32_t(n / 64);
}
constexpr uint32_t W_SPLIT_MIN = 256; // W-projection: an entry has up to 4096 taps in a tile
constexpr size_t SPLIT_EXTRA_MAX = 512;
constexpr size_t SPLIT_PLAN_BYTES = 16384;
static_assert(256 + SPLIT_EXTRA_MAX * 20 <= SPLIT_PLAN_BYTES, "plan layout");
struct Split {
    uint32_t* hdr;     // extra chunks, split tiles, ch (null: no splitting)
    uint32_t* ext;     // per extra chunk: tile, chunk
    uint32_t* spl;     // per split tile (in tile order): tile, first slot, chunks
    double* part;      // slots of chans x tile columns x TILE_R sums
    size_t room;       // bytes for slots
};

inline int split_extra_max(size_t n, uint32_t least) { return int(std::min(SPLIT_EXTRA_MAX, n / least)); }
// Merge workgroups (four tile columns each).
inline size_t merge_blocks(int ext_host, int tc) { return size_t(ext_host) * (tc / 4); }

__device__ __forceinline__ Split split_view(Entry* entries, uint32_t cap, uint32_t nent, int ext_host, int tc, int chans)
{
    Split sp{ nullptr, nullptr, nullptr, nullptr, 0 };
    const size_t used = (size_t(nent) * sizeof(Entry) + 255) & ~size_t(255);
    const size_t room = size_t(cap) * sizeof(Entry), slot = size_t(chans) * tc * TILE_R * sizeof(double);
    if (ext_host <= 0 || room < used + SPLIT_PLAN_BYTES + 2 * slot)
        return sp;
    sp.room = room - used - SPLIT_PLAN_BYTES;
    uint8_t* base = reinterpret_cast<uint8_t*>(entries) + used;
    sp.hdr = reinterpret_cast<uint32_t*>(base);
    sp.ext = sp.hdr + 64;
    sp.spl = sp.ext + 2 * SPLIT_EXTRA_MAX;
    sp.part = reinterpret_cast<double*>(base + SPLIT_PLAN_BYTES);
    return sp;
}

// The plan from the tile totals, by one workgroup of BWG threads.
__device__ void split_plan(const Split& sp, const uint32_t* totals, int ntiles, uint32_t total, int ext_host, int tc,
    int chans, uint32_t least, uint32_t* wsum)
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const size_t slot = size_t(chans) * tc * TILE_R * sizeof(double);
    const uint32_t ext_max = uint32_t(min(size_t(ext_host), sp.room / (2 * slot)));
    const uint32_t ch = max(least, (total + ext_max - 1) / ext_max);
    const int per = (ntiles + BWG - 1) / BWG;
    const int i0 = min(ntiles, tid * per), i1 = min(ntiles, i0 + per);
    uint32_t s = 0; // extra chunks | split tiles << 16
    for (int t = i0; t < i1; t++) {
        const uint32_t c = totals[t];
        if (c > ch)
            s += (c - 1) / ch + (1u << 16);
    }
    uint32_t x = s;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off)
            x += y;
    }
    __syncthreads();
    if (lane == 63)
        wsum[w] = x;
    __syncthreads();
    uint32_t sum = 0;
    for (int k = 0; k < BWG / 64; k++) {
        sum += wsum[k];
        if (k < w)
            x += wsum[k];
    }
    uint32_t e = (x - s) & 0xffffu, i = (x - s) >> 16;
    for (int t = i0; t < i1; t++) {
        const uint32_t c = totals[t];
        if (c <= ch)
            continue;
        const uint32_t n = (c - 1) / ch + 1;
        sp.spl[3 * i] = uint32_t(t);
        sp.spl[3 * i + 1] = e + i;
        sp.spl[3 * i + 2] = n;
        for (uint32_t k = 1; k < n; k++, e++) {
            sp.ext[2 * e] = uint32_t(t);
            sp.ext[2 * e + 1] = k;
        }
        i++;
    }
    if (tid == 0) {
        sp.hdr[0] = sum & 0xffffu;
        sp.hdr[1] = sum >> 16;
        sp.hdr[2] = ch;
    }
}

// Block b's entries go to cursors tile offset + block offset; the tile offsets (the
// scan of the tile totals) are computed by every block in LDS, and block 0 also
// writes them to tile_off[0..ntiles] for the tile kernel, and the split plan.
__device__ __forceinline__ void bin_scatter_body(const GridGeom& g, const double* uv, const double* vis, const double* wts,
    const uint32_t* totals, const uint32_t* block_off, Entry* entries, uint32_t cap, uint32_t* tile_off, int ext_host,
    int bid)
{
    extern __shared__ uint32_t cur[];
    __shared__ uint32_t wsum[BWG / 64];
    const int ntiles = g.tiles_r * g.tiles_c;
    const uint32_t total = scan_tile_totals(totals, ntiles, cur, wsum);
    __syncthreads();
    if (bid == 0) {
        for (int t = threadIdx.x; t < ntiles; t += BWG)
            tile_off[t] = cur[t];
        if (threadIdx.x == 0)
            tile_off[ntiles] = total;
    }
    for (int t = threadIdx.x; t < ntiles; t += BWG)
        cur[t] += block_off[size_t(bid) * ntiles + t];
    __syncthreads();
    const long long base = (long long)bid * VPB;
    VisIn in[VPB / BWG];
#pragma unroll
    for (int j = 0; j < VPB / BWG; j++) {
        const long long i = base + threadIdx.x + j * BWG;
        if (i < g.n)
            in[j] = load_vis(g, uv, vis, wts, i);
    }
#pragma unroll
    for (int j = 0; j < VPB / BWG; j++) {
        const long long i = base + threadIdx.x + j * BWG;
        if (i >= g.n)
            break;
        const Prep p = prep_in(g, in[j]);
        if (!p.good)
            continue;
        const int sup = plane_support(g, i);
        for (int pass = 0; pass <= p.dup; pass++) {
            const Entry e = make_entry(g, p, pass, i);
            visit_tiles(g, e.gx, e.gy, sup, [&](int ct, int rt) {
                const uint32_t slot = atomicAdd(&cur[ct * g.tiles_r + rt], 1u);
                if (slot < cap)
                    entries[slot] = e;
            });
        }
    }
    if (bid == 0 && g.planes > 0) {
        // tile_off[ntiles + 1]: the W tile sums in one phase
        double taps = 0.0;
        for (int p = threadIdx.x; p < g.planes; p += BWG)
            taps += double(2 * g.psup[p] + 1) * double(2 * g.psup[p] + 1);
        for (int off = 32; off >= 1; off >>= 1)
            taps += __shfl_xor(taps, off, 64);
        __shared__ double tsum[BWG / 64];
        if ((threadIdx.x & 63) == 0)
            tsum[threadIdx.x >> 6] = taps;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int k = 1; k < BWG / 64; k++)
                taps += tsum[k];
            tile_off[ntiles + 1] = taps < g.phase_taps ? 1u : 0u;
        }
    }
    if (bid == 0 && ext_host > 0) {
        const int chans = g.wproj ? 4 : 3;
        const Split sp = split_view(entries, cap, total, ext_host, g.tc, chans);
        if (sp.hdr)
            split_plan(sp, totals, ntiles, total, ext_host, g.tc, chans, g.wproj ? W_SPLIT_MIN : split_min(ntiles, g.n), wsum);
    }
}

__global__ __launch_bounds__(BWG) void grid_bin_scatter_kernel(GridGeom g, const double* uv, const double* vis,
    const double* wts, const uint32_t* totals, const uint32_t* block_off, Entry* entries, uint32_t cap, uint32_t* tile_off,
    int ext_host)
{
    bin_scatter_body(g, uv, vis, wts, totals, block_off, entries, cap, tile_off, ext_host, int(blockIdx.x));
}

// ---------------------------------------------------------------------------
// Tile sums on the FP64 matrix cores.  The taps of an entry are the outer product of
// its kernel row and column values, so the entries that touch a block of 16 x 16 cells
// sum as a matrix product: v_mfma_f64_16x16x4 adds four entries at once, A = kx times
// the entry's (vis w) re, (vis w) im or w over the block's columns, B = ky over its rows,
// both zero outside the footprint.  A wave owns one block (three accumulators of four
// doubles per lane) and a workgroup the tile's TC / 4 blocks.  The workgroup stages its
// entries in LDS in batches, a thread for each, which queues the entry's index for the
// blocks that it touches; each wave then takes its queue four at a time.
// (Waves that each walked all entries spent more on the walk than on the products: 123 us
// at 1 M visibilities, N = 4096.)
//
// Bound: FP64 matrix products and vector instructions share their issue (a wave's
// products and another wave's integer instructions take the sum of their times), so the
// time is the sum of both: a 7 x 7 footprint touches (22 / 16)^2 = 1.9 blocks, each 3 x 64
// cycles per four entries plus 17 vector instructions, 57 us for 1 M visibilities at 2.1
// GHz, and staging.  DPP broadcasts inside rows of 16 lanes hand the entries' values out,
// since the LDS is nearly as busy with the kernel values.  Measured with N = 4096 and 1 M
// visibilities: 99 us (uniform uv disk), 150 us (centrally condensed array, FP64) against
// 144 and 554 us for LDS FP64 atomics, three per tap, the form before; exact PSWF
// kernels, 300 k visibilities, N = 2048: 146 us against 3500.  The sums stay FP64 on the FP32
// path too, whose kernel values are no longer rounded to FP32.
//
// Heavy tiles are summed in chunks (Split); the chunks of a split tile store their sums
// in slots that grid_total's merge workgroups add in chunk order.
typedef double double4v __attribute__((ext_vector_type(4)));

// Where the kernel values come from: the oversampled table in LDS with 15 zeros on both
// sides of each kernel, so that a block's 16 rows or columns read it without a range
// check; the plain table, for oversampling factors whose padded table would take the LDS
// of several workgroups; or exact kernels, evaluated into LDS for each batch.
enum { KERNEL_PADDED = 0, KERNEL_TABLE = 1, KERNEL_EXACT = 2 };
constexpr int KV_DOUBLES = 3584;          // kernel table, or exact kernel vectors of a batch (28 KB)
constexpr int KPAD = 15;
constexpr int PADDED_DOUBLES = 2560;      // largest padded table (20 KB: four workgroups per CU at 32 columns)
constexpr int OUT_STRIDE = TILE_R + 4;

inline int table_form(int cs, int ks) { return cs * (ks + 2 * KPAD) <= PADDED_DOUBLES ? KERNEL_PADDED : KERNEL_TABLE; }

struct Staged {
    double a, b, w;  // (vis w) re, im and w
    int oy, ox;      // kernel row of the tile's first row and kernel column of its first column as padded
                     // table indices; other forms: as 16-bit offsets | the kernel's table index << 16
};

__host__ __device__ constexpr int tile_threads(int tc) { return tc * 16; }
// Waves per SIMD asked of the register allocator: six keep three 32-column workgroups on
// a CU (eight spilled: 103 against 101 us at 1 M visibilities); exact kernels need the
// registers.
constexpr int tile_waves(int form) { return form == KERNEL_EXACT ? 2 : 6; }
// Entries staged at a time: one per thread; exact kernels take two threads for each (its
// row and its column values).
__host__ __device__ constexpr int tile_batch(int tc, bool exact) { return exact ? tile_threads(tc) / 2 : tile_threads(tc); }

// LDS of a tile workgroup: the kernel table, then the staged entries and the blocks'
// queues or the tile's sums on their way to memory.
inline size_t tiles_lds(int tc, int form, int cs, int ks)
{
    const size_t table = form == KERNEL_EXACT ? size_t(KV_DOUBLES)
                                              : size_t(cs) * (form == KERNEL_PADDED ? ks + 2 * KPAD : ks);
    const size_t batch = tile_batch(tc, form == KERNEL_EXACT);
    const size_t stage = batch * sizeof(Staged) + batch * (tc / 4 + 1) * sizeof(uint16_t);
    const size_t out = 2 * size_t(tc) * OUT_STRIDE * sizeof(double);
    return ((table + 1) & ~size_t(1)) * sizeof(double) + std::max(stage, out);
}

// Lane R of each row of 16 lanes, to the whole row (DPP row_newbcast: no LDS traffic,
// which the kernel-value reads need).
template <int R>
__device__ __forceinline__ int row_lane(int x)
{
    return __builtin_amdgcn_mov_dpp(x, 0x150 + R, 0xf, 0xf, true);
}
template <int R>
__device__ __forceinline__ double row_lane(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = row_lane<R>(int(b)), hi = row_lane<R>(int(b >> 32));
    return __longlong_as_double((long long)((unsigned long long)(unsigned)hi << 32 | (unsigned)lo));
}

// f(integral_constant<int, R>) for R = 0 .. n - 1 (n <= 16, uniform)
template <int R = 0, typename F>
__device__ __forceinline__ void for_rows(int n, F f)
{
    if constexpr (R < 16) {
        if (R < n) {
            f(std::integral_constant<int, R>{});
            for_rows<R + 1>(n, f);
        }
    }
}

template <typename T, int TC, int FORM>
__device__ __forceinline__ void tiles_mfma_body(const GridGeom& g, Entry* entries, const uint32_t* offsets, uint32_t cap,
    const double* ktab, const double* uv, cplx<T>* vgrid, cplx<T>* bgrid, int ext_host, int bid)
{
#pragma clang fp contract(off)
    constexpr int NTH = tile_threads(TC), NB = TC / 4; // threads, blocks (one per wave)
    constexpr int QCAP = tile_batch(TC, FORM == KERNEL_EXACT);
    extern __shared__ __align__(16) double dyn[];
    __shared__ int qcnt[NB];
    __shared__ int oddcnt[2];
    const int ks = g.ks, s = g.s, N = g.N;
    const int cs = (g.os / 2) * 2 + 1;
    const int ntiles = g.tiles_r * g.tiles_c;
    Split sp{ nullptr, nullptr, nullptr, nullptr, 0 };
    uint32_t chunk = 0;
    int t = bid - ext_host;
    if (t < 0) {
        // an extra chunk of a split tile
        sp = split_view(entries, cap, offsets[ntiles], ext_host, TC, 3);
        if (!sp.hdr || uint32_t(bid) >= sp.hdr[0])
            return;
        t = int(sp.ext[2 * bid]);
        chunk = sp.ext[2 * bid + 1];
    }
    uint32_t eb = min(offsets[t], cap), ee = min(offsets[t + 1], cap);
    uint32_t ch = 0xffffffffu;
    if (ee - eb > split_min(ntiles, g.n)) { // light tiles do not wait for the plan
        if (bid >= ext_host)
            sp = split_view(entries, cap, offsets[ntiles], ext_host, TC, 3);
        ch = sp.hdr ? sp.hdr[2] : ch;
    }
    const bool split = ee - eb > ch;
    if (split) {
        const uint32_t e0 = eb + chunk * ch;
        ee = min(ee, e0 + ch);
        eb = e0;
    }
    const int rt = t % g.tiles_r, ct = t / g.tiles_r;
    const int r0 = rt * TILE_R, c0 = ct * TC;
    // the tile's rows and columns on the grid (pieces of a footprint past them are not stored:
    // with a 32-column tile on a 16 x 16 grid most entries had one)
    const int nr = min(TILE_R, g.rows - r0), nc = min(TC, N - c0);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int pitch = FORM == KERNEL_PADDED ? ks + 2 * KPAD : ks;
    double* kt = dyn;
    double* area = dyn + (FORM == KERNEL_EXACT ? KV_DOUBLES : ((cs * pitch + 1) & ~1));
    Staged* staged = reinterpret_cast<Staged*>(area);
    uint16_t* queues = reinterpret_cast<uint16_t*>(staged + QCAP);
    uint16_t* oddq = queues + NB * QCAP;
    const int br = 16 * (wave & 3), bc = 16 * (wave >> 2); // the wave's block inside the tile
    const int m = lane & 15, kk = lane >> 4;
    double4v ar = { 0, 0, 0, 0 }, ai = { 0, 0, 0, 0 }, ab = { 0, 0, 0, 0 };

    // kernel value i of an entry whose values start at kt[base], zero outside the kernel
    auto checked = [&](int base, int i) -> double { return unsigned(i) < unsigned(ks) ? kt[base + i] : 0.0; };
    // row (column) value m of the wave's block for staged entry q with offsets o
    auto block_value = [&](int q, int o, int at, int axis) -> double {
        if constexpr (FORM == KERNEL_PADDED)
            return kt[o + at + m];
        else
            return checked(FORM == KERNEL_TABLE ? int(uint32_t(o) >> 16) : (q * 2 + axis) * ks, int(short(o & 0xffff)) + at + m);
    };

    if (eb < ee) {
        if (threadIdx.x < NB)
            qcnt[threadIdx.x] = 0;
        if (threadIdx.x < 2)
            oddcnt[threadIdx.x] = 0;
        const int batch = FORM == KERNEL_EXACT ? min(QCAP, KV_DOUBLES / (2 * ks)) : QCAP;
        // exact kernels: thread k + QCAP evaluates the columns of thread k's entry
        const int slot = FORM == KERNEL_EXACT ? int(threadIdx.x) % QCAP : int(threadIdx.x);
        const bool lead = FORM != KERNEL_EXACT || int(threadIdx.x) < QCAP;
        // the next batch's loads are in flight while this one is summed
        int ngx, ngy, ncp, nidx;
        double nvr, nvi, nw;
        auto fetch = [&](uint32_t e) {
            const Entry* p = entries + min(e + uint32_t(slot), ee - 1);
            ngx = p->gx;
            ngy = p->gy;
            ncp = p->cp;
            nidx = p->idx;
            nvr = p->vr;
            nvi = p->vi;
            nw = p->w;
        };
        fetch(eb);
        if constexpr (FORM == KERNEL_PADDED) {
            for (int k = threadIdx.x; k < cs * pitch; k += NTH) {
                const int c = k / pitch, i = k - c * pitch - KPAD;
                kt[k] = unsigned(i) < unsigned(ks) ? ktab[c * ks + i] : 0.0;
            }
        } else if constexpr (FORM == KERNEL_TABLE) {
            for (int k = threadIdx.x; k < cs * ks; k += NTH)
                kt[k] = ktab[k];
        }
        __syncthreads();
        int round = 0;
        for (uint32_t e0 = eb; e0 < ee; e0 += uint32_t(batch)) {
            const int gx = ngx, gy = ngy, cp = ncp;
            const double vr = nvr, vi = nvi;
            double w = nw;
            const bool valid = slot < batch && e0 + uint32_t(slot) < ee;
            if constexpr (FORM == KERNEL_EXACT) {
                // exact kernel of this visibility pass (make_kernel_array, conv_func.h:279-303),
                // its tap sum folded into the weight
                double sum = 0.0;
                if (valid) {
                    const long long k = nidx >> 1;
                    double uu = uv[k] * g.scale;
                    double vv = uv[g.n + k] * g.scale;
                    if (g.halfplane && vv < 0.0) {
                        uu = -uu;
                        vv = -vv;
                    }
                    const double x = lead ? vv : uu;
                    double f = x - int(rint(x));
                    if (nidx & 1)
                        f = -f;
                    double* kv = kt + (slot * 2 + (lead ? 0 : 1)) * ks;
                    for (int q = 0; q < ks; q++) {
                        const double v = dev_kernel(g, double(q - s) - f);
                        kv[q] = v;
                        sum += v;
                    }
                    if (!lead)
                        staged[slot].a = sum;
                }
                __syncthreads();
                if (valid && lead)
                    w = w / (sum * staged[slot].a);
            }
            fetch(e0 + uint32_t(batch));
            const double a = vr * w, b = vi * w;
            // the products multiply zeros outside the footprint: entries that are not
            // finite (among them an infinite visibility of weight 0, whose product is not) are
            // added tap by tap instead, so they touch their own taps only
            const bool odd = !(fabs(a) < 1.0e290 && fabs(b) < 1.0e290 && fabs(w) < 1.0e290);
            // the footprint and its wrapped pieces that overlap the tile: raw rows at +N (rows
            // past N wrap) and, for exact kernels, -N; raw columns at +-N.  One piece a round:
            // a second one exists only on grids hardly wider than the tile.
            const int iraw = r0 - (gy - s), jraw = c0 - (gx - s);
            uint32_t pieces = 0;
            if (valid && lead) {
                uint32_t rp = 0, cpz = 0;
                auto meets = [&](int o, int len) { return o < ks && o > -len; };
                rp = (meets(iraw, nr) ? 1u : 0u) | (meets(iraw + N, nr) ? 2u : 0u) |
                    (FORM == KERNEL_EXACT && meets(iraw - N, nr) ? 4u : 0u);
                cpz = (meets(jraw, nc) ? 1u : 0u) | (meets(jraw + N, nc) ? 2u : 0u) | (meets(jraw - N, nc) ? 4u : 0u);
                pieces = ((rp & 1u) ? cpz : 0u) | ((rp & 2u) ? cpz << 3 : 0u) | ((rp & 4u) ? cpz << 6 : 0u);
            }
            bool more;
            do {
                uint32_t hits = 0; // blocks touched
                if (pieces) {
                    const int p = __builtin_ctz(pieces);
                    pieces &= pieces - 1;
                    const int pr = p / 3, pc = p % 3;
                    const int i0 = iraw + (pr == 0 ? 0 : (pr == 1 ? N : -N)), j0 = jraw + (pc == 0 ? 0 : (pc == 1 ? N : -N));
                    uint32_t rh = 0;
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        rh |= (i0 + 16 * k < ks && i0 + 16 * k > -16) ? 1u << k : 0u;
#pragma unroll
                    for (int k = 0; k < NB / 4; k++)
                        hits |= (j0 + 16 * k < ks && j0 + 16 * k > -16) ? rh << (4 * k) : 0u;
                    Staged st;
                    st.a = odd ? vr : a;
                    st.b = odd ? vi : b;
                    st.w = w;
                    const int by = FORM == KERNEL_EXACT ? 0 : (cp >> 16) * pitch + (FORM == KERNEL_PADDED ? KPAD : 0);
                    const int bx = FORM == KERNEL_EXACT ? 0 : (cp & 0xffff) * pitch + (FORM == KERNEL_PADDED ? KPAD : 0);
                    st.oy = FORM == KERNEL_PADDED && !odd ? by + i0 : (i0 & 0xffff) | by << 16;
                    st.ox = FORM == KERNEL_PADDED && !odd ? bx + j0 : (j0 & 0xffff) | bx << 16;
                    staged[slot] = st;
                    if (odd) {
                        oddq[atomicAdd(&oddcnt[round & 1], 1)] = uint16_t(slot);
                        hits = 0;
                    }
                }
                while (hits) {
                    const int k = __builtin_ctz(hits);
                    hits &= hits - 1;
                    queues[k * QCAP + atomicAdd(&qcnt[k], 1)] = uint16_t(slot);
                }
                __syncthreads();
                const int cnt = __builtin_amdgcn_readfirstlane(qcnt[wave]), nodd = __builtin_amdgcn_readfirstlane(oddcnt[round & 1]);
                const uint16_t* queue = queues + wave * QCAP;
                for (int q0 = 0; q0 < cnt; q0 += 64) {
                    // 64 queued entries at once: lane (m, kk) holds entry kk of product m, and
                    // product G takes lane G of each row of 16 lanes
                    const int at = q0 + 4 * m + kk;
                    const int q = queue[min(at, cnt - 1)];
                    const Staged e = staged[q];
                    const bool on = at < cnt;
                    const double ea = on ? e.a : 0.0, eb4 = on ? e.b : 0.0, ew = on ? e.w : 0.0;
                    const int groups = min(16, (cnt - q0 + 3) >> 2);
                    for_rows(groups, [&](auto G) {
                        constexpr int R = decltype(G)::value;
                        const int qg = FORM == KERNEL_EXACT ? row_lane<R>(q) : 0;
                        const double ky = block_value(qg, row_lane<R>(e.oy), br, 0);
                        const double kx = block_value(qg, row_lane<R>(e.ox), bc, 1);
                        ar = __builtin_amdgcn_mfma_f64_16x16x4f64(kx * row_lane<R>(ea), ky, ar, 0, 0, 0);
                        ai = __builtin_amdgcn_mfma_f64_16x16x4f64(kx * row_lane<R>(eb4), ky, ai, 0, 0, 0);
                        if (g.beam)
                            ab = __builtin_amdgcn_mfma_f64_16x16x4f64(kx * row_lane<R>(ew), ky, ab, 0, 0, 0);
                    });
                }
                for (int k = 0; k < nodd; k++) {
                    const int q = oddq[k];
                    const Staged e = staged[q];
                    const int i = int(short(e.oy & 0xffff)) + br + m, j = int(short(e.ox & 0xffff)) + bc;
                    const double ky = checked(FORM == KERNEL_EXACT ? q * 2 * ks : int(uint32_t(e.oy) >> 16), i);
                    // lane m holds column value m
                    const double kx = checked(FORM == KERNEL_EXACT ? (q * 2 + 1) * ks : int(uint32_t(e.ox) >> 16), j + m);
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const double kw = (ky * __shfl(kx, kk + 4 * v, 64)) * e.w;
                        if (unsigned(i) < unsigned(ks) && unsigned(j + kk + 4 * v) < unsigned(ks)) {
                            ar[v] += e.a * kw;
                            ai[v] += e.b * kw;
                            ab[v] += kw;
                        }
                    }
                }
                if (lane == 0)
                    qcnt[wave] = 0;
                if (threadIdx.x == 0)
                    oddcnt[(round + 1) & 1] = 0;
                round++;
                more = __syncthreads_or(int(pieces != 0)) != 0;
            } while (more);
        }
    }
    // lane (m, kk) holds the block's row m, columns kk + 4 v
    const int lr0 = br + m, lc0 = bc + kk;
    if (split) {
        uint32_t lo = 0, hi = sp.hdr[1] - 1; // the tile's record among the split tiles
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if (sp.spl[3 * mid] < uint32_t(t))
                lo = mid + 1;
            else
                hi = mid;
        }
        double* out = sp.part + size_t(sp.spl[3 * lo + 1] + chunk) * (3 * TC * TILE_R);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            double* o = out + (lc0 + 4 * v) * TILE_R + lr0;
            o[0] = ar[v];
            o[TC * TILE_R] = ai[v];
            if (g.beam)
                o[2 * TC * TILE_R] = ab[v];
        }
        return;
    }
    // through LDS, so that a wave stores 64 consecutive rows of a column; the beam grid is
    // complex (imaginary part 0) or, with g.bpack, packed real: cell (r, c) is component
    // c & 1 of element (r, c / 2) of a rows x N/2 complex array
    const bool some = eb < ee;
    if (!some && g.skip)
        return;
    double* o0 = area;
    double* o1 = area + TC * OUT_STRIDE;
    if (some) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            o0[(lc0 + 4 * v) * OUT_STRIDE + lr0] = ar[v];
            o1[(lc0 + 4 * v) * OUT_STRIDE + lr0] = ai[v];
        }
        __syncthreads();
    }
    const int lr = threadIdx.x & 63, r = r0 + lr;
    for (int lc = threadIdx.x >> 6; lc < TC; lc += NTH / 64) {
        const int c = c0 + lc;
        if (r < g.rows && c < N) {
            cplx<T> v = { T(0), T(0) };
            if (some)
                v = { T(o0[lc * OUT_STRIDE + lr]), T(o1[lc * OUT_STRIDE + lr]) };
            vgrid[size_t(r) + size_t(c) * g.rows] = v;
        }
    }
    if (!g.beam)
        return;
    if (some) {
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; v++)
            o0[(lc0 + 4 * v) * OUT_STRIDE + lr0] = ab[v];
        __syncthreads();
    }
    for (int lc = threadIdx.x >> 6; lc < (g.bpack ? TC / 2 : TC); lc += NTH / 64) {
        const int c = c0 + (g.bpack ? 2 * lc : lc);
        if (r < g.rows && c < N) {
            cplx<T> v = { T(0), T(0) };
            if (some && g.bpack)
                v = { T(o0[2 * lc * OUT_STRIDE + lr]), T(o0[(2 * lc + 1) * OUT_STRIDE + lr]) };
            else if (some)
                v = { T(o0[lc * OUT_STRIDE + lr]), T(0) };
            bgrid[size_t(r) + size_t(g.bpack ? c / 2 : c) * g.rows] = v;
        }
    }
}

template <typename T, int TC, int FORM>
__global__ __launch_bounds__(tile_threads(TC), tile_waves(FORM)) void grid_tiles_kernel(GridGeom g, Entry* entries, const uint32_t* offsets,
    uint32_t cap, const double* ktab, const double* uv, cplx<T>* vgrid, cplx<T>* bgrid, int ext_host)
{
    tiles_mfma_body<T, TC, FORM>(g, entries, offsets, cap, ktab, uv, vgrid, bgrid, ext_host, int(blockIdx.x));
}

// Workgroup q of the merges: columns 4 (q % (tc / 4)) .. + 3 of split tile q / (tc / 4), the
// sum of its chunks' slots in chunk order.  lds: 4 x TILE_R doubles.
template <typename T>
__device__ __forceinline__ void merge_body(const GridGeom& g, Entry* entries, uint32_t cap, uint32_t nent, int ext_host,
    cplx<T>* vgrid, cplx<T>* bgrid, int q, double* lds)
{
    const int chans = g.wproj ? 4 : 3; // W-projection: a complex beam grid
    const Split sp = split_view(entries, cap, nent, ext_host, g.tc, chans);
    const int groups = g.tc / 4;
    const uint32_t i = uint32_t(q / groups);
    if (!sp.hdr || i >= sp.hdr[1])
        return;
    const int t = int(sp.spl[3 * i]);
    const uint32_t slot = sp.spl[3 * i + 1], n = sp.spl[3 * i + 2];
    const int lr = threadIdx.x & 63, lq = threadIdx.x >> 6, lc = 4 * (q % groups) + lq;
    const size_t plane = size_t(g.tc) * TILE_R;
    const double* p = sp.part + slot * chans * plane + size_t(lc) * TILE_R + lr;
    double a = 0.0, b = 0.0, w = 0.0, wi = 0.0;
#pragma unroll 4
    for (uint32_t k = 0; k < n; k++, p += chans * plane) {
        a += p[0];
        b += p[plane];
        if (g.beam) {
            w += p[2 * plane];
            if (g.wproj)
                wi += p[3 * plane];
        }
    }
    const int r = (t % g.tiles_r) * TILE_R + lr, c = (t / g.tiles_r) * g.tc + lc;
    const bool cell = r < g.rows && c < g.N;
    if (cell)
        vgrid[size_t(r) + size_t(c) * g.rows] = { T(a), T(b) };
    if (!g.beam)
        return;
    if (!g.bpack) {
        if (cell)
            bgrid[size_t(r) + size_t(c) * g.rows] = { T(w), T(wi) };
        return;
    }
    lds[threadIdx.x] = w;
    __syncthreads();
    if (cell && !(lq & 1))
        bgrid[size_t(r) + size_t(c / 2) * g.rows] = { T(w), T(lds[threadIdx.x + 64]) };
}

// Workgroup 0: the last canonical level of the (good weights, good count) block pairs,
// which gives the sampling grid total 2 * sum(weights) and the good count, and the number
// of gridding entries (the end of the last tile's range).  The others merge split tiles.
template <typename T>
__global__ __launch_bounds__(CANON_LANES) void grid_total_kernel(const double* part, unsigned m, double* total,
    unsigned long long* ngood, const uint32_t* entries_end, unsigned long long* nentries, GridGeom g, Entry* entries,
    uint32_t cap, int ext_host, cplx<T>* vgrid, cplx<T>* bgrid)
{
    __shared__ double lds[2 * CANON_LANES];
    if (blockIdx.x > 0) {
        merge_body<T>(g, entries, cap, *entries_end, ext_host, vgrid, bgrid, int(blockIdx.x) - 1, lds);
        return;
    }
    double a, b;
    canon_last_level(part, m, a, b, lds);
    if (threadIdx.x == 0) {
        total[0] = a * 2.0;
        if (ngood)
            *ngood = (unsigned long long)b;
        if (nentries)
            *nentries = *entries_end;
    }
}

// ---------------------------------------------------------------------------
// Two-float tile sums (STP_PRECISION_FP32_TWOFLOAT): one workgroup per tile
// accumulates the taps of every entry binned to it in LDS, then writes the tile once.
// Lane mapping for supports up to 31: a wave takes 64 / ks entries at a time, lane
// (entry e, kernel column j) walks the ks kernel rows, so one load of kx[j] serves ks
// taps and the ks LDS atomics of a lane are independent.  Wider kernels take one entry
// per wave, lanes striding columns.  Each channel keeps an unevaluated pair hi + lo:
// the returning atomic add on hi yields the old value, so the rounding error of the
// sum it stored is known exactly (Knuth's TwoSum on old and x) and is added to lo.
constexpr int TWG = 512;
constexpr int TEB = 256;                  // entries staged per batch

constexpr int RG = 4;                     // kernel rows per group of LDS atomics

// Error of the rounded sum s = fl(old + x) (TwoSum).
__device__ __forceinline__ float two_sum_err(float old, float x)
{
    const float sum = old + x;
    const float bp = sum - old;
    return (old - (sum - bp)) + (x - bp);
}
// Two-float accumulation of FP32 taps: hi planes (re, im, beam), then lo planes.
struct AccTwoFloat {
    using S = float;
    static constexpr int arrays = 6;
    template <int R, typename T>
    __device__ static void add_rows(float* base, int plane, const int* aa, const T* xr, const T* xi,
        const T* xb, bool beam)
    {
        float orr[R], oi[R], ob[R];
        // returning adds on hi: each yields the old value, so the stored sum is fl(old + x)
#pragma unroll
        for (int u = 0; u < R; u++) {
            orr[u] = oi[u] = ob[u] = 0.f;
            if (aa[u] < 0)
                continue;
            orr[u] = atomicAdd(&base[aa[u]], xr[u]);
            oi[u] = atomicAdd(&base[plane + aa[u]], xi[u]);
            if (beam)
                ob[u] = atomicAdd(&base[2 * plane + aa[u]], xb[u]);
        }
        // the exact rounding errors go to the lo planes
#pragma unroll
        for (int u = 0; u < R; u++) {
            if (aa[u] < 0)
                continue;
            const float er = two_sum_err(orr[u], xr[u]), ei = two_sum_err(oi[u], xi[u]);
            if (er != 0.f)
                atomicAdd(&base[3 * plane + aa[u]], er);
            if (ei != 0.f)
                atomicAdd(&base[4 * plane + aa[u]], ei);
            if (beam) {
                const float eb = two_sum_err(ob[u], xb[u]);
                if (eb != 0.f)
                    atomicAdd(&base[5 * plane + aa[u]], eb);
            }
        }
    }
    __device__ static float value(const float* base, int plane, int ch, int a)
    {
        return base[ch * plane + a] + base[(3 + ch) * plane + a];
    }
};

// Writes a tile's sums once: the vis grid complex; the beam grid complex (imaginary
// part 0) or, with g.bpack, packed real: cell (r, c) is component c & 1 of element
// (r, c / 2) of a rows x N/2 complex array (tile columns come in even pairs).
template <typename T, typename Acc>
__device__ __forceinline__ void write_tile(const GridGeom& g, const typename Acc::S* acc, int plane, int S, int r0, int c0,
    cplx<T>* vgrid, cplx<T>* bgrid)
{
    for (int k = threadIdx.x; k < g.tc * TILE_R; k += TWG) {
        const int lr = k % TILE_R, lc = k / TILE_R;
        const int r = r0 + lr, c = c0 + lc;
        if (r < g.rows && c < g.N) {
            const size_t o = size_t(r) + size_t(c) * g.rows;
            const int a = lc * S + lr;
            vgrid[o] = { T(Acc::value(acc, plane, 0, a)), T(Acc::value(acc, plane, 1, a)) };
            if (g.beam && !g.bpack)
                bgrid[o] = { T(Acc::value(acc, plane, 2, a)), T(0) };
        }
    }
    if (g.beam && g.bpack)
        for (int k = threadIdx.x; k < (g.tc / 2) * TILE_R; k += TWG) {
            const int lr = k % TILE_R, lp = k / TILE_R;
            const int r = r0 + lr, c = c0 + 2 * lp;
            if (r < g.rows && c < g.N) {
                const int a = 2 * lp * S + lr;
                bgrid[size_t(r) + size_t(c / 2) * g.rows] = { T(Acc::value(acc, plane, 2, a)), T(Acc::value(acc, plane, 2, a + S)) };
            }
        }
}

template <typename T, typename Acc>
__global__ __launch_bounds__(TWG) void grid_tiles_twofloat_kernel(GridGeom g, const Entry* entries, const uint32_t* offsets, int ostride,
    uint32_t cap, const double* ktab, const double* uv, cplx<T>* vgrid, cplx<T>* bgrid)
{
#pragma clang fp contract(off)
    using AS = typename Acc::S;
    extern __shared__ double dyn[];
    __shared__ Entry ebuf[TEB];
    const int ks = g.ks, s = g.s;
    const int S = TILE_R + (ks <= 15 ? ks : 1);     // column stride of the LDS tile
    const int plane = g.tc * S;
    AS* acc = reinterpret_cast<AS*>(dyn);
    const int acc_bytes = Acc::arrays * plane * int(sizeof(AS));
    double* kv = dyn + (acc_bytes + 7) / 8;          // kernel table, or exact-mode vectors then sums
    const int cs = (g.os / 2) * 2 + 1;
    T* kt = reinterpret_cast<T*>(kv);
    double* ksum = kv + KV_DOUBLES;
    if (!g.exact)
        for (int k = threadIdx.x; k < cs * ks; k += TWG)
            kt[k] = T(ktab[k]);
    for (int k = threadIdx.x; k < Acc::arrays * plane; k += TWG)
        acc[k] = AS(0);
    const int t = blockIdx.x;
    const int rt = t % g.tiles_r, ct = t / g.tiles_r;
    const int r0 = rt * TILE_R, c0 = ct * g.tc;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int epw = ks <= 64 ? 64 / ks : 1;          // entries per wave pass
    const int slot = ks <= 64 ? lane / ks : 0;
    const int jl = ks <= 64 ? lane - slot * ks : lane;
    const bool lane_on = slot < epw;
    const uint32_t eb = min(offsets[size_t(t) * ostride], cap), ee = min(offsets[size_t(t + 1) * ostride], cap);
    const int batch = g.exact ? min(TEB, KV_DOUBLES / (2 * ks)) : TEB;
    for (uint32_t e0 = eb; e0 < ee; e0 += uint32_t(batch)) {
        const int cnt = int(min(uint32_t(batch), ee - e0));
        __syncthreads();
        if (int(threadIdx.x) < cnt) {
            const Entry E = entries[e0 + threadIdx.x];
            ebuf[threadIdx.x] = E;
            if (g.exact) {
                // exact kernel of this visibility pass (make_kernel_array, conv_func.h:279-303)
                const long long vi = E.idx >> 1;
                double uu = uv[vi] * g.scale, vv = uv[g.n + vi] * g.scale;
                if (g.halfplane && vv < 0.0) {
                    uu = -uu;
                    vv = -vv;
                }
                double fx = uu - int(rint(uu)), fy = vv - int(rint(vv));
                if (E.idx & 1) {
                    fx = -fx;
                    fy = -fy;
                }
                double* ky = &kv[2 * ks * threadIdx.x];
                double* kx = ky + ks;
                double sx = 0.0, sy = 0.0;
                for (int q = 0; q < ks; q++) {
                    ky[q] = dev_kernel(g, double(q - s) - fy);
                    kx[q] = dev_kernel(g, double(q - s) - fx);
                    sy += ky[q];
                    sx += kx[q];
                }
                ksum[threadIdx.x] = sx * sy;
            }
        }
        __syncthreads();
        for (int q0 = wave * epw; q0 < cnt; q0 += (TWG / 64) * epw) {
            const int q = q0 + slot;
            if (!lane_on || q >= cnt)
                continue;
            const Entry& E = ebuf[q];
            const int cpx = E.cp & 0xffff, cpy = E.cp >> 16;
            const T w = T(E.w), vr = T(E.vr), vim = T(E.vi);
            const double* kyd = g.exact ? &kv[2 * ks * q] : nullptr;
            const double inv = g.exact ? ksum[q] : 1.0;
            for (int j = jl; j < ks; j += (ks <= 64 ? ks : 64)) {
                const int c = tap_col(g, E.gx, j);
                const int lc = c - c0;
                if (lc < 0 || lc >= g.tc)
                    continue;
                const double kxd = g.exact ? kyd[ks + j] : 0.0;
                const T kx = g.exact ? T(0) : kt[cpx * ks + j];
                // RG kernel rows at a time: their atomics are issued back to back
                for (int i0 = 0; i0 < ks; i0 += RG) {
                    int aa[RG];
                    T xr[RG], xi[RG], xb[RG];
#pragma unroll
                    for (int u = 0; u < RG; u++) {
                        const int i = i0 + u;
                        aa[u] = -1;
                        xr[u] = xi[u] = xb[u] = T(0);
                        if (i >= ks)
                            continue;
                        const int r = tap_row(g, E.gy, i);
                        const int lr = r - r0;
                        if (r < 0 || lr < 0 || lr >= TILE_R)
                            continue;
                        T K;
                        if (g.exact)
                            K = T((kyd[i] * kxd) / inv);
                        else
                            K = kt[cpy * ks + i] * kx;
                        const T kw = K * w; // gridder.h:854-858
                        aa[u] = lc * S + lr;
                        xr[u] = vr * kw;
                        xi[u] = vim * kw;
                        xb[u] = kw;
                    }
                    Acc::template add_rows<RG, T>(acc, plane, aa, xr, xi, xb, g.beam != 0);
                }
            }
        }
    }
    __syncthreads();
    write_tile<T, Acc>(g, acc, plane, S, r0, c0, vgrid, bgrid);
}

// Oversampled-kernel tiles with ks <= KSM taps per side (the common case): the
// same lane mapping and tap arithmetic as grid_tiles_twofloat_kernel, specialised so a
// lane preloads its entry's ks kernel-row values and computes row validity
// without branches; taps that miss the tile issue no LDS atomic.
template <typename T, typename Acc, int KSM>
__device__ __forceinline__ void tiles_os_body(const GridGeom& g, const Entry* entries, const uint32_t* offsets, int ostride,
    uint32_t cap, const double* ktab, cplx<T>* vgrid, cplx<T>* bgrid, int t)
{
#pragma clang fp contract(off)
    using AS = typename Acc::S;
    extern __shared__ double dyn[];
    __shared__ Entry ebuf[TEB];
    const int ks = g.ks, s = g.s;
    const int S = TILE_R + (ks <= 15 ? ks : 1);     // column stride of the LDS tile
    const int plane = g.tc * S;
    AS* acc = reinterpret_cast<AS*>(dyn);
    const int acc_bytes = Acc::arrays * plane * int(sizeof(AS));
    T* kt = reinterpret_cast<T*>(dyn + (acc_bytes + 7) / 8);
    const int cs = (g.os / 2) * 2 + 1;
    for (int k = threadIdx.x; k < cs * ks; k += TWG)
        kt[k] = T(ktab[k]);
    for (int k = threadIdx.x; k < Acc::arrays * plane; k += TWG)
        acc[k] = AS(0);
    const int rt = t % g.tiles_r, ct = t / g.tiles_r;
    const int r0 = rt * TILE_R, c0 = ct * g.tc;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int epw = 64 / ks;                         // entries per wave pass
    const int slot = lane / ks;
    const int jl = lane - slot * ks;
    const bool lane_on = slot < epw;
    const uint32_t eb = min(offsets[size_t(t) * ostride], cap), ee = min(offsets[size_t(t + 1) * ostride], cap);
    for (uint32_t e0 = eb; e0 < ee; e0 += uint32_t(TEB)) {
        const int cnt = int(min(uint32_t(TEB), ee - e0));
        __syncthreads();
        if (int(threadIdx.x) < cnt)
            ebuf[threadIdx.x] = entries[e0 + threadIdx.x];
        __syncthreads();
        for (int q0 = wave * epw; q0 < cnt; q0 += (TWG / 64) * epw) {
            const int q = q0 + slot;
            if (!lane_on || q >= cnt)
                continue;
            const Entry& E = ebuf[q];
            const int lc = tap_col(g, E.gx, jl) - c0;
            if (lc < 0 || lc >= g.tc)
                continue;
            const int cpx = E.cp & 0xffff, cpy = E.cp >> 16;
            const T w = T(E.w), vr = T(E.vr), vim = T(E.vi);
            const T kx = kt[cpx * ks + jl];
            T ky[KSM];
#pragma unroll
            for (int i = 0; i < KSM; i++)
                ky[i] = i < ks ? kt[cpy * ks + i] : T(0);
            const int rb = E.gy - s, cb = lc * S;
#pragma unroll
            for (int i0 = 0; i0 < KSM; i0 += RG) {
                int aa[RG];
                T xr[RG], xi[RG], xb[RG];
#pragma unroll
                for (int u = 0; u < RG; u++) {
                    const int i = i0 + u;
                    // tap_row: rows < 0 skipped, rows >= N wrapped, rows >= rows dropped
                    int r = rb + i;
                    bool ok = i < ks && r >= 0;
                    r = r >= g.N ? r - g.N : r;
                    const int lr = r - r0;
                    ok = ok && r < g.rows && lr >= 0 && lr < TILE_R;
                    const T kw = (ky[i] * kx) * w; // gridder.h:854-858
                    aa[u] = ok ? cb + lr : -1;
                    xr[u] = vr * kw;
                    xi[u] = vim * kw;
                    xb[u] = kw;
                }
                Acc::template add_rows<RG, T>(acc, plane, aa, xr, xi, xb, g.beam != 0);
            }
        }
    }
    __syncthreads();
    write_tile<T, Acc>(g, acc, plane, S, r0, c0, vgrid, bgrid);
}

template <typename T, typename Acc, int KSM>
__global__ __launch_bounds__(TWG) void grid_tiles_os_kernel(GridGeom g, const Entry* entries, const uint32_t* offsets,
    int ostride, uint32_t cap, const double* ktab, cplx<T>* vgrid, cplx<T>* bgrid)
{
    tiles_os_body<T, Acc, KSM>(g, entries, offsets, ostride, cap, ktab, vgrid, bgrid, int(blockIdx.x));
}

// ---------------------------------------------------------------------------
// W-projection (gridder.h:311-367,467-486,767-842; aw_projection.cpp:19-210,366-474)
//
//  1. |w| order: stable LSD radix sort of the 64-bit keys bits(|w|) with the
//     visibility index as payload (the reference's arma::sort_index, gridder.h:324,
//     with ties kept in index order).
//  2. planes: good flags in |w| order, their prefix sum, then the equal-count plane
//     boundaries and plane |w| (mean or median) of average_w_planes
//     (gridder.cpp:68-146) on the device.
//  3. W-kernels per plane: the image-domain kernel aa(x) aa(y) exp(-2 pi i w (n-1)) / n
//     on an (workarea * os)^2 array, its forward 2-D DFT at the frequencies the cuts
//     read, and the oversampled (2s+1)^2 kernels cut from it, each normalised by its real sum.
//  4. gridding: the entries of every plane binned by tile together; the tile
//     kernel reads each entry's complex kernel from its plane's cache, so the grid
//     is written once for all planes.
// Radix sort of the 63 key bits by seven digits of nine.  A block of eight waves takes
// RS_STEPS x 512 keys, a wave RS_STEPS x 64 of them in order.  Bound by the latency of its
// launches at some hundred thousand keys (300 k: 175 us), then by the scattered stores
// (2 M: 440 us).  With eight-bit digits, one wave per 1024 keys and a scan in between an
// image of 300 k visibilities took 694 us in all, now 593 us.
constexpr int RS_BITS = 9, RS_DIGITS = 1 << RS_BITS, RS_WAVES = 8, RS_THREADS = 64 * RS_WAVES, RS_PASSES = 7;
static_assert(RS_DIGITS == RS_THREADS, "a thread per digit");
static_assert(RS_BITS * RS_PASSES == 63, "|w| has no sign bit");
// Up to this many blocks every scatter block adds up their counts itself: 7 x 18 us against
// 7 x (14 + 6) us for 74 blocks and a scan between; 7 x 55 us against 7 x (44 + 9) us for 245.
constexpr int RS_SELF = 128;

// Key k of a pass; the first pass (src NULL) reads |w|.
__device__ __forceinline__ unsigned long long rs_key(const unsigned long long* src, const double* w, long long k)
{
    return src ? src[k] : (unsigned long long)__double_as_longlong(fabs(w[k]));
}

// counts[block][digit]
template <int RS_STEPS>
__global__ __launch_bounds__(RS_THREADS) void rs_hist_kernel(const unsigned long long* key, const double* w, long long n, int shift,
    uint32_t* counts)
{
    __shared__ uint32_t h[RS_DIGITS];
    h[threadIdx.x] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * RS_STEPS * RS_THREADS;
    unsigned long long k[RS_STEPS];
#pragma unroll
    for (int j = 0; j < RS_STEPS; j++)
        k[j] = rs_key(key, w, min(base + j * RS_THREADS + threadIdx.x, n - 1));
#pragma unroll
    for (int j = 0; j < RS_STEPS; j++)
        if (base + j * RS_THREADS + threadIdx.x < n)
            atomicAdd(&h[(k[j] >> shift) & (RS_DIGITS - 1)], 1u);
    __syncthreads();
    counts[size_t(blockIdx.x) * RS_DIGITS + threadIdx.x] = h[threadIdx.x];
}

// Stable scatter of a block's keys.  A wave ranks its keys 64 at a time: lanes with
// equal digits find each other by ballots on the digit's bits and follow the wave's
// earlier ones; the waves' counts, in order, and the block's offset place them.
// totals: per digit, and counts[block][digit] the keys of earlier blocks (column scan);
// NULL: the counts themselves (few blocks), added up here.
template <int RS_STEPS>
__global__ __launch_bounds__(RS_THREADS) void rs_scatter_kernel(const unsigned long long* kin, const uint32_t* iin, const double* w,
    long long n, int shift, const uint32_t* counts, const uint32_t* totals, int nblk, unsigned long long* kout, uint32_t* iout)
{
    __shared__ uint32_t cnt[RS_WAVES][RS_DIGITS];
    __shared__ uint32_t wsum[RS_WAVES];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const long long base = (long long)blockIdx.x * RS_STEPS * RS_THREADS + (long long)wave * RS_STEPS * 64 + lane;
    unsigned long long k[RS_STEPS];
    uint32_t idx[RS_STEPS], rank[RS_STEPS];
#pragma unroll
    for (int j = 0; j < RS_STEPS; j++) {
        const long long i = min(base + j * 64, n - 1);
        k[j] = rs_key(kin, w, i);
        idx[j] = kin ? iin[i] : uint32_t(i);
    }
    // this thread's digit: its keys in earlier blocks, and in all
    uint32_t before = 0, total = 0;
    if (totals) {
        before = counts[size_t(blockIdx.x) * RS_DIGITS + t];
        total = totals[t];
    } else {
        for (int b0 = 0; b0 < nblk; b0 += 16) {
            uint32_t v[16];
#pragma unroll
            for (int j = 0; j < 16; j++)
                v[j] = counts[size_t(min(b0 + j, nblk - 1)) * RS_DIGITS + t];
#pragma unroll
            for (int j = 0; j < 16; j++) {
                total += b0 + j < nblk ? v[j] : 0u;
                before += b0 + j < int(blockIdx.x) ? v[j] : 0u;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < RS_WAVES; q++)
        cnt[q][t] = 0;
    uint32_t x = total;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off)
            x += y;
    }
    if (lane == 63)
        wsum[wave] = x;
    __syncthreads();
    uint32_t start = x - total + before;
    for (int q = 0; q < wave; q++)
        start += wsum[q];
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int j = 0; j < RS_STEPS; j++) {
        const bool valid = base + j * 64 < n;
        const uint32_t d = uint32_t(k[j] >> shift) & (RS_DIGITS - 1);
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < RS_BITS; b++) {
            const bool bit = (d >> b) & 1u;
            const unsigned long long m = __ballot(valid && bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t mine = uint32_t(__popcll(peers & below));
        const uint32_t prev = cnt[wave][d];
        __builtin_amdgcn_wave_barrier();
        if (valid && mine == 0)
            cnt[wave][d] = prev + uint32_t(__popcll(peers));
        __builtin_amdgcn_wave_barrier();
        rank[j] = prev + mine;
    }
    __syncthreads();
    // the waves' first places, in wave order
#pragma unroll
    for (int q = 0; q < RS_WAVES; q++) {
        const uint32_t c = cnt[q][t];
        cnt[q][t] = start;
        start += c;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_STEPS; j++) {
        if (base + j * 64 >= n)
            continue;
        const uint32_t at = cnt[wave][uint32_t(k[j] >> shift) & (RS_DIGITS - 1)] + rank[j];
        kout[at] = k[j];
        iout[at] = idx[j];
    }
}

// The inputs in |w| order, gathered once: uv (u, v, w columns), vis and weights of
// sorted position k from original position perm[k], so the later passes read them
// in sequence instead of gathering each time.
__global__ void wpermute_kernel(const double* uvw, const double* vis, const double* wts, const uint32_t* perm, long long n,
    double* uvw_s, double* vis_s, double* wts_s)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n)
        return;
    const long long i = perm[k];
    const double u = uvw[i], v = uvw[n + i], w = uvw[2 * n + i];
    const double vr = vis[2 * i], vi = vis[2 * i + 1], wt = wts[i];
    uvw_s[k] = u;
    uvw_s[n + k] = v;
    uvw_s[2 * n + k] = w;
    vis_s[2 * k] = vr;
    vis_s[2 * k + 1] = vi;
    wts_s[k] = wt;
}

__global__ void wgood_kernel(GridGeom g, const double* uvw, const double* vis, const double* wts, uint32_t* flag)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= g.n)
        return;
    flag[k] = prep_vis(g, uvw, vis, wts, k).good ? 1u : 0u;
}

// Smallest k in [lo, hi) with G[k] >= target (G non-decreasing), or hi, found by
// one full wave: 64 probes per step narrow the range 64-fold, so a search over 2^21
// positions takes four dependent loads instead of 21.  Every lane returns the result.
__device__ unsigned long long lower_bound_wave(const uint32_t* G, unsigned long long lo, unsigned long long hi,
    unsigned long long target)
{
    const unsigned long long lane = threadIdx.x & 63;
    // with few values that do not count, the answer lies near lo + target - G[lo - 1] - 1
    if (hi - lo > 64 && lo > 0) {
        const unsigned long long skip = target - min(target, (unsigned long long)G[lo - 1] + 1);
        const unsigned long long mid = lo + min(skip, hi - lo), a = mid - min(mid - lo, 32ull);
        const unsigned long long m = __ballot((unsigned long long)G[min(a + lane, hi - 1)] >= target);
        if (m && (a == lo || !(m & 1ull)))
            return a + (unsigned long long)__builtin_ctzll(m);
    }
    while (hi - lo > 64) {
        const unsigned long long step = (hi - lo + 63) / 64;
        const unsigned long long q = lo + lane * step;
        const unsigned long long m = __ballot(q >= hi || (unsigned long long)G[q] >= target);
        const int f = m ? __builtin_ctzll(m) : 64;
        if (f == 0)
            return lo;
        // the answer lies in (probe f-1, probe f]
        const unsigned long long nlo = lo + (unsigned long long)(f - 1) * step + 1;
        const unsigned long long nhi = f == 64 ? hi : min(hi, lo + (unsigned long long)f * step);
        lo = nlo;
        hi = nhi;
    }
    const unsigned long long q = lo + lane;
    const unsigned long long m = __ballot(q >= hi || (unsigned long long)G[q] >= target);
    return m ? lo + (unsigned long long)__builtin_ctzll(m) : hi;
}

// average_w_planes (gridder.cpp:68-146) over the |w|-sorted good flags: G is their
// exclusive prefix sum (G[n] = number of good visibilities).  One wave (the planes
// are sequential: each starts where the last stopped).  Writes first[0..P]
// (first[P] = n), first[P+1] (where the last plane's count stopped), the good count
// of each plane, and for the median variant the plane |w|.
__global__ __launch_bounds__(64) void wplane_bounds_kernel(const uint32_t* G, long long n, int P, int median,
    const unsigned long long* skey, uint32_t* first, uint32_t* count, double* w_plane)
{
    const bool lead = threadIdx.x == 0;
    const unsigned long long num_gvis = G[n];
    unsigned long long begin = 0;
    auto wv = [&](unsigned long long k) { return __longlong_as_double((long long)skey[k]); };
    for (int p = 0; p < P; p++) {
        // with many rejected visibilities the position `begin` passes the good count and the
        // unsigned difference wraps (the reference's own arithmetic): a size past 64 bits, which
        // only the last plane can have, is none, as the reference's conversion gives on x86
        const double size = ceil(double(num_gvis - begin) / double(P - p));
        const unsigned long long plane_size = size < 18446744073709551616.0 ? (unsigned long long)size : 0ull;
        unsigned long long k = begin, counter = 0;
        if (plane_size > 0 && begin < (unsigned long long)n) {
            const unsigned long long target = (unsigned long long)G[begin] + plane_size;
            k = lower_bound_wave(G, begin + 1, (unsigned long long)n, target);
            counter = (unsigned long long)G[k] - G[begin];
        }
        if (lead) {
            first[p] = uint32_t(begin);
            count[p] = uint32_t(counter);
        }
        if (median) {
            unsigned long long middle = plane_size / 2;
            if ((begin + plane_size) > num_gvis)
                middle = (num_gvis - begin) / 2;
            double v = 0.0;
            if (counter > 0) {
                // the good element with counter == middle: the first position whose
                // inclusive good count reaches middle + 1
                const unsigned long long mid = lower_bound_wave(G, begin + 1, k, (unsigned long long)G[begin] + middle + 1) - 1;
                v = (plane_size % 2 == 0 && mid > 0) ? (wv(mid - 1) + wv(mid)) / 2.0 : wv(mid);
            }
            if (lead)
                w_plane[p] = v;
        }
        begin = k;
    }
    // the last plane grids every position up to n (gridder.h:532-533); its count
    // stopped at `begin`
    if (lead) {
        first[P] = uint32_t(n);
        first[P + 1] = uint32_t(begin);
    }
}

// Mean |w| of each plane's counted good visibilities: those in [first[p],
// first[p+1]), except for the last plane, whose count stops at first[P+1] (with
// rejected visibilities before it, the reference's plane size, computed from a
// position rather than a good count, stops short of n).  WMS blocks per plane sum
// fixed slices (part[p * WMS + slice]); a second kernel adds the slices in order.
constexpr int WMS = 32;
__global__ __launch_bounds__(256) void wplane_sum_kernel(const unsigned long long* skey, const uint32_t* flag,
    const uint32_t* first, double* part)
{
    __shared__ double red[256];
    const int p = blockIdx.x, sl = blockIdx.y;
    const unsigned long long b = first[p];
    const unsigned long long end = p + 1 == int(gridDim.x) ? first[p + 2] : first[p + 1];
    const unsigned long long len = end > b ? end - b : 0, per = (len + WMS - 1) / WMS;
    const unsigned long long s0 = b + min(len, sl * per), s1 = b + min(len, (sl + 1) * per);
    double sum = 0.0;
    for (unsigned long long k = s0 + threadIdx.x; k < s1; k += 256)
        if (flag[k])
            sum += __longlong_as_double((long long)skey[k]);
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off)
            red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        part[p * WMS + sl] = red[0];
}

__global__ void wplane_mean_kernel(const double* part, const uint32_t* count, int P, double* w_plane)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P)
        return;
    double sum = 0.0;
    for (int sl = 0; sl < WMS; sl++)
        sum += part[p * WMS + sl];
    w_plane[p] = count[p] > 0 ? sum / double(count[p]) : 0.0;
}

__global__ void wplane_ids_kernel(const uint32_t* first, int P, long long n, uint16_t* plane)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n)
        return;
    int lo = 0, hi = P - 1; // last plane p with first[p] <= k
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if ((long long)first[mid] <= k)
            lo = mid;
        else
            hi = mid - 1;
    }
    plane[k] = uint16_t(lo);
}

// generate_image_domain_convolution_kernel (aw_projection.cpp:50-111): the quadrant
// q[p + r half] of the image-domain kernel at pixel offsets p, r = 0 .. half - 1 (the kernel
// is even along both axes and zero beyond).  blockIdx.y: plane p0 + blockIdx.y.
__global__ void wk_fill_kernel(cplx<double>* quad, int half, const double* aa, const double* w_plane, int p0,
    double scaled_cell)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= half * half)
        return;
    const int pi = e % half, pj = e / half;
    // combine_2d_kernel_value (aw_projection.cpp:455-474)
    const double a = aa[half + pi] * aa[half + pj];
    cplx<double> v{ a, 0.0 };
    if (pi != 0 || pj != 0) {
        const double dx = double(pi) * scaled_cell, dy = double(pj) * scaled_cell;
        const double r2 = dx * dx + dy * dy;
        if (r2 < 1.0) {
            const double nn = sqrt(1.0 - r2);
            const double ph = (-2.0 * M_PI) * w_plane[p0 + int(blockIdx.y)] * (nn - 1.0);
            double sn, cs;
            sincos(ph, &sn, &cs);
            v.x = ((cs / nn) * aa[half + pi]) * aa[half + pj];
            v.y = ((sn / nn) * aa[half + pi]) * aa[half + pj];
        }
    }
    quad[size_t(blockIdx.y) * half * half + e] = v;
}

// One axis of the forward 2-D DFT of the even image-domain kernel (aw_projection.cpp:194),
// which is a cosine sum over the quadrant:
//   out[i * ldo + pos] = sum_k c_k x[k * ldx + i] cos(2 pi n(pos) k / arr),  c_0 = 1, c_k = 2,
// for the output frequencies that the oversampled cuts read: n(pos) = (pos % len) os + pos / len,
// so that a cut's samples, os apart, lie side by side.  As FP64 matrix products, a wave per
// 16 x 16 outputs; cos from the twiddle table of arr points.  A quadrant of 64 x 64 and 264
// frequencies take 22 Mflop per plane; the padded 1024 x 1024 FFT moved 48 MB for it (0.87 ms
// for 32 planes against 0.06).
__global__ __launch_bounds__(256) void wk_cosine_kernel(const cplx<double>* x, size_t xstride, int ldx, int ni, int nk,
    cplx<double>* out, size_t ostride, int npos, int len, int os, const cplx<double>* tw, int arr)
{
    const int lane = threadIdx.x & 63, m = lane & 15, kk = lane >> 4;
    const int ib = 16 * blockIdx.y, jb = 64 * blockIdx.x + 16 * (threadIdx.x >> 6);
    x += blockIdx.z * xstride;
    out += blockIdx.z * ostride;
    const int i = min(ib + m, ni - 1), pos = min(jb + m, npos - 1);
    const int n = (pos % len) * os + pos / len;
    double4v re = { 0, 0, 0, 0 }, im = { 0, 0, 0, 0 };
#pragma unroll 4
    for (int k0 = 0; k0 < nk; k0 += 4) {
        const int k = min(k0 + kk, nk - 1);
        const cplx<double> v = x[size_t(k) * ldx + i];
        double c = tw[(n * k) & (arr - 1)].x;
        c = k0 + kk >= nk ? 0.0 : (k == 0 ? c : 2.0 * c);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(v.x, c, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(v.y, c, im, 0, 0, 0);
    }
    // lane (m, kk) holds rows i = kk + 4 v, position m of the block
#pragma unroll
    for (int v = 0; v < 4; v++)
        if (ib + kk + 4 * v < ni && jb + m < npos)
            out[size_t(ib + kk + 4 * v) * npos + jb + m] = { re[v], im[v] };
}

// Each sub-kernel is stored column-major with WPAD zero columns on both sides, so that the
// W tile kernel's column runs starting up to WPAD columns outside the kernel read zeros.
constexpr int WPAD = W_KERNEL_PAD_COLS;
// A kernel of ks taps per side is a zero, then ks + 2 WPAD columns of ks values and a zero
// each, so that the rows before and after every column read zero too.
__host__ __device__ constexpr size_t w_slot(int ks) { return size_t(1) + size_t(ks + 1) * (ks + 2 * WPAD); }

// ---------------------------------------------------------------------------
// Hankel W-kernels (hankel_opt; aw_projection.cpp:211-287,380-411, aw_projection.h:127-213)
//
// Per plane: a 1-D profile (the radial screen times the AA kernel, or the
// projection of the 2-D image-domain kernel onto one axis), its transform (the
// DHT, or the forward DFT), the truncated support, a natural cubic or linear
// spline through the transform at radii 0, 1, ..., the spline sampled on the half
// quadrant {(ii, j): ii <= j < ko}, ko = (s + 1) os, at radius sqrt(ii^2 + j^2), and
// the (os+1)^2 cuts of that radially symmetric kernel, each normalised by its real
// sum.  One block per plane for the sequential parts (the spline's tridiagonal
// solve), one thread per output for the transforms.
struct HankelArgs {
    int n;          // transform length: arr / 2 (DHT) or arr (projection slice)
    int half;       // workarea / 2
    int arr;        // workarea * os
    int os, support;
    int proj_slice, cubic;
    double scaled_cell, trunc_frac;
    int kh_stride;  // half-quadrant values per plane (for the maximum support)
};

// combine_2d_kernel_value (aw_projection.cpp:455-474) at pixel offsets (px, py)
__device__ cplx<double> wk_combine(const double* aa, int half, int px, int py, double w, double sc)
{
    const double dx = double(px) * sc, dy = double(py) * sc;
    const double r2 = dx * dx + dy * dy;
    if (r2 >= 1.0)
        return { aa[half + px] * aa[half + py], 0.0 };
    const double nn = sqrt(1.0 - r2);
    const double ph = (-2.0 * M_PI) * w * (nn - 1.0);
    double sn, cs;
    sincos(ph, &sn, &cs);
    return { ((cs / nn) * aa[half + px]) * aa[half + py], ((sn / nn) * aa[half + px]) * aa[half + py] };
}

// Profiles of one plane per block: prof[p * n + i].
__global__ __launch_bounds__(256) void wk_hankel_profile_kernel(HankelArgs h, const double* aa, const double* w_plane,
    cplx<double>* prof)
{
#pragma clang fp contract(off)
    const int p = blockIdx.x;
    const double w = w_plane[p];
    cplx<double>* out = prof + size_t(p) * h.n;
    if (!h.proj_slice) {
        // the radial screen along x times aa(x) (aw_projection.cpp:224-239)
        for (int i = threadIdx.x; i < h.n; i += 256) {
            cplx<double> v{ 0.0, 0.0 };
            if (i < h.half) {
                const double dx = double(i) * h.scaled_cell;
                const double r2 = dx * dx;
                double tr = 1.0, ti = 0.0;
                if (r2 < 1.0) {
                    const double nn = sqrt(1.0 - r2);
                    const double ph = (-2.0 * M_PI) * w * (nn - 1.0);
                    double sn, cs;
                    sincos(ph, &sn, &cs);
                    tr = cs / nn;
                    ti = sn / nn;
                }
                v = { tr * aa[h.half + i], ti * aa[h.half + i] };
            }
            out[i] = v;
        }
        return;
    }
    // generate_projected_image_domain_kernel (aw_projection.cpp:113-171): column sums
    // of the 2-D kernel, each sum in the reference's order
    for (int j = threadIdx.x; j < h.n; j += 256) {
        cplx<double> v{ 0.0, 0.0 };
        if (j == 0) {
            // twice the axis values (1 .. half-1) plus the centre
            double sr = 0.0, si = 0.0;
            for (int i = 1; i < h.half; i++) {
                const cplx<double> c = wk_combine(aa, h.half, i, 0, w, h.scaled_cell);
                sr += c.x;
                si += c.y;
            }
            v = { sr * 2.0 + aa[h.half] * aa[h.half], si * 2.0 };
        } else {
            const int jj = j < h.half ? j : (j > h.arr - h.half ? h.arr - j : -1);
            if (jj > 0) {
                v = wk_combine(aa, h.half, jj, 0, w, h.scaled_cell);
                for (int i = 1; i < h.half; i++) {
                    const cplx<double> c = wk_combine(aa, h.half, i, jj, w, h.scaled_cell);
                    v.x += c.x * 2.0;
                    v.y += c.y * 2.0;
                }
            }
        }
        out[j] = v;
    }
}

// y[p * n + i] = sum_j T(j, i) prof[p * n + j], j in order: T = the DHT (tab[j * n + i])
// or the forward DFT (tab = exp(-2 pi i m / n) interleaved, m = j i mod n).
__global__ __launch_bounds__(256) void wk_hankel_transform_kernel(HankelArgs h, const double* tab,
    const cplx<double>* prof, cplx<double>* y)
{
#pragma clang fp contract(off)
    const int i = blockIdx.x * 256 + threadIdx.x, p = blockIdx.y;
    if (i >= h.n)
        return;
    const cplx<double>* x = prof + size_t(p) * h.n;
    double ar = 0.0, ai = 0.0;
    if (!h.proj_slice) {
        for (int j = 0; j < h.n; j++) {
            const double d = tab[size_t(j) * h.n + i];
            ar += d * x[j].x;
            ai += d * x[j].y;
        }
    } else {
        unsigned long long m = 0;
        for (int j = 0; j < h.n; j++) {
            const double c = tab[2 * m], sn = tab[2 * m + 1];
            ar += x[j].x * c - x[j].y * sn;
            ai += x[j].x * sn + x[j].y * c;
            m += (unsigned long long)i;
            if (m >= (unsigned long long)h.n)
                m -= (unsigned long long)h.n;
        }
    }
    y[size_t(p) * h.n + i] = { ar, ai };
}

// Truncated support (aw_projection.h:132-148) and spline coefficients of one plane:
// lane 0 the real part, lane 1 the imaginary part.  coef[(p * 2 + part) * 5 + {a, b,
// c, d, r}][k]; the natural cubic spline on the knots 0, 1, ... solves its
// tridiagonal system (rows 0 and n-1: 2 b = 0; else (1/3, 4/3, 1/3) against the
// second differences) by forward elimination and back substitution.
__global__ __launch_bounds__(64) void wk_hankel_spline_kernel(HankelArgs h, const cplx<double>* y, double* coef, int* psup)
{
#pragma clang fp contract(off)
    const int p = blockIdx.x, part = threadIdx.x;
    const int n = h.n;
    const cplx<double>* yp = y + size_t(p) * n;
    if (part == 0) {
        int ts = h.support;
        if (h.trunc_frac > 0.0) {
            const double min_value = hypot(yp[0].x, yp[0].y) * h.trunc_frac;
            int idx = h.support * h.os;
            const double scale = 1.0 / double(h.os);
            while (idx > h.os) {
                if (hypot(yp[idx].x, yp[idx].y) > min_value)
                    break;
                idx -= h.os;
            }
            ts = min(int(ceil(double(idx) * scale)), h.support);
        }
        psup[p] = ts;
    }
    if (part > 1)
        return;
    double* a = coef + (size_t(p) * 2 + part) * 5 * n;
    double* b = a + n;
    double* c = b + n;
    double* d = c + n;
    double* r = d + n;
    auto yv = [&](int k) { return part ? yp[k].y : yp[k].x; };
    if (!h.cubic) {
        for (int k = 0; k + 1 < n; k++) {
            c[k] = (yv(k + 1) - yv(k)) / 1.0;
            a[k] = b[k] = 0.0;
        }
        c[n - 1] = c[n - 2];
        a[n - 1] = b[n - 1] = 0.0;
        return;
    }
    const double lo = 1.0 / 3.0 * 1.0, di = 2.0 / 3.0 * 2.0, up = 1.0 / 3.0 * 1.0;
    d[0] = 2.0;
    r[0] = 0.0;
    for (int k = 1; k < n; k++) {
        const bool last = k == n - 1;
        const double lk = last ? 0.0 : lo, dk = last ? 2.0 : di;
        const double rk = last ? 0.0 : (yv(k + 1) - yv(k)) / 1.0 - (yv(k) - yv(k - 1)) / 1.0;
        const double m = lk / d[k - 1];
        d[k] = dk - m * (k == 1 ? 0.0 : up);
        r[k] = rk - m * r[k - 1];
    }
    b[n - 1] = r[n - 1] / d[n - 1];
    for (int k = n - 2; k >= 0; k--)
        b[k] = (r[k] - (k == 0 ? 0.0 : up) * b[k + 1]) / d[k];
    for (int k = 0; k + 1 < n; k++) {
        a[k] = 1.0 / 3.0 * (b[k + 1] - b[k]) / 1.0;
        c[k] = (yv(k + 1) - yv(k)) / 1.0 - 1.0 / 3.0 * (2.0 * b[k] + b[k + 1]) * 1.0;
    }
    a[n - 1] = 0.0;
    c[n - 1] = 3.0 * a[n - 2] * 1.0 * 1.0 + 2.0 * b[n - 2] * 1.0 + c[n - 2];
}

// The spline on the half quadrant of one plane (RadialInterpolate's loop): row ii
// holds j = ii .. ko-1 at kh[p * stride + ii ko - ii (ii - 1) / 2 + j - ii].
__global__ __launch_bounds__(256) void wk_hankel_quad_kernel(HankelArgs h, const cplx<double>* y, const double* coef,
    const int* psup, cplx<double>* kh)
{
#pragma clang fp contract(off)
    const int p = blockIdx.y, n = h.n;
    const int ko = (psup[p] * 2 + 2) * h.os / 2;
    const long long total = (long long)ko * (ko + 1) / 2;
    const cplx<double>* yp = y + size_t(p) * n;
    const double* cr = coef + size_t(p) * 2 * 5 * n;
    const double* ci = cr + 5 * size_t(n);
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < total; q += (long long)gridDim.x * 256) {
        // row ii: the largest with ii ko - ii (ii - 1) / 2 <= q
        int ii = int((double(2 * ko + 1) - sqrt(double(2 * ko + 1) * double(2 * ko + 1) - 8.0 * double(q))) / 2.0);
        ii = max(0, min(ii, ko - 1));
        while (ii > 0 && (long long)ii * ko - (long long)ii * (ii - 1) / 2 > q)
            ii--;
        while (ii + 1 < ko && (long long)(ii + 1) * ko - (long long)(ii + 1) * ii / 2 <= q)
            ii++;
        const int j = int(q - ((long long)ii * ko - (long long)ii * (ii - 1) / 2)) + ii;
        const double nx = ii == 0 ? double(j) : sqrt(double((long long)ii * ii + (long long)j * j));
        int k = int(nx);
        if (k >= n)
            k = n - 1;
        const double hh = nx - double(k);
        double vr, vi;
        if (h.cubic) {
            vr = ((cr[k] * hh + cr[n + k]) * hh + cr[2 * n + k]) * hh + yp[k].x;
            vi = ((ci[k] * hh + ci[n + k]) * hh + ci[2 * n + k]) * hh + yp[k].y;
        } else {
            vr = cr[2 * n + k] * hh + yp[k].x;
            vi = ci[2 * n + k] * hh + yp[k].y;
        }
        kh[size_t(p) * h.kh_stride + q] = { vr, vi };
    }
}

// generate_kernel_cache, Hankel branch (aw_projection.cpp:380-411): cut (x, y) of the
// radially symmetric kernel, element (row tx, column ty) at offsets
// cx = -ts os + os/2 - x + ty os, cy = ... - y + tx os, divided by the cut's real sum;
// stored like wk_extract_kernel's cuts (padded columns, truncated kernels centred).
template <typename KT>
__global__ __launch_bounds__(256) void wk_hankel_extract_kernel(HankelArgs h, const cplx<double>* kh, const int* psup,
    int p0, cplx<KT>* cache)
{
    __shared__ double red[256];
    const int p = p0 + int(blockIdx.y);
    const int cs = h.os / 2 + 1;
    const int x = blockIdx.x % cs, yy = blockIdx.x / cs;
    const int ts = psup[p], ko = (ts * 2 + 2) * h.os / 2;
    const int ks = 2 * ts + 1;
    const long long os = h.os, op = h.os / 2;
    const cplx<double>* khp = kh + size_t(p) * h.kh_stride;
    auto value = [&](int i, int j) -> cplx<double> {
        const long long cx = -(long long)ts * os + op - x + (long long)j * os;
        const long long cy = -(long long)ts * os + op - yy + (long long)i * os;
        const long long dcx = cx < 0 ? -cx : cx, dcy = cy < 0 ? -cy : cy;
        const long long vi = dcx > dcy ? dcy * ko - ((dcy * (dcy + 1)) >> 1) + dcx : dcx * ko - ((dcx * (dcx + 1)) >> 1) + dcy;
        return khp[vi];
    };
    double sum = 0.0;
    for (int e = threadIdx.x; e < ks * ks; e += 256) {
        const int i = e % ks, j = e / ks;
        sum += value(i, j).x;
    }
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off)
            red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    const double ksum = red[0];
    cplx<KT>* out = cache + (size_t(p) * cs * cs + blockIdx.x) * w_slot(2 * h.support + 1);
    for (int e = threadIdx.x; e < int(w_slot(ks)); e += 256) {
        const int i = (e - 1) % (ks + 1), j = (e - 1) / (ks + 1) - WPAD;
        if (e == 0 || i == ks || j < 0 || j >= ks) {
            out[e] = { KT(0), KT(0) };
            continue;
        }
        const cplx<double> v = value(i, j);
        out[e] = { KT(v.x / ksum), KT(v.y / ksum) };
    }
}

// Truncated support of each plane of a batch (aw_projection.cpp:176-179,197-209):
// the largest s <= support whose sample conv(s * os, 0) (position s of row 0) exceeds
// trunc_frac times |conv(0, 0)|.  A plane truncated to 0 (the reference asserts there,
// gridder.h:584) keeps support 1.
__global__ void wk_trunc_kernel(const cplx<double>* conv, size_t stride, int support, double trunc_frac, int nb,
    int* plane_support)
{
    const int b = blockIdx.x * 64 + threadIdx.x;
    if (b >= nb)
        return;
    const cplx<double>* c = conv + size_t(b) * stride;
    const double min_value = hypot(c[0].x, c[0].y) * trunc_frac;
    int s = support;
    while (s > 0 && !(hypot(c[s].x, c[s].y) > min_value))
        s--;
    plane_support[b] = max(1, s);
}

// generate_kernel_cache, non-Hankel branch (aw_projection.cpp:415-443): kernel (x, y) of the
// oversampled offsets 0 .. os / 2 (the others are these, mirrored), element (row i, column
// j) = conv at frequencies |(j - s) os + os / 2 - x| and |(i - s) os + os / 2 - y|,
// normalised by the sum of its real parts.  One block per (x, y); blockIdx.y: array
// blockIdx.y of conv (wk_cosine_kernel's positions, npos a side), written to plane
// blockIdx.y of cache.  A truncated plane's kernels (plane_support non-NULL) have its own
// support s.
template <typename KT>
__global__ __launch_bounds__(256) void wk_extract_kernel(const cplx<double>* conv, int npos, int len, int os, int support,
    const int* plane_support, cplx<KT>* cache)
{
    __shared__ double red[4];
    conv += size_t(blockIdx.y) * npos * npos;
    const int op = os / 2, cs = op + 1;
    const int x = blockIdx.x % cs, y = blockIdx.x / cs;
    const int s = plane_support ? plane_support[blockIdx.y] : support;
    const int ks = 2 * s + 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // position of sample d os + o, d = -s .. s, o = 0 .. os / 2
    auto at = [&](int d, int o) { return d >= 0 ? o * len + d : (o ? (os - o) * len - d - 1 : -d); };
    double sum = 0.0;
    for (int j = wave; j < ks; j += 4) {
        const cplx<double>* c = conv + size_t(at(j - s, op - x)) * npos;
        for (int i = lane; i < ks; i += 64)
            sum += c[at(i - s, op - y)].x;
    }
    for (int off = 32; off > 0; off >>= 1)
        sum += __shfl_down(sum, off, 64);
    if (lane == 0)
        red[wave] = sum;
    __syncthreads();
    const double inv = 1.0 / ((red[0] + red[1]) + (red[2] + red[3]));
    cplx<KT>* out = cache + (size_t(blockIdx.y) * cs * cs + blockIdx.x) * w_slot(2 * support + 1);
    if (threadIdx.x == 0)
        out[0] = { KT(0), KT(0) };
    for (int jc = wave; jc < ks + 2 * WPAD; jc += 4) {
        const int j = jc - WPAD;
        const bool in = j >= 0 && j < ks;
        const cplx<double>* c = conv + size_t(in ? at(j - s, op - x) : 0) * npos;
        for (int i = lane; i <= ks; i += 64) {
            cplx<KT> v{ KT(0), KT(0) };
            if (in && i < ks) {
                const cplx<double> k = c[at(i - s, op - y)];
                v = { KT(k.x * inv), KT(k.y * inv) };
            }
            out[1 + size_t(jc) * (ks + 1) + i] = v;
        }
    }
}

// W-projection tile sums without atomics.  A wave sums 64 rows x W_COLS columns of a
// tile: its FP64 sums stay in registers and each cell is written once.  Every lane loads
// 16 bytes of kernel at a time (two rows of FP32 values, one of FP64), and the lanes of
// each 16 rows take entries of their own from a queue of those that touch them, so a
// footprint of ks rows wastes at most 15 rows at either end (one entry across all 64 rows
// used half of the lanes at 65 taps).  Per tap (gridder.h:826-861): kval = K w with K the
// plane's complex kernel, conjugated for w < 0, grid += vis kval, beam += kval, as six
// FP64 FMAs with the entry's coefficients.
//
// The waves walk the tile's entries 64 at a time, each by itself, and keep those that
// touch their cells in LDS, so there is no barrier.  Kernels of mirrored oversampled
// offsets are stored once and read backwards (the plane's kernel is even): 1.0 MB per FP32
// plane at 65 taps and oversampling 8.
//
// Phases: the entries are in |w| order, and workgroups that start together read the
// kernels of about the same planes, from L2.  Later ones start over at plane 0 while the
// others are further on, so a launch covers a run of binning blocks (a phase) of about
// W_PHASE_BYTES of kernels and continues the FP64 sums of the launch before: with 32
// planes (33 MB of FP32 kernels) one launch read 66 GB past L2.
//
// Measured with N = 4096, 2 M visibilities, 32 planes, 65 taps, FP32: 7.2 ms (12.0 with a
// lane per row of 64 and 81 kernels per plane), of which 4.3 are vector instructions and
// as much the 1.2 G cache lines of the kernel reads; with all kernels in L2 it takes 6.8.
// Truncated kernels (N = 2048, 300 k visibilities of a condensed array, FP64): 0.2 ms against 25,
// from footprints of each plane's own support and from splitting the heavy tiles.
constexpr int W_COLS = 8;
constexpr int W_WAVES = 4;               // waves per workgroup (tiles of 16 columns: 2)
constexpr int W_KEEP = 128;              // kept entries of a wave: summed above 64
constexpr uint32_t W_OOB = 0xc0000000u;  // buffer offset past every kernel
constexpr size_t W_BUFFER_MAX = size_t(1) << 31; // largest kernel cache of the 32-bit buffer offsets
constexpr double W_PHASE_BYTES = 4.5 * (1 << 20); // 32 planes, 65 taps, FP32: 9.7 ms in one launch, 7.6 at 9 MB, 7.2 at 4.5 MB
constexpr double W_PHASE_READS = 4e9;    // least kernel bytes read per phase: below, its own 50-100 us cost more
// With truncated kernels the host counts the reads of the whole ones, and the device takes
// one phase where the planes' own come to less than two phases' worth (WPhase::one); the
// other phases then cost 5 us each for nothing.  N = 4096, 2 M visibilities, 32 planes, FP64,
// truncated at 0.01 % (whole supports remain): 22.2 ms in one phase, 11.6 in eight; at 1 % 1.65
// and 1.68 ms.  Below 32 GB of reads one phase loses less than 1.5 ms.
constexpr double W_TRUNC_PHASE_READS = 16e9;
constexpr int BUF_DWORD3 = 0x00020000;   // raw (untyped) buffer access
static_assert(W_COLS - 1 <= WPAD, "column runs must stay within the zero padding");

struct WPhase {
    const uint32_t* bcur = nullptr; // bcur[b * ntiles + t]: entries of tile t in blocks < b (null: one phase)
    const uint32_t* btot = nullptr; // entries of tile t
    int b0 = 0, b1 = 0, nblk = 0;
    int first = 1, last = 1;        // first: sums start at zero; last: write the grids
    const uint32_t* one = nullptr;  // not 0: the first phase takes all blocks after all (null: no)
    cplx<double>* acc_v = nullptr;  // FP64 running sums between phases (rows x N, grid layout)
    cplx<double>* acc_b = nullptr;
};

struct alignas(16) WKept {
    double a, b, w;      // (vis w) re, im and w
    uint32_t first;      // byte offset of the kernel row of the wave's first row in the run's first column
    int step;            // bytes to the next column (negative: columns mirrored)
    int row;             // kernel row of the wave's first row
    int ks;              // taps per side, negative for the conjugate kernel
    int sub, pad;        // sub-kernel (BIG)
};
struct WaveKeep {
    WKept e[W_KEEP + 1];             // the last one: no taps
    uint8_t queue[2][4][W_KEEP];     // per row direction and 16 rows: positions in e
};

// 16 bytes of kernel values at an offset of the cache (zero past its end).
template <typename KT>
struct KRow {
    cplx<KT> v[16 / sizeof(cplx<KT>)];
};
template <typename KT>
__device__ __forceinline__ KRow<KT> load_krow(__amdgpu_buffer_rsrc_t rs, uint32_t voff)
{
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    const u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, 0, 0);
    if constexpr (std::is_same<KT, double>::value)
        return { { { __longlong_as_double((long long)((unsigned long long)v.y << 32 | v.x)),
            __longlong_as_double((long long)((unsigned long long)v.w << 32 | v.z)) } } };
    else
        return { { { __uint_as_float(v.x), __uint_as_float(v.y) }, { __uint_as_float(v.z), __uint_as_float(v.w) } } };
}

// -x where `sign` is negative
__device__ __forceinline__ double flip_if(double x, int sign)
{
    return __longlong_as_double(__double_as_longlong(x) ^ ((unsigned long long)(uint32_t(sign) & 0x80000000u) << 32));
}

// BIG: kernel caches past the reach of a buffer's 32-bit offsets, by 64-bit addresses
// (rows outside the kernel read its zero padding).
template <typename T, typename KT, bool BEAM, bool BIG>
__global__ __launch_bounds__(64 * W_WAVES) void grid_wtiles_kernel(GridGeom g, Entry* entries,
    const uint32_t* __restrict__ offsets, uint32_t cap, const cplx<KT>* __restrict__ cache, uint32_t cache_bytes,
    cplx<T>* __restrict__ vgrid, cplx<T>* __restrict__ bgrid, int ext_host, WPhase ph)
{
    constexpr int SZ = int(sizeof(cplx<KT>));
    constexpr int RPL = 16 / SZ, CPL = W_COLS / RPL; // rows and columns of a lane
    constexpr int LS = 16 / RPL;                     // lanes per 16 rows
    __shared__ WaveKeep keeps[W_WAVES];
    const int N = g.N, waves = int(blockDim.x) / 64, strips = g.tc / (W_COLS * waves);
    const int ntiles = g.tiles_r * g.tiles_c;
    const Split sp = split_view(entries, cap, offsets[ntiles], ext_host, g.tc, 4);
    uint32_t chunk = 0;
    const int unit = int(blockIdx.x) / strips;
    int t = unit - ext_host;
    if (ph.one && *ph.one) {
        if (!ph.first)
            return;
        ph.b1 = ph.nblk;
        ph.last = 1;
    }
    if (t < 0) {
        if (!sp.hdr || uint32_t(unit) >= sp.hdr[0])
            return;
        t = int(sp.ext[2 * unit]);
        chunk = sp.ext[2 * unit + 1];
    }
    const uint32_t tb = min(offsets[t], cap), te = min(offsets[t + 1], cap);
    const uint32_t ch = sp.hdr ? sp.hdr[2] : 0xffffffffu;
    const bool split = te - tb > ch;
    uint32_t eb = tb, ee = te;
    bool fresh = ph.first; // sums start at zero
    if (split) {
        eb = tb + chunk * ch;
        ee = min(te, eb + ch);
    }
    if (ph.bcur) {
        const uint32_t p0 = tb + (ph.b0 < ph.nblk ? ph.bcur[size_t(ph.b0) * ntiles + t] : ph.btot[t]);
        const uint32_t p1 = tb + (ph.b1 < ph.nblk ? ph.bcur[size_t(ph.b1) * ntiles + t] : ph.btot[t]);
        if (split)
            fresh = eb >= p0;
        eb = max(eb, min(p0, te));
        ee = min(ee, min(p1, te));
    }
    // FP32 grids take the sums at the last phase; FP64 grids are their own running sums
    constexpr bool narrow = !std::is_same<T, double>::value;
    if (eb >= ee && (split || !(ph.first || (narrow && ph.last))))
        return; // no entry in the phase: the sums stay as they are
    const int rt = t % g.tiles_r, ct = t / g.tiles_r;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int kk = (lane / LS) & 3;                      // the lane's 16 rows
    const int lr = 16 * kk + RPL * (lane % LS);          // its first row
    const int lh = CPL * (lane / (4 * LS));              // its first column among the wave's
    const int lw = W_COLS * (int(blockIdx.x) % strips * waves + wave);
    const int rb = rt * TILE_R, cb = ct * g.tc + lw;     // the wave's cells
    const uint32_t slot = uint32_t(w_slot(g.ks));
    WaveKeep& keep = keeps[wave];
    // the running sums of cell (row lr + v, column lh + u): grid or slot elements
    double* slot_out = nullptr;
    if (split) {
        uint32_t lo = 0, hi = sp.hdr[1] - 1; // the tile's record among the split tiles
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if (sp.spl[3 * mid] < uint32_t(t))
                lo = mid + 1;
            else
                hi = mid;
        }
        slot_out = sp.part + size_t(sp.spl[3 * lo + 1] + chunk) * (4 * g.tc * TILE_R) + (lw + lh) * TILE_R + lr;
    }
    const int plane = g.tc * TILE_R;
    double ar[8], ai[8], br[8], bi[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int v = k % RPL, u = k / RPL;
        ar[k] = ai[k] = br[k] = bi[k] = 0.0;
        if (fresh)
            continue;
        if (split) {
            const double* o = slot_out + u * TILE_R + v;
            ar[k] = o[0];
            ai[k] = o[plane];
            if (BEAM) {
                br[k] = o[2 * plane];
                bi[k] = o[3 * plane];
            }
        } else if (rb + lr + v < g.rows && cb + lh + u < N) {
            const size_t o = size_t(rb + lr + v) + size_t(cb + lh + u) * g.rows;
            ar[k] = ph.acc_v[o].x;
            ai[k] = ph.acc_v[o].y;
            if (BEAM) {
                br[k] = ph.acc_b[o].x;
                bi[k] = ph.acc_b[o].y;
            }
        }
    }
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)cache, (short)0, cache_bytes, BUF_DWORD3);

    int cnt[2][4] = {}, kept = 0;
    // one queue of each 16 rows, up to the longest one's length; MIRROR: the kernel's rows
    // run backwards, and so do the rows of a load
    auto sum_queues = [&](auto MIRROR) {
        constexpr bool MR = decltype(MIRROR)::value;
        const int* c = cnt[MR];
        const int n = max(max(c[0], c[1]), max(c[2], c[3]));
        const int mine = kk == 0 ? c[0] : (kk == 1 ? c[1] : (kk == 2 ? c[2] : c[3]));
        const uint8_t* queue = keep.queue[MR][kk];
        int nx = 0 < mine ? queue[0] : W_KEEP;
        for (int q = 0; q < n; q++) {
            const WKept e = keep.e[nx];
            nx = q + 1 < mine ? queue[q + 1] : W_KEEP;
            const int ks = e.ks < 0 ? -e.ks : e.ks;
            // rows -1 and ks are zeros of the padding
            const bool row = unsigned(e.row + lr + RPL - 1) < unsigned(ks + RPL - 1);
            const int off = (MR ? -lr - (RPL - 1) : lr) * SZ + lh * e.step;
            KRow<KT> kv[CPL];
            if constexpr (BIG) {
                const char* p = reinterpret_cast<const char*>(cache + size_t(e.sub) * slot);
#pragma unroll
                for (int u = 0; u < CPL; u++)
                    kv[u] = row ? *reinterpret_cast<const KRow<KT>*>(p + (int(e.first) + off + u * e.step)) : KRow<KT>{};
            } else {
                uint32_t v = row ? e.first + uint32_t(off) : W_OOB;
#pragma unroll
                for (int u = 0; u < CPL; u++) {
                    kv[u] = load_krow<KT>(rs, v);
                    v += uint32_t(e.step);
                }
            }
            const double a = e.a, b = e.b, w = e.w;
            const double sa = flip_if(a, e.ks), sb = flip_if(b, e.ks), sw = flip_if(w, e.ks);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const cplx<KT> K = kv[k / RPL].v[MR ? RPL - 1 - k % RPL : k % RPL];
                const double kr = double(K.x), ki = double(K.y);
                ar[k] = fma(a, kr, ar[k]);
                ar[k] = fma(-sb, ki, ar[k]);
                ai[k] = fma(b, kr, ai[k]);
                ai[k] = fma(sa, ki, ai[k]);
                if (BEAM) {
                    br[k] = fma(w, kr, br[k]);
                    bi[k] = fma(sw, ki, bi[k]);
                }
            }
        }
    };
    auto sum_kept = [&]() {
        // the wave's LDS accesses complete in order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        sum_queues(std::integral_constant<bool, false>{});
        sum_queues(std::integral_constant<bool, true>{});
        kept = 0;
#pragma unroll
        for (int k = 0; k < 4; k++)
            cnt[0][k] = cnt[1][k] = 0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };

    if (eb < ee) {
        if (lane == 0) {
            WKept none{};
            none.row = -(1 << 20);
            none.ks = 1;
            keep.e[W_KEEP] = none;
        }
        int ngx, ngy, ncp, nidx;
        double nvr, nvi, nw;
        auto fetch = [&](uint32_t e) {
            const Entry* p = entries + min(e + uint32_t(lane), ee - 1);
            ngx = p->gx;
            ngy = p->gy;
            ncp = p->cp;
            nidx = p->idx;
            nvr = p->vr;
            nvi = p->vi;
            nw = p->w;
        };
        fetch(eb);
        const unsigned long long below = (1ull << lane) - 1ull;
        for (uint32_t e0 = eb; e0 < ee; e0 += 64) {
            const int gx = ngx, gy = ngy, cp = ncp, idx = nidx;
            const double a = nvr, b = nvi, w = nw;
            const bool valid = e0 + uint32_t(lane) < ee;
            fetch(e0 + 64);
            const int s = cp & 127, ks = 2 * s + 1;
            // the footprint and its wrapped pieces: the cells' rows at +N (rows past N wrap,
            // rows below 0 are dropped), their columns at +-N
            const int iraw = rb - (gy - s), jraw = cb - (gx - s);
            const bool wrapped = valid && (gy + s >= N || gx - s < 0 || gx + s >= N);
            const int pieces = __ballot(wrapped) ? 6 : 1;
            for (int p = 0; p < pieces; p++) {
                const int pr = p & 1, pc = p >> 1;
                const int i0 = iraw + (pr ? N : 0), j0 = jraw + (pc == 0 ? 0 : (pc == 1 ? N : -N));
                const bool hit = valid && i0 < ks && i0 > -64 && j0 < ks && j0 > -W_COLS;
                const unsigned long long mask = __ballot(hit);
                if (!mask)
                    continue;
                const int pos = kept + __popcll(mask & below);
                const bool mr = (cp >> 30) & 1, mc = (cp >> 29) & 1;
                if (hit) {
                    const int jp = (mc ? 2 * s - j0 : j0) + WPAD; // padded column of the run's start
                    WKept e;
                    e.a = a;
                    e.b = b;
                    e.w = w;
                    e.first = (BIG ? 0u : uint32_t(idx) * slot * SZ) + uint32_t((1 + jp * (ks + 1) + (mr ? 2 * s - i0 : i0)) * SZ);
                    e.step = (mc ? -(ks + 1) : ks + 1) * SZ;
                    e.row = i0;
                    e.ks = cp < 0 ? -ks : ks;
                    e.sub = idx;
                    e.pad = 0;
                    keep.e[pos] = e;
                }
                kept += __popcll(mask);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const bool in = hit && i0 + 16 * k < ks && i0 + 16 * k > -16;
                    const unsigned long long m0 = __ballot(in && !mr), m1 = __ballot(in && mr);
                    if (in)
                        keep.queue[mr][k][mr ? cnt[1][k] + __popcll(m1 & below) : cnt[0][k] + __popcll(m0 & below)] = uint8_t(pos);
                    cnt[0][k] += __popcll(m0);
                    cnt[1][k] += __popcll(m1);
                }
                if (kept > W_KEEP - 64)
                    sum_kept();
            }
        }
        if (kept)
            sum_kept();
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int v = k % RPL, u = k / RPL;
        const int r = rb + lr + v, c = cb + lh + u;
        if (split) {
            double* o = slot_out + u * TILE_R + v;
            o[0] = ar[k];
            o[plane] = ai[k];
            if (BEAM) {
                o[2 * plane] = br[k];
                o[3 * plane] = bi[k];
            }
        } else if (r < g.rows && c < N) {
            const size_t o = size_t(r) + size_t(c) * g.rows;
            if (narrow && !ph.last) {
                ph.acc_v[o] = { ar[k], ai[k] };
                if (BEAM)
                    ph.acc_b[o] = { br[k], bi[k] };
            } else {
                vgrid[o] = { T(ar[k]), T(ai[k]) };
                if (BEAM)
                    bgrid[o] = { T(br[k]), T(bi[k]) };
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Fused batches: the snapshots of a batch are gridded by one launch per stage.
// Each stage's workgroups are numbered across the snapshots; pre[k] is the first
// workgroup of snapshot k (pre[0] = 0, non-decreasing, snapshots without work
// in a stage repeat the next start) and a workgroup finds its snapshot by a
// binary search over pre (uniform, so scalar loads).
struct BItem {
    GridGeom g;
    const double* uv;
    const double* vis;
    const double* wts;
    const double* ktab;        // oversampled 1-D kernel table
    uint32_t* counts;          // nblk x ntiles block counts, then block cursors
    uint32_t* totals;          // entries per tile
    uint32_t* toffs;           // tile entry offsets (ntiles + 1)
    Entry* entries;
    double* wpart;             // canonical weight / good-count pairs, one per block
    void* vgrid;
    void* bgrid;
    double* total;
    unsigned long long* ngood;
    uint32_t cap;
    int nblk;
    int ext_host;              // extra chunk workgroups of split tiles
};

__device__ __forceinline__ int batch_item(const uint32_t* __restrict__ pre, int K, uint32_t b)
{
    int lo = 0, hi = K - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(BWG) void batch_count_kernel(const BItem* __restrict__ items, const uint32_t* __restrict__ pre,
    int K)
{
    const int k = batch_item(pre, K, blockIdx.x);
    const BItem& it = items[k];
    bin_count_body(it.g, it.uv, it.vis, it.wts, it.counts, it.wpart, int(blockIdx.x - pre[k]));
}

__global__ __launch_bounds__(1024) void batch_colscan_kernel(const BItem* __restrict__ items, const uint32_t* __restrict__ pre,
    int K)
{
    const int k = batch_item(pre, K, blockIdx.x);
    const BItem& it = items[k];
    colscan_body(it.counts, it.nblk, it.g.tiles_r * it.g.tiles_c, it.totals, int(blockIdx.x - pre[k]));
}

__global__ __launch_bounds__(BWG) void batch_scatter_kernel(const BItem* __restrict__ items, const uint32_t* __restrict__ pre,
    int K)
{
    const int k = batch_item(pre, K, blockIdx.x);
    const BItem& it = items[k];
    bin_scatter_body(it.g, it.uv, it.vis, it.wts, it.totals, it.counts, it.entries, it.cap, it.toffs, it.ext_host,
        int(blockIdx.x - pre[k]));
}

template <typename Acc, int KSM>
__global__ __launch_bounds__(TWG) void batch_tiles_twofloat_kernel(const BItem* __restrict__ items,
    const uint32_t* __restrict__ pre, int K)
{
    const int k = batch_item(pre, K, blockIdx.x);
    const BItem& it = items[k];
    tiles_os_body<float, Acc, KSM>(it.g, it.entries, it.toffs, 1, it.cap, it.ktab, (cplx<float>*)it.vgrid,
        (cplx<float>*)it.bgrid, int(blockIdx.x - pre[k]));
}

template <typename T, int TC, int FORM>
__global__ __launch_bounds__(tile_threads(TC), tile_waves(FORM)) void batch_tiles_kernel(const BItem* __restrict__ items, const uint32_t* __restrict__ pre,
    int K)
{
    const int k = batch_item(pre, K, blockIdx.x);
    const BItem& it = items[k];
    tiles_mfma_body<T, TC, FORM>(it.g, it.entries, it.toffs, it.cap, it.ktab, it.uv, (cplx<T>*)it.vgrid,
        (cplx<T>*)it.bgrid, it.ext_host, int(blockIdx.x - pre[k]));
}

// Workgroups 0 .. K-1: the last canonical level of a snapshot's weight pairs (at most
// CANON_BLOCK blocks), sample_grid_total and the good count; the others: the merges of
// split tiles.
template <typename T>
__global__ __launch_bounds__(CANON_LANES) void batch_total_kernel(const BItem* __restrict__ items,
    const uint32_t* __restrict__ pre, int K)
{
    __shared__ double lds[2 * CANON_LANES];
    if (blockIdx.x < unsigned(K)) {
        const BItem& it = items[blockIdx.x];
        double a, b;
        canon_last_level(it.wpart, unsigned(it.nblk), a, b, lds);
        if (threadIdx.x == 0) {
            it.total[0] = a * 2.0;
            if (it.ngood)
                *it.ngood = (unsigned long long)b;
        }
        return;
    }
    const uint32_t q = blockIdx.x - unsigned(K);
    const int k = batch_item(pre, K, q);
    const BItem& it = items[k];
    merge_body<T>(it.g, it.entries, it.cap, it.toffs[it.g.tiles_r * it.g.tiles_c], it.ext_host, (cplx<T>*)it.vgrid,
        (cplx<T>*)it.bgrid, int(q - pre[k]), lds);
}

} // namespace

// Grid geometry of one call (validated); the kernel functor in kf.
static GridGeom make_geom(const GridderArgs& a, size_t n, bool beam, KernelFn& kf)
{
    const int N = a.image_size;
    const bool wproj = a.wproj.num_wplanes > 0;
    // W-projection grids with max_wpconv_support (gridder.h:260-268)
    const int support = wproj ? int(a.wproj.max_wpconv_support) : a.support;
    STP_REQUIRE(N >= 4 && (N % 2) == 0, "image_size must be even and >= 4");
    STP_REQUIRE(support >= 1 && support <= 127, "kernel support must be in [1, 127]");
    STP_REQUIRE(2 * support + 1 <= N, "kernel wider than the grid");
    STP_REQUIRE(n < (size_t(1) << 30), "at most 2^30 visibilities per call");
    if (wproj) {
        STP_REQUIRE(!a.kernel_exact, "W-projection requires kernel_exact == false");
        STP_REQUIRE(a.wproj.num_wplanes <= 65535, "at most 65535 w-planes");
        STP_REQUIRE(n < (size_t(1) << 31), "too many visibilities for W-projection");
    }
    int os = a.oversampling;
    if (a.kernel_exact) {
        os = 1;
    } else {
        os = (os >> 1) << 1; // gridder.h:297-303
        if (os == 0)
            os = 1;
    }
    STP_REQUIRE(os <= 1024, "oversampling must be <= 1024");
    GridGeom g;
    g.N = N;
    g.half = N / 2;
    g.rows = a.halfplane ? g.half + 1 : N;
    g.s = support;
    g.ks = 2 * support + 1;
    g.os = os;
    g.halfplane = a.halfplane;
    g.shift = a.shift_uv;
    g.exact = a.kernel_exact;
    g.beam = beam;
    g.bpack = beam && a.beam_packed ? 1 : 0;
    STP_REQUIRE(!g.bpack || (!wproj && a.halfplane), "a packed real beam grid needs the half-plane grid without W-projection");
    g.tiles_r = int(div_up(g.rows, TILE_R));
    g.tc = a.tile_cols > 0 ? a.tile_cols : (wproj ? W_TILE_C : TILE_C);
    STP_REQUIRE(g.tc == 16 || g.tc == 32 || g.tc == 64, "tile width must be 16, 32 or 64 columns");
    g.tiles_c = int(div_up(N, g.tc));
    g.scale = a.uv_scale;
    g.n = (long long)n;
    kf = kernel_fn(a.kernel);
    g.kfunc = kf.kind;
    g.kparam = kf.param;
    g.kwg = kf.width_g;
    g.kws = kf.width_s;
    return g;
}

template <typename T, int FORM>
static auto tiles_kernel_of(int tc)
{
    return tc == 16 ? grid_tiles_kernel<T, 16, FORM> : (tc == 32 ? grid_tiles_kernel<T, 32, FORM> : grid_tiles_kernel<T, 64, FORM>);
}

// The two-float tile sums of one call (ostride: stride of the tile offsets).
static void twofloat_tiles(stp_ctx* ctx, const GridGeom& g, int cs, const Entry* entries, const uint32_t* offsets, int ostride,
    uint32_t cap, const double* d_tab, const double* d_uv, cplx<float>* vgrid, cplx<float>* bgrid)
{
    const int ntiles = g.tiles_r * g.tiles_c;
    const int S = TILE_R + (g.ks <= 15 ? g.ks : 1);
    const size_t acc_bytes = ((6 * size_t(g.tc) * S * sizeof(float) + 7) / 8) * 8;
    if (!g.exact && g.ks <= 16) {
        // oversampled kernels up to 16 taps: the specialised tile kernel
        const size_t bytes = acc_bytes + sizeof(double) * size_t(cs) * g.ks;
        auto kern = g.ks <= 8 ? grid_tiles_os_kernel<float, AccTwoFloat, 8> : grid_tiles_os_kernel<float, AccTwoFloat, 16>;
        HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
        launch(ctx, "grid_tiles", kern, dim3(unsigned(ntiles)), dim3(TWG), bytes, g, entries, offsets, ostride, cap, d_tab, vgrid,
            bgrid);
    } else {
        const size_t bytes = acc_bytes + (g.exact ? sizeof(double) * (KV_DOUBLES + TEB) : sizeof(double) * size_t(cs) * g.ks);
        auto kern = grid_tiles_twofloat_kernel<float, AccTwoFloat>;
        HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
        launch(ctx, "grid_tiles", kern, dim3(unsigned(ntiles)), dim3(TWG), bytes, g, entries, offsets, ostride, cap, d_tab, d_uv,
            vgrid, bgrid);
    }
}

template <typename T>
void grid_visibilities(stp_ctx* ctx, const GridderArgs& a, size_t n, const double* d_uv, const double* d_vis,
    const double* d_w, cplx<T>* d_vis_grid, cplx<T>* d_sampling_grid, double* d_total, unsigned long long* d_ngood, TileOcc* occ)
{
    const bool wproj = a.wproj.num_wplanes > 0;
    KernelFn kf;
    GridGeom g = make_geom(a, n, a.generate_beam && d_sampling_grid != nullptr, kf);
    const int N = g.N, os = g.os;
    const int ntiles = g.tiles_r * g.tiles_c;
    // kernel table (oversampled 1-D kernels), computed on the host once per configuration
    const double* d_tab = nullptr;
    const int cs = (os / 2) * 2 + 1;
    if (wproj) {
        d_tab = dev_table(ctx, "k1d:none", std::vector<double>(1, 0.0));
    } else if (!a.kernel_exact) {
        char key[160];
        snprintf(key, sizeof(key), "k1d:%d:%.17g:%.17g:%.17g:%d:%d", kf.kind, kf.param, kf.width_g, kf.width_s, a.support, os);
        d_tab = has_table(ctx, key) ? dev_table(ctx, key, {}) : dev_table(ctx, key, kernel_1d_table(kf, a.support, os));
    } else {
        d_tab = dev_table(ctx, "k1d:none", std::vector<double>(1, 0.0));
    }

    // FP64 tile sums (every path but two-float and W-projection) run on the matrix cores
    const bool twofloat = std::is_same<T, float>::value && a.twofloat;
    const bool mfma = !wproj && !twofloat;
    const size_t nblk = std::max<size_t>(1, (n + VPB - 1) / VPB);
    double* wpart = (double*)ws_get(ctx, "grid_wpart", sizeof(double) * (2 * nblk + 2));
    double* wscr = (double*)ws_get(ctx, "grid_wscr", sizeof(double) * canon_scratch_doubles(nblk));
    // worst-case entries: the most tiles one footprint can touch (every centre
    // checked on the host), times two passes
    const size_t cap64 = std::max<size_t>(1, 2 * footprint_tiles_max(g) * n);
    STP_REQUIRE(cap64 < (size_t(1) << 32), "too many gridding entries for one call");
    const uint32_t cap = uint32_t(cap64);
    Entry* entries = (Entry*)ws_get(ctx, "grid_entries", sizeof(Entry) * cap64);

    // W-kernel cache in the grid precision: FP64 kernels on the FP64 path, FP32
    // kernels (half the bytes the W tile kernel reads per tap) on the FP32 paths
    using KT = T;
    cplx<KT>* wcache = nullptr;
    size_t wcache_bytes = 0;
    if (wproj) {
        const int P = int(a.wproj.num_wplanes);
        // 1. |w| order
        unsigned long long* k0 = (unsigned long long*)ws_get(ctx, "w_key0", sizeof(unsigned long long) * n);
        unsigned long long* k1 = (unsigned long long*)ws_get(ctx, "w_key1", sizeof(unsigned long long) * n);
        uint32_t* i0 = (uint32_t*)ws_get(ctx, "w_idx0", sizeof(uint32_t) * n);
        uint32_t* i1 = (uint32_t*)ws_get(ctx, "w_idx1", sizeof(uint32_t) * n);
        // 4096 keys per block, 8192 where that still fills the chip: at 2 M keys counts, scan
        // and scatter take 62 + 66 + 310 us against 56 + 110 + 274 us
        const bool wide = n > (size_t(1) << 20);
        const size_t nrb = div_up(n, (wide ? 16 : 8) * RS_THREADS);
        uint32_t* rcounts = (uint32_t*)ws_get(ctx, "w_rcounts", sizeof(uint32_t) * RS_DIGITS * nrb);
        uint32_t* rtotals = (uint32_t*)ws_get(ctx, "w_rtotals", sizeof(uint32_t) * RS_DIGITS);
        auto hist = wide ? rs_hist_kernel<16> : rs_hist_kernel<8>;
        auto scatter = wide ? rs_scatter_kernel<16> : rs_scatter_kernel<8>;
        const double* wcol = d_uv + 2 * n;
        const bool self = nrb <= size_t(RS_SELF);
        for (int pass = 0; pass < RS_PASSES; pass++) {
            const unsigned long long* src = pass ? k0 : nullptr;
            launch(ctx, "w_sort_hist", hist, dim3(unsigned(nrb)), dim3(RS_THREADS), 0, src, wcol, (long long)n, RS_BITS * pass,
                rcounts);
            if (!self)
                launch(ctx, "w_sort_scan", bin_colscan_kernel, dim3(RS_DIGITS / 64), dim3(1024), 0, rcounts, int(nrb), RS_DIGITS,
                    rtotals);
            launch(ctx, "w_sort_scatter", scatter, dim3(unsigned(nrb)), dim3(RS_THREADS), 0, src, (const uint32_t*)i0, wcol,
                (long long)n, RS_BITS * pass, (const uint32_t*)rcounts, (const uint32_t*)(self ? nullptr : rtotals), int(nrb), k1,
                i1);
            std::swap(k0, k1);
            std::swap(i0, i1);
        }
        {
            double* uvw_s = (double*)ws_get(ctx, "w_uvw_sorted", sizeof(double) * 3 * n);
            double* vis_s = (double*)ws_get(ctx, "w_vis_sorted", sizeof(double) * 2 * n);
            double* wts_s = (double*)ws_get(ctx, "w_wts_sorted", sizeof(double) * n);
            launch(ctx, "w_permute", wpermute_kernel, dim3(unsigned(div_up(n, 256))), dim3(256), 0, d_uv, d_vis, d_w,
                (const uint32_t*)i0, (long long)n, uvw_s, vis_s, wts_s);
            d_uv = uvw_s;
            d_vis = vis_s;
            d_w = wts_s;
        }
        // 2. planes
        uint32_t* flag = (uint32_t*)ws_get(ctx, "w_flag", sizeof(uint32_t) * n);
        uint32_t* G = (uint32_t*)ws_get(ctx, "w_gscan", sizeof(uint32_t) * (n + 1));
        uint32_t* first = (uint32_t*)ws_get(ctx, "w_first", sizeof(uint32_t) * (P + 2));
        uint32_t* pcount = (uint32_t*)ws_get(ctx, "w_pcount", sizeof(uint32_t) * P);
        double* w_plane = (double*)ws_get(ctx, "w_plane", sizeof(double) * P);
        uint16_t* plane_of = (uint16_t*)ws_get(ctx, "w_planeof", sizeof(uint16_t) * n);
        launch(ctx, "w_good", wgood_kernel, dim3(unsigned(div_up(n, 256))), dim3(256), 0, g, d_uv, d_vis, d_w, flag);
        scan_u32(ctx, flag, n, G);
        launch(ctx, "w_planes", wplane_bounds_kernel, dim3(1), dim3(64), 0, (const uint32_t*)G, (long long)n, P,
            int(a.wproj.wplanes_median != 0), (const unsigned long long*)k0, first, pcount, w_plane);
        if (!a.wproj.wplanes_median) {
            double* wpart = (double*)ws_get(ctx, "w_plane_part", sizeof(double) * size_t(P) * WMS);
            launch(ctx, "w_plane_sum", wplane_sum_kernel, dim3(unsigned(P), unsigned(WMS)), dim3(256), 0,
                (const unsigned long long*)k0, (const uint32_t*)flag, (const uint32_t*)first, wpart);
            launch(ctx, "w_plane_mean", wplane_mean_kernel, dim3(unsigned(div_up(P, 256))), dim3(256), 0,
                (const double*)wpart, (const uint32_t*)pcount, P, w_plane);
        }
        launch(ctx, "w_plane_ids", wplane_ids_kernel, dim3(unsigned(div_up(n, 256))), dim3(256), 0, (const uint32_t*)first, P,
            (long long)n, plane_of);
        g.plane = plane_of;
        g.wproj = 1;
        // 3. W-kernels: workarea (gridder.h:467-486), image-domain AA kernel, cosine sums per plane
        const int us = a.wproj.undersampling_opt > 0 ? (1 << (a.wproj.undersampling_opt - 1)) : 0;
        int workarea = 2;
        if (us > 0)
            while (workarea / us < g.ks)
                workarea *= 2;
        else
            while (workarea < N)
                workarea *= 2;
        const int arr = workarea * os;
        STP_REQUIRE(arr <= 4096, "W-kernel work array (workarea * oversampling) must be <= 4096");
        const double scaling = double(N) / double(workarea);
        char key[192];
        snprintf(key, sizeof(key), "waa:%d:%.17g:%.17g:%.17g:%d:%d", kf.kind, kf.param, kf.width_g, kf.width_s, workarea,
            a.analytic_gcf ? 1 : 0);
        const double* d_aa = has_table(ctx, key) ? dev_table(ctx, key, {})
                                                 : dev_table(ctx, key, img_dom_kernel(kf, size_t(workarea), false, a.analytic_gcf));
        const int csw = os / 2 + 1; // offsets per axis without their mirror images
        const size_t per_plane = size_t(csw) * csw * w_slot(g.ks);
        wcache_bytes = sizeof(cplx<KT>) * per_plane * P;
        STP_REQUIRE(size_t(P) * cs * cs < (size_t(1) << 31), "too many W sub-kernels (planes x oversampling^2)");
        wcache = (cplx<KT>*)ws_get(ctx, "w_cache", sizeof(cplx<KT>) * per_plane * P);
        // kernel_trunc_perc > 0: every plane grids with its own truncated support
        const bool trunc = a.wproj.kernel_trunc_perc > 0.0;
        if (a.wproj.hankel_opt) {
            // Hankel W-kernels: profile, DHT or DFT, spline, half quadrant, cuts
            HankelArgs h;
            h.proj_slice = a.wproj.hankel_proj_slice != 0;
            h.cubic = a.wproj.interp_type == 2;
            h.n = h.proj_slice ? arr : arr / 2;
            h.half = workarea / 2;
            h.arr = arr;
            h.os = os;
            h.support = g.s;
            h.scaled_cell = a.cell_rad * scaling;
            h.trunc_frac = trunc ? a.wproj.kernel_trunc_perc / 100.0 : 0.0;
            const long long ko_max = (long long)(g.s + 1) * os;
            h.kh_stride = int(ko_max * (ko_max + 1) / 2);
            STP_REQUIRE(h.n >= 3, "Hankel W-kernels need a transform of at least 3 points");
            STP_REQUIRE(h.n <= 8192, "Hankel W-kernel transform longer than 8192 points (workarea * oversampling)");
            const double* tab;
            char tkey[64];
            if (!h.proj_slice) {
                snprintf(tkey, sizeof(tkey), "dht:%d", h.n);
                tab = has_table(ctx, tkey) ? dev_table(ctx, tkey, {}) : dev_table(ctx, tkey, dht_table(size_t(h.n)));
            } else {
                snprintf(tkey, sizeof(tkey), "dft:%d", h.n);
                tab = has_table(ctx, tkey) ? dev_table(ctx, tkey, {}) : dev_table(ctx, tkey, dft_twiddles(size_t(h.n)));
            }
            cplx<double>* prof = (cplx<double>*)ws_get(ctx, "w_hk_prof", sizeof(cplx<double>) * size_t(h.n) * P);
            cplx<double>* yv = (cplx<double>*)ws_get(ctx, "w_hk_y", sizeof(cplx<double>) * size_t(h.n) * P);
            double* coef = (double*)ws_get(ctx, "w_hk_coef", sizeof(double) * 10 * size_t(h.n) * P);
            cplx<double>* kh = (cplx<double>*)ws_get(ctx, "w_hk_quad", sizeof(cplx<double>) * size_t(h.kh_stride) * P);
            int* psup = (int*)ws_get(ctx, "w_psupport", sizeof(int) * P);
            launch(ctx, "w_hankel_profile", wk_hankel_profile_kernel, dim3(unsigned(P)), dim3(256), 0, h, d_aa,
                (const double*)w_plane, prof);
            g.psup = psup;
            launch(ctx, "w_hankel_transform", wk_hankel_transform_kernel, dim3(unsigned(div_up(h.n, 256)), unsigned(P)),
                dim3(256), 0, h, tab, (const cplx<double>*)prof, yv);
            launch(ctx, "w_hankel_spline", wk_hankel_spline_kernel, dim3(unsigned(P)), dim3(64), 0, h, (const cplx<double>*)yv,
                coef, psup);
            launch(ctx, "w_hankel_quad", wk_hankel_quad_kernel,
                dim3(unsigned(std::min<long long>(1024, div_up((long long)h.kh_stride, 256))), unsigned(P)), dim3(256), 0, h,
                (const cplx<double>*)yv, (const double*)coef, (const int*)psup, kh);
            launch(ctx, "w_kernel_extract", wk_hankel_extract_kernel<KT>, dim3(unsigned(csw * csw), unsigned(P)), dim3(256), 0,
                h, (const cplx<double>*)kh, (const int*)psup, 0, wcache);
        } else {
            STP_REQUIRE(arr >= 4 && (arr & (arr - 1)) == 0, "W-kernel work array (workarea * oversampling) must be a power of two >= 4");
            const int half = workarea / 2, len = g.s + 1, npos = os * len;
            const size_t q2 = size_t(half) * half, t2 = size_t(half) * npos, c2 = size_t(npos) * npos;
            const int PB = int(w_group_planes(size_t(P), size_t(half), size_t(npos)));
            // planes in groups of PB, each stage one launch per group
            cplx<double>* quad = (cplx<double>*)ws_get(ctx, "w_quad", sizeof(cplx<double>) * q2 * PB);
            cplx<double>* axis = (cplx<double>*)ws_get(ctx, "w_axis", sizeof(cplx<double>) * t2 * PB);
            cplx<double>* conv = (cplx<double>*)ws_get(ctx, "w_conv", sizeof(cplx<double>) * c2 * PB);
            const cplx<double>* tw = (const cplx<double>*)twiddles_for(ctx, arr).d;
            int* psup = trunc ? (int*)ws_get(ctx, "w_psupport", sizeof(int) * P) : nullptr;
            g.psup = psup;
            for (int p0 = 0; p0 < P; p0 += PB) {
                const int nb = std::min(PB, P - p0);
                launch(ctx, "w_kernel_fill", wk_fill_kernel, dim3(unsigned(div_up(q2, 256)), unsigned(nb)), dim3(256), 0, quad,
                    half, d_aa, (const double*)w_plane, p0, a.cell_rad * scaling);
                launch(ctx, "w_kernel_axis", wk_cosine_kernel, dim3(div_up(npos, 64), div_up(half, 16), unsigned(nb)), dim3(256), 0,
                    (const cplx<double>*)quad, q2, half, half, half, axis, t2, npos, len, os, tw, arr);
                launch(ctx, "w_kernel_axis", wk_cosine_kernel, dim3(div_up(npos, 64), div_up(npos, 16), unsigned(nb)), dim3(256), 0,
                    (const cplx<double>*)axis, t2, npos, npos, half, conv, c2, npos, len, os, tw, arr);
                if (trunc)
                    launch(ctx, "w_kernel_trunc", wk_trunc_kernel, dim3(div_up(nb, 64)), dim3(64), 0, (const cplx<double>*)conv, c2,
                        g.s, a.wproj.kernel_trunc_perc / 100.0, nb, psup + p0);
                launch(ctx, "w_kernel_extract", wk_extract_kernel<KT>, dim3(unsigned(csw * csw), unsigned(nb)), dim3(256), 0,
                    (const cplx<double>*)conv, npos, len, os, g.s, (const int*)(trunc ? psup + p0 : nullptr),
                    wcache + size_t(p0) * per_plane);
            }
        }
    }

    int nph = 1; // W-projection: phases of the tile sums
    if (wproj && ntiles <= MAX_LDS_TILES) {
        const bool trunc = a.wproj.kernel_trunc_perc > 0.0;
        const double tap_bytes = sizeof(cplx<KT>);
        nph = int(std::max(1.0, std::min({ double(nblk), std::ceil(double(wcache_bytes) / W_PHASE_BYTES),
            double(n) * g.ks * g.ks * tap_bytes / (trunc ? W_TRUNC_PHASE_READS : W_PHASE_READS) })));
        if (trunc && nph > 1) {
            // two phases' reads and one phase's bytes for the planes' own supports
            const int csw = os / 2 + 1;
            g.planes = int(a.wproj.num_wplanes);
            g.phase_taps = std::max(2.0 * W_PHASE_READS / (double(n) * tap_bytes) * g.planes, W_PHASE_BYTES / (tap_bytes * csw * csw));
        }
    }
    int ext_host = 0; // extra workgroups for split tiles
    const uint32_t* offsets;
    int ostride;
    const uint32_t* bcur = nullptr; // block cursors inside each tile (block binning only)
    const uint32_t* btot = nullptr;
    if (ntiles <= MAX_LDS_TILES) {
        const size_t m = size_t(ntiles) * nblk;
        uint32_t* counts = (uint32_t*)ws_get(ctx, "grid_bcounts", sizeof(uint32_t) * m);
        uint32_t* totals = (uint32_t*)ws_get(ctx, "grid_btotals", sizeof(uint32_t) * ntiles);
        uint32_t* toffs = (uint32_t*)ws_get(ctx, "grid_boffsets", sizeof(uint32_t) * (ntiles + 2));
        const size_t hist_bytes = sizeof(uint32_t) * size_t(ntiles);
        HIP_CHECK(hipFuncSetAttribute((const void*)grid_bin_count_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(hist_bytes)));
        HIP_CHECK(hipFuncSetAttribute((const void*)grid_bin_scatter_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(hist_bytes)));
        ext_host = wproj ? split_extra_max(n, W_SPLIT_MIN) : (mfma ? split_extra_max(n, split_min(int(ntiles), (long long)n)) : 0);
        launch(ctx, "grid_count", grid_bin_count_kernel, dim3(unsigned(nblk)), dim3(BWG), hist_bytes, g, d_uv, d_vis, d_w, counts,
            wpart);
        launch(ctx, "grid_colscan", bin_colscan_kernel, dim3(div_up(ntiles, 64)), dim3(1024), 0, counts, int(nblk), int(ntiles),
            totals);
        launch(ctx, "grid_scatter", grid_bin_scatter_kernel, dim3(unsigned(nblk)), dim3(BWG), hist_bytes, g, d_uv, d_vis, d_w,
            (const uint32_t*)totals, (const uint32_t*)counts, entries, cap, toffs, ext_host);
        if (mfma && a.skip_empty && occ) {
            g.skip = 1;
            *occ = { totals, g.tiles_r, __builtin_ctz(unsigned(g.tc)) };
        }
        offsets = toffs;
        ostride = 1;
        bcur = counts;
        btot = totals;
    } else {
        // very large grids: global per-tile counters
        uint32_t* counts = (uint32_t*)ws_get(ctx, "grid_counts", sizeof(uint32_t) * ntiles);
        uint32_t* offs = (uint32_t*)ws_get(ctx, "grid_offsets", sizeof(uint32_t) * (ntiles + 1));
        uint32_t* cursor = (uint32_t*)ws_get(ctx, "grid_cursor", sizeof(uint32_t) * ntiles);
        fill_u32(ctx, counts, 0u, ntiles);
        launch(ctx, "grid_count", grid_count_kernel, dim3(unsigned(nblk)), dim3(GWG), 0, g, d_uv, d_vis, d_w, counts, wpart);
        exclusive_scan_u32(ctx, counts, ntiles, offs, cursor);
        launch(ctx, "grid_scatter", grid_scatter_kernel, dim3(div_up(n, GWG)), dim3(GWG), 0, g, d_uv, d_vis, d_w, cursor,
            entries, cap);
        offsets = offs;
        ostride = 1;
    }
    if (wproj) {
        const bool big = wcache_bytes > W_BUFFER_MAX;
        const int wv = std::min(W_WAVES, g.tc / W_COLS);
        auto kern = big ? (g.beam ? grid_wtiles_kernel<T, KT, true, true> : grid_wtiles_kernel<T, KT, false, true>)
                        : (g.beam ? grid_wtiles_kernel<T, KT, true, false> : grid_wtiles_kernel<T, KT, false, false>);
        WPhase ph;
        if (nph > 1) {
            ph.one = g.planes > 0 ? offsets + ntiles + 1 : nullptr;
            ph.bcur = bcur;
            ph.btot = btot;
            ph.nblk = int(nblk);
            if (std::is_same<T, double>::value) {
                ph.acc_v = (cplx<double>*)d_vis_grid;
                ph.acc_b = (cplx<double>*)d_sampling_grid;
            } else {
                const size_t cells = size_t(g.rows) * N;
                ph.acc_v = (cplx<double>*)ws_get(ctx, "w_acc", sizeof(cplx<double>) * cells * (g.beam ? 2 : 1));
                ph.acc_b = g.beam ? ph.acc_v + cells : nullptr;
            }
        }
        for (int f = 0; f < nph; f++) {
            ph.b0 = int(size_t(f) * nblk / nph);
            ph.b1 = int(size_t(f + 1) * nblk / nph);
            ph.first = f == 0;
            ph.last = f == nph - 1;
            launch(ctx, "grid_wtiles", kern, dim3(unsigned(ntiles + ext_host) * unsigned(g.tc / (W_COLS * wv))),
                dim3(unsigned(64 * wv)), 0, g, entries, offsets, cap, (const cplx<KT>*)wcache,
                uint32_t(big ? 0 : wcache_bytes), d_vis_grid, d_sampling_grid, ext_host, ph);
        }
    } else {
        STP_REQUIRE(a.kernel_exact || cs * g.ks <= KV_DOUBLES, "oversampled kernel table too large");
        if constexpr (std::is_same<T, float>::value) {
            if (twofloat)
                twofloat_tiles(ctx, g, cs, entries, offsets, ostride, cap, d_tab, d_uv, d_vis_grid, d_sampling_grid);
        }
        if (mfma) {
            const int form = a.kernel_exact ? KERNEL_EXACT : table_form(cs, g.ks);
            auto kern = form == KERNEL_PADDED ? tiles_kernel_of<T, KERNEL_PADDED>(g.tc)
                                              : (form == KERNEL_TABLE ? tiles_kernel_of<T, KERNEL_TABLE>(g.tc)
                                                                      : tiles_kernel_of<T, KERNEL_EXACT>(g.tc));
            const size_t lds = tiles_lds(g.tc, form, cs, g.ks);
            HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
            launch(ctx, "grid_tiles", kern, dim3(unsigned(ntiles + ext_host)), dim3(unsigned(g.tc * 16)), lds, g, entries,
                offsets, cap, d_tab, d_uv, d_vis_grid, d_sampling_grid, ext_host);
        }
    }
    // sample_grid_total = 2 * sum(good weights) (gridder.h:415-423); the good count
    size_t mfin = 0;
    const double* fin = canon_reduce_to_block(ctx, wpart, nblk, wscr, &mfin);
    launch(ctx, "grid_total", grid_total_kernel<T>, dim3(unsigned(1 + merge_blocks(ext_host, g.tc))), dim3(CANON_LANES), 0, fin,
        unsigned(mfin), d_total, d_ngood, offsets + size_t(ntiles) * ostride, a.d_nentries, g, entries, cap, ext_host, d_vis_grid,
        d_sampling_grid);
}

bool grid_batch_eligible(const GridderArgs& a, size_t n)
{
    if (a.wproj.num_wplanes > 0 || a.kernel_exact || a.support < 1 || 2 * a.support + 1 > 16)
        return false;
    const int N = a.image_size;
    const int tc = a.tile_cols > 0 ? a.tile_cols : TILE_C;
    const int rows = a.halfplane ? N / 2 + 1 : N;
    const long long ntiles = (long long)div_up(rows, TILE_R) * div_up(N, tc);
    const int os = std::max(1, (a.oversampling >> 1) << 1);
    const int cs = (os / 2) * 2 + 1;
    return N >= 8 && ntiles <= MAX_LDS_TILES && std::max<size_t>(1, div_up(n, VPB)) <= size_t(CANON_BLOCK) &&
           cs * (2 * a.support + 1) <= KV_DOUBLES;
}

template <typename T>
BatchPlan grid_batch_bin(stp_ctx* ctx, const std::vector<BatchGridItem>& items, const std::vector<uint8_t>& extra)
{
    const int K = int(items.size());
    STP_REQUIRE(K >= 1 && K <= 65535, "1 to 65535 snapshots per fused batch");
    const bool twofloat = std::is_same<T, float>::value && items[0].a.twofloat;
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    // per snapshot: geometry, kernel table, workspace offsets inside one pool
    struct Place {
        size_t counts, totals, toffs, wpart, entries;
    };
    std::vector<BItem> bi(K);
    std::vector<Place> pl(K);
    // tile launches per class: kernel width (up to 8 or 16 taps) x tile width (16, 32,
    // 64 columns), so each launch reserves the LDS its own tiles need
    constexpr int NCLS = BatchPlan::CLASSES;
    std::vector<uint32_t> pre_b(K), pre_c(K), pre_t(size_t(NCLS) * K), pre_m(K);
    size_t nb = 0, nc = 0, nm = 0, nt[NCLS] = {}, pool = 0, hist_bytes = 4, tile_bytes[NCLS] = {};
    for (int k = 0; k < K; k++) {
        const BatchGridItem& it = items[k];
        STP_REQUIRE(grid_batch_eligible(it.a, it.n), "snapshot not eligible for a fused batch");
        STP_REQUIRE((std::is_same<T, float>::value && it.a.twofloat) == twofloat, "one tile-sum form per fused batch");
        KernelFn kf;
        BItem& b = bi[k];
        b.g = make_geom(it.a, it.n, it.a.generate_beam && it.bgrid != nullptr, kf);
        const GridGeom& g = b.g;
        const int ntiles = g.tiles_r * g.tiles_c;
        const size_t nblk = std::max<size_t>(1, div_up(it.n, VPB));
        const size_t cap64 = std::max<size_t>(1, 2 * footprint_tiles_max(g) * it.n);
        STP_REQUIRE(cap64 < (size_t(1) << 32), "too many gridding entries for one snapshot");
        char key[160];
        snprintf(key, sizeof(key), "k1d:%d:%.17g:%.17g:%.17g:%d:%d", kf.kind, kf.param, kf.width_g, kf.width_s, it.a.support,
            g.os);
        b.ktab = has_table(ctx, key) ? dev_table(ctx, key, {}) : dev_table(ctx, key, kernel_1d_table(kf, it.a.support, g.os));
        b.uv = it.uv;
        b.vis = it.vis;
        b.wts = it.wts;
        b.vgrid = it.vgrid;
        b.bgrid = g.beam ? it.bgrid : nullptr;
        b.total = it.total;
        b.ngood = it.ngood;
        b.g.skip = it.a.skip_empty && !twofloat ? 1 : 0;
        b.cap = uint32_t(cap64);
        b.nblk = int(nblk);
        Place& p = pl[k];
        p.counts = pool;
        pool = al(pool + sizeof(uint32_t) * nblk * ntiles);
        p.totals = pool;
        pool = al(pool + sizeof(uint32_t) * ntiles);
        p.toffs = pool;
        pool = al(pool + sizeof(uint32_t) * (ntiles + 1));
        p.wpart = pool;
        pool = al(pool + sizeof(double) * (2 * nblk + 2));
        p.entries = pool;
        pool = al(pool + sizeof(Entry) * cap64);
        b.ext_host = twofloat ? 0 : split_extra_max(it.n, split_min(int(ntiles), (long long)it.n));
        pre_m[k] = uint32_t(nm);
        nm += merge_blocks(b.ext_host, g.tc);
        pre_b[k] = uint32_t(nb);
        nb += nblk;
        pre_c[k] = uint32_t(nc);
        nc += div_up(ntiles, 64);
        const int form = table_form((g.os / 2) * 2 + 1, g.ks);
        const int cls = ((twofloat ? g.ks <= 8 : form == KERNEL_PADDED) ? 0 : 3) + (g.tc == 16 ? 0 : (g.tc == 32 ? 1 : 2));
        for (int c = 0; c < NCLS; c++)
            pre_t[size_t(c) * K + k] = uint32_t(nt[c]);
        nt[cls] += size_t(ntiles) + b.ext_host;
        hist_bytes = std::max(hist_bytes, sizeof(uint32_t) * size_t(ntiles));
        const int cs = (g.os / 2) * 2 + 1;
        size_t lds;
        if (twofloat) {
            const int S = TILE_R + (g.ks <= 15 ? g.ks : 1);
            lds = ((6 * sizeof(float) * (size_t(g.tc) * S) + 7) / 8) * 8 + sizeof(double) * size_t(cs) * g.ks;
        } else {
            lds = tiles_lds(g.tc, form, cs, g.ks);
        }
        tile_bytes[cls] = std::max(tile_bytes[cls], lds);
    }
    STP_REQUIRE(nb < (size_t(1) << 31) && *std::max_element(nt, nt + NCLS) < (size_t(1) << 31),
        "too many workgroups for one fused batch");
    uint8_t* base = (uint8_t*)ws_get(ctx, "bat_pool", pool);
    std::vector<TileOcc> occ(K);
    for (int k = 0; k < K; k++) {
        bi[k].counts = (uint32_t*)(base + pl[k].counts);
        bi[k].totals = (uint32_t*)(base + pl[k].totals);
        bi[k].toffs = (uint32_t*)(base + pl[k].toffs);
        bi[k].wpart = (double*)(base + pl[k].wpart);
        bi[k].entries = (Entry*)(base + pl[k].entries);
        if (bi[k].g.skip)
            occ[k] = { bi[k].totals, bi[k].g.tiles_r, __builtin_ctz(unsigned(bi[k].g.tc)) };
    }
    // tables: items, the stage prefixes, the occupied tiles, the caller's tables; one upload from the
    // page-locked stage once the previous batch's upload has left it
    const size_t o_items = 0, o_b = al(sizeof(BItem) * K), o_c = o_b + al(4 * K), o_t = o_c + al(4 * K);
    const size_t o_m = o_t + al(4 * size_t(NCLS) * K), o_o = o_m + al(4 * K), o_x = o_o + al(sizeof(TileOcc) * K), tab_bytes = o_x + std::max<size_t>(extra.size(), 1);
    hipEvent_t& up = ctx->batch_tab_events[ctx->ws_slot];
    if (!up)
        HIP_CHECK(hipEventCreateWithFlags(&up, hipEventDisableTiming));
    HIP_CHECK(hipEventSynchronize(up));
    uint8_t* h = (uint8_t*)host_stage(ctx, "bat_tabs#" + std::to_string(ctx->ws_slot), tab_bytes);
    uint8_t* d = (uint8_t*)ws_get(ctx, "bat_tabs", tab_bytes);
    memcpy(h + o_items, bi.data(), sizeof(BItem) * K);
    memcpy(h + o_b, pre_b.data(), 4 * K);
    memcpy(h + o_c, pre_c.data(), 4 * K);
    memcpy(h + o_t, pre_t.data(), 4 * size_t(NCLS) * K);
    memcpy(h + o_m, pre_m.data(), 4 * K);
    memcpy(h + o_o, occ.data(), sizeof(TileOcc) * K);
    if (!extra.empty())
        memcpy(h + o_x, extra.data(), extra.size());
    HIP_CHECK(hipMemcpyAsync(d, h, tab_bytes, hipMemcpyHostToDevice, ctx->stream));
    HIP_CHECK(hipEventRecord(up, ctx->stream));
    const BItem* d_items = (const BItem*)(d + o_items);
    const uint32_t* d_pre_b = (const uint32_t*)(d + o_b);
    HIP_CHECK(hipFuncSetAttribute((const void*)batch_count_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(hist_bytes)));
    HIP_CHECK(hipFuncSetAttribute((const void*)batch_scatter_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(hist_bytes)));
    launch(ctx, "batch_count", batch_count_kernel, dim3(unsigned(nb)), dim3(BWG), hist_bytes, d_items, d_pre_b, K);
    launch(ctx, "batch_colscan", batch_colscan_kernel, dim3(unsigned(nc)), dim3(1024), 0, d_items, (const uint32_t*)(d + o_c), K);
    launch(ctx, "batch_scatter", batch_scatter_kernel, dim3(unsigned(nb)), dim3(BWG), hist_bytes, d_items, d_pre_b, K);
    BatchPlan plan;
    plan.d_tab = d;
    plan.d_extra = d + o_x;
    plan.d_occ = (const TileOcc*)(d + o_o);
    plan.items = K;
    plan.twofloat = twofloat;
    plan.pre_t_off = o_t;
    plan.pre_m_off = o_m;
    plan.merges = nm;
    for (int c = 0; c < NCLS; c++) {
        plan.tiles[c] = nt[c];
        plan.tile_lds[c] = tile_bytes[c];
    }
    return plan;
}

template <typename T>
void grid_batch_tiles(stp_ctx* ctx, const BatchPlan& plan)
{
    const BItem* d_items = (const BItem*)plan.d_tab;
    const int K = plan.items;
    for (int c = 0; c < BatchPlan::CLASSES; c++) {
        if (plan.tiles[c] == 0)
            continue;
        const uint32_t* pre = (const uint32_t*)((const uint8_t*)plan.d_tab + plan.pre_t_off) + size_t(c) * K;
        if constexpr (std::is_same<T, float>::value) {
            if (plan.twofloat) {
                auto kern = c < 3 ? batch_tiles_twofloat_kernel<AccTwoFloat, 8> : batch_tiles_twofloat_kernel<AccTwoFloat, 16>;
                HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(plan.tile_lds[c])));
                launch(ctx, "batch_tiles", kern, dim3(unsigned(plan.tiles[c])), dim3(TWG), plan.tile_lds[c], d_items, pre, K);
                continue;
            }
        }
        const int w = c % 3;
        auto kern = c < 3 ? (w == 0 ? batch_tiles_kernel<T, 16, KERNEL_PADDED>
                                    : (w == 1 ? batch_tiles_kernel<T, 32, KERNEL_PADDED> : batch_tiles_kernel<T, 64, KERNEL_PADDED>))
                          : (w == 0 ? batch_tiles_kernel<T, 16, KERNEL_TABLE>
                                    : (w == 1 ? batch_tiles_kernel<T, 32, KERNEL_TABLE> : batch_tiles_kernel<T, 64, KERNEL_TABLE>));
        HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(plan.tile_lds[c])));
        launch(ctx, "batch_tiles", kern, dim3(unsigned(plan.tiles[c])), dim3(256u << w),
            plan.tile_lds[c], d_items, pre, K);
    }
    launch(ctx, "batch_total", batch_total_kernel<T>, dim3(unsigned(K + plan.merges)), dim3(CANON_LANES), 0, d_items,
        (const uint32_t*)((const uint8_t*)plan.d_tab + plan.pre_m_off), K);
}

template <typename T>
const void* grid_batch(stp_ctx* ctx, const std::vector<BatchGridItem>& items, const std::vector<uint8_t>& extra)
{
    const BatchPlan plan = grid_batch_bin<T>(ctx, items, extra);
    grid_batch_tiles<T>(ctx, plan);
    return plan.d_extra;
}

template BatchPlan grid_batch_bin<double>(stp_ctx*, const std::vector<BatchGridItem>&, const std::vector<uint8_t>&);
template BatchPlan grid_batch_bin<float>(stp_ctx*, const std::vector<BatchGridItem>&, const std::vector<uint8_t>&);
template void grid_batch_tiles<double>(stp_ctx*, const BatchPlan&);
template void grid_batch_tiles<float>(stp_ctx*, const BatchPlan&);
template const void* grid_batch<double>(stp_ctx*, const std::vector<BatchGridItem>&, const std::vector<uint8_t>&);
template const void* grid_batch<float>(stp_ctx*, const std::vector<BatchGridItem>&, const std::vector<uint8_t>&);

size_t gridder_entry_capacity(int N, bool halfplane, int support, bool exact, int tile_cols, size_t n)
{
    GridGeom g;
    g.N = N;
    g.rows = halfplane ? N / 2 + 1 : N;
    g.s = support;
    g.ks = 2 * support + 1;
    g.exact = exact ? 1 : 0;
    g.tc = tile_cols > 0 ? tile_cols : TILE_C;
    return std::max<size_t>(1, 2 * footprint_tiles_max(g) * n);
}

template void grid_visibilities<double>(stp_ctx*, const GridderArgs&, size_t, const double*, const double*,
    const double*, cplx<double>*, cplx<double>*, double*, unsigned long long*, TileOcc*);
template void grid_visibilities<float>(stp_ctx*, const GridderArgs&, size_t, const double*, const double*,
    const double*, cplx<float>*, cplx<float>*, double*, unsigned long long*, TileOcc*);

} // namespace stp_hip
