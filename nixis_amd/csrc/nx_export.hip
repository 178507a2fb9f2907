// nx_export.hip -- equirectangular export on the device (nixis.py:270-302,
// util.py:275-366): pixel coordinates (make_ll_arr), the k nearest mesh
// vertices of each pixel (the reference's scipy KD-tree query) and the
// inverse-distance sampling of make_gray_array.
//
// Nearest neighbours come from a bin structure instead of a tree: points are
// counted into bins and stored bin by bin, and a query scans the bins around
// it, in growing blocks, until the k-th best distance is no larger than the
// least distance that a point outside the block can have, so the result is
// the exact k nearest (ties ordered by point index, whatever the order inside
// a bin).  Two kinds of bins, chosen on the device when the grid is built:
//   shell  points that surround the origin at nearly one radius (a planet's
//          vertices): bands of equal latitude height, each cut into cells of
//          about the same width in longitude.  A band's cells are consecutive
//          in memory, so a block of 3 x 3 cells is three runs of points with
//          no search; the band table has about 0.74 sqrt(V) entries.
//   cells  any other points: cubes of a uniform grid, hashed into at least
//          2V bins.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "nx_ctx.h"
#include "nx_erosion_dev.h"
#include "nx_reduce_dev.h"

namespace nx {

namespace {

constexpr int kKnnMax = 8;                // largest k
constexpr int kAxisBits = 21;             // cell coordinate bits per axis
// Height of a band, in mean spacings sqrt(4 pi / V) of V points on the unit
// sphere.  The third nearest vertex of an icosphere lies within 1.18 of
// them, so a block reaching one band and cell beyond the query's own settles
// the reference's k = 3 in one round, over about 13 points.
constexpr double kBandSpacings = 1.2;
// Slack of the FP32 latitudes and longitudes, in radians (their rounding is
// below 1e-6), and of the FP64 comparison of squared distances.
constexpr float kAngleSlack = 2e-6f;
constexpr double kGuardSlack = 1e-6;
constexpr int kBoxBlocks = 256;           // one per CU
constexpr int kScanBlocks = 1024;

struct GridHead {
    double origin[3];
    double cell;
    int32_t dims[3];
    int32_t shell;              // 1: latitude bands, 0: hashed cells
    int64_t nbins;
    double rmin, rmax;          // shell: least and largest |p|
    double cosa[2], sin2a[2];   // shell: cos a and sin^2 (a / 2) of blocks of 1 and 2 bands
    float sina[2];              // sin of 1 and 2 band heights
    float perband;              // bands per radian
    double unit, fixed;         // 1 and kFixed over rmax
};
static_assert(sizeof(GridHead) <= 256, "grid head must fit its 256 bytes");

// A point in bin order.  Shell: its coordinates in units of rmax / 2^29, so a
// query's differences to it are exact integers (kFixed).  Cells use the index
// alone.
struct alignas(16) GridEntry {
    int32_t x, y, z, idx;
};
constexpr double kFixed = 0x1p29;
constexpr int kStage = 256;   // entries a wave stages (16 KB for a block's four waves)

inline size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

uint64_t table_size(int64_t V)
{
    uint64_t t = 64;
    while (t < 2 * (uint64_t)V) t <<= 1;
    return t;
}

int32_t band_count(int64_t V)
{
    const double h = kBandSpacings * std::sqrt(4.0 * 3.141592653589793 / (double)V);
    return (int32_t)std::max(1.0, std::floor(3.141592653589793 / h));
}

struct GridLayout {
    size_t head, band, start, entry, pts, bin, rank, part, total;
    uint64_t tsize;    // bins for hashed cells
    int32_t bands;
};

GridLayout grid_layout(int64_t V)
{
    GridLayout L;
    L.bands = band_count(V);
    L.tsize = table_size(V);
    size_t o = 0;
    L.head = o;
    o += 256;
    L.band = o;
    o += a256(4 * ((size_t)L.bands + 1));
    L.start = o;
    o += a256(4 * ((size_t)L.tsize + 1));
    L.entry = o;
    o += a256(sizeof(GridEntry) * (size_t)V);
    L.pts = o;
    o += a256(24 * (size_t)V);
    L.bin = o;
    o += a256(4 * (size_t)V);
    L.rank = o;
    o += a256(4 * (size_t)V);
    L.part = o;
    o += a256(8 * 8 * kBoxBlocks);
    L.total = o;
    return L;
}

// MurmurHash3's 64-bit finaliser.
__device__ __forceinline__ uint64_t mix64(uint64_t x)
{
    x ^= x >> 33;
    x *= 0xff51afd7ed558ccdULL;
    x ^= x >> 33;
    x *= 0xc4ceb9fe1a85ec53ULL;
    x ^= x >> 33;
    return x;
}

__device__ __forceinline__ unsigned long long cell_key(int x, int y, int z)
{
    return ((unsigned long long)x << (2 * kAxisBits)) | ((unsigned long long)y << kAxisBits) |
           (unsigned long long)z;
}

// The bin of a cell: blocks of 4 x 4 x 4 cells are hashed, a block's bins are
// consecutive, so that the bins and points around a query share their lines.
__device__ __forceinline__ uint64_t cell_bin(int x, int y, int z, uint64_t mask)
{
    return (mix64(cell_key(x >> 2, y >> 2, z >> 2)) << 6 |
            (uint64_t)((x & 3) << 4 | (y & 3) << 2 | (z & 3))) & mask;
}

__device__ __forceinline__ int cell_of(double q, double o, double cell, int dim)
{
    const double t = floor((q - o) / cell);
    if (!(t >= 0.0)) return 0;  // below the grid, or NaN
    return t >= (double)(dim - 1) ? dim - 1 : (int)t;
}

// Latitude + pi / 2, longitude + pi and the cosine of the latitude of a
// direction, in FP32 (within kAngleSlack); scale brings it near length 1.
__device__ __forceinline__ void angles_of(double x, double y, double z, double scale, float &lat,
                                          float &lon, float &clat)
{
    const float fx = (float)(x * scale), fy = (float)(y * scale), fz = (float)(z * scale);
    const float rho = sqrtf(fx * fx + fy * fy);
    lat = atan2f(fz, rho) + 1.57079633f;
    lon = atan2f(fy, fx) + 3.14159265f;
    clat = rho / sqrtf(rho * rho + fz * fz);
}

__device__ __forceinline__ int clamp_cell(float t, int n) { return min(max((int)t, 0), n - 1); }

__device__ __forceinline__ int band_of(float lat, int bands, float perband)
{
    return clamp_cell(lat * perband, bands);
}

}  // namespace

// Box of the points and least / largest squared norm, one record of eight
// order-preserving keys per block.
__global__ __launch_bounds__(1024) void k_grid_box(const double *__restrict__ pts, int64_t V,
                                                   unsigned long long *__restrict__ part)
{
    unsigned long long lo[4], hi[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        lo[k] = ~0ull;
        hi[k] = 0ull;
    }
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
#pragma unroll 2
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < V; i += step) {
        const double p[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
        const unsigned long long q[4] = {dkey(p[0]), dkey(p[1]), dkey(p[2]),
                                         dkey(p[0] * p[0] + p[1] * p[1] + p[2] * p[2])};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lo[k] = q[k] < lo[k] ? q[k] : lo[k];
            hi[k] = q[k] > hi[k] ? q[k] : hi[k];
        }
    }
    __shared__ unsigned long long red[16][8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long a = __shfl_xor(lo[k], off, 64), b = __shfl_xor(hi[k], off, 64);
            lo[k] = a < lo[k] ? a : lo[k];
            hi[k] = b > hi[k] ? b : hi[k];
        }
        if ((threadIdx.x & 63) == 0) {
            red[threadIdx.x >> 6][2 * k] = lo[k];
            red[threadIdx.x >> 6][2 * k + 1] = hi[k];
        }
    }
    __syncthreads();
    if (threadIdx.x < 8) {   // minima are even
        unsigned long long a = red[0][threadIdx.x];
        for (int w = 1; w < 16; ++w) {
            const unsigned long long c = red[w][threadIdx.x];
            a = ((c < a) != (threadIdx.x & 1)) ? c : a;
        }
        part[8 * blockIdx.x + threadIdx.x] = a;
    }
}

// Grid geometry (one block).  Points with norms in [0.8, 1] of the largest
// that reach 0.7 of it on both sides of every axis get latitude bands: those
// are sized for points over the whole sphere, and a band's cells bound the
// distance of their points by direction alone.  Others get cells with an edge
// of twice the mean spacing of V points spread over the sphere that fits the
// box, at most 2^21 - 1 per axis.  The geometry only sets the speed; the
// search is exact for any.
__global__ __launch_bounds__(1024) void k_grid_setup(GridHead *__restrict__ g, int64_t V,
                                                     const unsigned long long *__restrict__ part,
                                                     int parts, int32_t bands, uint64_t tsize,
                                                     int32_t *__restrict__ band)
{
    __shared__ double box[8];
    __shared__ int shell;
    const int t = threadIdx.x;
    if (t < 512) {   // wave w joins key w: minima are even
        const int w = t >> 6;
        unsigned long long a = part[w];
        for (int i = t & 63; i < parts; i += 64) {
            const unsigned long long c = part[8 * i + w];
            a = ((c < a) != (w & 1)) ? c : a;
        }
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long c = __shfl_xor(a, off, 64);
            a = ((c < a) != (w & 1)) ? c : a;
        }
        if ((t & 63) == 0) box[w] = dunkey(a);
    }
    __syncthreads();
    const double pi = 3.141592653589793, h = pi / bands;
    if (t == 0) {
        double ext[3], R = 0.0;
        const double n0 = box[6], n1 = box[7];
        bool s = n1 >= 0x1p-600 && n1 <= 0x1p600 && n0 >= 0.64 * n1;
        for (int k = 0; k < 3; ++k) {
            ext[k] = box[2 * k + 1] - box[2 * k];
            R = fmax(R, 0.5 * ext[k]);
            s = s && box[2 * k] <= -0.7 * sqrt(n1) && box[2 * k + 1] >= 0.7 * sqrt(n1);
        }
        double cell = 2.0 * sqrt(4.0 * pi * R * R / (double)V);
        for (int k = 0; k < 3; ++k) {
            const double need = ext[k] / 2097150.0;
            if (cell < need) cell = need;
        }
        if (!(cell > 0.0)) cell = 1.0;  // all points equal
        g->cell = cell;
        for (int k = 0; k < 3; ++k) {
            g->origin[k] = box[2 * k];
            const double n = floor(ext[k] / cell) + 1.0;
            g->dims[k] = (int32_t)fmin(n, 2097151.0);
        }
        g->shell = shell = s;
        g->rmin = sqrt(n0) * (1.0 - kGuardSlack);
        g->rmax = sqrt(n1) * (1.0 + kGuardSlack);
        g->unit = 1.0 / g->rmax;
        g->fixed = kFixed / g->rmax;
        g->perband = (float)bands * 0.318309886f;
        if (!s) g->nbins = (int64_t)tsize;
    }
    if ((t & 63) == 0 && (t >> 6) >= 1 && (t >> 6) <= 2) {
        const int r = t >> 6;
        const double a = r * h - 2.0 * kAngleSlack, s2 = sin(0.5 * a);
        g->cosa[r - 1] = 1.0 - 2.0 * s2 * s2;
        g->sin2a[r - 1] = s2 * s2;
        g->sina[r - 1] = r * h < 1.5 ? sinf((float)(r * h)) : 2.0f;
    }
    __syncthreads();
    if (!shell) return;
    // cells of each band and their running sum
    __shared__ int32_t wsum[16];
    int32_t carry = 0;
    for (int32_t b0 = 0; b0 < bands; b0 += 1024) {
        const int32_t b = b0 + t;
        int32_t n = 0;
        if (b < bands) n = max(1, (int32_t)(2.0f * (float)bands * sinf(((float)b + 0.5f) * (float)h)));
        int32_t inc = n;
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t o = __shfl_up(inc, off, 64);
            if ((t & 63) >= off) inc += o;
        }
        if ((t & 63) == 63) wsum[t >> 6] = inc;
        __syncthreads();
        int32_t before = carry, all = carry;
        for (int w = 0; w < 16; ++w) {
            if (w < (t >> 6)) before += wsum[w];
            all += wsum[w];
        }
        if (b < bands) band[b] = before + inc - n;
        carry = all;
        __syncthreads();
    }
    if (t == 0) {
        band[bands] = carry;
        g->nbins = carry;
    }
}

__global__ __launch_bounds__(256) void k_grid_clear(const GridHead *__restrict__ g,
                                                    int32_t *__restrict__ count)
{
    const int64_t n = g->nbins;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        count[i] = 0;
}

// Each point's bin and its rank among the bin's points.  Bound by the counters'
// atomics, which run at the memory side: 10,000,002 points take 308 us (337
// with a contiguous eighth of the points on each XCD).
__global__ __launch_bounds__(256) void k_grid_count(const double *__restrict__ pts, int64_t V,
                                                    const GridHead *__restrict__ g,
                                                    const int32_t *__restrict__ band, int32_t bands,
                                                    int32_t *__restrict__ count,
                                                    uint32_t *__restrict__ bin,
                                                    int32_t *__restrict__ rank)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= V) return;
    const double x = pts[3 * i], y = pts[3 * i + 1], z = pts[3 * i + 2];
    uint32_t b;
    if (g->shell) {
        float lat, lon, clat;
        angles_of(x, y, z, g->unit, lat, lon, clat);
        const int r = band_of(lat, bands, g->perband);
        const int n = band[r + 1] - band[r];
        b = (uint32_t)(band[r] + clamp_cell(lon * ((float)n * 0.159154943f), n));
    } else {
        const double c = g->cell;
        b = (uint32_t)cell_bin(cell_of(x, g->origin[0], c, g->dims[0]),
                               cell_of(y, g->origin[1], c, g->dims[1]),
                               cell_of(z, g->origin[2], c, g->dims[2]), (uint64_t)(g->nbins - 1));
    }
    bin[i] = b;
    rank[i] = __hip_atomic_fetch_add(&count[b], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Points of each of gridDim.x equal runs of bins.
__global__ __launch_bounds__(256) void k_grid_sums(const GridHead *__restrict__ g,
                                                   const int32_t *__restrict__ count,
                                                   int32_t *__restrict__ sums)
{
    const int64_t n = g->nbins, per = (n + gridDim.x - 1) / gridDim.x;
    const int64_t a = per * blockIdx.x, e = min(n, a + per);
    int32_t s = 0;
    for (int64_t i = a + threadIdx.x; i < e; i += 256) s += count[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    __shared__ int32_t w[4];
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = w[0] + w[1] + w[2] + w[3];
}

// Counts to the first point of each bin, in place, over the same runs;
// start[nbins] = V.
__global__ __launch_bounds__(256) void k_grid_starts(const GridHead *__restrict__ g, int64_t V,
                                                     const int32_t *__restrict__ sums,
                                                     int32_t *__restrict__ start)
{
    const int64_t n = g->nbins, per = (n + gridDim.x - 1) / gridDim.x;
    const int64_t a = per * blockIdx.x, e = min(n, a + per);
    const int t = threadIdx.x, wave = t >> 6;
    __shared__ int32_t w[4];
    int32_t s = 0;
    for (int i = t; i < (int)blockIdx.x; i += 256) s += sums[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((t & 63) == 0) w[wave] = s;
    __syncthreads();
    int32_t carry = w[0] + w[1] + w[2] + w[3];
    for (int64_t i0 = a; i0 < e; i0 += 256) {
        const int64_t i = i0 + t;
        const int32_t c = i < e ? start[i] : 0;
        int32_t inc = c;
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t o = __shfl_up(inc, off, 64);
            if ((t & 63) >= off) inc += o;
        }
        __syncthreads();
        if ((t & 63) == 63) w[wave] = inc;
        __syncthreads();
        int32_t before = carry;
        for (int k = 0; k < 4; ++k)
            if (k < wave) before += w[k];
        if (i < e) start[i] = before + inc - c;
        carry += w[0] + w[1] + w[2] + w[3];
    }
    if (blockIdx.x == 0 && t == 0) start[n] = (int32_t)V;
}

// Entries in bin order; the points themselves stay in the caller's order for
// a shell (read once per result) and go into bin order for cells (read once
// per candidate).
__global__ __launch_bounds__(256) void k_grid_place(const double *__restrict__ pts, int64_t V,
                                                    const GridHead *__restrict__ g,
                                                    const int32_t *__restrict__ start,
                                                    const uint32_t *__restrict__ bin,
                                                    const int32_t *__restrict__ rank,
                                                    GridEntry *__restrict__ entry,
                                                    double *__restrict__ out)
{
    const int64_t i = xcd_tile(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (i >= V) return;
    const double x = pts[3 * i], y = pts[3 * i + 1], z = pts[3 * i + 2];
    const int64_t at = (int64_t)start[bin[i]] + rank[i];
    GridEntry e{0, 0, 0, (int32_t)i};
    int64_t to = at;
    if (g->shell) {
        const double f = g->fixed;
        e.x = (int32_t)rint(x * f);
        e.y = (int32_t)rint(y * f);
        e.z = (int32_t)rint(z * f);
        to = i;
    }
    entry[at] = e;
    out[3 * to] = x;
    out[3 * to + 1] = y;
    out[3 * to + 2] = z;
}

namespace {

struct GridView {
    const GridHead *g;
    const int32_t *band;
    const int32_t *start;
    const GridEntry *entry;
    const double *pts;
    int32_t bands;
};

__device__ __forceinline__ bool before(double s, int32_t i, double t, int32_t j)
{
    return s < t || (s == t && i < j);
}

// Squared distance as the reference's KD-tree sums it.
__device__ __forceinline__ double dist2(const double *__restrict__ p, double qx, double qy,
                                        double qz)
{
    double s = 0.0, d;
    d = qx - p[0];
    s += d * d;
    d = qy - p[1];
    s += d * d;
    d = qz - p[2];
    s += d * d;
    return s;
}

__device__ __forceinline__ void order(double &s, int32_t &i, double &t, int32_t &j)
{
    const bool swap = before(t, j, s, i);
    const double a = swap ? t : s, b = swap ? s : t;
    const int32_t c = swap ? j : i, d = swap ? i : j;
    s = a;
    t = b;
    i = c;
    j = d;
}

// (s, id) into the K best so far, which are in order.
template <int K>
__device__ __forceinline__ void insert(double s, int32_t id, double (&bd)[K], int32_t (&bi)[K])
{
    bd[K - 1] = s;
    bi[K - 1] = id;
#pragma unroll
    for (int m = K - 1; m > 0; --m) order(bd[m - 1], bi[m - 1], bd[m], bi[m]);
}

template <int K>
__device__ __forceinline__ void none_yet(double (&bd)[K], int32_t (&bi)[K])
{
#pragma unroll
    for (int j = 0; j < K; ++j) {
        bd[j] = INFINITY;
        bi[j] = INT32_MAX;
    }
}

// How many points a query reads together from a dense run (scan).  More cover
// more latency but take registers, which the pixels' kernels need for waves
// (8192 x 4096 on d=1000, K = 3: 939 us at 2 and seven waves, 1,055 at 4 and six;
// points in the caller's order are faster with fewer waves anyway: 3,333,334
// queries on d=1000, 497 us at 4 and four waves, 643 at 2 and seven).
constexpr int kPointScan = 4;
constexpr int pixel_scan(int k) { return k <= 3 ? 2 : 4; }

// The points of entries j..e-1 among the K best, T at a time, so that a long
// run's loads go out together.  SHELL: an entry lies within 0.87 of its unit of
// its point, so its own distance tells whether the point can be among the K
// (most: squared, in units, the largest that can, with slack for FP32); where
// none of T can, no point is read.  AGAIN: points may come that were met before.
// 499,281 queries of 998,562 vertices off the origin (cells): 263 us, 670 where
// each candidate's entry was read and compared before its point and cells were
// hashed one by one.
template <int K, int T, bool SHELL, bool AGAIN>
__device__ __forceinline__ void scan(const GridView &v, int j, int e, double qx, double qy,
                                     double qz, double f, float &most, double (&bd)[K],
                                     int32_t (&bi)[K])
{
    for (; j < e; j += T) {
        double s[T];
        int32_t id[T];
        if (SHELL) {
            bool near = false;
#pragma unroll
            for (int u = 0; u < T; ++u) {
                const GridEntry p = v.entry[min(j + u, e - 1)];
                const float dx = (float)fma(qx, f, -(double)p.x), dy = (float)fma(qy, f, -(double)p.y),
                            dz = (float)fma(qz, f, -(double)p.z);
                near = near || !(fmaf(dz, dz, fmaf(dy, dy, dx * dx)) > most);
                id[u] = p.idx;
            }
            if (!near) continue;
        }
        double least = INFINITY;
#pragma unroll
        for (int u = 0; u < T; ++u) {
            const int at = min(j + u, e - 1);
            if (!SHELL) id[u] = v.entry[at].idx;
            s[u] = dist2(v.pts + 3 * (int64_t)(SHELL ? id[u] : at), qx, qy, qz);
            least = fmin(least, s[u]);
        }
        if (!(least <= bd[K - 1])) continue;
        bool better = false;   // (not for ties with a lower index)
#pragma unroll
        for (int u = 0; u < T; ++u) {
            if (u > 0 && j + u >= e) {
                s[u] = INFINITY;
                id[u] = INT32_MAX;
            }
            better = better || before(s[u], id[u], bd[K - 1], bi[K - 1]);
        }
        if (!better) continue;
#pragma unroll 1
        for (int u = 0; u < T; ++u) {
            bool held = false;
            if (AGAIN)
#pragma unroll
                for (int h = 0; h < K; ++h) held = held || bi[h] == id[0];
            if (!held && before(s[0], id[0], bd[K - 1], bi[K - 1])) insert<K>(s[0], id[0], bd, bi);
#pragma unroll
            for (int w = 1; w < T; ++w) {
                s[w - 1] = s[w];
                id[w - 1] = id[w];
            }
        }
        if (SHELL) {
            const float far = (float)(sqrt(bd[K - 1]) * f) + 2.0f;
            most = far * far * (1.0f + 2e-6f);
        }
    }
}

// The K nearest points of q among hashed cells: shells of cells around q's
// cell until the K-th squared distance is within the block's guaranteed
// radius (the distance from q to the nearest face of the block that does not
// lie on the grid's border, less a margin for rounding of the cell bounds).
template <int K, int T>
__device__ __forceinline__ void knn_cells(const GridView &v, double qx, double qy, double qz,
                                       double (&bd)[K], int32_t (&bi)[K])
{
    const GridHead &g = *v.g;
    const double ox = g.origin[0], oy = g.origin[1], oz = g.origin[2], cell = g.cell;
    const int dx = g.dims[0], dy = g.dims[1], dz = g.dims[2];
    const uint64_t mask = (uint64_t)(g.nbins - 1);
    none_yet<K>(bd, bi);
    const int cx = cell_of(qx, ox, cell, dx);
    const int cy = cell_of(qy, oy, cell, dy);
    const int cz = cell_of(qz, oz, cell, dz);
    const int rmax = max(dx, max(dy, dz));
    const double margin = 1e-9 * cell;
    float most = 0.0f;   // (shells only)
    for (int r = 0; r <= rmax; ++r) {
        for (int z = cz - r; z <= cz + r; ++z) {
            if (z < 0 || z >= dz) continue;
            for (int y = cy - r; y <= cy + r; ++y) {
                if (y < 0 || y >= dy) continue;
                const bool face = (z == cz - r || z == cz + r || y == cy - r || y == cy + r);
                const int step = (face || r == 0) ? 1 : 2 * r;
                for (int x = cx - r; x <= cx + r; x += step) {
                    if (x < 0 || x >= dx) continue;
                    const int32_t *s = v.start + cell_bin(x, y, z, mask);
                    // other cells' points in the bin are no worse candidates
                    scan<K, T, false, true>(v, s[0], s[1], qx, qy, qz, 0.0, most, bd, bi);
                }
            }
        }
        double guar = INFINITY;
        if (cx - r > 0) guar = fmin(guar, qx - (ox + (cx - r) * cell));
        if (cx + r + 1 < dx) guar = fmin(guar, (ox + (cx + r + 1) * cell) - qx);
        if (cy - r > 0) guar = fmin(guar, qy - (oy + (cy - r) * cell));
        if (cy + r + 1 < dy) guar = fmin(guar, (oy + (cy + r + 1) * cell) - qy);
        if (cz - r > 0) guar = fmin(guar, qz - (oz + (cz - r) * cell));
        if (cz + r + 1 < dz) guar = fmin(guar, (oz + (cz + r + 1) * cell) - qz);
        if (guar == INFINITY) break;  // the block covers the whole grid
        guar -= margin;
        if (guar > 0.0 && bd[K - 1] <= guar * guar) break;
    }
}

// Latitude bands.  A round of reach a visits the bands within a of q's latitude
// (or r bands on either side, a = r h for a band height h) and, in each, the
// cells within longitude D of q, sin D = sin a / cos(latitude of q) (all cells
// where that passes 1, near the poles).  Every point not visited then lies at
// an angle of at least a from q (its latitude differs by that, or its meridian
// passes q no nearer), and with a norm in [rmin, rmax] its squared distance is
// at least (|q| - t)^2 + 4 |q| t sin^2(a / 2), t = |q| cos a clamped to those
// norms.
struct ShellQuery {
    double x, y, z, norm;
    float lat, lon, clat;
    int own;   // q's band
};

// The visited part of a band: entries ja.. (na of them), then jb.. (to n): a
// window past either end of the band continues at the other end.
struct Run {
    int ja, na, jb, n;
    __device__ __forceinline__ int at(int i) const { return i + (i < na ? ja : jb - na); }
};

__device__ __forceinline__ Run band_run(const GridView &v, const ShellQuery &q, int b, float D,
                                        bool circle)
{
    Run run{0, 0, 0, 0};
    if (b < 0 || b >= v.bands) return run;
    const int base = v.band[b], n = v.band[b + 1] - base;
    const int32_t *start = v.start + base;
    const float per = (float)n * 0.159154943f;
    int c0 = (int)floorf((q.lon - D) * per), c1 = (int)floorf((q.lon + D) * per);
    if (circle || c1 - c0 >= n - 1) {
        c0 = 0;
        c1 = n - 1;
    }
    const bool wrap = c0 < 0 || c1 >= n;
    const int a = c0 < 0 ? c0 + n : c0, e = c1 >= n ? c1 - n : c1;
    run.ja = start[a];
    run.na = start[wrap ? n : e + 1] - run.ja;
    run.n = run.na;
    if (wrap) {
        run.jb = start[0];
        run.n += start[e + 1] - run.jb;
    }
    return run;
}

// asin x <= x + (pi / 2 - 1) x^3 on [0, 1].
__device__ __forceinline__ float window(float sina, float clat, bool &circle)
{
    const float x = sina * __builtin_amdgcn_rcpf(clat);   // within the slack
    circle = !(x < 0.99f);
    return circle ? 0.0f : x * (1.0f + 0.5709f * x * x) + 4.0f * kAngleSlack;
}

// Least squared distance of a point at an angle with these terms or more.
__device__ __forceinline__ double beyond(const GridHead &g, double qn, double ca, double s2)
{
    const double t = fmin(fmax(qn * ca, g.rmin), g.rmax);
    return ((qn - t) * (qn - t) + 4.0 * qn * t * s2) * (1.0 - kGuardSlack);
}

// Candidates whose number fits the words of knn_near where they are not staged.
constexpr int kMost = 64;

// The first round, of reach R: the candidates' squared distances in FP32 from
// exact integer differences, the K + 1 least kept as one word each (the
// number of the candidate in the low bits), then FP64 for the K.  False where
// that does not settle it: more than 64 candidates (not staged), a candidate
// beyond the K-th that rounding (2^-17 or 2^-15 in the words, 2^-24 in the
// sum, 2^-29 of rmax in the coordinates) could place before it, or a block
// too small.
// STAGED: the wave's queries lie in one row of an image, in order of
// longitude, so their runs of a band make one run (or two, where it passes
// the band's end, which LDS joins); where those hold at most kStage entries
// together they are read once into LDS, as FP32 differences to the wave's
// first query.  Bound by VALU issue (70% busy: 695 instructions per wave, 14
// per candidate) and the FP64 points' gathers.  8192 x 4096 on d=1000: 971 us
// (1666 with every candidate loaded by its query, 2392 with every candidate
// in FP64); 2048 x 1024 on d=320: 76 (86, 137).
template <int K, int R, bool STAGED>
__device__ __forceinline__ bool knn_near(const GridView &v, const ShellQuery &q, float4 *lds,
                                         double (&bd)[K], int32_t (&bi)[K], int &total)
{
    constexpr int kBands = 2 * R + 1;
    const GridHead &g = *v.g;
    if (!(q.norm <= 2.0 * g.rmax)) return false;   // the differences stay within 31 bits
    const double f = g.fixed;
    const int fx = (int)rint(q.x * f), fy = (int)rint(q.y * f), fz = (int)rint(q.z * f);
    bool circle;
    const float D = window(g.sina[R - 1], q.clat, circle);
    const int own = STAGED ? __builtin_amdgcn_readfirstlane(q.own) : q.own;
    Run run[kBands];
    // Most waves' windows are parts of their bands, with no end in between:
    // then each band's runs are one, from the first query's start to the last's end.
    bool simple = STAGED && !__any(circle);
    if (simple) {
        int c0[kBands], c1[kBands];
        const int32_t *start[kBands];
#pragma unroll
        for (int k = 0; k < kBands; ++k) {
            const int b = own + k - R;
            c0[k] = 0;
            c1[k] = -1;
            start[k] = v.start;
            if (b < 0 || b >= v.bands) continue;
            const int first = v.band[b], n = v.band[b + 1] - first;
            const float per = (float)n * 0.159154943f;
            start[k] += first;
            c0[k] = (int)floorf((q.lon - D) * per);
            c1[k] = (int)floorf((q.lon + D) * per);
            simple = simple && c0[k] >= 0 && c1[k] < n && c1[k] - c0[k] < n - 1;
        }
        simple = __all(simple);
        if (simple) {
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                run[k].ja = start[k][(uint32_t)c0[k]];
                run[k].n = run[k].na = start[k][(uint32_t)(c1[k] + 1)] - run[k].ja;
                run[k].jb = 0;
                total += run[k].n;
            }
        }
    }
    if (!simple) {
#pragma unroll
        for (int k = 0; k < kBands; ++k) {
            run[k] = band_run(v, q, own + k - R, D, circle);
            total += run[k].n;
        }
    }
    // words as floats: positive, never subnormal (the squares start from 1),
    // so a median of three places a word among the best
    float best[K + 1];
#pragma unroll
    for (int m = 0; m <= K; ++m) best[m] = INFINITY;
    uint32_t low = kMost - 1;   // the words' low bits
    auto take = [&](float dx, float dy, float dz, uint32_t number) {
        const float d2 = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, 1.0f)));
        const float w = __uint_as_float((__float_as_uint(d2) & ~low) | (number & low));
#pragma unroll
        for (int m = K; m > 0; --m) best[m] = __builtin_amdgcn_fmed3f(best[m - 1], best[m], w);
        best[0] = __builtin_amdgcn_fmed3f(0.0f, best[0], w);
    };
    // each difference is off by at most 1 per axis, so a distance by 1.74, and
    // by 1 more for the squares' 1
    float slack = 5.0f;
    bool staged = false;
    if (STAGED) {
        const int lane = threadIdx.x & 63;
        // per band: the joined run's first piece (len entries from base), the
        // second's start, its length, and this query's place in it
        int base[kBands], len[kBands], from[kBands], joined[kBands], place[kBands], all = 0;
        if (simple) {
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                base[k] = __builtin_amdgcn_readfirstlane(run[k].ja);
                len[k] = joined[k] = __builtin_amdgcn_readlane(run[k].ja + run[k].n, 63) - base[k];
                from[k] = 0;
                place[k] = run[k].ja - base[k];
                all += joined[k];
            }
            staged = all <= kStage;
        } else {
            bool inside = true;
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                const bool wraps = run[k].n > run[k].na;
                const unsigned long long some = __ballot(wraps);
                base[k] = __builtin_amdgcn_readfirstlane(run[k].ja);
                const int last = __builtin_amdgcn_readlane(
                    wraps ? run[k].jb + run[k].n - run[k].na : run[k].ja + run[k].na, 63);
                if (some) {
                    const int l = __builtin_ctzll(some);
                    from[k] = __builtin_amdgcn_readlane(run[k].jb, l);
                    len[k] = __builtin_amdgcn_readlane(run[k].ja + run[k].na, l) - base[k];
                    joined[k] = len[k] + last - from[k];
                } else {
                    from[k] = last;
                    len[k] = joined[k] = last - base[k];
                }
                all += joined[k];
                const bool second = run[k].ja < base[k];
                place[k] = run[k].ja + (second ? len[k] - from[k] : -base[k]);
                // (not so near the poles, where a window may be a whole band for
                // some of the queries only)
                inside = inside && place[k] >= 0 && place[k] + run[k].n <= joined[k] &&
                         !(second && wraps) && len[k] >= 0 && last <= base[k] + (some ? 0 : len[k]);
            }
            staged = all <= kStage && __all(inside);
        }
        if (staged) {
            const int ox = __builtin_amdgcn_readfirstlane(fx);
            const int oy = __builtin_amdgcn_readfirstlane(fy);
            const int oz = __builtin_amdgcn_readfirstlane(fz);
            const float qx = (float)(fx - ox), qy = (float)(fy - oy), qz = (float)(fz - oz);
            // rounding of the differences to the first query, of either end
            slack += (fabsf(qx) + fabsf(qy) + fabsf(qz)) * 0x1p-21f;
            int at = 0;
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                for (int t = lane; t < joined[k]; t += 64) {
                    const GridEntry p =
                        v.entry[(uint32_t)(simple || t < len[k] ? base[k] + t : from[k] + t - len[k])];
                    lds[at + t] = make_float4((float)(p.x - ox), (float)(p.y - oy),
                                              (float)(p.z - oz), __int_as_float(p.idx));
                }
                run[k].ja = at + place[k];
                at += joined[k];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            low = kStage - 1;   // a candidate's number is its place in LDS
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                int j = run[k].ja;
                const int e = j + run[k].n;
                for (; j < e; ++j) {
                    const float4 p = lds[j];
                    take(qx - p.x, qy - p.y, qz - p.z, (uint32_t)j);
                }
            }
        }
    }
    if (!staged) {
        if (total > kMost) return false;
        uint32_t number = 0;
        auto visit = [&](int j, int e) {
            for (; j < e; ++j, ++number) {
                const GridEntry p = v.entry[j];
                take((float)(fx - p.x), (float)(fy - p.y), (float)(fz - p.z), number);
            }
        };
#pragma unroll
        for (int k = 0; k < kBands; ++k) {
            visit(run[k].ja, run[k].ja + run[k].na);
            if (run[k].n > run[k].na) visit(run[k].jb, run[k].jb + run[k].n - run[k].na);
        }
    }
    if (total > K) {
        // d of the K-th rounded up and of the next rounded down, in units of
        // rmax / 2^29
        const float dk = __builtin_amdgcn_sqrtf(__uint_as_float(__float_as_uint(best[K - 1]) | low));
        const float dn = __builtin_amdgcn_sqrtf(__uint_as_float(__float_as_uint(best[K]) & ~low));
        if (!(dn > dk * (1.0f + 2e-6f) + slack)) return false;
    }
#pragma unroll
    for (int m = 0; m < K; ++m) {
        int i = (int)(__float_as_uint(best[m]) & low), j = i;
        if (!staged) {
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                if (i >= 0 && i < run[k].n) j = run[k].at(i);
                i -= run[k].n;
            }
        }
        bd[m] = INFINITY;
        bi[m] = INT32_MAX;
        if (m < total) {
            bi[m] = staged ? __float_as_int(lds[j].w) : v.entry[j].idx;
            bd[m] = dist2(v.pts + 3 * (int64_t)bi[m], q.x, q.y, q.z);
        }
    }
    // in order but for rounding
#pragma unroll
    for (int e = 1; e < K; ++e)
#pragma unroll
        for (int m = e; m > 0; --m) order(bd[m - 1], bi[m - 1], bd[m], bi[m]);
    if (circle && q.own - R <= 0 && q.own + R >= v.bands - 1) return true;   // all points visited
    return bd[K - 1] <= beyond(g, q.norm, g.cosa[R - 1], g.sin2a[R - 1]);
}

// From this far rounding leaves every point of a shell (norms up to 2^300) at
// one distance, infinite where its square overflows: a coordinate of 2^353 or
// more takes no change from a point's, and the square of a smaller one none
// of the sum.  The nearest are then the first by index.
constexpr double kFar = 0x1p500;

// Rounds in FP64 for queries knn_near does not settle: of reach a0, then of a1
// and its doubles.  sin a is bounded by a from above and by a - a^3 / 6 from below.
template <int K, int T>
__device__ __forceinline__ void knn_rounds(const GridView &v, const ShellQuery &q, float a0,
                                           float a1, double (&bd)[K], int32_t (&bi)[K])
{
    const GridHead &g = *v.g;
    none_yet<K>(bd, bi);
    if (q.norm != q.norm) return;   // a NaN: no distance to compare
    if (q.norm >= kFar) {
        const int32_t n = v.start[g.nbins];   // the number of points
#pragma unroll
        for (int m = 0; m < K; ++m)
            if (m < n) {
                bd[m] = dist2(v.pts + 3 * m, q.x, q.y, q.z);
                bi[m] = m;
            }
        return;
    }
    const double f = g.fixed;
    for (float a = a0;; a = fmaxf(2.0f * a, a1)) {
        none_yet<K>(bd, bi);
        float most = INFINITY;
        const bool whole = a >= 3.2f;
        bool circle;
        const float D = window(a < 1.5f ? a : 2.0f, q.clat, circle), up = a + 2.0f * kAngleSlack;
        const int lo = whole ? 0 : band_of(q.lat - up, v.bands, g.perband);
        const int hi = whole ? v.bands - 1 : band_of(q.lat + up, v.bands, g.perband);
        const int reach = max(q.own - lo, hi - q.own);
        for (int k = 0; k <= 2 * reach; ++k) {   // q's band, then outwards
            const int b = q.own + ((k & 1) ? -((k + 1) >> 1) : (k >> 1));
            if (b < lo || b > hi) continue;
            const Run run = band_run(v, q, b, D, circle);
#pragma unroll 1
            for (int part = 0; part < 2; ++part) {
                const int j = part ? run.jb : run.ja, n = part ? run.n - run.na : run.na;
                scan<K, T, true, false>(v, j, j + n, q.x, q.y, q.z, f, most, bd, bi);
            }
        }
        if (whole || (circle && lo == 0 && hi == v.bands - 1)) return;   // all points visited
        const float x = 0.5f * (a - 2.0f * kAngleSlack), s = fmaxf(x * (1.0f - x * x / 6.0f), 0.0f);
        const double s2 = (double)s * s * (1.0 - kGuardSlack);
        if (bd[K - 1] <= beyond(g, q.norm, 1.0 - 2.0 * s2, s2)) return;
    }
}

template <int K, int T, bool STAGED>
__device__ __forceinline__ void knn_shell(const GridView &v, const ShellQuery &q, float4 *lds,
                                          double (&bd)[K], int32_t (&bi)[K])
{
    constexpr int R = K <= 3 ? 1 : 2;
    int total = 0;
    if (knn_near<K, R, STAGED>(v, q, lds, bd, bi, total)) return;
    // where the window holds more than kMost points, the first round's takes about
    // that many at their density (400,000 points, half of them in a cap of 1 degree,
    // 2,000 queries: 6.1 ms, 92 where every round took the whole window)
    const float a1 = (float)R * (3.14159265f / (float)v.bands);
    const float a0 = a1 * __builtin_amdgcn_sqrtf((float)kMost / (float)max(total, kMost));
    knn_rounds<K, T>(v, q, fmaxf(a0, 16.0f * kAngleSlack), a1, bd, bi);
}

__device__ __forceinline__ ShellQuery shell_query(const GridView &v, double x, double y, double z)
{
    ShellQuery q{x, y, z, sqrt(x * x + y * y + z * z), 0.0f, 0.0f, 0.0f, 0};
    angles_of(x, y, z, v.g->unit, q.lat, q.lon, q.clat);
    q.own = band_of(q.lat, v.bands, v.g->perband);
    return q;
}

// LDS of a query block: the staged entries of its four waves, then its results.
template <int K>
union KnnLds {
    float4 entry[4][kStage];
    struct {
        double d[256 * K];
        int32_t i[256 * K];
    } out;
};

// Results of a block's `count` (up to 256) consecutive queries from p0 on,
// through LDS so that the stores are contiguous (K doubles per query are not).
template <int K>
__device__ __forceinline__ void knn_store(KnnLds<K> &lds, int64_t p0, int count,
                                          const double (&bd)[K], const int32_t (&bi)[K], int64_t V,
                                          double *dists, int64_t *nbrs)
{
    double *sd = lds.out.d;
    int32_t *si = lds.out.i;
    const int t = threadIdx.x;
    __syncthreads();   // every wave is done with its entries
#pragma unroll
    for (int j = 0; j < K; ++j) {
        sd[t * K + j] = sqrt(bd[j]);  // +inf where fewer than K points exist
        si[t * K + j] = bi[j];
    }
    __syncthreads();
    dists += p0 * K;
    nbrs += p0 * K;
    const int m = count * K;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int e = j * 256 + t;
        if (e < m) {
            dists[e] = sd[e];
            nbrs[e] = si[e] == INT32_MAX ? V : si[e];
        }
    }
}

}  // namespace

template <int K>
__global__ __launch_bounds__(256) void k_knn_points(GridView v, int64_t V,
                                                    const double *__restrict__ q, int64_t nq,
                                                    double *__restrict__ dists,
                                                    int64_t *__restrict__ nbrs)
{
    const int64_t p0 = (int64_t)blockIdx.x * 256, p = min(p0 + threadIdx.x, nq - 1);
    __shared__ KnnLds<K> lds;
    double bd[K];
    int32_t bi[K];
    const double x = q[3 * p], y = q[3 * p + 1], z = q[3 * p + 2];
    if (v.g->shell)
        knn_shell<K, kPointScan, false>(v, shell_query(v, x, y, z), nullptr, bd, bi);
    else
        knn_cells<K, kPointScan>(v, x, y, z, bd, bi);
    knn_store<K>(lds, p0, (int)min((int64_t)256, nq - p0), bd, bi, V, dists, nbrs);
}

// trig: cos(lat_h), sin(lat_h) for each row, then cos(lon_w), sin(lon_w) for
// each column, computed on the host with the C library the reference's
// numba code calls; x = (r * cos lat) * cos lon, y = (r * cos lat) * sin lon,
// z = r * sin lat as util.py:86-88.
// ROWS: a block's pixels lie in one row, and stripes of 1 << stripe rows go to
// the XCDs in turn (blockIdx.x is the XCD: consecutive blocks go round them),
// so that an XCD's L2 reads the points of its stripes once: 8192 x 4096 on
// d=1000 947 us in stripes of 16, 982 row by row.  Otherwise blocks take 256
// pixels across rows.
template <int K, bool ROWS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(K <= 3 ? 7 : 4))) void
k_knn_pixels(GridView v, int64_t V, int64_t width, int64_t height, double radius, int stripe,
             float dlat, float dlon, const double *__restrict__ trig, double *__restrict__ dists,
             int64_t *__restrict__ nbrs)
{
    int64_t p0, h, w;
    int count;
    if (ROWS) {
        const int z = blockIdx.z, row = z & ((1 << stripe) - 1);
        h = ((((z >> stripe) << 3) + (int)blockIdx.x) << stripe) + row;
        if (h >= height) return;
        const int w0 = blockIdx.y * 256;
        count = min(256, (int)width - w0);
        w = w0 + min((int)threadIdx.x, count - 1);
        p0 = h * width + w0;
    } else {
        const int64_t n = width * height;
        p0 = (int64_t)blockIdx.x * 256;
        count = (int)min((int64_t)256, n - p0);
        const int64_t p = p0 + min((int)threadIdx.x, count - 1);
        h = p / width;
        w = p - h * width;
    }
    const double clat = trig[2 * h], slat = trig[2 * h + 1];
    const double clon = trig[2 * height + 2 * w], slon = trig[2 * height + 2 * w + 1];
    const double x = radius * clat * clon, y = radius * clat * slon, z = radius * slat;
    __shared__ KnnLds<K> lds;
    double bd[K];
    int32_t bi[K];
    if (!v.g->shell) {
        knn_cells<K, pixel_scan(K)>(v, x, y, z, bd, bi);
    } else if (radius > 0.0) {
        // the angles are the pixel's own
        ShellQuery q{x, y, z, radius, 0.0f, 0.0f, (float)clat, 0};
        q.lat = 3.14159265f - (float)(int)h * dlat;
        q.lon = (float)(int)w * dlon;
        q.own = band_of(q.lat, v.bands, v.g->perband);
        knn_shell<K, pixel_scan(K), ROWS>(v, q, lds.entry[threadIdx.x >> 6], bd, bi);
    } else {
        knn_shell<K, pixel_scan(K), false>(v, shell_query(v, x, y, z), nullptr, bd, bi);
    }
    knn_store<K>(lds, p0, count, bd, bi, V, dists, nbrs);
}

__global__ __launch_bounds__(256) void k_ll_arr(int64_t width, int64_t height, double radius,
                                                const double *__restrict__ trig,
                                                double *__restrict__ out)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= width * height) return;
    const int64_t h = p / width, w = p - h * width;
    const double clat = trig[2 * h], slat = trig[2 * h + 1];
    const double clon = trig[2 * height + 2 * w], slon = trig[2 * height + 2 * w + 1];
    out[3 * p] = radius * clat * clon;
    out[3 * p + 1] = radius * clat * slon;
    out[3 * p + 2] = radius * slat;
}

// util.py:356-364 over K neighbours: sd = sum(d); w_i = 1 / ((d_i + 0.00001)
// / sd); t = sum(w); value = int(sum(colors[n_i] * (w_i / t))), each sum
// accumulated from 0 in neighbour order; truncation toward zero.
template <int K>
__device__ __forceinline__ int32_t gray_value(const double (&d)[K], const int64_t (&n)[K],
                                              const double *__restrict__ colors, int64_t ncolors,
                                              bool &bad)
{
    double c[K], w[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const bool out = n[i] < 0 || n[i] >= ncolors;
        bad = bad || out;
        c[i] = out ? 0.0 : colors[n[i]];
    }
    double sd = 0.0, t = 0.0, v = 0.0;
#pragma unroll
    for (int i = 0; i < K; ++i) sd += d[i];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        w[i] = 1.0 / ((d[i] + 0.00001) / sd);
        t += w[i];
    }
#pragma unroll
    for (int i = 0; i < K; ++i)
        if (n[i] >= 0 && n[i] < ncolors) v += c[i] * (w[i] / t);
    return (int32_t)(int64_t)v;
}

// A block's 256 K distances and indices come through LDS, so that the loads
// are contiguous (K doubles per pixel are not).  Bound by reading 16 K bytes
// per pixel: 8192 x 4096, K = 3: 409 us, 500 with a pixel's own loads.
template <int K>
__global__ __launch_bounds__(256) void k_gray(int64_t npix, const double *__restrict__ dists,
                                              const int64_t *__restrict__ nbrs,
                                              const double *__restrict__ colors, int64_t ncolors,
                                              int32_t *__restrict__ out, int *__restrict__ err)
{
    __shared__ double sd[256 * K];
    __shared__ int64_t sn[256 * K];
    const int t = threadIdx.x;
    const int64_t p0 = (int64_t)blockIdx.x * 256;
    const int count = (int)min((int64_t)256, npix - p0), m = count * K;
    double a[K];
    int64_t b[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int e = min(i * 256 + t, m - 1);
        b[i] = __builtin_nontemporal_load(&nbrs[p0 * K + e]);
        a[i] = __builtin_nontemporal_load(&dists[p0 * K + e]);
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
        sn[i * 256 + t] = b[i];
        sd[i * 256 + t] = a[i];
    }
    __syncthreads();
    if (t >= count) return;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        b[i] = sn[t * K + i];
        a[i] = sd[t * K + i];
    }
    bool bad = false;
    out[p0 + t] = gray_value<K>(a, b, colors, ncolors, bad);
    if (bad) __hip_atomic_fetch_or(err, NX_ERR_INDEX_BIT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int K>
static void launch_gray(int64_t npix, const double *dists, const int64_t *nbrs,
                        const double *colors, int64_t ncolors, int32_t *out, int *err,
                        hipStream_t stream)
{
    hipLaunchKernelGGL(k_gray<K>, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, stream, npix,
                       dists, nbrs, colors, ncolors, out, err);
}

size_t knn_grid_bytes(int64_t V)
{
    if (V <= 0 || V >= INT32_MAX) return 256;
    return grid_layout(V).total;
}

int knn_grid_build(nx_ctx *ctx, const double *pts, int64_t V, void *grid, hipStream_t stream)
{
    if (!ctx || !pts || !grid || V <= 0 || V >= INT32_MAX)
        return set_error(NX_EINVAL, "grid build needs points, a workspace and 0 < V < 2^31 - 1");
    if (((uintptr_t)grid & 255) != 0) return set_error(NX_EINVAL, "grid workspace must be 256-byte aligned");
    NX_HIP(hipSetDevice(ctx->device));
    const GridLayout L = grid_layout(V);
    char *w = (char *)grid;
    auto *g = (GridHead *)(w + L.head);
    auto *band = (int32_t *)(w + L.band);
    auto *start = (int32_t *)(w + L.start);
    auto *bin = (uint32_t *)(w + L.bin);
    auto *rank = (int32_t *)(w + L.rank);
    auto *part = (unsigned long long *)(w + L.part);
    auto *sums = (int32_t *)(w + L.part);   // the box records are read by then
    const unsigned blocks = (unsigned)((V + 255) / 256), by8 = (blocks + 7) / 8 * 8;
    const int parts = (int)std::min<int64_t>((V + 1023) / 1024, kBoxBlocks);
    hipLaunchKernelGGL(k_grid_box, dim3(parts), dim3(1024), 0, stream, pts, V, part);
    hipLaunchKernelGGL(k_grid_setup, dim3(1), dim3(1024), 0, stream, g, V,
                       (const unsigned long long *)part, parts, L.bands, L.tsize, band);
    hipLaunchKernelGGL(k_grid_clear, dim3(std::min<unsigned>(blocks, 2048u)), dim3(256), 0, stream,
                       (const GridHead *)g, start);
    hipLaunchKernelGGL(k_grid_count, dim3(blocks), dim3(256), 0, stream, pts, V,
                       (const GridHead *)g, (const int32_t *)band, L.bands, start, bin, rank);
    const unsigned scan = std::min<unsigned>(blocks, kScanBlocks);
    hipLaunchKernelGGL(k_grid_sums, dim3(scan), dim3(256), 0, stream, (const GridHead *)g,
                       (const int32_t *)start, sums);
    hipLaunchKernelGGL(k_grid_starts, dim3(scan), dim3(256), 0, stream, (const GridHead *)g, V,
                       (const int32_t *)sums, start);
    hipLaunchKernelGGL(k_grid_place, dim3(by8), dim3(256), 0, stream, pts, V,
                       (const GridHead *)g, (const int32_t *)start, (const uint32_t *)bin,
                       (const int32_t *)rank, (GridEntry *)(w + L.entry),
                       (double *)(w + L.pts));
    NX_HIP(hipGetLastError());
    return NX_OK;
}

static GridView grid_view(const void *grid, int64_t V)
{
    const GridLayout L = grid_layout(V);
    const char *w = (const char *)grid;
    return GridView{(const GridHead *)(w + L.head), (const int32_t *)(w + L.band),
                    (const int32_t *)(w + L.start), (const GridEntry *)(w + L.entry),
                    (const double *)(w + L.pts), L.bands};
}

template <int K>
static void launch_points(const GridView &v, int64_t V, const double *q, int64_t nq,
                          double *dists, int64_t *nbrs, hipStream_t stream)
{
    hipLaunchKernelGGL(k_knn_points<K>, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, stream,
                       v, V, q, nq, dists, nbrs);
}

template <int K>
static void launch_pixels(const GridView &v, int64_t V, int64_t width, int64_t height,
                          double radius, const double *trig, double *dists, int64_t *nbrs,
                          hipStream_t stream)
{
    const float dlat = 3.14159265f / (float)(height - 1), dlon = 6.28318531f / (float)width;
    if (width >= 256 && width <= (1 << 23) && height <= (1 << 18)) {
        int stripe = 4;
        while (stripe > 0 && (64 << stripe) > height) --stripe;   // 8 stripes or more to an XCD
        const int64_t groups = (height + (8 << stripe) - 1) >> (3 + stripe);
        hipLaunchKernelGGL((k_knn_pixels<K, true>),
                           dim3(8, (unsigned)((width + 255) / 256), (unsigned)(groups << stripe)),
                           dim3(256), 0, stream, v, V, width, height, radius, stripe, dlat, dlon,
                           trig, dists, nbrs);
        return;
    }
    hipLaunchKernelGGL((k_knn_pixels<K, false>), dim3((unsigned)((width * height + 255) / 256)),
                       dim3(256), 0, stream, v, V, width, height, radius, 0, dlat, dlon,
                       trig, dists, nbrs);
}

#define NX_K_DISPATCH(FN, ...)                  \
    switch (k) {                                \
    case 1: FN<1>(__VA_ARGS__); break;          \
    case 2: FN<2>(__VA_ARGS__); break;          \
    case 3: FN<3>(__VA_ARGS__); break;          \
    case 4: FN<4>(__VA_ARGS__); break;          \
    case 5: FN<5>(__VA_ARGS__); break;          \
    case 6: FN<6>(__VA_ARGS__); break;          \
    case 7: FN<7>(__VA_ARGS__); break;          \
    default: FN<8>(__VA_ARGS__); break;         \
    }

int knn_query(nx_ctx *ctx, const void *grid, int64_t V, const double *q, int64_t nq, int k,
              double *dists, int64_t *nbrs, hipStream_t stream)
{
    if (!ctx || !grid || V <= 0 || V >= INT32_MAX || nq < 0 || (nq > 0 && (!q || !dists || !nbrs)))
        return set_error(NX_EINVAL, "query needs a built grid, query points and outputs");
    if (k < 1 || k > kKnnMax) return set_error(NX_EINVAL, "k=%d outside 1..%d", k, kKnnMax);
    if (nq == 0) return NX_OK;
    if (nq > (int64_t)UINT32_MAX * 256) return set_error(NX_EINVAL, "too many query points");
    NX_HIP(hipSetDevice(ctx->device));
    NX_K_DISPATCH(launch_points, grid_view(grid, V), V, q, nq, dists, nbrs, stream);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

size_t pixel_workspace_bytes(int64_t width, int64_t height)
{
    return width > 0 && height > 0 ? a256(16 * (size_t)(width + height)) : 256;
}

// cos/sin of each row's latitude and each column's longitude in radians, as
// util.py:300-309 computes lat, lon and latlon2xyz its arguments.  One
// sincos per angle: compilers pair a sin and a cos of the same operand into
// the C library's sincos (LLVM for numba's intrinsics, GCC for C), and
// glibc's sincos differs from separate sin and cos in the last bit for a
// few arguments.
static int stage_trig(nx_ctx *ctx, int64_t width, int64_t height, void *ws, hipStream_t stream)
{
    const size_t bytes = 16 * (size_t)(width + height);
    int slot = 0;
    double *t = (double *)stage_begin(ctx, bytes, &slot);
    if (!t) return set_error(NX_ENOMEM, "pinned staging buffer allocation failed");
    const double latpercent = 180.0 / (double)(height - 1);
    const double lonpercent = 360.0 / (double)width;
    const double d2r = 3.141592653589793 / 180.0;  // np.pi / 180
    for (int64_t h = 0; h < height; ++h) {
        double lat = 90.0 - ((double)h * latpercent);
        if (lat < -90.0) lat = -90.0;
        sincos(lat * d2r, &t[2 * h + 1], &t[2 * h]);
    }
    for (int64_t w = 0; w < width; ++w) {
        double lon = -180.0 + ((double)w * lonpercent);
        if (lon < -180.0) lon = -180.0;
        sincos(lon * d2r, &t[2 * height + 2 * w + 1], &t[2 * height + 2 * w]);
    }
    return stage_commit(ctx, slot, ws, bytes, stream);
}

static int pixel_check(nx_ctx *ctx, int64_t width, int64_t height, const void *ws)
{
    if (!ctx || !ws) return set_error(NX_EINVAL, "pixel grid needs a context and a workspace");
    if (width < 1 || height < 2 || width > (1 << 24) || height > (1 << 24) ||
        width * height > (int64_t)UINT32_MAX * 256)
        return set_error(NX_EINVAL, "image %lld x %lld outside 1..2^24 x 2..2^24",
                         (long long)width, (long long)height);
    return NX_OK;
}

int knn_query_pixels(nx_ctx *ctx, const void *grid, int64_t V, int64_t width, int64_t height,
                     double radius, int k, double *dists, int64_t *nbrs, void *ws,
                     hipStream_t stream)
{
    int rc = pixel_check(ctx, width, height, ws);
    if (rc) return rc;
    if (!grid || V <= 0 || V >= INT32_MAX || !dists || !nbrs)
        return set_error(NX_EINVAL, "query needs a built grid and outputs");
    if (k < 1 || k > kKnnMax) return set_error(NX_EINVAL, "k=%d outside 1..%d", k, kKnnMax);
    NX_HIP(hipSetDevice(ctx->device));
    if ((rc = stage_trig(ctx, width, height, ws, stream))) return rc;
    NX_K_DISPATCH(launch_pixels, grid_view(grid, V), V, width, height, radius,
                  (const double *)ws, dists, nbrs, stream);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

int make_ll_arr(nx_ctx *ctx, int64_t width, int64_t height, double radius, double *out, void *ws,
                hipStream_t stream)
{
    int rc = pixel_check(ctx, width, height, ws);
    if (rc) return rc;
    if (!out) return set_error(NX_EINVAL, "null output");
    NX_HIP(hipSetDevice(ctx->device));
    if ((rc = stage_trig(ctx, width, height, ws, stream))) return rc;
    const int64_t n = width * height;
    hipLaunchKernelGGL(k_ll_arr, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, width,
                       height, radius, (const double *)ws, out);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

int make_gray_array(nx_ctx *ctx, int64_t npix, int k, const double *dists, const int64_t *nbrs,
                    const double *colors, int64_t ncolors, int32_t *out, hipStream_t stream)
{
    if (!ctx || npix < 0 || (npix > 0 && (!dists || !nbrs || !colors || !out)) || ncolors <= 0)
        return set_error(NX_EINVAL, "gray array needs query results, colors and an output");
    if (k < 1 || k > kKnnMax) return set_error(NX_EINVAL, "k=%d outside 1..%d", k, kKnnMax);
    if (npix == 0) return NX_OK;
    if (npix > (int64_t)UINT32_MAX * 256) return set_error(NX_EINVAL, "too many pixels");
    NX_HIP(hipSetDevice(ctx->device));
    NX_K_DISPATCH(launch_gray, npix, dists, nbrs, colors, ncolors, out, ctx->d_err, stream);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

}  // namespace nx
