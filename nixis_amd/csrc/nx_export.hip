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
};
static_assert(sizeof(GridHead) <= 256, "grid head must fit its 256 bytes");

// A point in bin order; `tag` is the upper half of its cell's hash (cells).
struct alignas(16) GridPoint {
    double x, y, z;
    int32_t idx;
    uint32_t tag;
};

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
    size_t head, band, start, pts, bin, rank, part, total;
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
    L.pts = o;
    o += a256(sizeof(GridPoint) * (size_t)V);
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

__device__ __forceinline__ int band_of(float lat, int bands)
{
    return clamp_cell(lat * ((float)bands * 0.318309886f), bands);
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
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        block_minmax(lo[k], hi[k]);
        if (threadIdx.x == 0) {
            part[8 * blockIdx.x + 2 * k] = lo[k];
            part[8 * blockIdx.x + 2 * k + 1] = hi[k];
        }
        __syncthreads();
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
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        unsigned long long lo = ~0ull, hi = 0ull;
        for (int i = t; i < parts; i += 1024) {
            const unsigned long long a = part[8 * i + 2 * k], b = part[8 * i + 2 * k + 1];
            lo = a < lo ? a : lo;
            hi = b > hi ? b : hi;
        }
        block_minmax(lo, hi);
        if (t == 0) {
            box[2 * k] = dunkey(lo);
            box[2 * k + 1] = dunkey(hi);
        }
        __syncthreads();
    }
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
        for (int r = 1; r <= 2; ++r) {
            const double a = r * h - 2.0 * kAngleSlack;
            g->cosa[r - 1] = cos(a);
            g->sin2a[r - 1] = sin(0.5 * a) * sin(0.5 * a);
        }
        if (!s) g->nbins = (int64_t)tsize;
    }
    __syncthreads();
    if (!shell) return;
    // cells of each band and their running sum
    __shared__ int32_t wsum[16];
    int32_t carry = 0;
    for (int32_t b0 = 0; b0 < bands; b0 += 1024) {
        const int32_t b = b0 + t;
        int32_t n = 0;
        if (b < bands) n = max(1, (int32_t)(2.0 * bands * cos((b + 0.5) * h - 0.5 * pi)));
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

// Each point's bin and its rank among the bin's points.
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
        angles_of(x, y, z, 1.0 / g->rmax, lat, lon, clat);
        const int r = band_of(lat, bands);
        const int n = band[r + 1] - band[r];
        b = (uint32_t)(band[r] + clamp_cell(lon * ((float)n * 0.159154943f), n));
    } else {
        const double c = g->cell;
        const uint64_t m = mix64(cell_key(cell_of(x, g->origin[0], c, g->dims[0]),
                                          cell_of(y, g->origin[1], c, g->dims[1]),
                                          cell_of(z, g->origin[2], c, g->dims[2])));
        b = (uint32_t)(m & (uint64_t)(g->nbins - 1));
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

__global__ __launch_bounds__(256) void k_grid_place(const double *__restrict__ pts, int64_t V,
                                                    const GridHead *__restrict__ g,
                                                    const int32_t *__restrict__ start,
                                                    const uint32_t *__restrict__ bin,
                                                    const int32_t *__restrict__ rank,
                                                    GridPoint *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= V) return;
    GridPoint p;
    p.x = pts[3 * i];
    p.y = pts[3 * i + 1];
    p.z = pts[3 * i + 2];
    p.idx = (int32_t)i;
    p.tag = 0;
    if (!g->shell) {
        const double c = g->cell;
        p.tag = (uint32_t)(mix64(cell_key(cell_of(p.x, g->origin[0], c, g->dims[0]),
                                          cell_of(p.y, g->origin[1], c, g->dims[1]),
                                          cell_of(p.z, g->origin[2], c, g->dims[2]))) >> 32);
    }
    out[(int64_t)start[bin[i]] + rank[i]] = p;
}

namespace {

struct GridView {
    const GridHead *g;
    const int32_t *band;
    const int32_t *start;
    const GridPoint *pts;
    int32_t bands;
};

__device__ __forceinline__ bool before(double s, int32_t i, double t, int32_t j)
{
    return s < t || (s == t && i < j);
}

// Points j0..j1-1 against the K best.  HASHED skips points of other cells
// (another tag) and points already held (another visited cell with this tag).
template <int K, bool HASHED>
__device__ __forceinline__ void scan_points(const GridPoint *__restrict__ pts, int j0, int j1,
                                            uint32_t tag, double qx, double qy, double qz,
                                            double (&bd)[K], int32_t (&bi)[K])
{
    for (int j = j0; j < j1; ++j) {
        const GridPoint p = pts[j];
        if (HASHED && p.tag != tag) continue;
        double s = 0.0, d;
        d = qx - p.x;
        s += d * d;
        d = qy - p.y;
        s += d * d;
        d = qz - p.z;
        s += d * d;
        const int32_t id = p.idx;
        if (!before(s, id, bd[K - 1], bi[K - 1])) continue;
        if (HASHED) {
            bool held = false;
#pragma unroll
            for (int m = 0; m < K; ++m) held = held || bi[m] == id;
            if (held) continue;
        }
        bd[K - 1] = s;
        bi[K - 1] = id;
#pragma unroll
        for (int m = K - 1; m > 0; --m)
            if (before(bd[m], bi[m], bd[m - 1], bi[m - 1])) {
                const double td = bd[m];
                bd[m] = bd[m - 1];
                bd[m - 1] = td;
                const int32_t ti = bi[m];
                bi[m] = bi[m - 1];
                bi[m - 1] = ti;
            }
    }
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

// The K nearest points of q among hashed cells: shells of cells around q's
// cell until the K-th squared distance is within the block's guaranteed
// radius (the distance from q to the nearest face of the block that does not
// lie on the grid's border, less a margin for rounding of the cell bounds).
template <int K>
__device__ __noinline__ void knn_cells(const GridView &v, double qx, double qy, double qz,
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
    for (int r = 0; r <= rmax; ++r) {
        for (int z = cz - r; z <= cz + r; ++z) {
            if (z < 0 || z >= dz) continue;
            for (int y = cy - r; y <= cy + r; ++y) {
                if (y < 0 || y >= dy) continue;
                const bool face = (z == cz - r || z == cz + r || y == cy - r || y == cy + r);
                const int step = (face || r == 0) ? 1 : 2 * r;
                for (int x = cx - r; x <= cx + r; x += step) {
                    if (x < 0 || x >= dx) continue;
                    const uint64_t m = mix64(cell_key(x, y, z));
                    const int32_t *s = v.start + (m & mask);
                    scan_points<K, true>(v.pts, s[0], s[1], (uint32_t)(m >> 32), qx, qy, qz, bd,
                                         bi);
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

// The K nearest points of q among latitude bands.  A round of reach r visits
// the bands within r of q's and, in each, the cells within longitude D of q,
// sin D = sin(r h) / cos(latitude of q) for a band height h (all cells where
// that passes 1, near the poles).  Every point not visited then lies at an
// angle of at least r h from q (its latitude differs by that, or its meridian
// passes q no nearer), and at an angle a and norms in [rmin, rmax] its squared
// distance is at least (|q| - t)^2 + 4 |q| t sin^2(a / 2), t = |q| cos a
// clamped to those norms.
template <int K>
__device__ __forceinline__ void knn_shell(const GridView &v, double qx, double qy, double qz,
                                          double (&bd)[K], int32_t (&bi)[K])
{
    const GridHead &g = *v.g;
    const int bands = v.bands;
    float lat, lon, clat;
    angles_of(qx, qy, qz, 1.0 / g.rmax, lat, lon, clat);
    const double qn = sqrt(qx * qx + qy * qy + qz * qz);
    const int own = band_of(lat, bands);
    const float h = 3.14159265f / (float)bands;
    for (int r = K <= 3 ? 1 : 2;; r *= 2) {
        none_yet<K>(bd, bi);
        if (!(qn < INFINITY)) break;   // no distance to compare
        const float a = (float)r * h;
        const float ratio = a < 1.5f ? sinf(a) / clat : 1.0f;
        const bool circle = !(ratio < 0.99f);
        const float D = circle ? 0.0f : asinf(ratio) + 4.0f * kAngleSlack;
        for (int k = 0; k <= 2 * r; ++k) {   // q's band, then outwards
            const int b = own + ((k & 1) ? -((k + 1) >> 1) : (k >> 1));
            if (b < 0 || b >= bands) continue;
            const int base = v.band[b], n = v.band[b + 1] - base;
            const int32_t *start = v.start + base;
            const float per = (float)n * 0.159154943f;
            int c0 = (int)floorf((lon - D) * per), c1 = (int)floorf((lon + D) * per);
            if (circle || c1 - c0 >= n - 1) {
                c0 = 0;
                c1 = n - 1;
            }
            // cells beyond either end of the band continue at the other end
            if (c0 < 0) {
                scan_points<K, false>(v.pts, start[c0 + n], start[n], 0, qx, qy, qz, bd, bi);
                c0 = 0;
            }
            if (c1 >= n) {
                scan_points<K, false>(v.pts, start[0], start[c1 - n + 1], 0, qx, qy, qz, bd, bi);
                c1 = n - 1;
            }
            scan_points<K, false>(v.pts, start[c0], start[c1 + 1], 0, qx, qy, qz, bd, bi);
        }
        if (circle && own - r <= 0 && own + r >= bands - 1) break;   // every point visited
        double ca, s2;
        if (r <= 2) {
            ca = g.cosa[r - 1];
            s2 = g.sin2a[r - 1];
        } else {
            const double ad = r * (3.141592653589793 / bands) - 2.0 * kAngleSlack;
            if (ad >= 3.141592653589793) continue;   // more bands than the sphere has
            ca = cos(ad);
            s2 = sin(0.5 * ad) * sin(0.5 * ad);
        }
        const double t = fmin(fmax(qn * ca, g.rmin), g.rmax);
        const double least = (qn - t) * (qn - t) + 4.0 * qn * t * s2;
        if (bd[K - 1] <= least * (1.0 - kGuardSlack)) break;
    }
}

template <int K>
__device__ __forceinline__ void knn_point(const GridView &v, double qx, double qy, double qz,
                                          double (&bd)[K], int32_t (&bi)[K])
{
    if (v.g->shell)
        knn_shell<K>(v, qx, qy, qz, bd, bi);
    else
        knn_cells<K>(v, qx, qy, qz, bd, bi);
}

// Results of a block's 256 consecutive queries p0..p0+255 (of n), through
// LDS so that the stores are contiguous (K doubles per query are not).
template <int K>
__device__ __forceinline__ void knn_store(int64_t p0, int64_t n, const double (&bd)[K],
                                          const int32_t (&bi)[K], int64_t V, double *dists,
                                          int64_t *nbrs)
{
    __shared__ double sd[256 * K];
    __shared__ int32_t si[256 * K];
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        sd[t * K + j] = sqrt(bd[j]);  // +inf where fewer than K points exist
        si[t * K + j] = bi[j];
    }
    __syncthreads();
    const int m = (int)min((int64_t)256, n - p0) * K;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int e = j * 256 + t;
        if (e < m) {
            dists[p0 * K + e] = sd[e];
            nbrs[p0 * K + e] = si[e] == INT32_MAX ? V : si[e];
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
    double bd[K];
    int32_t bi[K];
    knn_point<K>(v, q[3 * p], q[3 * p + 1], q[3 * p + 2], bd, bi);
    knn_store<K>(p0, nq, bd, bi, V, dists, nbrs);
}

// trig: cos(lat_h), sin(lat_h) for each row, then cos(lon_w), sin(lon_w) for
// each column, computed on the host with the C library the reference's
// numba code calls; x = (r * cos lat) * cos lon, y = (r * cos lat) * sin lon,
// z = r * sin lat as util.py:86-88.
template <int K>
__global__ __launch_bounds__(256) void k_knn_pixels(GridView v, int64_t V, int64_t width,
                                                    int64_t height, double radius,
                                                    const double *__restrict__ trig,
                                                    double *__restrict__ dists,
                                                    int64_t *__restrict__ nbrs)
{
    const int64_t n = width * height;
    const int64_t p0 = (int64_t)blockIdx.x * 256, p = min(p0 + threadIdx.x, n - 1);
    const int64_t h = p / width, w = p - h * width;
    const double clat = trig[2 * h], slat = trig[2 * h + 1];
    const double clon = trig[2 * height + 2 * w], slon = trig[2 * height + 2 * w + 1];
    double bd[K];
    int32_t bi[K];
    knn_point<K>(v, radius * clat * clon, radius * clat * slon, radius * slat, bd, bi);
    knn_store<K>(p0, n, bd, bi, V, dists, nbrs);
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

// util.py:356-364 over k neighbours: sd = sum(d); w_i = 1 / ((d_i + 0.00001)
// / sd); t = sum(w); value = int(sum(colors[n_i] * (w_i / t))), each sum
// accumulated from 0 in neighbour order; truncation toward zero.
__global__ __launch_bounds__(256) void k_gray(int64_t npix, int k, const double *__restrict__ dists,
                                              const int64_t *__restrict__ nbrs,
                                              const double *__restrict__ colors, int64_t ncolors,
                                              int32_t *__restrict__ out, int *__restrict__ err)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    double d[kKnnMax], ws[kKnnMax];
    double sd = 0.0;
    for (int i = 0; i < k; ++i) {
        d[i] = dists[p * k + i];
        sd += d[i];
    }
    double t = 0.0;
    for (int i = 0; i < k; ++i) {
        ws[i] = 1.0 / ((d[i] + 0.00001) / sd);
        t += ws[i];
    }
    double v = 0.0;
    bool bad = false;
    for (int i = 0; i < k; ++i) {
        const int64_t n = nbrs[p * k + i];
        if (n < 0 || n >= ncolors) {
            bad = true;
            continue;
        }
        v += colors[n] * (ws[i] / t);
    }
    out[p] = (int32_t)(int64_t)v;
    if (bad) __hip_atomic_fetch_or(err, NX_ERR_INDEX_BIT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
    const unsigned blocks = (unsigned)((V + 255) / 256);
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
    hipLaunchKernelGGL(k_grid_place, dim3(blocks), dim3(256), 0, stream, pts, V,
                       (const GridHead *)g, (const int32_t *)start, (const uint32_t *)bin,
                       (const int32_t *)rank, (GridPoint *)(w + L.pts));
    NX_HIP(hipGetLastError());
    return NX_OK;
}

static GridView grid_view(const void *grid, int64_t V)
{
    const GridLayout L = grid_layout(V);
    const char *w = (const char *)grid;
    return GridView{(const GridHead *)(w + L.head), (const int32_t *)(w + L.band),
                    (const int32_t *)(w + L.start), (const GridPoint *)(w + L.pts), L.bands};
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
    const int64_t n = width * height;
    hipLaunchKernelGGL(k_knn_pixels<K>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       v, V, width, height, radius, trig, dists, nbrs);
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
    hipLaunchKernelGGL(k_gray, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, stream, npix, k,
                       dists, nbrs, colors, ncolors, out, ctx->d_err);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

}  // namespace nx
