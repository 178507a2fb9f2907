// nx_climate.hip -- insolation at the top of the atmosphere on the device
// (climate.py:193-201, 416-590).
//
// Per vertex and rotation step: rotate about z, tilt about y, convert to
// latitude / longitude (util.py:60-76) and add max(cos|lat|, 0) *
// max(cos lon, 0) to a float32 accumulator the way numba adds a double to a
// float32 array element (sum in double, round to float).  The sines and
// cosines of the rotation, tilt and seasonal angles are the same for every
// vertex; they are computed on the host with the C library the reference's
// numba code calls (one sincos per angle, as LLVM pairs a sin and a cos of
// one operand) and uploaded as tables.
//
// cos(latitude) * cos(longitude) of a rotated vertex t is, without the
// angles, sqrt(1 - (t.z / r)^2) * t.x / sqrt(t.x^2 + t.y^2); on the sphere of
// radius r the two roots cancel and it is t.x / |r|, the sun's direction
// component.  k_insolation, k_slice and k_year_slice use the second form for
// vertices on the sphere to within rounding, the first (insol_vector) elsewhere
// and at angles that are not finite, and the angles themselves (insol_value)
// only where the first form's quotients could overflow or a value is not finite.  The kernels are bound by FP64 issue:
// six FP64 instructions per vertex and step on the sphere.
#include <hip/hip_runtime.h>

#include <cmath>

#include "nx_ctx.h"

namespace nx {

namespace {

constexpr int kMaxSteps = 360;  // rotation steps per call (a day of 1-degree steps)
constexpr int kDays = 360;      // climate.py:581
constexpr int kSlice = 181;     // latitudes -90..90, index = lat mod 181

struct ClimateLayout {
    size_t rot, tilt, sverts, table, total;
};

constexpr size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

constexpr ClimateLayout climate_layout()
{
    ClimateLayout L{};
    size_t o = 0;
    L.rot = o;
    o += a256(16 * kMaxSteps);       // cos, sin per rotation step
    L.tilt = o;
    o += a256(16 * kDays);           // cos, sin per day's tilt
    L.sverts = o;
    o += a256(24 * kSlice);          // the slice's vertices
    L.table = o;
    o += a256(8 * kSlice);           // a day's table (float) or the year's (double)
    L.total = o;
    return L;
}

__device__ __forceinline__ double py_max(double a, double b) { return b > a ? b : a; }
__device__ __forceinline__ double py_min(double a, double b) { return b < a ? b : a; }

// util.py:60-76: degrees(v) = v * (180 / pi).
__device__ __forceinline__ double lat_of(double z, double r)
{
    return asin(py_min(py_max(z / r, -1.0), 1.0)) * (180.0 / 3.141592653589793);
}

// climate.py:421-440 and 444 for one rotation step.
__device__ __forceinline__ double insol_value(double x, double y, double z, double r, double cr,
                                              double sr, double ct, double st)
{
    const double pi = 3.141592653589793;
    const double rx = x * cr - y * sr;
    const double ry = x * sr + y * cr;
    const double rz = z;
    const double tx = rx * ct + rz * st;
    const double ty = ry;
    const double tz = rz * ct - rx * st;
    const double lat = lat_of(tz, r);
    const double lon = atan2(ty, tx) * (180.0 / 3.141592653589793);
    return py_max(cos(fabs(lat) * pi / 180), 0.0) * py_max(cos(lon * pi / 180), 0.0);
}

// Largest |(|v|^2 - r^2)| / r^2 of a vertex taken to lie on the sphere: 16
// units of FP64 rounding, above what normalising and scaling a vertex leave
// (a few units).  The first form's own rounding, 1 unit of q near |q| = 1,
// moves its value as much as this does.
constexpr double kOnSphere = 0x1p-48;

// insol_value without the angles, for finite radii whose square is finite.
__device__ __forceinline__ double insol_vector(double x, double y, double z, double r, double cr,
                                               double sr, double ct, double st)
{
    const double rx = x * cr - y * sr, ty = x * sr + y * cr;
    const double tx = rx * ct + z * st, tz = z * ct - rx * st;
    const double n2 = tx * tx + ty * ty;
    if (!(n2 >= 0x1p-900 && n2 <= 0x1p900)) return insol_value(x, y, z, r, cr, sr, ct, st);
    if (!(tx > 0.0)) return 0.0;
    const double q = py_min(py_max(tz / r, -1.0), 1.0);
    return tx * sqrt((1.0 - q) * (1.0 + q) / n2);
}

// nsteps rotations of one vertex added to acc, each step as numba adds a
// double to a float32 element.  finite: every angle's cosine and sine are (the
// maximum below takes a NaN for 0).  Day of 360 steps at d=320 (1,024,002
// vertices): 3215 us a call with the angles, 97 us this way, every float equal.
__device__ __forceinline__ float insol_sum(double x, double y, double z, double r,
                                           const double *__restrict__ rot, int nsteps, double ct,
                                           double st, bool finite, float acc)
{
    const double r2 = r * r, v2 = x * x + y * y + z * z;
    const bool r_ok = r2 >= 0x1p-900 && r2 <= 0x1p900;
    if (finite && r_ok && fabs(v2 - r2) <= kOnSphere * r2) {
        const double d = fabs(r);   // the longitude does not depend on the radius's sign
        const double xs = x * ct / d, ys = -y * ct / d, zs = z * st / d;
#pragma unroll 4
        for (int s = 0; s < nsteps; ++s) {
            const double t = fma(xs, rot[2 * s], fma(ys, rot[2 * s + 1], zs));
            acc = (float)((double)acc + fmax(t, 0.0));
        }
    } else if (r_ok) {
        for (int s = 0; s < nsteps; ++s)
            acc = (float)((double)acc +
                          insol_vector(x, y, z, r, rot[2 * s], rot[2 * s + 1], ct, st));
    } else {
        for (int s = 0; s < nsteps; ++s)
            acc = (float)((double)acc +
                          insol_value(x, y, z, r, rot[2 * s], rot[2 * s + 1], ct, st));
    }
    return acc;
}

// climate.py:351-412 (assign_surface_temp).  The reference's altitude weight
// is 0 (climate.py:373-374), so h2 = rescale(altitudes, 0, 0) is 0 at every
// vertex and every vertex takes the else branch (climate.py:408):
// max(cos(|lat - tilt| * pi / 180), 0), stored as float32.
__global__ __launch_bounds__(256) void k_surface_temp(const double *__restrict__ verts,
                                                      int64_t V, double r, double tilt,
                                                      float *__restrict__ out)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const double pi = 3.141592653589793;
    const double dist = lat_of(verts[3 * v + 2], r) - tilt;
    out[v] = (float)py_max(cos(fabs(dist) * pi / 180), 0.0);
}

}  // namespace

// nsteps rotations of each vertex, accumulated into arr (float32).
__global__ __launch_bounds__(256) void k_insolation(const double *__restrict__ verts, int64_t V,
                                                    double radius, const double *__restrict__ rot,
                                                    int nsteps, double ct, double st, int finite,
                                                    float *__restrict__ arr)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    arr[v] = insol_sum(verts[3 * v], verts[3 * v + 1], verts[3 * v + 2], radius, rot, nsteps, ct,
                       st, finite != 0, arr[v]);
}

// climate.py:503-533 for one tilt: table[k] over the 181 slice vertices, 360
// rotation steps each.
__global__ __launch_bounds__(64) void k_slice(const double *__restrict__ sverts, double radius,
                                              const double *__restrict__ rot, int nsteps,
                                              double ct, double st, float *__restrict__ table)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= kSlice) return;
    table[k] = insol_sum(sverts[3 * k], sverts[3 * k + 1], sverts[3 * k + 2], radius, rot, nsteps,
                         ct, st, ct == ct, 0.0f);
}

// The year's table: a block per slice vertex, a thread per day (the daily
// values of k_slice with that day's tilt), summed over the days in FP64 in a
// fixed order.
constexpr int kYearThreads = 384;
__global__ __launch_bounds__(kYearThreads) void k_year_slice(const double *__restrict__ sverts,
                                                            double radius,
                                                            const double *__restrict__ rot,
                                                            int nsteps,
                                                            const double *__restrict__ tilt,
                                                            double *__restrict__ year)
{
    const int k = blockIdx.x, d = threadIdx.x;
    double sum = 0.0;
    if (d < kDays)
        sum = (double)insol_sum(sverts[3 * k], sverts[3 * k + 1], sverts[3 * k + 2], radius, rot,
                                nsteps, tilt[2 * d], tilt[2 * d + 1], tilt[2 * d] == tilt[2 * d], 0.0f);
    __shared__ double part[kYearThreads / 64];
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if ((d & 63) == 0) part[d >> 6] = sum;
    __syncthreads();
    if (d == 0) {
        double t = 0.0;
        for (int w = 0; w < kYearThreads / 64; ++w) t += part[w];
        year[k] = t;
    }
}

// climate.py:547-573 with a day's table (float), or the year's (double):
// interpolating each day and adding up (climate.py:581-584) is interpolating
// in the sum of the tables, so the year is one pass over the vertices, bound
// by reading them.  The daily values were added in float32 before; the
// FP64 sum is rounded once (relative error against 64 bits 3.2e-8, 3.1e-7
// before).  A year and the surface temperatures of 10,000,002 vertices: 2815
// us before the vector form and this, 2519 with the first, 146 with both.
template <class T>
__global__ __launch_bounds__(256) void k_interpolate(const double *__restrict__ verts, int64_t V,
                                                     double radius, const T *__restrict__ table,
                                                     float *__restrict__ out)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const double lat = lat_of(verts[3 * v + 2], radius);
    const int64_t lower = (int64_t)floor(lat), upper = (int64_t)ceil(lat);
    const T tl = table[lower < 0 ? kSlice + lower : lower];
    const T tu = table[upper < 0 ? kSlice + upper : upper];
    if (lower == upper) {
        out[v] = (float)tl;
        return;
    }
    const T diff = tu - tl;
    out[v] = (float)((double)tl + (lat - (double)lower) * ((double)diff / (double)(upper - lower)));
}

size_t climate_workspace_bytes() { return climate_layout().total; }

// rot[2s], rot[2s+1] = cos, sin of (rotation * pi) / 180 for s = 0..nsteps-1;
// whether all are finite (not for an infinite angle or a NaN).
static bool fill_rot(double *t, double rot0, double rot_step, int nsteps)
{
    const double pi = 3.141592653589793;
    double rotation = rot0;
    bool finite = true;
    for (int s = 0; s < nsteps; ++s) {
        sincos(rotation * pi / 180, &t[2 * s + 1], &t[2 * s]);
        finite = finite && std::isfinite(t[2 * s]);
        rotation += rot_step;
    }
    return finite;
}

static int climate_check(nx_ctx *ctx, const void *ws)
{
    if (!ctx || !ws) return set_error(NX_EINVAL, "insolation needs a context and a workspace");
    if (((uintptr_t)ws & 255) != 0) return set_error(NX_EINVAL, "workspace must be 256-byte aligned");
    return NX_OK;
}

int sample_insolation(nx_ctx *ctx, const double *verts, int64_t V, double radius, double rot0,
                      double rot_step, int nsteps, double tilt, float *arr, void *ws,
                      hipStream_t stream)
{
    int rc = climate_check(ctx, ws);
    if (rc) return rc;
    if (V < 0 || (V > 0 && (!verts || !arr))) return set_error(NX_EINVAL, "bad vertices / output");
    if (nsteps < 0 || nsteps > kMaxSteps)
        return set_error(NX_EINVAL, "nsteps=%d outside 0..%d", nsteps, kMaxSteps);
    if (V == 0 || nsteps == 0) return NX_OK;
    NX_HIP(hipSetDevice(ctx->device));
    const ClimateLayout L = climate_layout();
    int slot = 0;
    double *t = (double *)stage_begin(ctx, 16 * (size_t)nsteps, &slot);
    if (!t) return set_error(NX_ENOMEM, "pinned staging buffer allocation failed");
    const bool finite = fill_rot(t, rot0, rot_step, nsteps);
    if ((rc = stage_commit(ctx, slot, (char *)ws + L.rot, 16 * (size_t)nsteps, stream))) return rc;
    double st, ct;
    sincos(tilt * 3.141592653589793 / 180, &st, &ct);
    hipLaunchKernelGGL(k_insolation, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, stream, verts,
                       V, radius, (const double *)((char *)ws + L.rot), nsteps, ct, st,
                       finite && std::isfinite(ct) ? 1 : 0, arr);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

// The slice's rotations, tilts and vertices (climate.py:510-528) into the
// workspace's head.
static int stage_slice(nx_ctx *ctx, double radius, const double *tilts, int days, void *ws,
                       hipStream_t stream)
{
    const ClimateLayout L = climate_layout();
    const size_t bytes = L.table;  // rot, tilt and slice vertices
    int slot = 0;
    char *h = stage_begin(ctx, bytes, &slot);
    if (!h) return set_error(NX_ENOMEM, "pinned staging buffer allocation failed");
    fill_rot((double *)(h + L.rot), -180.0, 360.0 / 360, kMaxSteps);
    double *tl = (double *)(h + L.tilt);
    for (int d = 0; d < days; ++d) sincos(tilts[d] * 3.141592653589793 / 180, &tl[2 * d + 1], &tl[2 * d]);
    double *sv = (double *)(h + L.sverts);
    const double d2r = 3.141592653589793 / 180.0;
    for (int i = -90; i <= 90; ++i) {  // latlon2xyz(i, 0, radius), util.py:86-88
        const int k = i < 0 ? kSlice + i : i;
        double s, c;
        sincos((double)i * d2r, &s, &c);
        sv[3 * k] = radius * c * 1.0;
        sv[3 * k + 1] = radius * c * 0.0;
        sv[3 * k + 2] = radius * s;
    }
    return stage_commit(ctx, slot, ws, bytes, stream);
}

// One day's table into `table`.
static int slice(nx_ctx *ctx, double radius, double tilt, float *table, void *ws,
                 hipStream_t stream)
{
    const ClimateLayout L = climate_layout();
    int rc = stage_slice(ctx, radius, &tilt, 1, ws, stream);
    if (rc) return rc;
    double st, ct;
    sincos(tilt * 3.141592653589793 / 180, &st, &ct);
    hipLaunchKernelGGL(k_slice, dim3((kSlice + 63) / 64), dim3(64), 0, stream,
                       (const double *)((char *)ws + L.sverts), radius,
                       (const double *)((char *)ws + L.rot), kMaxSteps, ct, st, table);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

int insolation_slice(nx_ctx *ctx, double radius, double tilt, float *out, void *ws,
                     hipStream_t stream)
{
    int rc = climate_check(ctx, ws);
    if (rc) return rc;
    if (!out) return set_error(NX_EINVAL, "null output");
    NX_HIP(hipSetDevice(ctx->device));
    return slice(ctx, radius, tilt, out, ws, stream);
}

int daily_insolation(nx_ctx *ctx, const double *verts, int64_t V, double radius, double tilt,
                     float *out, void *ws, hipStream_t stream)
{
    int rc = climate_check(ctx, ws);
    if (rc) return rc;
    if (V < 0 || (V > 0 && (!verts || !out))) return set_error(NX_EINVAL, "bad vertices / output");
    NX_HIP(hipSetDevice(ctx->device));
    float *table = (float *)((char *)ws + climate_layout().table);
    if ((rc = slice(ctx, radius, tilt, table, ws, stream))) return rc;
    if (V == 0) return NX_OK;
    hipLaunchKernelGGL(k_interpolate<float>, dim3((unsigned)((V + 255) / 256)), dim3(256), 0,
                       stream, verts, V, radius, (const float *)table, out);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

int interpolate_insolation(nx_ctx *ctx, const double *verts, int64_t V, const float *table,
                           double radius, float *out, hipStream_t stream)
{
    if (!ctx || V < 0 || (V > 0 && (!verts || !table || !out)))
        return set_error(NX_EINVAL, "bad vertices / table / output");
    if (V == 0) return NX_OK;
    NX_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(k_interpolate<float>, dim3((unsigned)((V + 255) / 256)), dim3(256), 0,
                       stream, verts, V, radius, table, out);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

int surface_temp(nx_ctx *ctx, const double *verts, int64_t V, double radius, double tilt,
                 float *out, hipStream_t stream)
{
    if (!ctx) return set_error(NX_EINVAL, "null context");
    if (V < 0 || (V > 0 && (!verts || !out))) return set_error(NX_EINVAL, "bad vertices / output");
    if (V == 0) return NX_OK;
    NX_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(k_surface_temp, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, stream,
                       verts, V, radius, tilt, out);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

int yearly_insolation(nx_ctx *ctx, const double *verts, int64_t V, double radius,
                      double axial_tilt, float *out, void *ws, hipStream_t stream)
{
    int rc = climate_check(ctx, ws);
    if (rc) return rc;
    if (V < 0 || (V > 0 && (!verts || !out))) return set_error(NX_EINVAL, "bad vertices / output");
    NX_HIP(hipSetDevice(ctx->device));
    double tilts[kDays];
    for (int x = 0; x < kDays; ++x)  // climate.py:201
        tilts[x] = std::sin((double)x * 3.141592653589793 / 180) * axial_tilt;
    if ((rc = stage_slice(ctx, radius, tilts, kDays, ws, stream))) return rc;
    const ClimateLayout L = climate_layout();
    double *year = (double *)((char *)ws + L.table);
    hipLaunchKernelGGL(k_year_slice, dim3(kSlice), dim3(kYearThreads), 0, stream,
                       (const double *)((char *)ws + L.sverts), radius,
                       (const double *)((char *)ws + L.rot), kMaxSteps,
                       (const double *)((char *)ws + L.tilt), year);
    if (V > 0)
        hipLaunchKernelGGL(k_interpolate<double>, dim3((unsigned)((V + 255) / 256)), dim3(256), 0,
                           stream, verts, V, radius, (const double *)year, out);
    NX_HIP(hipGetLastError());
    return NX_OK;
}

}  // namespace nx
