// nx_plan_dev.hip -- four-step tile plans on the device.
//
// The plan of nx_tiles.cpp (four steps), byte for byte, from a neighbour
// table that is on the device: the host planner took 85 ms per pass over a
// mesh of 316,842 vertices, and needs the table copied there and the plan
// copied back.  A block makes a tile: its rings are collected in an LDS hash
// set and sorted, the local table, the owners of the edge lengths and the
// labels of their rounds stay in LDS.
//   k_plan_cut     cuts each chunk into tiles that fit (sizes only)
//   k_plan_offsets numbers the tiles and adds up their sections
//   k_plan_owners  rings, slot codes and length columns of each tile
//   k_plan_lengths adds up the length blocks
//   k_plan_write   the image
// A tile takes about 20 synchronous steps to collect and number and 40 to
// settle its owners, so the kernels are bound by barriers and LDS latency, two
// tiles to a CU.  Neighbour tables, order and plan of a new mesh of 316,842
// vertices: 178 ms with the host planner, 0.99 ms so.  A table that is not
// symmetric is left to the host planner.
#include <hip/hip_runtime.h>

#include <cstring>

#include "nx_ctx.h"
#include "nx_pair_dev.h"

namespace nx {

namespace {

constexpr int kSteps = kMultiSteps;
constexpr int kThreads = 1024;
constexpr int kHash = 4096;                 // slots of a tile's ring set
constexpr int kPieces = kQuadStepOne / kTileMin;   // tiles a chunk can be cut into
constexpr int kScanThreads = 1024;
static_assert(kQuadLoadMax + kThreads < kHash, "room for the entries in flight past the limit");

struct TileRec {
    int32_t a;                 // first vertex
    int32_t pref[kSteps + 1];  // tile, tile + ring 1, ..., tile + rings 1..kSteps
};

struct PlanTotals {
    int64_t ntiles, nring, ncs, nlen;
    int32_t max_tile, max_load, max_step1;
    int32_t refused;           // a chunk does not cut, or the table is not symmetric
};

inline size_t a256(size_t x) { return (x + 255) & ~(size_t)255; }

struct PlanScratch {
    size_t totals, count, rec, tile, rbase, cbase, ebase, kt, ring, code, total;
    int64_t chunks;
};

// Tiles hold at least kTileMin vertices, and a plan whose rings hold more
// than kSteps / 2 vertices per owned one is refused.
PlanScratch plan_scratch(int64_t V, int64_t chunk)
{
    PlanScratch L;
    L.chunks = (V + chunk - 1) / chunk;
    const size_t tiles = (size_t)(V / kTileMin + L.chunks);
    const size_t nring = (size_t)(kSteps / 2) * (size_t)V;
    size_t o = 0;
    auto take = [&o](size_t bytes) {
        const size_t at = o;
        o += a256(bytes);
        return at;
    };
    L.totals = take(sizeof(PlanTotals));
    L.count = take(4 * (size_t)L.chunks);
    L.rec = take(sizeof(TileRec) * kPieces * (size_t)L.chunks);
    L.tile = take(sizeof(TileRec) * tiles);
    L.rbase = take(8 * (tiles + 1));
    L.cbase = take(8 * (tiles + 1));
    L.ebase = take(8 * (tiles + 1));
    L.kt = take(4 * tiles);
    L.ring = take(4 * nring);
    L.code = take(2 * 6 * (nring + (size_t)V));
    L.total = o;
    return L;
}

// The rings of one tile: a hash set of the vertices, and the list of them.
struct RingSet {
    int32_t key[kHash];
    int32_t ring[kQuadLoadMax];
    int32_t count;
    int32_t bad;               // a neighbour index outside 0..V-1 was met
    int32_t pref[kSteps + 1];
};

__device__ __forceinline__ uint32_t ring_hash(int32_t n) { return (uint32_t)n * 2654435761u >> 20; }

__device__ __forceinline__ void ring_add(RingSet &S, int32_t n)
{
    // past the limit the tile is refused anyway; the set never fills up
    if (__hip_atomic_load(&S.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > kQuadLoadMax)
        return;
    for (uint32_t h = ring_hash(n);; h = (h + 1) & (kHash - 1)) {
        const int32_t prev = atomicCAS(&S.key[h], -1, n);
        if (prev == n) return;
        if (prev != -1) continue;
        const int32_t i = atomicAdd(&S.count, 1);
        if (i < kQuadLoadMax) S.ring[i] = n;
        return;
    }
}

// Rings 1..kSteps of [a, a + T) into S, each sorted when SORT; false where the
// tile and its rings do not fit.  All threads of the block call it.
template <bool SORT>
__device__ bool tile_rings(RingSet &S, const int32_t *__restrict__ col, int64_t V, int64_t a, int T)
{
    const int t = threadIdx.x;
    for (int i = t; i < kHash; i += kThreads) S.key[i] = -1;
    if (t == 0) {
        S.count = 0;
        S.bad = 0;
        S.pref[0] = T;
    }
    __syncthreads();
    int lo = 0, hi = 0;   // the ring before the one being collected
    for (int m = 0; m < kSteps; ++m) {
        const int n = m == 0 ? T : hi - lo;
        for (int k = 0; k < 6; ++k)
            for (int i = t; i < n; i += kThreads) {
                const int64_t v = m == 0 ? a + i : S.ring[lo + i];
                const int32_t u = col[(int64_t)k * V + v];
                if (u < 0 || u >= V)
                    S.bad = 1;
                else if (u < a || u >= a + T)
                    ring_add(S, u);
            }
        __syncthreads();
        lo = hi;
        hi = S.count;
        const int total = T + hi;
        const bool bad = S.bad != 0;
        __syncthreads();
        if (bad || total > kQuadLoadMax || (m == kSteps - 2 && total > kQuadStepOne)) return false;
        if (t == 0) S.pref[m + 1] = total;
        if (SORT) {   // by rank; the entries of a ring are distinct
            constexpr int kMine = (kQuadLoadMax + kThreads - 1) / kThreads;
            int32_t e[kMine], r[kMine];
#pragma unroll
            for (int q = 0; q < kMine; ++q) {
                r[q] = 0;
                e[q] = lo + t + q * kThreads < hi ? S.ring[lo + t + q * kThreads] : 0;
            }
            const int mine = (hi - lo + kThreads - 1) / kThreads;
            for (int i = lo; i < hi; ++i) {
                const int32_t x = S.ring[i];
#pragma unroll
                for (int q = 0; q < kMine; ++q)
                    if (q < mine) r[q] += x < e[q];
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kMine; ++q)
                if (lo + t + q * kThreads < hi) S.ring[lo + r[q]] = e[q];
        }
        __syncthreads();
    }
    return true;
}

}  // namespace

// Tiles of each chunk: halved until they fit, in order (a stack of the
// pieces still to try).  count[chunk] is -1 where a piece would be cut below
// kTileMin.
__global__ __launch_bounds__(kThreads) void k_plan_cut(const int32_t *__restrict__ col, int64_t V,
                                                       int64_t chunk, TileRec *__restrict__ rec,
                                                       int32_t *__restrict__ count)
{
    __shared__ RingSet S;
    __shared__ int32_t todo[16][2];   // (offset, length), the next piece last
    __shared__ int32_t left, made;
    const int64_t c0 = blockIdx.x * chunk;
    if (threadIdx.x == 0) {
        todo[0][0] = 0;
        todo[0][1] = (int32_t)min(chunk, V - c0);
        left = 1;
        made = 0;
    }
    __syncthreads();
    while (left > 0) {
        const int off = todo[left - 1][0], len = todo[left - 1][1];
        const bool fits = tile_rings<false>(S, col, V, c0 + off, len);
        __syncthreads();
        if (threadIdx.x == 0) {
            --left;
            if (S.bad) {   // refused: the host planner names the error
                made = -1;
                left = 0;
            } else if (fits) {
                TileRec &r = rec[blockIdx.x * (int64_t)kPieces + made++];
                r.a = (int32_t)(c0 + off);
                for (int m = 0; m <= kSteps; ++m) r.pref[m] = S.pref[m];
            } else if (len / 2 < kTileMin) {
                made = -1;
                left = 0;
            } else {
                const int h = len / 2;
                todo[left][0] = off + h;
                todo[left++][1] = len - h;
                todo[left][0] = off;
                todo[left++][1] = h;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) count[blockIdx.x] = made;
}

namespace {

// Exclusive sums of three values over a block's threads, and their totals.
__device__ __forceinline__ void block_sums(int64_t (&x)[3], int64_t (&total)[3])
{
    __shared__ int64_t w[3][kScanThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        int64_t inc = x[q];
        for (int off = 1; off < 64; off <<= 1) {
            const int64_t o = __shfl_up(inc, off, 64);
            if (lane >= off) inc += o;
        }
        if (lane == 63) w[q][wave] = inc;
        x[q] = inc - x[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        total[q] = 0;
        for (int k = 0; k < kScanThreads / 64; ++k) {
            if (k < wave) x[q] += w[q][k];
            total[q] += w[q][k];
        }
    }
    __syncthreads();
}

__device__ __forceinline__ int block_max(int v)
{
    __shared__ int w[kScanThreads / 64];
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    for (int k = 0; k < kScanThreads / 64; ++k) v = max(v, w[k]);
    __syncthreads();
    return v;
}

}  // namespace

// The chunks' tiles in order, with the first entry of each in the ring list
// and among the first-step vertices (one block).
__global__ __launch_bounds__(kScanThreads) void k_plan_offsets(
    const TileRec *__restrict__ rec, const int32_t *__restrict__ count, int64_t chunks,
    TileRec *__restrict__ tile, int64_t *__restrict__ rbase, int64_t *__restrict__ cbase,
    PlanTotals *__restrict__ out)
{
    const int64_t per = (chunks + kScanThreads - 1) / kScanThreads;
    const int64_t b = min(chunks, per * threadIdx.x), e = min(chunks, b + per);
    int64_t x[3] = {0, 0, 0}, total[3];   // tiles, ring entries, first-step vertices
    int tmax = 0, lmax = 0, smax = 0, refused = 0;
    for (int64_t c = b; c < e; ++c) {
        if (count[c] < 0) refused = 1;
        for (int i = 0; i < count[c]; ++i) {
            const TileRec &r = rec[c * kPieces + i];
            x[0] += 1;
            x[1] += r.pref[kSteps] - r.pref[0];
            x[2] += r.pref[kSteps - 1];
            tmax = max(tmax, r.pref[0]);
            lmax = max(lmax, r.pref[kSteps]);
            smax = max(smax, r.pref[kSteps - 1]);
        }
    }
    block_sums(x, total);
    tmax = block_max(tmax);
    lmax = block_max(lmax);
    smax = block_max(smax);
    refused = block_max(refused);
    if (!refused)   // else some counts are -1 and the tiles are not used
        for (int64_t c = b; c < e; ++c)
            for (int i = 0; i < count[c]; ++i) {
                const TileRec r = rec[c * kPieces + i];
                tile[x[0]] = r;
                rbase[x[0]] = x[1];
                cbase[x[0]] = x[2];
                x[0] += 1;
                x[1] += r.pref[kSteps] - r.pref[0];
                x[2] += r.pref[kSteps - 1];
            }
    if (threadIdx.x == 0) {
        out->ntiles = total[0];
        out->nring = total[1];
        out->ncs = total[2];
        out->nlen = 0;
        out->max_tile = tmax;
        out->max_load = lmax;
        out->max_step1 = smax;
        out->refused = refused;
        if (!refused) {
            rbase[total[0]] = total[1];
            cbase[total[0]] = total[2];
        }
    }
}

// Rings, slot codes and length columns of each tile (nx_tiles.cpp, tile_edges).
__global__ __launch_bounds__(kThreads) void k_plan_owners(const int32_t *__restrict__ col, int64_t V,
                                                          const TileRec *__restrict__ tile,
                                                          const int64_t *__restrict__ rbase,
                                                          const int64_t *__restrict__ cbase,
                                                          int32_t *__restrict__ ring_out,
                                                          uint16_t *__restrict__ code_out,
                                                          int32_t *__restrict__ kt_out,
                                                          PlanTotals *__restrict__ totals)
{
    constexpr int kPer = kQuadStepOne / kThreads;
    __shared__ RingSet S;
    __shared__ uint16_t place[kHash];                // a ring vertex's local index
    __shared__ uint16_t slot[6][kQuadStepOne];       // neighbour (bits 0-11), back slot (12-14), movable
    __shared__ uint32_t own[kQuadStepOne];
    __shared__ uint8_t dist[kQuadStepOne];
    const int t = threadIdx.x;
    const int64_t a = tile[blockIdx.x].a;
    const int T = tile[blockIdx.x].pref[0], c = tile[blockIdx.x].pref[kSteps - 1];
    if (!tile_rings<true>(S, col, V, a, T)) return;   // (it fitted when it was cut)
    const int nring = S.pref[kSteps] - T;
    int32_t *ring = ring_out + rbase[blockIdx.x];
    for (int i = t; i < nring; i += kThreads) {
        const int32_t n = S.ring[i];
        ring[i] = n;
        uint32_t h = ring_hash(n);
        while (S.key[h] != n) h = (h + 1) & (kHash - 1);
        place[h] = (uint16_t)(T + i);
    }
    __syncthreads();
    auto device_index = [&](int j) { return j < T ? (int32_t)(a + j) : S.ring[j - T]; };
    // every neighbour of a first-step vertex is in the tile or its rings
    for (int j = t; j < c; j += kThreads) {
        const int32_t v = device_index(j);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int32_t n = col[(int64_t)k * V + v];
            int l;
            if (n >= a && n < a + T) {
                l = (int)(n - a);
            } else {
                uint32_t h = ring_hash(n);
                while (S.key[h] != n && S.key[h] != -1) h = (h + 1) & (kHash - 1);
                l = place[h];
            }
            slot[k][j] = (uint16_t)l;
        }
    }
    __syncthreads();
    // first owners; slots that do not name each other first are left to the host
    bool odd = false;
    uint16_t full[kPer][6];
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
        const int j = t + m * kThreads;
        if (j >= c) continue;
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int n = slot[k][j];
            full[m][k] = (uint16_t)n;
            if (n == j) continue;
            if (n >= c) {
                mine |= 1u << k;
                continue;
            }
            int q = -1, self = -1;
#pragma unroll
            for (int z = 5; z >= 0; --z) {
                if (slot[z][n] == j) q = z;
                if (slot[z][j] == n) self = z;
            }
            odd = odd || q < 0 || self != k;
            full[m][k] = (uint16_t)(n | (q & 7) << 12 | 0x8000);
            if ((j >= T) != (n >= T) ? j >= T : device_index(j) < device_index(n)) mine |= 1u << k;
        }
        own[j] = mine;
    }
    odd = __syncthreads_or(odd);
    if (odd) {
        if (t == 0) totals->refused = 1;
        return;
    }
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
        const int j = t + m * kThreads;
        if (j < c)
#pragma unroll
            for (int k = 0; k < 6; ++k) slot[k][j] = full[m][k];
    }
    __syncthreads();
    // this thread's slots in registers: local neighbours two to a word, and
    // the movable ones
    uint32_t nb[kPer][3], movable[kPer];
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
        const int j = t + m * kThreads;
        movable[m] = 0;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const uint32_t x = j < c ? slot[k][j] : 0;
            nb[m][k >> 1] = k & 1 ? nb[m][k >> 1] | (x & 4095) << 16 : x & 4095;
            movable[m] |= (x >> 15) << k;
        }
    }
    auto nbr = [&](int m, int k) { return (int)(nb[m][k >> 1] >> (16 * (k & 1)) & 4095); };
    int kr = kOwnRing;
    auto cap = [&](int j) { return j < T ? kLenFull : kr; };
    for (int round = 0;; ++round) {
        bool over[kPer];
        uint32_t free_[kPer];   // movable edges held
        bool any = false;
#pragma unroll
        for (int m = 0; m < kPer; ++m) {
            const int j = t + m * kThreads;
            over[m] = false;
            free_[m] = 0;
            if (j >= c) continue;
            const int held = __popc(own[j]);
            over[m] = held > cap(j);
            any = any || over[m];
            dist[j] = held < cap(j) ? 0 : kOwnFar;
            free_[m] = own[j] & movable[m];
        }
        if (!__syncthreads_or(any)) break;
        if (round == kOwnRounds) {
            if (t == 0) totals->refused = 1;
            return;
        }
        for (int s = 1; s < kOwnFar; ++s) {
            bool changed = false, far = false;
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                const int j = t + m * kThreads;
                if (j >= c || dist[j] != kOwnFar) continue;
                bool near = false;
#pragma unroll
                for (int k = 0; k < 6; ++k)
                    if (free_[m] >> k & 1) near = near || dist[nbr(m, k)] == s - 1;
                if (near) dist[j] = (uint8_t)s;
                changed = changed || near;
                far = far || (over[m] && !near);
            }
            changed = __syncthreads_or(changed);
            far = __syncthreads_or(far);
            if (!changed || !far) break;
        }
        bool moved = false;
        for (;;) {
            int move[kPer];
            bool moves = false;
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                const int j = t + m * kThreads;
                move[m] = -1;
                if (j >= c || __popc(own[j]) <= cap(j)) continue;
                const int at = dist[j];
                if (at == 0 || at == kOwnFar) continue;
                const uint32_t f = own[j] & movable[m];
#pragma unroll
                for (int k = 5; k >= 0; --k)
                    if ((f >> k & 1) && dist[nbr(m, k)] == at - 1) move[m] = k;
                moves = moves || move[m] >= 0;
            }
            if (!__syncthreads_or(moves)) break;
            moved = true;
#pragma unroll
            for (int m = 0; m < kPer; ++m) {
                if (move[m] < 0) continue;
                const int j = t + m * kThreads, x = slot[move[m]][j];
                atomicAnd(&own[j], ~(1u << move[m]));
                atomicOr(&own[x & 4095], 1u << (x >> 12 & 7));
            }
            __syncthreads();
        }
        if (!moved) {
            if (kr >= 6) {
                if (t == 0) totals->refused = 1;
                return;
            }
            ++kr;
        }
    }
    // slot codes
    uint16_t *code = code_out + 6 * cbase[blockIdx.x];
    int kt = 1;
    for (int j = t; j < c; j += kThreads) {
        const uint32_t o = own[j];
        kt = max(kt, __popc(o));
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int x = slot[k][j], n = x & 4095;
            uint32_t e;
            if (n == j)
                e = (uint32_t)j | 0x8000u;
            else if (o >> k & 1)
                e = (uint32_t)n | (uint32_t)__popc(o & ((1u << k) - 1)) << 12 | 0x8000u;
            else
                e = (uint32_t)n | (uint32_t)__popc(own[n] & ((1u << (x >> 12 & 7)) - 1)) << 12;
            code[(int64_t)k * c + j] = (uint16_t)e;
        }
    }
    kt = block_max(kt);
    if (t == 0) kt_out[blockIdx.x] = kt;
}

// First length of each tile, and their number (one block).
__global__ __launch_bounds__(kScanThreads) void k_plan_lengths(const TileRec *__restrict__ tile,
                                                               const int32_t *__restrict__ kt,
                                                               int64_t ntiles,
                                                               int64_t *__restrict__ ebase,
                                                               PlanTotals *__restrict__ out)
{
    if (out->refused) return;   // some kt were not written
    const int64_t per = (ntiles + kScanThreads - 1) / kScanThreads;
    const int64_t b = min(ntiles, per * threadIdx.x), e = min(ntiles, b + per);
    int64_t x[3] = {0, 0, 0}, total[3];
    for (int64_t i = b; i < e; ++i)
        x[0] += len_block(kt[i], tile[i].pref[kSteps - 1], tile[i].pref[0]);
    block_sums(x, total);
    for (int64_t i = b; i < e; ++i) {
        ebase[i] = x[0];
        x[0] += len_block(kt[i], tile[i].pref[kSteps - 1], tile[i].pref[0]);
    }
    if (threadIdx.x == 0) {
        ebase[ntiles] = total[0];
        out->nlen = total[0];
    }
}

// The image: a block copies its tile's sections and fills in its lengths.
__global__ __launch_bounds__(kThreads) void k_plan_write(
    const double *__restrict__ elen, int64_t V, const TileRec *__restrict__ tile,
    const int64_t *__restrict__ rbase, const int64_t *__restrict__ cbase,
    const int64_t *__restrict__ ebase, const int32_t *__restrict__ kt,
    const int32_t *__restrict__ ring, const uint16_t *__restrict__ code, nx_tile_plan q,
    char *__restrict__ img)
{
    const int64_t i = blockIdx.x;
    const TileRec r = tile[i];
    const int t = threadIdx.x, T = r.pref[0], c = r.pref[kSteps - 1];
    if (t == 0) {
        ((int32_t *)(img + q.off_start))[i] = r.a;
        ((int32_t *)(img + q.off_cs))[i] = c;
        ((int32_t *)(img + q.off_load))[i] = r.pref[kSteps];
        ((int64_t *)(img + q.off_rbase))[i] = rbase[i];
        ((int64_t *)(img + q.off_cbase))[i] = cbase[i];
        ((int64_t *)(img + q.off_ebase))[i] = ebase[i];
        if (i == q.ntiles - 1) {
            ((int32_t *)(img + q.off_start))[i + 1] = (int32_t)V;
            ((int64_t *)(img + q.off_rbase))[i + 1] = rbase[i + 1];
            ((int64_t *)(img + q.off_cbase))[i + 1] = cbase[i + 1];
            ((int64_t *)(img + q.off_ebase))[i + 1] = ebase[i + 1];
        }
    }
    if (t <= kSteps) ((int32_t *)(img + q.off_pref))[i * (kSteps + 1) + t] = r.pref[t];
    const int32_t *rg = ring + rbase[i];
    int32_t *ro = (int32_t *)(img + q.off_ring) + rbase[i];
    for (int j = t; j < r.pref[kSteps] - T; j += kThreads) ro[j] = rg[j];
    const uint16_t *cd = code + 6 * cbase[i];
    uint16_t *co = (uint16_t *)(img + q.off_lcol) + 6 * cbase[i];
    for (int j = t; j < 6 * c; j += kThreads) co[j] = cd[j];
    double *lens = (double *)(img + q.off_lel) + ebase[i];
    for (int j = t; j < c; j += kThreads) {
        const int64_t v = j < T ? r.a + j : rg[j - T];
        const int columns = j < T ? min(kt[i], kLenFull) : kt[i];
        int m = 0;
        for (int k = 0; k < 6; ++k) {
            const int e = cd[(int64_t)k * c + j];
            if (e & 0x8000 && slot_nbr(e) != j) lens[len_index(m++, j, c, T)] = elen[(int64_t)k * V + v];
        }
        for (; m < columns; ++m) lens[len_index(m, j, c, T)] = 0.0;
    }
}

size_t tile_plan_device_workspace_bytes(int64_t V, int chunk)
{
    if (V <= 0 || V > INT32_MAX || chunk < 0 || (chunk != 0 && chunk < kTileMin)) return 256;
    return plan_scratch(V, chunk ? chunk : quad_chunk(V)).total;
}

int tile_plan_build_device(nx_ctx *ctx, const int32_t *col, const double *elen, int64_t V,
                           int chunk_in, void *ws, void *out, int64_t cap, nx_tile_plan *plan,
                           hipStream_t stream)
{
    if (!ctx || !col || !elen || !plan || !ws || V <= 0 || V > INT32_MAX)
        return set_error(NX_EINVAL, "tile plan needs col, elen, plan, a workspace and 0 < V < 2^31");
    if (((uintptr_t)ws & 255) != 0) return set_error(NX_EINVAL, "workspace must be 256-byte aligned");
    if (chunk_in != 0 && (chunk_in < kTileMin || chunk_in > kQuadStepOne))
        return set_error(NX_EINVAL, "tile chunk %d outside %d..%d (0 for the default)", chunk_in,
                         kTileMin, kQuadStepOne);
    NX_HIP(hipSetDevice(ctx->device));
    const int64_t chunk = chunk_in ? chunk_in : quad_chunk(V);
    const PlanScratch L = plan_scratch(V, chunk);
    char *w = (char *)ws;
    auto *totals = (PlanTotals *)(w + L.totals);
    auto *count = (int32_t *)(w + L.count);
    auto *rec = (TileRec *)(w + L.rec), *tile = (TileRec *)(w + L.tile);
    auto *rbase = (int64_t *)(w + L.rbase), *cbase = (int64_t *)(w + L.cbase);
    auto *ebase = (int64_t *)(w + L.ebase);
    auto *kt = (int32_t *)(w + L.kt), *ring = (int32_t *)(w + L.ring);
    auto *code = (uint16_t *)(w + L.code);
    if (out) {   // the image of the plan that the call before sized
        if (plan->V != V || plan->steps != kSteps || cap < plan->bytes)
            return set_error(NX_EINVAL, "tile plan image needs the plan sized with this workspace");
        hipLaunchKernelGGL(k_plan_write, dim3((unsigned)plan->ntiles), dim3(kThreads), 0, stream, elen, V,
                           tile, rbase, cbase, ebase, kt, ring, code, *plan, (char *)out);
        NX_HIP(hipGetLastError());
        return NX_OK;
    }
    PlanTotals h;
    hipLaunchKernelGGL(k_plan_cut, dim3((unsigned)L.chunks), dim3(kThreads), 0, stream, col, V, chunk,
                       rec, count);
    hipLaunchKernelGGL(k_plan_offsets, dim3(1), dim3(kScanThreads), 0, stream, rec, count, L.chunks,
                       tile, rbase, cbase, totals);
    NX_HIP(hipGetLastError());
    NX_HIP(hipMemcpyAsync(&h, totals, sizeof(h), hipMemcpyDeviceToHost, stream));
    NX_HIP(hipStreamSynchronize(stream));
    if (h.refused || h.nring > (int64_t)(kSteps / 2) * V)
        return set_error(NX_ERANGE, "vertices do not cut into tiles whose %d rings fit %d vertices, or "
                         "the rings hold more than %d vertices per owned one", kSteps, kQuadLoadMax,
                         kSteps / 2);
    hipLaunchKernelGGL(k_plan_owners, dim3((unsigned)h.ntiles), dim3(kThreads), 0, stream, col, V,
                       tile, rbase, cbase, ring, code, kt, totals);
    hipLaunchKernelGGL(k_plan_lengths, dim3(1), dim3(kScanThreads), 0, stream, tile, kt, h.ntiles,
                       ebase, totals);
    NX_HIP(hipGetLastError());
    NX_HIP(hipMemcpyAsync(&h, totals, sizeof(h), hipMemcpyDeviceToHost, stream));
    NX_HIP(hipStreamSynchronize(stream));
    if (h.refused)
        return set_error(NX_ERANGE, "tile plan: a neighbour table that is not symmetric");
    nx_tile_plan q;
    std::memset(&q, 0, sizeof(q));
    q.V = V;
    q.max_tile = h.max_tile;
    q.max_load = h.max_load;
    q.max_step1 = h.max_step1;
    plan_layout(q, h.ntiles, h.nring, h.ncs, h.nlen, kSteps);
    q.blob = plan->blob;
    *plan = q;
    return NX_OK;
}

}  // namespace nx
