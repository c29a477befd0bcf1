// Samples in tile order: degridding and the density iterations' gridding.
//
// Degridding reads, and single-channel gridding writes, about 34 (2D: 13)
// cells per sample.  In acquisition order those cells are all over the grid;
// here a plan's samples are sorted once by the tile (8^3 cells, 16^2 in 2D
// and per frame) that holds the first cell of their kernel box, so that a
// workgroup finds every cell its samples touch in one region (11^3 or 19^2
// cells) in LDS:
//   k_tile_degrid   stages the region of up to 4 (2D: 8) coils and sums each
//                   sample's taps, one lane per sample, in the reference's z,
//                   y, x order (bit-identical to k_degrid);
//   k_dens_grid     real weights only (Pipe-Menon grids w itself): one lane
//                   per tap, a wave's samples one after the other into a box
//                   of its own with LDS adds.  The taps of a sample are
//                   distinct cells and LDS instructions of a wave execute in
//                   order, so the sums do not depend on timing;
//   k_dens_slices, k_dens_combine   add the boxes of a tile's slices and of
//                   the up to 8 tiles that reach a cell, in a fixed order;
//   k_dens_update   the same region scheme for w <- w / (G^H G w).
//
// The order exists only for position-weight plans (which own their sample
// positions) with kernels of width <= 4: at most 4 cells per axis have
// |x - c| < hw.  It is built on first use, from the plan's positions, and
// serves a samples handle only while that handle's trajectory is the one the
// plan was built on (uid and version); others take the general kernels of
// fr_dcf.hip.
#include "fr_internal.h"
#include "fr_taps.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// samples per work item (workgroup): a slice of a tile.  Tiles of usual 3D
// scans hold 200 to 800 samples; the central ones, up to half a million, are
// cut so that no workgroup runs much longer than the others
constexpr uint32_t SLICE = 1024;
constexpr int WAVES = 4;

template <int DIM> struct shape;
template <> struct shape<3> {
    static constexpr int LOG = 3, TILE = 8, EDGE = 11, CELLS = 11 * 11 * 11, TAPS = 64;
};
template <> struct shape<2> {
    static constexpr int LOG = 4, TILE = 16, EDGE = 19, CELLS = 19 * 19, TAPS = 16;
};

struct tgeom {
    float hw;
    int N, frames;
    int ntx, nty, ntz;
    uint32_t nt;                 // tiles; samples without a cell in reach sort behind them
};

// First cell of a sample's kernel box along one axis: cells with fl(x - c)
// outside (-hw, hw) fail the reference tap test whatever the other axes
// (sqrtf of anything >= fl(hw hw) is >= hw), and fl(x - c) is monotone in x,
// so lo .. lo + 3 hold every accepted cell for hw <= 2.  False when no cell
// of the grid is in reach.
__device__ __forceinline__ bool first_cell(float c, float hw, int N, int &lo)
{
    int a = (int)ceilf(c - hw), e = (int)floorf(c + hw);
    if (a > N - 1 || e < 0) return false;
    a = max(a, 0);
    e = min(e, N - 1);
    if (__fsub_rn((float)a, c) <= -hw) ++a;
    if (__fsub_rn((float)e, c) >= hw) --e;
    lo = a;
    return a <= e;
}

template <int DIM>
__device__ __forceinline__ bool box_of(const float4 &p, const tgeom &g, int (&lo)[3])
{
    lo[0] = lo[1] = lo[2] = 0;
    bool in = first_cell(p.x, g.hw, g.N, lo[0]) && first_cell(p.y, g.hw, g.N, lo[1]);
    if constexpr (DIM == 3) in = in && first_cell(p.z, g.hw, g.N, lo[2]);
    else lo[2] = (int)p.z;       // the frame (0 for one grid)
    return in;
}

template <int DIM>
__global__ void k_tile_key(const float4 *__restrict__ pos, int64_t M, tgeom g, uint32_t *__restrict__ key,
                           uint32_t *__restrict__ val)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    int lo[3];
    const bool in = box_of<DIM>(pos[i], g, lo);
    const int tz = DIM == 3 ? lo[2] >> shape<DIM>::LOG : lo[2];
    key[i] = in ? (uint32_t)((tz * g.nty + (lo[1] >> shape<DIM>::LOG)) * g.ntx + (lo[0] >> shape<DIM>::LOG)) : g.nt;
    val[i] = (uint32_t)i;
}

// tpos[i] = the position of the i-th sample in tile order and its index
__global__ void k_tile_place(const float4 *__restrict__ pos, const uint32_t *__restrict__ val, int64_t M,
                             float4 *__restrict__ tpos)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    const uint32_t s = val[i];
    float4 p = pos[s];
    p.w = __uint_as_float(s);
    tpos[i] = p;
}

// start[t] = first sample of tile t in the sorted keys (t = 0 .. nt + 1)
__global__ void k_tile_start(const uint32_t *__restrict__ key, int64_t M, uint32_t nt, uint32_t *__restrict__ start)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > nt + 1) return;
    int64_t lo = 0, hi = M;
    while (lo < hi) {
        const int64_t mid = (lo + hi) / 2;
        if (key[mid] < t) lo = mid + 1; else hi = mid;
    }
    start[t] = (uint32_t)lo;
}

__global__ void k_tile_slices(const uint32_t *__restrict__ start, uint32_t nt, uint32_t *__restrict__ n)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > nt + 1) return;
    n[t] = t <= nt ? (start[t + 1] - start[t] + SLICE - 1) / SLICE : 0u;
}

// items of tile t: [first[t], first[t + 1]); tiles with several go to the list
__global__ void k_tile_items(const uint32_t *__restrict__ start, const uint32_t *__restrict__ first, uint32_t nt,
                             fr_titem *__restrict__ items, uint32_t *__restrict__ many, uint32_t *__restrict__ nmany)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > nt) return;
    const uint32_t a = start[t], b = start[t + 1], f = first[t], n = first[t + 1] - f;
    for (uint32_t q = 0; q < n; ++q)
        items[f + q] = fr_titem{t, a + q * SLICE, min(SLICE, b - (a + q * SLICE)), 0u};
    if (n > 1 && t < nt) many[atomicAdd(nmany, 1u)] = t;
}

template <int DIM>
__device__ __forceinline__ void tile_origin(uint32_t t, const tgeom &g, int &ox, int &oy, int &oz)
{
    ox = (int)(t % g.ntx) * shape<DIM>::TILE;
    oy = (int)(t / g.ntx % g.nty) * shape<DIM>::TILE;
    oz = (int)(t / (g.ntx * g.nty)) * (DIM == 3 ? shape<DIM>::TILE : 1);
}

// region cell q of the tile at (ox, oy, oz): its grid index, or -1 outside the grid
template <int DIM>
__device__ __forceinline__ int64_t region_cell(int q, int ox, int oy, int oz, int N)
{
    constexpr int E = shape<DIM>::EDGE;
    const int x = ox + q % E, y = oy + q / E % E, z = oz + (DIM == 3 ? q / (E * E) : 0);
    if (x >= N || y >= N || (DIM == 3 && z >= N)) return -1;
    return ((int64_t)z * N + y) * N + x;
}

// The selection table in LDS as two arrays of 4-byte entries: thr[m] = least
// d2 of index m + 1, lut[0 .. L].  Two dependent 4-byte reads of random
// entries cost the LDS fewer cycles than one 16-byte read (k_dens_update at
// 13.1M samples: 400 us against 492).
struct table {
    float *thr, *lut;
    float dacc, cidx, lmax;
};
__host__ __device__ constexpr int table_floats(int L) { return (2 * L + 1 + 3) & ~3; }

template <int NW = WAVES>
__device__ __forceinline__ table stage_table(float *sm, const float4 *__restrict__ tbl, int L, float dacc, float cidx)
{
    const table T{sm, sm + L, dacc, cidx, (float)(L - 1)};
    for (int q = threadIdx.x; q < L; q += 64 * NW) {
        const float4 e = tbl[q];
        T.thr[q] = e.x;
        T.lut[q] = e.y;
        if (q == L - 1) T.lut[L] = e.z;
    }
    return T;
}

// fr_tap_weight without the tap test
__device__ __forceinline__ float lut_weight(const table &T, float d2)
{
    const int e = (int)fminf(__builtin_fmaf(__builtin_amdgcn_sqrtf(d2), T.cidx, 0.49f), T.lmax);
    return T.lut[e + (d2 >= T.thr[e] ? 1 : 0)];
}

// ------------------------------------------------------------- degridding
// Sum of one sample's taps over the region: f(cell, w) for the 4^DIM box in
// z, y, x order with w = 0 where the reference tap test fails.  The four
// weights of a row are independent, so their table reads overlap.
template <int DIM, typename F>
__device__ __forceinline__ void box_taps(const float4 &p, const int (&lo)[3], int ox, int oy, int oz,
                                         const table &T, F &&f)
{
    constexpr int E = shape<DIM>::EDGE;
    float dx2[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const float dx = __fsub_rn((float)(lo[0] + x), p.x);
        dx2[x] = __fmul_rn(dx, dx);
    }
    const int base = (DIM == 3 ? (lo[2] - oz) * E * E : 0) + (lo[1] - oy) * E + (lo[0] - ox);
#pragma unroll 1
    for (int z = 0; z < (DIM == 3 ? 4 : 1); ++z) {
        float dz2 = 0.f;
        if constexpr (DIM == 3) {
            const float dz = __fsub_rn((float)(lo[2] + z), p.z);
            dz2 = __fmul_rn(dz, dz);
        }
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const float dy = __fsub_rn((float)(lo[1] + y), p.y);
            const float dzy = __fadd_rn(dz2, __fmul_rn(dy, dy));
            float w[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const float d2 = __fadd_rn(dzy, dx2[x]);
                w[x] = lut_weight(T, d2);
                w[x] = d2 < T.dacc ? w[x] : 0.f;
            }
            f(base + (z * E + y) * E, w);
        }
    }
}

// f(cell, w) for a sample's accepted taps alone, in the same order.  For
// regions with an infinite or NaN value, which a weight of 0 does not leave
// out of a sum.
template <int DIM, typename F>
__device__ __forceinline__ void accepted_taps(const float4 &p, const int (&lo)[3], int ox, int oy, int oz, int N,
                                              const table &T, F &&f)
{
    constexpr int E = shape<DIM>::EDGE;
#pragma unroll 1
    for (int t = 0; t < shape<DIM>::TAPS; ++t) {
        const int x = t & 3, y = t >> 2 & 3, z = t >> 4;
        const float dz = DIM == 3 ? __fsub_rn((float)(lo[2] + z), p.z) : 0.f;
        const float dy = __fsub_rn((float)(lo[1] + y), p.y), dx = __fsub_rn((float)(lo[0] + x), p.x);
        const float d2 = fr_tap_dk2(__fmul_rn(dz, dz), __fmul_rn(dy, dy), dx);
        // a cell past the grid's edge is no tap (its region value is 0)
        if (!(d2 < T.dacc) || lo[0] + x >= N || lo[1] + y >= N || (DIM == 3 && lo[2] + z >= N)) continue;
        f(((DIM == 3 ? lo[2] - oz + z : 0) * E + lo[1] - oy + y) * E + lo[0] - ox + x, lut_weight(T, d2));
    }
}

// out[s][c0 + c] for the samples of one item.  The region's coils lie side by
// side in LDS, a cell's in an odd multiple of 4 words for pairs of coils, of 2
// words for an odd number (16- or 8-byte reads of random cells then spread
// over all banks).  A rejected tap adds 0 * v, which leaves a sum unchanged
// bit for bit unless v is infinite or NaN; a region with such a value takes
// the second loop, of accepted taps.  Bound by the LDS: per tap two table
// reads and the cell's coils, all at random addresses.
template <int NC> constexpr int cell_words() { return NC % 4 == 0 ? 2 * NC + 4 : 2 * NC; }

// the NC coils of a region cell
template <int NC>
__device__ __forceinline__ void load_cell(const float *cell, float2 (&v)[NC])
{
    if constexpr (NC % 2 == 0) {
#pragma unroll
        for (int c = 0; c < NC; c += 2) {
            const float4 a = *reinterpret_cast<const float4 *>(cell + 2 * c);
            v[c] = make_float2(a.x, a.y);
            v[c + 1] = make_float2(a.z, a.w);
        }
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = *reinterpret_cast<const float2 *>(cell + 2 * c);
    }
}

template <int DIM, int NC, int NW>
__global__ void __launch_bounds__(64 * NW) k_tile_degrid(const fr_titem *__restrict__ items,
                                                            const float4 *__restrict__ tpos, tgeom g,
                                                            const float4 *__restrict__ tbl, int L, float dacc,
                                                            float cidx, const float2 *__restrict__ grid, size_t cells,
                                                            int C, float2 *__restrict__ out)
{
    constexpr int CELLS = shape<DIM>::CELLS, CW = cell_words<NC>();
    extern __shared__ float4 sm[];
    float *reg = reinterpret_cast<float *>(sm) + table_floats(L);
    __shared__ int odd;
    const fr_titem it = items[blockIdx.x];
    const int c0 = blockIdx.y * NC, nc = min(NC, C - c0);
    if (it.tile == g.nt) {       // samples that reach no cell
        for (uint32_t i = threadIdx.x; i < it.n; i += 64 * NW) {
            const size_t s = __float_as_uint(tpos[it.s0 + i].w);
            for (int c = 0; c < nc; ++c) out[s * C + c0 + c] = make_float2(0.f, 0.f);
        }
        return;
    }
    if (threadIdx.x == 0) odd = 0;
    const table T = stage_table<NW>(reinterpret_cast<float *>(sm), tbl, L, dacc, cidx);
    __syncthreads();
    int ox, oy, oz;
    tile_origin<DIM>(it.tile, g, ox, oy, oz);
    bool fine = true;
    for (int q = threadIdx.x; q < CELLS; q += 64 * NW) {
        const int64_t at = region_cell<DIM>(q, ox, oy, oz, g.N);
        float2 v[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c)
            v[c] = at >= 0 && c < nc ? grid[(size_t)(c0 + c) * cells + at] : make_float2(0.f, 0.f);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            *reinterpret_cast<float2 *>(reg + q * CW + 2 * c) = v[c];
            // a - a is 0 for finite a, NaN for the others
            fine = fine && __fadd_rn(__fsub_rn(v[c].x, v[c].x), __fsub_rn(v[c].y, v[c].y)) == 0.f;
        }
    }
    if (!fine) odd = 1;
    __syncthreads();
    const bool skip = odd != 0;
    for (uint32_t i = threadIdx.x; i < it.n; i += 64 * NW) {
        const float4 p = tpos[it.s0 + i];
        int lo[3];
        box_of<DIM>(p, g, lo);
        float2 a[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) a[c] = make_float2(0.f, 0.f);
        if (!skip) {
            box_taps<DIM>(p, lo, ox, oy, oz, T, [&](int cell, const float (&w)[4]) {
                float2 v[4][NC];
#pragma unroll
                for (int x = 0; x < 4; ++x) load_cell<NC>(reg + (cell + x) * CW, v[x]);
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        a[c].x = __fadd_rn(a[c].x, __fmul_rn(w[x], v[x][c].x));
                        a[c].y = __fadd_rn(a[c].y, __fmul_rn(w[x], v[x][c].y));
                    }
            });
        } else {
            accepted_taps<DIM>(p, lo, ox, oy, oz, g.N, T, [&](int cell, float w) {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const float2 v = *reinterpret_cast<const float2 *>(reg + cell * CW + 2 * c);
                    a[c].x = __fadd_rn(a[c].x, __fmul_rn(w, v.x));
                    a[c].y = __fadd_rn(a[c].y, __fmul_rn(w, v.y));
                }
            });
        }
        float2 *o = out + (size_t)__float_as_uint(p.w) * C + c0;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (c < nc) o[c] = a[c];
    }
}

// ---------------------------------------------------------------- density
// A wave's LDS instructions execute in order; this keeps the compiler from
// moving one lane's read before another lane's write (no instruction).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int STAGED = 16;       // floats per staged sample
constexpr int AHEAD = 8;         // samples (2D: groups of 4) whose weights are computed before their adds

__device__ __forceinline__ float4 axis_d2(int lo, float c)
{
    const float a = __fsub_rn((float)lo, c), b = __fsub_rn((float)(lo + 1), c);
    const float e = __fsub_rn((float)(lo + 2), c), f = __fsub_rn((float)(lo + 3), c);
    return make_float4(__fmul_rn(a, a), __fmul_rn(b, b), __fmul_rn(e, e), __fmul_rn(f, f));
}

// Boxes of real sums per item: each wave (2D: each 16 lanes) adds its share
// of the item's samples into a box of its own, lane = tap.  13.1M samples on
// 256^3: 830 us (2240 with the many-coil gridding kernel, whose 8 records per
// sample each cost the same weights again); LDS float atomics instead of the
// wave's own read-add-write took 3031, weights and adds sample by sample 935.
// Bound by LDS (staged values, two table reads, the cell's read and write)
// and VALU issue, about 40 cycles of each per sample and CU.
template <int DIM>
__global__ void __launch_bounds__(64 * WAVES) k_dens_grid(const fr_titem *__restrict__ items,
                                                          const float4 *__restrict__ tpos,
                                                          const float *__restrict__ w, tgeom g,
                                                          const float4 *__restrict__ tbl, int L, float dacc,
                                                          float cidx, float *__restrict__ part)
{
    constexpr int CELLS = shape<DIM>::CELLS, E = shape<DIM>::EDGE, TAPS = shape<DIM>::TAPS, SUB = 64 / TAPS;
    extern __shared__ float4 sm[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    // 64 staged samples per wave: the squared distances of the box's 4 cells
    // along each axis, the weight and the box's offset in the region
    float *stage = reinterpret_cast<float *>(sm) + table_floats(L) + wv * 64 * STAGED;
    float *boxes = reinterpret_cast<float *>(sm) + table_floats(L) + WAVES * 64 * STAGED;
    const fr_titem it = items[blockIdx.x];
    if (it.tile == g.nt) return;
    const table T = stage_table(reinterpret_cast<float *>(sm), tbl, L, dacc, cidx);
    for (int q = threadIdx.x; q < CELLS * WAVES * SUB; q += 64 * WAVES) boxes[q] = 0.f;
    __syncthreads();
    int ox, oy, oz;
    tile_origin<DIM>(it.tile, g, ox, oy, oz);
    const int tap = lane & (TAPS - 1), sub = lane / TAPS;
    const float *sx = stage + sub * STAGED + (tap & 3), *sy = stage + sub * STAGED + 4 + (tap >> 2 & 3),
                *sz = stage + sub * STAGED + 8 + (tap >> 4), *sw = stage + sub * STAGED + 12;
    float *box = boxes + (wv * SUB + sub) * CELLS + ((tap >> 4) * E + (tap >> 2 & 3)) * E + (tap & 3);
    float *none = boxes + CELLS * WAVES * SUB + threadIdx.x;
    const uint32_t share = (it.n + WAVES - 1) / WAVES;
    const uint32_t a = min(it.n, wv * share), b = min(it.n, a + share);
    for (uint32_t i = a; i < b; i += 64) {
        const uint32_t n = min(64u, b - i);
        float4 d[3] = {make_float4(3e30f, 3e30f, 3e30f, 3e30f)};         // no tap
        float2 wo = make_float2(0.f, 0.f);
        if ((uint32_t)lane < n) {
            const float4 p = tpos[it.s0 + i + lane];
            int lo[3];
            box_of<DIM>(p, g, lo);
            d[0] = axis_d2(lo[0], p.x);
            d[1] = axis_d2(lo[1], p.y);
            d[2] = DIM == 3 ? axis_d2(lo[2], p.z) : make_float4(0.f, 0.f, 0.f, 0.f);
            wo = make_float2(w[it.s0 + i + lane],
                             __int_as_float(((DIM == 3 ? lo[2] - oz : 0) * E + lo[1] - oy) * E + lo[0] - ox));
        }
        wave_sync();                         // the samples before are no longer read
        float4 *row = reinterpret_cast<float4 *>(stage + lane * STAGED);
        row[0] = d[0];
        row[1] = d[1];
        row[2] = d[2];
        *reinterpret_cast<float2 *>(row + 3) = wo;
        wave_sync();
        // AHEAD samples' values first, then their adds (the compiler cannot
        // tell the boxes from the staged samples, so it would not move a
        // read past an add); rejected taps add 0 to a cell of the lane's own
        const uint32_t steps = (n + SUB - 1) / SUB;
        for (uint32_t k = 0; k < steps; k += AHEAD) {
            float v[AHEAD];
            float *c[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int o = (k + u) * SUB * STAGED;
                const float d2 = __fadd_rn(DIM == 3 ? __fadd_rn(sz[o], sy[o]) : sy[o], sx[o]);
                const float2 q = *reinterpret_cast<const float2 *>(sw + o);
                v[u] = __fmul_rn(q.x, lut_weight(T, d2));
                c[u] = d2 < dacc ? box + __float_as_int(q.y) : none;
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                *c[u] = __fadd_rn(*c[u], v[u]);
                // the next sample's lanes may add to the same cells (ordered for
                // the compiler alone: a fence costs 3% of the kernel here)
                asm volatile("" ::: "memory");
            }
        }
    }
    __syncthreads();
    float *o = part + (size_t)blockIdx.x * CELLS;
    for (int q = threadIdx.x; q < CELLS; q += 64 * WAVES) {
        float v = boxes[q];
#pragma unroll
        for (int k = 1; k < WAVES * SUB; ++k) v = __fadd_rn(v, boxes[k * CELLS + q]);
        o[q] = v;
    }
}

// tiles with several items: their boxes added into the first one, 64 cells a
// workgroup, each wave taking every SLICE_WAVES-th box
constexpr int SLICE_WAVES = 4;
__global__ void __launch_bounds__(64 * SLICE_WAVES) k_dens_slices(const uint32_t *__restrict__ many,
                                                                  const uint32_t *__restrict__ first, int box_cells,
                                                                  float *__restrict__ part)
{
    __shared__ float sums[SLICE_WAVES][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t t = many[blockIdx.x], a = first[t], b = first[t + 1];
    const int q = blockIdx.y * 64 + lane;
    float v = 0.f;
    if (q < box_cells)
#pragma unroll 8
        for (uint32_t k = a + wv; k < b; k += SLICE_WAVES) v = __fadd_rn(v, part[(size_t)k * box_cells + q]);
    sums[wv][lane] = v;
    __syncthreads();
    if (wv != 0 || q >= box_cells) return;
#pragma unroll
    for (int k = 1; k < SLICE_WAVES; ++k) v = __fadd_rn(v, sums[k][lane]);
    part[(size_t)a * box_cells + q] = v;
}

// every cell of the real grid: its own tile's box, then those of the tiles
// before it whose regions reach it
template <int DIM>
__global__ void __launch_bounds__(256) k_dens_combine(const float *__restrict__ part,
                                                      const uint32_t *__restrict__ first, tgeom g, uint32_t cells,
                                                      float *__restrict__ grid)
{
    constexpr int T = shape<DIM>::TILE, E = shape<DIM>::EDGE, LOG = shape<DIM>::LOG, CELLS = shape<DIM>::CELLS;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cells) return;
    const uint32_t N = (uint32_t)g.N, r = i / N;
    const int x = (int)(i - r * N), z = (int)(r / N), y = (int)(r - (uint32_t)z * N);
    const int lx = x & (T - 1), ly = y & (T - 1), lz = DIM == 3 ? z & (T - 1) : 0;
    const int X = x >> LOG, Y = y >> LOG, Z = DIM == 3 ? z >> LOG : z;
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < (DIM == 3 ? 8 : 4); ++k) {
        const int dx = k & 1, dy = k >> 1 & 1, dz = k >> 2;
        if ((dx && (lx >= E - T || X == 0)) || (dy && (ly >= E - T || Y == 0)) || (dz && (lz >= E - T || Z == 0)))
            continue;
        const uint32_t t = (uint32_t)(((Z - dz) * g.nty + (Y - dy)) * g.ntx + (X - dx));
        const uint32_t f = first[t];
        if (f == first[t + 1]) continue;
        v = __fadd_rn(v, part[(size_t)f * CELLS + ((lz + dz * T) * E + ly + dy * T) * E + lx + dx * T]);
    }
    grid[i] = v;
}

// w <- w / (G^H G w); samples whose denominator is not positive get 0
template <int DIM>
__global__ void __launch_bounds__(64 * WAVES) k_dens_update(const fr_titem *__restrict__ items,
                                                            const float4 *__restrict__ tpos, tgeom g,
                                                            const float4 *__restrict__ tbl, int L, float dacc,
                                                            float cidx, const float *__restrict__ grid,
                                                            float *__restrict__ w)
{
    extern __shared__ float4 sm[];
    __shared__ int odd[WAVES];                  // a wave met an infinite or NaN cell
    float *reg = reinterpret_cast<float *>(sm) + table_floats(L);
    const fr_titem it = items[blockIdx.x];
    if (it.tile == g.nt) {
        for (uint32_t i = threadIdx.x; i < it.n; i += 64 * WAVES) w[it.s0 + i] = 0.f;
        return;
    }
    const table T = stage_table(reinterpret_cast<float *>(sm), tbl, L, dacc, cidx);
    int ox, oy, oz;
    tile_origin<DIM>(it.tile, g, ox, oy, oz);
    bool fine = true;
    for (int q = threadIdx.x; q < shape<DIM>::CELLS; q += 64 * WAVES) {
        const int64_t at = region_cell<DIM>(q, ox, oy, oz, g.N);
        const float v = at >= 0 ? grid[at] : 0.f;
        reg[q] = v;
        fine = fine && __fsub_rn(v, v) == 0.f;
    }
    const bool all_fine = __all(fine);
    if ((threadIdx.x & 63) == 0) odd[threadIdx.x >> 6] = !all_fine;
    __syncthreads();
    const bool skip = (odd[0] | odd[1] | odd[2] | odd[3]) != 0;
    static_assert(WAVES == 4, "flags read above");
    for (uint32_t i = threadIdx.x; i < it.n; i += 64 * WAVES) {
        const float4 p = tpos[it.s0 + i];
        int lo[3];
        box_of<DIM>(p, g, lo);
        float d = 0.f;
        if (!skip)
            box_taps<DIM>(p, lo, ox, oy, oz, T, [&](int cell, const float (&t)[4]) {
#pragma unroll
                for (int x = 0; x < 4; ++x) d = __fadd_rn(d, __fmul_rn(t[x], reg[cell + x]));
            });
        else
            accepted_taps<DIM>(p, lo, ox, oy, oz, g.N, T,
                               [&](int cell, float t) { d = __fadd_rn(d, __fmul_rn(t, reg[cell])); });
        w[it.s0 + i] = d > 0.f ? __fdiv_rn(w[it.s0 + i], d) : 0.f;
    }
}

__global__ void k_fill(float *__restrict__ d, int64_t n, float v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = v;
}

// the density between acquisition order and tile order
__global__ void k_to_tiles(const float4 *__restrict__ tpos, const float *__restrict__ dcf, int64_t M,
                           float *__restrict__ w)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) w[i] = dcf[__float_as_uint(tpos[i].w)];
}
__global__ void k_from_tiles(const float4 *__restrict__ tpos, const float *__restrict__ w, int64_t M,
                             float *__restrict__ dcf)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) dcf[__float_as_uint(tpos[i].w)] = w[i];
}

tgeom geom_of(const fr_plan *p)
{
    tgeom g{};
    const int T = p->dim == 3 ? shape<3>::TILE : shape<2>::TILE;
    g.hw = p->kHW;
    g.N = (int)p->N;
    g.frames = p->frames;
    g.ntx = g.nty = (g.N + T - 1) / T;
    g.ntz = p->dim == 3 ? g.ntx : std::max(p->frames, 1);
    g.nt = (uint32_t)g.ntx * g.nty * g.ntz;
    return g;
}

template <typename T>
struct dbuf {
    T *p = nullptr;
    ~dbuf() { if (p) (void)hipFree(p); }
};

template <int DIM>
fr_status build(fr_plan *p, fr_tiles *t, const tgeom &g)
{
    fr_ctx *ctx = p->ctx;
    hipStream_t st = ctx->stream;
    const int64_t M = p->M;
    const uint32_t nt = g.nt;
    dbuf<uint32_t> key, val, key2, val2, start, n, nmany;
    dbuf<char> tmp;
    fr_status e;
    int bits = 1;
    while (bits < 32 && (uint64_t(1) << bits) <= nt) ++bits;
    size_t sort_bytes = 0, scan_bytes = 0;
    FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, key.p, key2.p, val.p, val2.p, (int)M, 0, bits,
                                                   st));
    FR_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, n.p, t->first, (int)(nt + 2), st));
    if ((e = fr_alloc(ctx, (void **)&t->tpos, sizeof(float4) * M)) ||
        (e = fr_alloc(ctx, (void **)&t->first, 4 * (size_t)(nt + 2))) ||
        (e = fr_alloc(ctx, (void **)&t->many, 4 * (size_t)(M / SLICE + 1))) ||
        (e = fr_alloc(ctx, (void **)&key.p, 4 * M)) || (e = fr_alloc(ctx, (void **)&val.p, 4 * M)) ||
        (e = fr_alloc(ctx, (void **)&key2.p, 4 * M)) || (e = fr_alloc(ctx, (void **)&val2.p, 4 * M)) ||
        (e = fr_alloc(ctx, (void **)&start.p, 4 * (size_t)(nt + 2))) ||
        (e = fr_alloc(ctx, (void **)&n.p, 4 * (size_t)(nt + 2))) || (e = fr_alloc(ctx, (void **)&nmany.p, 4)) ||
        (e = fr_alloc(ctx, (void **)&tmp.p, std::max(sort_bytes, scan_bytes) + 16)))
        return e;
    hipLaunchKernelGGL(k_tile_key<DIM>, dim3(nblk(M, 256)), dim3(256), 0, st, p->pos, M, g, key.p, val.p);
    FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(tmp.p, sort_bytes, key.p, key2.p, val.p, val2.p, (int)M, 0, bits,
                                                   st));
    hipLaunchKernelGGL(k_tile_place, dim3(nblk(M, 256)), dim3(256), 0, st, p->pos, val2.p, M, t->tpos);
    hipLaunchKernelGGL(k_tile_start, dim3(nblk(nt + 2, 256)), dim3(256), 0, st, key2.p, M, nt, start.p);
    hipLaunchKernelGGL(k_tile_slices, dim3(nblk(nt + 2, 256)), dim3(256), 0, st, start.p, nt, n.p);
    FR_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(tmp.p, scan_bytes, n.p, t->first, (int)(nt + 2), st));
    FR_HIP(ctx, hipMemsetAsync(nmany.p, 0, 4, st));
    uint32_t total = 0;
    FR_HIP(ctx, hipMemcpyAsync(&total, t->first + nt + 1, 4, hipMemcpyDeviceToHost, st));
    FR_HIP(ctx, hipStreamSynchronize(st));
    if ((e = fr_alloc(ctx, (void **)&t->items, sizeof(fr_titem) * (size_t)total))) return e;
    hipLaunchKernelGGL(k_tile_items, dim3(nblk(nt + 1, 256)), dim3(256), 0, st, start.p, t->first, nt, t->items,
                       t->many, nmany.p);
    FR_HIP(ctx, hipGetLastError());
    FR_HIP(ctx, hipMemcpyAsync(&t->nmany, nmany.p, 4, hipMemcpyDeviceToHost, st));
    FR_HIP(ctx, hipStreamSynchronize(st));
    t->nitems = total;
    return FR_OK;
}

template <int DIM, int NC, int NW>
fr_status degrid(const fr_plan *p, const tgeom &g, const float2 *grid, int C, float2 *out)
{
    fr_ctx *ctx = p->ctx;
    const fr_tiles *t = p->tord;
    const size_t lds = sizeof(float) * (table_floats(p->L) + shape<DIM>::CELLS * cell_words<NC>());
    auto kern = k_tile_degrid<DIM, NC, NW>;
    FR_HIP(ctx, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(t->nitems, (C + NC - 1) / NC), dim3(64 * NW), lds, ctx->stream, t->items, t->tpos,
                       g, p->tsel, p->L, p->mfma_dacc, p->mfma_cidx, grid, fr_plan_cells(p->dim, p->N, p->frames), C,
                       out);
    FR_HIP(ctx, hipGetLastError());
    return FR_OK;
}

// As few chunks of coils as the region's LDS allows, none of them much
// emptier than the others: a sample's weights are computed once per chunk and
// its region is read once per chunk.  Measured at 1.6M samples on 128^3: 8
// coils 2182 us in acquisition order, 309 as 4 chunks of 2 (4 waves), 287 as
// 2 of 4 (8 waves; 398 with 4), 335 as one of 8 (96 KB of LDS, one workgroup
// per CU); 12 coils 379 as 2 of 6; 1 coil 234 -> 76.  2D, 205,824 samples on
// 512^2: 8 coils 95 -> 23, 32 coils 476 -> 57, 1 coil 15 -> 8.
template <int DIM>
fr_status degrid_coils(const fr_plan *p, const tgeom &g, const float2 *grid, int C, float2 *out)
{
    constexpr int MOST = DIM == 3 ? 6 : 8;
    const int chunks = (C + MOST - 1) / MOST, nc = (C + chunks - 1) / chunks;
    if (nc == 1) return degrid<DIM, 1, 8>(p, g, grid, C, out);
    if (nc == 2) return degrid<DIM, 2, DIM == 3 ? 4 : 8>(p, g, grid, C, out);
    if (nc == 3) return degrid<DIM, 3, DIM == 3 ? 4 : 8>(p, g, grid, C, out);
    if (nc == 4) return degrid<DIM, 4, 8>(p, g, grid, C, out);
    if constexpr (DIM == 2)
        if (nc > 6) return degrid<DIM, 8, 8>(p, g, grid, C, out);
    return degrid<DIM, 6, 8>(p, g, grid, C, out);
}

template <int DIM>
fr_status density(fr_plan *p, const tgeom &g, fr_samples *s, int iters, bool ones)
{
    fr_ctx *ctx = p->ctx;
    hipStream_t st = ctx->stream;
    fr_tiles *t = p->tord;
    const int64_t M = p->M, cells = (int64_t)fr_plan_cells(p->dim, p->N, p->frames);
    constexpr int CELLS = shape<DIM>::CELLS, SUB = 64 / shape<DIM>::TAPS;
    const size_t gl = sizeof(float) * (table_floats(p->L) + WAVES * 64 * STAGED + CELLS * WAVES * SUB + 64 * WAVES);
    const size_t ul = sizeof(float) * (table_floats(p->L) + CELLS);
    auto kg = k_dens_grid<DIM>;
    auto ku = k_dens_update<DIM>;
    FR_HIP(ctx, hipFuncSetAttribute((const void *)kg, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gl));
    FR_HIP(ctx, hipFuncSetAttribute((const void *)ku, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ul));
    if (ones)
        hipLaunchKernelGGL(k_fill, dim3(nblk(M, 256)), dim3(256), 0, st, t->w, M, 1.f);
    else
        hipLaunchKernelGGL(k_to_tiles, dim3(nblk(M, 256)), dim3(256), 0, st, t->tpos, s->dcf, M, t->w);
    for (int it = 0; it < iters; ++it) {
        hipLaunchKernelGGL(kg, dim3(t->nitems), dim3(64 * WAVES), gl, st, t->items, t->tpos, t->w, g, p->tsel, p->L,
                           p->mfma_dacc, p->mfma_cidx, t->part);
        if (t->nmany > 0)
            hipLaunchKernelGGL(k_dens_slices, dim3(t->nmany, (CELLS + 63) / 64), dim3(64 * SLICE_WAVES), 0, st, t->many,
                               t->first, CELLS, t->part);
        hipLaunchKernelGGL(k_dens_combine<DIM>, dim3(nblk(cells, 256)), dim3(256), 0, st, t->part, t->first, g,
                           (uint32_t)cells, t->grid);
        hipLaunchKernelGGL(ku, dim3(t->nitems), dim3(64 * WAVES), ul, st, t->items, t->tpos, g, p->tsel, p->L,
                           p->mfma_dacc, p->mfma_cidx, t->grid, t->w);
    }
    hipLaunchKernelGGL(k_from_tiles, dim3(nblk(M, 256)), dim3(256), 0, st, t->tpos, t->w, M, s->dcf);
    FR_HIP(ctx, hipGetLastError());
    return FR_OK;
}

}  // namespace

void fr_tiles_free(fr_tiles *t)
{
    if (!t) return;
    hipFree(t->tpos);
    hipFree(t->items);
    hipFree(t->first);
    hipFree(t->many);
    hipFree(t->part);
    hipFree(t->grid);
    hipFree(t->w);
    delete t;
}

bool fr_tiles_fit(const fr_plan *p, const fr_samples *s)
{
    return p->accumulate == FR_ACC_POS && p->pos && p->tsel && p->kHW <= 2.f && p->M > 0 && s->uid == p->traj_uid &&
           s->traj_version == p->traj_version;
}

fr_status fr_tiles_build(fr_plan *p)
{
    if (p->tord) return FR_OK;
    fr_tiles *t = new (std::nothrow) fr_tiles;
    if (!t) return FR_ERR_NOMEM;
    const tgeom g = geom_of(p);
    const fr_status e = p->dim == 3 ? build<3>(p, t, g) : build<2>(p, t, g);
    if (e) {
        hipStreamSynchronize(p->ctx->stream);
        fr_tiles_free(t);
        return e;
    }
    p->tord = t;
    return FR_OK;
}

fr_status fr_tile_degrid(const fr_plan *p, const float2 *grid, int C, float2 *out)
{
    const tgeom g = geom_of(p);
    return p->dim == 3 ? degrid_coils<3>(p, g, grid, C, out) : degrid_coils<2>(p, g, grid, C, out);
}

fr_status fr_tile_density(fr_plan *p, fr_samples *s, int iters, bool ones)
{
    fr_ctx *ctx = p->ctx;
    fr_status e = fr_tiles_build(p);
    if (e) return e;
    fr_tiles *t = p->tord;
    const size_t box = p->dim == 3 ? shape<3>::CELLS : shape<2>::CELLS;
    if ((!t->w && (e = fr_alloc(ctx, (void **)&t->w, sizeof(float) * p->M))) ||
        (!t->grid &&
         (e = fr_alloc(ctx, (void **)&t->grid, sizeof(float) * fr_plan_cells(p->dim, p->N, p->frames)))) ||
        (!t->part && (e = fr_alloc(ctx, (void **)&t->part, sizeof(float) * box * t->nitems)))) {
        hipFree(t->w);                          // all of it for the general path
        hipFree(t->grid);
        t->w = t->grid = nullptr;
        return e;
    }
    const tgeom g = geom_of(p);
    return p->dim == 3 ? density<3>(p, g, s, iters, ones) : density<2>(p, g, s, iters, ones);
}
