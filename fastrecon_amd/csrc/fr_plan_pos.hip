// Gridding plan of the position-weight matrix-core mode (FR_ACC_POS).
//
// Replaces cuGridLut::plan (ReconData/cuGridLut.cu:151-226) for this mode.
// The grid is tiled by fixed boxes of at most 16 cells (4 x 2 x 2 by
// default; 8 x 2 in 2D and for batched frames, one frame deep).  For every
// box the plan lists the samples with at least one accepted tap in it
// (tap test of GridLut.cpp:99-136), in ascending sample order, padded to a
// multiple of FR_POS_BATCH (16) with the null sample M.  No taps are stored: the gridding
// kernel recomputes each weight from the sample position.
//
// Everything runs on the device; the host reads two small totals.
//   1. positions and per-sample record counts, and their scan;
//   2. (box, sample) pairs in sample order, stable-sorted by box; the ends of
//      each box's run give its count;
//   3. box order: boxes with more than a quarter slice of records first,
//      heaviest first, then Morton order (a radix sort of the boxes);
//   4. per-box padded offsets, item and slot counts (one scan of all five);
//   5. the sorted samples placed at their boxes' padded offsets;
//   6. items: each box's records cut into slices of at most S records
//      (a multiple of 16); boxes with several slices write partial sums to
//      scratch slots, combined afterwards in slice order (k_combine);
//   7. tiles: the light boxes grouped by TW x-adjacent boxes, in Morton
//      order of the tiles: pairs (TW = 2, the default), which a wave grids
//      one after the other and writes out in rows of two units (64 bytes for
//      4-cell-wide units), or fours (TW = 4), which a workgroup grids and
//      writes out in whole rows.
//
// What bounds it is the traffic of the R records (the sort's three passes,
// 8 bytes in and out a record each) once the allocations are out of the way:
// all device memory comes from the context's pool.  At 3.84 million samples
// on 192^3 (30.2 million records, 442,368 boxes): 12 ms before, of which 2.7
// in kernels and the rest in some 45 calls each of hipMalloc and hipFree;
// 1.75 ms now.  Sorting by box and taking the counts from the sorted runs
// spares a count of the boxes in advance (a hash table in LDS, then atomics).
#include "fr_internal.h"
#include "fr_taps.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

namespace {

struct pgeom {
    float hw;
    int L, dim, N, frames;
    int bx, by, bz;
    int nbx, nby, nbz;
    float dacc;                 // least rejected squared distance
    int bits;                   // bits of one axis' box index in a Morton code
};

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// pieces of one block of the context's pool, each aligned to 256 bytes
struct chunk {
    fr_ctx *ctx;
    char *p = nullptr;
    size_t used = 0;
    explicit chunk(fr_ctx *c) : ctx(c) {}
    ~chunk() { fr_pool_free(ctx, p); }
    size_t add(size_t bytes)
    {
        const size_t at = used;
        used += (bytes + 255) & ~size_t(255);
        return at;
    }
    fr_status alloc() { return fr_pool_alloc(ctx, (void **)&p, used); }
    template <typename T>
    T *at(size_t off) const { return (T *)(p + off); }
};

// least fl((x - c)^2) over the cells [a, b], a <= b
__device__ __forceinline__ float least_d2(float c, int a, int b)
{
    const int f = min(max((int)floorf(c), a), b), g = min(f + 1, b);
    const float p = __fsub_rn((float)f, c), q = __fsub_rn((float)g, c);
    return fminf(__fmul_rn(p, p), __fmul_rn(q, q));
}

// f(box id, n) for the n-th box in which a sample at c has an accepted tap,
// in box order (z, y, x); returns their count.  A box holds one if its cell
// nearest along every axis does: rounding is monotone, so the nearest cell has
// the least of the reference's squared distances (dz2 + dy2) + dx2, and
// sqrtf(d2) < hw (GridLut.cpp:133) is d2 < dacc.  One comparison a box in
// place of a root for each of its cells: the counting pass 734 -> 93 us, the
// emitting one 670 -> 218 us (3.84 million samples, 192^3).
template <typename F>
__device__ __forceinline__ uint32_t sample_boxes(const float *__restrict__ traj, int64_t M, int64_t s,
                                                 const pgeom &g, F &&f)
{
    fr_box b;
    fr_sample_box(g.dim, g.N, traj, M, s, g.hw, b, g.frames);
    if (b.s[0] > b.e[0] || b.s[1] > b.e[1] || b.s[2] > b.e[2]) return 0;
    uint32_t n = 0;
    for (int Z = b.s[2] / g.bz; Z <= b.e[2] / g.bz; ++Z) {
        const float dz = least_d2(b.c[2], max(b.s[2], Z * g.bz), min(b.e[2], Z * g.bz + g.bz - 1));
        for (int Y = b.s[1] / g.by; Y <= b.e[1] / g.by; ++Y) {
            const float dzy =
                __fadd_rn(dz, least_d2(b.c[1], max(b.s[1], Y * g.by), min(b.e[1], Y * g.by + g.by - 1)));
            for (int X = b.s[0] / g.bx; X <= b.e[0] / g.bx; ++X) {
                const float d2 =
                    __fadd_rn(dzy, least_d2(b.c[0], max(b.s[0], X * g.bx), min(b.e[0], X * g.bx + g.bx - 1)));
                if (d2 < g.dacc) {
                    f(((uint32_t)Z * g.nby + Y) * g.nbx + X, n);
                    ++n;
                }
            }
        }
    }
    return n;
}

// Grid positions as float4 (x, y, z, 0) and the samples' record counts.  2D
// samples get z = 0 and batched frames their frame index (the box of
// fr_sample_box); entry M is the null sample, far outside the grid.
__global__ void k_positions(const float *__restrict__ traj, int64_t M, pgeom g, float4 *__restrict__ pos,
                            uint32_t *__restrict__ nrec)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > M) return;
    if (i == M) {
        pos[i] = make_float4(3e30f, 3e30f, 3e30f, 0.f);
        nrec[i] = 0u;
        return;
    }
    float z = 0.f;
    if (g.frames > 0)
        z = (float)min(max((int)traj[2 * M + i], 0), g.frames - 1);
    else if (g.dim == 3)
        z = traj[2 * M + i];
    pos[i] = make_float4(traj[i], traj[M + i], z, 0.f);     // .w: the DCF, set before each pass
    nrec[i] = sample_boxes(traj, M, i, g, [](uint32_t, uint32_t) {});
}

__global__ void k_emit(const float *__restrict__ traj, int64_t M, pgeom g, const uint64_t *__restrict__ spos,
                       uint32_t *__restrict__ keys, uint32_t *__restrict__ vals)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= M) return;
    const uint64_t p = spos[s];
    sample_boxes(traj, M, s, g, [&](uint32_t box, uint32_t n) {
        keys[p + n] = box;
        vals[p + n] = (uint32_t)s;
    });
}

// first and one past the last record of every box that has any (keys sorted)
__global__ void k_runs(const uint32_t *__restrict__ keys, int64_t R, uint32_t *__restrict__ first,
                       uint32_t *__restrict__ end)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= R) return;
    const uint32_t k = keys[r];
    if (r == 0 || keys[r - 1] != k) first[k] = (uint32_t)r;
    if (r == R - 1 || keys[r + 1] != k) end[k] = (uint32_t)(r + 1);
}

__device__ __forceinline__ uint64_t spread3(uint32_t v)
{
    uint64_t m = 0;
    for (int bit = 0; bit < 21; ++bit) m |= (uint64_t)((v >> bit) & 1u) << (3 * bit);
    return m;
}

__device__ __forceinline__ uint64_t spread2(uint32_t v)
{
    uint64_t m = 0;
    for (int bit = 0; bit < 21; ++bit) m |= (uint64_t)((v >> bit) & 1u) << (2 * bit);
    return m;
}

// Morton code of a box or tile; frame-major for batched frames, which share
// no samples.
__device__ __forceinline__ uint64_t place_code(uint32_t X, uint32_t Y, uint32_t Z, const pgeom &g)
{
    return g.frames > 0 ? ((uint64_t)Z << (2 * g.bits)) | spread2(X) | (spread2(Y) << 1)
                        : spread3(X) | (spread3(Y) << 1) | (spread3(Z) << 2);
}

// Sort key of a box: boxes above the heavy cut first, most records first;
// the rest, marked by the bit `light`, in place order.
__global__ void k_box_keys(const uint32_t *__restrict__ first, const uint32_t *__restrict__ end, int64_t nbox, pgeom g,
                           uint32_t heavy_cut, int light, uint64_t *__restrict__ key, uint32_t *__restrict__ val)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbox) return;
    const uint32_t X = (uint32_t)(b % g.nbx), Y = (uint32_t)((b / g.nbx) % g.nby), Z = (uint32_t)(b / ((int64_t)g.nbx * g.nby));
    const uint32_t c = end[b] - first[b];
    key[b] = c > heavy_cut ? (uint64_t)(0xffffffffu - c) : (uint64_t(1) << light) | place_code(X, Y, Z, g);
    val[b] = (uint32_t)b;
}

// What a unit takes, and (scanned) where it starts.  The sums stay below
// 2^32: checked on the padded record count before.
struct ustat {
    uint32_t recs;              // records, padded to FR_POS_BATCH
    uint32_t items, slots;      // items; slots of partial sums (units with several items)
    uint32_t heavy, front;      // 1: several items; more records than the heavy cut
};

struct ustat_sum {
    __host__ __device__ __forceinline__ ustat operator()(const ustat &a, const ustat &b) const
    {
        return ustat{a.recs + b.recs, a.items + b.items, a.slots + b.slots, a.heavy + b.heavy, a.front + b.front};
    }
};

// per unit, in rank order; entry nu is null, so that the scan ends with the totals
__global__ void k_unit_stats(const uint32_t *__restrict__ order, int64_t nu, const uint32_t *__restrict__ first,
                             const uint32_t *__restrict__ end, uint32_t S, uint32_t heavy_cut, ustat *__restrict__ us)
{
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u > nu) return;
    if (u == nu) {
        us[u] = ustat{0u, 0u, 0u, 0u, 0u};
        return;
    }
    const uint32_t b = order[u];
    const uint32_t c = end[b] - first[b], c4 = (c + (FR_POS_BATCH - 1)) & ~(uint32_t)(FR_POS_BATCH - 1);
    const uint32_t nit = c4 == 0 ? 1u : (c4 + S - 1) / S;
    us[u] = ustat{c4, nit, nit > 1 ? nit : 0u, nit > 1, c > heavy_cut};
}

struct totals {
    ustat sum;
    uint32_t front_items;
};

__global__ void k_totals(int64_t nu, const ustat *__restrict__ at, totals *__restrict__ t)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    t->sum = at[nu];
    t->front_items = at[at[nu].front].items;        // front units rank first
}

// unit records, their items and heavy entries, their padding (null sample M)
// and shift[box]: what added to a record's rank in box order gives its place
__global__ void k_units(const uint32_t *__restrict__ order, int64_t nu, pgeom g, uint32_t S, uint32_t null_sample,
                        const uint32_t *__restrict__ first, const uint32_t *__restrict__ end,
                        const ustat *__restrict__ us, const ustat *__restrict__ at, uint32_t *__restrict__ shift,
                        fr_unit *__restrict__ units, fr_item *__restrict__ items, fr_heavy *__restrict__ heavy,
                        uint32_t *__restrict__ recs)
{
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u < FR_POS_PAD) recs[at[nu].recs + u] = null_sample;
    if (u >= nu) return;
    const int64_t b = order[u];
    const int X = (int)(b % g.nbx), Y = (int)((b / g.nbx) % g.nby), Z = (int)(b / ((int64_t)g.nbx * g.nby));
    const int ox = X * g.bx, oy = Y * g.by, oz = Z * g.bz;
    const int ux = min(g.bx, g.N - ox), uy = min(g.by, g.N - oy);
    const int uz = g.dim == 3 && g.frames == 0 ? min(g.bz, g.N - oz) : 1;
    const uint32_t c = end[b] - first[b], c4 = us[u].recs, nit = us[u].items;
    const ustat p = at[u];
    shift[b] = p.recs - first[b];
    units[u] = fr_unit{ox, oy, oz, ux | (uy << 8) | (uz << 16), p.recs, 0, c4, c};
    for (uint32_t i = c; i < c4; ++i) recs[p.recs + i] = null_sample;
    // the unit's box travels with its items (the kernel reads no unit record)
    const uint32_t box0 = (uint32_t)ox | ((uint32_t)oy << 16);
    const uint32_t box1 = (uint32_t)oz | (((uint32_t)ux | ((uint32_t)uy << 5) | ((uint32_t)uz << 10)) << 16);
    for (uint32_t q = 0; q < nit; ++q) {
        const uint32_t r0 = p.recs + q * S, end = p.recs + c4;
        const uint32_t r1 = r0 + min(S, end - r0);
        items[p.items + q] = fr_item{(uint32_t)u, nit > 1 ? (int32_t)(p.slots + q) : -1, r0, r1, box0, box1};
    }
    if (nit > 1) heavy[p.heavy] = fr_heavy{(uint32_t)u, nit, p.slots, 0u};
}

__global__ void k_place(const uint32_t *__restrict__ keys, const uint32_t *__restrict__ vals, int64_t R,
                        const uint32_t *__restrict__ shift, uint32_t *__restrict__ recs)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < R) recs[shift[keys[r]] + (uint32_t)r] = vals[r];
}

// Tiles: TW x-adjacent units, in place order of the tile coordinates.
__global__ void k_tile_keys(int64_t ntiles, int ntx, pgeom g, uint64_t *__restrict__ key, uint32_t *__restrict__ val)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntiles) return;
    const uint32_t X = (uint32_t)(t % ntx), Y = (uint32_t)((t / ntx) % g.nby),
                   Z = (uint32_t)(t / ((int64_t)ntx * g.nby));
    key[t] = place_code(X, Y, Z, g);
    val[t] = (uint32_t)t;
}

// tiles in launch order: box and no items yet; tpos = inverse permutation
__global__ void k_tile_init(const uint32_t *__restrict__ torder, int64_t ntiles, int ntx, int nty, pgeom g, int tw,
                            fr_tile *__restrict__ tiles, uint32_t *__restrict__ tpos)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ntiles) return;
    const uint32_t t = torder[q];
    tpos[t] = (uint32_t)q;
    const uint32_t X = t % ntx, Y = (t / ntx) % nty, Z = t / (ntx * nty);
    tiles[q] = fr_tile{{-1, -1, -1, -1}, (X * tw * g.bx) | ((Y * g.by) << 16), Z * g.bz};
}

// every light unit's (single) item into its tile slot
__global__ void k_tile_fill(const uint32_t *__restrict__ order, int64_t nu, int64_t nfront_units, pgeom g, int ntx, int tw,
                            const uint32_t *__restrict__ tpos, const ustat *__restrict__ at,
                            fr_tile *__restrict__ tiles)
{
    const int64_t u = nfront_units + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nu) return;
    const int64_t b = order[u];
    const uint32_t X = (uint32_t)(b % g.nbx), Y = (uint32_t)((b / g.nbx) % g.nby),
                   Z = (uint32_t)(b / ((int64_t)g.nbx * g.nby));
    const uint32_t t = (Z * g.nby + Y) * ntx + X / tw;
    tiles[tpos[t]].item[X % tw] = (int32_t)at[u].items;
}

}  // namespace

fr_status fr_plan_build_pos(fr_plan *p, const fr_samples *s, const fr_tune *tune)
{
    fr_ctx *ctx = p->ctx;
    hipStream_t st = ctx->stream;
    auto t0 = std::chrono::steady_clock::now();
    const int N = (int)p->N;
    const int64_t M = s->M;
    FR_CHECK(ctx, p->L <= FR_POS_MAX_L, FR_ERR_UNSUPPORTED,
             "position-weight gridding (accumulate 6) takes LUTs of at most %d entries (have %d)", FR_POS_MAX_L, p->L);
    FR_CHECK(ctx, !(tune && tune->exact_order), FR_ERR_INVALID,
             "exact_order needs a sequential accumulation mode (1, 2 or 4); the matrix cores sum four products at "
             "a time");

    // unit box: 4 x 2 x 2 in 3D; 8 x 2 in 2D and per frame (the 64 uneven
    // spiral frames on 384^2: 1.01 ms against 1.12 with 4 x 4; the 402-spoke
    // radial case on 512^2 is the same with both)
    fr_geom geom{};
    geom.dim = p->dim;
    geom.N = N;
    const bool flat = p->dim == 2;
    geom.bx = flat ? 8 : 4;
    geom.by = 2;
    geom.bz = flat ? 1 : 2;
    if (tune) {
        if (tune->tile_x > 0) geom.bx = tune->tile_x;
        if (tune->tile_y > 0) geom.by = tune->tile_y;
        if (!flat && tune->tile_z > 0) geom.bz = tune->tile_z;
    }
    geom.bx = std::min(geom.bx, N);
    geom.by = std::min(geom.by, N);
    geom.bz = flat ? 1 : std::min(geom.bz, N);
    geom.cells_max = geom.bx * geom.by * geom.bz;
    geom.waves = FR_POS_WAVES;
    FR_CHECK(ctx, geom.bx >= 1 && geom.by >= 1 && geom.bz >= 1 && geom.cells_max <= 16, FR_ERR_INVALID,
             "position-weight gridding (accumulate 6) takes unit boxes of at most 16 cells (have %dx%dx%d)",
             geom.bx, geom.by, geom.bz);
    p->geom = geom;
    p->accumulate = FR_ACC_POS;
    p->exact_order = 0;
    // defaults measured on the 32-coil 256^3 kooshball (4.70 ms with pairs;
    // 4.95 unit by unit, 5.41 with tiles of four; streaming stores slower)
    p->pos_ipw = 1;
    p->xcd_run = 256;
    p->pos_stores = 2;
    p->pos_waves = 4;
    if (tune && tune->items_per_wave > 0) p->pos_ipw = tune->items_per_wave;
    if (tune && tune->xcd_run > 0) p->xcd_run = tune->xcd_run;
    if (tune && tune->stores > 0) p->pos_stores = tune->stores;
    if (tune && tune->waves_per_simd > 0) p->pos_waves = tune->waves_per_simd;
    const int tile_writes = tune ? tune->tile_writes : 0;
    FR_CHECK(ctx, tile_writes >= 0 && tile_writes <= 3, FR_ERR_INVALID, "tile_writes %d out of range", tile_writes);
    FR_CHECK(ctx, (p->pos_stores == 1 || p->pos_stores == 2) && (p->pos_waves == 3 || p->pos_waves == 4),
             FR_ERR_INVALID, "stores %d / waves_per_simd %d out of range", p->pos_stores, p->pos_waves);
    FR_CHECK(ctx, p->pos_ipw <= 64 && p->xcd_run <= (1 << 20), FR_ERR_INVALID, "items_per_wave %d / xcd_run %d "
             "out of range", p->pos_ipw, p->xcd_run);

    fr_status e = fr_plan_thresholds(p, true);
    if (e) return e;

    pgeom g{p->kHW, p->L, p->dim, N, p->frames, geom.bx, geom.by, geom.bz, 0, 0, 0, p->mfma_dacc, 0};
    g.nbx = (N + geom.bx - 1) / geom.bx;
    g.nby = (N + geom.by - 1) / geom.by;
    g.nbz = p->frames > 0 ? p->frames : (flat ? 1 : (N + geom.bz - 1) / geom.bz);
    const int64_t nbox = (int64_t)g.nbx * g.nby * g.nbz;
    FR_CHECK(ctx, nbox < (int64_t(1) << 31), FR_ERR_UNSUPPORTED, "%lld unit boxes", (long long)nbox);
    FR_CHECK(ctx, N <= 65535 && g.nbz * geom.bz <= 65535, FR_ERR_UNSUPPORTED, "grid too large for packed unit boxes");
    // bits of a Morton code: of the boxes along an axis (frames go above them)
    const int axis = std::max({g.nbx, g.nby, p->frames > 0 ? 1 : g.nbz});
    while ((1 << g.bits) < axis) ++g.bits;
    int code_bits = (p->frames > 0 ? 2 : 3) * g.bits;
    for (int f = 1; p->frames > f; f *= 2) ++code_bits;
    code_bits = std::max(1, code_bits);
    int box_bits = 1;
    while (box_bits < 32 && (int64_t(1) << box_bits) < nbox) ++box_bits;
    const int light = std::max(32, code_bits);
    const int64_t nu = nbox;

    // scratch whose size the samples and boxes give
    size_t scan_bytes = 0, sort_bytes = 0, stat_bytes = 0;
    using wide = hipcub::TransformInputIterator<uint64_t, hipcub::CastOp<uint64_t>, const uint32_t *>;
    FR_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, wide(nullptr, hipcub::CastOp<uint64_t>()),
                                                 (uint64_t *)nullptr, (int)(M + 1), st));
    hipcub::DoubleBuffer<uint64_t> bkey(nullptr, nullptr);
    hipcub::DoubleBuffer<uint32_t> bval(nullptr, nullptr);
    FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, bkey, bval, (int)nbox, 0, light + 1, st));
    FR_HIP(ctx, hipcub::DeviceScan::ExclusiveScan(nullptr, stat_bytes, (ustat *)nullptr, (ustat *)nullptr, ustat_sum(),
                                                  ustat{}, (int)(nu + 1), st));
    const size_t tmp_bytes = std::max({scan_bytes, sort_bytes, stat_bytes}) + 256;
    chunk w(ctx);
    const size_t o_nrec = w.add(4 * (M + 1)), o_spos = w.add(8 * (M + 1)), o_first = w.add(8 * nbox);
    const size_t o_k0 = w.add(8 * nbox), o_k1 = w.add(8 * nbox), o_v0 = w.add(4 * nbox), o_v1 = w.add(4 * nbox);
    const size_t o_us = w.add(sizeof(ustat) * (nu + 1)), o_at = w.add(sizeof(ustat) * (nu + 1));
    const size_t o_shift = w.add(4 * nbox), o_tot = w.add(sizeof(totals)), o_tmp = w.add(tmp_bytes);
    if ((e = w.alloc()) || (e = fr_pool_alloc(ctx, (void **)&p->pos, sizeof(float4) * (M + 1)))) return e;
    uint32_t *nrec = w.at<uint32_t>(o_nrec), *first = w.at<uint32_t>(o_first), *end = first + nbox;
    uint64_t *spos = w.at<uint64_t>(o_spos);
    void *tmp = w.at<char>(o_tmp);

    // 1. positions (entry M: the null sample) and counts
    hipLaunchKernelGGL(k_positions, dim3(nblk(M + 1, 256)), dim3(256), 0, st, s->traj, M, g, p->pos, nrec);
    FR_HIP(ctx, hipMemsetAsync(first, 0, 8 * nbox, st));
    FR_HIP(ctx, hipGetLastError());
    size_t bytes = tmp_bytes;
    FR_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(tmp, bytes, wide(nrec, hipcub::CastOp<uint64_t>()), spos, (int)(M + 1),
                                                 st));
    uint64_t R = 0;
    FR_HIP(ctx, hipMemcpyAsync(&R, spos + M, 8, hipMemcpyDeviceToHost, st));
    FR_HIP(ctx, hipStreamSynchronize(st));
    // Sorts take below 2^31 records, and the padded ones (a box without any
    // takes none) are counted in 32 bits.
    const uint64_t padded = R + (FR_POS_BATCH - 1) * std::min<uint64_t>(R, nbox) + FR_POS_PAD;
    FR_CHECK(ctx, R + 4 * (uint64_t)nbox + 64 < (uint64_t(1) << 31) && padded < (uint64_t(1) << 32), FR_ERR_UNSUPPORTED,
             "plan has %llu records (max about 2^31)", (unsigned long long)R);

    // slice size S (records, a multiple of 16): about 32 slices' worth of
    // work per CU, at least 64 and at most 16384 (the 384^3 FP16 kooshball's
    // 300M records would give 36,600: 16384 grids it 3% faster; the 256^3
    // kooshball's 12,600 stays)
    const int cus = std::max(1, ctx->cu_count);
    uint64_t S = std::min<uint64_t>(16384, std::max<uint64_t>(64, R / ((uint64_t)cus * 32)));
    if (tune && tune->split_taps > 0) S = (uint64_t)tune->split_taps;
    // (at most 2^25: the gridding kernel counts a wave's records in 32-bit
    // byte offsets, of a slice or of up to 64 units below the heavy cut)
    S = std::min<uint64_t>((S + 15) / 16 * 16, uint64_t(1) << 25);
    const uint32_t heavy_cut = (uint32_t)std::max<uint64_t>(4, S / 4);

    // 2. records by box, in sample order
    chunk rw(ctx);
    hipcub::DoubleBuffer<uint32_t> rkey(nullptr, nullptr), rval(nullptr, nullptr);
    if (R > 0) {
        size_t need = 0;
        FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, need, rkey, rval, (int)R, 0, box_bits, st));
        const size_t o0 = rw.add(4 * R), o1 = rw.add(4 * R), o2 = rw.add(4 * R), o3 = rw.add(4 * R),
                     o4 = rw.add(need + 256);
        if ((e = rw.alloc())) return e;
        rkey = hipcub::DoubleBuffer<uint32_t>(rw.at<uint32_t>(o0), rw.at<uint32_t>(o1));
        rval = hipcub::DoubleBuffer<uint32_t>(rw.at<uint32_t>(o2), rw.at<uint32_t>(o3));
        hipLaunchKernelGGL(k_emit, dim3(nblk(M, 256)), dim3(256), 0, st, s->traj, M, g, spos, rkey.Current(),
                           rval.Current());
        FR_HIP(ctx, hipGetLastError());
        FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(rw.at<char>(o4), need, rkey, rval, (int)R, 0, box_bits, st));
        hipLaunchKernelGGL(k_runs, dim3(nblk((int64_t)R, 256)), dim3(256), 0, st, rkey.Current(), (int64_t)R, first,
                           end);
    }

    // 3. box order
    bkey = hipcub::DoubleBuffer<uint64_t>(w.at<uint64_t>(o_k0), w.at<uint64_t>(o_k1));
    bval = hipcub::DoubleBuffer<uint32_t>(w.at<uint32_t>(o_v0), w.at<uint32_t>(o_v1));
    hipLaunchKernelGGL(k_box_keys, dim3(nblk(nbox, 256)), dim3(256), 0, st, first, end, nbox, g, heavy_cut, light,
                       bkey.Current(), bval.Current());
    FR_HIP(ctx, hipGetLastError());
    bytes = tmp_bytes;
    FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(tmp, bytes, bkey, bval, (int)nbox, 0, light + 1, st));
    const uint32_t *order = bval.Current();

    // 4. what the units take and where they start
    ustat *us = w.at<ustat>(o_us), *at = w.at<ustat>(o_at);
    hipLaunchKernelGGL(k_unit_stats, dim3(nblk(nu + 1, 256)), dim3(256), 0, st, order, nu, first, end, (uint32_t)S,
                       heavy_cut, us);
    FR_HIP(ctx, hipGetLastError());
    bytes = tmp_bytes;
    FR_HIP(ctx, hipcub::DeviceScan::ExclusiveScan(tmp, bytes, us, at, ustat_sum(), ustat{}, (int)(nu + 1), st));
    totals *tot_d = w.at<totals>(o_tot);
    hipLaunchKernelGGL(k_totals, dim3(1), dim3(64), 0, st, nu, at, tot_d);
    totals tot{};
    FR_HIP(ctx, hipMemcpyAsync(&tot, tot_d, sizeof(totals), hipMemcpyDeviceToHost, st));
    FR_HIP(ctx, hipStreamSynchronize(st));

    // 5., 6. units, items, heavy units and records
    p->nunits = nu;
    p->nrecords = (int64_t)R;
    p->nrecs_padded = (int64_t)tot.sum.recs;
    p->nitems = (int64_t)tot.sum.items;
    p->nitems_front = (int64_t)tot.front_items;
    p->nheavy = (int64_t)tot.sum.heavy;
    p->nslots = (int64_t)tot.sum.slots;
    if ((e = fr_pool_alloc(ctx, (void **)&p->units, sizeof(fr_unit) * nu)) ||
        (e = fr_pool_alloc(ctx, (void **)&p->recs, sizeof(uint32_t) * ((size_t)tot.sum.recs + FR_POS_PAD))) ||
        (e = fr_pool_alloc(ctx, (void **)&p->items, sizeof(fr_item) * std::max<size_t>(1, tot.sum.items))) ||
        (e = fr_pool_alloc(ctx, (void **)&p->heavy, sizeof(fr_heavy) * std::max<size_t>(1, tot.sum.heavy))))
        return e;
    uint32_t *shift = w.at<uint32_t>(o_shift);
    hipLaunchKernelGGL(k_units, dim3(nblk(std::max<int64_t>(nu, FR_POS_PAD), 256)), dim3(256), 0, st, order, nu, g,
                       (uint32_t)S, (uint32_t)M, first, end, us, at, shift, p->units, p->items, p->heavy, p->recs);
    if (R > 0)
        hipLaunchKernelGGL(k_place, dim3(nblk((int64_t)R, 256)), dim3(256), 0, st, rkey.Current(), rval.Current(),
                           (int64_t)R, shift, p->recs);
    FR_HIP(ctx, hipGetLastError());

    // 7. tiles of TW x-adjacent whole units (unit box of 16 cells with
    // power-of-two sides; the grid divides into whole tiles): pairs by
    // default (tile_writes 0 or 3), rows of 2 bx cells; fours with
    // tile_writes 1, rows of 4 bx cells; none with tile_writes 2
    const bool pow2 = (geom.bx & (geom.bx - 1)) == 0 && (geom.by & (geom.by - 1)) == 0 &&
                      (geom.bz & (geom.bz - 1)) == 0;
    const int TW = tile_writes == 1 ? FR_POS_WAVES : (tile_writes == 2 ? 0 : 2);
    p->ntiles = 0;
    p->tile_units = 0;
    if (TW > 0 && pow2 && geom.cells_max == 16 && N % (TW * geom.bx) == 0 && N % geom.by == 0 &&
        (flat || N % geom.bz == 0) && nu > (int64_t)tot.sum.front) {
        const int ntx = g.nbx / TW;
        const int64_t ntiles = (int64_t)ntx * g.nby * g.nbz, nfront = tot.sum.front;
        // the keys and values of the boxes' sort are free again but for `order`
        hipcub::DoubleBuffer<uint64_t> tkey(bkey.Current(), bkey.Alternate());
        chunk tw(ctx);
        const size_t o0 = tw.add(4 * ntiles), o1 = tw.add(4 * ntiles), o2 = tw.add(4 * ntiles);
        if ((e = tw.alloc()) || (e = fr_pool_alloc(ctx, (void **)&p->tiles, sizeof(fr_tile) * ntiles))) return e;
        hipcub::DoubleBuffer<uint32_t> tval(tw.at<uint32_t>(o0), tw.at<uint32_t>(o1));
        uint32_t *tpos = tw.at<uint32_t>(o2);
        hipLaunchKernelGGL(k_tile_keys, dim3(nblk(ntiles, 256)), dim3(256), 0, st, ntiles, ntx, g, tkey.Current(),
                           tval.Current());
        bytes = 0;
        FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, tkey, tval, (int)ntiles, 0, code_bits, st));
        chunk ts(ctx);
        ts.add(bytes + 256);
        if ((e = ts.alloc())) return e;
        FR_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ts.p, bytes, tkey, tval, (int)ntiles, 0, code_bits, st));
        hipLaunchKernelGGL(k_tile_init, dim3(nblk(ntiles, 256)), dim3(256), 0, st, tval.Current(), ntiles, ntx, g.nby,
                           g, TW, p->tiles, tpos);
        hipLaunchKernelGGL(k_tile_fill, dim3(nblk(nu - nfront, 256)), dim3(256), 0, st, order, nu, nfront, g, ntx, TW,
                           tpos, at, p->tiles);
        FR_HIP(ctx, hipGetLastError());
        p->ntiles = ntiles;
        p->tile_units = TW;
    }
    FR_HIP(ctx, hipStreamSynchronize(st));
    p->max_unit_taps = 0;
    p->ntaps = 0;
    p->build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return FR_OK;
}
