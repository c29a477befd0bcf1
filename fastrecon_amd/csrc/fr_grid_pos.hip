// Gridding on the matrix cores with tap weights computed from the sample
// positions (accumulate mode FR_ACC_POS, the default for plans that are not
// exact-order).
//
// A unit is a box of at most 16 cells (4 x 2 x 2 by default, the most
// compact 16-cell box: a radius-2 kernel ball meets about 8 such boxes per
// sample, against 10 for 8 x 2 x 1).  The plan lists, per unit, the samples
// that have at least one accepted tap in it (ascending sample order, padded
// to a multiple of 16 with a null sample).  Four records at a time are one
// dense product per 16 components
//
//     acc[16 cells][16 components] += A[16 cells][4 records] * B[4 records][16 components]
//
// on v_mfma_f32_16x16x4_f32, with
//   A[i][k] = LUT weight of record k's sample at cell i, 0 where the sample
//             has no tap there: computed here, lane (i, k) evaluating the
//             reference tap test and LUT index for its own cell;
//   B[k][j] = dcf * sample component j of record k (GridLut.cpp:109); the
//             DCF travels in the .w of the record's position entry, which
//             k_pos_dcf refreshes from the samples before every pass.
//
// Tap test and LUT index (GridLut.cpp:112-136) without the reference's
// correctly rounded square root and division: the squared distance d2 is
// formed with the reference's FP32 operations in its order ((dz*dz + dy*dy)
// + dx*dx); the tap is accepted iff d2 < dacc, the least d2 whose sqrtf is >=
// hw; the reference index roundf(sqrtf(d2) / hw * (L - 1)) is monotone in d2,
// so with B[m] = least d2 whose index is >= m (computed on the host with the
// reference arithmetic) the index is the m with B[m] <= d2 < B[m + 1].  An
// estimate e = floor(sqrt~(d2) * (L - 1) / hw + 0.49) from the hardware's
// 1-ulp square root is the index or one below it, so one comparison with
// B[e + 1] selects LUT[e] or LUT[e + 1] from the table entry (B[e + 1],
// LUT[e], LUT[e + 1]).  Every tap set and LUT index is the reference's; only
// the order of the sum over samples differs (four products per matrix
// instruction), so results agree with the CPU loop to FP32 rounding and are
// deterministic.
//
// Cells a sample does not tap get weight 0, so a NaN or Inf sample value
// spreads to the other cells of the units it touches (0 * NaN), unlike the
// reference, which leaves those cells alone.
//
// Lane layout of v_mfma_f32_16x16x4_f32 (wave64): lane l supplies A[l % 16][l
// / 16] and B[l / 16][l % 16]; accumulator register r of lane l holds
// D[4 (l / 16) + r][l % 16].  Lane l evaluates cell l % 16 for record l / 16
// of a group, and holds component slice l % 16: with NCB component blocks,
// components [NCB j, NCB j + NCB) of a chunk of 8 NCB coils.
#include "fr_internal.h"
#include "fr_taps.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int RB = 16;               // records per batch: four groups of four
constexpr int PW = FR_POS_WAVES;     // waves per workgroup
constexpr int CS = 17;               // LDS row stride of the write-out transpose (16 cells + 1)
constexpr int PS = 68;               // and of a pair's (32 cells of a coil, + 16 bytes)
// the pipeline reads record indices up to 191 past a batch's first
static_assert(3 * 64 <= FR_POS_PAD, "record padding");

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float2 ld_coil(const float2 *__restrict__ row, int c) { return row[c]; }
__device__ __forceinline__ float2 ld_coil(const __half2 *__restrict__ row, int c) { return __half22float2(row[c]); }
__device__ __forceinline__ float4 ld_pair(const float2 *__restrict__ row, int c)
{
    return *reinterpret_cast<const float4 *>(row + c);
}
__device__ __forceinline__ float4 ld_pair(const __half2 *__restrict__ row, int c)
{
    const uint2 u = *reinterpret_cast<const uint2 *>(row + c);
    const float2 a = __half22float2(*reinterpret_cast<const __half2 *>(&u.x));
    const float2 b = __half22float2(*reinterpret_cast<const __half2 *>(&u.y));
    return make_float4(a.x, a.y, b.x, b.y);
}

// element at a 32-bit byte offset from a uniform base: positions (at most 2^27
// samples, 2 GiB), or the records of a stream, from its first one on (a plan's
// records take up to 16 GiB)
template <typename E>
__device__ __forceinline__ E ld_off(const E *__restrict__ base, uint32_t byte_off)
{
    return *reinterpret_cast<const E *>(reinterpret_cast<const char *>(base) + byte_off);
}

// The rows of one batch of RB records in flight: lane (j, k) holds its
// component slice of group q's record 4 q + k.
struct batch_rows {
    float2 a[4], b[4];
};

// Rows of the batch whose samples lanes 16 s .. 16 s + 15 hold: in `at`, the
// byte offset of a sample's row (SMALL: the data is below 4 GiB; one 32-bit
// addition per load in place of a 64-bit product and sum) or its index.
template <int NCB, bool PAIR, bool SMALL, typename TS>
__device__ __forceinline__ void issue_rows(batch_rows &S, uint32_t at, int s, const TS *__restrict__ data, uint32_t C,
                                           int ca, int cbb, int k)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t m = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (16 * s + 4 * q + k), (int)at);
        if constexpr (SMALL) {
            const uint32_t o = m + (uint32_t)(ca * (int)sizeof(TS));
            if constexpr (NCB == 4 && PAIR) {
                const float4 v = ld_pair(reinterpret_cast<const TS *>(reinterpret_cast<const char *>(data) + o), 0);
                S.a[q] = make_float2(v.x, v.y);
                S.b[q] = make_float2(v.z, v.w);
            } else {
                S.a[q] = ld_coil(reinterpret_cast<const TS *>(reinterpret_cast<const char *>(data) + o), 0);
                if constexpr (NCB == 4)
                    S.b[q] = ld_coil(reinterpret_cast<const TS *>(reinterpret_cast<const char *>(data) +
                                                                  (m + (uint32_t)(cbb * (int)sizeof(TS)))), 0);
            }
        } else {
            const TS *row = data + (uint64_t)m * C;
            if constexpr (NCB == 4 && PAIR) {
                const float4 v = ld_pair(row, ca);
                S.a[q] = make_float2(v.x, v.y);
                S.b[q] = make_float2(v.z, v.w);
            } else {
                S.a[q] = ld_coil(row, ca);
                if constexpr (NCB == 4) S.b[q] = ld_coil(row, cbb);
            }
        }
    }
}

// Weight of the lane's cell for a sample at p: the reference tap test and
// LUT index through the selection table (file comment).
__device__ __forceinline__ float tap_weight(const float4 &p, const float4 *stbl, float fx, float fy, float fz,
                                            float cidx, float lmax)
{
    // d2 with the reference's operations and order (GridLut.cpp:120-131)
    const float dz = __fsub_rn(fz, p.z);
    const float dy = __fsub_rn(fy, p.y);
    const float dx = __fsub_rn(fx, p.x);
    return fr_tap_weight(fr_tap_dk2(__fmul_rn(dz, dz), __fmul_rn(dy, dy), dx), stbl, cidx, lmax);
}

// B = dcf * sample (GridLut.cpp:109).  Columns past the chunk's coils repeat
// its last coil; their sums are not written.
template <int NCB>
__device__ __forceinline__ void b_values(float (&bv)[NCB], float w, float2 a, float2 b, int j)
{
    if constexpr (NCB == 4) {
        bv[0] = __fmul_rn(w, a.x); bv[1] = __fmul_rn(w, a.y);
        bv[2] = __fmul_rn(w, b.x); bv[3] = __fmul_rn(w, b.y);
    } else if constexpr (NCB == 2) {
        bv[0] = __fmul_rn(w, a.x); bv[1] = __fmul_rn(w, a.y);
    } else {
        bv[0] = __fmul_rn(w, (j & 1) ? a.y : a.x);
    }
}

// Apply the four groups of one batch, its positions and DCFs in pb[0 .. 15].
// The null sample (index M) sits far outside the grid with DCF 0 and a zero
// row, so padding records add exact zeros.  The four weight computations are
// independent (their table reads overlap); the matrix instructions then cycle
// through the NCB accumulators.
template <int NCB>
__device__ __forceinline__ void apply_batch(f4 (&acc)[NCB], const batch_rows &S, const float4 *pb, const float4 *stbl,
                                            float fx, float fy, float fz, float cidx, float lmax, int j, int k)
{
    float aw[4], w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 p = pb[4 * q + k];
        w[q] = p.w;
        aw[q] = tap_weight(p, stbl, fx, fy, fz, cidx, lmax);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float bv[NCB];
        b_values<NCB>(bv, w[q], S.a[q], S.b[q], j);
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) acc[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(aw[q], bv[cb], acc[cb], 0, 0, 0);
    }
}

// Lane j's cell of an item's unit box (t0 = ox | oy << 16, pad = oz | (ux |
// uy << 5 | uz << 10) << 16): cell index j, x fastest; lanes past the box's
// cells sit far away, so every tap test rejects them.
struct item_box {
    int ox, oy, oz, ux, uy, uz, ncell;
};

__device__ __forceinline__ item_box unpack_box(uint32_t b0, uint32_t b1)
{
    item_box b;
    b.ox = (int)(b0 & 0xffffu);
    b.oy = (int)(b0 >> 16);
    b.oz = (int)(b1 & 0xffffu);
    b.ux = (int)((b1 >> 16) & 31u);
    b.uy = (int)((b1 >> 21) & 31u);
    b.uz = (int)((b1 >> 26) & 31u);
    b.ncell = b.ux * b.uy * b.uz;
    return b;
}

__device__ __forceinline__ void lane_cell(const item_box &b, int j, float &fx, float &fy, float &fz)
{
    fx = fy = fz = -3e30f;
    if (j < b.ncell) {
        fx = (float)(b.ox + j % b.ux);
        fy = (float)(b.oy + (j / b.ux) % b.uy);
        fz = (float)(b.oz + j / (b.ux * b.uy));
    }
}

// Grid the records from recs[0] on into acc, batch by batch, until
// after_batch(r), called with the number of records applied so far (below
// 2^30), returns false.
//
// Records come in blocks of 64, one per lane: one load brings a block's
// sample indices and one its positions and DCFs, which go through LDS (pbuf)
// to the 16 lanes that need each; the indices reach the lanes
// that load a record's row by a lane exchange.  (Loaded where they are used,
// each by 16 lanes, positions and indices took 16 times the load
// instructions and return traffic of these.)  Software pipeline: while batch
// b is applied, batch b + 1's rows, the next block's positions and the block
// after's indices are in flight (past the last record they read the next
// records or the FR_POS_PAD padding records at the end).  Bound by the
// latency of a batch's chain (row loads, table reads, matrix products) over
// the waves that fit a SIMD, and at 32 coils by the traffic of the rows past
// L2 as well: up to 16 coils, where six waves fit instead of five (a wave's
// records and its write-out share their LDS, 80 VGPRs), 16 FP16 coils at
// 384^3 went from 7.00 to 6.7 - 6.9 ms, by the run, and 12 coils of 64 frames
// on 384^2 from 1.19 to 1.14, while a third fewer VALU instructions a weight
// (squared distances along each axis formed once a record) gained nothing: 7.01.  By
// blocks at all: 32 coils at 256^3 4.71 -> 4.13 ms (now 4.06), 16 FP16 coils
// at 384^3 7.75 -> 7.12.  Rows fetched two or three batches ahead were slower
// (the extra ones past an item's end cost as much as useful ones): 8.1 and
// 8.5 ms there.
template <int NCB, bool PAIR, bool SMALL, typename TS, typename After>
__device__ __forceinline__ void grid_stream(f4 (&acc)[NCB], const uint32_t *__restrict__ recs,
                                            const float4 *__restrict__ pos, const TS *__restrict__ data, uint32_t C,
                                            int ca, int cbb, const float4 *stbl, float4 *pbuf, float &fx, float &fy,
                                            float &fz, float cidx, float lmax, int j,
                                            int k, After after_batch)
{
    const uint32_t lane = (uint32_t)(16 * k + j);
    uint32_t r = 0;
    const uint32_t id = ld_off(recs, (r + lane) * 4u);
    uint32_t id1 = ld_off(recs, (r + 64 + lane) * 4u);
    float4 P = ld_off(pos, id * 16u);
    batch_rows S0, S1;
    auto row_at = [&](uint32_t m) __attribute__((always_inline)) { return SMALL ? m * (C * (uint32_t)sizeof(TS)) : m; };
    uint32_t at = row_at(id);
    issue_rows<NCB, PAIR, SMALL>(S0, at, 0, data, C, ca, cbb, k);
    auto apply = [&](const batch_rows &S, int s) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        apply_batch<NCB>(acc, S, pbuf + 16 * s, stbl, fx, fy, fz, cidx, lmax, j, k);
        r += RB;
    };
    while (true) {
        wave_sync();                       // the block before is no longer read
        pbuf[lane] = P;
        P = ld_off(pos, id1 * 16u);
        const uint32_t at1 = row_at(id1);
        const uint32_t id2 = ld_off(recs, (r + 128 + lane) * 4u);
        wave_sync();
#pragma unroll 1
        for (int q = 0; q < 4; q += 2) {
            issue_rows<NCB, PAIR, SMALL>(S1, at, q + 1, data, C, ca, cbb, k);
            apply(S0, q);
            if (!after_batch(r)) return;
            issue_rows<NCB, PAIR, SMALL>(S0, q == 0 ? at : at1, (q + 2) & 3, data, C, ca, cbb, k);
            apply(S1, q + 1);
            if (!after_batch(r)) return;
        }
        at = at1;
        id1 = id2;
    }
}

template <int NCB, bool PAIR, bool SMALL, typename TS>
__device__ __forceinline__ void grid_records(f4 (&acc)[NCB], uint32_t r, uint32_t r1,
                                             const uint32_t *__restrict__ recs, const float4 *__restrict__ pos,
                                             const TS *__restrict__ data, uint32_t C, int ca, int cbb,
                                             const float4 *stbl, float4 *pbuf, float fx, float fy, float fz,
                                             float cidx, float lmax, int j, int k)
{
    const uint32_t n = r1 - r;
    grid_stream<NCB, PAIR, SMALL>(acc, recs + r, pos, data, C, ca, cbb, stbl, pbuf, fx, fy, fz, cidx, lmax, j, k,
                                  [&](uint32_t q) __attribute__((always_inline)) { return q < n; });
}

// grid_records over [r, r1) with a switch at rmid (a multiple of RB): the
// records up to rmid belong to one unit, the rest to the next; at rmid the
// pipeline keeps running and on_mid() moves the lane to the next unit's
// cell (fx, fy, fz) and accumulators.
template <int NCB, bool PAIR, bool SMALL, typename TS, typename Mid>
__device__ __forceinline__ void grid_records_mid(f4 (&acc)[NCB], uint32_t r, uint32_t rmid, uint32_t r1,
                                                 const uint32_t *__restrict__ recs, const float4 *__restrict__ pos,
                                                 const TS *__restrict__ data, uint32_t C, int ca, int cbb,
                                                 const float4 *stbl, float4 *pbuf, float &fx, float &fy, float &fz,
                                                 float cidx, float lmax, int j, int k, Mid on_mid)
{
    const uint32_t mid = rmid - r, n = r1 - r;
    grid_stream<NCB, PAIR, SMALL>(acc, recs + r, pos, data, C, ca, cbb, stbl, pbuf, fx, fy, fz, cidx, lmax, j, k,
                                  [&](uint32_t q) __attribute__((always_inline)) {
                                      if (q == mid) on_mid();
                                      return q < n;
                                  });
}

// Waves a SIMD that the registers have to leave room for: of the variants for
// 4 (OCC 4) and for 3 (OCC 1), which up to 16 coils need fewer registers.
template <int NCB, int OCC>
constexpr int pos_waves()
{
    return NCB == 1 ? 6 : NCB == 2 ? (OCC == 4 ? 6 : 5) : OCC;
}

// NCB component blocks (chunks of 8 NCB coils).  PAIR: C even, so lane j's
// two coils (2j, 2j+1 of a 32-coil chunk) are one aligned 16-byte (8-byte
// for FP16) load.
//
// Three kinds of workgroup:
//  * front: one heavy-unit item per wave (a whole unit, or a slice written
//    to its scratch slot), written out by the wave;
//  * tile (when the plan has tiles): the PW waves grid the PW x-adjacent
//    units of a tile, stage their sums in LDS and store the tile in whole
//    rows of PW * bx cells (128 bytes for 4-cell-wide units);
//  * otherwise a run of ipw consecutive light items per wave, as one
//    record stream, each unit written out by its wave.
template <int NCB, bool PAIR, bool SMALL, typename TS, int OCC>
__global__ void __launch_bounds__(64 * PW) __attribute__((amdgpu_waves_per_eu(pos_waves<NCB, OCC>(), 8))) k_grid_pos(
    const fr_item *__restrict__ items, int64_t nitems, const fr_tile *__restrict__ tiles, int64_t ntiles,
    int lbx, int lby, int lbz, const uint32_t *__restrict__ recs, const float4 *__restrict__ pos,
    const float4 *__restrict__ tbl, int L, float cidx, const TS *__restrict__ data,
    int C, int N, size_t cells, float2 *__restrict__ out, float2 *__restrict__ partial,
    int64_t nslots, int cells_max, int64_t nfront, int64_t front_wg, int ipw, int64_t xr, int nt, int tw,
    int wave_floats, int osm_at, int64_t tstride, int fsub)
{
    extern __shared__ float4 smem_pos[];
    float4 *stbl = smem_pos;                                         // L entries
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    // the wave's block of positions and, after them (its LDS instructions stay
    // in order), its write-out transpose in the same place; beside them for
    // runs of items
    float4 *pbuf = smem_pos + L + wv * (wave_floats / 4);
    float *osm = reinterpret_cast<float *>(pbuf) + osm_at;
    for (int q = threadIdx.x; q < L; q += 64 * PW) stbl[q] = tbl[q];
    __syncthreads();

    const int j = lane & 15;                    // A row (cell) / B column (component slice)
    const int k = lane >> 4;                    // A column / B row (record in group)
    const int chunk = 8 * NCB;                  // coils per chunk
    const int c0 = blockIdx.y * chunk;
    const int nc = min(chunk, C - c0);
    const int cl0 = NCB == 4 ? 2 * j : (NCB == 2 ? j : j >> 1);
    const int ca = PAIR ? c0 + min(cl0, nc - 2) : c0 + min(cl0, nc - 1), cbb = c0 + min(cl0 + 1, nc - 1);
    const float lmax = (float)(L - 1);

    f4 acc[NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) acc[cb] = f4{0.f, 0.f, 0.f, 0.f};

    // Launch order: the front items first; then tiles (or runs of light
    // items) in Morton order, remapped so that each XCD (workgroups are dealt
    // to the 8 XCDs round-robin) takes runs of xr consecutive workgroups, a
    // compact patch of neighbouring units sharing samples in its L2.
    const int64_t bid = blockIdx.x;
    const int64_t rr = bid - front_wg, gg = rr / 8;
    const int64_t grp = (gg / xr) * (8 * xr) + (bid % 8) * xr + gg % xr;

    if (bid >= front_wg && ntiles > 0 && tw == PW) {
        // ---------------------------------------------------------- tile
        if (grp >= ntiles) return;              // the whole workgroup
        const fr_tile T = tiles[grp];
        // (a select, not T.item[wv]: a per-lane index would put T in scratch)
        const int32_t myitem = wv == 0 ? T.item[0] : wv == 1 ? T.item[1] : wv == 2 ? T.item[2] : T.item[3];
        const int bx = 1 << lbx, by = 1 << lby;
        const int W = PW * bx, rows = by << lbz;    // tile row length, rows per coil
        float *tb = reinterpret_cast<float *>(smem_pos + L) + PW * wave_floats;
        const int cstride = rows * W * 2 + 4;       // floats per coil (+4: fewer bank conflicts)
        if (myitem >= 0) {
            const fr_item it = items[myitem];
            float fx, fy, fz;
            lane_cell(unpack_box(it.t0, it.pad), j, fx, fy, fz);
            if (it.r0 < it.r1)
                grid_records<NCB, PAIR, SMALL>(acc, it.r0, it.r1, recs, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf, fx,
                                              fy, fz, cidx, lmax, j, k);
            // register r holds cell q = 4 k + r of the unit, component NCB j + cb
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int q = 4 * k + r;
                    const int cx = q & (bx - 1), cy = (q >> lbx) & (by - 1), cz = q >> (lbx + lby);
                    const int comp = NCB * j + cb;
                    tb[(comp >> 1) * cstride + ((cz * by + cy) * W + wv * bx + cx) * 2 + (comp & 1)] = acc[cb][r];
                }
        }
        __syncthreads();
        // 16 bytes (two cells) per thread and step, whole rows; cells of
        // units without an item here are left alone
        const int ox = (int)(T.box0 & 0xffffu), oy = (int)(T.box0 >> 16), oz = (int)T.box1;
        const int lhalf = lbx + __builtin_ctz((unsigned)PW) - 1;       // log2(W / 2)
        const int lrows = lby + lbz;
        const int total = nc << (lrows + lhalf);
        for (int ci = threadIdx.x; ci < total; ci += 64 * PW) {
            const int ch = ci & ((1 << lhalf) - 1);
            const int line = ci >> lhalf;
            const int coil = line >> lrows, row = line & (rows - 1);
            const int x = 2 * ch;
            const int slot = x >> lbx;
            const int32_t owner = slot == 0 ? T.item[0] : slot == 1 ? T.item[1] : slot == 2 ? T.item[2] : T.item[3];
            if (owner < 0) continue;
            const int cz = row >> lby, cy = row & (by - 1);
            const f4 v = *reinterpret_cast<const f4 *>(tb + coil * cstride + (row * W + x) * 2);
            f4 *dst = reinterpret_cast<f4 *>(out + (size_t)(c0 + coil) * cells +
                                             ((size_t)(oz + cz) * N + (oy + cy)) * N + (ox + x));
            if (nt)
                __builtin_nontemporal_store(v, dst);
            else
                *dst = v;
        }
        return;
    }

    // Write the accumulators of item it (unit box b) through an LDS
    // transpose: register r holds cell 4 k + r, component NCB j + cb (coil
    // c: re 2c, im 2c + 1); consecutive lanes then store consecutive cells
    // of one coil.
    auto write_out = [&](const fr_item &it, const item_box &b) __attribute__((always_inline)) {
        wave_sync();
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r) osm[(NCB * j + cb) * CS + 4 * k + r] = acc[cb][r];
        wave_sync();
        auto put = [&](int cl, int q, size_t go) __attribute__((always_inline)) {
            const float2 v = make_float2(osm[(2 * cl) * CS + q], osm[(2 * cl + 1) * CS + q]);
            const int c = c0 + cl;
            if (it.slot < 0) {
                if (nt)
                    __builtin_nontemporal_store(__builtin_bit_cast(unsigned long long, v),
                                                reinterpret_cast<unsigned long long *>(out + (size_t)c * cells + go));
                else
                    out[(size_t)c * cells + go] = v;
            } else {
                const size_t slot = ((size_t)(c >> 5) * nslots + it.slot) * 32 + (c & 31);
                partial[slot * cells_max + q] = v;
            }
        };
        if ((16 % b.ncell) == 0) {
            // the cell count divides 16 (full units): each lane keeps one cell
            const int sh = __builtin_ctz((unsigned)b.ncell);
            const int q = lane & (b.ncell - 1);
            const size_t go =
                ((size_t)(b.oz + q / (b.ux * b.uy)) * N + (b.oy + (q / b.ux) % b.uy)) * N + (b.ox + q % b.ux);
            for (int cl = lane >> sh; cl < nc; cl += 64 >> sh) put(cl, q, go);
        } else {
            for (int t = lane; t < nc * b.ncell; t += 64) {
                const int cl = t / b.ncell;
                const int q = t - cl * b.ncell;
                const size_t go =
                    ((size_t)(b.oz + q / (b.ux * b.uy)) * N + (b.oy + (q / b.ux) % b.uy)) * N + (b.ox + q % b.ux);
                put(cl, q, go);
            }
        }
        wave_sync();   // the next item reuses the transpose buffer
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) acc[cb] = f4{0.f, 0.f, 0.f, 0.f};
    };

    // ----------------------------------------------------------- pairs
    // One wave grids the two x-adjacent units of a pair one after the other,
    // the first unit's sums held in registers, and writes them out together:
    // rows of 2 bx cells (64 bytes for 4-cell-wide units) instead of bx.
    // (Stored straight from the accumulators, 16 bytes of a row at a time, 32
    // coils at 256^3 took 4.87 ms against 4.31 with an LDS transpose by 4-byte
    // words and 4.13 with this one by 16-byte words.)
    if (bid >= front_wg && ntiles > 0) {
        const int64_t pidx = fr_sampled_tile(grp * PW + wv, tstride);   // (tstride 1: every pair)
        if (pidx >= ntiles) return;
        const fr_tile T = tiles[pidx];
        const int32_t ia = T.item[0], ib = T.item[1];
        if (ia < 0 && ib < 0) return;
        // a unit alone (its partner is a front unit): the single write-out
        if (ia < 0 || ib < 0) {
            const fr_item it = items[ia >= 0 ? ia : ib];
            const item_box b = unpack_box(it.t0, it.pad);
            float fx, fy, fz;
            lane_cell(b, j, fx, fy, fz);
            if (it.r0 < it.r1)
                grid_records<NCB, PAIR, SMALL>(acc, it.r0, it.r1, recs, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf, fx, fy,
                                              fz, cidx, lmax, j, k);
            write_out(it, b);
            return;
        }
        const fr_item ita = items[ia], itb = items[ib];
        const item_box ba = unpack_box(ita.t0, ita.pad), bb = unpack_box(itb.t0, itb.pad);
        float fx, fy, fz;
        lane_cell(ba, j, fx, fy, fz);
        // at the end of A: its sums aside, B's cell and fresh accumulators
        f4 acc_a[NCB];
        auto to_b = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) {
                acc_a[cb] = acc[cb];
                acc[cb] = f4{0.f, 0.f, 0.f, 0.f};
            }
            lane_cell(bb, j, fx, fy, fz);
        };
        if (ita.r0 < ita.r1 && itb.r0 < itb.r1 && itb.r0 == ita.r1) {
            // A's and B's records are consecutive: one pipelined stream
            grid_records_mid<NCB, PAIR, SMALL>(acc, ita.r0, ita.r1, itb.r1, recs, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf,
                                              fx, fy, fz, cidx, lmax, j, k, to_b);
        } else {
            if (ita.r0 < ita.r1)
                grid_records<NCB, PAIR, SMALL>(acc, ita.r0, ita.r1, recs, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf, fx,
                                              fy, fz, cidx, lmax, j, k);
            to_b();
            if (itb.r0 < itb.r1)
                grid_records<NCB, PAIR, SMALL>(acc, itb.r0, itb.r1, recs, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf, fx,
                                              fy, fz, cidx, lmax, j, k);
        }
        // Lane (j, k) holds cells 4 k .. 4 k + 3 of both units, neighbours
        // along x in boxes at least 4 wide.  By way of LDS, [coil][cell of the pair's 2 bx x by x bz
        // box][re, im], 16 coils a step, each lane then stores two
        // neighbouring cells of a coil and 2 bx cells make one write.
        const int px = (4 * k) & ((1 << lbx) - 1), prow = (4 * k) >> lbx;
        const int cell = 2 * (lane & 15), x = cell & ((2 << lbx) - 1), row = cell >> (lbx + 1);
        const size_t go = ((size_t)(ba.oz + (row >> lby)) * N + (ba.oy + (row & ((1 << lby) - 1)))) * N + (ba.ox + x);
        // floats from the lane's first cell to its second and third: boxes
        // less than 4 wide hold those in a next row (2 x 2 x 4, 32 coils on
        // 128^3: 498 us, 883 as single units)
        const int d1 = lbx >= 1 ? 2 : 4, d2 = lbx >= 2 ? 4 : 8;
        constexpr int steps = NCB == 4 ? 2 : 1, ncs = NCB == 1 ? 8 : 16;
#pragma unroll
        for (int h = 0; h < steps; ++h) {
            wave_sync();
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float *o = osm + (NCB == 1 ? j >> 1 : j) * PS + 2 * ((prow << (lbx + 1)) + px + (u << lbx));
                if constexpr (NCB == 1) {
                    const f4 v = u ? acc[0] : acc_a[0];
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[(r & 1) * d1 + (r >> 1) * d2 + (j & 1)] = v[r];
                } else {
                    const f4 re = u ? acc[2 * h] : acc_a[2 * h], im = u ? acc[2 * h + 1] : acc_a[2 * h + 1];
                    if (lbx >= 1) {
                        *reinterpret_cast<f4 *>(o) = f4{re[0], im[0], re[1], im[1]};
                        *reinterpret_cast<f4 *>(o + d2) = f4{re[2], im[2], re[3], im[3]};
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            *reinterpret_cast<float2 *>(o + 4 * r) = make_float2(re[r], im[r]);
                    }
                }
            }
            wave_sync();
#pragma unroll
            for (int t = 0; t < ncs / 4; ++t) {
                const int cs = (lane >> 4) + 4 * t, cl = NCB == 4 ? 2 * cs + h : cs;
                if (cl >= nc) continue;
                const f4 v = *reinterpret_cast<const f4 *>(osm + cs * PS + 2 * cell);
                f4 *d = reinterpret_cast<f4 *>(out + (size_t)(c0 + cl) * cells + go);
                if (nt)
                    __builtin_nontemporal_store(v, d);
                else
                    *d = v;
            }
        }
        return;
    }

    int64_t i, iend;
    const int64_t fw = bid * PW + wv;
    if (bid < front_wg) {
        // fsub > 1 (a sample of the grid): wave fw takes sub-slice fw % fsub
        // of front item fw / fsub
        i = fsub > 1 ? fw / fsub : fw;
        iend = min(i + 1, nfront);
    } else {
        i = nfront + (grp * PW + wv) * ipw;
        iend = min(i + ipw, nitems);
    }
    if (i >= iend) return;

    fr_item it = items[i];
    item_box box = unpack_box(it.t0, it.pad);
    float fx, fy, fz;
    if (ipw > 1 && bid >= front_wg) {
        // A run of light items (one each a unit, their records consecutive)
        // as one record stream: at an item's end the pipeline keeps running
        // while the unit is written out, from LDS beside the positions (4
        // items a wave, 8 coils on 180^3: 283 us, drained at each item 317).
        // Units without records are written as zeros.
        auto next = [&]() __attribute__((always_inline)) {
            write_out(it, box);
            while (++i < iend) {
                it = items[i];
                box = unpack_box(it.t0, it.pad);
                if (it.r0 < it.r1) return true;
                write_out(it, box);
            }
            return false;
        };
        if (it.r0 == it.r1 && !next()) return;
        lane_cell(box, j, fx, fy, fz);
        const uint32_t first = it.r0;
        grid_stream<NCB, PAIR, SMALL>(acc, recs + first, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf, fx, fy, fz, cidx,
                                      lmax, j, k, [&](uint32_t q) __attribute__((always_inline)) {
                                          if (q != it.r1 - first) return true;
                                          const bool more = next();
                                          if (more) lane_cell(box, j, fx, fy, fz);
                                          return more;
                                      });
        return;
    }
    if (bid < front_wg && fsub > 1) {
        // only the front units of every tstride-th rank; the sub-slice's
        // records (a multiple of FR_POS_BATCH, possibly none) go to
        // virtual slot fw
        if (it.unit % (uint32_t)tstride != 0) return;
        const uint32_t sub = (uint32_t)(fw % fsub), len = it.r1 - it.r0;
        const uint32_t sl = ((len + fsub - 1) / fsub + (FR_POS_BATCH - 1)) & ~(uint32_t)(FR_POS_BATCH - 1);
        const uint32_t a = min(it.r0 + sub * sl, it.r1);
        it.r0 = a;
        it.r1 = min(a + sl, it.r1);
        it.slot = (int32_t)fw;
    }
    lane_cell(box, j, fx, fy, fz);
    if (it.r0 < it.r1)
        grid_records<NCB, PAIR, SMALL>(acc, it.r0, it.r1, recs, pos, data, (uint32_t)C, ca, cbb, stbl, pbuf, fx, fy, fz,
                                      cidx, lmax, j, k);
    write_out(it, box);
}

template <int NCB, bool PAIR, bool SMALL, typename TS, int OCC>
fr_status launch(fr_plan *p, const fr_samples *s, float2 *out, float2 *partial, int64_t tstride, int fsub)
{
    fr_ctx *ctx = p->ctx;
    const size_t cells = fr_plan_cells(p->dim, p->N, p->frames);
    const int chunks = (s->C + 8 * NCB - 1) / (8 * NCB);
    const int64_t light = p->nitems - p->nitems_front;
    // tstride > 1 (pair plans only): the sampled pairs (fr_sampled_tile), and
    // the front items cut into fsub sub-slices each (one wave per sub-slice)
    const int64_t front_wg = (p->nitems_front * (tstride > 1 ? fsub : 1) + PW - 1) / PW;
    const int64_t npairs = fr_sampled_tiles(p->ntiles, tstride);
    // light work: tiles of four (one per workgroup), pairs (PW per
    // workgroup) or runs of ipw items per wave; longer runs where one wave an
    // item would be more work-items than a launch takes (grids above 1024^3
    // that do not divide into pairs)
    const bool fours = p->ntiles > 0 && p->tile_units == PW;
    int ipw = std::max(1, p->pos_ipw);
    int64_t xr = 0, W = 0;
    for (;; ipw *= 2) {
        const int64_t per_wg = (int64_t)PW * ipw;
        const int64_t groups = p->ntiles > 0 ? (fours ? p->ntiles : (npairs + PW - 1) / PW)
                                             : (light + per_wg - 1) / per_wg;
        xr = std::max<int64_t>(1, p->xcd_run / (p->ntiles > 0 ? (fours ? PW : 2 * PW) : per_wg));
        const int64_t span = 8 * xr;
        W = front_wg + span * ((groups + span - 1) / span);
        if (W * 64 * PW < (int64_t(1) << 32) || p->ntiles > 0 || ipw > 64) break;
    }
    FR_CHECK(ctx, W * 64 * PW < (int64_t(1) << 32), FR_ERR_UNSUPPORTED, "gridding launch of %lld workgroups",
             (long long)W);
    // per wave: the write-out transpose (16 cells x 16 NCB components, or a
    // step of a pair; a tile of four needs less from its four waves together)
    const int osm_floats = std::max(16 * NCB * CS, (NCB == 1 ? 8 : 16) * PS);
    // in the place of the block of positions before it; a tile of four, whose
    // waves write each other's cells, has its own
    const int osm_at = p->ntiles == 0 && ipw > 1 ? 64 * 4 : 0;
    const int wave_floats = std::max(64 * 4, osm_at + osm_floats);
    const size_t lds = sizeof(float4) * p->L + sizeof(float) * PW * (wave_floats + (fours ? osm_floats : 0));
    auto kern = k_grid_pos<NCB, PAIR, SMALL, TS, OCC>;
    FR_HIP(ctx, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int lbx = __builtin_ctz((unsigned)p->geom.bx), lby = __builtin_ctz((unsigned)p->geom.by),
              lbz = __builtin_ctz((unsigned)p->geom.bz);
    hipLaunchKernelGGL(kern, dim3((unsigned)W, chunks), dim3(64 * PW), lds, ctx->stream, p->items, p->nitems,
                       p->tiles, p->ntiles, lbx, lby, lbz, p->recs, p->pos, p->tsel, p->L, p->mfma_cidx,
                       (const TS *)s->data, s->C, (int)p->N, cells, out, partial, p->nslots,
                       p->geom.cells_max, p->nitems_front, front_wg, ipw, xr, p->pos_stores == 1 ? 1 : 0,
                       p->tile_units, wave_floats, osm_at, tstride, tstride > 1 ? fsub : 1);
    FR_HIP(ctx, hipGetLastError());
    return FR_OK;
}

template <int NCB, bool PAIR, typename TS, int OCC>
fr_status launch_size(fr_plan *p, const fr_samples *s, float2 *out, float2 *partial, int64_t ts, int fs)
{
    const uint64_t bytes = (uint64_t)(p->M + 1) * s->C * sizeof(TS);
    return bytes < (uint64_t(1) << 32) ? launch<NCB, PAIR, true, TS, OCC>(p, s, out, partial, ts, fs)
                                       : launch<NCB, PAIR, false, TS, OCC>(p, s, out, partial, ts, fs);
}

template <typename TS, int OCC>
fr_status launch_ncb(fr_plan *p, const fr_samples *s, float2 *out, float2 *partial, int64_t ts, int fs)
{
    if (s->C <= 8) return launch_size<1, false, TS, OCC>(p, s, out, partial, ts, fs);
    if (s->C <= 16) return launch_size<2, false, TS, OCC>(p, s, out, partial, ts, fs);
    if (s->C % 2 == 0) return launch_size<4, true, TS, OCC>(p, s, out, partial, ts, fs);
    return launch_size<4, false, TS, OCC>(p, s, out, partial, ts, fs);
}

// pos[i].w <- the samples' DCF (the null sample keeps 0)
__global__ void k_pos_dcf(float4 *__restrict__ pos, const float *__restrict__ dcf, int64_t M)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) pos[i].w = dcf[i];
}

template <typename TS>
fr_status launch_occ(fr_plan *p, const fr_samples *s, float2 *out, float2 *partial, int64_t ts, int fs)
{
    return p->pos_waves == 4 ? launch_ncb<TS, 4>(p, s, out, partial, ts, fs)
                             : launch_ncb<TS, 1>(p, s, out, partial, ts, fs);
}

}  // namespace

fr_status fr_launch_grid_pos(fr_plan *p, const fr_samples *s, float2 *out, float2 *partial, int64_t tile_stride,
                             const fr_samples *dcf, int front_sub)
{
    FR_CHECK(p->ctx, p->recs && p->pos && p->tsel && p->geom.cells_max <= 16 && p->L <= FR_POS_MAX_L,
             FR_ERR_STATE, "position-weight gridding needs a plan built for it (accumulate 6)");
    FR_CHECK(p->ctx, tile_stride == 1 || (tile_stride > 1 && p->ntiles > 0 && p->tile_units == 2), FR_ERR_STATE,
             "a tile stride needs a plan with unit pairs");
    FR_CHECK(p->ctx, tile_stride == 1 || (front_sub >= 1 && s->C == 1), FR_ERR_INVALID,
             "a sample of the grid is single-channel, with at least one sub-slice per front item");
    const fr_samples *w = dcf ? dcf : s;
    FR_CHECK(p->ctx, w->M == s->M, FR_ERR_INVALID, "the DCF's samples handle has another sample count");
    // the DCF into the positions' .w when the copy there is not this
    // handle's current DCF (another samples handle, or a changed DCF), and
    // always under graph capture: a replay may follow DCF changes that no
    // host call sees, so the captured pass carries its copy and the next
    // eager pass refreshes again
    fr_ctx *ctx = p->ctx;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    FR_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
    const bool capturing = cs != hipStreamCaptureStatusNone;
    if (p->M > 0 && (capturing || p->pos_dcf_uid != w->uid || p->pos_dcf_version != w->dcf_version)) {
        hipLaunchKernelGGL(k_pos_dcf, dim3((unsigned)((p->M + 255) / 256)), dim3(256), 0, ctx->stream, p->pos,
                           w->dcf, p->M);
        FR_HIP(ctx, hipGetLastError());
        p->pos_dcf_uid = capturing ? 0 : w->uid;
        p->pos_dcf_version = w->dcf_version;
    }
    return s->type == FR_SAMPLES_C64 ? launch_occ<float2>(p, s, out, partial, tile_stride, front_sub)
                                     : launch_occ<__half2>(p, s, out, partial, tile_stride, front_sub);
}
