// Batched in-place FFTs of the grids along each axis in turn (unnormalised,
// exp(sign 2 pi i / N)), for the sizes that fr_fft_radices takes: the
// transform of ImageFilter/FFT.cpp:40-51,82-84.
//
// One pass per axis over the whole array, so what bounds it is memory: each
// pass reads and writes the array once.  A workgroup transforms a tile of TC
// rows (along x: whole rows; along y and z: TC neighbouring columns, so that
// reads and writes are runs of 8 TC bytes) in mixed-radix Stockham stages.
// The first stage's inputs come from memory straight into registers and the
// last stage's outputs go straight back, so a length of three stages makes
// two exchanges through LDS, in place: every thread holds its one or two
// butterflies of a stage in registers, and a barrier parts all reads from all
// writes.  Twiddles come from a table evaluated in FP64.
//
// Measured against rocFFT, whose plans of these sizes take strided passes and
// transposes besides: 4 x 180^3 466 -> 213 us, 8 x 192^3 738 -> 651, 8 x 256^3
// 1799 -> 1451, 8 x 96^3 98 -> 74, 8 x 512^2 30 -> 21 (about 4 TB/s where the
// array is larger than the caches).  White noise comes out 1.3e-7 .. 1.7e-7
// from FP64, 4 to 18% nearer than rocFFT's at each of 34 sizes from 40^3 and
// 96^2 to 288^3 and 640^2.
#include "fr_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace {

constexpr int MAX_STAGES = FR_FFT_STAGES, MAX_THREADS = 512;
using stage_desc = fr_fft_desc::stage;
using fft_desc = fr_fft_desc;

// t / d by the high word of t m, m = ceil(2^32 / d) (0: d = 1), for the t
// below 2^16 that occur
__device__ __forceinline__ uint32_t quot(uint32_t t, uint32_t m) { return m ? __umulhi(t, m) : t; }

__device__ __forceinline__ float2 operator+(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 operator-(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
// A butterfly's constant: its FP32 rounding and the rest.  The rounding alone
// is the same relative error (1.8e-8 for sqrt(3) / 2) at every element of
// every stage, which an image of several coils does not average out as it
// does the elements' own roundings.  By the transform alone, 5 coils on 180^3
// are 4.2e-8 from FP64 with both parts and 5.2e-8 with the first one (rocFFT
// 5.5e-8).  The five-point butterfly's are in a form of fewer products, whose
// one more rounding is not a bias; with it the pair costs nothing that can be
// seen (up to 4% at 2D sizes of radix 10).
struct real2 {
    float hi, lo;
};
__host__ __device__ constexpr real2 two(double c) { return {(float)c, (float)(c - (double)(float)c)}; }
// a + b c
__device__ __forceinline__ float fma2(float b, real2 c, float a)
{
    if (__builtin_constant_p(c.lo) && c.lo == 0.f) return __builtin_fmaf(b, c.hi, a);
    return __builtin_fmaf(b, c.hi, __builtin_fmaf(b, c.lo, a));
}
__device__ __forceinline__ float mul2(float b, real2 c)
{
    if (__builtin_constant_p(c.lo) && c.lo == 0.f) return b * c.hi;
    return __builtin_fmaf(b, c.hi, b * c.lo);
}
__device__ __forceinline__ float2 axpy(float2 a, float2 b, real2 c)
{
    return make_float2(fma2(b.x, c, a.x), fma2(b.y, c, a.y));
}
__device__ __forceinline__ float2 scale(float2 b, real2 c) { return make_float2(mul2(b.x, c), mul2(b.y, c)); }
// a + i b c and a - i b c
__device__ __forceinline__ float2 add_i(float2 a, float2 b, real2 c)
{
    return make_float2(fma2(-b.y, c, a.x), fma2(b.x, c, a.y));
}
__device__ __forceinline__ float2 sub_i(float2 a, float2 b, real2 c)
{
    return make_float2(fma2(b.y, c, a.x), fma2(-b.x, c, a.y));
}
// a (c + i d)
__device__ __forceinline__ float2 cmul(float2 a, real2 c, real2 d)
{
    return make_float2(fma2(a.x, c, mul2(-a.y, d)), fma2(a.x, d, mul2(a.y, c)));
}
// a + i b, a - i b
__device__ __forceinline__ float2 add_i(float2 a, float2 b) { return make_float2(a.x - b.y, a.y + b.x); }
__device__ __forceinline__ float2 sub_i(float2 a, float2 b) { return make_float2(a.x + b.y, a.y - b.x); }

// R-point DFTs with w = exp(S 2 pi i / R), S = 1 or -1, in place, natural order
template <int R, int S>
__device__ __forceinline__ void dft(float2 (&x)[R])
{
    if constexpr (R == 2) {
        const float2 a = x[0], b = x[1];
        x[0] = a + b;
        x[1] = a - b;
    } else if constexpr (R == 3) {
        constexpr real2 r3 = two(0.86602540378443864676);
        const float2 p = x[1] + x[2], d = S > 0 ? x[1] - x[2] : x[2] - x[1];
        const float2 m = make_float2(__builtin_fmaf(p.x, -0.5f, x[0].x), __builtin_fmaf(p.y, -0.5f, x[0].y));
        x[0] = x[0] + p;
        x[1] = add_i(m, d, r3);
        x[2] = sub_i(m, d, r3);
    } else if constexpr (R == 4) {
        const float2 a = x[0] + x[2], b = x[0] - x[2], c = x[1] + x[3], d = S > 0 ? x[1] - x[3] : x[3] - x[1];
        x[0] = a + c;
        x[1] = add_i(b, d);
        x[2] = a - c;
        x[3] = sub_i(b, d);
    } else if constexpr (R == 5) {
        // (cosines as -1/4 +- sqrt(5) / 4 take fewer products, but round once
        // more: 160^3 1.66e-7 from FP64 against 1.6e-7)
        constexpr real2 c1 = two(0.30901699437494742410), c2 = two(-0.80901699437494742410);
        constexpr real2 s1 = two(0.95105651629515357212), s2 = two(0.58778525229247312917);
        constexpr real2 m1 = two(-0.95105651629515357212);
        const float2 p1 = x[1] + x[4], p2 = x[2] + x[3];
        const float2 d1 = S > 0 ? x[1] - x[4] : x[4] - x[1], d2 = S > 0 ? x[2] - x[3] : x[3] - x[2];
        const float2 a = axpy(axpy(x[0], p1, c1), p2, c2), b = axpy(axpy(x[0], p1, c2), p2, c1);
        const float2 u = axpy(scale(d1, s1), d2, s2), v = axpy(scale(d1, s2), d2, m1);
        x[0] = x[0] + (p1 + p2);
        x[1] = add_i(a, u);
        x[4] = sub_i(a, u);
        x[2] = add_i(b, v);
        x[3] = sub_i(b, v);
    } else if constexpr (R == 7) {
        constexpr real2 c1 = two(0.62348980185873353053), c2 = two(-0.22252093395631440429),
                        c3 = two(-0.90096886790241912624);
        constexpr real2 s1 = two(0.78183148246802980871), s2 = two(0.97492791218182360702),
                        s3 = two(0.43388373911755812048);
        constexpr real2 m1 = two(-0.78183148246802980871), m3 = two(-0.43388373911755812048);
        const float2 p1 = x[1] + x[6], p2 = x[2] + x[5], p3 = x[3] + x[4];
        const float2 d1 = S > 0 ? x[1] - x[6] : x[6] - x[1], d2 = S > 0 ? x[2] - x[5] : x[5] - x[2],
                     d3 = S > 0 ? x[3] - x[4] : x[4] - x[3];
        auto even = [&](real2 a, real2 b, real2 c) __attribute__((always_inline)) {
            return axpy(axpy(axpy(x[0], p1, a), p2, b), p3, c);
        };
        auto odd = [&](real2 a, real2 b, real2 c) __attribute__((always_inline)) {
            return axpy(axpy(scale(d1, a), d2, b), d3, c);
        };
        const float2 e1 = even(c1, c2, c3), e2 = even(c2, c3, c1), e3 = even(c3, c1, c2);
        const float2 o1 = odd(s1, s2, s3), o2 = odd(s2, m3, m1), o3 = odd(s3, m1, s2);
        x[0] = x[0] + ((p1 + p2) + p3);
        x[1] = add_i(e1, o1);
        x[6] = sub_i(e1, o1);
        x[2] = add_i(e2, o2);
        x[5] = sub_i(e2, o2);
        x[3] = add_i(e3, o3);
        x[4] = sub_i(e3, o3);
    } else {
        // R = 2 H: halves of even and odd inputs, X[k] = E[k] + w^k O[k], X[k + H] = E[k] - w^k O[k]
        constexpr int H = R / 2;
        static_assert(R == 6 || R == 8 || R == 10, "radix");
        float2 e[H], o[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            e[i] = x[2 * i];
            o[i] = x[2 * i + 1];
        }
        dft<H, S>(e);
        dft<H, S>(o);
        constexpr double r3 = 0.86602540378443864676, C1 = 0.80901699437494742410, C2 = 0.30901699437494742410;
        constexpr double S1 = 0.58778525229247312917, S2 = 0.95105651629515357212;
        constexpr real2 wc[5] = {two(1.), two(R == 6 ? 0.5 : C1), two(R == 6 ? -0.5 : C2), two(-C2), two(-C1)};
        constexpr real2 ws[5] = {two(0.), two(S * (R == 6 ? r3 : S1)), two(S * (R == 6 ? r3 : S2)), two(S * S2),
                                   two(S * S1)};
        constexpr real2 r2 = two(0.70710678118654752440);
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const float2 si = S > 0 ? make_float2(-o[i].y, o[i].x) : make_float2(o[i].y, -o[i].x);
            const float2 t = i == 0    ? o[0]
                             : R != 8  ? cmul(o[i], wc[i], ws[i])
                             : i == 1  ? scale(o[i] + si, r2)
                             : i == 2  ? si
                                       : scale(si - o[i], r2);
            x[i] = e[i] + t;
            x[i + H] = e[i] - t;
        }
    }
}

// A tile's place in memory: element n of row q at base + n step + q pitch.
struct tile_at {
    char *base;
    int64_t step;                               // bytes, as pitch
    uint32_t pitch;
    int rows;                                   // rows of the tile that exist
};

// crop position of output k (fftshifted if asked) or -1
__device__ __forceinline__ int crop_pos(int k, int N, int rc, int shift)
{
    const int kp = (shift ? (k < N / 2 ? k + N / 2 : k - N / 2) : k) - (N - rc) / 2;
    return kp >= 0 && kp < rc ? kp : -1;
}

// Where the last pass leaves the image of its one coil: rc kept outputs of its
// axis at out + k' outK, one element a kept column.  The arithmetic of k_sos
// (fr_image.hip).
struct sos_out {
    float *acc;                                 // LDS [rc][TC]
    float *out;
    const float *deapod;
    int64_t outK;
    int rc, shift;
    int rcx, rcy;                               // columns kept: x and, in 3D, y
};

// An element of a row in LDS.  Rows: one after the
// other, an element of padding after every eighth (the first stage writes at
// a stride of its radix); columns: side by side.
template <bool ROWS>
__device__ __forceinline__ int lds_at(const fft_desc &d, int n, int row)
{
    return ROWS ? row * d.pitch + n + (n >> 3) : (n << d.ltc) + row;
}

// Stage i for the whole tile, NB butterflies a thread.  ROWS: rows lie one
// after the other (step 1) and lanes run along a row; otherwise they lie side
// by side (pitch 1) and lanes run across them.  Memory addresses are a
// uniform base for each input (output) of the butterflies and one offset a
// butterfly, below 2^32 bytes.
template <int R, bool ROWS, int NB, int S, bool SOS>
__device__ __forceinline__ void stage(const fft_desc &d, int i, const tile_at &t, float2 *buf, float2 *tw,
                                      const float2 *__restrict__ gtw, const sos_out &o)
{
    const stage_desc &g = d.st[i];
    const bool first = i == 0, last = i == d.stages - 1;
    const int total = g.nb << d.ltc;
    float2 x[NB][R];
    int row[NB], j[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int q = threadIdx.x + b * blockDim.x;
        if (ROWS) {
            row[b] = (int)quot(q, g.m_nb);
            j[b] = q - row[b] * g.nb;
        } else {
            row[b] = q & ((1 << d.ltc) - 1);
            j[b] = q >> d.ltc;
        }
        if (q >= total || row[b] >= t.rows) row[b] = -1;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (row[b] < 0) continue;
        if (first) {
            const uint32_t off = (uint32_t)j[b] * (uint32_t)t.step + (uint32_t)row[b] * t.pitch;
#pragma unroll
            for (int r = 0; r < R; ++r)
                x[b][r] = *reinterpret_cast<const float2 *>(t.base + r * (g.nb * t.step) + off);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) x[b][r] = buf[lds_at<ROWS>(d, j[b] + r * g.nb, row[b])];
        }
    }
    // the table on its way behind the first inputs; otherwise all reads before the writes below
    if (first)
        for (int q = threadIdx.x; q < d.N; q += blockDim.x) tw[q] = gtw[q];
    else
        __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (row[b] < 0) continue;
        const int jq = (int)quot(j[b], g.m_ns), jm = j[b] - jq * g.Ns;
        if (!first) {
#pragma unroll
            for (int r = 1; r < R; ++r) x[b][r] = cmul(x[b][r], tw[r * jm * g.step]);
        }
        dft<R, S>(x[b]);
        const int n = jq * g.Ns * R + jm;
        if (last) {
            const uint32_t off = (uint32_t)n * (uint32_t)t.step + (uint32_t)row[b] * t.pitch;
#pragma unroll
            for (int r = 0; r < R; ++r) *reinterpret_cast<float2 *>(t.base + r * (g.Ns * t.step) + off) = x[b][r];
            if constexpr (SOS) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int kp = crop_pos(n + r * g.Ns, d.N, o.rc, o.shift);
                    if (kp >= 0)
                        o.acc[(kp << d.ltc) + row[b]] =
                            __fadd_rn(__fmul_rn(x[b][r].x, x[b][r].x), __fmul_rn(x[b][r].y, x[b][r].y));
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) buf[lds_at<ROWS>(d, n + r * g.Ns, row[b])] = x[b][r];
        }
    }
    if (!last) __syncthreads();
}

template <bool ROWS, int NB, int S, bool SOS>
__device__ __forceinline__ void transform(const fft_desc &d, const tile_at &t, float2 *buf, float2 *tw,
                                          const float2 *__restrict__ gtw, const sos_out &o)
{
    for (int i = 0; i < d.stages; ++i)
        switch (d.st[i].R) {                    // the barrier after stage 0 also covers the twiddles
        case 2: stage<2, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        case 3: stage<3, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        case 4: stage<4, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        case 5: stage<5, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        case 6: stage<6, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        case 7: stage<7, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        case 8: stage<8, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        default: stage<10, ROWS, NB, S, SOS>(d, i, t, buf, tw, gtw, o); break;
        }
}

// Rows (ROWS): `count` rows of N, tile T the rows from T TC.  Columns: planes
// of count columns, N apart by `step`; tile T the columns from (T mod tiles)
// TC of plane T / tiles, planes `plane` elements apart.  SOS: one plane, and
// the image.
template <bool ROWS, int NB, int S, bool SOS>
__global__ void __launch_bounds__(MAX_THREADS) __attribute__((amdgpu_waves_per_eu(NB == 1 || ROWS ? 8 : SOS ? 6 : 7)))
k_fft(float2 *data, const float2 *__restrict__ gtw, fft_desc d, int64_t count, uint32_t tiles, uint32_t all,
      int64_t step, int64_t plane, sos_out o)
{
    extern __shared__ float2 sm[];              // twiddles [N], tile, sums
    float2 *buf = sm + d.N;
    // a compact eighth of the tiles for each XCD (workgroups go to them in
    // turn): what fits an XCD's L2 is still there for the next axis (8 x
    // 512^2: x and y pass together 31 -> 23 us, 8 x 320^2 24 -> 15)
    const uint32_t T = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (T >= all) return;
    const uint32_t P = ROWS ? 0u : T / tiles;
    const int64_t q0 = (int64_t)(T - P * tiles) << d.ltc;
    tile_at t;
    t.base = reinterpret_cast<char *>(ROWS ? data + q0 * d.N : data + P * plane + q0);
    t.step = 8 * (ROWS ? 1 : step);
    t.pitch = 8u * (ROWS ? (uint32_t)d.N : 1u);
    t.rows = (int)min((int64_t)1 << d.ltc, count - q0);
    if constexpr (!SOS) {
        transform<ROWS, NB, S, false>(d, t, buf, sm, gtw, o);
    } else {
        o.acc = reinterpret_cast<float *>(buf + ((size_t)d.N << d.ltc));
        transform<ROWS, NB, S, true>(d, t, buf, sm, gtw, o);
        __syncthreads();
        for (int i = threadIdx.x; i < o.rc << d.ltc; i += blockDim.x) {
            const int kp = i >> d.ltc, row = i & ((1 << d.ltc) - 1);
            if (row >= t.rows) continue;
            const uint32_t col = (uint32_t)q0 + row, y = col / (uint32_t)d.N;       // (2D: y = 0)
            const int xp = crop_pos((int)(col - y * d.N), d.N, o.rcx, o.shift);
            const int yp = count > d.N ? crop_pos((int)y, d.N, o.rcy, o.shift) : 0;
            if (xp < 0 || yp < 0) continue;
            const int64_t at = kp * o.outK + (int64_t)yp * o.rcx + xp;
            float m = sqrtf(o.acc[i]);
            if (o.deapod) m = __fdiv_rn(m, o.deapod[at]);
            o.out[at] = m;
        }
    }
}

// The fewest stages, then the largest least radix; odd radices first (the
// first stage's LDS writes go at a stride of the radix along a row).
void search(int n, int least, int *cur, int depth, int *best, int &best_depth, int &best_min)
{
    if (n == 1) {
        const int mn = depth ? cur[0] : 0;      // radices ascend
        if (depth > 0 && (best_depth == 0 || depth < best_depth || (depth == best_depth && mn > best_min))) {
            best_depth = depth;
            best_min = mn;
            std::copy(cur, cur + depth, best);
        }
        return;
    }
    if (depth == MAX_STAGES) return;
    for (int r : {2, 3, 4, 5, 6, 7, 8, 10})
        if (r >= least && n % r == 0) {
            cur[depth] = r;
            search(n / r, r, cur, depth + 1, best, best_depth, best_min);
        }
}

constexpr uint32_t magic(uint32_t d) { return d > 1 ? (uint32_t)(((uint64_t(1) << 32) + d - 1) / d) : 0u; }

// radices of N: false if it has other factors, a single stage (whose inputs
// and outputs would share no barrier) or rows too long for a tile of 8
bool plan(int N, fft_desc &d)
{
    if (N < 8 || N > 1024) return false;
    int cur[MAX_STAGES], best[MAX_STAGES], n = 0, mn = 0;
    search(N, 2, cur, 0, best, n, mn);
    if (n < 2) return false;
    std::stable_sort(best, best + n, [](int a, int b) { return (a & 1) > (b & 1); });
    d.N = N;
    d.stages = n;
    d.pitch = N + N / 8 + 1;
    d.nbmax = 0;
    int Ns = 1;
    for (int i = 0; i < n; ++i) {
        const int R = best[i], nb = N / R;
        d.st[i] = stage_desc{R, nb, Ns, N / (R * Ns), magic(nb), magic(Ns)};
        d.nbmax = std::max(d.nbmax, nb);
        Ns *= R;
    }
    return d.nbmax * 8 <= 2 * MAX_THREADS;
}

template <bool ROWS>
fr_status pass(fr_fft *f, float2 *data, int64_t planes, int64_t count, int64_t step,
               int64_t plane, const sos_out *sos = nullptr)
{
    fr_ctx *ctx = f->ctx;
    fft_desc d = f->desc;
    // rows a tile: at most 16 (128-byte runs) and two butterflies a thread;
    // fewer, down to 4, for one tile a CU, and along x, where that breaks no
    // runs, for four.  At 8 x 512^2 and 16, 8, 4 rows: x 13.1, 13.3, 11.1 us,
    // y 14.2, 17.1, 20.2; 4 x 240^2 at 4 against 2 rows: y 7.6, 9.0.
    d.ltc = 4;
    while (d.nbmax << d.ltc > 2 * MAX_THREADS) --d.ltc;
    auto tiles = [&] { return (count + (1 << d.ltc) - 1) >> d.ltc; };
    while (d.ltc > 2 && planes * tiles() < (ROWS ? 4 : 1) * ctx->cu_count) --d.ltc;
    const int work = d.nbmax << d.ltc, each = work > MAX_THREADS ? 2 : 1;
    const int threads = ((work + each - 1) / each + 63) & ~63;
    const size_t lds = sizeof(float2) * (d.N + ((size_t)(ROWS ? d.pitch : d.N) << d.ltc)) +
                       (sos ? sizeof(float) * ((size_t)sos->rc << d.ltc) : 0);
    const int64_t W = planes * tiles();
    FR_CHECK(ctx, (W + 8) * threads < (int64_t(1) << 32), FR_ERR_UNSUPPORTED, "FFT launch of %lld workgroups",
             (long long)W);
    const bool pos = f->sign > 0;
    auto kern = each == 1 ? (pos ? k_fft<ROWS, 1, 1, false> : k_fft<ROWS, 1, -1, false>)
                          : (pos ? k_fft<ROWS, 2, 1, false> : k_fft<ROWS, 2, -1, false>);
    if constexpr (!ROWS)
        if (sos)
            kern = each == 1 ? (pos ? k_fft<ROWS, 1, 1, true> : k_fft<ROWS, 1, -1, true>)
                             : (pos ? k_fft<ROWS, 2, 1, true> : k_fft<ROWS, 2, -1, true>);
    if (lds > 65536)
        FR_HIP(ctx, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)((W + 7) / 8 * 8)), dim3(threads), lds, ctx->stream, data, f->tw, d, count,
                       (uint32_t)tiles(), (uint32_t)W, step, plane, sos ? *sos : sos_out{});
    FR_HIP(ctx, hipGetLastError());
    return FR_OK;
}

// Where rocFFT's kernels are the faster ones by more than 6% somewhere.  It
// has kernels that transform these sizes in one pass over a small 2D grid, or
// in one pass an axis without transposes, and a launch or two less, or more
// threads at work in each stage, beats these passes on few elements (4 x 240^2:
// 9.3 us against 11.5; 16^2 to 48^2: half) and, where the radices of a size
// leave threads idle in some stages (the 7s and 2 of 98), on many (16 x 98^3:
// 175 against 199).  A listed size is transformed here from `from` to `to` thousand
// elements in all (measured at 10 to 23 batches each, the lines between the two
// that they part; where both are within 6%, here: rocFFT's plan takes 2 to 40
// ms to make).  At the sizes not listed, of all that plan() takes up to 1000^2
// and 400^3, these passes took 0.45 to 1.06 of rocFFT's time from 1 grid to 2^26
// elements (3D 2^27), up to 1.15 (24^2: 1.2) at few elements of 12^2 to 24^2,
// 70^2, 144^2, 224^2, 48^3 and 60^3.
constexpr int64_t ALL = int64_t(1) << 40;
struct window {
    int dim, N;
    int64_t from, to;
};
constexpr window windows[] = {
    {2, 14, 280, ALL}, {2, 15, ALL, ALL}, {2, 16, ALL, ALL}, {2, 18, ALL, ALL}, {2, 21, 280, ALL}, {2, 25, ALL, ALL},
    {2, 27, ALL, ALL}, {2, 28, 250, ALL}, {2, 30, 100, ALL}, {2, 32, ALL, ALL}, {2, 35, ALL, ALL}, {2, 36, 290, ALL},
    {2, 40, 130, ALL}, {2, 42, 390, ALL}, {2, 45, 220, ALL}, {2, 48, ALL, ALL}, {2, 49, 380, ALL},
    {2, 50, 390, 1600}, {2, 54, 230, 1300}, {2, 56, 250, ALL}, {2, 60, 280, ALL}, {2, 63, 310, ALL},
    {2, 64, 320, ALL}, {2, 72, 290, 2300}, {2, 75, 220, ALL}, {2, 80, 350, ALL}, {2, 81, 360, 2100},
    {2, 84, 200, 2200}, {2, 98, 380, 1100}, {2, 100, 0, 780}, {2, 105, 220, 3000}, {2, 108, 320, 3700},
    {2, 112, 350, 3900}, {2, 125, 310, ALL}, {2, 128, 320, 2600}, {2, 135, 0, 1400}, {2, 160, 180, 4000},
    {2, 162, 320, 1800}, {2, 168, 200, ALL}, {2, 200, 280, ALL}, {2, 216, 320, ALL}, {2, 240, 400, ALL},
    {2, 243, 410, ALL}, {2, 256, 450, ALL}, {2, 280, 350, ALL}, {2, 336, 280, ALL}, {2, 343, 410, ALL},
    {2, 512, 370, ALL}, {3, 16, ALL, ALL}, {3, 25, ALL, ALL}, {3, 27, ALL, ALL}, {3, 32, 450, ALL},
    {3, 64, 640, ALL}, {3, 72, 530, 1800}, {3, 84, 0, 2100}, {3, 98, 0, 4500}, {3, 108, 0, 12000},
    {3, 112, 0, 2000}, {3, 125, 0, 38000}};

}  // namespace

// Whether f's grids are transformed here; lays out the stages.
bool fr_fft_radices(fr_fft *f)
{
    // (a grid below 2^32 bytes: 32-bit offsets)
    if (f->N > (f->dim == 3 ? 800u : 1024u) || !plan((int)f->N, f->desc)) return false;
    const int64_t thousands = (int64_t)f->batch * f->N * f->N * (f->dim == 3 ? f->N : 1) / 1000;
    for (const window &w : windows)
        if (w.dim == f->dim && w.N == (int)f->N) return thousands >= w.from && thousands < w.to;
    return true;
}

// The grids of f's batch, in place; f->tw is set.  With an image (of one coil
// and grid, kept outputs rcx x rcy x rcz), the last pass forms it.
static fr_status passes(fr_fft *f, float2 *data, const sos_out *sos)
{
    const int64_t N = f->N, B = f->batch, last = sos ? 1 : B;
    fr_status e = pass<true>(f, data, 1, B * N * (f->dim == 3 ? N : 1), 1, 0);
    if (!e && f->dim == 3) e = pass<false>(f, data, B * N, N, N, N * N);
    if (!e) e = f->dim == 3 ? pass<false>(f, data, last, N * N, N * N, N * N * N, sos)
                            : pass<false>(f, data, last, N, N, N * N, sos);
    return e;
}

fr_status fr_fft_passes(fr_fft *f, float2 *data) { return passes(f, data, nullptr); }

// Whether the image comes out of the last pass: of one coil, in 2D and of 3D
// grids up to 2^20 cells (a launch less: 96^2 9.9 us against 11.8 with k_sos,
// 40^3 13.6 and 15.0, 96^3 24.6 and 26.4).  Above, the pass with its image is
// the slower one (144^3 52.9 us and 52.2, 240^3 156.9 and 150.9), and several
// coils would go one after the other, nothing loaded ahead.
bool fr_fft_sos_last(const fr_fft *f, const fr_grids *g)
{
    return f->own && g->frames == 0 && g->C == 1 && (g->dim == 2 || g->cells <= (size_t(1) << 20));
}

fr_status fr_fft_passes_sos(fr_fft *f, const fr_grids *g, int rcx, int rcy, int rcz, int shift, const float *deapod,
                            float *out)
{
    sos_out o{};
    o.out = out;
    o.deapod = deapod;
    o.rc = g->dim == 3 ? rcz : rcy;
    o.outK = g->dim == 3 ? (int64_t)rcy * rcx : rcx;
    o.rcx = rcx;
    o.rcy = rcy;
    o.shift = shift;
    return passes(f, g->data, &o);
}
