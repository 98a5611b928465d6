// Launchers of the band tile (nemo_band.h) for one domain: FP64 into the other
// state set or in place, mixed precision, and the table of metrics by row.
#include <algorithm>

#include "nemo_band.h"
#include "nemo_hip_common.h"

namespace nemo {
namespace {

using band::Flather;

// SPLIT: wavefronts a tile, each with its part of the outputs: 1 (all) or 2 (u;
// v and ssh).
template <typename T, bool ROWM, int R, int OW, int PF, bool NEXT, bool STREAM, int SPLIT>
__global__ __launch_bounds__(64) void k_band(typename band::Types<T>::In f,
                                             const T *__restrict__ tab, StepScalars<T> p,
                                             typename band::Types<T>::Out o, Flather<T> fl,
                                             int W, Bounds b, int nstrip,
                                             const double *__restrict__ tide_tab, int tide_k,
                                             double tide_val)
{
    static_assert(OW <= 61, "one neighbour lane below, two above");
    static_assert(SPLIT == 1 || SPLIT == 2, "parts of a tile");
    const int item = wave::xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int logical = item / SPLIT, part = item - logical * SPLIT;
    const int bd = logical / nstrip, strip = logical - bd * nstrip;
    const int jlo = b.ys - 1 + bd * R, jhi = min(jlo + R, b.ye + 2);
    auto tide = [&]() __attribute__((always_inline)) {
        const double t = tide_tab ? tide_tab[tide_k] : tide_val;
        if constexpr (sizeof(T) == 8)
            return t;
        else
            return wave::split(t);
    };
    auto run = [&](auto parts) __attribute__((always_inline)) {
        band::tile<T, ROWM, R, PF, NEXT, STREAM, decltype(parts)::value>(
            f, tab, p, o, fl, W, 0u, b, OW, strip, jlo, jhi, tide);
    };
    using band::PART_SSH, band::PART_U, band::PART_V;
    if constexpr (SPLIT == 1)
        run(std::integral_constant<int, band::ALL_PARTS>{});
    else if (part == 0)
        run(std::integral_constant<int, PART_U>{});
    else
        run(std::integral_constant<int, PART_V | PART_SSH>{});
}

template <typename T>
struct Args {
    hipStream_t s;
    const typename band::Types<T>::In &f;
    const T *tab;
    const StepScalars<T> &p;
    const typename band::Types<T>::Out &o;
    const Flather<T> &fl;
    int W;
    const Bounds &b;
    const double *tide_tab;
    int tide_k;
    double tide_val;
};

template <typename T, bool ROWM, int R, int OW, int PF, bool NEXT, bool STREAM, int SPLIT = 1>
void launch(const Args<T> &a)
{
    const int nstrip = wave::strips(a.b, OW);
    const dim3 grid((unsigned)(nstrip * wave::bands(a.b, R) * SPLIT));
    k_band<T, ROWM, R, OW, PF, NEXT, STREAM, SPLIT><<<grid, dim3(64), 0, a.s>>>(
        a.f, a.tab, a.p, a.o, a.fl, a.W, a.b, nstrip, a.tide_tab, a.tide_k, a.tide_val);
    NEMO_LAUNCH_CHECK();
}

// The 13 arrays of the row table, in this order.
constexpr int kRowArrays = 13;
template <typename T>
struct RowSource {
    const T *a[kRowArrays];
};
template <typename T, typename In>
RowSource<T> row_source(const In &f)
{
    return RowSource<T>{{f.area_t, f.area_u, f.area_v, f.dx_u, f.dx_v, f.dx_t, f.dy_u, f.dy_v,
                         f.dy_t, f.fcor_u, f.fcor_v, f.ssha_u, f.ssha_v}};
}

// A divisor that uniform_quotient takes (FP64).
__device__ bool divisor_ok(double d)
{
    return isfinite(d) && d != 0.0 && abs(__builtin_amdgcn_frexp_exp(d)) <= kDivisorExp;
}
__device__ bool divisor_ok(float) { return true; }
__device__ double reciprocal(double d) { return band::refined_reciprocal(d); }
__device__ float reciprocal(float d) { return __builtin_amdgcn_rcpf(d); }

// One workgroup per row: writes the row's record from its first column and
// stores `mark` to *bad when another column of the row holds other bits or a
// divisor is out of range. Reads 13 arrays once at most; a grid whose metrics
// vary is mostly recognised in the first 256 columns of each row. The others
// are read kRowBatch loads of each array at a time, without a barrier: 33 us
// with a barrier for every 256 columns -> 19 us at 1024^2, 128 -> 79 at 2048^2
// (5.5 TB/s).
constexpr int kRowBatch = 4;
template <typename T>
__global__ __launch_bounds__(256) void k_row_metrics(RowSource<T> src, int W, unsigned base,
                                                     int ncol, T *__restrict__ tab, int *bad,
                                                     int mark)
{
    using B = std::conditional_t<sizeof(T) == 8, unsigned long long, unsigned>;
    const int j = (int)blockIdx.x, nrow = (int)gridDim.x;
    const unsigned row = base + (unsigned)(j * W);
    B first[kRowArrays];
#pragma unroll
    for (int q = 0; q < kRowArrays; q++) first[q] = __builtin_bit_cast(B, ld32(src.a[q], row));
    bool differs = false;
    // columns x + 256 k of every array, all loads before the first comparison
    auto compare = [&](int x, auto batch) __attribute__((always_inline)) {
        constexpr int N = decltype(batch)::value;
        B v[N][kRowArrays];
#pragma unroll
        for (int k = 0; k < N; k++)
#pragma unroll
            for (int q = 0; q < kRowArrays; q++)
                v[k][q] = __builtin_bit_cast(
                    B, ld32(src.a[q], row + (unsigned)min(x + 256 * k, ncol - 1)));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < N; k++)
#pragma unroll
            for (int q = 0; q < kRowArrays; q++) differs |= v[k][q] != first[q];
    };
    const int x0 = (int)threadIdx.x;
    compare(x0, std::integral_constant<int, 1>{});
    differs = __syncthreads_or(differs);  // the workgroup's answer in every thread
    for (int x = 256; x < ncol && !differs; x += 256 * kRowBatch)
        compare(x + x0, std::integral_constant<int, kRowBatch>{});
    differs = __syncthreads_or(differs);
    if (threadIdx.x != 0) return;
    T v[kRowArrays];
#pragma unroll
    for (int q = 0; q < kRowArrays; q++) v[q] = __builtin_bit_cast(T, first[q]);
    const T e2u_n = ld32(src.a[6], base + (unsigned)(min(j + 1, nrow - 1) * W));
    T *r = tab + (size_t)j * band::ROW_WIDTH;
    using namespace band;
    r[M_AT] = v[0];
    r[M_ARU] = v[1];
    r[M_ARV] = v[2];
    r[M_E1U] = v[3];
    r[M_E1V] = v[4];
    r[M_E1V2] = v[4] + v[4];
    r[M_E1T] = v[5];
    r[M_E2U] = v[6];
    r[M_E2US] = v[6] + e2u_n;
    r[M_E2V] = v[7];
    r[M_E2T] = v[8];
    r[M_FCU] = v[9];
    r[M_FCV] = v[10];
    r[M_SAU] = v[11];
    r[M_SAV] = v[12];
    auto divisor = [&](int slot, T d) {
        differs |= !divisor_ok(d);
        r[slot] = reciprocal(d);
    };
    divisor(R_AT, v[0]);
    divisor(R_ARU, v[1]);
    divisor(R_ARV, v[2]);
    divisor(R_E1V2, v[4] + v[4]);
    divisor(R_E1T, v[5]);
    divisor(R_E2US, v[6] + e2u_n);
    divisor(R_E2T, v[8]);
    if (differs) *bad = mark;
}

template <typename T, typename In>
void row_metrics(hipStream_t s, const In &f, int W, unsigned base, const Bounds &b, T *tab,
                 int *bad, int mark)
{
    k_row_metrics<T><<<dim3((unsigned)(b.ye + 2)), dim3(256), 0, s>>>(
        row_source<T>(f), W, base, b.xe + 2, tab, bad, mark);
    NEMO_LAUNCH_CHECK();
}

// In-place step, second half: now <- after over the reference's copy region
// (time_step.cpp:115-122), and the face ssh from the new cell ssh (which the
// copy region covers, so the after field stands for the now field).
__global__ __launch_bounds__(256) void k_finish(double *__restrict__ un,
                                                const double *__restrict__ ua,
                                                double *__restrict__ vn,
                                                const double *__restrict__ va,
                                                double *__restrict__ sshn_t,
                                                const double *__restrict__ ssha_t,
                                                double *__restrict__ sshn_u,
                                                double *__restrict__ sshn_v,
                                                const int *__restrict__ tm,
                                                const double *__restrict__ area_t,
                                                const double *__restrict__ area_u,
                                                const double *__restrict__ area_v, int W,
                                                Bounds b)
{
    const int i = b.xs - 1 + (int)(blockIdx.x * 64 + threadIdx.x);
    const int j = b.ys - 1 + (int)(blockIdx.y * 4 + threadIdx.y);
    if (i > b.xe + 1 || j > b.ye) return;
    const int c = j * W + i;
    un[c] = ua[c];
    vn[c] = va[c];
    const double s = ssha_t[c];
    sshn_t[c] = s;
    if (i < b.xs || j < b.ys || i > b.xe) return;
    double v;
    if (i <= b.xe - 1 &&
        next_ssh_pt(s, ssha_t[c + 1], area_t[c], area_t[c + 1], area_u[c], tm[c], tm[c + 1], &v))
        sshn_u[c] = v;
    if (j <= b.ye - 1 &&
        next_ssh_pt(s, ssha_t[c + W], area_t[c], area_t[c + W], area_v[c], tm[c], tm[c + W], &v))
        sshn_v[c] = v;
}

// Tiles of a launch with R-row bands of ow columns.
long tiles(const Bounds &b, int rows, int ow)
{
    return (long)wave::strips(b, ow) * wave::bands(b, rows);
}

// Band height by the number of tiles. A wavefront takes about 2 us a row when
// it has a SIMD to itself, so a grid that does not fill the chip wants
// one-row bands, although each also evaluates the faces of the row before it
// (565 against 390 instructions a row); a large one wants the fewest halo
// rows, in 56-column strips (64-byte-aligned stores). Measured, us a step
// with one / two / four or eight rows:
//   FP64 by row  128^2 4.2 / 5.6 / 10;  384^2 7.1 / 7.5 / 11;  512^2 10.1 /
//                9.7 / 13.7;  1400^2 46 / 39 / 46;  2048^2 136 / 109 / 106;
//                4096^2 540 / 430 / 406
//   FP64         400^2 8.1 / 9.3 / 13.6;  700^2 20.3 / 22 / 23.5;  2048^2 207
//                / 193 / 195;  4096^2 809 / 751 / 741
//   FP32         512^2 6.2 / 7.1 / 10.3;  1024^2 16.6 / 16.7 / 17.7;  2048^2
//                65 / 58 / 56;  4096^2 314 / 266 / 242 (by row)
// The largest FP64 bands store past the caches (STREAM): by then a step's
// output is gone from them before the next step reads it (us a step, with and
// without: 1800^2 82 / 88, 2048^2 102 / 113, 4096^2 404 / 423). Below, and in
// FP32, the next step finds it there (1024^2 31.1 / 25.4, 1500^2 61 / 54;
// FP32 1500^2 79 / 69, 2048^2 116 / 110 with the read-back).
// The smallest grids leave most SIMDs without a wavefront even so, and a step
// takes one wavefront's chain of arithmetic. There two wavefronts share a tile
// (SPLIT), each reading all of it and evaluating half of its outputs. One / two
// wavefronts a tile:
//   FP64 by row  48^2 4.4 / 3.4;  128^2 4.6 / 3.9;  256^2 5.7 / 5.4;  320^2 6.4 /
//                6.6
//   FP64         48^2 4.0 / 3.3;  128^2 4.4 / 4.0;  181^2 4.7 / 4.6;  256^2 5.9 /
//                6.1
//   FP32         48^2 2.8 / 2.4;  128^2 3.1 / 2.8;  256^2 3.8 / 3.4;  320^2 3.9 /
//                3.8;  400^2 4.6 / 4.7
// (three wavefronts a tile are no better anywhere but at 48^2, by 0.1 us).
constexpr long kSplitTilesByRowF64 = 1400, kSplitTilesF64 = 600, kSplitTilesF32 = 1950;
constexpr long kOneRowTilesF64 = 12000, kOneRowTilesByRowF64 = 3500;
constexpr long kTwoRowTilesF64 = 48000, kTwoRowTilesByRowF64 = 24000;
constexpr long kOneRowTilesF32 = 16000, kTwoRowTilesF32 = 20000;

}  // namespace

size_t row_table_values(const Bounds &b) { return (size_t)(b.ye + 2) * band::ROW_WIDTH; }

void launch_row_metrics(hipStream_t s, const StepIn<double> &f, int W, unsigned base,
                        const Bounds &b, double *tab, int *bad, int mark)
{
    row_metrics<double>(s, f, W, base, b, tab, bad, mark);
}

void launch_row_metrics(hipStream_t s, const MixedIn &f, int W, unsigned base, const Bounds &b,
                        float *tab, int *bad, int mark)
{
    row_metrics<float>(s, f, W, base, b, tab, bad, mark);
}

void launch_band_f64(hipStream_t s, const StepIn<double> &f, const double *tab,
                     const StepScalars<double> &p, const StepOut<double> &o,
                     const double *u_prev, const double *v_prev, int W, const Bounds &b,
                     const double *tide_tab, int tide_k, double tide_val)
{
    const Flather<double> fl{u_prev, v_prev, nullptr, nullptr, 1, 0.0, 0.0};
    const Args<double> a{s, f, tab, p, o, fl, W, b, tide_tab, tide_k, tide_val};
    if (tab) {
        if (tiles(b, 1, 61) <= kSplitTilesByRowF64)
            launch<double, true, 1, 61, 0, true, false, 2>(a);
        else if (tiles(b, 1, 61) <= kOneRowTilesByRowF64)
            launch<double, true, 1, 61, 0, true, false>(a);
        else if (tiles(b, 2, 61) <= kTwoRowTilesByRowF64)
            launch<double, true, 2, 61, 0, true, false>(a);
        else
            launch<double, true, 8, 56, 0, true, true>(a);
    } else {
        if (tiles(b, 1, 61) <= kSplitTilesF64)
            launch<double, false, 1, 61, 0, true, false, 2>(a);
        else if (tiles(b, 1, 61) <= kOneRowTilesF64)
            launch<double, false, 1, 61, 0, true, false>(a);
        else if (tiles(b, 2, 61) <= kTwoRowTilesF64)
            launch<double, false, 2, 61, 0, true, false>(a);
        else
            launch<double, false, 4, 56, 1, true, true>(a);
    }
}

// FP32 shapes asked for by rows and prefetch: time of 20 steps with the
// overlapped-wavefront tile over that with the band tile. 4 rows: by row 1.06
// .. 2.2, by point 0.98 .. 1.13 (100 x 3000 0.95). 8 rows by row: 1.07 .. 1.95
// without prefetch; with it 0.93 .. 1.03 up to 640^2 (7062 tiles of one row),
// 1.00 .. 1.9 from 768^2 (10010). 8 rows by point: without prefetch 1.00 .. 1.10
// up to 300 x 250 (1260), 0.89 .. 1.03 above; with it 0.66 .. 0.98.
constexpr long kBandByRowTilesF32 = 10000, kBandByPointTilesF32 = 1500;

bool band_f32_shape(int rows, int cols, int prefetch, bool by_row, const Bounds &b)
{
    if (band_f32_auto(rows, cols, prefetch)) return true;
    if ((rows != 4 && rows != 8) || (cols != 61 && cols != 56)) return false;
    if (rows == 4) return true;
    if (by_row) return prefetch == 0 || tiles(b, 1, 61) > kBandByRowTilesF32;
    return prefetch == 0 && tiles(b, 1, 61) <= kBandByPointTilesF32;
}

void launch_band_f32(hipStream_t s, int rows, int cols, int prefetch, const MixedIn &f,
                     const float *tab, const StepScalars<float> &p, const MixedOut &o,
                     const float *u_prev, const float *v_prev, const float *cu,
                     const float *cv, int W, const Bounds &b, const double *tide_tab, int tide_k,
                     double tide_val)
{
    const Flather<float> fl{u_prev, v_prev, cu, cv, cu != nullptr, 0.0f, 0.0f};
    const Args<float> a{s, f, tab, p, o, fl, W, b, tide_tab, tide_k, tide_val};
    if (band_f32_auto(rows, cols, prefetch)) {
        if (tiles(b, 1, 61) <= kSplitTilesF32) {
            tab ? launch<float, true, 1, 61, 0, true, false, 2>(a)
                : launch<float, false, 1, 61, 0, true, false, 2>(a);
            return;
        }
        if (tiles(b, 1, 61) <= kOneRowTilesF32) {
            tab ? launch<float, true, 1, 61, 0, true, false>(a)
                : launch<float, false, 1, 61, 0, true, false>(a);
            return;
        }
        if (tiles(b, 2, 61) <= kTwoRowTilesF32) {
            tab ? launch<float, true, 2, 61, 0, true, false>(a)
                : launch<float, false, 2, 61, 0, true, false>(a);
            return;
        }
        rows = 4;
        prefetch = tab ? 2 : 0;
    }
#define NEMO_BAND_F32(R, OW, PF, BY_ROW)                                             \
    if (rows == R && cols == OW && prefetch == PF && (tab != nullptr) == BY_ROW) {   \
        launch<float, BY_ROW, R, OW, PF, true, false>(a);                            \
        return;                                                                      \
    }
    NEMO_BAND_F32(4, 61, 0, true)
    NEMO_BAND_F32(4, 61, 0, false)
    NEMO_BAND_F32(4, 61, 1, true)
    NEMO_BAND_F32(4, 61, 1, false)
    NEMO_BAND_F32(4, 61, 2, true)
    NEMO_BAND_F32(4, 61, 2, false)
    NEMO_BAND_F32(4, 56, 0, true)
    NEMO_BAND_F32(4, 56, 0, false)
    NEMO_BAND_F32(4, 56, 1, true)
    NEMO_BAND_F32(4, 56, 1, false)
    NEMO_BAND_F32(4, 56, 2, true)
    NEMO_BAND_F32(4, 56, 2, false)
    NEMO_BAND_F32(8, 61, 0, true)
    NEMO_BAND_F32(8, 61, 0, false)
    NEMO_BAND_F32(8, 61, 1, true)
    NEMO_BAND_F32(8, 61, 2, true)
    NEMO_BAND_F32(8, 56, 0, true)
    NEMO_BAND_F32(8, 56, 0, false)
    NEMO_BAND_F32(8, 56, 1, true)
    NEMO_BAND_F32(8, 56, 2, true)
#undef NEMO_BAND_F32
    NEMO_FATAL("mixed step: no band kernel for %d rows x %d columns, prefetch %d", rows, cols,
               prefetch);
}

void launch_band_inplace(hipStream_t s, const StepIn<double> &f, const StepScalars<double> &p,
                         const StepOut<double> &o, double omega, double d2r, int W,
                         const Bounds &b, double tide)
{
    // the after arrays hold the previous step's velocities until their faces
    // are written
    const Flather<double> fl{o.u, o.v, nullptr, nullptr, 1, 2. * omega, d2r};
    const Args<double> a{s, f, nullptr, p, o, fl, W, b, nullptr, 0, tide};
    if (tiles(b, 1, 61) <= kOneRowTilesF64)
        launch<double, false, 1, 61, 0, false, false>(a);
    else
        launch<double, false, 2, 61, 0, false, false>(a);
}

void launch_finish(hipStream_t s, double *un, const double *ua, double *vn, const double *va,
                   double *sshn_t, const double *ssha_t, double *sshn_u, double *sshn_v,
                   const int *tmask, const double *area_t, const double *area_u,
                   const double *area_v, int W, const Bounds &b)
{
    const dim3 grid((unsigned)((b.xe - b.xs + 3 + 63) / 64), (unsigned)((b.ye - b.ys + 2 + 3) / 4));
    k_finish<<<grid, dim3(64, 4), 0, s>>>(un, ua, vn, va, sshn_t, ssha_t, sshn_u, sshn_v, tmask,
                                          area_t, area_u, area_v, W, b);
    NEMO_LAUNCH_CHECK();
}

}  // namespace nemo
