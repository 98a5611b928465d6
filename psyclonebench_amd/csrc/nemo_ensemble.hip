// Batched ensemble step (CDNA4 / gfx950): one launch per step advances
// every domain of the ensemble.
//
// Work list: every domain is cut into tiles of one strip (OW output columns:
// 61, or 56 so that every strip's stores start on a 64-byte boundary, or per
// domain whichever of the two suits its width) by one band (R rows); the list
// holds one self-contained descriptor per tile (domain geometry, strip, band,
// width), domain by domain. Two launch forms run on the domain's arrays of
// each tile:
//
//  * one wavefront per tile: a grid of one-wavefront workgroups, one per
//    tile of the list, as the single-domain kernels launch, so that the
//    dispatcher starts a new tile wherever a wavefront slot frees up. The
//    default shape, and bands of 4 and 8 rows where they are the faster
//    (ens_band), are band tiles (nemo_band.h), which write the Flather faces
//    themselves; the others run wave::tile_f64 / tile_mixed;
//  * persistent: a fixed number of workgroups (a multiple of 8) of 1, 2 or
//    4 wavefronts; every wavefront takes tiles from the list with a stride,
//    so uneven domain sizes cost nothing but the partial tiles at their
//    edges. These run wave::tile_f64 / tile_mixed.
//
// Every form has the loads of the next row issued at the top of the row that
// needs them (PF = 0), or one or two rows earlier.
//
// XCD locality: the dispatcher hands workgroup b to XCD b % 8. The list is
// cut into 8 contiguous chunks and the workgroups of XCD x take tiles of
// chunk x only, so neighbouring strips of a domain (which share the cache
// lines of their overlap columns) are processed under one L2.
#include "nemo_band.h"
#include "nemo_ensemble.h"
#include "nemo_hip_common.h"
#include "nemo_wave.h"

namespace nemo {
namespace {

// Tiles [first, last) of this wavefront's XCD chunk, and its stride. Every
// quantity is wavefront-uniform, so the list and domain reads are scalar.
struct Walk {
    int first, last, stride;
};

__device__ __forceinline__ Walk walk(int ntiles)
{
    const int wpb = (int)(blockDim.x >> 6);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int bid = (int)blockIdx.x, nblk = (int)gridDim.x;
    const int xcd = bid & 7, k = bid >> 3, per = nblk >> 3;  // nblk % 8 == 0
    const int chunk = (ntiles + 7) >> 3;
    const int t0 = xcd * chunk;
    return Walk{t0 + k * wpb + wave, min(t0 + chunk, ntiles), per * wpb};
}

// Tile `tl` of the FP64 step; OW = 0 takes the tile width from the tile
// (wavefront-uniform branch between the 61- and 56-column bodies).
template <int R, int OW, int PF>
__device__ __forceinline__ void ens_tile_f64(const StepIn<double> &f,
                                             const StepScalars<double> &p,
                                             const StepOut<double> &o, const EnsTile &tl,
                                             double tide)
{
    if constexpr (OW == 0) {
        if (tl.cols == 61)
            ens_tile_f64<R, 61, PF>(f, p, o, tl, tide);
        else
            ens_tile_f64<R, 56, PF>(f, p, o, tl, tide);
    } else {
        wave::tile_f64<R, OW, PF>(f, p, o, tl.W, tl.off, Bounds{tl.xs, tl.xe, tl.ys, tl.ye},
                                  tl.strip, tl.band, tide);
    }
}

template <int R, int OW, int PF>
__device__ __forceinline__ void ens_tile_mixed(const MixedIn &f, const StepScalars<float> &p,
                                               const MixedOut &o, const EnsTile &tl,
                                               double tide)
{
    if constexpr (OW == 0) {
        if (tl.cols == 61)
            ens_tile_mixed<R, 61, PF>(f, p, o, tl, tide);
        else
            ens_tile_mixed<R, 56, PF>(f, p, o, tl, tide);
    } else {
        wave::tile_mixed<R, OW, PF>(f, p, o, tl.W, tl.off, Bounds{tl.xs, tl.xe, tl.ys, tl.ye},
                                    tl.strip, tl.band, wave::split(tide));
    }
}

// Band tile, one wavefront each, or two that share it (SPLIT = 2: u; v and ssh);
// the grid has exactly SPLIT * ntiles workgroups. The strip's width comes with
// the tile. ROWM: every domain has a table of metrics
// by row (records tl.rec and on).
template <typename T, bool ROWM, int R, int PF, bool STREAM, int SPLIT = 1>
__global__ __launch_bounds__(64) void k_ens_band(typename band::Types<T>::In f,
                                                 const T *__restrict__ tab, StepScalars<T> p,
                                                 typename band::Types<T>::Out o,
                                                 band::Flather<T> fl,
                                                 const EnsTile *__restrict__ tiles,
                                                 const double *__restrict__ tide)
{
    static_assert(SPLIT == 1 || SPLIT == 2, "parts of a tile");
    const int item = wave::xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const EnsTile tl = tiles[item / SPLIT];
    const Bounds b{tl.xs, tl.xe, tl.ys, tl.ye};
    const int jlo = tl.ys - 1 + tl.band * R, jhi = min(jlo + R, tl.ye + 2);
    const T *const rec = ROWM ? tab + (size_t)tl.rec * band::ROW_WIDTH : nullptr;
    auto tide_of = [&]() __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 8)
            return tide[tl.dom];
        else
            return wave::split(tide[tl.dom]);
    };
    auto run = [&](auto parts) __attribute__((always_inline)) {
        band::tile<T, ROWM, R, PF, true, STREAM, decltype(parts)::value>(
            f, rec, p, o, fl, tl.W, tl.off, b, tl.cols, tl.strip, jlo, jhi, tide_of);
    };
    if constexpr (SPLIT == 1)
        run(std::integral_constant<int, band::ALL_PARTS>{});
    else if (item % SPLIT == 0)
        run(std::integral_constant<int, band::PART_U>{});
    else
        run(std::integral_constant<int, band::PART_V | band::PART_SSH>{});
}

template <int R, int OW, int PF>
__global__ __launch_bounds__(256) void k_ens_f64(StepIn<double> f, StepScalars<double> p,
                                                 StepOut<double> o,
                                                 const EnsTile *__restrict__ tiles,
                                                 int ntiles,
                                                 const double *__restrict__ tide)
{
    const Walk w = walk(ntiles);
    for (int t = w.first; t < w.last; t += w.stride) {
        const EnsTile tl = tiles[t];
        ens_tile_f64<R, OW, PF>(f, p, o, tl, tide[tl.dom]);
    }
}

// One wavefront per tile; the grid has exactly ntiles workgroups.
template <int R, int OW, int PF>
__global__ __launch_bounds__(64) void k_ens_f64_grid(StepIn<double> f, StepScalars<double> p,
                                                     StepOut<double> o,
                                                     const EnsTile *__restrict__ tiles,
                                                     const double *__restrict__ tide)
{
    const EnsTile tl = tiles[wave::xcd_tile((int)blockIdx.x, (int)gridDim.x)];
    ens_tile_f64<R, OW, PF>(f, p, o, tl, tide[tl.dom]);
}

template <int R, int OW, int PF>
__global__ __launch_bounds__(256) void k_ens_mixed(MixedIn f, StepScalars<float> p,
                                                   MixedOut o,
                                                   const EnsTile *__restrict__ tiles,
                                                   int ntiles,
                                                   const double *__restrict__ tide)
{
    const Walk w = walk(ntiles);
    for (int t = w.first; t < w.last; t += w.stride) {
        const EnsTile tl = tiles[t];
        ens_tile_mixed<R, OW, PF>(f, p, o, tl, tide[tl.dom]);
    }
}

template <int R, int OW, int PF>
__global__ __launch_bounds__(64) void k_ens_mixed_grid(MixedIn f, StepScalars<float> p,
                                                       MixedOut o,
                                                       const EnsTile *__restrict__ tiles,
                                                       const double *__restrict__ tide)
{
    const EnsTile tl = tiles[wave::xcd_tile((int)blockIdx.x, (int)gridDim.x)];
    ens_tile_mixed<R, OW, PF>(f, p, o, tl, tide[tl.dom]);
}

void check_shape(const EnsShape &sh)
{
    if (sh.blocks < 0 || sh.blocks % 8)
        NEMO_FATAL("ensemble launch: %d workgroups is not 0 (one per tile) or a positive "
                   "multiple of 8", sh.blocks);
    if (sh.waves_per_block != 1 && sh.waves_per_block != 2 && sh.waves_per_block != 4)
        NEMO_FATAL("ensemble launch: %d wavefronts per workgroup", sh.waves_per_block);
    if (sh.blocks == 0 && sh.waves_per_block != 1)
        NEMO_FATAL("ensemble launch: one workgroup per tile takes 1 wavefront, not %d",
                   sh.waves_per_block);
    if (sh.cols != 61 && sh.cols != 56 && sh.cols != 0)
        NEMO_FATAL("ensemble launch: %d columns per wavefront", sh.cols);
    if (sh.prefetch < 0 || sh.prefetch > 2)
        NEMO_FATAL("ensemble launch: prefetch depth %d", sh.prefetch);
}

// rows x columns x prefetch depth of the tile -> one kernel instantiation
// per launch form
#define NEMO_ENS_PERSISTENT(X)                                                         \
    X(4, 61, 0) X(8, 61, 0) X(16, 61, 0) X(32, 61, 0) X(64, 61, 0) X(4, 56, 0)         \
    X(8, 56, 0) X(16, 56, 0) X(32, 56, 0) X(64, 56, 0) X(4, 61, 1) X(8, 61, 1)         \
    X(16, 61, 1) X(4, 56, 1) X(8, 56, 1) X(16, 56, 1)
#define NEMO_ENS_GRID(X)                                                               \
    X(4, 61, 1) X(4, 56, 1) X(4, 0, 1) X(4, 61, 2) X(4, 56, 2) X(8, 61, 0) X(8, 56, 0)  \
    X(8, 0, 0) X(8, 61, 1) X(8, 56, 1) X(8, 0, 1) X(8, 61, 2) X(8, 56, 2) X(8, 0, 2)    \
    X(16, 61, 0) X(16, 56, 0) X(16, 61, 1) X(16, 56, 1)
// shapes whose tiles are always band tiles: 4 rows without prefetch, and the
// default one
#define NEMO_ENS_BAND_ONLY(X) X(4, 61, 0) X(4, 56, 0) X(4, 0, 0) X(4, 0, 2)

// Tiles of the default shape, by how many bands of one and of two rows there
// are (the reasons are those of the single domain: a wavefront with a SIMD to
// itself wants one row, a full chip fewer halo rows; non-temporal stores where
// a step's output is gone from the last-level cache before the next step).
// Measured on ensembles of uneven domains, us a step:
//   points       one row / two / four / four, non-temporal
//   FP64 by row  54 k 6.8 / 7.0 / 11;  0.4 M 19.5 / 16.4 / 18;  1.2 M 50 / 36 /
//                39 / 45;  2.9 M 133 / 93 / 86 / 83;  24 M 1029 / 711 / 679 / 647
//   FP64         54 k 5.9 / 7.2 / 12;  0.4 M 18.4 / 19.6 / 22;  1.0 M 44.4 /
//                43.4 / 48;  7.2 M 353 / 345 / 351, two rows non-temporal 334
//   FP32 by row  54 k 4.2 / 5.4 / 8.9;  1.2 M 18.2 / 19.0 / 22;  2.9 M 33.7 /
//                33.0 / 41 / 55;  24 M 441 / 394 / 410 / 442
//   FP32         1.0 M 22 / 25 / 28;  2.9 M 85 / 76 / 76;  7.2 M 211 / 202 / 211
// The overlapped-wavefront tiles took 13, 33, 68, 180 (2.9 M) and 81 us (FP32,
// 2.9 M), with a Flather launch after each step.
// On the smallest two wavefronts share a tile, as in a single domain (one / two,
// by row: 306 tiles FP64 4.1 / 3.4, FP32 3.2 / 2.7; 1193 tiles 5.7 / 5.3 and 3.9 /
// 3.5).
constexpr long kEnsSplitTilesByRowF64 = 1400, kEnsSplitTilesF64 = 600, kEnsSplitTilesF32 = 1950;
constexpr long kEnsOneRowTilesByRowF64 = 3500, kEnsOneRowTilesF64 = 12000;
constexpr long kEnsOneRowTilesF32 = 24000;
constexpr long kEnsTwoRowTilesByRowF64 = 24000, kEnsCachedTilesF64 = 48000;

// Shapes asked for by rows and prefetch run band tiles where these are the
// faster. Time of a step with the overlapped-wavefront tile (and its Flather
// launch) over that with the band tile, over ensembles of 146 to 73 thousand
// one-row tiles:
//   by row     every FP64 shape 1.00 .. 1.8, FP32 4 rows 1.04 .. 1.9, 8 rows
//              without prefetch 1.08 .. 1.8; with it 0.89 .. 1.02 up to 9659
//              tiles, 1.04 .. 1.6 from 22581
//   by point   4 rows without prefetch 0.97 .. 1.2; with it 1.01 .. 1.07 up to
//              2841 tiles, 0.93 .. 1.01 from 9659; 8 rows FP64 0.65 .. 1.03,
//              FP32 without prefetch 1.02 .. 1.15 up to 2841 tiles and 0.90 ..
//              1.02 from 5092, with it 0.75 .. 0.94
constexpr long kEnsBandByRowTilesF32 = 10000, kEnsBandByPointTiles = 4000;

bool default_shape(const EnsShape &sh)
{
    return sh.blocks == 0 && sh.rows == 4 && sh.cols == 0 && sh.prefetch == 2;
}

void unsupported(const EnsShape &sh)
{
    NEMO_FATAL("ensemble launch: no %s kernel for %d rows x %d columns, prefetch %d",
               sh.blocks ? "persistent" : "one-wavefront-per-tile", sh.rows, sh.cols,
               sh.prefetch);
}

}  // namespace

bool ens_shape_supported(const EnsShape &sh)
{
#define NEMO_ENS_HAS(R, OW, PF)                                                        \
    if (sh.rows == R && sh.cols == OW && sh.prefetch == PF) return true;
    if (sh.blocks) {
        NEMO_ENS_PERSISTENT(NEMO_ENS_HAS)
    } else {
        NEMO_ENS_GRID(NEMO_ENS_HAS)
        NEMO_ENS_BAND_ONLY(NEMO_ENS_HAS)
    }
#undef NEMO_ENS_HAS
    return false;
}

bool ens_band(const EnsShape &sh, int precision, bool by_row, long one_row_tiles)
{
    if (default_shape(sh)) return true;
    if (sh.blocks || (sh.rows != 4 && sh.rows != 8)) return false;
    if (sh.rows == 4 && sh.prefetch == 0) return true;
    if (by_row)
        return precision == 64 || sh.rows == 4 || sh.prefetch == 0 ||
               one_row_tiles > kEnsBandByRowTilesF32;
    return one_row_tiles <= kEnsBandByPointTiles &&
           (sh.rows == 4 || (precision == 32 && sh.prefetch == 0));
}

EnsBand ens_band_tiles(const EnsShape &sh, int precision, bool by_row, long one_row_tiles,
                       long two_row_tiles)
{
    if (!default_shape(sh))
        return EnsBand{sh.rows, sh.cols, sh.prefetch, false, false};
    const long one = precision == 32 ? kEnsOneRowTilesF32
                     : by_row        ? kEnsOneRowTilesByRowF64
                                     : kEnsOneRowTilesF64;
    const long split = precision == 32 ? kEnsSplitTilesF32
                       : by_row        ? kEnsSplitTilesByRowF64
                                       : kEnsSplitTilesF64;
    if (one_row_tiles <= one) return EnsBand{1, 61, 0, false, one_row_tiles <= split};
    if (precision == 32) return EnsBand{2, 61, 0, false, false};
    if (by_row)
        return two_row_tiles <= kEnsTwoRowTilesByRowF64 ? EnsBand{2, 61, 0, false, false}
                                                        : EnsBand{4, 0, 0, true, false};
    return EnsBand{2, 61, 0, two_row_tiles > kEnsCachedTilesF64, false};
}

template <typename T, typename In, typename Out>
void launch_band(hipStream_t s, const EnsBand &bt, const In &in, const T *tab,
                 const StepScalars<T> &p, const Out &out, const T *u_prev, const T *v_prev,
                 const T *cu, const T *cv, const EnsTile *tiles, int ntiles, const double *tide)
{
    if (ntiles <= 0) return;
    const band::Flather<T> fl{u_prev, v_prev, cu, cv, sizeof(T) == 8 || cu, T(0), T(0)};
    const dim3 grid((unsigned)(bt.split ? 2 * ntiles : ntiles)), block(64);
    auto run = [&](auto kernel) {
        kernel<<<grid, block, 0, s>>>(in, tab, p, out, fl, tiles, tide);
        NEMO_LAUNCH_CHECK();
    };
    if (bt.split && bt.rows == 1)
        return tab ? run(k_ens_band<T, true, 1, 0, false, 2>)
                   : run(k_ens_band<T, false, 1, 0, false, 2>);
    if constexpr (sizeof(T) == 8) {
        if (bt.stream && bt.rows == 4 && tab) return run(k_ens_band<T, true, 4, 0, true>);
        if (bt.stream && bt.rows == 2 && !tab) return run(k_ens_band<T, false, 2, 0, true>);
    }
#define NEMO_ENS_BAND(R, PF, BY_ROW)                                                   \
    if (bt.rows == R && bt.prefetch == PF && !bt.stream && !bt.split &&                \
        (tab != nullptr) == BY_ROW)                                                    \
        return run(k_ens_band<T, BY_ROW, R, PF, false>);
    NEMO_ENS_BAND(1, 0, true)
    NEMO_ENS_BAND(1, 0, false)
    NEMO_ENS_BAND(2, 0, true)
    NEMO_ENS_BAND(2, 0, false)
    NEMO_ENS_BAND(4, 0, true)
    NEMO_ENS_BAND(4, 0, false)
    NEMO_ENS_BAND(4, 1, true)
    NEMO_ENS_BAND(4, 1, false)
    NEMO_ENS_BAND(4, 2, true)
    NEMO_ENS_BAND(4, 2, false)
    NEMO_ENS_BAND(8, 0, true)
    NEMO_ENS_BAND(8, 1, true)
    NEMO_ENS_BAND(8, 2, true)
    if constexpr (sizeof(T) == 4) {
        NEMO_ENS_BAND(8, 0, false)
    }
#undef NEMO_ENS_BAND
    NEMO_FATAL("ensemble launch: no band kernel for %d rows, prefetch %d", bt.rows, bt.prefetch);
}

void launch_ens_band(hipStream_t s, const EnsBand &bt, const StepIn<double> &in,
                     const double *tab, const StepScalars<double> &p, const StepOut<double> &out,
                     const double *u_prev, const double *v_prev, const EnsTile *tiles,
                     int ntiles, const double *tide)
{
    launch_band<double>(s, bt, in, tab, p, out, u_prev, v_prev, nullptr, nullptr, tiles, ntiles,
                        tide);
}

void launch_ens_band(hipStream_t s, const EnsBand &bt, const MixedIn &in, const float *tab,
                     const StepScalars<float> &p, const MixedOut &out, const float *u_prev,
                     const float *v_prev, const float *cu, const float *cv,
                     const EnsTile *tiles, int ntiles, const double *tide)
{
    launch_band<float>(s, bt, in, tab, p, out, u_prev, v_prev, cu, cv, tiles, ntiles, tide);
}

void launch_ens_f64(hipStream_t s, const EnsShape &sh, const StepIn<double> &in,
                    const StepScalars<double> &p, const StepOut<double> &out,
                    const EnsTile *tiles, int ntiles, const double *tide)
{
    check_shape(sh);
    if (ntiles <= 0) return;
    const dim3 grid((unsigned)sh.blocks), block((unsigned)(64 * sh.waves_per_block));
#define NEMO_ENS_F64(R, OW, PF)                                                        \
    if (sh.rows == R && sh.cols == OW && sh.prefetch == PF) {                          \
        k_ens_f64<R, OW, PF><<<grid, block, 0, s>>>(in, p, out, tiles, ntiles, tide);  \
        NEMO_LAUNCH_CHECK();                                                           \
        return;                                                                        \
    }
#define NEMO_ENS_F64_GRID(R, OW, PF)                                                   \
    if (sh.rows == R && sh.cols == OW && sh.prefetch == PF) {                          \
        k_ens_f64_grid<R, OW, PF><<<dim3((unsigned)ntiles), dim3(64), 0, s>>>(         \
            in, p, out, tiles, tide);                                                  \
        NEMO_LAUNCH_CHECK();                                                           \
        return;                                                                        \
    }
    if (sh.blocks) {
        NEMO_ENS_PERSISTENT(NEMO_ENS_F64)
    } else {
        NEMO_ENS_GRID(NEMO_ENS_F64_GRID)
    }
#undef NEMO_ENS_F64
#undef NEMO_ENS_F64_GRID
    unsupported(sh);
}

void launch_ens_mixed(hipStream_t s, const EnsShape &sh, const MixedIn &in,
                      const StepScalars<float> &p, const MixedOut &out,
                      const EnsTile *tiles, int ntiles, const double *tide)
{
    check_shape(sh);
    if (ntiles <= 0) return;
    const dim3 grid((unsigned)sh.blocks), block((unsigned)(64 * sh.waves_per_block));
#define NEMO_ENS_MIXED(R, OW, PF)                                                      \
    if (sh.rows == R && sh.cols == OW && sh.prefetch == PF) {                          \
        k_ens_mixed<R, OW, PF><<<grid, block, 0, s>>>(in, p, out, tiles, ntiles,       \
                                                      tide);                           \
        NEMO_LAUNCH_CHECK();                                                           \
        return;                                                                        \
    }
#define NEMO_ENS_MIXED_GRID(R, OW, PF)                                                 \
    if (sh.rows == R && sh.cols == OW && sh.prefetch == PF) {                          \
        k_ens_mixed_grid<R, OW, PF><<<dim3((unsigned)ntiles), dim3(64), 0, s>>>(       \
            in, p, out, tiles, tide);                                                  \
        NEMO_LAUNCH_CHECK();                                                           \
        return;                                                                        \
    }
    if (sh.blocks) {
        NEMO_ENS_PERSISTENT(NEMO_ENS_MIXED)
    } else {
        NEMO_ENS_GRID(NEMO_ENS_MIXED_GRID)
    }
#undef NEMO_ENS_MIXED
#undef NEMO_ENS_MIXED_GRID
    unsupported(sh);
}

int ens_domain_cols(const Bounds &b)
{
    // 61-column strips cost about 27/25 of 56-column ones
    return 27 * wave::strips(b, 61) < 25 * wave::strips(b, 56) ? 61 : 56;
}

int ens_max_waves_per_cu(int precision, int rows, int cols, int prefetch)
{
    int blocks = 0;
#define NEMO_ENS_OCC(R, OW, PF)                                                        \
    if (rows == R && cols == OW && prefetch == PF) {                                   \
        const void *k = precision == 64 ? reinterpret_cast<const void *>(&k_ens_f64<R, OW, PF>) \
                                        : reinterpret_cast<const void *>(&k_ens_mixed<R, OW, PF>); \
        NEMO_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, 64, 0)); \
        return blocks;                                                                 \
    }
    NEMO_ENS_PERSISTENT(NEMO_ENS_OCC)
#undef NEMO_ENS_OCC
    NEMO_FATAL("ensemble launch: no persistent kernel for %d rows x %d columns, prefetch %d",
               rows, cols, prefetch);
}

}  // namespace nemo
