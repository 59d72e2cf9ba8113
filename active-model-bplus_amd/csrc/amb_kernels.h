// amb_kernels.h -- host-side declarations of the HIP kernels' launchers (internal).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace amb {

// Coefficients of one step with dx, dy, dt and the model folded in (host-computed
// in double, cast to the arithmetic type T).
template <typename T>
struct StepCoef {
    T a, b, c, kappa, lam, zeta;
    T gxc, gxe, gyc, gye;  // G3: centre/edge smoothing weights times 1/dx (1/dy)
    T lcc, lex, ley, lck;  // L3: centre, x-neighbours, y-neighbours, corners
    T p0;                  // D8oD8 centre weight of -(mu_p'' along x and y)
    T px[9], py[9];        // D8oD8 weights (index 1..8) times -1/dx^2, -1/dy^2
    T lxx[3], lyy[3];      // G3xoG3x row weights times -1/dx^2; lyy[0] = -1/dy^2
    T zx, zy;              // 1/dx, 1/dy (divergence of the circulating current)
    T dxw[5], dyw[5];      // D8 weights (index 1..4) times 1/dx, 1/dy (currents through D8)
    T dt;
    T amp;                 // sqrt(2T) sqrt(1/(dt dx dy))
};

template <typename T>
struct StepArgs {
    const T* in;
    T* out;
    int ny, nx;
    int seg_rows;     // > 0: strips, this many output rows per workgroup
    int ntx, nty;     // tiles along x and y
    int xcd_chunk;    // tiles per XCD: block b takes tile (b % 8) xcd_chunk + b / 8 (xcd_chunk below)
    uint32_t ntx_inv; // floor(2^32 / ntx) + 1, or 0 to divide by ntx (tile_row)
    StepCoef<T> k;
    uint32_t key0, key1;
    const long long* step_base;  // device step counter; noise uses *step_base + step_off
    int step_off;
    const double* noise;         // explicit normals [2][ny][nx] of this step (noise mode 2)
    double* part;                // nullable: per-tile (sum, non-finite count) of the new field
};

// kNoisePhiloxOdd: Philox on fields whose columns do not split into groups of four.  It is a
// kernel of its own: compiled into kNoisePhilox's, its paths cost aligned fields up to 4%
// (FP64 2048^2 65.8 -> 68.2 us a step, 109 instead of 97 VGPRs).  The host chooses it from
// the field's columns (philox_mode); callers name kNoisePhilox.
enum NoiseMode { kNoiseNone = 0, kNoisePhilox = 1, kNoiseBuffer = 2, kNoisePhiloxOdd = 3 };
inline int philox_mode(int64_t nx) { return nx % 4 == 0 ? kNoisePhilox : kNoisePhiloxOdd; }

struct TileShape {
    int tw, th, nt;  // tile columns, tile rows, workgroup size
};

// Compiled tile configurations (index = autotuner choice): X(index, TW, TH, NT).  A field
// without a chosen one runs in run_tile's; options name the occupancy rule's, which follows an
// order of preference per kernel (default_tile in amb_capi.hip).
#define AMB_F32_TILES(X) X(0, 32, 48, 512) X(1, 32, 24, 256) X(2, 32, 32, 256) X(3, 64, 32, 512) X(4, 64, 16, 256) X(5, 32, 16, 256) X(6, 16, 16, 128) X(7, 16, 8, 128) X(8, 8, 8, 64) X(9, 32, 32, 512) X(10, 32, 16, 512)
#define AMB_F64_TILES(X) X(0, 32, 32, 256) X(1, 64, 16, 256) X(2, 32, 16, 256) X(3, 32, 32, 512) X(4, 16, 16, 128) X(5, 16, 8, 128) X(6, 8, 8, 64) X(7, 32, 16, 512)
constexpr int kSquare512F32 = 9, kSquare512F64 = 3;  // 32x32 tiles of 512 threads
// FP32 orders of preference, measured on MI355X (the times below predate the step's wave
// priorities, which took 2-4% off every shape).  Noisy: 32x32 tiles of 512 threads are
// fastest at 4096^2 (108.1 us per step; 32x48 111.5 us, 32x16 116.9 us, the others 120-139
// us): their 35 KB of LDS and 61 VGPRs let four workgroups, 8 waves per SIMD, share a CU,
// against three for 32x48, and the extra halo work costs less than the extra waves hide;
// at 1024^2 they tie with 64x32 (11.02 / 11.04 us).  Noiseless, measured with the current
// step (stage B's rows formed just before use, so its 17-tap windows fit 58 VGPRs without
// spilling): 32x32 tiles of 512 threads are fastest at 4096^2 (84.9 us; 32x48 86.3 us, 32x16
// 93.4 us), 2048^2 (25.0 / 25.6 us) and 1024^2 (8.92 us, 64x32 8.94 us, 32x48 9.79 us).
// 16x8 serves the smallest fields (256^2: 5.1 us noiseless, 6.2 us noisy, 8x8 6.0 us).
#define AMB_F32_NOISY_ORDER 9, 0, 3, 2, 1, 4, 5, 6, 7, 8
#define AMB_F32_NOISELESS_ORDER 9, 0, 3, 1, 5, 2, 4, 6, 7, 8
// FP64, noisy and noiseless alike: 32x32 tiles of 512 threads (held to 128 VGPRs, so two
// workgroups, 16 waves, share a CU) are fastest at 4096^2 (291.0 / 178.6 us per step against
// 321.0 / 213.2 us for 256 threads, both before the fitted noise polynomials and the priorities); 16x8 serves the smallest fields (256^2: 5.56 us, 16x16
// 5.77 us, 8x8 5.88 us).
#define AMB_F64_ORDER 3, 0, 2, 1, 4, 5, 6

// The tile that a field runs in when none was chosen: 32x16 tiles of 512 threads while one
// round of them holds the field, else 32x32 tiles of 512 threads, or kStrips (step_grid).  us a
// step, 32x16 / 32x32 / the tile of the orders above:
//   side      FP32 T = 0.05        FP32 T = 0           FP64 T = 0.05        FP64 T = 0
//   64        4.41 / 5.26 / 4.89   3.64 / 4.59 / 4.05   5.64 / 7.16 / 6.16   4.48 / 5.41 / 4.27
//   128       4.76 / 5.44 / 5.54   3.89 / 4.79 / 4.43   6.28 / 7.26 / 7.17   4.63 / 5.48 / 4.76
//   256       5.31 / 5.89 / 5.91   4.31 / 5.24 / 4.73   7.00 / 8.02 / 7.96   5.08 / 6.15 / 5.19
//   512       5.96 / 6.08 / 6.08   4.85 / 5.40 / 5.40   8.33 / 8.00 / 8.00   6.23 / 6.20 / 6.20
//   608       6.84 / 7.52 / 7.77   5.72 / 6.55 / 6.78   10.1 / 10.6 / 10.6   7.82 / 8.34 / 8.34
//   704       7.40 / 7.37 / 9.46   6.25 / 6.47 / 8.40   13.5 / 10.6 / 12.6   9.60 / 8.30 / 9.34
//   768       9.21 / 7.79 / 9.88   7.29 / 6.93 / 8.38   15.1 / 14.7 / 16.0   11.1 / 11.2 / 11.4
//   1088      14.4 / 11.3 / 15.5   11.2 / 10.2 / 13.4   26.3 / 22.0 / 26.5   18.5 / 16.5 / 19.6
// (a round is four workgroups per compute unit in FP32, three in FP64).  FP64 32x32 tiles that
// fit one to a compute unit beat more than 1.5 32x16 tiles to each (448^2 8.30 / 8.46).
constexpr int kWide512F32 = 10, kWide512F64 = 7;
int run_tile(int precision, int noise, int64_t ny, int64_t nx);
constexpr int kStrips = -1;  // in a tile's place: strips of columns (step_grid)

// Tile shapes compiled per precision (index = autotuner choice).
int tile_count(int precision);
TileShape tile_shape(int precision, int index);

// Workgroups of one step of a whole field: ntx x nty tiles of a shape or, on large fields for
// which none was chosen, strips of columns each seg_rows rows long (amb_march.h; the rule and its
// reason are at strip_grid).
struct StepGrid {
    int ntx, nty;
    int seg_rows;  // 0: tiles
};
constexpr int kMarchCols = 112;  // columns of a strip
constexpr int march_threads(int noise) { return noise != kNoiseNone ? 512 : 256; }
StepGrid step_grid(int precision, int tile, int noise, int64_t ny, int64_t nx);
int device_cus();  // compute units of the current device

// Order of a step's tiles.  gfx950 dispatches block b to XCD b % 8, and neighbouring tiles read
// each other's rows, so each XCD takes a contiguous run of xcd_chunk(tiles) tiles and finds
// those rows in its own L2; the grid is 8 xcd_chunk blocks, those without a tile leave at once.
// In plain order a step is 1 to 1.5 us longer (640^2 in 800 tiles 7.2 us, 608^2 in 722, which
// no multiple of eight used to leave in plain order, 8.7).  Fields of few tiles keep to as few
// XCDs as hold them one to a compute unit: 128^2 FP32 T = 0.05 in 32 tiles 4.9 us on one XCD, 5.3
// on two, 5.5 on eight; FP64 6.4, 6.8, 7.1; from 3/8 of the device on all eight are as fast.
// Several such fields at once share the first XCD and still gain: 128^2 FP64 on 1, 2, 4 and 8 threads
// 6.4, 6.4, 12.9 and 19.5 us a step of all of them, spread over the XCDs in larger tiles 7.4, 7.5,
// 15.2 and 23.9; in four processes 6.4 to 7.1 us against 8.6 where each has a hardware queue.
inline int xcd_chunk(int64_t tiles)
{
    const int64_t cus = device_cus();
    const int xcds = 8 * tiles <= cus ? 1 : 4 * tiles <= cus ? 2 : 8 * tiles <= 3 * cus ? 4 : 8;
    return (int)((tiles + xcds - 1) / xcds);
}

// The tile coordinates of index t without a division at the head of every workgroup: exact
// while t ntx < 2^32, the host passes 0 where that may not hold.
inline uint32_t ntx_inverse(int64_t ntx, int64_t nty)
{
    return ntx > 1 && ntx * nty * ntx < ((int64_t)1 << 32) ? (uint32_t)(((uint64_t)1 << 32) / (uint64_t)ntx) + 1 : 0;
}

// Launches one fused step.  Returns a hipError_t.
hipError_t launch_step_f32(const StepArgs<float>& a, int tile, int noise, hipStream_t s);
hipError_t launch_step_f64(const StepArgs<double>& a, int tile, int noise, hipStream_t s);
hipError_t prepare_step_kernels();  // raises the dynamic-LDS limit of large tiles
int tile_occupancy(int precision, int tile, int noise);  // resident workgroups per CU (>= 1)

// Adds `n` to the device step counter (a one-lane kernel, graph-capturable).
hipError_t launch_advance(long long* step, long long n, hipStream_t s);

// One observable (AMB_OBS_*) of the current step into `out` (n = ny*nx doubles for the
// chemical potentials, 2n for currents); `tmp` is 2n doubles of workspace.
hipError_t launch_observable_f32(const StepArgs<float>& a, int which, double* tmp, double* out, hipStream_t s);
hipError_t launch_observable_f64(const StepArgs<double>& a, int which, double* tmp, double* out, hipStream_t s);

// Final reduction of the per-tile partials (sum, non-finite count) that the last step of
// a run writes: one block, fixed order.
hipError_t launch_reduce_tiles(const double* part, int64_t ntiles, double* sum, unsigned long long* bad,
                               hipStream_t s);

// FP64 sum and non-finite count of a field: deterministic two-pass reduction (at most
// kReduceBlocks partials; their number depends only on the field's size).
constexpr int kReduceBlocks = 2048;
hipError_t launch_reduce_f32(const float* phi, int64_t n, double* part, unsigned long long* bad_part,
                             double* sum, unsigned long long* bad, hipStream_t s);
hipError_t launch_reduce_f64(const double* phi, int64_t n, double* part, unsigned long long* bad_part,
                             double* sum, unsigned long long* bad, hipStream_t s);

}  // namespace amb
