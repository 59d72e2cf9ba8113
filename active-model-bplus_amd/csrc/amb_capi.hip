// amb_capi.hip -- host runtime behind the C ABI declared in include/amb.h.
//
// One handle owns: two device field buffers (ping-pong; the fused step cannot
// update in place because each tile reads its neighbours' halo), a device step
// counter that keys the Philox noise, a private stream, cached hipGraph
// executables of kGraphSteps steps, and small reduction buffers.  The reference's
// Integrator (src/integrator.cu:286-538) instead owns 11 FP64 arrays plus cuRAND
// state and launches three kernels per step from a host loop.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <tuple>
#include <vector>

#include "amb.h"
#include "amb_internal.h"
#include "amb_kernels.h"
#include "amb_math.h"

namespace {

thread_local std::string g_error;

}  // namespace

namespace amb {

int fail(int code, const std::string& msg)
{
    g_error = msg;
    return code;
}

int fail_hip(hipError_t e, const char* what)
{
    g_error = std::string(what) + ": " + hipGetErrorString(e);
    return AMB_E_HIP;
}

void clear_error() { g_error.clear(); }

int check_device()
{
    int n = 0;
    const hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        return fail(AMB_E_NODEVICE, "no HIP device is visible (the integrator runs on an AMD GPU only)");
    }
    return AMB_OK;
}

template <typename T>
StepCoef<T> make_coef(const amb_stencil& st, const amb_model& m)
{
    StepCoef<T> k{};
    const double idx = 1.0 / st.dx, idy = 1.0 / st.dy;
    const double idx2 = idx * idx, idy2 = idy * idy;
    k.a = (T)m.a;
    k.b = (T)m.b;
    k.c = (T)m.c;
    k.kappa = (T)m.kappa;
    k.lam = (T)m.lamb;
    k.zeta = (T)m.zeta;
    k.gxc = (T)(kG3S[0] * idx);
    k.gxe = (T)(kG3S[1] * idx);
    k.gyc = (T)(kG3S[0] * idy);
    k.gye = (T)(kG3S[1] * idy);
    // L3 = S2x/dx^2 + S2y/dy^2 written per neighbour class.
    k.lcc = (T)(-3.0 * (idx2 + idy2));
    k.lex = (T)(1.5 * idx2 + 0.5 * idy2);
    k.ley = (T)(0.5 * idx2 + 1.5 * idy2);
    k.lck = (T)(-0.25 * (idx2 + idy2));
    k.p0 = (T)(-(idx2 + idy2) * kD8D8[0]);
    for (int j = 0; j < 9; ++j) {
        k.px[j] = (T)(-idx2 * kD8D8[j]);
        k.py[j] = (T)(-idy2 * kD8D8[j]);
    }
    // G3xoG3x: the smoothing weights across rows are folded in (lxx[|a|]); for
    // G3yoG3y the smoothing is applied to each row first, so lyy[0] = -1/dy^2.
    for (int a = 0; a < 3; ++a) {
        k.lxx[a] = (T)(-idx2 * kG3G3S[a]);
        k.lyy[a] = (T)(a == 0 ? -idy2 : 0.0);
    }
    k.zx = (T)idx;
    k.zy = (T)idy;
    // Noise amplitude sqrt(2T) * sqrt(1/(dt dx dy)) (src/parameters.h:50,86).
    const double amp = std::sqrt(2.0 * m.T) * std::sqrt(1.0 / (st.dt * st.dx * st.dy));
    for (int j = 0; j < 5; ++j) {
        k.dxw[j] = (T)(idx * kD8[j]);
        k.dyw[j] = (T)(idy * kD8[j]);
    }
    k.dt = (T)st.dt;
    k.amp = (T)amp;
    return k;
}

template StepCoef<float> make_coef<float>(const amb_stencil&, const amb_model&);
template StepCoef<double> make_coef<double>(const amb_stencil&, const amb_model&);

int validate_params(int64_t ny, int64_t nx, const amb_stencil* st, const amb_model* m)
{
    if (!st || !m) return fail(AMB_E_ARG, "stencil and model must not be null");
    if (ny <= 0 || nx <= 0) return fail(AMB_E_ARG, "field must have at least one row and one column");
    if (ny > (int64_t)0x7fffffff || nx > (int64_t)0x7fffffff || ny * nx > ((int64_t)1 << 40))
        return fail(AMB_E_ARG, "field is too large");
    const double v[] = {st->dt, st->dx, st->dy, m->a, m->b, m->c, m->kappa, m->lamb, m->zeta, m->T};
    for (double x : v)
        if (!std::isfinite(x)) return fail(AMB_E_ARG, "stencil and model parameters must be finite");
    if (!(st->dx > 0.0) || !(st->dy > 0.0)) return fail(AMB_E_ARG, "dx and dy must be positive");
    if (m->T < 0.0) return fail(AMB_E_ARG, "temperature must be non-negative");
    if (m->T > 0.0 && !(st->dt > 0.0)) return fail(AMB_E_ARG, "noise needs a positive dt");
    return AMB_OK;
}

// The pieces and their events, made on the stream's device, whichever is current (a stream takes
// its own device's events only).
static hipError_t make_pieces(HostStage& st, size_t bytes, hipStream_t s)
{
    int current = 0;
    hipDevice_t own = 0;
    hipError_t e = hipGetDevice(&current);
    if (e == hipSuccess) e = hipStreamGetDevice(s, &own);
    if (e == hipSuccess && own != current) e = hipSetDevice(own);
    if (e != hipSuccess) return e;
    for (int k = 0; k < 2 && e == hipSuccess; ++k) {
        if (!st.piece[k]) e = hipHostMalloc(&st.piece[k], bytes, hipHostMallocDefault);
        if (e == hipSuccess && !st.filled[k]) e = hipEventCreateWithFlags(&st.filled[k], hipEventDisableTiming);
    }
    const hipError_t back = own != current ? hipSetDevice(current) : hipSuccess;
    return e == hipSuccess ? back : e;
}

// Fields above one piece of doubles go through two pinned pieces: the copy engine fills one while the
// host empties the other into the caller's memory, whose first touch and the widening of FP32
// values are what takes the time.  A copy to pageable memory stages one piece after the other,
// and FP32 fields took a vector of their own: a run of 400 steps of 1024^2 FP32 and its field
// 4.23 ms, now 4.03; a run of 640 steps of 48 members and their fields 22.2 ms, now 20.7.  Small
// fields are quicker copied at once (128^2 FP64 by 9 us; a copy on the stream that is not pinned
// also made the next integrator 45 us slower to create), and four threads, each with pieces
// of its own, gained on mu and J of 1024^2 FP64 (2.0 -> 1.8 ms) but lost on its FP32 field (0.3 ms).
hipError_t copy_out(HostStage& st, const void* dev, int64_t n, int precision, double* out, hipStream_t s)
{
    constexpr size_t kPiece = kStageDoubles * sizeof(double);
    const size_t esize = precision == AMB_F32 ? sizeof(float) : sizeof(double);
    hipError_t e = hipSuccess;
    if (n <= kStageDoubles) {
        std::vector<float> tmp(precision == AMB_F32 ? n : 0);
        void* dst = precision == AMB_F32 ? static_cast<void*>(tmp.data()) : out;
        if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
        if ((e = hipMemcpy(dst, dev, (size_t)n * esize, hipMemcpyDeviceToHost)) != hipSuccess) return e;
        for (size_t i = 0; i < tmp.size(); ++i) out[i] = (double)tmp[i];
        return hipSuccess;
    }
    if (!st.filled[1] && (e = make_pieces(st, kPiece, s)) != hipSuccess) return e;
    const int64_t per = (int64_t)(kPiece / esize), pieces = (n + per - 1) / per;
    auto fill = [&](int64_t i) {
        const int64_t count = std::min(per, n - i * per);
        const hipError_t f = hipMemcpyAsync(st.piece[i & 1], static_cast<const char*>(dev) + (size_t)(i * per) * esize,
                                            (size_t)count * esize, hipMemcpyDeviceToHost, s);
        return f == hipSuccess ? hipEventRecord(st.filled[i & 1], s) : f;
    };
    for (int64_t i = 0; i < 2 && i < pieces && e == hipSuccess; ++i) e = fill(i);
    for (int64_t i = 0; i < pieces && e == hipSuccess; ++i) {
        if ((e = hipEventSynchronize(st.filled[i & 1])) != hipSuccess) break;
        const int64_t count = std::min(per, n - i * per);
        double* dst = out + i * per;
        if (precision == AMB_F32) {
            const float* src = static_cast<const float*>(st.piece[i & 1]);
            for (int64_t j = 0; j < count; ++j) dst[j] = (double)src[j];
        } else {
            std::memcpy(dst, st.piece[i & 1], (size_t)count * sizeof(double));
        }
        if (i + 2 < pieces) e = fill(i + 2);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no copy into a piece outlives the call
    return e;
}

void release(HostStage& st)
{
    for (int k = 0; k < 2; ++k) {
        if (st.piece[k]) (void)hipHostFree(st.piece[k]);
        if (st.filled[k]) (void)hipEventDestroy(st.filled[k]);
        st.piece[k] = nullptr;
        st.filled[k] = nullptr;
    }
}

int grid_tiles(int64_t n, int t) { return (int)((n + t - 1) / t); }

// The occupancy rule's tile, which options report when none was chosen (such a field runs in
// run_tile's; amb_get_step_shape tells) and whose tiles bound amb_run_noalloc's fields: in order of
// preference (AMB_F32_NOISY_ORDER, AMB_F32_NOISELESS_ORDER or AMB_F64_ORDER), the first shape of 256 or more threads whose tiles fill the device's
// resident workgroups either for at least 8 rounds or in whole-or-mostly-full rounds (a
// last round under half full leaves most CUs idle for a round).  Fields too small for one
// round of such a shape take the shape that puts nearest 8 waves on each CU (in ratio; the
// earlier in the order on a tie): fewer waves leave each CU a single workgroup's latency to
// hide, while many small tiles pay their halo several times over.  The tiles of 64 and 128
// threads only serve that way: their boxes hold 4.5-10.6x their area of phi (32x32 tiles
// 2.4x), so where they fill a round (FP64 16x8 at 512^2) a half round of 32x32 tiles is
// still faster (9.0 against 10.2 us).  It picked the fastest of the shapes it lists, or one within
// 2% of it, before the tiles were handed to the XCDs in runs; run_tile's are up to 1.4 times as
// fast now (its table).
int default_tile(int precision, int64_t ny, int64_t nx, int noise)
{
    int device = 0, cus = 256;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) {
        (void)hipGetLastError();
        cus = 256;
    }
    static constexpr int kNoisyF32[] = {AMB_F32_NOISY_ORDER};
    static constexpr int kNoiselessF32[] = {AMB_F32_NOISELESS_ORDER};
    static constexpr int kF64[] = {AMB_F64_ORDER};
#define AMB_COUNT_ONE(i, tw, th, nt) +1
    static_assert(sizeof(kNoisyF32) / sizeof(kNoisyF32[0]) == kWide512F32 &&
                      sizeof(kNoiselessF32) / sizeof(kNoiselessF32[0]) == kWide512F32 &&
                      kWide512F32 + 1 == 0 AMB_F32_TILES(AMB_COUNT_ONE),
                  "the FP32 orders must list every FP32 tile shape but the last");
    static_assert(sizeof(kF64) / sizeof(kF64[0]) == kWide512F64 && kWide512F64 + 1 == 0 AMB_F64_TILES(AMB_COUNT_ONE),
                  "the FP64 order must list every FP64 tile shape but the last");
#undef AMB_COUNT_ONE
    // fields that run in strips: the tile that comes next to them
    if (run_tile(precision, noise, ny, nx) == kStrips) return precision == AMB_F32 ? kSquare512F32 : kSquare512F64;
    const int n = precision == AMB_F32 ? kWide512F32 : kWide512F64;
    const int* order = precision != AMB_F32 ? kF64 : noise == kNoiseNone ? kNoiselessF32 : kNoisyF32;
    int best = 0;
    double best_gap = 0.0;
    for (int k = 0; k < n; ++k) {
        const int i = order ? order[k] : k;
        const TileShape t = tile_shape(precision, i);
        const int64_t tiles = (int64_t)grid_tiles(nx, t.tw) * grid_tiles(ny, t.th);
        const int64_t slots = (int64_t)cus * tile_occupancy(precision, i, noise);
        const int64_t full = tiles / slots, rest = tiles % slots;
        if (t.nt >= 256 && (full >= 8 || (full >= 1 && (rest == 0 || 2 * rest >= slots)))) return i;
        const double waves = (double)tiles * (t.nt / 64);
        const double gap = std::fabs(std::log(waves / (8.0 * cus)));
        if (k == 0 || gap < best_gap - 1e-9) {
            best = i;
            best_gap = gap;
        }
    }
    return best;
}

// ---- tuning table: the autotuners' choices, per (precision, grid, noise) ------------
namespace {
struct Tuned {
    int tile;
    int timed;  // AMB_TUNED_*
};
std::mutex g_tune_mutex;
std::map<std::tuple<int, int64_t, int64_t, int>, Tuned> g_tune;
}  // namespace

bool tuned_tile(int precision, int64_t ny, int64_t nx, int noise, int* tile, int* timed)
{
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    const auto it = g_tune.find({precision, ny, nx, noise != kNoiseNone});
    if (it == g_tune.end()) return false;
    *tile = it->second.tile;
    if (timed) *timed = it->second.timed;
    return true;
}

// An ensemble's timing knows nothing of strips: it does not replace an entry that decides between
// them and a tile for single fields.
void record_tile(int precision, int64_t ny, int64_t nx, int noise, int tile, int timed)
{
    const bool strips = timed == AMB_TUNED_TILES && run_tile(precision, noise, ny, nx) == kStrips;
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    const auto at = g_tune.insert({{precision, ny, nx, noise != kNoiseNone}, {tile, timed}});
    if (!at.second && !(strips && at.first->second.timed != AMB_TUNED_TILES)) at.first->second = {tile, timed};
}

}  // namespace amb

using namespace amb;

struct amb_handle {
    int device = 0;
    hipStream_t stream = nullptr;
    int64_t ny = 0, nx = 0;
    amb_stencil stencil{};
    amb_model model{};
    amb_options options{};
    int precision = AMB_F64;
    size_t esize = 8;
    void* buf[2] = {nullptr, nullptr};
    int cur = 0;
    long long* d_step = nullptr;
    int64_t timestep = 0;
    double* d_part = nullptr;
    unsigned long long* d_bad_part = nullptr;
    double* d_tile_part = nullptr;         // (sum, non-finite count) per tile, written by a run's last step
    int64_t parts = 0;                     // how many of them the last step wrote
    double* d_sum = nullptr;
    unsigned long long* d_bad = nullptr;   // after d_sum
    double last_sum = 0.0;                 // mass and non-finite count found by the last amb_run
    int64_t last_bad = 0;
    double* h_sum = nullptr;               // pinned
    unsigned long long* h_bad = nullptr;   // after h_sum
    double* d_obs = nullptr;               // 10 n doubles, allocated by the first getter
    double* d_noise = nullptr;             // explicit normals (test mode)
    int64_t noise_steps = 0, noise_used = 0;
    int tile = 0;                          // index into the precision's tile table: chosen, or default_tile's
    bool tile_chosen = false;              // by an option, the tuning table, amb_set_tile or the autotuner
    hipGraphExec_t graph[2] = {nullptr, nullptr};
    int graph_tile[2] = {-1, -1};
    int graph_noise[2] = {-1, -1};
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    SkCache* sk = nullptr;                 // structure-factor plan and buffers (lazy)
    HostStage stage;                       // getters
};

namespace {

constexpr int kGraphSteps = 32;  // even: a graph returns the field to the buffer it started in

// The tile (or kStrips) of the handle's launches.
int launch_tile(const amb_handle* h, int noise)
{
    return h->tile_chosen ? h->tile : run_tile(h->precision, noise, h->ny, h->nx);
}

template <typename T>
StepArgs<T> step_args(const amb_handle* h, int tile, int parity_in, int step_off, int noise_mode, bool reduce = false)
{
    StepArgs<T> a{};
    const StepGrid g = step_grid(h->precision, tile, noise_mode, h->ny, h->nx);
    a.in = static_cast<const T*>(h->buf[parity_in & 1]);
    a.out = static_cast<T*>(h->buf[(parity_in + 1) & 1]);
    a.ny = (int)h->ny;
    a.nx = (int)h->nx;
    a.ntx = g.ntx;
    a.nty = g.nty;
    a.seg_rows = g.seg_rows;
    a.xcd_chunk = xcd_chunk((int64_t)a.ntx * a.nty);
    a.ntx_inv = ntx_inverse(a.ntx, a.nty);
    a.k = make_coef<T>(h->stencil, h->model);
    a.key0 = (uint32_t)h->options.seed;
    a.key1 = (uint32_t)(h->options.seed >> 32);
    a.step_base = h->d_step;
    a.step_off = step_off;
    a.noise = nullptr;
    if (noise_mode == kNoiseBuffer)
        a.noise = h->d_noise + (size_t)h->noise_used * 2 * (size_t)(h->ny * h->nx);
    a.part = reduce ? h->d_tile_part : nullptr;
    return a;
}

// One step; with `reduce` (the last step of a run) every tile also writes its partial
// of the fused finite check and FP64 mass.
hipError_t launch_step(const amb_handle* h, int parity_in, int step_off, int noise_mode, bool reduce = false)
{
    const int tile = launch_tile(h, noise_mode);
    if (h->precision == AMB_F32)
        return launch_step_f32(step_args<float>(h, tile, parity_in, step_off, noise_mode, reduce), tile, noise_mode,
                               h->stream);
    return launch_step_f64(step_args<double>(h, tile, parity_in, step_off, noise_mode, reduce), tile, noise_mode,
                           h->stream);
}

void choose_tile(amb_handle* h, int tile, bool strips = false)
{
    h->tile = tile;
    h->tile_chosen = !strips;
}

// The tuning table's entry, when it has one for the handle's field (one timed among tiles alone
// is none for a field that runs in strips).
bool take_tuned(amb_handle* h, int noise)
{
    int tile = 0, timed = 0;
    if (!tuned_tile(h->precision, h->ny, h->nx, noise, &tile, &timed)) return false;
    if (timed == AMB_TUNED_TILES && run_tile(h->precision, noise, h->ny, h->nx) == kStrips) return false;
    choose_tile(h, tile, timed == AMB_TUNED_STRIPS);
    return true;
}

// Workgroups of one step, each writing one partial of the fused finite check.
int64_t parts_of(const amb_handle* h, int noise)
{
    const StepGrid g = step_grid(h->precision, launch_tile(h, noise), noise, h->ny, h->nx);
    return (int64_t)g.ntx * g.nty;
}

int noise_mode_of(const amb_handle* h)
{
    if (h->noise_used < h->noise_steps) return kNoiseBuffer;
    return h->model.T > 0.0 ? kNoisePhilox : kNoiseNone;
}

void drop_graphs(amb_handle* h)
{
    for (int p = 0; p < 2; ++p) {
        if (h->graph[p]) (void)hipGraphExecDestroy(h->graph[p]);
        h->graph[p] = nullptr;
        h->graph_tile[p] = -1;
        h->graph_noise[p] = -1;
    }
}

int build_graph(amb_handle* h, int parity, int noise_mode)
{
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return fail_hip(e, "hipStreamBeginCapture");
    for (int k = 0; k < kGraphSteps && e == hipSuccess; ++k)
        e = launch_step(h, parity + k, k, noise_mode, k == kGraphSteps - 1);
    if (e == hipSuccess) e = launch_advance(h->d_step, kGraphSteps, h->stream);
    const hipError_t e2 = hipStreamEndCapture(h->stream, &g);
    if (e != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return fail_hip(e, "step launch during graph capture");
    }
    if (e2 != hipSuccess) return fail_hip(e2, "hipStreamEndCapture");
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return fail_hip(e, "hipGraphInstantiate");
    if (h->graph[parity]) (void)hipGraphExecDestroy(h->graph[parity]);
    h->graph[parity] = exec;
    h->graph_tile[parity] = launch_tile(h, noise_mode);
    h->graph_noise[parity] = noise_mode;
    return AMB_OK;
}

// Enqueues nsteps steps on the handle's stream (no synchronisation).
int enqueue_steps(amb_handle* h, int64_t nsteps)
{
    hipError_t e;
    int64_t left = nsteps;
    while (left > 0) {
        const int mode = noise_mode_of(h);
        if (mode == kNoiseBuffer) {
            if ((e = launch_step(h, h->cur, 0, mode, true)) != hipSuccess) return fail_hip(e, "step launch");
            if ((e = launch_advance(h->d_step, 1, h->stream)) != hipSuccess) return fail_hip(e, "advance launch");
            h->parts = parts_of(h, mode);
            h->cur ^= 1;
            ++h->noise_used;
            --left;
            continue;
        }
        if (left >= kGraphSteps) {
            const int p = h->cur;
            if (!h->graph[p] || h->graph_tile[p] != launch_tile(h, mode) || h->graph_noise[p] != mode) {
                const int rc = build_graph(h, p, mode);
                if (rc != AMB_OK) return rc;
            }
            const int64_t reps = left / kGraphSteps;
            for (int64_t r = 0; r < reps; ++r)
                if ((e = hipGraphLaunch(h->graph[p], h->stream)) != hipSuccess) return fail_hip(e, "hipGraphLaunch");
            h->parts = parts_of(h, mode);
            left -= reps * kGraphSteps;
            continue;
        }
        for (int k = 0; k < left; ++k)
            if ((e = launch_step(h, h->cur + k, k, mode, k == left - 1)) != hipSuccess) return fail_hip(e, "step launch");
        if ((e = launch_advance(h->d_step, left, h->stream)) != hipSuccess) return fail_hip(e, "advance launch");
        h->parts = parts_of(h, mode);
        h->cur = (int)((h->cur + left) & 1);
        left = 0;
    }
    return AMB_OK;
}

// FP64 sum and non-finite count of the field into *sum and *bad (device or pinned memory).
hipError_t enqueue_reduce(amb_handle* h, double* sum, unsigned long long* bad)
{
    const int64_t n = h->ny * h->nx;
    return h->precision == AMB_F32
               ? launch_reduce_f32(static_cast<const float*>(h->buf[h->cur]), n, h->d_part, h->d_bad_part, sum, bad,
                                   h->stream)
               : launch_reduce_f64(static_cast<const double*>(h->buf[h->cur]), n, h->d_part, h->d_bad_part, sum, bad,
                                   h->stream);
}

// The last kernel of a reduction writes its two results straight into the handle's pinned
// memory: two copies of eight bytes after it cost as much as two steps of a small field (a run of
// 20 steps of 128^2 FP64 192 us with them, 181 without).
int wait_reduce(amb_handle* h, double* sum, int64_t* bad)
{
    const hipError_t e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return fail_hip(e, "hipStreamSynchronize");
    *sum = *h->h_sum;
    *bad = (int64_t)*h->h_bad;
    return AMB_OK;
}

int reduce_now(amb_handle* h, double* sum, int64_t* bad)
{
    const hipError_t e = enqueue_reduce(h, h->h_sum, h->h_bad);
    if (e != hipSuccess) return fail_hip(e, "reduction launch");
    return wait_reduce(h, sum, bad);
}

// Mass and non-finite count after a run of nsteps: the last step of the run wrote one
// partial per tile, summed here by one small fixed-order reduction; for nsteps = 0 the
// field is read in full.
int finish_run(amb_handle* h, int64_t nsteps, double* sum, int64_t* bad)
{
    if (nsteps == 0) {
        const int rc = reduce_now(h, sum, bad);
        if (rc == AMB_OK) {
            h->last_sum = *sum;
            h->last_bad = *bad;
        }
        return rc;
    }
    const hipError_t e = launch_reduce_tiles(h->d_tile_part, h->parts, h->h_sum, h->h_bad, h->stream);
    if (e != hipSuccess) return fail_hip(e, "reduction launch");
    const int rc = wait_reduce(h, sum, bad);
    if (rc != AMB_OK) return rc;
    h->last_sum = *sum;
    h->last_bad = *bad;
    return AMB_OK;
}

void release(amb_handle* h)
{
    if (!h) return;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    drop_graphs(h);
    sk_cache_free(h->sk);
    for (void* p : {h->buf[0], h->buf[1], (void*)h->d_step, (void*)h->d_part, (void*)h->d_bad_part,
                    (void*)h->d_tile_part, (void*)h->d_sum, (void*)h->d_obs, (void*)h->d_noise})
        if (p) (void)hipFree(p);
    release(h->stage);
    if (h->h_sum) (void)hipHostFree(h->h_sum);
    if (h->ev0) (void)hipEventDestroy(h->ev0);
    if (h->ev1) (void)hipEventDestroy(h->ev1);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
}

int upload_field(amb_handle* h, const double* field, int which)
{
    const size_t n = (size_t)(h->ny * h->nx);
    hipError_t e;
    if (h->precision == AMB_F32) {
        std::vector<float> tmp(n);
        for (size_t i = 0; i < n; ++i) tmp[i] = (float)field[i];
        e = hipMemcpy(h->buf[which], tmp.data(), n * sizeof(float), hipMemcpyHostToDevice);
    } else {
        e = hipMemcpy(h->buf[which], field, n * sizeof(double), hipMemcpyHostToDevice);
    }
    return e == hipSuccess ? AMB_OK : fail_hip(e, "hipMemcpy (field upload)");
}

// Computes observable `which` into d_obs + 2n (workspace d_obs[0, 2n)); allocated on
// the first getter call.
int compute_observable(amb_handle* h, int which)
{
    const size_t n = (size_t)(h->ny * h->nx);
    hipError_t e;
    if (!h->d_obs) {
        if ((e = hipMalloc(&h->d_obs, 4 * n * sizeof(double))) != hipSuccess) return fail_hip(e, "hipMalloc");
    }
    const int mode = noise_mode_of(h), tile = launch_tile(h, mode);
    if (h->precision == AMB_F32) {
        StepArgs<float> a = step_args<float>(h, tile, h->cur, 0, mode);
        if (mode != kNoiseBuffer) a.noise = nullptr;
        e = launch_observable_f32(a, which, h->d_obs, h->d_obs + 2 * n, h->stream);
    } else {
        StepArgs<double> a = step_args<double>(h, tile, h->cur, 0, mode);
        if (mode != kNoiseBuffer) a.noise = nullptr;
        e = launch_observable_f64(a, which, h->d_obs, h->d_obs + 2 * n, h->stream);
    }
    if (e != hipSuccess) return fail_hip(e, "observable launch");
    return AMB_OK;
}

}  // namespace

namespace amb {

int handle_view(amb_handle* h, FieldView* v)
{
    if (!h || !v) return fail(AMB_E_ARG, "handle must not be null");
    v->cur = h->buf[h->cur];
    v->other = h->buf[h->cur ^ 1];
    v->ny = h->ny;
    v->nx = h->nx;
    v->precision = h->precision;
    v->stream = h->stream;
    return AMB_OK;
}

int handle_field_sum(amb_handle* h, const double** sum)
{
    const hipError_t e = enqueue_reduce(h, h->d_sum, h->d_bad);
    if (e != hipSuccess) return fail_hip(e, "reduction launch");
    *sum = h->d_sum;
    return AMB_OK;
}

int handle_commit(amb_handle* h, int64_t steps, bool swapped)
{
    if (swapped) h->cur ^= 1;
    h->timestep += steps;
    const hipError_t e = launch_advance(h->d_step, steps, h->stream);
    return e == hipSuccess ? AMB_OK : fail_hip(e, "advance launch");
}

int handle_enqueue(amb_handle* h, int64_t steps)
{
    const int rc = enqueue_steps(h, steps);
    if (rc == AMB_OK) h->timestep += steps;
    return rc;
}

int handle_set_timestep(amb_handle* h, int64_t timestep)
{
    const long long v = timestep;
    hipError_t e = hipStreamSynchronize(h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(h->d_step, &v, sizeof v, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return fail_hip(e, "set timestep");
    h->timestep = timestep;
    return AMB_OK;
}

int64_t handle_timestep(const amb_handle* h) { return h->timestep; }

SkCache** handle_sk_cache(amb_handle* h) { return &h->sk; }

}  // namespace amb

extern "C" {

const char* amb_last_error(void) { return g_error.c_str(); }

int amb_set_field(amb_handle* h, const double* field)
{
    clear_error();
    if (!h || !field) return fail(AMB_E_ARG, "handle and field must not be null");
    hipError_t e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return fail_hip(e, "hipStreamSynchronize");
    return upload_field(h, field, h->cur);
}

int amb_device_count(int* count)
{
    if (!count) return fail(AMB_E_ARG, "count must not be null");
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) {
        (void)hipGetLastError();
        n = 0;
    }
    *count = n;
    return AMB_OK;
}

int amb_tile_count(int precision, int* count)
{
    if (!count || (precision != AMB_F32 && precision != AMB_F64)) return fail(AMB_E_ARG, "bad precision");
    *count = tile_count(precision);
    return AMB_OK;
}

int amb_tile_shape(int precision, int index, int* tile_cols, int* tile_rows, int* threads)
{
    if (precision != AMB_F32 && precision != AMB_F64) return fail(AMB_E_ARG, "bad precision");
    if (index < 0 || index >= tile_count(precision)) return fail(AMB_E_ARG, "tile index out of range");
    const TileShape t = tile_shape(precision, index);
    if (tile_cols) *tile_cols = t.tw;
    if (tile_rows) *tile_rows = t.th;
    if (threads) *threads = t.nt;
    return AMB_OK;
}

int amb_create(const double* field, int64_t ny, int64_t nx, const amb_stencil* stencil, const amb_model* model,
               const amb_options* options, amb_handle** out)
{
    clear_error();
    if (!out) return fail(AMB_E_ARG, "out must not be null");
    *out = nullptr;
    if (!field) return fail(AMB_E_ARG, "field must not be null");
    int rc = validate_params(ny, nx, stencil, model);
    if (rc != AMB_OK) return rc;
    amb_options opt{AMB_F64, 0, 0, 0};
    if (options) opt = *options;
    if (opt.precision != AMB_F32 && opt.precision != AMB_F64)
        return fail(AMB_E_ARG, "precision must be AMB_F32 or AMB_F64");
    if (opt.tile < 0 || opt.tile > tile_count(opt.precision)) return fail(AMB_E_ARG, "tile index out of range");
    if ((rc = check_device()) != AMB_OK) return rc;

    amb_handle* h = new (std::nothrow) amb_handle();
    if (!h) return fail(AMB_E_ARG, "out of host memory");
    h->ny = ny;
    h->nx = nx;
    h->stencil = *stencil;
    h->model = *model;
    h->options = opt;
    h->precision = opt.precision;
    h->esize = opt.precision == AMB_F32 ? 4 : 8;
    h->timestep = opt.timestep;
    const size_t n = (size_t)(ny * nx);
    hipError_t e;
#define AMB_CHECK(call)                                  \
    do {                                                 \
        e = (call);                                      \
        if (e != hipSuccess) {                           \
            const int code_ = fail_hip(e, #call);        \
            release(h);                                  \
            return code_;                                \
        }                                                \
    } while (0)
    AMB_CHECK(hipGetDevice(&h->device));
    AMB_CHECK(prepare_step_kernels());
    {
        const int noise = model->T > 0.0 ? kNoisePhilox : kNoiseNone;
        if (opt.tile > 0) choose_tile(h, opt.tile - 1);
        else if (!take_tuned(h, noise)) h->tile = default_tile(opt.precision, ny, nx, noise);
    }
    AMB_CHECK(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    AMB_CHECK(hipMalloc(&h->buf[0], n * h->esize));
    AMB_CHECK(hipMalloc(&h->buf[1], n * h->esize));
    AMB_CHECK(hipMalloc(&h->d_step, sizeof(long long)));
    AMB_CHECK(hipMalloc(&h->d_part, kReduceBlocks * sizeof(double)));
    AMB_CHECK(hipMalloc(&h->d_bad_part, kReduceBlocks * sizeof(unsigned long long)));
    {
        // partials for the tile shape with the most tiles (the tile may change); strips, on
        // large fields only, are far fewer
        int64_t most = 1;
        for (int t = 0; t < tile_count(h->precision); ++t) {
            const TileShape ts = tile_shape(h->precision, t);
            most = std::max(most, (int64_t)grid_tiles(nx, ts.tw) * grid_tiles(ny, ts.th));
        }
        AMB_CHECK(hipMalloc(&h->d_tile_part, (size_t)most * 2 * sizeof(double)));
    }
    static_assert(sizeof(double) == sizeof(unsigned long long), "one allocation for both results");
    AMB_CHECK(hipMalloc(&h->d_sum, 2 * sizeof(double)));
    h->d_bad = reinterpret_cast<unsigned long long*>(h->d_sum + 1);
    AMB_CHECK(hipHostMalloc(&h->h_sum, 2 * sizeof(double), hipHostMallocDefault));
    h->h_bad = reinterpret_cast<unsigned long long*>(h->h_sum + 1);
    AMB_CHECK(hipEventCreate(&h->ev0));
    AMB_CHECK(hipEventCreate(&h->ev1));
    const long long step0 = (long long)h->timestep;
    AMB_CHECK(hipMemcpy(h->d_step, &step0, sizeof(long long), hipMemcpyHostToDevice));
#undef AMB_CHECK
    rc = upload_field(h, field, 0);
    if (rc != AMB_OK) {
        release(h);
        return rc;
    }
    *out = h;
    return AMB_OK;
}

int amb_destroy(amb_handle* h)
{
    clear_error();
    release(h);
    return AMB_OK;
}

int amb_run(amb_handle* h, int64_t nsteps)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    if (nsteps < 0) return fail(AMB_E_ARG, "nsteps must be non-negative");
    int rc = enqueue_steps(h, nsteps);
    if (rc != AMB_OK) return rc;
    h->timestep += nsteps;
    double sum;
    int64_t bad;
    if ((rc = finish_run(h, nsteps, &sum, &bad)) != AMB_OK) return rc;
    if (bad != 0) return fail(AMB_E_NONFINITE, "an unknown numerical error occurred during simulation");
    return AMB_OK;
}

int amb_run_timed(amb_handle* h, int64_t nsteps, double* device_ms)
{
    clear_error();
    if (!h || !device_ms) return fail(AMB_E_ARG, "handle and device_ms must not be null");
    if (nsteps < 0) return fail(AMB_E_ARG, "nsteps must be non-negative");
    hipError_t e;
    if ((e = hipEventRecord(h->ev0, h->stream)) != hipSuccess) return fail_hip(e, "hipEventRecord");
    int rc = enqueue_steps(h, nsteps);
    if (rc != AMB_OK) return rc;
    if ((e = hipEventRecord(h->ev1, h->stream)) != hipSuccess) return fail_hip(e, "hipEventRecord");
    if ((e = hipEventSynchronize(h->ev1)) != hipSuccess) return fail_hip(e, "hipEventSynchronize");
    float ms = 0.f;
    if ((e = hipEventElapsedTime(&ms, h->ev0, h->ev1)) != hipSuccess) return fail_hip(e, "hipEventElapsedTime");
    *device_ms = ms;
    h->timestep += nsteps;
    double sum;
    int64_t bad;
    if ((rc = finish_run(h, nsteps, &sum, &bad)) != AMB_OK) return rc;
    if (bad != 0) return fail(AMB_E_NONFINITE, "an unknown numerical error occurred during simulation");
    return AMB_OK;
}

int amb_get_field(amb_handle* h, double* out)
{
    clear_error();
    if (!h || !out) return fail(AMB_E_ARG, "handle and out must not be null");
    const std::lock_guard<std::mutex> turn(h->stage.turn);
    const hipError_t e = copy_out(h->stage, h->buf[h->cur], h->ny * h->nx, h->precision, out, h->stream);
    return e == hipSuccess ? AMB_OK : fail_hip(e, "hipMemcpy (field download)");
}

int amb_get_observable(amb_handle* h, int which, double* out)
{
    return amb_get_observable_parts(h, which, out, h && out ? out + h->ny * h->nx : nullptr);
}

int amb_get_observable_parts(amb_handle* h, int which, double* out, double* second)
{
    clear_error();
    if (!h || !out) return fail(AMB_E_ARG, "handle and out must not be null");
    if (which < AMB_OBS_MU || which > AMB_OBS_J_RANDOM) return fail(AMB_E_ARG, "unknown observable");
    if (which > AMB_OBS_MU_ACTIVE && !second) return fail(AMB_E_ARG, "a current needs both components' arrays");
    const std::lock_guard<std::mutex> turn(h->stage.turn);  // d_obs too is one for all getters
    const int rc = compute_observable(h, which);
    if (rc != AMB_OK) return rc;
    const int64_t n = h->ny * h->nx;
    const double* result = h->d_obs + 2 * n;
    // Up to 16 KB a copy that waits on the stream itself is quicker than a wait and a copy (mu of
    // 30x64 18.7 us, 27), beyond it is not (mu of 64x64 34 us, 22.5).
    auto copy = [&](const double* from, int64_t count, double* to) {
        if (count <= 2048)
            return hipMemcpyWithStream(to, from, (size_t)count * sizeof(double), hipMemcpyDeviceToHost, h->stream);
        return copy_out(h->stage, from, count, AMB_F64, to, h->stream);
    };
    // A current's components lie one after the other.  A copy costs 11 us, so on small fields both
    // come in one and are dealt out on the host: mu and J of 64x64 55 us, in a copy each 63, of
    // 128x128 FP64 67 and 77; from 32768 sites on the array between costs more than the copy.
    hipError_t e = hipSuccess;
    std::unique_ptr<double[]> both;
    if (which <= AMB_OBS_MU_ACTIVE) {
        e = copy(result, n, out);
    } else if (second == out + n) {
        e = copy(result, 2 * n, out);
    } else if (n <= 16384 && (both.reset(new (std::nothrow) double[2 * n]), both)) {
        if ((e = copy(result, 2 * n, both.get())) == hipSuccess) {
            std::memcpy(out, both.get(), (size_t)n * sizeof(double));
            std::memcpy(second, both.get() + n, (size_t)n * sizeof(double));
        }
    } else {
        if ((e = copy(result, n, out)) == hipSuccess) e = copy(result + n, n, second);
    }
    return e == hipSuccess ? AMB_OK : fail_hip(e, "hipMemcpy (observable)");
}

int amb_get_timestep(const amb_handle* h, int64_t* timestep)
{
    if (!h || !timestep) return fail(AMB_E_ARG, "handle and timestep must not be null");
    *timestep = h->timestep;
    return AMB_OK;
}

int amb_get_params(const amb_handle* h, amb_stencil* stencil, amb_model* model)
{
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    if (stencil) *stencil = h->stencil;
    if (model) *model = h->model;
    return AMB_OK;
}

int amb_get_shape(const amb_handle* h, int64_t* ny, int64_t* nx)
{
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    if (ny) *ny = h->ny;
    if (nx) *nx = h->nx;
    return AMB_OK;
}

int amb_get_options(const amb_handle* h, amb_options* options)
{
    if (!h || !options) return fail(AMB_E_ARG, "handle and options must not be null");
    *options = h->options;
    options->timestep = h->timestep;
    options->tile = h->tile + 1;
    return AMB_OK;
}

int amb_get_step_shape(const amb_handle* h, int* cols, int* rows, int* threads, int* strips)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    const int noise = noise_mode_of(h), tile = launch_tile(h, noise);
    TileShape ts;
    if (tile == kStrips) ts = {kMarchCols, step_grid(h->precision, tile, noise, h->ny, h->nx).seg_rows, march_threads(noise)};
    else ts = tile_shape(h->precision, tile);
    if (cols) *cols = ts.tw;
    if (rows) *rows = ts.th;
    if (threads) *threads = ts.nt;
    if (strips) *strips = tile == kStrips;
    return AMB_OK;
}

int amb_mass(amb_handle* h, double* sum, int64_t* nonfinite)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    double s;
    int64_t b;
    const int rc = reduce_now(h, &s, &b);
    if (rc != AMB_OK) return rc;
    if (sum) *sum = s;
    if (nonfinite) *nonfinite = b;
    return AMB_OK;
}

int amb_last_mass(amb_handle* h, double* sum, int64_t* nonfinite)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    if (sum) *sum = h->last_sum;
    if (nonfinite) *nonfinite = h->last_bad;
    return AMB_OK;
}

int amb_set_noise(amb_handle* h, const double* noise, int64_t nsteps)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    if (nsteps < 0 || (nsteps > 0 && !noise)) return fail(AMB_E_ARG, "noise buffer must cover nsteps >= 0 steps");
    hipError_t e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return fail_hip(e, "hipStreamSynchronize");
    if (h->d_noise) (void)hipFree(h->d_noise);
    h->d_noise = nullptr;
    h->noise_steps = h->noise_used = 0;
    if (nsteps == 0) return AMB_OK;
    const size_t bytes = (size_t)nsteps * 2 * (size_t)(h->ny * h->nx) * sizeof(double);
    if ((e = hipMalloc(&h->d_noise, bytes)) != hipSuccess) return fail_hip(e, "hipMalloc (noise)");
    if ((e = hipMemcpy(h->d_noise, noise, bytes, hipMemcpyHostToDevice)) != hipSuccess)
        return fail_hip(e, "hipMemcpy (noise)");
    h->noise_steps = nsteps;
    return AMB_OK;
}

int amb_autotune(amb_handle* h, int reps, int* chosen)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    const int mode0 = h->model.T > 0.0 ? kNoisePhilox : kNoiseNone;
    if (reps < 0) {  // the tuning table's choice, when it has one
        if (take_tuned(h, mode0)) {
            if (chosen) *chosen = h->tile;
            return AMB_OK;
        }
        reps = -reps;
    }
    if (reps < 1) reps = 8;
    const size_t bytes = (size_t)(h->ny * h->nx) * h->esize;
    amb_handle trial = {};
    // A shallow trial handle on scratch buffers and a scratch step counter.
    hipError_t e = hipStreamSynchronize(h->stream);
    void* scratch[2] = {nullptr, nullptr};
    long long* step = nullptr;
    if (e == hipSuccess) e = hipMalloc(&scratch[0], bytes);
    if (e == hipSuccess) e = hipMalloc(&scratch[1], bytes);
    if (e == hipSuccess) e = hipMalloc(&step, sizeof(long long));
    if (e == hipSuccess) e = hipMemcpyAsync(scratch[0], h->buf[h->cur], bytes, hipMemcpyDeviceToDevice, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(step, h->d_step, sizeof(long long), hipMemcpyDeviceToDevice, h->stream);
    float best = 1e30f;
    int best_t = h->tile;
    const int mode = h->model.T > 0.0 ? kNoisePhilox : kNoiseNone;
    // every tile shape, then strips where the field runs in them without a choice
    bool strips = false;
    const int shapes = tile_count(h->precision);
    const int trials = shapes + (run_tile(h->precision, mode, h->ny, h->nx) == kStrips ? 1 : 0);
    for (int t = 0; t < trials && e == hipSuccess; ++t) {
        trial.ny = h->ny;
        trial.nx = h->nx;
        trial.stencil = h->stencil;
        trial.model = h->model;
        trial.options = h->options;
        trial.precision = h->precision;
        trial.buf[0] = scratch[0];
        trial.buf[1] = scratch[1];
        trial.d_step = step;
        trial.stream = h->stream;
        trial.tile = t < shapes ? t : kStrips;
        trial.tile_chosen = true;
        for (int k = 0; k <= reps && e == hipSuccess; ++k) {
            if (k == 1) e = hipEventRecord(h->ev0, h->stream);
            if (e == hipSuccess) e = launch_step(&trial, k, 0, mode);
        }
        if (e == hipSuccess) e = hipEventRecord(h->ev1, h->stream);
        if (e == hipSuccess) e = hipEventSynchronize(h->ev1);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, h->ev0, h->ev1);
        if (e == hipSuccess && ms < best) {
            best = ms;
            if (t < shapes) best_t = t;
            else strips = true;
        }
    }
    (void)hipStreamSynchronize(h->stream);
    for (void* p : {scratch[0], scratch[1], (void*)step})
        if (p) (void)hipFree(p);
    trial.stream = nullptr;
    if (e != hipSuccess) return fail_hip(e, "autotune");
    choose_tile(h, best_t, strips);
    record_tile(h->precision, h->ny, h->nx, mode0, best_t, strips ? AMB_TUNED_STRIPS : AMB_TUNED_ALL);
    if (chosen) *chosen = best_t;
    return AMB_OK;
}

int amb_tuning_set(int precision, int64_t ny, int64_t nx, int noisy, int tile)
{
    clear_error();
    if (precision != AMB_F32 && precision != AMB_F64) return fail(AMB_E_ARG, "bad precision");
    if (ny <= 0 || nx <= 0) return fail(AMB_E_ARG, "bad grid");
    if (tile < 0 || tile >= tile_count(precision)) return fail(AMB_E_ARG, "tile index out of range");
    record_tile(precision, ny, nx, noisy ? kNoisePhilox : kNoiseNone, tile, AMB_TUNED_ALL);
    return AMB_OK;
}

int amb_tuning_get(int precision, int64_t ny, int64_t nx, int noisy, int* tile)
{
    clear_error();
    if (!tile) return fail(AMB_E_ARG, "tile must not be null");
    if (!tuned_tile(precision, ny, nx, noisy ? kNoisePhilox : kNoiseNone, tile)) *tile = -1;
    return AMB_OK;
}

int amb_tuning_timed(int precision, int64_t ny, int64_t nx, int noisy, int set, int* timed)
{
    clear_error();
    if (set > AMB_TUNED_STRIPS) return fail(AMB_E_ARG, "unknown kind of tuning entry");
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    const auto it = g_tune.find({precision, ny, nx, noisy != 0});
    if (it == g_tune.end()) return fail(AMB_E_ARG, "no tuning entry");
    if (set >= 0) it->second.timed = set;
    if (timed) *timed = it->second.timed;
    return AMB_OK;
}

int amb_tuning_count(int64_t* count)
{
    if (!count) return fail(AMB_E_ARG, "count must not be null");
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    *count = (int64_t)g_tune.size();
    return AMB_OK;
}

int amb_tuning_entry(int64_t index, int* precision, int64_t* ny, int64_t* nx, int* noisy, int* tile)
{
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    if (index < 0 || index >= (int64_t)g_tune.size()) return fail(AMB_E_ARG, "tuning entry out of range");
    auto it = g_tune.begin();
    std::advance(it, index);
    if (precision) *precision = std::get<0>(it->first);
    if (ny) *ny = std::get<1>(it->first);
    if (nx) *nx = std::get<2>(it->first);
    if (noisy) *noisy = std::get<3>(it->first);
    if (tile) *tile = it->second.tile;
    return AMB_OK;
}

int amb_tuning_clear(void)
{
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    g_tune.clear();
    return AMB_OK;
}

int amb_set_tile(amb_handle* h, int index)
{
    clear_error();
    if (!h) return fail(AMB_E_ARG, "handle must not be null");
    if (index < 0 || index >= tile_count(h->precision)) return fail(AMB_E_ARG, "tile index out of range");
    choose_tile(h, index);
    return AMB_OK;
}

}  // extern "C"
