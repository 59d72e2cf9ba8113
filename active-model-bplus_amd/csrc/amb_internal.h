// amb_internal.h -- helpers shared by the host runtime's translation units (internal).
#pragma once

#include <mutex>
#include <hip/hip_runtime.h>

#include <string>

#include "amb.h"
#include "amb_kernels.h"

namespace amb {

int fail(int code, const std::string& msg);
int fail_hip(hipError_t e, const char* what);
void clear_error();
int check_device();
int validate_params(int64_t ny, int64_t nx, const amb_stencil* st, const amb_model* m);
int grid_tiles(int64_t n, int t);
int default_tile(int precision, int64_t ny, int64_t nx, int noise);
// The autotuners' table (process-wide): lookup and record (timed: AMB_TUNED_*).
bool tuned_tile(int precision, int64_t ny, int64_t nx, int noise, int* tile, int* timed = nullptr);
void record_tile(int precision, int64_t ny, int64_t nx, int noise, int tile, int timed);

template <typename T>
StepCoef<T> make_coef(const amb_stencil& st, const amb_model& m);

constexpr int64_t kStageDoubles = (int64_t)1 << 17;  // of a piece
// Two pinned pieces through which results go to the caller's memory, made on first use.  Getters
// of one handle may be called from several threads: each holds `turn` until its result is out.
struct HostStage {
    std::mutex turn;
    void* piece[2] = {nullptr, nullptr};
    hipEvent_t filled[2] = {nullptr, nullptr};
};
// n values of a field (FP32 or FP64) at dev, as doubles to out, after the work on `s`.  The caller
// holds st.turn.
hipError_t copy_out(HostStage& st, const void* dev, int64_t n, int precision, double* out, hipStream_t s);
void release(HostStage& st);

// Access to an integrator's state for other parts of the library (the surrogate).
struct FieldView {
    void* cur;          // current field (ny*nx elements of the handle's precision)
    void* other;        // the second ping-pong buffer
    int64_t ny, nx;
    int precision;
    hipStream_t stream;
};
int handle_view(amb_handle* h, FieldView* v);
// Enqueues the FP64 sum of the current field on the handle's stream; *sum is where it will be
// (device memory of the handle, rewritten by the next reduction).
int handle_field_sum(amb_handle* h, const double** sum);
// Advances the step counter by `steps` (host and device); with `swapped` the field
// now lives in the buffer that was `other`.
int handle_commit(amb_handle* h, int64_t steps, bool swapped);
// Enqueues `steps` explicit-Euler steps on the handle's stream without waiting (no
// finite check) and advances the step counter.
int handle_enqueue(amb_handle* h, int64_t steps);
// Sets the step counter (host and device), after the handle's stream is idle.
int handle_set_timestep(amb_handle* h, int64_t timestep);
int64_t handle_timestep(const amb_handle* h);

// Per-handle state of the structure factor (FFT plan and buffers), created by
// amb_structure_factor on first use and freed with the handle.
struct SkCache;
SkCache** handle_sk_cache(amb_handle* h);
void sk_cache_free(SkCache* c);

}  // namespace amb
