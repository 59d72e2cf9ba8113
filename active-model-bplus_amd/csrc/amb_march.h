// amb_march.h -- device code of one fused step over a strip of rows (large fields).
//
// A square tile recomputes its halo on every side: at 32x32 outputs the terms of stage A,
// the noise and the currents cost about twice what their sites need.  Here a workgroup
// advances a strip of 112 columns down a segment of rows and keeps the rows in flight in LDS
// rings, so nothing is recomputed along y except 16 rows at the top of the segment.
//
// Its waves have fixed roles, each marching down the strip four rows a step, a barrier per
// step; the later roles trail the earlier ones by what they read:
//   A (2 waves, a column a lane)   phi -> mu_p, mu_a = lambda |G3 phi|^2, q = zeta L3phi G3phi;
//                                  with the active current also C = q - G3 mu_a, a step later
//   X (2 waves, noisy)             J_x = amp xi_x - D8 mu_p, four columns a lane
//   Y (2 waves, noisy)             J_y
//   B (2 waves, a column a lane)   div J -> phi^{n+1}
// The rows a role needs again (three rows of phi, nine of J_y, five of mu_a ...) stay in its
// registers: step indices are unrolled over 16 rows, the length of the longest ring, so
// every LDS access has a constant offset from a per-lane base and no row is moved.
// 112 columns: the 16 halo columns of mu_p make 128, two waves; 240 (four waves a role) would
// save 7% of the lanes but lock 16 waves to each barrier.  Four rows a step: rings of 16 rows
// then let four workgroups share a CU's LDS.  The longer roles run at higher priority: the
// noisy FP32 step at 4096^2 took 83 us with every role at the same.
// Row counts below are from the segment's first mu_p row, rho = row - (y0 - 8).  At step n
//   A forms rho = 4n .. 4n+3             C       4n-5 .. 4n-2
//   Y       rho = 4n-8 .. 4n-5           X       4n-12 .. 4n-9
//   B       rho = 4n-16 .. 4n-13 (noisy) or 4n-12 .. 4n-9 (noiseless).
// Every site's arithmetic is that of step_tile, in the same order: the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "amb_kernels.h"
#include "amb_tile.h"

namespace amb {

constexpr int kMarchRows = 4;  // of a step

// LDS rings of a strip (elements).  Columns: mu_p from -8, mu_a, q and C from -2, J_x from -4,
// J_y from 0.  A ring of 16 or 8 rows holds row rho at slot rho mod 16 or
// mod 8 (C: rho + 1).
template <typename T, bool NOISY, bool ACTIVE>
struct MarchLds {
    static constexpr int TW = kMarchCols;
    static constexpr int MP = TW + 16, AP = TW + 4, XP = TW + 8, YP = TW;
    // three rows past the ring repeat its first three: a lane of role Y reads nine rows from
    // its own first row (0 .. 3 past the step's) without wrapping
    static constexpr int MR = NOISY ? 19 : 16, AR = NOISY && !ACTIVE ? 16 : 8, QR = NOISY ? 16 : 8;
    static constexpr int off_mu = 0;
    static constexpr int off_ma = off_mu + MR * MP;
    static constexpr int off_qx = off_ma + AR * AP;
    static constexpr int off_qy = off_qx + QR * AP;
    static constexpr int off_jx = off_qy + QR * AP;
    static constexpr int off_jy = off_jx + (NOISY ? 8 * XP : 0);
    static constexpr int total = off_jy + (NOISY ? 8 * YP : 0);
    static constexpr size_t red_off = (sizeof(T) * (size_t)total + 15) / 16 * 16;
    static constexpr size_t bytes = red_off + 16 * 128;  // a (sum, count) pair per lane of role B
    static constexpr int NT = march_threads(NOISY);
    static constexpr int wg = (int)((160 * 1024) / bytes);
    static constexpr int waves_want = wg * (NT / 64) / 4;
    // registers bind the noiseless step (its 17-row window) before LDS does
    static constexpr int most = NOISY ? 8 : sizeof(T) == 4 ? 5 : 2;
    static constexpr int min_waves = waves_want < 1 ? 1 : waves_want > most ? most : waves_want;
    // workgroups a CU: by LDS and registers, and at most four (the noiseless FP32 kernel, of
    // which five fit, takes 70.2 us at 4096^2 with five and 67.5 us with four, whose segments
    // are longer)
    static constexpr int by_regs = min_waves * 4 / (NT / 64);
    static constexpr int per_cu = wg < by_regs ? (wg < 4 ? wg : 4) : (by_regs < 4 ? by_regs : 4);
};

// A field as a buffer resource: an access takes a lane's byte offset within a row and the
// row's byte offset as a scalar, with no address arithmetic on the vector unit, and a lane
// whose offset is kNoLane reads zero and writes nothing.  Fields of at most 2^31 bytes.
constexpr uint32_t kNoLane = 0xffffff00u;
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t field_buffer(const T* field, int ny, int nx)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(field), 0, (int)((uint32_t)sizeof(T) * (uint32_t)ny * (uint32_t)nx),
                                             0x00020000);
}
__device__ __forceinline__ void buf_load(__amdgpu_buffer_rsrc_t b, uint32_t lane, uint32_t row, float& v)
{
    v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, lane, row, 0));
}
__device__ __forceinline__ void buf_load(__amdgpu_buffer_rsrc_t b, uint32_t lane, uint32_t row, double& v)
{
    v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, lane, row, 0));
}
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t b, uint32_t lane, uint32_t row, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), b, lane, row, 0);
}
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t b, uint32_t lane, uint32_t row, double v)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2v, v), b, lane, row, 0);
}

// rows: the segment's output rows (the last segment's may end short of a multiple of 4).
template <typename T, int NOISE, bool ACTIVE>
__device__ __forceinline__ void march_strip(T* const sm, const T* __restrict__ in, T* __restrict__ out, const int ny,
                                            const int nx, const int x0, const int y0, const int rows,
                                            const StepCoef<T>& K, const uint32_t key0, const uint32_t key1,
                                            const uint64_t step, double* const red_out)
{
    constexpr bool NOISY = NOISE == kNoisePhilox;
    static_assert(NOISY || !ACTIVE, "the active current is formed in noisy steps only");
    using L = MarchLds<T, NOISY, ACTIVE>;
    constexpr int TW = L::TW, MP = L::MP, AP = L::AP, XP = L::XP, YP = L::YP;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    enum { kA, kX, kY, kB };
    const int role = wave < 2 ? kA : NOISY ? wave >> 1 : kB;
    const int w = wave & 1;
    const uint32_t pitch = (uint32_t)sizeof(T) * (uint32_t)nx;  // bytes a row
    const int s4 = (rows + 3) >> 2;
    constexpr int N0 = NOISY ? 6 : 5;  // first step with an output
    // without the active current mu_a and q follow mu_p by LAG rows, to stay in their rings
    // no longer than stage B needs them
    constexpr int LAG = ACTIVE ? 0 : NOISY ? 8 : 4;
    const int n_end = s4 + N0;   // steps
    double* const red = reinterpret_cast<double*>(reinterpret_cast<unsigned char*>(sm) + L::red_off);
    const bool reduce = __builtin_amdgcn_readfirstlane(red_out != nullptr) != 0;
    // Every role runs n_end steps, each ended by one barrier: first `from` idle ones, then its
    // own body(u, n) at steps [from, to), u = n mod 4 a constant, then idle ones again.
    auto march = [&](auto from_c, int to, auto body, auto started) {
        constexpr int from = decltype(from_c)::value;
        if constexpr (!decltype(started)::value)
            for (int n = 0; n < from; ++n) __syncthreads();
        for (int n = from; n < to; n += 4) {
            body(std::integral_constant<int, from & 3>{});
            __syncthreads();
            if (n + 1 >= to) break;
            body(std::integral_constant<int, (from + 1) & 3>{});
            __syncthreads();
            if (n + 2 >= to) break;
            body(std::integral_constant<int, (from + 2) & 3>{});
            __syncthreads();
            if (n + 3 >= to) break;
            body(std::integral_constant<int, (from + 3) & 3>{});
            __syncthreads();
        }
        for (int n = to; n < n_end; ++n) __syncthreads();
    };

    if (role == kA) {
        __builtin_amdgcn_s_setprio(1);
        const int j = 64 * w + lane;  // column j - 8
        const uint32_t cm = (uint32_t)sizeof(T) * (uint32_t)wrap_index(x0 + j - 9, nx),
                       cc = (uint32_t)sizeof(T) * (uint32_t)wrap_index(x0 + j - 8, nx),
                       cp = (uint32_t)sizeof(T) * (uint32_t)wrap_index(x0 + j - 7, nx);
        const bool box = j >= 6 && j < TW + 10;
        const bool core = j >= 7 && j < TW + 9;  // columns [-1, TW+1): C
        const auto Mw = lds_base(sm + L::off_mu + j);
        const auto Aw = lds_base(sm + L::off_ma + (box ? j - 6 : 0));
        const auto Qxw = lds_base(sm + L::off_qx + (box ? j - 6 : 0));
        const auto Qyw = lds_base(sm + L::off_qy + (box ? j - 6 : 0));
        const T kb = in_vgpr(K.b);
        T f0[4], h1[4], h2[4];  // phi, its x-difference and x-sum at rows rho mod 4
        T pf[2][3];           // the next rows, in flight
        T e0[4], e1[4], e2[4], pe[2][3];  // the same LAG rows above, for mu_a and q
        T d[4], sum[4];         // mu_a's x-difference and y-smoothed sum at rows rho mod 4
        const auto field = field_buffer(in, ny, nx);
        uint32_t row = (uint32_t)wrap_index(y0 - 9, ny) * pitch;  // the next phi row to load
        uint32_t erow = (uint32_t)wrap_index(y0 - 9 - LAG, ny) * pitch;
        auto load_row = [&](T* v, uint32_t& row) {
            buf_load(field, cm, row, v[0]);
            buf_load(field, cc, row, v[1]);
            buf_load(field, cp, row, v[2]);
            row = row + pitch == pitch * (uint32_t)ny ? 0 : row + pitch;
        };
        {
            T a[3], b[3];
            load_row(a, row);
            load_row(b, row);
#pragma unroll
            for (int k = 0; k < 2; ++k) load_row(pf[k], row);
            f0[3] = a[1]; h1[3] = a[2] - a[0]; h2[3] = a[2] + a[0];
            f0[0] = b[1]; h1[0] = b[2] - b[0]; h2[0] = b[2] + b[0];
            if constexpr (LAG > 0) {
                load_row(a, erow);
                load_row(b, erow);
#pragma unroll
                for (int k = 0; k < 2; ++k) load_row(pe[k], erow);
                e0[3] = a[1]; e1[3] = a[2] - a[0]; e2[3] = a[2] + a[0];
                e0[0] = b[1]; e1[0] = b[2] - b[0]; e2[0] = b[2] + b[0];
            }
        }
        march(std::integral_constant<int, 0>{}, s4 + (LAG == 8 ? 5 : 4), [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if constexpr (ACTIVE) {
                // C at rows 4n-5 .. 4n-2, from mu_a rows up to 4n-1
                if (core) {
                    const auto Ar = Aw + 4 * ((u + 1) & 1) * AP;
                    // every read ahead of the writes (the compiler would wait out each in turn)
                    T ml[4], mc[4], mr[4], qx[4], qy[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int s = (4 * u + 12 + k) & 15;
                        ml[k] = Ar[k * AP - 1];
                        mc[k] = Ar[k * AP];
                        mr[k] = Ar[k * AP + 1];
                        qx[k] = Qxw[s * AP];
                        qy[k] = Qyw[s * AP];
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int s = (4 * u + 12 + k) & 15;
                        d[k] = mr[k] - ml[k];
                        sum[k] = fma(K.gye, ml[k] + mr[k], K.gyc * mc[k]);
                        Qxw[s * AP] = fma(-K.gxc, d[(k + 3) & 3], fma(-K.gxe, d[(k + 2) & 3] + d[k], qx[k]));
                        Qyw[s * AP] = qy[k] - (sum[k] - sum[(k + 2) & 3]);
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                constexpr int R4 = 4 * u;
                const int a = (k + 3) & 3, m = k, b = (k + 1) & 3;
                T* const v = pf[k & 1];
                f0[b] = v[1];
                if constexpr (LAG == 0) h1[b] = v[2] - v[0];
                h2[b] = v[2] + v[0];
                load_row(v, row);
                const T lap = laplacian3(K, f0[m], h2[m], f0[a] + f0[b], h2[a] + h2[b]);
                const T mu = mu_passive(K, kb, f0[m], lap);
                Mw[(R4 + k) * MP] = mu;
                if (NOISY && R4 + k < 3) Mw[(16 + R4 + k) * MP] = mu;
                // mu_a and q, of this row or of the row LAG above
                T gx, gy, zl;
                if constexpr (LAG == 0) {
                    gx = K.gxe * (h1[a] + h1[b]) + K.gxc * h1[m];
                    gy = K.gye * (h2[b] - h2[a]) + K.gyc * (f0[b] - f0[a]);
                    zl = K.zeta * lap;
                } else {
                    T* const p = pe[k & 1];
                    e0[b] = p[1];
                    e1[b] = p[2] - p[0];
                    e2[b] = p[2] + p[0];
                    load_row(p, erow);
                    gx = K.gxe * (e1[a] + e1[b]) + K.gxc * e1[m];
                    gy = K.gye * (e2[b] - e2[a]) + K.gyc * (e0[b] - e0[a]);
                    zl = K.zeta * laplacian3(K, e0[m], e2[m], e0[a] + e0[b], e2[a] + e2[b]);
                }
                const T ma = K.lam * (gy * gy + gx * gx);
                if (box) {
                    const int s = R4 + k + 16 - LAG;
                    Aw[(s & (L::AR - 1)) * AP] = ma;
                    Qxw[((s + (ACTIVE ? 1 : 0)) & (L::QR - 1)) * AP] = zl * gx;
                    Qyw[((s + (ACTIVE ? 1 : 0)) & (L::QR - 1)) * AP] = zl * gy;
                }
            }
        }, std::false_type{});
    } else if (NOISY && role == kX) {
        __builtin_amdgcn_s_setprio(1);
        // lane = (row k of the step, group of four columns)
        const int k = lane >> 4, g = 15 * w + (lane & 15);  // columns 4 g - 4 .. 4 g - 1
        const bool live = (lane & 15) < 15;
        const T* const M = sm + L::off_mu + k * MP + 4 * g;  // mu_p at column 4 g - 8
        T* const J = sm + L::off_jx + k * XP + 4 * g;
        const int gc = wrap_index(x0 + 4 * g - 4, nx);  // the group's first column
        // whether its four columns are one Philox group, as everywhere but at the periodic
        // seam of a field whose columns do not split into fours
        const bool whole = __all(((gc & 3) == 0 && gc + 3 < nx) || !live);
        // Across the seam the groups straddle two Philox groups.  A lane then draws the Philox
        // group of its first column and takes its other columns from the next lane's draw; the
        // spare lane of each row draws for the last one, or in the first strip for the group
        // left of column 0.  (Fields narrower than a strip: a call per site.)
        const bool left = x0 == 0 && w == 0, neighbours = nx >= TW + 16;
        const int drawn = left && !live ? nx - 1 : gc;
        const int from = left && (lane & 15) == 0 ? lane + 15 : lane + 1;
        const int own = min(4 - (gc & 3), nx - gc);  // columns in the lane's own Philox group
        const uint32_t group = (uint32_t)drawn >> 2;
        int row = wrap_index(y0 + k, ny);  // rho = 8 + k, at step 5
        march(std::integral_constant<int, 5>{}, s4 + 5, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            T z[4];
            if (whole || neighbours) normals4<T>(group, (uint32_t)row, step, 1, key0, key1, z);
            if (!whole) {
                T n[4];
                if (neighbours) {
                    T o[4];
#pragma unroll
                    for (int l = 0; l < 4; ++l) {
                        o[l] = __shfl(z[l], from, 64);
                        n[l] = z[l];
                    }
                    const int at = gc & 3;
#pragma unroll
                    for (int l = 0; l < 4; ++l) {  // own: column l is z[at + l]; else o[l - own]
                        T v = o[0];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if (l < own && i == at + l) v = n[i];
                            if (l >= own && i == l - own) v = o[i];
                        }
                        z[l] = v;
                    }
                } else {
#pragma unroll 1
                    for (int l = 0; l < 4; ++l) {
                        const T v = normal1<T>(row, (gc + l) % nx, step, 1, key0, key1);
                        if (l == 0) z[0] = v;
                        if (l == 1) z[1] = v;
                        if (l == 2) z[2] = v;
                        if (l == 3) z[3] = v;
                    }
                }
            }
            if (live) {
                const T* const Ms = M + ((4 * u + 4) & 15) * MP;
                T m[12], jv[4];
                lds_load4(Ms, m);
                lds_load4(Ms + 4, m + 4);
                lds_load4(Ms + 8, m + 8);
#pragma unroll
                for (int l = 0; l < 4; ++l) {
                    T acc = K.amp * z[l];
#pragma unroll
                    for (int i = 1; i <= 4; ++i) acc = fma(-K.dxw[i], m[4 + l + i] - m[4 + l - i], acc);
                    jv[l] = acc;
                }
                lds_store4(J + 4 * ((u + 1) & 1) * XP, jv);
            }
            row += 4;
            row = (int)min((uint32_t)row, (uint32_t)(row - ny));
        }, std::false_type{});
    } else if (NOISY && role == kY) {
        __builtin_amdgcn_s_setprio(0);
        const int k = lane >> 4, g = 14 * w + (lane & 15);  // columns 4 g .. 4 g + 3
        const bool live = (lane & 15) < 14;
        const T* const M = sm + L::off_mu + k * MP + 4 * g + 8;
        T* const J = sm + L::off_jy + k * YP + 4 * g;
        const uint32_t group = (uint32_t)(x0 >> 2) + (uint32_t)g;  // columns past nx are not used
        int row = wrap_index(y0 - 4 + k, ny);                      // rho = 4 + k, at step 3
        march(std::integral_constant<int, 3>{}, s4 + 5, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if (live) {
                T z[4], acc[4];
                normals4<T>(group, (uint32_t)row, step, 0, key0, key1, z);
#pragma unroll
                for (int l = 0; l < 4; ++l) acc[l] = K.amp * z[l];
#pragma unroll
                for (int i = 1; i <= 4; ++i) {
                    // row rho + e sits at slot 4u + 8 + e of the step's first row, plus k
                    T up[4], dn[4];
                    lds_load4(M + ((4 * u + 8 + i) & 15) * MP, up);
                    lds_load4(M + ((4 * u + 8 - i) & 15) * MP, dn);
#pragma unroll
                    for (int l = 0; l < 4; ++l) acc[l] = fma(-K.dyw[i], up[l] - dn[l], acc[l]);
                }
                lds_store4(J + 4 * (u & 1) * YP, acc);
            }
            row += 4;
            row = (int)min((uint32_t)row, (uint32_t)(row - ny));
        }, std::false_type{});
    } else {
        __builtin_amdgcn_s_setprio(3);
        const int c = 64 * w + lane;
        const bool live = c < TW;
        const int cs = live ? c : 0;
        const bool col_ok = live && x0 + c < nx;
        const uint32_t off = col_ok ? (uint32_t)sizeof(T) * (uint32_t)(x0 + c) : kNoLane;
        const auto src = field_buffer(in, ny, nx);
        const auto Ab = lds_base(sm + L::off_ma + cs + 2);
        const auto Qxb = lds_base(sm + L::off_qx + cs + 2);
        const auto Qyb = lds_base(sm + L::off_qy + cs + 2);
        const auto Xb = lds_base(sm + L::off_jx + cs + 4);
        const auto Mc = lds_base(sm + L::off_mu + cs + 8);
        const auto Yb = lds_base(sm + L::off_jy + cs);
        // windows, by row: J_y or mu_p (mod 16), mu_a, q or C (mod 8); phi at the step's outputs
        T col[16], d2x[8], sx[8], hx[8], sy[8], pc[4];
        double* const mine = red + 2 * (64 * w + lane);
        if (reduce) mine[0] = mine[1] = 0.0;
        // rows ahead at which mu_a and q (or C) are read: two and one at least, more where their
        // rings would be overwritten by then
        constexpr int AL = NOISY ? 2 : 4, QL = NOISY && !ACTIVE ? 1 : 4;
        // byte offset of the step's first output row from the segment's first
        uint32_t orow = 0;
        const uint32_t first = (uint32_t)y0 * pitch, len = (uint32_t)rows * pitch;
        auto load_centers = [&]() {  // (past the segment's last row: its first row's)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t at = orow + (uint32_t)k * pitch;
                buf_load(src, off, first + (at < len ? at : 0u), pc[k]);
            }
        };
        // Output rows are rho = 4n-16 .. 4n-13 (noiseless 4n-12 .. 4n-9), at slot S + k.  A row
        // completes its windows with row rho + 4 of J_y (rho + 8 of mu_p, here `last`), rho + AL
        // of mu_a and rho + QL of q or C.
        auto slot = [](int u) { return 4 * u + (NOISY ? 0 : 4); };
        auto windows = [&](auto uc, int k, T& last) {
            const int S = slot(decltype(uc)::value);
            if constexpr (NOISY) col[(S + k + 4) & 15] = Yb[((S + k + 4) & 7) * YP];
            else last = Mc[((S + k + 8) & 15) * MP];
            if constexpr (!ACTIVE) {
                const auto A = Ab + ((S + k + AL) & (L::AR - 1)) * AP;
                const T o2 = A[-2] + A[2];
                d2x[(S + k + AL) & 7] = o2 - A[0] - A[0];
                sx[(S + k + AL) & 7] = T(kG3G3S[0]) * A[0] + T(kG3G3S[1]) * (A[-1] + A[1]) + T(kG3G3S[2]) * o2;
            }
            const int qslot = (S + k + QL + (ACTIVE ? 1 : 0)) & (L::QR - 1);
            const auto Qx = Qxb + qslot * AP;
            const auto Qy = Qyb + qslot * AP;
            hx[(S + k + QL) & 7] = Qx[1] - Qx[-1];
            sy[(S + k + QL) & 7] = K.gyc * Qy[0] + K.gye * (Qy[-1] + Qy[1]);
        };
        // the steps before the first output fill the windows: two steps of J_y, mu_a, q; four of mu_p
        T last;
        for (int n = 0; n < (NOISY ? 4 : 1); ++n) __syncthreads();
        if constexpr (!NOISY) {
#pragma unroll
            for (int n = 1; n < 5; ++n) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (n >= 3) windows(std::integral_constant<int, 0>{}, 4 * n + k, last);
                    col[(4 * n - 4 + k) & 15] = Mc[((4 * n - 4 + k) & 15) * MP];
                }
                if (n == 4) load_centers();
                __syncthreads();
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) windows(std::integral_constant<int, 0>{}, k, last);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 4; ++k) windows(std::integral_constant<int, 1>{}, k, last);
            load_centers();
            __syncthreads();
        }
        march(std::integral_constant<int, N0>{}, n_end, [&](auto uc) {
            constexpr int u = decltype(uc)::value;
            const int S = slot(u);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                T last;
                windows(uc, k, last);
                T acc;
                if constexpr (NOISY) {
                    const auto X = Xb + ((S + k) & 7) * XP;
                    auto yv = [&](int e) { return col[(S + k + 16 + e) & 15]; };
                    acc = K.dxw[1] * (X[1] - X[-1]);
                    acc = fma(K.dyw[1], yv(1) - yv(-1), acc);
#pragma unroll
                    for (int i = 2; i <= 4; ++i) {
                        acc = fma(K.dxw[i], X[i] - X[-i], acc);
                        acc = fma(K.dyw[i], yv(i) - yv(-i), acc);
                    }
                } else {
                    const auto m = Mc + ((S + k) & 15) * MP;
                    auto mv = [&](int e) { return e == 8 ? last : col[(S + k + 16 + e) & 15]; };
                    acc = K.p0 * mv(0);
#pragma unroll
                    for (int i = 1; i <= 8; ++i) {
                        acc = fma(K.px[i], m[i] + m[-i], acc);
                        acc = fma(K.py[i], mv(i) + mv(-i), acc);
                    }
                    col[(S + k + 8) & 15] = last;
                }
                auto at = [&](int e) { return (S + k + 8 + e) & 7; };
                if constexpr (!ACTIVE) {
                    acc = fma(K.lxx[0], d2x[at(0)], acc);
                    acc = fma(K.lxx[1], d2x[at(-1)] + d2x[at(1)], acc);
                    acc = fma(K.lxx[2], d2x[at(-2)] + d2x[at(2)], acc);
                    acc = fma(K.lyy[0], (sx[at(-2)] + sx[at(2)]) - sx[at(0)] - sx[at(0)], acc);
                }
                acc = fma(K.gxc, hx[at(0)], acc);
                acc = fma(K.gxe, hx[at(-1)] + hx[at(1)], acc);
                acc += sy[at(1)] - sy[at(-1)];
                pc[k] = fma(-K.dt, acc, pc[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                // an empty buffer for rows past the segment: no branch, and nothing stored
                const uint32_t at = orow + (uint32_t)k * pitch;
                const bool in_seg = at < len;
                buf_store(field_buffer(out, in_seg ? ny : 0, nx), off, in_seg ? first + at : 0u, pc[k]);
            }
            if (reduce) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const double dv = (double)pc[k];
                    if (orow + (uint32_t)k * pitch >= len) continue;
                    if (isfinite(dv)) mine[0] += dv;
                    else mine[1] += 1.0;
                }
            }
            orow += 4 * pitch;
            load_centers();
        }, std::true_type{});
        if (reduce) {
            double rs = col_ok ? mine[0] : 0.0, rbad = col_ok ? mine[1] : 0.0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                rs += __shfl_xor(rs, o, 64);
                rbad += __shfl_xor(rbad, o, 64);
            }
            if (lane == 0) {
                mine[0] = rs;
                mine[1] = rbad;
            }
        }
    }
    if (reduce) {
        __syncthreads();
        if (threadIdx.x == 0) {
            red_out[0] = red[0] + red[128];
            red_out[1] = red[1] + red[129];
        }
    }
}

}  // namespace amb
