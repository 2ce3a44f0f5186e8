// tridiag_real.hip — Householder reduction of a real symmetric H(k) to
// tridiagonal form (gfx950): the matrices of crystals with an inversion centre
// and no spin-orbit, in FP32 for the precision form and FP64 for the FP64 form.
// A chain of shrinking kernels as for complex matrices (tridiag_reg.hip): real
// lower-triangle grids (tridiag_grid.hpp) down to a trailing block of 128, then
// one-row-per-lane kernels (tridiag_row.hpp); FP32 blocks of 65 .. 96 start in a grid.
//
// A real element takes a quarter of a complex one's multiply-adds and half its
// registers, so each grid reaches twice the dimension or twice the workgroups
// per CU.  Si, n = 181, 2048 k-points alone on the chip: FP32 1.08 ms, FP64 1.87; the
// complex kernels took 2.4 and 5.8 on the same matrices.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "solver.hpp"
#include "tridiag_grid.hpp"
#include "tridiag_row.hpp"

namespace uepm {

namespace {

// Sizes the stages take, largest first, and where each hands over (next()).  A
// grid hands over after 32 steps to the next one, except from 192 to 128 (the
// 160-wide stage in between gains as much as its hand-over costs: FP32 2.14 ms
// both ways at n = 181, FP64 3.39 against 3.42); 96 and 128 end in the one-wave
// 64-row kernel (FP32 n = 128: 0.69 ms against 0.78 for all steps in one kernel).
constexpr int kSize[] = {448, 384, 320, 288, 256, 224, 192, 160, 128, 96, 64};
constexpr int kNum = sizeof(kSize) / sizeof(kSize[0]);
constexpr int kMax32 = 448, kMax64 = 320;

int stage_of(int n) {
    int g = 0;
    while (g < kNum - 1 && n <= kSize[g + 1]) ++g;
    return g;
}
// trailing size handed over by the stage that takes n; 0: it runs to the end
int next(int n) {
    const int size = kSize[stage_of(n)];
    return size > 192 ? kSize[stage_of(n) + 1] : size > 128 ? 128 : size > 64 ? 64 : 0;
}

// One stage.  Shapes and register budgets (waves per SIMD) are the fastest of a
// sweep that did not spill in the steps; 16 x 16 lanes where a grid fits their
// registers (four waves meet at a barrier instead of eight), 32 x 16 above.
// Measured, ms per 32 steps and 2048 matrices: FP32 448: 3.04, 384: 2.24, 320:
// 1.73, 288: 1.09, 256: 0.77, 224: 0.62 (16 x 16 lanes: the same), 160: 0.31; FP64 320: 2.53, 288: 1.87, 256: 1.54,
// 224: 1.35, 160: 0.52 (0.58 without blocks in LDS).  Per 4096: FP32 192 (53 steps):
// 1.17 (1.43 at three waves per SIMD without), 128 (64 steps): 0.55 (32 steps of a grid
// alone: 0.47), 96 (32 steps): 0.28 (rows: 0.34), 64: 0.15; FP64 2.19, 128: 1.01 (32 steps
// of a grid alone: 0.70), 96: 0.44 (grid: 0.49), 64: 0.19.
template <typename THin>
void stage(const THin* H, int64_t hk, int n, int ld, int64_t nk, float* V, int ldv, int64_t vk, double* dd, double* de,
           float* dtau, int64_t dk, int s_end, float* B, int ldb, hipStream_t s) {
    using S = r1<float>;
    constexpr bool kFromH = sizeof(THin) == sizeof(double);  // no stage hands over to these three
#define UEPM_GRID(...) reg_stage<S, __VA_ARGS__>(H, hk, n, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s)
#define UEPM_ROWS(...) row_stage<S, __VA_ARGS__, 1>(H, hk, n, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s)
    switch (kSize[stage_of(n)]) {
        case 448:
            if constexpr (kFromH) UEPM_GRID(32, 14, 2, 1, THin, true, 30, true);
            break;
        case 384: UEPM_GRID(32, 12, 2, 1, THin, true, 0, true); break;
        case 320: UEPM_GRID(32, 10, 2, 1, THin, false, 0, true); break;
        case 288: UEPM_GRID(32, 9, 4, 1, THin, true, 8, true); break;
        case 256: UEPM_GRID(32, 8, 4, 1, THin, true, 0, true); break;
        case 224: UEPM_GRID(32, 7, 4, 1, THin, false, 0, true); break;
        case 192: UEPM_GRID(16, 12, 4, 1, THin, true, 16, true); break;
        case 160:
            if constexpr (kFromH) UEPM_GRID(16, 10, 4, 1, THin, false, 0, true);
            break;
        case 128: UEPM_ROWS(2, 2, 4, 5); break;
        case 96:
            if constexpr (kFromH) UEPM_GRID(16, 6, 8, 1, THin, true, 0, true);
            break;
        default: UEPM_ROWS(1, 1, 4, 5); break;
    }
#undef UEPM_GRID
#undef UEPM_ROWS
}
void stage(const double* H, int64_t hk, int n, int ld, int64_t nk, double* V, int ldv, int64_t vk, double* dd, double* de,
           double* dtau, int64_t dk, int s_end, double* B, int ldb, hipStream_t s) {
    using S = r1<double>;
#define UEPM_GRID(...) reg_stage<S, __VA_ARGS__>(H, hk, n, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s)
#define UEPM_ROWS(...) row_stage<S, __VA_ARGS__, 1>(H, hk, n, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s)
    switch (kSize[stage_of(n)]) {
        case 320: UEPM_GRID(32, 10, 2, 1, double, true, 24, true); break;
        case 288: UEPM_GRID(32, 9, 2, 1, double, true, 0, true); break;
        case 256: UEPM_GRID(32, 8, 2, 1, double, true, 0, true); break;
        case 224: UEPM_GRID(32, 7, 2, 1, double, true, 0, true); break;
        case 192: UEPM_GRID(16, 12, 2, 1, double, true, 0, true); break;
        case 160: UEPM_GRID(16, 10, 3, 1, double, true, 16, true); break;
        case 128: UEPM_ROWS(2, 2, 4, 2); break;
        case 96: UEPM_ROWS(2, 1, 6, 2); break;
        default: UEPM_ROWS(1, 1, 4, 3); break;
    }
#undef UEPM_GRID
#undef UEPM_ROWS
}

template <typename R>
hipError_t chain(const double* H, int n, int64_t nk, R* V, double* dd, double* de, R* dtau, R* work, hipStream_t s) {
    const int64_t nn = (int64_t)n * n;
    const int t1 = next(n);
    if (t1 && !work) return hipErrorInvalidValue;
    R* buf[2] = {work, t1 ? work + nk * (int64_t)t1 * t1 : nullptr};
    stage(H, nn, n, n, nk, V, n, nn, dd, de, dtau, n, t1 ? n - t1 : n, buf[0], t1, s);
    int r = t1, cur = 0;
    while (r) {
        const int off = n - r, t = next(r);
        stage((const R*)buf[cur], (int64_t)r * r, r, r, nk, V + off + (int64_t)off * n, n, nn, dd + off, de + off,
              dtau + off, n, t ? r - t : r, t ? buf[cur ^ 1] : (R*)nullptr, t, s);
        r = t;
        cur ^= 1;
    }
    return hipGetLastError();
}

}  // namespace

int tridiag_real_max_n(bool f32) { return f32 ? kMax32 : kMax64; }

size_t tridiag_real_work_bytes(int n, bool f32) {
    const int t1 = next(n), t2 = t1 ? next(t1) : 0;
    return (f32 ? sizeof(float) : sizeof(double)) * ((size_t)t1 * t1 + (size_t)t2 * t2);
}

hipError_t launch_tridiag_real_f32(const double* dH, int n, int64_t nk, float* V, double* dd, double* de, float* dtau,
                                   float* work, hipStream_t s) {
    if (n < 1 || n > kMax32 || nk <= 0) return hipErrorInvalidValue;
    return chain<float>(dH, n, nk, V, dd, de, dtau, work, s);
}

hipError_t launch_tridiag_real_f64(const double* dH, int n, int64_t nk, double* V, double* dd, double* de, double* dtau,
                                   double* work, hipStream_t s) {
    if (n < 1 || n > kMax64 || nk <= 0) return hipErrorInvalidValue;
    return chain<double>(dH, n, nk, V, dd, de, dtau, work, s);
}

}  // namespace uepm
