// tridiag_quaternion.hip — Householder reduction of a quaternion Hermitian H(k)
// to real symmetric tridiagonal form (gfx950): the spinor matrices of crystals
// with an inversion centre (equal atoms, spin-orbit), an N x N quaternion matrix
// for a 2N x 2N complex one.  Half the multiply-adds, half the elements and half
// the steps; the N x N tridiagonal T holds each Kramers pair of levels once.
// The grids of tridiag_grid.hpp in quaternion arithmetic, shrinking as the
// complex chain does (tridiag_reg.hip).  Shapes are the fastest of a sweep; 32 steps of
// 2048 matrices, ms, 32 x 16 lanes against 16 x 16: FP32 160 1.98, 2.21; 137 -> 128 (9
// steps, the 160 against the 144 grid) 0.80, 0.59, FP64 2.30, 1.35 (512 registers, AGPRs
// among them, one wave per SIMD); FP32 128 1.50 (1.19 with
// 6 of 20 blocks in LDS), 1.15; 96 0.74, 0.63; 64 (63 steps) 0.68, 0.49; FP64 128 2.48 (2.74
// with no blocks in LDS), too large; 96 1.69, 1.33; 64 1.31, 1.05.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "solver.hpp"
#include "tridiag_grid.hpp"

namespace uepm {

namespace {

constexpr int kSize[] = {192, 160, 144, 128, 96, 64};
constexpr int kNum = sizeof(kSize) / sizeof(kSize[0]);
constexpr int kMax32 = 192, kMax64 = 160;

int stage_of(int n) {
    int g = 0;
    while (g < kNum - 1 && n <= kSize[g + 1]) ++g;
    return g;
}
// 144 takes first blocks only: 16 steps are not worth a hand-over
int next(int n) {
    const int g = stage_of(n);
    return n > 128 ? (n > 160 ? 160 : 128) : g < kNum - 1 ? kSize[g + 1] : 0;
}

template <int IN, typename R>
void stage(const q4<double>* H0, const q4<R>* Hb, int64_t hk, int n, int64_t nk, q4<R>* V, int ldv, int64_t vk, double* dd,
           double* de, q4<R>* dtau, int64_t dk, int s_end, q4<R>* B, int ldb, hipStream_t s) {
    using S = q4<R>;
    auto grid = [&](const auto* H) {
        using THin = std::remove_const_t<std::remove_pointer_t<decltype(H)>>;
#define UEPM_GRID(pr, lr, w, nl)                                                                                            \
    reg_stage<S, pr, lr, w, IN, THin, true, nl>(H, hk, n, n, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s)
        if constexpr (sizeof(R) == sizeof(float)) {
            switch (kSize[stage_of(n)]) {
                case 192: UEPM_GRID(32, 6, 2, 0); break;
                case 160: UEPM_GRID(32, 5, 2, 0); break;
                case 144:
                    if constexpr (IN == 1) UEPM_GRID(16, 9, 2, 12);
                    break;
                case 128: UEPM_GRID(16, 8, 2, 0); break;
                case 96: UEPM_GRID(16, 6, 3, 3); break;
                default: UEPM_GRID(16, 4, 4, 0); break;
            }
        } else {
            switch (kSize[stage_of(n)]) {
                case 160: UEPM_GRID(32, 5, 2, 5); break;
                case 144:
                    if constexpr (IN == 1) UEPM_GRID(16, 9, 1, 14);
                    break;
                case 128: UEPM_GRID(32, 4, 2, 4); break;
                case 96: UEPM_GRID(16, 6, 2, 6); break;
                default: UEPM_GRID(16, 4, 2, 0); break;
            }
        }
#undef UEPM_GRID
    };
    if constexpr (IN == 1) grid(H0);
    else grid(Hb);
}

template <typename R>
hipError_t chain(const q4<double>* H, int n, int64_t nk, q4<R>* V, double* dd, double* de, q4<R>* dtau, q4<R>* work,
                 hipStream_t s) {
    const int64_t nn = (int64_t)n * n;
    const int t1 = next(n);
    if (t1 && !work) return hipErrorInvalidValue;
    q4<R>* buf[2] = {work, t1 ? work + nk * (int64_t)t1 * t1 : nullptr};
    stage<1, R>(H, nullptr, nn, n, nk, V, n, nn, dd, de, dtau, n, t1 ? n - t1 : n, buf[0], t1, s);
    int r = t1, cur = 0;
    while (r) {
        const int off = n - r, t = next(r);
        stage<2, R>(nullptr, buf[cur], (int64_t)r * r, r, nk, V + off + (int64_t)off * n, n, nn, dd + off, de + off,
                    dtau + off, n, t ? r - t : r, t ? buf[cur ^ 1] : nullptr, t, s);
        r = t;
        cur ^= 1;
    }
    return hipGetLastError();
}

}  // namespace

int tridiag_quaternion_max_n(bool f32) { return f32 ? kMax32 : kMax64; }

size_t tridiag_quaternion_work_bytes(int n, bool f32) {
    const int t1 = next(n), t2 = t1 ? next(t1) : 0;
    return (f32 ? sizeof(q4<float>) : sizeof(q4<double>)) * ((size_t)t1 * t1 + (size_t)t2 * t2);
}

hipError_t launch_tridiag_quaternion_f32(const q4<double>* dH, int n, int64_t nk, q4<float>* V, double* dd, double* de,
                                         q4<float>* dtau, q4<float>* work, hipStream_t s) {
    if (n < 1 || n > kMax32 || nk <= 0) return hipErrorInvalidValue;
    return chain<float>(dH, n, nk, V, dd, de, dtau, work, s);
}

hipError_t launch_tridiag_quaternion_f64(const q4<double>* dH, int n, int64_t nk, q4<double>* V, double* dd, double* de,
                                         q4<double>* dtau, q4<double>* work, hipStream_t s) {
    if (n < 1 || n > kMax64 || nk <= 0) return hipErrorInvalidValue;
    return chain<double>(dH, n, nk, V, dd, de, dtau, work, s);
}

}  // namespace uepm
