// solver_f64.hip — tridiagonal eigen-stage of the band solve on gfx950.
//
//   (c) tri_eig_wave_kernel bisection (Sturm counts, multisection) for the lowest
//                           nb eigenvalues of T, one wave per k
//       tri_vec_kernel      inverse iteration for their vectors, one lane per band
//
// The assembly (a) lives in assemble.hip, the Householder reduction (b) in
// tridiag_*.hip and the back-transform (d) in backtransform.hip; (b)-(d) replace
// Eigen::SelfAdjointEigenSolver::compute (Hamiltonian.cpp:129): same
// eigenvalues to within the backward-stability envelope of a Householder
// reduction, eigenvectors up to phase (and basis inside degenerate clusters).
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <cstdlib>

#include "epm_physics.hpp"
#include "solver.hpp"

namespace uepm {

// ------------------------------------- (c) tridiagonal eigenvalues / vectors
// Start vector of inverse iteration: a fixed pseudo-random value per (row, band).
__device__ __forceinline__ double lane_rand(uint32_t i, uint32_t b) {
    uint32_t h = i * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u;
    h ^= h >> 15;
    h *= 0x2C1B3C6Du;
    h ^= h >> 12;
    h *= 0x297A2D39u;
    h ^= h >> 15;
    return (double)(h >> 8) * (1.0 / 8388608.0) - 1.0;
}

// 1/x: hardware reciprocal and Newton steps to full precision
__device__ __forceinline__ double rcp_nr64(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// number of eigenvalues of T below x: sign changes of the leading principal
// minors p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}, T scaled to norm 1..2 and e^2
// held above 2^-160, so that no two neighbours vanish.  Of two neighbours the larger
// falls by at most that (and a factor of eight) six times in eight steps, after which
// the pair is rescaled by a power of two, so it stays in range.  One multiply-add
// long per step, against a reciprocal and its Newton step for the quotients
// p_i / p_{i-1}; the two have the same backward error.  n and the LDS arrays are
// padded to whole pairs of blocks of eight (kSturmPad, rows that change no sign).
__device__ __forceinline__ int sturm_count(const double* __restrict__ sd, const double* __restrict__ se2, int np, double x) {
    struct Block {
        double d[8], e[8];
    };
    auto load = [&](Block& r, int i) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            r.d[u] = sd[i + u];
            r.e[u] = se2[i + u];
        }
    };
    double p = 1.0, pp = 0.0;
    unsigned signs = 0;  // sign bits of the last minors, the newest lowest
    int c = 0;
    auto step = [&](const Block& r) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double pn = fma(r.d[u] - x, p, -(r.e[u] * pp));
            signs = __builtin_amdgcn_alignbit(signs, (unsigned)__double2hiint(pn), 31);
            pp = p;
            p = pn;
        }
        c += __popc((signs ^ signs >> 1) & 0xffu);
        const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(p), fabs(pp)));
        p = __builtin_amdgcn_ldexp(p, -ex);
        pp = __builtin_amdgcn_ldexp(pp, -ex);
    };
    Block r0, r1;  // the block after the current one is always in flight
    load(r0, 0);
    for (int i = 0; i < np; i += 16) {
        load(r1, i + 8);
        step(r0);
        load(r0, i + 16 < np ? i + 16 : i);
        step(r1);
    }
    return c;
}
// d of a padding row: far above every probe, so p keeps its sign
constexpr double kSturmPad = 16.0;

// Eigenvalues of T by multisection, one wave per k-point and 64 / S bands (S probes
// per band): a sweep narrows the bracket of every band S + 1-fold.  d and e^2,
// scaled, sit in LDS, uniform reads across the wave.  A bracket is final at the
// rounding level of its eigenvalue or narrower than abstol_rel ||T||_inf; where every
// coupling is felt (e^2 >= eps ||T||^2) also at a sixteenth of the rounding of ||T||, of
// which the reduction has put several into such a T: levels near zero then close one to
// three sweeps earlier (240 k-points, N = 137: 71 us instead of 86).  A T that decouples
// may hold levels of H(k) to their own digits, and keeps them.  At N = 181,
// 16 bands, 4096 k-points (two chunks in flight) the precision form's takes 0.26 ms
// against 0.45 ms with the ratio form of the count (a division a row) and unpadded
// rows.  Alone on the chip it is bound by those reads (LDS busy 80% of the cycles, FP64
// issue 57%), at one k-point by the chain of fmas (69 us).
template <int S>
__global__ __launch_bounds__(64, 4) void tri_eig_wave_kernel(const double* __restrict__ dall,
                                                          const double* __restrict__ eall, int n, int nb,
                                                          double* __restrict__ evals, double* __restrict__ tnorms,
                                                          double abstol_rel, int* __restrict__ kstat,
                                                          unsigned long long* __restrict__ status, int64_t k0) {
    constexpr int NBW = 64 / S;  // bands per wave
    const int64_t kk = blockIdx.x;
    const int lane = threadIdx.x, sub = lane % S;
    const int b = blockIdx.y * NBW + lane / S;
    const bool live = b < nb;
    const double* d = dall + kk * n;
    const double* e = eall + kk * n;
    extern __shared__ double tri_lds[];
    const int np = (n + 15) & ~15;
    double* const sd = tri_lds;
    double* const se2 = tri_lds + np;
    // Gershgorin interval and scale
    double lo = DBL_MAX, hi = -DBL_MAX, tnorm = 0.0, emin = DBL_MAX;
    bool finite = true;
    for (int i = lane; i < n; i += 64) {
        const double di = d[i], el = i > 0 ? fabs(e[i - 1]) : 0.0, er = i + 1 < n ? fabs(e[i]) : 0.0;
        finite = finite && isfinite(di) && isfinite(er);
        lo = fmin(lo, di - el - er);
        hi = fmax(hi, di + el + er);
        tnorm = fmax(tnorm, fabs(di) + el + er);
        if (i + 1 < n || n == 1) emin = fmin(emin, er);
    }
    for (int o = 32; o > 0; o >>= 1) {
        emin = fmin(emin, __shfl_xor(emin, o, 64));
        lo = fmin(lo, __shfl_xor(lo, o, 64));
        hi = fmax(hi, __shfl_xor(hi, o, 64));
        tnorm = fmax(tnorm, __shfl_xor(tnorm, o, 64));
    }
    finite = __all(finite) && isfinite(tnorm);
    // A non-finite T (a non-finite k-point, or H(k) overflowing) has no
    // eigen-decomposition (the reference's Eigen solver reports NoConvergence,
    // Hamiltonian.cpp:130-133): NaN eigenvalues (and, in tri_vec_kernel, vectors), and
    // the k-point is flagged -- in kstat for a later stage to report, or in status
    // directly when this is the last stage.  Both conditions are the same in every wave.
    if (blockIdx.y == 0 && lane == 0) {
        if (tnorms) tnorms[kk] = tnorm;
        if (kstat) kstat[kk] = finite ? 0 : 1;
        else if (status && !finite) {
            atomicAdd(&status[0], 1ull);
            atomicMin(&status[1], (unsigned long long)(k0 + kk));
        }
    }
    if (!finite) {
        if (live && sub == 0) evals[kk * nb + b] = __builtin_nan("");
        return;
    }
    if (tnorm == 0.0) {  // the floor of e^2 would split the levels
        if (live && sub == 0) evals[kk * nb + b] = 0.0;
        return;
    }
    // scaled by a power of two (exact) to 1 <= ||T|| < 2
    const int ex = 1 - __builtin_amdgcn_frexp_exp(tnorm);
    auto scaled = [&](double v) { return __builtin_amdgcn_ldexp(v, ex); };
    for (int i = lane; i < np; i += 64) {
        const double ei = i > 0 && i < n ? scaled(e[i - 1]) : 0.0;
        sd[i] = i < n ? scaled(d[i]) : kSturmPad;
        se2[i] = i < n ? fmax(ei * ei, 0x1p-160) : 0.0;
    }
    __syncthreads();
    const double eps = DBL_EPSILON;
    tnorm = scaled(tnorm);
    lo = scaled(lo) - 2.0 * eps * tnorm - 0x1p-58;  // and what the floor of e^2 may move
    hi = scaled(hi) + 2.0 * eps * tnorm + 0x1p-58;
    emin = scaled(emin);
    const bool coupled = emin * emin >= eps * tnorm * tnorm;
    const double abstol = fmax(abstol_rel, coupled ? eps / 16.0 : 0.0) * tnorm;
    // two shared sweeps first: the wave's 64 lanes probe one interval that holds
    // every band of the wave, and each band takes the probes around its index
    // (a count c at x puts eigenvalues 0..c-1 below x and c.. at or above it)
    {
        const int bw0 = blockIdx.y * NBW;
        const int bw1 = min(nb, bw0 + NBW) - 1;  // last band of this wave
        double L = lo, U = hi;
        for (int sw = 0; sw < 2; ++sw) {
            const double x = L + (double)(lane + 1) * ((U - L) / 65.0);
            const int cnt = sturm_count(sd, se2, np, x);
            double nlo = lo, nhi = hi;
            for (int u = 0; u < 64; ++u) {
                const int cu = __shfl(cnt, u, 64);
                const double xu = __shfl(x, u, 64);
                if (cu > b) nhi = fmin(nhi, xu);
                else nlo = fmax(nlo, xu);
            }
            lo = nlo;
            hi = nhi;
            L = __shfl(lo, 0, 64);  // band bw0 sits on lane 0, band bw1 on lane (bw1 - bw0) S
            U = __shfl(hi, (bw1 - bw0) * S, 64);
        }
    }
    // multisection: lane `sub` of a band probes lo + (sub+1) (hi-lo)/(S+1)
    for (int it = 0; it < 200; ++it) {
        const double w = hi - lo;
        const bool done = !live || w <= 2.0 * eps * fmax(fabs(lo), fabs(hi)) || w <= abstol;
        if (__all(done)) break;
        const double x = lo + (double)(sub + 1) * (w * (1.0 / (double)(S + 1)));
        const int cnt = done ? 0 : sturm_count(sd, se2, np, x);
        // gather the S probes of this band
        double nlo = lo, nhi = hi;
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int cu = __shfl(cnt, lane - sub + u, 64);
            const double xu = __shfl(x, lane - sub + u, 64);
            if (cu > b) nhi = fmin(nhi, xu);
            else nlo = fmax(nlo, xu);
        }
        if (!done) {
            if (nlo >= nhi || (nlo <= lo && nhi >= hi)) {  // no progress possible (rounding): stop here
                lo = hi = 0.5 * (lo + hi);
            } else {
                lo = nlo;
                hi = nhi;
            }
        }
    }
    if (live && sub == 0) evals[kk * nb + b] = __builtin_amdgcn_ldexp(0.5 * (lo + hi), -ex);
}

// Eigenvectors of T by inverse iteration, one lane per (k, band): LU factorisation
// of T - lam I with partial pivoting (rows k, k+1 interchanged when |e_k| >
// |pivot|), `sweeps` sweeps from a fixed pseudo-random start.
//
// The factors of n rows and 16 bands do not fit registers or LDS, and writing them
// out and back bounded the stage (nineteen words a row and band over two sweeps).  Here a
// sweep goes forward once keeping only the elimination's state at every kRows-th
// row, then walks those blocks backwards: each is eliminated again in registers
// (the same operations, so the same values) and substituted back at once.  A sweep
// reads the previous iterate twice and writes one (work arrays interleaved over
// the (k, band) pairs, one coalesced access a row); the last one writes Z, not
// normalised: cluster_orth_kernel does that.  N = 181, 16 bands, 4096 k-points, two
// chunks in flight: 0.33 ms against 0.58 ms with the factors in memory.
constexpr int kRows = 8;
size_t tri_eig_work_doubles(int n, int nb) { return (size_t)(2 * n + 3 * ((n - 1 + kRows - 1) / kRows)) * nb + 1; }
__global__ __launch_bounds__(64, 2) void tri_vec_kernel(const double* __restrict__ dall, const double* __restrict__ eall,
                                                        int n, int nb, int64_t T, const double* __restrict__ evals,
                                                        const double* __restrict__ tnorms, const int* __restrict__ kstat,
                                                        double* __restrict__ W, double* __restrict__ Z, int sweeps) {
    const int64_t t = blockIdx.x * (int64_t)64 + threadIdx.x;
    if (t >= T) return;
    const int64_t kk = t / nb;
    const uint32_t b = (uint32_t)(t - kk * nb);
    double* z = Z + t * n;
    if (kstat[kk]) {
        for (int i = 0; i < n; ++i) z[i] = __builtin_nan("");
        return;
    }
    const double* d = dall + kk * n;
    const double* e = eall + kk * n;
    // T scaled by a power of two (exact), or the last iterate of a tiny T would have no
    // norm in range; a T of zeros counts as of norm 1
    const double tnorm = tnorms[kk];
    const double scl = tnorm > 0.0 ? __builtin_amdgcn_ldexp(1.0, min(1 - __builtin_amdgcn_frexp_exp(tnorm), 1000)) : 1.0;
    const double lam = evals[t] * scl;
    // smallest pivot: under the rounding of T, and large enough that a run of equal
    // levels with next to no coupling cannot grow the iterate out of range
    const double tiny = 0x1p-10 * DBL_EPSILON * (tnorm > 0.0 ? tnorm * scl : 1.0);
    auto at_least_tiny = [&](double a) { return fabs(a) < tiny ? copysign(tiny, a) : a; };
    const int nblk = (n - 1 + kRows - 1) / kRows;  // blocks of eliminated rows 0 .. n - 2
    double* __restrict__ C = W + (size_t)2 * n * T;  // (a, c, y) at every block's first row
    struct State {
        double a, c, y;  // pivot row: a x_k + c x_{k+1} (+ ...) = y
    };
    double sc = 1.0;  // scaling of the previous iterate
    for (int iter = 0; iter < sweeps; ++iter) {
        const double* __restrict__ Xin = W + (size_t)(iter & 1) * n * T;          // previous iterate (iter > 0)
        double* __restrict__ Xout = W + (size_t)((iter & 1) ^ 1) * n * T;
        const bool first = iter == 0, last = iter == sweeps - 1;
        // the rows k0 .. k0 + kRows - 1: d, e and the right-hand side one row ahead
        struct Rows {
            double e[kRows + 1], d[kRows], y[kRows];
        };
        auto load = [&](int k0, Rows& r) {
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
                const int k = k0 + u;
                r.e[u] = e[min(k, n - 1)] * scl;
                r.d[u] = d[min(k + 1, n - 1)];
                if (!first) r.y[u] = Xin[(size_t)min(k + 1, n - 1) * T + t];
            }
            r.e[kRows] = e[min(k0 + kRows, n - 1)] * scl;
        };
        // eliminates row k = k0 + u: multipliers and interchange applied to the state;
        // out: reciprocal pivot, first and second super-diagonal of U, forward result
        auto eliminate = [&](State& s, const Rows& r, int k, int u, double* out) {
            const double sub = r.e[u];
            const double dn = fma(r.d[u], scl, -lam);
            const double en = k + 2 < n ? r.e[u + 1] : 0.0;
            const double y1 = first ? lane_rand((uint32_t)(k + 1), b) : r.y[u] * sc;
            const double a = at_least_tiny(s.a);
            const bool keep = fabs(a) >= fabs(sub);
            const double piv = keep ? a : sub;
            const double rp = rcp_nr64(piv);
            const double mult = (keep ? sub : a) * rp;
            const double u1 = keep ? s.c : dn, u2 = keep ? 0.0 : en;
            const double top = keep ? s.y : y1, bot = keep ? y1 : s.y;
            s.a = (keep ? dn : s.c) - mult * u1;
            s.c = keep ? en : -mult * en;
            s.y = bot - mult * top;
            if (out) {
                out[0] = rp;
                out[1] = u1;
                out[2] = u2;
                out[3] = top;
            }
        };
        State s{fma(d[0], scl, -lam), n > 1 ? e[0] * scl : 0.0, first ? lane_rand(0u, b) : Xin[t] * sc};
        for (int blk = 0; blk < nblk; ++blk) {
            C[(size_t)(3 * blk) * T + t] = s.a;
            C[(size_t)(3 * blk + 1) * T + t] = s.c;
            C[(size_t)(3 * blk + 2) * T + t] = s.y;
            Rows r;
            load(kRows * blk, r);
#pragma unroll
            for (int u = 0; u < kRows; ++u)
                if (kRows * blk + u + 1 < n) eliminate(s, r, kRows * blk + u, u, nullptr);
        }
        auto put = [&](int k, double x) {
            if (last) z[k] = x;
            else Xout[(size_t)k * T + t] = x;
        };
        double x1 = s.y * rcp_nr64(at_least_tiny(s.a)), x2 = 0.0;
        put(n - 1, x1);
        double amax = fabs(x1);
        for (int blk = nblk - 1; blk >= 0; --blk) {
            State q{C[(size_t)(3 * blk) * T + t], C[(size_t)(3 * blk + 1) * T + t], C[(size_t)(3 * blk + 2) * T + t]};
            Rows r;
            load(kRows * blk, r);
            double f[kRows][4];
#pragma unroll
            for (int u = 0; u < kRows; ++u)
                if (kRows * blk + u + 1 < n) eliminate(q, r, kRows * blk + u, u, f[u]);
#pragma unroll
            for (int u = kRows - 1; u >= 0; --u) {
                const int k = kRows * blk + u;
                if (k + 1 < n) {
                    const double x = (f[u][3] - f[u][1] * x1 - f[u][2] * x2) * f[u][0];
                    put(k, x);
                    x2 = x1;
                    x1 = x;
                    amax = fmax(amax, fabs(x));
                }
            }
        }
        sc = 1.0 / amax;
    }
}

// ------------------------------------------------------------ launchers
hipError_t launch_tri_eig(const double* dd, const double* de, int n, int nb, int64_t nk, double* devals, double* dZ,
                          double* dW, int inv_sweeps, double abstol_rel, int* kstat, unsigned long long* status,
                          int64_t k0, hipStream_t s) {
    const size_t shm = sizeof(double) * 2 * (size_t)((n + 15) & ~15);  // d and e^2 of the k-point
    const int64_t T = nk * nb;
    // the work array holds two iterates, the elimination states and, last, the norms
    double* tnorms = inv_sweeps > 0 ? dW + nk * (tri_eig_work_doubles(n, nb) - 1) : nullptr;
    auto eig = [&](auto kern, int bands) {
        hipLaunchKernelGGL(kern, dim3((unsigned)nk, (unsigned)((nb + bands - 1) / bands)), dim3(64), shm, s, dd, de, n, nb,
                           devals, tnorms, abstol_rel, kstat, status, k0);
    };
    if (nb <= 16) eig(tri_eig_wave_kernel<4>, 16);
    else if (nb <= 32) eig(tri_eig_wave_kernel<2>, 32);
    else eig(tri_eig_wave_kernel<1>, 64);
    if (inv_sweeps > 0)
        hipLaunchKernelGGL(tri_vec_kernel, dim3((unsigned)((T + 63) / 64)), dim3(64), 0, s, dd, de, n, nb, T, devals, tnorms,
                           kstat, dW, dZ, inv_sweeps);
    return hipGetLastError();
}

__global__ void pair_levels_kernel(const double* __restrict__ levels, int nb, int64_t n, double* __restrict__ evals) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t < n) evals[t] = levels[t / nb * ((nb + 1) / 2) + t % nb / 2];
}

hipError_t launch_pair_levels(const double* levels, int nb, int64_t nk, double* devals, hipStream_t s) {
    const int64_t n = nk * nb;
    hipLaunchKernelGGL(pair_levels_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, levels, nb, n, devals);
    return hipGetLastError();
}

// status[0] = 0 failed k-points, status[1] = no first index (a kernel node, so
// that a solve captured into a graph clears it on every replay)
__global__ void status_reset_kernel(unsigned long long* status) {
    status[0] = 0ull;
    status[1] = ~0ull;
}

hipError_t launch_status_reset(unsigned long long* status, hipStream_t s) {
    hipLaunchKernelGGL(status_reset_kernel, dim3(1), dim3(1), 0, s, status);
    return hipGetLastError();
}

}  // namespace uepm
