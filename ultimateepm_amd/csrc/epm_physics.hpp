// epm_physics.hpp — per-element physics of the EPM Hamiltonian H(k) on gfx950.
//
// Device-side statement of the reference's element functions:
//   local V(G_i - G_j)      Pseudopotential::GetValue           src/EPP/Pseudopotential.cpp:24-56
//   kinetic diagonal        Hamiltonian::SetMatrix              src/EPP/Hamiltonian.cpp:61-74
//   non-local correction    Material::compute_pseudopotential_non_local_correction,
//                           F_l_function, F_2_function_gaussian src/EPP/Material.cpp:87-208
//   spherical Bessel j_l    generalized_bessel / J_neg_v        src/EPP/bessel_func.hpp:17-45
//   modified Bessel i_2     bessel_2nd_order_first_kind         src/EPP/bessel_func.hpp:47-52
//   spin-orbit 2x2 block    SpinOrbitCorrection                 src/EPP/SpinOrbitFunctional.cpp:20-138
//
// Expressions keep the reference's operation order and are compiled without
// FMA contraction (the pragma below), so an element differs from the
// reference only through the last-ulp behaviour of sin/cos/exp/sqrt and of
// the Bessel functions: those are evaluated here in closed form (with power
// series where the closed form cancels) instead of libstdc++'s
// std::cyl_bessel_j(l + 1/2, x), which the reference calls per element.  The
// rearrangements, each worth a few ulp of its term: the non-local phase
// exp(2 pi i (tau/a) . (K_i - K_j)) and the spin-orbit phase are products of
// per-vector ones, so is exp(-(K_i^2 + K_j^2) R^2 / 4) of a gaussian well,
// divisions by |K_i| |K_j| and |K_i|^2 - |K_j|^2 are products with reciprocals,
// and each element is formed hermitised at once.
//
// The per-basis-vector quantities (|K_i|, j_l(|K_i| R), SOC radial factors)
// are k-dependent but element-independent, so they are computed once per
// (k, i) and the O(N^2) element loop only combines them.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace uepm {

// Everything an element needs, precomputed on the host from uepm_material
// with the reference's expressions (src/Common/physical_constants.hpp:18-41).
struct DevParams {
    int32_t N;          // basis size
    int32_t dim;        // N or 2N
    int32_t nl;         // non-local correction on
    int32_t soc;        // spin-orbit on
    int32_t well;       // 0 square, 1 gaussian (anything else: gaussian, as the reference's else-branch)
    int32_t nb;         // bands kept per k
    int32_t need_l0_a, need_l0_c;  // F_0 needed (R0 != 0) for anion / cation
    int32_t need_l2_a, need_l2_c;  // A2 != 0
    int32_t period_a, period_c;    // SOC radial-factor periods
    int32_t same_r0;    // need_l0_a && need_l0_c && R0_a == R0_c
    int32_t same_r2;    // need_l2_a && need_l2_c && R2_a == R2_c
    double a;           // lattice constant [m]
    double tau;         // a / 8 [m]
    double tpa;         // 2 pi / a
    double kin;         // (2 pi / a)^2 * hbar^2 / (2 m_e q_e): tpa * tpa * diag_factor
    double VS[4], VA[4];
    // non-local
    double fourier;     // 2 pi / a
    double diag_factor; // hbar^2 / (2 m_e q_e)
    double kF2;         // pow(kF, 2.0)
    double V_pre;       // 4 pi / Omega_at
    double tau_over_a;  // (a / 8) / a
    double alpha0_a, dfbeta_a, A2_a, R0_a, R2_a, gpre_a;  // dfbeta = diag_factor * beta_0
    double alpha0_c, dfbeta_c, A2_c, R0_c, R2_c, gpre_c;  // gpre = 5 pi^1.5 R2^3 / Omega
    // products the element loop would otherwise keep in vector registers (a double
    // that every lane shares is a scalar operand only if the host forms it)
    double w2_a, w2_c;                      // l = 2: V_pre A2 5 (square well), gpre A2 (gaussian)
    double h2_a, h2_c;                      // R2^2 / 2 (gaussian)
    struct Radius {
        double R2, R3_2, R3_3;              // R^2, R^3 / 2, and for l = 0 R^3 / 3 (else 0)
    } r0_a, r0_c, r2_a, r2_c;
    // spin-orbit
    double soc_kfac;    // (2 pi) / a
    double xi_a, xi_c;  // radial extents
    double mu, alpha_mu;// mu_soc, alpha_soc * mu_soc
    double bohr;        // Bohr radius [m]
    // gradient
    double grad_pref;   // 2 * diag_factor * tpa^2
    double frac_to_phys;// 1 / tpa
};

#pragma clang fp contract(off)

// Spherical Bessel j_l(x), l in {-1, 0, 1, 2, 3}, x >= 0, with the special
// cases of generalized_bessel (bessel_func.hpp:29-45): x < 1e-14 gives 1 for
// l = 0 and 0 for l >= 1.  Closed forms (DLMF 10.49.3) above the cancellation
// region, the ascending series (DLMF 10.53.1) below it.
__device__ __forceinline__ double sph_series(int l, double x) {
    // x^l / (2l+1)!! * sum_k (-x^2/2)^k / (k! (2l+3)(2l+5)...(2l+2k+1))
    double dfact = 1.0;
    double xl = 1.0;
    for (int i = 1; i <= l; ++i) {
        dfact *= (double)(2 * i + 1);
        xl *= x;
    }
    const double h = -0.5 * x * x;
    double term = 1.0, sum = 1.0;
    for (int k = 1; k < 24; ++k) {
        term *= h / ((double)k * (double)(2 * l + 2 * k + 1));
        sum += term;
    }
    return xl / dfact * sum;
}

__device__ __forceinline__ double sph_j(int l, double x) {
    if (l == -1) return cos(x) / x;
    if (x < 1e-14) return l == 0 ? 1.0 : 0.0;
    const double lim = (l == 0) ? 0.25 : (double)l;
    if (x < lim) return sph_series(l, x);
    double s, c;
    sincos(x, &s, &c);
    const double ix = 1.0 / x;
    switch (l) {
        case 0: return s * ix;
        case 1: return (s * ix - c) * ix;
        case 2: return ((3.0 * ix * ix - 1.0) * s * ix - 3.0 * c * ix * ix);
        default: return ((15.0 * ix * ix * ix - 6.0 * ix) * s * ix - (15.0 * ix * ix - 1.0) * c * ix);
    }
}

// Modified spherical Bessel function i_2(x), x >= 0 (bessel_func.hpp:47-52:
// ((x^2 + 3) sinh x - 3 x cosh x) / x^3).  That difference cancels like x^5
// below x = 2; the ascending series (DLMF 10.53.3) does not, and costs no
// exponential.  Above, sinh and cosh come from one exponential.
__device__ __forceinline__ double mod_i2(double x) {
    const double x2 = x * x;
    if (x < 2.0) {
        // x^2 / 15 sum_k prod_{i <= k} x^2 / (2 i (2 i + 5)); at x = 2 the thirteenth term is below 1e-17
        double s = 1.0;
#pragma unroll
        for (int k = 12; k >= 1; --k) s = fma(s, x2 * (1.0 / (double)(2 * k * (2 * k + 5))), 1.0);
        return x2 * (1.0 / 15.0) * s;
    }
    const double e = exp(x), m = 1.0 / e;
    const double sh = 0.5 * (e - m), ch = 0.5 * (e + m);
    return ((x2 + 3) * sh - 3 * x * ch) / (x2 * x);
}

// SpinOrbitFunctional.cpp:20-49 (period 2, 3, 4; others rejected on the host)
__device__ __forceinline__ double soc_radial(int period, double Klen, double bohr, double xi) {
    const double kappa = Klen * bohr / xi;
    const double q = 1.0 + kappa * kappa;
    if (period == 2) return 1.0 / (q * q * q);
    if (period == 3) return (5.0 - kappa * kappa) / (5.0 * (q * q * q * q));
    return (5.0 - 3.0 * kappa * kappa) / (5.0 * (q * q * q * q * q));
}

// Per-basis-vector state of one k-point, in LDS as arrays of N doubles (lanes
// of consecutive vectors then read consecutive words), with only the arrays
// that the plan's terms use: the fewer bytes per k-point, the more k-points a
// CU assembles at once.  Offsets in arrays; a radial integral takes three:
//   j_l(x), j_{l+1}(x) and, for equal norms, j_l^2 - j_{l-1} j_{l+1}, x = |K| R
// (a gaussian l = 2 well one: exp(-(|K| R)^2 / 4)).
struct VecLayout {
    int32_t k = 0;                    // k + G, reduced: 3 arrays
    int32_t nK = 0;                   // |K|
    int32_t ph = 0;                   // cos, sin of theta = 2 pi (tau/a) sum_c (k + G)_c
    int32_t ik = 0;                   // 1 / |k + G|
    int32_t l0a = 0, l0c = 0, l2a = 0, l2c = 0;  // radial integrals (cation: the anion's when the radii are equal)
    int32_t B = 0;                    // spin-orbit radial factors of anion and cation
    int32_t q = 0;                    // cos, sin of the spin-orbit phase of G
    int32_t count = 0;                // arrays in all (and three of int32 after them: the components of G)
};
__host__ __device__ inline VecLayout vec_layout(const DevParams& P) {
    VecLayout L;
    int n = 0;
    L.k = n; n += 3;
    if (P.nl) {
        const int l2 = P.well == 0 ? 3 : 1;
        L.nK = n; n += 1;
        L.ph = n; n += 2;
        if (P.need_l2_a || P.need_l2_c) { L.ik = n; n += 1; }
        if (P.need_l0_a) { L.l0a = n; n += 3; }
        if (P.need_l0_c) { L.l0c = P.same_r0 ? L.l0a : n; n += P.same_r0 ? 0 : 3; }
        if (P.need_l2_a) { L.l2a = n; n += l2; }
        if (P.need_l2_c) { L.l2c = P.same_r2 ? L.l2a : n; n += P.same_r2 ? 0 : l2; }
    }
    if (P.soc) {
        L.B = n; n += 2;
        L.q = n; n += 2;
    }
    L.count = n;
    return L;
}
__host__ __device__ inline size_t vec_bytes(const DevParams& P) {
    return (sizeof(double) * (size_t)vec_layout(P).count + 3 * sizeof(int32_t)) * (size_t)P.N;
}

__device__ __forceinline__ void radial_init(int l, double nK, double R, double* S, int N, int i) {
    const double x = nK * R;
    const double jm = sph_j(l - 1, x), j0 = sph_j(l, x), jp = sph_j(l + 1, x);
    S[i] = j0;
    S[N + i] = jp;
    S[2 * N + i] = j0 * j0 - jm * jp;
}

__device__ __forceinline__ void vector_init(const DevParams& P, const VecLayout& L, const double* k, const int32_t* G,
                                            int i, double* S, int32_t* Gs) {
    const int N = P.N;
    const int gx = G[3 * i], gy = G[3 * i + 1], gz = G[3 * i + 2];
    const double kx = k[0] + (double)gx, ky = k[1] + (double)gy, kz = k[2] + (double)gz;
    Gs[i] = gx;
    Gs[N + i] = gy;
    Gs[2 * N + i] = gz;
    S[L.k * N + i] = kx;
    S[(L.k + 1) * N + i] = ky;
    S[(L.k + 2) * N + i] = kz;
    const double Kx = kx * P.fourier, Ky = ky * P.fourier, Kz = kz * P.fourier;
    const double nK = sqrt(Kx * Kx + Ky * Ky + Kz * Kz);
    if (P.nl) {
        S[L.nK * N + i] = nK;
        double s, c;
        sincos(2.0 * 3.14159265358979323846 * (P.tau_over_a * kx + P.tau_over_a * ky + P.tau_over_a * kz), &s, &c);
        S[L.ph * N + i] = c;
        S[(L.ph + 1) * N + i] = s;
        if (P.need_l2_a || P.need_l2_c) S[L.ik * N + i] = P.fourier / nK;
        if (P.need_l0_a) radial_init(0, nK, P.R0_a, S + L.l0a * N, N, i);
        if (P.need_l0_c && !P.same_r0) radial_init(0, nK, P.R0_c, S + L.l0c * N, N, i);
        if (P.well == 0) {
            if (P.need_l2_a) radial_init(2, nK, P.R2_a, S + L.l2a * N, N, i);
            if (P.need_l2_c && !P.same_r2) radial_init(2, nK, P.R2_c, S + L.l2c * N, N, i);
        } else {
            if (P.need_l2_a) S[L.l2a * N + i] = exp(-0.25 * (nK * nK) * (P.R2_a * P.R2_a));
            if (P.need_l2_c && !P.same_r2) S[L.l2c * N + i] = exp(-0.25 * (nK * nK) * (P.R2_c * P.R2_c));
        }
    }
    if (P.soc) {
        // Kphys = kfac * K (SpinOrbitFunctional.cpp:109-110) is K above: soc_kfac == fourier
        S[L.B * N + i] = soc_radial(P.period_a, nK, P.bohr, P.xi_a);
        S[(L.B + 1) * N + i] = soc_radial(P.period_c, nK, P.bohr, P.xi_c);
        double s, c;
        // soc_kfac tau is pi / 4: the phase has eight values, formed from the smallest
        // argument (that of G itself grows with a basis far from the origin)
        sincos(P.soc_kfac * (P.tau * (double)(((unsigned)gx + (unsigned)gy + (unsigned)gz) & 7u)), &s, &c);
        S[L.q * N + i] = c;
        S[(L.q + 1) * N + i] = s;
    }
}

// (cos, sin) of the phase of V(G) for integer G (Pseudopotential.cpp:24-56).
__device__ __forceinline__ double2 local_phase(const DevParams& P, int gx, int gy, int gz) {
    const double Gtau = P.tpa * (P.tau * (double)gx + P.tau * (double)gy + P.tau * (double)gz);
    double s, c;
    sincos(Gtau, &s, &c);
    return make_double2(c, s);
}

// The form factors vanish outside G^2 in {3, 4, 8, 11}, which bounds every
// component of G by 3: a table of local_phase over [-3, 3]^3 (343 entries,
// built on the device with the same expression) serves every pair.
constexpr int kVPhaseTab = 343;
__device__ __forceinline__ int local_phase_index(int gx, int gy, int gz) { return (gx + 3) * 49 + (gy + 3) * 7 + (gz + 3); }

// Pseudopotential::GetValue for integer G = G_i - G_j (Pseudopotential.cpp:24-56);
// tab: nullptr to evaluate the phase here, else the table above.
__device__ __forceinline__ void local_V(const DevParams& P, int gx, int gy, int gz, double& re, double& im,
                                        const double2* tab = nullptr) {
    const int G2 = gx * gx + gy * gy + gz * gz;
    double VS = 0.0, VA = 0.0;
    switch (G2) {
        case 3: VS = P.VS[0]; VA = P.VA[0]; break;
        case 4: VS = P.VS[1]; VA = P.VA[1]; break;
        case 8: VS = P.VS[2]; VA = P.VA[2]; break;
        case 11: VS = P.VS[3]; VA = P.VA[3]; break;
        default: re = 0.0; im = 0.0; return;  // VS = VA = 0: 0*cos = 0, 0*sin = 0
    }
    const double2 cs = tab ? tab[local_phase_index(gx, gy, gz)] : local_phase(P, gx, gy, gz);
    re = VS * cs.x;
    im = VA * cs.y;
}

// F_l (Material.cpp:87-109) of the pair (i, j), averaged over its two orders.
// The general branch is symmetric in them.  Norms within 1e-4 of each other
// take the first vector's own value: the mean of both orders, as the
// hermitisation 0.5 (H + H^dagger) leaves it.  id: 1 / (n1^2 - n2^2).
__device__ __forceinline__ double F_l(double n1, double n2, double id, const DevParams::Radius& R, const double* S, int N,
                                      int i, int j) {
    constexpr double EPSILON = 1.0e-4;
    if (fabs(n1 - n2) > EPSILON) {
        const double F = n1 * S[N + i] * S[j] - n2 * S[N + j] * S[i];
        return R.R2 * id * F;
    }
    return 0.5 * ((n1 > EPSILON ? R.R3_2 * S[2 * N + i] : R.R3_3) + (n2 > EPSILON ? R.R3_2 * S[2 * N + j] : R.R3_3));
}

// Material::compute_pseudopotential_non_local_correction (Material.cpp:139-208),
// hermitised: every factor is symmetric in the pair or (the phase) conjugated by
// its exchange, so one evaluation serves both elements.
__device__ __forceinline__ void nonlocal(const DevParams& P, const VecLayout& L, const double* S, int i, int j, double& re,
                                         double& im) {
    const int N = P.N;
    const double n1 = S[L.nK * N + i], n2 = S[L.nK * N + j];
    double leg2 = 0.0;  // P_2(cos angle(K1, K2)), used by the l = 2 terms only
    if (P.need_l2_a || P.need_l2_c) {
        const double* kx = S + L.k * N;
        const double dp = kx[i] * kx[j] + kx[N + i] * kx[N + j] + kx[2 * N + i] * kx[2 * N + j];
        const double cosang = (n1 * n2 < 1.0e-13) ? 1.0 : dp * (S[L.ik * N + i] * S[L.ik * N + j]);
        leg2 = 0.5 * (3 * cosang * cosang - 1);
    }
    const double nn = n1 * n2 - P.kF2;
    const bool any_F = P.need_l0_a || P.need_l0_c || P.well == 0;
    const double id = any_F ? 1.0 / (n1 * n1 - n2 * n2) : 0.0;
    double Va = 0.0, Vc = 0.0;
    double F0 = 0.0, F2 = 0.0;
    auto radial2 = [&](const DevParams::Radius& R, double h2, int at) {
        if (P.well == 0) return F_l(n1, n2, id, R, S + at * N, N, i, j);
        return mod_i2(h2 * (n1 * n2)) * (S[at * N + i] * S[at * N + j]);
    };
    if (P.need_l0_a) {
        F0 = F_l(n1, n2, id, P.r0_a, S + L.l0a * N, N, i, j);
        Va = P.V_pre * (P.alpha0_a + P.dfbeta_a * nn) * F0;
    }
    if (P.need_l2_a) {
        F2 = radial2(P.r2_a, P.h2_a, L.l2a);
        Va += P.w2_a * leg2 * F2;
    }
    if (P.need_l0_c) {
        if (!P.same_r0) F0 = F_l(n1, n2, id, P.r0_c, S + L.l0c * N, N, i, j);
        Vc = P.V_pre * (P.alpha0_c + P.dfbeta_c * nn) * F0;
    }
    if (P.need_l2_c) {
        if (!P.same_r2) F2 = radial2(P.r2_c, P.h2_c, L.l2c);
        Vc += P.w2_c * leg2 * F2;
    }
    const double Vs = 1.0 * (Va + Vc) / 2.0;
    const double Vas = 1.0 * (Va - Vc) / 2.0;
    // cos / sin of 2 pi (tau/a) sum_c (K_a - K_b)_c from the per-vector phases
    // (the reference forms the difference first; the two agree to rounding)
    const double *pc = S + L.ph * N, *ps = pc + N;
    const double c = pc[i] * pc[j] + ps[i] * ps[j];
    const double s = ps[i] * pc[j] - pc[i] * ps[j];
    re = c * Vs;
    im = s * Vas;
}

// SpinOrbitCorrection::compute_soc_contribution (SpinOrbitFunctional.cpp:111-138):
// s[0..5] = s00, s01, s10 as (re, im) pairs; s11 = -s00.  Exchanging the pair
// conjugate-transposes the block exactly, so it is its own hermitisation.
__device__ __forceinline__ void soc_block(const DevParams& P, const VecLayout& L, const double* S, int i, int j, double* s) {
    const int N = P.N;
    const double *Ba = S + L.B * N, *Bc = Ba + N, *qc = S + L.q * N, *qs = qc + N;
    const double l1 = P.mu * (Bc[i] * Bc[j]);
    const double l2 = P.alpha_mu * (Ba[i] * Ba[j]);
    const double lsym = (l1 + l2) / 2.0;
    const double lanti = (l1 - l2) / 2.0;
    const double *kx = S + L.k * N, *ky = kx + N, *kz = ky + N;
    const double cz = kx[i] * ky[j] - ky[i] * kx[j];
    const double cx = ky[i] * kz[j] - kz[i] * ky[j];
    const double cy = kx[i] * kz[j] - kz[i] * kx[j];
    // the phase of G_i - G_j from the per-vector phases
    const double cs = qc[i] * qc[j] + qs[i] * qs[j];
    const double sn = qs[i] * qc[j] - qc[i] * qs[j];
    const double pr = lanti * sn, pi = -lsym * cs;
    s[0] = cz * pr;            s[1] = cz * pi;
    s[2] = cx * pr - cy * pi;  s[3] = cx * pi + cy * pr;
    s[4] = cx * pr + cy * pi;  s[5] = cx * pi - cy * pr;
}

#pragma clang fp contract(on)

}  // namespace uepm
