// tridiag_reg.hip — Householder reduction of a complex Hermitian H(k) to real
// symmetric tridiagonal form, one workgroup per k-point and kernel (gfx950): a
// chain of shrinking register grids (256 or 512 lanes, tridiag_grid.hpp) that ends
// in a wave (complex64) or the row kernel (complex128, tridiag_row.hpp).
// Complex64 for the precision form: whole matrices to dim 288, to 384 after the
// strip kernel (tridiag_strip.hpp); complex128 for the FP64 form: to dim 192.
// Larger ones come from the blocked reduction (tridiag_blocked.hip).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>

#include "solver.hpp"
#include "tridiag_grid.hpp"
#include "tridiag_row.hpp"
#include "tridiag_strip.hpp"
#include "wave_ops.hpp"

namespace uepm {

// One wave per k-point for a block of size n <= 64 (complex64; the chain's
// last stage, or the whole reduction of a small matrix).  Lane i keeps row i
// of the Hermitian block in VGPRs, both triangles, in shifted columns: at step
// s, R[t] = A(i, s + t).  Column s is then R[0] on every lane, the product
// y = A v is a local dot product of the row with v (read from LDS, where each
// lane publishes its v_i and w_i), and the rank-2 update writes R[t - 1] from
// R[t], which moves the columns along at no cost.  No barriers: the wave is
// the workgroup.  Columns are processed in blocks of 8, skipped once they are
// past the live part (those registers are never read again).  Same outputs
// as the grid kernels (d, e, tau, reflectors below the sub-diagonal of column
// s of Vout).  The block is read as the grids read it (IN: 1 conjugate of the
// upper triangle of a full Hermitian matrix, 2 lower triangle by rows).
template <int IN, typename THin>
__global__ __launch_bounds__(64, 2) void tridiag_wave64_kernel(const THin* __restrict__ Hin, int64_t h_kstride, int n,
                                                               int ld, float2* __restrict__ Vout, int ldv,
                                                               int64_t v_kstride, double* __restrict__ dout,
                                                               double* __restrict__ eout, float2* __restrict__ tauout,
                                                               int64_t de_kstride) {
    using f2 = c2<float>;
    constexpr int W = 64;
    // (v, w) of lane j at VW[j]; entries W..2W-1 stay zero (columns past the block)
    __shared__ float4 VW[2 * W];
    const int i = threadIdx.x;
    const int64_t kk = blockIdx.x;
    const THin* H = Hin + kk * h_kstride;
    float2* Vk = Vout + kk * v_kstride;
    double* d = dout + kk * de_kstride;
    double* e = eout + kk * de_kstride;
    float2* tau_o = tauout + kk * de_kstride;
    const f2 zero = f2{0.f, 0.f}, one = f2{1.f, 0.f};
    VW[W + i] = make_float4(0.f, 0.f, 0.f, 0.f);

    // ---- row i of the block (zero outside it) ----
    f2 R[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        f2 a = zero;
        if (i < n && j < n) {
            // lower element A(r, c), r >= c, as the grids read it
            const int r = j <= i ? i : j, c = j <= i ? j : i;
            const THin h = H[c + (int64_t)r * ld];
            const float hx = (float)h.x, hy = IN == 1 ? -(float)h.y : (float)h.y;
            a = j <= i ? f2{hx, hy} : f2{hx, -hy};  // A(i, j) = conj(A(j, i)) above the diagonal
        }
        R[j] = a;
    }

    for (int s = 0; s < n - 1; ++s) {
        const int L = n - 1 - s;  // live columns s + 1 .. n - 1 sit in R[1 .. L]
        // ---- reflector from x = A(s+1:, s), redundantly in every lane ----
        const f2 x = R[0];
        const bool below = i > s + 1 && i < n;
        const float xn2 = wave::sum(below ? fmaf(x.x, x.x, x.y * x.y) : 0.f);
        const float alx = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x.x), s + 1));
        const float aly = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x.y), s + 1));
        const float dss = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x.x), s));
        float beta = alx, tr = 0, ti = 0, sr = 1, si = 0;
        if (reflects(xn2, c2<float>{alx, aly})) {
            const float nrm = sqrtf(fmaf(alx, alx, fmaf(aly, aly, xn2)));
            beta = alx >= 0.f ? -nrm : nrm;
            const float ib = rcp_full(beta);
            tr = (beta - alx) * ib;
            ti = -aly * ib;
            const float br = alx - beta, iden = rcp_full(fmaf(br, br, aly * aly));
            sr = br * iden;
            si = -aly * iden;
        }
        const f2 tau = f2{tr, ti}, sc = f2{sr, si};
        if (i == 0) {
            d[s] = (double)dss;
            e[s] = (double)beta;
            tau_o[s] = make_float2(tau.x, tau.y);
        }
        const f2 v = i == s + 1 ? one : (below ? mul(x, sc) : zero);
        if (below) Vk[i + (int64_t)s * ldv] = make_float2(v.x, v.y);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        VW[i] = make_float4(v.x, v.y, 0.f, 0.f);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // ---- y = A v over the live columns (v_j = 0 for j <= s) ----
        f2 y = zero;
#pragma unroll
        for (int b = 0; b < W / 8; ++b) {
            if (8 * b + 1 <= L) {  // wave-uniform
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int t = 8 * b + u + 1;
                    if (t < W) {
                        const float4 q = VW[s + t];
                        fma_ab(y, R[t], f2{q.x, q.y});
                    }
                }
            }
        }
        // ---- w = tau y + alpha v, alpha = -(1/2) |tau|^2 v^H A v ----
        const float vav = wave::sum(fmaf(v.x, y.x, v.y * y.y));
        const float alpha = -0.5f * (tau.x * tau.x + tau.y * tau.y) * vav;
        f2 w = mul(tau, y);
        w.x = fmaf(alpha, v.x, w.x);
        w.y = fmaf(alpha, v.y, w.y);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        VW[i] = make_float4(v.x, v.y, w.x, w.y);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // ---- A -= v w^H + w v^H on the live columns, shifted down by one ----
#pragma unroll
        for (int b = 0; b < W / 8; ++b) {
            if (8 * b + 1 <= L) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int t = 8 * b + u + 1;
                    if (t < W) {
                        const float4 q = VW[s + t];  // (v_j, w_j), j = s + t
                        f2 a = R[t];
                        a.x = fmaf(-v.x, q.z, a.x);
                        a.x = fmaf(-v.y, q.w, a.x);
                        a.x = fmaf(-w.x, q.x, a.x);
                        a.x = fmaf(-w.y, q.y, a.x);
                        a.y = fmaf(-v.y, q.z, a.y);
                        a.y = fmaf(v.x, q.w, a.y);
                        a.y = fmaf(-w.y, q.x, a.y);
                        a.y = fmaf(w.x, q.y, a.y);
                        R[t - 1] = a;
                    }
                }
            }
        }
    }
    // last diagonal element
    {
        const int s = n - 1;
        const float dss = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, R[0].x), s));
        if (i == 0) {
            d[s] = (double)dss;
            e[s] = 0.0;
            tau_o[s] = make_float2(0.f, 0.f);
        }
    }
}

int tridiag_reg_max_n() { return 288; }

// Hand-over between grids.  The late steps of a large grid carry its full
// per-step overhead for a small trailing matrix, so each grid stops where the
// next smaller one can take the trailing block: 288 -> 256 -> 224 -> 192 -> 160 ->
// 128 -> 96 -> 64 (one wave); a first block of 129 .. 144 takes a grid of its own (16 steps
// at 144: 0.34 ms, the 160 grid 0.44).  From 160 down the lanes are 16 x 16, not 32 x 16: four waves
// meet at a step's barriers instead of eight and twice the workgroups share a CU, so
// one's barriers and chains hide behind another's work.  Low-register form throughout
// but for 96, blocks in LDS where that is what one more workgroup takes.  VGPRs and
// workgroups per CU: 288: 256, 16 of 90 blocks in LDS (1); 256: 244 (1); 224: 204 (1); 192:
// 128, 14 of 42 blocks in LDS (2); 160: 168, 12 of 55 (3); 128: 128, 10 of 36 (4); 96: 127
// (4).  32 steps of 2048 matrices, 32 x 16 -> 16 x 16 lanes: 160 0.68 -> 0.63 ms, 128 0.51 ->
// 0.41, 96 0.32 -> 0.26; at 192 (21 steps) 32 x 16 stays the faster, 0.65 against 0.74.
namespace {
constexpr int kNumGrids = 9;
constexpr int kGrid[kNumGrids] = {288, 256, 224, 192, 160, 144, 128, 96, 64};
// index of the smallest grid that holds n
int grid_of(int n) {
    int g = 0;
    while (g < kNumGrids - 1 && n <= kGrid[g + 1]) ++g;
    return g;
}
}  // namespace

int tridiag_reg_split(int n) {
    if (n > kGrid[0]) return kGrid[0];
    if (n > 128 && n <= 160) return 128;  // 144 takes first blocks only
    if (n > 160 && n <= 192) return 160;
    const int g = grid_of(n);
    return g < kNumGrids - 1 ? kGrid[g + 1] : 0;
}

namespace {
template <int IN, typename THin>
void wave64_stage(const THin* H, int64_t h_kstride, int n, int ld, int64_t nk, float2* V, int ldv, int64_t v_kstride,
                  double* dd, double* de, float2* dtau, int64_t de_kstride, hipStream_t s) {
    hipLaunchKernelGGL((tridiag_wave64_kernel<IN, THin>), dim3((unsigned)nk), dim3(64), 0, s, H, h_kstride, n, ld, V, ldv,
                       v_kstride, dd, de, dtau, de_kstride);
}

constexpr int NL288 = 16, NL192 = 14, NL160 = 12, NL144 = 14, NL128 = 10;  // blocks held in LDS by these grids

template <typename THin, int IN>
void grid_stage(int g, const THin* H, int64_t hk, int m, int ld, int64_t nk, float2* V, int ldv, int64_t vk,
                double* dd, double* de, float2* dtau, int64_t dk, int s_end, float2* B, int ldb, int64_t bk, hipStream_t s) {
    switch (g) {
        case 0: reg_stage<c2<float>, 32, 9, 2, IN, THin, true, NL288>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        case 1: reg_stage<c2<float>, 32, 8, 2, IN, THin, true>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        case 2: reg_stage<c2<float>, 32, 7, 2, IN, THin, true>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        case 3: reg_stage<c2<float>, 32, 6, 4, IN, THin, true, NL192>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        case 4: reg_stage<c2<float>, 16, 10, 3, IN, THin, true, NL160>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        case 5:
            if constexpr (IN == 1) reg_stage<c2<float>, 16, 9, 4, IN, THin, true, NL144>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk);
            break;
        case 6: reg_stage<c2<float>, 16, 8, 4, IN, THin, true, NL128>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        case 7: reg_stage<c2<float>, 16, 6, 4, IN, THin>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s, bk); break;
        default: wave64_stage<IN, THin>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s); break;  // last: s_end >= m - 1
    }
}
}  // namespace

namespace {
// The rest of a complex64 chain: the hand-over block of size r in work (bk per k), then
// each smaller grid's over it (a stage reads its whole block before its first step and
// writes the next after its last); outputs at the block's own offset.
hipError_t c64_blocks(int r, float2* work, int64_t bk, int64_t nk, float2* V, int ldv, int64_t vk, double* dd, double* de,
                      float2* dtau, int64_t dk, hipStream_t s) {
    for (int off = 0;;) {
        const int t = tridiag_reg_split(r);
        grid_stage<float2, 2>(grid_of(r), (const float2*)work, bk, r, r, nk, V + off + (int64_t)off * ldv, ldv, vk, dd + off,
                              de + off, dtau + off, dk, t ? r - t : r, t ? work : (float2*)nullptr, t, bk, s);
        if (!t) break;
        off += r - t;
        r = t;
    }
    return hipGetLastError();
}

// Larger blocks, up to 384: the strip kernel takes the leading m - 288 steps (2.7 times
// as fast as the blocked reduction at 362; every column of a longer strip adds as much to
// the first step's traffic, and at 96 columns that is what the blocked one streams).
constexpr int kStripMax = 384, kStripCols = (kStripMax - kGrid[0]) / 16, NLStrip = 30;
constexpr int kStripSlots = strip_slots(kStripMax / 32, kStripCols);

// The complex64 chain above 288 on a block of size m whose element (0, 0) sits at H
// (leading dimension ld, per-k stride hk; read as IN says, IN = 0 or 1); outputs at the
// block's offset of the full matrix's V (ldv, stride vk) and d, e, tau (stride dk).  work:
// the hand-over blocks of the k-points, then their strips.
template <int IN, typename THin>
hipError_t strip_chain(const THin* H, int64_t hk, int m, int ld, int64_t nk, float2* V, int ldv, int64_t vk, double* dd,
                       double* de, float2* dtau, int64_t dk, float2* work, hipStream_t s) {
    if (!work || m <= kGrid[0] || m > kStripMax) return hipErrorInvalidValue;
    constexpr int64_t bk = (int64_t)kGrid[0] * kGrid[0];
    hipLaunchKernelGGL((tridiag_strip_kernel<kStripMax / 32, kStripCols, NLStrip, IN, THin>), dim3((unsigned)nk), dim3(512),
                       0, s, H, hk, m, ld, V, ldv, vk, dd, de, dtau, dk, work, bk, work + nk * bk, (int64_t)kStripSlots);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int off = m - kGrid[0];
    return c64_blocks(kGrid[0], work, bk, nk, V + off + (int64_t)off * ldv, ldv, vk, dd + off, de + off, dtau + off, dk, s);
}
}  // namespace

size_t tridiag_reg_work_bytes(int n) {
    // the first hand-over block (the later ones go over it) and, above 288, the strip
    const int t = tridiag_reg_split(n);
    return sizeof(float2) * ((size_t)t * t + (n > kGrid[0] ? kStripSlots : 0));
}

hipError_t launch_tridiag_reg_c64(const double2* dH, int n, int ld, int64_t nk, float2* Vout, double* dd, double* de,
                                  float2* dtau, float2* work, hipStream_t s) {
    if (n < 1 || n > kStripMax || nk <= 0) return hipErrorInvalidValue;
    const int64_t hk = (int64_t)ld * n;
    if (n > kGrid[0]) return strip_chain<1>(dH, hk, n, ld, nk, Vout, ld, hk, dd, de, dtau, n, work, s);
    const int t = tridiag_reg_split(n);
    if (t && !work) return hipErrorInvalidValue;
    // first grid on the matrix, then each smaller grid on the trailing block of its size
    const int64_t bk = (int64_t)t * t;
    grid_stage<double2, 1>(grid_of(n), dH, hk, n, ld, nk, Vout, ld, hk, dd, de, dtau, n, t ? n - t : n,
                           t ? work : (float2*)nullptr, t, bk, s);
    if (!t) return hipGetLastError();
    const int off = n - t;
    return c64_blocks(t, work, bk, nk, Vout + off + (int64_t)off * ld, ld, hk, dd + off, de + off, dtau + off, n, s);
}

int tridiag_reg_c64_tail(int n) {
    if (n < 2) return 0;
    if (n <= kStripMax) return n;
    const int P = tridiag_blocked_panel((int)sizeof(float2));
    const int s0 = ((n - kStripMax + P - 1) / P) * P;
    return n - s0;
}

hipError_t launch_tridiag_reg_c64_block(const float2* H, int64_t hk, int m, int ld, int64_t nk, float2* V, int ldv,
                                        int64_t vk, double* dd, double* de, float2* dtau, int64_t dk, float2* work,
                                        hipStream_t s) {
    if (nk <= 0) return hipErrorInvalidValue;
    return strip_chain<0>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, work, s);
}

// ---- FP64: grids 192 (10 of 42 blocks in LDS) and 160 of 32 x 16 lanes, 256 and 236
// VGPRs, one workgroup per CU; 128 and 96 of 16 x 16 lanes, two and three (32 steps of
// 2048 matrices, 32 x 16 -> 16 x 16 lanes: 137 -> 128 0.58 -> 0.46, 128 1.15 -> 0.80 ms, 96 0.62 -> 0.49; 160 1.55
// against 1.65; one matrix alone takes a tenth longer on half the lanes).  The last 64 steps run one row per lane in two
// column waves, four workgroups per CU (tridiag_row.hpp; 4096 blocks of 64 take
// 0.59 ms, a 2 x 4 grid 1.48; blocks of 27 in one wave 0.14; at 96 the grid is
// the faster, 1.0 ms for 32 steps against 1.50).  A larger FP64 matrix runs the
// blocked reduction first and hands over its trailing block at a panel boundary.
namespace {
constexpr int kNumGrids64 = 6;
constexpr int kGrid64[kNumGrids64] = {192, 160, 144, 128, 96, 64};
int grid64_of(int n) {
    int g = 0;
    while (g < kNumGrids64 - 1 && n <= kGrid64[g + 1]) ++g;
    return g;
}
int split64(int n) {
    if (n > 128) return n > 160 ? 160 : 128;  // 144 takes first blocks only
    const int g = grid64_of(n);
    return g < kNumGrids64 - 1 ? kGrid64[g + 1] : 0;
}
constexpr int NL64_192 = 10, NL64_144 = 12, NL64_128 = 2, NL64_96 = 4;  // blocks held in LDS by these FP64 grids
template <int IN>
void grid64_stage(int g, const double2* H, int64_t hk, int m, int ld, int64_t nk, double2* V, int ldv, int64_t vk,
                  double* dd, double* de, double2* dtau, int64_t dk, int s_end, double2* B, int ldb, hipStream_t s) {
    if constexpr (IN == 0) {  // what the blocked reduction leaves: 189 .. 192
        reg_stage<c2<double>, 32, 6, 1, IN, double2, true, NL64_192>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
    } else {
        switch (g) {
            case 0:
                if constexpr (IN == 1) reg_stage<c2<double>, 32, 6, 1, IN, double2, true, NL64_192>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
                break;
            case 1: reg_stage<c2<double>, 32, 5, 1, IN, double2, true>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s); break;
            case 2:
                if constexpr (IN == 1) reg_stage<c2<double>, 16, 9, 2, IN, double2, true, NL64_144>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
                break;
            case 3: reg_stage<c2<double>, 16, 8, 2, IN, double2, true, NL64_128>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s); break;
            // hands both triangles to the row kernel
            case 4: reg_stage<c2<double>, 16, 6, 3, IN, double2, true, NL64_96, true>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s); break;
            default:
                if (m <= 32) row_stage<c2<double>, 1, 1, 2, 2, IN>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
                else row_stage<c2<double>, 1, 2, 2, 2, IN>(H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
                break;
        }
    }
}
}  // namespace

int tridiag_reg_c128_tail(int n) {
    if (n < 2) return 0;
    if (n <= kGrid64[0]) return n;
    // the blocked reduction stops at a panel boundary s0 >= n - 192
    const int P = tridiag_blocked_panel((int)sizeof(double2));
    const int s0 = ((n - kGrid64[0] + P - 1) / P) * P;
    return n - s0;
}

size_t tridiag_reg_c128_work_bytes(int m) {
    const int t1 = split64(m);
    if (!t1) return 0;
    const int t2 = split64(t1);
    return sizeof(double2) * ((size_t)t1 * t1 + (size_t)t2 * t2);
}

hipError_t launch_tridiag_reg_c128(const double2* H, int64_t hk, int m, int ld, bool hermitian_full, int64_t nk,
                                   double2* V, int ldv, int64_t vk, double* dd, double* de, double2* dtau, int64_t dk,
                                   double2* work, hipStream_t s) {
    if (m < 1 || m > kGrid64[0] || nk <= 0) return hipErrorInvalidValue;
    if (!hermitian_full && grid64_of(m) != 0) return hipErrorInvalidValue;
    // the first grid reads the block's rows (the conjugate upper triangle) when
    // the whole Hermitian matrix is there, its lower columns otherwise
    auto first = [&](int s_end, double2* B, int ldb) {
        if (hermitian_full)
            grid64_stage<1>(grid64_of(m), H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
        else
            grid64_stage<0>(grid64_of(m), H, hk, m, ld, nk, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb, s);
    };
    const int t1 = split64(m);
    if (!t1) {
        first(m, nullptr, 0);
        return hipGetLastError();
    }
    if (!work) return hipErrorInvalidValue;
    double2* buf[2] = {work, work + nk * (int64_t)t1 * t1};
    first(m - t1, buf[0], t1);
    int r = t1, cur = 0;
    while (true) {
        const int off = m - r;
        const int t = split64(r);
        grid64_stage<2>(grid64_of(r), buf[cur], (int64_t)r * r, r, r, nk, V + off + (int64_t)off * ldv, ldv, vk, dd + off,
                     de + off, dtau + off, dk, t ? r - t : r, t ? buf[cur ^ 1] : (double2*)nullptr, t, s);
        if (!t) break;
        r = t;
        cur ^= 1;
    }
    return hipGetLastError();
}

}  // namespace uepm
