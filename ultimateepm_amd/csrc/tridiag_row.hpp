// tridiag_row.hpp — Householder reduction of a real symmetric or complex Hermitian
// block, one matrix row per lane (gfx950).
//
// Layout.  A workgroup of RW x CW waves takes one k-point.  Lane l of a wave
// (rw, cw) keeps row i = 64 rw + l of the block in VGPRs (both triangles), the
// columns of every CW-th group of 16: group q = CW g + cw, register A[g][r] =
// A(i, 16 q + r).  Then
//
//   y_i = sum_j A(i, j) v_j                             is a sum over the lane's own registers,
//   A(i, j) += c1_i conj(y_j) + c2_i conj(v_j)          is the rank-2 update (below),
//
// and neither needs a cross-lane reduction.  v_j and y_j reach the lanes of a
// wave as DPP operands (row_ops.hpp): every 16-lane row holds the 16 values of a
// group, one LDS read per lane and group.
//
// Step s: the owner of column s publishes it in LDS | barrier | beta, tau, v in
// every wave; y = A v; each wave's share of y and of v^H A v to LDS | barrier |
// A -= v w^H + w v^H with w = y tau + alpha v, alpha = -(1/2) |tau|^2 v^H A v,
// written with c1_i = -v_i conj(tau), c2_i = -(y_i tau + 2 alpha v_i), so that w
// is never formed.  v and y are zero at rows <= s: dead rows and columns inside
// a live group take no part.
//
// Against the cyclic lower-triangle grid this does 1.5 times the multiply-adds
// (both triangles are updated) but none of the reductions, which were two thirds
// of a real step's instructions.  It pays where a wave's share of the square fits
// the registers of two or more waves per SIMD, in FP64 above all, where the DPP
// operand is free.
#pragma once
#include "row_ops.hpp"
#include "scalars.hpp"
#include "wave_ops.hpp"

namespace uepm {
namespace {

// A[r] for a wave-uniform r: a tree of selects (of values: a select of two array
// elements would be one of their addresses, and put the array in memory)
template <typename R>
__device__ __forceinline__ R pick(bool c, R a, R b) {
    return c ? a : b;
}
template <typename R>
__device__ __forceinline__ R pick16(const R (&A)[16], int r) {
    R t[8], u[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = pick<R>(r & 1, A[2 * i + 1], A[2 * i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = pick<R>(r & 2, t[2 * i + 1], t[2 * i]);
    const R v0 = pick<R>(r & 4, u[1], u[0]), v1 = pick<R>(r & 4, u[3], u[2]);
    return pick<R>(r & 8, v1, v0);
}

}  // namespace

// registers of a group of 16 columns, by component
template <typename S>
struct RowGroup {
    typename S::R x[16], y[S::NC == 2 ? 16 : 1];
};

// Arguments as tridiag_reg_kernel's; both triangles of the block are read.  IN 1:
// element (i, j) at i + j ld; IN 2: a hand-over block, row by row, element (i, j) at
// j + i ld.  The hand-over block written (s_end < n - 1) holds both triangles too.
template <typename S, int RW, int CW, int NG, int MINW, int IN, typename THin>
__global__ __launch_bounds__(64 * RW * CW, MINW) void tridiag_row_kernel(
    const THin* Hin, int64_t h_kstride, int n, int ld, typename ScMem<S>::T* Vout, int ldv,
    int64_t v_kstride, double* __restrict__ dout, double* __restrict__ eout, typename ScMem<S>::T* __restrict__ tauout,
    int64_t de_kstride, int s_end, typename ScMem<S>::T* __restrict__ Bout, int ldb) {
    using R = typename S::R;
    using VT = typename ScMem<S>::T;
    constexpr bool kCx = S::NC == 2;
    constexpr int NROW = 64 * RW, NCOL = 16 * CW * NG;
    constexpr int NX = NROW > NCOL ? NROW : NCOL;
    constexpr int NXR = NX / 64 + (NX % 64 ? 1 : 0);
    constexpr int NW = RW * CW;
    __shared__ S X[2][64 * NXR];      // column s (zero at rows <= s and >= n), by step parity
    __shared__ S YP[CW][64 * NXR];    // the column waves' shares of y
    __shared__ R QP[NW];              // the waves' shares of v^H A v
    __shared__ R XD;                  // A(s, s)
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wv % RW, cw = wv / RW;
    const int i = 64 * rw + lane;
    const int64_t kk = blockIdx.x;
    const THin* H = Hin + kk * h_kstride;
    VT* Vk = Vout + kk * v_kstride;
    double* d = dout + kk * de_kstride;
    double* e = eout + kk * de_kstride;
    VT* tau_o = tauout + kk * de_kstride;
    const int s_stop = s_end < n - 1 ? s_end : n - 1;
    const S zero{}, one = sc_real<S>(R(1));
    for (int t = threadIdx.x; t < 64 * NXR; t += 64 * NW) {
        X[0][t] = X[1][t] = zero;
#pragma unroll
        for (int q = 0; q < CW; ++q) YP[q][t] = zero;
    }
    // rows and columns past n load an in-range element and are masked by a 0 / 1
    // factor (a select would let the compiler turn each load into a branch); one
    // group's loads at a time, as all of them in flight would need registers that
    // the steps do not have
    RowGroup<S> A[NG];
    {
        const THin* Hi = H + (i < n ? i : n - 1);
        const R mi = i < n ? R(1) : R(0);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int j0 = 16 * (CW * g + cw);
            THin h[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) h[r] = Hi[(int64_t)(j0 + r < n ? j0 + r : n - 1) * ld];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const S a = scale(conj_if(sc_load<S>(h[r]), IN == 2), j0 + r < n ? mi : R(0));
                A[g].x[r] = a.x;
                if constexpr (kCx) A[g].y[r] = a.y;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // element (i, s) of the wave that holds column s
    auto column = [&](int s) -> S {
        S x{};
#pragma unroll
        for (int g = 0; g < NG; ++g)
            if (g == (s >> 4) / CW) {  // wave-uniform
                x.x = pick16(A[g].x, s & 15);
                if constexpr (kCx) x.y = pick16(A[g].y, s & 15);
            }
        return x;
    };
    // a group takes part while it has live columns
    auto live = [&](int g, int s) {
        const int j0 = 16 * (CW * g + cw);
        return j0 + 15 > s && j0 < n;
    };
    __syncthreads();

    for (int s = 0; s < s_stop; ++s) {
        S* Xs = X[s & 1];
        if ((s >> 4) % CW == cw) {
            const S x = column(s);
            if (i == s) XD = x.x;
            Xs[i] = sel(i > s, x, zero);
        }
        __syncthreads();
        // ---- reflector, in every wave: tau = (beta - alpha) / beta, sc = 1 / (alpha - beta) ----
        S vb[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) vb[g] = Xs[16 * (CW * g + cw) + l16];
        const S xi = Xs[i];
        const S al = Xs[s + 1];
        R part = 0;
#pragma unroll
        for (int q = 0; q < NXR; ++q) {
            const S t = Xs[lane + 64 * q];
            part = dot_acc(t, sel(lane + 64 * q == s + 1, zero, t), part);
        }
        const R xn2 = wave::sum(part);
        R beta = al.x;
        S tau{}, sc = one;
        if (reflects(xn2, al)) {
            const R nrm = sqrt(dot_acc(al, al, xn2));
            beta = al.x >= R(0) ? -nrm : nrm;
            const R ib = rcp_full(beta);
            tau = scale(al, -ib);
            tau.x = (beta - al.x) * ib;
            const R br = al.x - beta, iden = rcp_full(fma(br, br, imag2(al)));
            sc = scale(conj_if(al, true), iden);
            sc.x = br * iden;
        }
        const S vi = sel(i == s + 1, one, mul(xi, sc));
#pragma unroll
        for (int g = 0; g < NG; ++g) vb[g] = sel(16 * (CW * g + cw) + l16 == s + 1, one, mul(vb[g], sc));
        if (threadIdx.x == 0) {
            d[s] = (double)XD;
            e[s] = (double)beta;
            tau_o[s] = sc_store<S>(tau);
        }
        if (cw == 0 && i > s + 1 && i < n) Vk[i + (int64_t)s * ldv] = sc_store<S>(vi);
        // ---- this wave's share of y = A v ----
        S y{};
        if (64 * rw + 63 > s) {  // wave-uniform: the wave still has live rows
            R ax[4] = {0, 0, 0, 0}, ay[4] = {0, 0, 0, 0};
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (live(g, s)) {
                    rowop::dot16(ax, vb[g].x, A[g].x);
                    if constexpr (kCx) {
                        rowop::dot16(ay, vb[g].y, A[g].x);
                        rowop::dot16(ax, -vb[g].y, A[g].y);
                        rowop::dot16(ay, vb[g].x, A[g].y);
                    }
                }
            y.x = i > s ? (ax[0] + ax[1]) + (ax[2] + ax[3]) : R(0);
            if constexpr (kCx) y.y = i > s ? (ay[0] + ay[1]) + (ay[2] + ay[3]) : R(0);
        }
        YP[cw][i] = y;
        const R qv = wave::sum(dot_acc(vi, y, R(0)));
        if (lane == 0) QP[wv] = qv;
        __syncthreads();
        // ---- A += c1 y^H + c2 v^H ----
        if (64 * rw + 63 > s) {
            R vav = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) vav += QP[w];
            S yi = YP[0][i];
#pragma unroll
            for (int q = 1; q < CW; ++q) yi = add(yi, YP[q][i]);
            const R alpha2 = -dot_acc(tau, tau, R(0)) * vav;  // 2 alpha
            const S c1 = scale(mul(vi, conj_if(tau, true)), R(-1));
            const S c2 = scale(axpy(alpha2, vi, mul(yi, tau)), R(-1));
            S yb[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                yb[g] = YP[0][16 * (CW * g + cw) + l16];
#pragma unroll
                for (int q = 1; q < CW; ++q) yb[g] = add(yb[g], YP[q][16 * (CW * g + cw) + l16]);
            }
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (live(g, s)) {
                    rowop::axpy16(A[g].x, yb[g].x, c1.x);
                    rowop::axpy16(A[g].x, vb[g].x, c2.x);
                    if constexpr (kCx) {
                        rowop::axpy16(A[g].x, yb[g].y, c1.y);
                        rowop::axpy16(A[g].x, vb[g].y, c2.y);
                        rowop::axpy16(A[g].y, yb[g].x, c1.y);
                        rowop::axpy16(A[g].y, yb[g].y, -c1.x);
                        rowop::axpy16(A[g].y, vb[g].x, c2.y);
                        rowop::axpy16(A[g].y, vb[g].y, -c2.x);
                    }
                }
        }
    }
    if (s_stop < n - 1) {
        VT* B = Bout + kk * (int64_t)ldb * ldb;
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int j = 16 * (CW * g + cw) + r;
                if (j >= s_stop && j < n && i >= s_stop && i < n) {
                    S a{};
                    a.x = A[g].x[r];
                    if constexpr (kCx) a.y = -A[g].y[r];  // element (j, i) of the row-by-row block
                    B[(i - s_stop) + (int64_t)(j - s_stop) * ldb] = sc_store<S>(a);
                }
            }
        return;
    }
    // last diagonal element
    const int s = n - 1;
    if ((s >> 4) % CW == cw) {
        const S x = column(s);
        if (i == s) d[s] = (double)x.x;
    }
    if (threadIdx.x == 0) {
        e[s] = 0.0;
        tau_o[s] = sc_store<S>(zero);
    }
}

namespace {
template <typename S, int RW, int CW, int NG, int MINW, int IN, typename THin>
void row_stage(const THin* H, int64_t hk, int n, int ld, int64_t nk, typename ScMem<S>::T* V, int ldv, int64_t vk, double* dd,
               double* de, typename ScMem<S>::T* dtau, int64_t dk, int s_end, typename ScMem<S>::T* B, int ldb,
               hipStream_t s) {
    hipLaunchKernelGGL((tridiag_row_kernel<S, RW, CW, NG, MINW, IN, THin>), dim3((unsigned)nk), dim3(64 * RW * CW), 0, s, H,
                       hk, n, ld, V, ldv, vk, dd, de, dtau, dk, s_end, B, ldb);
}
}  // namespace

}  // namespace uepm
