// tridiag_row.hpp — Householder reduction of a real symmetric block, one matrix
// row per lane (gfx950).
//
// Layout.  A workgroup of RW x CW waves takes one k-point.  Lane l of a wave
// (rw, cw) keeps row i = 64 rw + l of the block in VGPRs (both triangles), the
// columns of every CW-th group of 16: group q = CW g + cw, register A[g][r] =
// A(i, 16 q + r).  Then
//
//   y_i = sum_j A(i, j) v_j           is a sum over the lane's own registers,
//   A(i, j) -= c1_i y_j + c2_i v_j    is the rank-2 update (below),
//
// and neither needs a cross-lane reduction.  v_j and y_j reach the lanes of a
// wave as DPP operands: every 16-lane row holds the 16 values of a group (one
// LDS read per lane and group), and v_fmac_*_dpp row_newbcast:r multiplies the
// register of column 16 q + r by the value in lane r of each row, in the one
// instruction of a plain multiply-add.
//
// Step s: the owner of column s publishes it in LDS | barrier | beta, tau, v in
// every wave; y = A v; each wave's share of y and of v^T A v to LDS | barrier |
// A -= v w^T + w v^T with w = tau y + alpha v, alpha = -(1/2) tau^2 v^T A v,
// written as A(i, j) += c1_i y_j + c2_i v_j, c1 = -tau v_i, c2 = -(tau y_i +
// 2 alpha v_i), so that w is never formed.  v and y are zero at rows <= s: dead
// rows and columns inside a live group take no part.
//
// Against the cyclic lower-triangle grid this does 1.5 times the multiply-adds
// (both triangles are updated) but none of the reductions, which were two thirds
// of a real step's instructions.
#pragma once

#include "row_ops.hpp"
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

// Arguments as tridiag_reg_kernel's; the block is symmetric and both triangles
// of it are read (element (i, j) at i + j ld), and the hand-over block written
// (s_end < n - 1) holds both triangles likewise.
template <typename R, int RW, int CW, int NG, int MINW, typename THin>
__global__ __launch_bounds__(64 * RW * CW, MINW) void tridiag_row_kernel(const THin* __restrict__ Hin,
                                                                         int64_t h_kstride, int n, int ld,
                                                                         R* __restrict__ Vout, int ldv,
                                                                         int64_t v_kstride, double* __restrict__ dout,
                                                                         double* __restrict__ eout,
                                                                         R* __restrict__ tauout, int64_t de_kstride,
                                                                         int s_end, R* __restrict__ Bout, int ldb) {
    constexpr int NROW = 64 * RW, NCOL = 16 * CW * NG;
    constexpr int NX = NROW > NCOL ? NROW : NCOL;
    constexpr int NXR = NX / 64 + (NX % 64 ? 1 : 0);
    constexpr int NW = RW * CW;
    __shared__ R X[2][64 * NXR];      // column s (zero at rows <= s and >= n), by step parity
    __shared__ R YP[CW][64 * NXR];    // the column waves' shares of y
    __shared__ R QP[NW];              // the waves' shares of v^T A v
    __shared__ R XD;                  // A(s, s)
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wv % RW, cw = wv / RW;
    const int i = 64 * rw + lane;
    const int64_t kk = blockIdx.x;
    const THin* H = Hin + kk * h_kstride;
    R* Vk = Vout + kk * v_kstride;
    double* d = dout + kk * de_kstride;
    double* e = eout + kk * de_kstride;
    R* tau_o = tauout + kk * de_kstride;
    const int s_stop = s_end < n - 1 ? s_end : n - 1;
    for (int t = threadIdx.x; t < 64 * NXR; t += 64 * NW) {
        X[0][t] = X[1][t] = R(0);
#pragma unroll
        for (int q = 0; q < CW; ++q) YP[q][t] = R(0);
    }
    // rows and columns past n load an in-range element and are masked by a 0 / 1
    // factor (a select would let the compiler turn each load into a branch); one
    // group's loads at a time, as all of them in flight would need registers that
    // the steps do not have
    R A[NG][16];
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
            for (int r = 0; r < 16; ++r) A[g][r] = (R)h[r] * (j0 + r < n ? mi : R(0));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();

    for (int s = 0; s < s_stop; ++s) {
        R* Xs = X[s & 1];
        const int gs = s >> 4;
        if (gs % CW == cw) {
            R x = 0;
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (g == gs / CW) x = pick16(A[g], s & 15);  // wave-uniform
            if (i == s) XD = x;
            Xs[i] = i > s ? x : R(0);
        }
        __syncthreads();
        // ---- reflector, in every wave ----
        R vb[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) vb[g] = Xs[16 * (CW * g + cw) + l16];
        const R xi = Xs[i];
        const R al = Xs[s + 1];
        R part = 0;
#pragma unroll
        for (int q = 0; q < NXR; ++q) {
            const R t = Xs[lane + 64 * q];
            part = fma(t, lane + 64 * q == s + 1 ? R(0) : t, part);
        }
        const R xn2 = wave::sum(part);
        R beta = al, tau = 0, sc = 1;
        if (xn2 != R(0)) {
            const R nrm = sqrt(fma(al, al, xn2));
            beta = al >= R(0) ? -nrm : nrm;
            tau = (beta - al) * rcp_full(beta);
            const R br = al - beta;
            sc = br * rcp_full(br * br);
        }
        const R vi = i == s + 1 ? R(1) : xi * sc;
#pragma unroll
        for (int g = 0; g < NG; ++g) vb[g] = 16 * (CW * g + cw) + l16 == s + 1 ? R(1) : vb[g] * sc;
        if (threadIdx.x == 0) {
            d[s] = (double)XD;
            e[s] = (double)beta;
            tau_o[s] = tau;
        }
        if (cw == 0 && i > s + 1 && i < n) Vk[i + (int64_t)s * ldv] = vi;
        // ---- this wave's share of y = A v ----
        R y = 0;
        if (64 * rw + 63 > s) {  // wave-uniform: the wave still has live rows
            R acc[4] = {0, 0, 0, 0};
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (16 * (CW * g + cw) + 15 > s) rowop::dot16(acc, vb[g], A[g]);
            y = i > s ? (acc[0] + acc[1]) + (acc[2] + acc[3]) : R(0);
        }
        YP[cw][i] = y;
        const R qv = wave::sum(vi * y);
        if (lane == 0) QP[wv] = qv;
        __syncthreads();
        // ---- A += c1 y^T + c2 v^T ----
        if (64 * rw + 63 > s) {
            R vav = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) vav += QP[w];
            R yi = YP[0][i];
#pragma unroll
            for (int q = 1; q < CW; ++q) yi += YP[q][i];
            const R alpha = -(tau * tau) * vav;  // 2 alpha
            const R c1 = -tau * vi, c2 = -fma(alpha, vi, tau * yi);
            R yb[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                yb[g] = YP[0][16 * (CW * g + cw) + l16];
#pragma unroll
                for (int q = 1; q < CW; ++q) yb[g] += YP[q][16 * (CW * g + cw) + l16];
            }
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (16 * (CW * g + cw) + 15 > s) {
                    rowop::axpy16(A[g], yb[g], c1);
                    rowop::axpy16(A[g], vb[g], c2);
                }
        }
    }
    if (s_stop < n - 1) {
        R* B = Bout + kk * (int64_t)ldb * ldb;
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int j = 16 * (CW * g + cw) + r;
                if (j >= s_stop && j < n && i >= s_stop && i < n) B[(i - s_stop) + (int64_t)(j - s_stop) * ldb] = A[g][r];
            }
        return;
    }
    // last diagonal element
    const int s = n - 1, gs = s >> 4;
    if (gs % CW == cw) {
        R x = 0;
#pragma unroll
        for (int g = 0; g < NG; ++g)
            if (g == gs / CW) x = pick16(A[g], s & 15);
        if (i == s) d[s] = (double)x;
    }
    if (threadIdx.x == 0) {
        e[s] = 0.0;
        tau_o[s] = R(0);
    }
}

}  // namespace uepm
