// tridiag_grid.hpp — register-resident Householder reduction of a Hermitian
// block on a grid of lanes, one workgroup per k-point (gfx950); real, complex
// and quaternion elements (scalars.hpp) in FP32 or FP64.  The chains of
// shrinking grids are in tridiag_reg.hip, tridiag_real.hip and tridiag_quaternion.hip.
//
// Layout.  The lanes form a PR x PC = 32 x 16 (or 16 x 16) grid: lane (r, c) with
// c = tid % 16, r = tid / 16 (a wave holds four r values and all sixteen c).
// Lane (r, c) keeps in VGPRs the lower-triangle elements A(i, j) with
// i = r + 32 l, j = c + 16 m (cyclic in both directions, so every lane keeps
// a share of the shrinking trailing matrix until the end).  Only blocks
// (l, m) that can hold i >= j are stored: 42 complex values per lane at
// dim <= 192.  The blocks of a row block that lie in its diagonal super-block
// (32 x 32) hold both triangles: their elements feed row i of the symmetric product
// only (A v_j), the elements of the other blocks row i and column j (conj(A) v_i).
// A grid whose blocks
// do not all fit its register budget keeps its last NL blocks in LDS instead,
// in lane-private slots (slot-major, so a wave's accesses are consecutive).
//
// Step s (LAPACK xHETD2, lower, restated; H_s = I - tau v v^H, v[s+1] = 1, and
// v = u sc with u = A(s+1:, s) but for u[s+1] = alpha - beta):
//   a. the lanes of column s put A(s+1:, s) in LDS                   | barrier
//   b. every wave forms beta, tau, sc from it (redundantly)
//   c. y = A u: row sums across the 16 lanes of a row group (DPP), column
//      sums across the 4 row groups of a wave (row swaps), one
//      partial per wave in LDS; each lane also sums its share of u^H A u,
//      so w^H u needs no separate dot product                         | barrier
//   d. y = sum of the partials, one row per lane                       | barrier
//   e. w = y ts - (1/2)|ts|^2 (u^H A u) u with ts = sc tau conj(sc);
//      A -= u w^H + w u^H on the live blocks
// (u is the column itself: rows and columns of it are read from LDS where v would be a
// product and a select each.  With that, and the diagonal super-blocks at full weight on
// one side instead of at half weight on both: quaternions 128 -> 96, 3000 k-points, 2.55
// -> 2.26 ms in FP32, 961 in FP64 1.69 -> 1.53; complex64 160 -> 128, 4096, two chunks in
// flight, 2.43 -> 2.35; real 181 -> 128 2.51 -> 2.44.  The three barriers of a step and
// the chains between them bound the small elements, issue the quaternions.)
// Blocks whose columns are all <= s are skipped (one wave-uniform test per
// block column: a stored block's rows are live while its columns are).
// Outputs match the LDS-blocked reduction: d, e (real), tau, reflectors below
// the sub-diagonal of column s of Vout (v[s+1] = 1 implied).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "scalars.hpp"
#include "wave_ops.hpp"

namespace uepm {

namespace {

// Reductions: DPP inside a 16-lane row, VALU row swaps across the rows of a
// wave (wave_ops.hpp; 64-bit values move as two 32-bit halves).
template <typename R>
__device__ __forceinline__ void swap16(R& a, R& b) {
    wave::Words<R> wa(a), wb(b);
#pragma unroll
    for (int i = 0; i < wave::Words<R>::n; ++i) wave::swap16(wa.w[i], wb.w[i]);
    a = wa.value();
    b = wb.value();
}
template <typename R>
__device__ __forceinline__ void swap32(R& a, R& b) {
    wave::Words<R> wa(a), wb(b);
#pragma unroll
    for (int i = 0; i < wave::Words<R>::n; ++i) wave::swap32(wa.w[i], wb.w[i]);
    a = wa.value();
    b = wb.value();
}
// Reduce-scatter of four column partials over the four rows of a wave: returns,
// in lane row q, partial q summed over the four rows (two block columns' (Re, Im)
// in complex arithmetic, four block columns in real, one in quaternion).
template <typename R>
__device__ __forceinline__ R cross_rows4(R p0, R p1, R p2, R p3) {
    swap16(p0, p1);  // rows 0,2: p0 parts; rows 1,3: p1 parts
    p0 += p1;
    swap16(p2, p3);
    p2 += p3;
    swap32(p0, p2);  // lanes 0-31: p0 (p0 | p1), lanes 32-63: p2 (p2 | p3)
    return p0 + p2;
}

// 1/x: hardware reciprocal and Newton steps to full precision
__device__ __forceinline__ float rcp_full(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, r, 1.f), r, r);
}
__device__ __forceinline__ double rcp_full(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// Stored blocks of the cyclic lower triangle.  With PR = Q PC and LC = Q LR
// (Q = 1 or 2) row block l stores block columns 0..Q l + Q - 1, so the
// offsets have closed forms: everything below folds to constants once the
// loops over l and m are unrolled, which keeps the slot array in registers.
template <int PR, int PC, int LR, int LC>
struct RegLayout {
    static constexpr int Q = PR / PC;
    static_assert((Q == 1 || Q == 2) && PR == Q * PC && LC == Q * LR, "closed forms below assume square coverage");
    static constexpr int mmax(int l) { return Q * l + Q - 1; }  // = min((PR l + PR - 1) / PC, LC - 1)
    static constexpr int base(int l) { return Q * l * (l + 1) / 2; }  // sum of mmax(q) + 1 over q < l
    static constexpr int count() { return base(LR); }
    static constexpr int idx(int l, int m) { return base(l) + m; }
    // first row block l with block (l, m) stored: the smallest l with mmax(l) >= m
    static constexpr int lmin(int m) { return m / Q; }
    // blocks (l, Q l) .. (l, Q l + Q - 1) lie in the diagonal PR x PR super-block
    // of rows PR l .. PR l + PR - 1: i and j there are in the same super-block, and
    // so are the mirror pair (j, i)
    static constexpr bool straddles(int l, int m) { return m >= Q * l; }
};

}  // namespace

// Stage arguments: steps s < s_end run here (s_end >= n - 1: the whole
// reduction); when s_end < n - 1 the updated trailing block A[s_end:, s_end:]
// (lower triangle, full diagonal) goes to Bout row by row (element (i, j) at
// j + i ldb, b_kstride per k; FULL: and its conjugate above the diagonal) for a
// smaller grid to continue.  IN says how
// the lower triangle of the input is read: 0, column-major (element (i, j) at
// i + j ld); 1, as the conjugate of the upper triangle of a full Hermitian
// matrix (element (j, i) at j + i ld); 2, row by row as a hand-over block.  Input (leading
// dimension ld), reflectors (ldv) and d, e, tau of k-point kk start at
// kk * h_kstride, kk * v_kstride and kk * de_kstride.  The reflectors may go over the
// input (the FP64 form) and so may the hand-over block (the complex64 chain), so none
// of the three pointers is __restrict__: the input is read before the first step, which
// writes the first reflector; the block is written after the last.
template <int PR, int PC, int LR, int LC, int MINWG, typename S, typename THin, bool LOW = false, int NL = 0, int IN = 0,
          bool FULL = false>
__global__ __launch_bounds__(PR* PC, MINWG) void tridiag_reg_kernel(const THin* Hin, int64_t h_kstride,
                                                                    int n, int ld,
                                                                    typename ScMem<S>::T* Vout, int ldv,
                                                                    int64_t v_kstride, double* __restrict__ dout,
                                                                    double* __restrict__ eout,
                                                                    typename ScMem<S>::T* __restrict__ tauout,
                                                                    int64_t de_kstride, int s_end,
                                                                    typename ScMem<S>::T* Bout, int ldb, int64_t b_kstride) {
    using R = typename S::R;
    using VT = typename ScMem<S>::T;
    constexpr int NC = S::NC;
    constexpr int GC = 4 / NC;  // block columns per reduce-scatter of the column sums
    constexpr int BS = PR * PC;
    constexpr int NW = BS / 64;
    using Lay = RegLayout<PR, PC, LR, LC>;
    constexpr int NS = Lay::count();
    constexpr int NX = PR * LR;  // rows covered by the grid
    constexpr int NXR = (NX + 63) / 64;
    constexpr int NXC = PC * ((LC + GC - 1) / GC * GC);  // columns of the column sums, whole groups
    constexpr int NYT = (NX + BS - 1) / BS;              // entries of y per lane
    static_assert(PC == 16 && BS % 64 == 0, "row groups are the 16-lane DPP rows of a wave");
    static_assert(PC * LC == NX, "square coverage");

    // column s: zero at rows <= s and >= n; two buffers by step parity, since the
    // LOW variant still reads the column of step s in its update phase while a
    // wave ahead may write the column of step s + 1 (no barrier in between)
    __shared__ S Xbuf[2][NX];
    __shared__ S XC[NX];      // column s as it is (rows of its diagonal super-block and below)
    __shared__ S RP[NX];      // row sums of the symmetric product
    __shared__ S CP[NW][NXC];  // column sums, one row per wave
    __shared__ S Y[NX];       // y = A v, zero at rows <= s and >= n
    __shared__ R Q[NW];    // per-wave partial v^H A v
    // the last NL stored blocks of every lane live in LDS (lane-private slots,
    // slot-major so that a wave's accesses are consecutive), the others in VGPRs
    static_assert(NL >= 0 && NL < NS, "LDS slots");
    constexpr int NR = NS - NL;
    __shared__ S AL[NL > 0 ? NL : 1][NL > 0 ? BS : 1];

    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int c = tid % PC, r = tid / PC;
    const int64_t kk = blockIdx.x;
    const THin* H = Hin + kk * h_kstride;
    VT* Vk = Vout + kk * v_kstride;
    double* d = dout + kk * de_kstride;
    double* e = eout + kk * de_kstride;
    VT* tau_o = tauout + kk * de_kstride;
    const int s_stop = s_end < n - 1 ? s_end : n - 1;

    // ---- load ----
    S A[NR];
    // slot i of this lane (i is a compile-time constant wherever these are used)
    auto aget = [&](int i) -> S {
        if constexpr (NL > 0)
            if (i >= NR) return AL[i - NR][tid];
        return A[i];
    };
    auto aset = [&](int i, S v) {
        if constexpr (NL > 0)
            if (i >= NR) {
                AL[i - NR][tid] = v;
                return;
            }
        A[i] = v;
    };
#pragma unroll
    for (int l = 0; l < LR; ++l) {
#pragma unroll
        for (int m = 0; m <= Lay::mmax(l); ++m) {
            const int i = r + PR * l, j = c + PC * m;
            S a{};
            if (i < n && j < n && (i >= j || Lay::straddles(l, m))) {
                // the lower element (p, q), p >= q: (i, j), or (j, i) conjugated above the
                // diagonal.  A wave's 16 columns j are consecutive: IN 1 and 2 read the
                // lower elements as contiguous runs (row i of the stored triangle)
                const bool up = i < j;
                const int p = up ? j : i, q = up ? i : j;
                const THin h = H[IN == 0 ? p + (int64_t)q * ld : q + (int64_t)p * ld];
                a = conj_if(sc_load<S>(h), (IN == 1) != up);
            }
            aset(Lay::idx(l, m), a);
        }
    }
    const S one = sc_real<S>(R(1)), zero{};

    for (int s = 0; s < s_stop; ++s) {
        S* X = Xbuf[s & 1];
        const int cs = s % PC, ms = s / PC;
        const int l0 = (s + 1) / PR, m0 = (s + 1) / PC;  // first live row / column blocks
        // ---- a. column s to LDS (every row of the grid) ----
        const bool own = c == cs;
#pragma unroll
        for (int m = 0; m < LC; ++m) {
            if (m == ms) {  // wave-uniform
                if (own) {
#pragma unroll
                    for (int l = 0; l < LR; ++l) {
                        const int i = r + PR * l;
                        if (m <= Lay::mmax(l)) {
                            const S a = aget(Lay::idx(l, m));
                            X[i] = sel(i > s, a, zero);
                            XC[i] = a;
                        } else {
                            X[i] = zero;  // block above the diagonal: rows < s
                        }
                    }
                }
            }
        }
        __syncthreads();
        // ---- b. reflector, redundantly in every wave ----
        R part = 0;
#pragma unroll
        for (int q = 0; q < NXR; ++q) {
            const int i = s + 2 + lane + 64 * q;
            const S a = X[i < NX ? i : NX - 1];
            const R t = norm2(a);
            part += i < NX ? t : R(0);
        }
        const R xn2 = wave::sum(part);
        // tau = (beta - alpha) / beta, sc = 1 / (alpha - beta); v = u sc with u the column
        // and alpha - beta in front, which is what the rest of the step works with:
        // tau v v^H = u ts u^H, ts = sc tau conj(sc), and ts takes tau's place throughout.
        const S al = XC[s + 1];
        R beta = al.x;
        S tau{}, sc = one, ts{};
        R iden = 0;  // |sc|^2
        if (reflects(xn2, al)) {
            const R nrm = sqrt(dot_acc(al, al, xn2));
            beta = al.x >= R(0) ? -nrm : nrm;
            const R ib = rcp_full(beta);
            tau = scale(al, -ib);
            tau.x = (beta - al.x) * ib;
            const R br = al.x - beta;
            iden = rcp_full(fma(br, br, imag2(al)));
            sc = scale(conj_if(al, true), iden);
            sc.x = br * iden;
            ts = mul(mul(sc, tau), conj_if(sc, true));
        }
        if (tid == 0) {
            d[s] = (double)XC[s].x;
            e[s] = (double)beta;
            tau_o[s] = sc_store<S>(tau);
        }
        // every wave puts u's first element in place, for itself: the others write the
        // same, and read X[s + 1] only after their own write
        if (lane == 0) {
            S u0 = al;
            u0.x = al.x - beta;
            X[s + 1] = u0;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int q = 0; q < NYT; ++q) {
            const int i = s + 2 + tid + q * BS;
            if (i < n) Vk[i + (int64_t)s * ldv] = sc_store<S>(mul(X[i], sc));
        }
        // u at this lane's rows and columns (X is zero outside s+1..n-1; loads
        // unconditional so they issue together)
        // LOW (fewer registers, for two workgroups per CU): the column values of u and
        // w are read from LDS where they are used instead of being kept, and each
        // pair of block columns is reduced as soon as its partial sums are complete
        // (the same operations in the same order)
        auto vcol = [&](int m) -> S { return X[c + PC * m]; };
        S vr[LR], vc[LOW ? 1 : LC];
#pragma unroll
        for (int l = 0; l < LR; ++l) vr[l] = X[r + PR * l];
        if constexpr (!LOW) {
#pragma unroll
            for (int m = 0; m < LC; ++m) vc[m] = vcol(m);
        }
        // ---- c. y = A u on the live blocks; local share of u^H A u ----
        S rp[LR], cp[LOW ? GC : NXC / PC];
#pragma unroll
        for (int l = 0; l < LR; ++l) rp[l] = zero;
#pragma unroll
        for (int m = 0; m < (LOW ? GC : NXC / PC); ++m) cp[m] = zero;
        R qv = 0;
        const int q4 = lane >> 4;
        R* cpw = &CP[wv][0].x;
        // column sums of GC block columns from m on: lane row q holds component
        // q % NC of block column m + q / NC
        auto col_sums = [&](int m, const S* p) {
            R t;
            if constexpr (NC == 1) t = cross_rows4(p[0].x, p[1].x, p[2].x, p[3].x);
            else if constexpr (NC == 2) t = cross_rows4(p[0].x, p[0].y, p[1].x, p[1].y);
            else t = cross_rows4(p[0].x, p[0].y, p[0].z, p[0].w);
            cpw[NC * (c + PC * (m + q4 / NC)) + q4 % NC] = t;
        };
#pragma unroll
        for (int m = LC - 1; m >= 0; --m) {
            const int mc = LOW ? m % GC : m;  // cp slot of block column m
            if (m >= m0) {  // a stored block is live while its block column is
                const S vcm = LOW ? vcol(m) : vc[LOW ? 0 : m];
#pragma unroll
                for (int l = Lay::lmin(m); l < LR; ++l) {
                    const S a = aget(Lay::idx(l, m));
                    fma_ab(rp[l], a, vcm);
                    if (!Lay::straddles(l, m)) fma_cab(cp[mc], a, vr[l]);
                }
            }
            // row block m / Q: its diagonal super-block, now complete, counts half in u^H A u
            if (m % Lay::Q == 0 && m + Lay::Q - 1 >= m0)
                qv = dot_acc(vr[Lay::lmin(m)], scale(rp[Lay::lmin(m)], R(-0.5)), qv);
            if constexpr (LOW) {
                if (m % GC == 0) {
                    if (m + GC - 1 >= m0) col_sums(m, cp);
#pragma unroll
                    for (int u = 0; u < GC; ++u) cp[u] = zero;
                }
            }
        }
        // half of u^H A u: the sum of conj(u_i) A_ij u_j over the blocks below the diagonal
        // super-blocks and half of it over those
#pragma unroll
        for (int l = 0; l < LR; ++l)
            if (l >= l0) qv = dot_acc(vr[l], rp[l], qv);
#pragma unroll
        for (int l = 0; l < LR; ++l) {
            if (l >= l0) {
                S t = rp[l];
                t.x = wave::row_sum16(t.x);
                if constexpr (NC >= 2) t.y = wave::row_sum16(t.y);
                if constexpr (NC == 4) {
                    t.z = wave::row_sum16(t.z);
                    t.w = wave::row_sum16(t.w);
                }
                if (c == 0) RP[r + PR * l] = t;
            }
        }
        if constexpr (!LOW) {
#pragma unroll
            for (int m = 0; m < LC; m += GC)
                if (m + GC - 1 >= m0) col_sums(m, cp + m);
        }
        qv = wave::sum(qv);
        if (lane == 0) Q[wv] = qv;
        __syncthreads();
        // ---- d. y = row sums + column sums of the waves, one row per lane; then
        // w = tau y + alpha v, alpha = -(tau/2) p^H v = -(1/2)|tau|^2 v^H A v, and v
        // itself, published for the update: w over y in Y, v over the row sums in RP
        // (the next writes of both come after a barrier that every wave passes only
        // once it has finished this step) ----
#pragma unroll
        for (int q = 0; q < NYT; ++q) {
            const int i = tid + q * BS;
            if (i >= NX) break;
            S y = zero;
            if (i > s && i < n) {
                y = RP[i];
#pragma unroll
                for (int w = 0; w < NW; ++w) y = add(y, CP[w][i]);
            }
            R vav = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) vav += Q[w];
            const R alpha = -dot_acc(tau, tau, R(0)) * (iden * (iden * vav));  // -(1/2)|ts|^2 u^H A u
            Y[i] = axpy(alpha, X[i], mul(y, ts));
        }
        __syncthreads();
        // ---- e. rank-2 update A -= u w^H + w u^H ----
        S wr[LR];
#pragma unroll
        for (int l = 0; l < LR; ++l) wr[l] = Y[r + PR * l];
#pragma unroll
        for (int m = LC - 1; m >= 0; --m) {
            if (m >= m0) {
                const S vcm = LOW ? vcol(m) : vc[LOW ? 0 : m];
                const S wcm = Y[c + PC * m];
#pragma unroll
                for (int l = Lay::lmin(m); l < LR; ++l) {
                    // a -= u_i conj(w_j) + w_i conj(u_j)
                    S a = aget(Lay::idx(l, m));
                    fms_abc(a, vr[l], wcm);
                    fms_abc(a, wr[l], vcm);
                    aset(Lay::idx(l, m), a);
                }
            }
        }
    }
    if (s_stop < n - 1) {
        // hand the trailing block A[s_stop:, s_stop:] over
        VT* B = Bout + kk * b_kstride;
#pragma unroll
        for (int l = 0; l < LR; ++l)
#pragma unroll
            for (int m = 0; m <= Lay::mmax(l); ++m) {
                const int i = r + PR * l, j = c + PC * m;
                if (i < n && j >= s_stop && i >= j) {
                    const S a = aget(Lay::idx(l, m));
                    B[(j - s_stop) + (int64_t)(i - s_stop) * ldb] = sc_store<S>(a);
                    if constexpr (FULL) B[(i - s_stop) + (int64_t)(j - s_stop) * ldb] = sc_store<S>(conj_if(a, true));
                }
            }
        return;
    }
    // last diagonal element
    {
        const int s = n - 1;
        const int cs = s % PC, ms = s / PC;
#pragma unroll
        for (int m = 0; m < LC; ++m)
            if (m == ms)
#pragma unroll
                for (int l = 0; l < LR; ++l)
                    if (m <= Lay::mmax(l) && c == cs && r + PR * l == s) d[s] = (double)aget(Lay::idx(l, m)).x;
        if (tid == 0) {
            e[s] = 0.0;
            tau_o[s] = sc_store<S>(zero);
        }
    }
}

namespace {
template <typename S, int PR, int LR, int MINWG, int IN, typename THin, bool LOW = false, int NL = 0, bool FULL = false>
void reg_stage(const THin* H, int64_t h_kstride, int n, int ld, int64_t nk, typename ScMem<S>::T* V, int ldv,
               int64_t v_kstride, double* dd, double* de, typename ScMem<S>::T* dtau, int64_t de_kstride, int s_end,
               typename ScMem<S>::T* B, int ldb, hipStream_t s, int64_t b_kstride = 0) {
    hipLaunchKernelGGL((tridiag_reg_kernel<PR, 16, LR, LR * PR / 16, MINWG, S, THin, LOW, NL, IN, FULL>),
                       dim3((unsigned)nk), dim3(PR * 16), 0, s, H, h_kstride, n, ld, V, ldv, v_kstride, dd, de, dtau,
                       de_kstride, s_end, B, ldb, b_kstride ? b_kstride : (int64_t)ldb * ldb);
}
}  // namespace

}  // namespace uepm
