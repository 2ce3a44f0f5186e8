// tridiag_strip.hpp — leading steps of a Householder reduction whose matrix is
// larger than the register grids (tridiag_grid.hpp) hold: the trailing block lives
// in the grid's registers and LDS, the leading columns (the strip) in memory, and
// the strip is used up by the steps run here.  One workgroup per k-point, complex64.
#pragma once
#include <type_traits>

#include "tridiag_grid.hpp"

namespace uepm {

namespace {
// f(constant B), .. f(constant E - 1)
template <int B, int E, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        unrolled<B + 1, E>(f);
    }
}
// First slot of block column m of the strip (its row blocks are m / 2 .. LR - 1).
__host__ __device__ constexpr int strip_base(int LR, int m) { return m * LR - (m / 2) * (m / 2 - 1) - (m & 1) * (m / 2); }

// Order in which a step visits the strip: pairs of block columns from the last to the
// first live one, row blocks from the diagonal's on; unit q is two slots.
template <int LR, int MG>
struct StripOrder {
    static constexpr int first(int p) { return p >= MG / 2 - 1 ? 0 : first(p + 1) + LR - (p + 1); }  // of pair p
    static constexpr int count() { return first(-1); }
    static constexpr int pair(int q) { return q >= first(0) ? 0 : q >= first(1) ? 1 : 2; }
    static constexpr int row(int q) { return pair(q) + q - first(pair(q)); }
    template <int q>
    static constexpr int slot0 = strip_base(LR, 2 * pair(q)) + row(q) - pair(q);
    template <int q>
    static constexpr int slot1 = strip_base(LR, 2 * pair(q) + 1) + row(q) - pair(q);
    static_assert(MG == 6, "pair()");
};
}  // namespace

// The grid covers NX = 32 LR rows and columns, lane (r, c) of 32 x 16 keeping blocks
// (l, m) of the lower triangle as in tridiag_grid.hpp, with half weight in the
// diagonal super-blocks; the matrix sits at its END, rows and columns NX - n .. NX - 1,
// so the trailing grid is always full and it is the strip that is short.  Block
// columns m < MG are the strip: lane-private slots in memory (slot-major, one run of
// 4 KB an access of the workgroup).  A step reads and writes them once, in its product:
// the rank-2 update of the step before is applied on the way (to the column that the
// next reflector needs, by itself).
// Steps NX - n .. 16 MG - 1 run here (m < MG columns are dead at their end); the
// updated trailing block of NX - 16 MG then goes to Bout row by row.
//
// The blocked reduction streams the columns that its LDS cannot hold (0.44 MB of
// the 0.53 at dim 362, FP32) for every step: 5 TB/s over the chip, so memory bounds
// it.  Here the first step moves 0.5 MB, the last a few KB, and every other element
// stays in registers or LDS: 74 steps at dim 362, 700 k-points, in 4.0 ms against the
// 10.8 of 80 blocked ones.  What is left is issue at two waves a SIMD (2.7 us of a step's
// 15 the update, 5 the trailing product) and the strip's latency (4.5, six units of
// 8 KB in flight; 4 and 8 units measure the same).
template <int LR, int MG, int NL, int IN, typename THin>
__global__ __launch_bounds__(512, 2) void tridiag_strip_kernel(const THin* Hin, int64_t h_kstride, int n, int ld,
                                                               float2* Vout, int ldv, int64_t v_kstride,
                                                               double* __restrict__ dout, double* __restrict__ eout,
                                                               float2* __restrict__ tauout, int64_t de_kstride,
                                                               float2* __restrict__ Bout, int64_t b_kstride,
                                                               float2* __restrict__ Sout, int64_t s_kstride) {
    using S = c2<float>;
    constexpr int PR = 32, PC = 16, BS = 512, NW = BS / 64;
    constexpr int LC = 2 * LR, NX = PR * LR, NXR = NX / 64;
    static_assert(MG % 2 == 0 && NX % 64 == 0 && NX <= BS, "whole super-blocks in the strip; a row a lane");
    constexpr int LT = LR - MG / 2, MT = LC - MG, NT = PR * LT;  // trailing grid: LT x MT blocks, NT rows
    using Lay = RegLayout<PR, PC, LT, MT>;
    using Or = StripOrder<LR, MG>;
    constexpr int Depth = 6;  // units of the strip in flight
    constexpr int NS = Lay::count(), NR = NS - NL;
    __shared__ S X[NX];        // the step's column: zero at rows <= s
    __shared__ float XD;       // its diagonal element
    __shared__ S XC[NX + 1];   // the next step's column before this step's update
    __shared__ S RP[NX];       // row sums
    __shared__ S CP[NW][NX];   // column sums of the waves
    __shared__ S V[NX], Y[NX]; // v and w of the step, read by the next one's strip pass too
    __shared__ float Q[NW];
    __shared__ S AL[NL][BS];

    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, q4 = lane >> 4;
    const int c = tid % PC, r = tid / PC;
    const int sh = NX - n;
    const int64_t kk = blockIdx.x;
    const THin* H = Hin + kk * h_kstride;
    float2* Vk = Vout + kk * v_kstride;
    double* d = dout + kk * de_kstride;
    double* e = eout + kk * de_kstride;
    float2* tau_o = tauout + kk * de_kstride;
    float2* G = Sout + kk * s_kstride;  // wave-uniform; strip slot i of this lane at slot(i)
    int g0 = 0;  // always 0, see the loop
    auto slot = [&](int i) -> float2& { return (G + g0 + i * BS)[(unsigned)tid]; };
    S A[NR];
    auto aget = [&](int i) -> S {
        if (i >= NR) return AL[i - NR][tid];
        return A[i];
    };
    auto aset = [&](int i, S v) {
        if (i >= NR) AL[i - NR][tid] = v;
        else A[i] = v;
    };
    // element (i, j) of the grid as stored: rows and columns in front of the matrix are zero
    auto element = [&](int l, int m) -> S {
        const int i = r + PR * l, j = c + PC * m;
        const bool half = l == m / 2, up = i < j;
        const int p = max((up ? j : i) - sh, 0), q = max((up ? i : j) - sh, 0);
        const THin h = H[IN == 0 ? p + (int64_t)q * ld : q + (int64_t)p * ld];
        const S a = scale(conj_if(sc_load<S>(h), (IN == 1) != up), half ? 0.5f : 1.f);
        return sel(i >= sh && j >= sh, a, S{});
    };
    const S one = sc_real<S>(1.f), zero{};
#pragma unroll
    for (int l = 0; l < LT; ++l)
#pragma unroll
        for (int m = 0; m <= Lay::mmax(l); ++m) aset(Lay::idx(l, m), element(l + MG / 2, m + MG));
    // block (l, m) of block column m, before the last step's update: column s to XC
    auto keep_column = [&](int s, int l, int m, S a) {  // (the other lanes: nowhere)
        XC[c == s % PC ? r + PR * l : NX] = scale(a, l == m / 2 ? 2.f : 1.f);
    };
#pragma unroll
    for (int m = 0; m < MG; ++m)
        if (m / 2 >= sh / PR) {  // whole pairs
#pragma unroll
            for (int l = m / 2; l < LR; ++l) {
                const S a = element(l, m);
                slot(strip_base(LR, m) + l - m / 2) = sc_store<S>(a);
                if (m == sh / PC) keep_column(sh, l, m, a);
            }
        }
    if (tid < NX) V[tid] = Y[tid] = zero;
    // XC to X, with the last step's update (v and w are zero at first)
    auto publish = [&](int s) {
        if (tid < NX) {
            const int i = tid;
            S a = XC[i];
            fms_abc(a, V[i], Y[s]);
            fms_abc(a, Y[i], V[s]);
            X[i] = sel(i > s, a, zero);
            if (i == s) XD = a.x;
        }
    };
    __syncthreads();
    publish(sh);
    __syncthreads();

    for (int s = sh; s < PC * MG; ++s) {
        const int m0 = (s + 1) / PC;  // first live block column
        asm volatile("" : "+s"(g0));  // the slots' addresses are formed where they are used, not kept
        float2 g[Depth][2];
        auto unit_load = [&](auto qc) {
            constexpr int q = decltype(qc)::value, s0 = Or::template slot0<q>, s1 = Or::template slot1<q>;
            g[q % Depth][0] = slot(s0);
            g[q % Depth][1] = slot(s1);
        };
        unrolled<0, Depth>(unit_load);
        // ---- reflector, redundantly in every wave ----
        float part = 0.f;
#pragma unroll
        for (int q = 0; q < NXR; ++q) {
            const int i = s + 2 + lane + 64 * q;
            const S a = X[i < NX ? i : NX - 1];
            const float t = norm2(a);
            part += i < NX ? t : 0.f;
        }
        const float xn2 = wave::sum(part);
        const S al = X[s + 1];
        float beta = al.x;
        S tau{}, sc = one;
        if (reflects(xn2, al)) {
            const float nrm = sqrt(dot_acc(al, al, xn2));
            beta = al.x >= 0.f ? -nrm : nrm;
            const float ib = rcp_full(beta);
            tau = scale(al, -ib);
            tau.x = (beta - al.x) * ib;
            const float br = al.x - beta, iden = rcp_full(fma(br, br, imag2(al)));
            sc = scale(conj_if(al, true), iden);
            sc.x = br * iden;
        }
        if (tid == 0) {
            d[s - sh] = (double)XD;
            e[s - sh] = (double)beta;
            tau_o[s - sh] = sc_store<S>(tau);
        }
        {
            const int i = s + 2 + tid;
            if (i < NX) Vk[(i - sh) + (int64_t)(s - sh) * ldv] = sc_store<S>(mul(X[i], sc));
        }
        auto vcol = [&](int m) -> S {
            const int j = c + PC * m;
            return sel(j == s + 1, one, mul(X[j], sc));
        };
        auto vrow = [&](int l) -> S {
            const int i = r + PR * l;
            return sel(i == s + 1, one, mul(X[i], sc));
        };
        // ---- y = A v ----
        S rp[LR];
#pragma unroll
        for (int l = 0; l < LR; ++l) rp[l] = zero;
        float qv = 0.f;  // sum over stored elements of conj(v_i) A_ij v_j
        float* cpw = &CP[wv][0].x;
        // column sums of block columns m, m + 1: lane row q holds component q % 2 of m + q / 2
        auto col_sums = [&](int m, S p0, S p1) {
            cpw[2 * (c + PC * (m + q4 / 2)) + q4 % 2] = cross_rows4(p0.x, p0.y, p1.x, p1.y);
        };
        unrolled<0, MG / 2>([&](auto pc) {
            constexpr int p = MG / 2 - 1 - decltype(pc)::value;
            if (p < m0 / 2) return;  // wave-uniform
            const S vc0 = vcol(2 * p), vp0 = V[c + PC * 2 * p], wp0 = Y[c + PC * 2 * p];
            const S vc1 = vcol(2 * p + 1), vp1 = V[c + PC * (2 * p + 1)], wp1 = Y[c + PC * (2 * p + 1)];
            S cp0 = zero, cp1 = zero;
            int ro = r;
            asm volatile("" : "+v"(ro));  // a row's v, v' and w': from LDS for every pair, not kept
            unrolled<p, LR>([&](auto lc) {
                constexpr int l = decltype(lc)::value, q = Or::first(p) + l - p, qn = q + Depth;
                constexpr float f = l == p ? 0.5f : 1.f;
                const int i = ro + PR * l;
                const S vi = sel(i == s + 1, one, mul(X[i], sc)), vpi = scale(V[i], f), wpi = scale(Y[i], f);
                S a0 = sc_load<S>(g[q % Depth][0]), a1 = sc_load<S>(g[q % Depth][1]);
                fms_abc(a0, vpi, wp0);
                fms_abc(a1, vpi, wp1);
                fms_abc(a0, wpi, vp0);
                fms_abc(a1, wpi, vp1);
                constexpr int s0 = Or::template slot0<q>, s1 = Or::template slot1<q>;
                if constexpr (qn < Or::count()) {
                    constexpr int n0 = Or::template slot0<qn>, n1 = Or::template slot1<qn>, pn = Or::pair(qn);
                    // of the next pair: not when that is dead (this unit again, unused)
                    g[q % Depth][0] = slot(pn == p || pn >= m0 / 2 ? n0 : s0);
                    g[q % Depth][1] = slot(pn == p || pn >= m0 / 2 ? n1 : s1);
                }
                slot(s0) = sc_store<S>(a0);
                slot(s1) = sc_store<S>(a1);
                keep_column(s + 1, l, 2 * p, sel(m0 & 1, a1, a0));
                fma_ab(rp[l], a0, vc0);
                fma_ab(rp[l], a1, vc1);
                fma_cab(cp0, a0, vi);
                fma_cab(cp1, a1, vi);
            });
            col_sums(2 * p, cp0, cp1);
        });
        S vr[LT];
#pragma unroll
        for (int l = 0; l < LT; ++l) vr[l] = vrow(l + MG / 2);
        unrolled<0, MT / 2>([&](auto uc) {  // block columns 2u, 2u + 1 of the trailing grid
            constexpr int u = decltype(uc)::value;
            S cp[2] = {zero, zero};
            const S vc0 = vcol(MG + 2 * u), vc1 = vcol(MG + 2 * u + 1);
            unrolled<u, LT>([&](auto lc) {  // row blocks from the diagonal's on
                constexpr int l = decltype(lc)::value;
                const S a0 = aget(Lay::idx(l, 2 * u)), a1 = aget(Lay::idx(l, 2 * u + 1));
                fma_ab(rp[l + MG / 2], a0, vc0);
                fma_cab(cp[0], a0, vr[l]);
                fma_ab(rp[l + MG / 2], a1, vc1);
                fma_cab(cp[1], a1, vr[l]);
            });
            col_sums(MG + 2 * u, cp[0], cp[1]);
        });
        __builtin_amdgcn_sched_barrier(0);
        S mine = zero;  // lane c writes the sum of row block c: one write, no branch a row block
#pragma unroll
        for (int l = 0; l < LR; ++l) {
            S t = rp[l];
            qv = dot_acc(l < MG / 2 ? vrow(l) : vr[l < MG / 2 ? 0 : l - MG / 2], t, qv);
            t.x = wave::row_sum16(t.x);
            t.y = wave::row_sum16(t.y);
            mine = sel(c == l, t, mine);
        }
        if (c < LR) RP[r + PR * c] = mine;
        qv = wave::sum(qv);
        if (lane == 0) Q[wv] = qv;
        __syncthreads();
        // ---- w = tau y - (1/2)|tau|^2 (v^H A v) v and v, published for the update ----
        if (tid < NX) {
            const int i = tid;
            S y = zero;
            if (i > s) {
                y = RP[i];
#pragma unroll
                for (int w = 0; w < NW; ++w) y = add(y, CP[w][i]);
            }
            float vav = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) vav += Q[w];
            const float alpha = -dot_acc(tau, tau, 0.f) * vav;
            const S v = sel(i == s + 1, one, mul(X[i], sc));
            Y[i] = axpy(alpha, v, mul(y, tau));
            V[i] = v;
        }
        __syncthreads();
        // ---- A -= v w^H + w v^H right of the strip; column s + 1 to X ----
        if (s + 1 < PC * MG) publish(s + 1);
        S wr[LT];
#pragma unroll
        for (int l = 0; l < LT; ++l) wr[l] = Y[r + PR * (l + MG / 2)];
        auto trailing_update = [&](auto mc) {
            constexpr int m = decltype(mc)::value;
            const S vcm = V[c + PC * (m + MG)], wcm = Y[c + PC * (m + MG)];
            unrolled<Lay::lmin(m), LT>([&](auto lc) {
                constexpr int l = decltype(lc)::value;
                constexpr float f = Lay::straddles(l, m) ? 0.5f : 1.f;
                S a = aget(Lay::idx(l, m));
                fms_abc(a, scale(vr[l], f), wcm);
                fms_abc(a, scale(wr[l], f), vcm);
                aset(Lay::idx(l, m), a);
            });
        };
        unrolled<0, MT>(trailing_update);
        __syncthreads();
    }
    float2* B = Bout + kk * b_kstride;
#pragma unroll
    for (int l = 0; l < LT; ++l)
#pragma unroll
        for (int m = 0; m <= Lay::mmax(l); ++m) {
            const int i = r + PR * l, j = c + PC * m;
            if (i >= j) B[j + (int64_t)i * NT] = sc_store<S>(scale(aget(Lay::idx(l, m)), Lay::straddles(l, m) ? 2.f : 1.f));
        }
}

// memory of the strip per k-point (elements): block columns 0 .. MG - 1
constexpr int strip_slots(int LR, int MG) { return strip_base(LR, MG) * 512; }

}  // namespace uepm
