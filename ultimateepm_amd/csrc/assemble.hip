// assemble.hip — H(k) for a batch of k-points on gfx950 (Hamiltonian::SetMatrix
// and the 0.5 (H + H^dagger) step of Diagonalize, src/EPP/Hamiltonian.cpp:50-127).
//
// Bound by the write of H where the pair terms are cheap, else by FP64 VALU work:
// one evaluation per pair, per-vector factors for everything separable, one
// division (and one exponential, gaussian wells) a pair.  Alone on the chip, ms
// per 4096 k-points, before (pairs evaluated both ways where their rounding
// differs) and now: GaAs N = 181 3.14 -> 0.92 (2.3 TB/s), InP N = 181 1.40 ->
// 1.03, InP N = 59 0.27 -> 0.18, Ge + SOC dim 274 3.11 -> 2.52, GaAs + SOC dim 362
// 5.50 -> 4.52 (1.9 TB/s); Si N = 181 0.87 -> 0.88 (already the write).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "epm_physics.hpp"
#include "scalars.hpp"
#include "solver.hpp"

namespace uepm {

// What a plan's H(k) is stored as.
enum class HForm { kComplex, kReal, kSpinor, kQuaternion };
template <HForm F>
struct HElem { using T = double2; };
template <>
struct HElem<HForm::kReal> { using T = double; };
template <>
struct HElem<HForm::kQuaternion> { using T = q4<double>; };

// One workgroup per k.  Per-basis-vector state in LDS, then 16 x 16 tiles of
// pairs (i, j), i >= j, one wave a tile: each wave evaluates its pairs once
// (the element formed is the reference's 0.5 (h_ij + conj(h_ji)), its Diagonalize
// hermitisation; epm_physics.hpp), writes the tile and, through its LDS slot,
// the conjugate transpose above the diagonal, so both halves go out in 16-element
// column runs.  Output: column-major dim x dim, leading dimension ld, one matrix
// per k.
//   kReal    the real parts alone, where the imaginary parts are exactly zero
//   kSpinor  2N x 2N: blocks [[M + S00, S01], [S10, M - S00]], each tile of pairs
//            writing its four blocks (and their transposes) in turn
//   kQuaternion  N x N: u = M + S00 and d = S10 of each spinor block, which is
//            [[u, -conj(d)], [d, conj(u)]] where the antisymmetric terms vanish
template <int BS, HForm F>
__global__ __launch_bounds__(BS, 4) void assemble_kernel(DevParams P, const int32_t* __restrict__ G,
                                                      const double* __restrict__ kpts,
                                                      typename HElem<F>::T* __restrict__ H, int ld) {
    using T = typename HElem<F>::T;
    extern __shared__ __align__(16) unsigned char smem[];
    double* S = reinterpret_cast<double*>(smem);
    __shared__ double2 vtab[kVPhaseTab];
    constexpr bool kSoc = F == HForm::kSpinor || F == HForm::kQuaternion;
    __shared__ T Tt[BS / 64][kSoc ? 4 : 16][17];
    const int kk = blockIdx.x;
    const double* k = kpts + 3 * (size_t)kk;
    const int N = P.N;
    const VecLayout L = vec_layout(P);
    int32_t* Gs = reinterpret_cast<int32_t*>(S + L.count * N);
    for (int i = threadIdx.x; i < N; i += BS) vector_init(P, L, k, G, i, S, Gs);
    for (int t = threadIdx.x; t < kVPhaseTab; t += BS) vtab[t] = local_phase(P, t / 49 - 3, (t / 7) % 7 - 3, t % 7 - 3);
    __syncthreads();
    T* A = H + (size_t)kk * ld * (F == HForm::kQuaternion ? N : P.dim);
    const int nt = (N + 15) >> 4, ntiles = nt * (nt + 1) / 2;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int il = lane & 15, jq = lane >> 4;
    T(*Tw)[17] = Tt[wv];
    auto wsync = [] {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    int bj = 0, rem = wv;  // tile -> (bj + rem, bj), column-major over the lower triangle of tiles
    for (int tile = wv; tile < ntiles; tile += BS / 64, rem += BS / 64) {
        while (rem >= nt - bj) {
            rem -= nt - bj;
            ++bj;
        }
        const int bi = bj + rem;
        // one pair per lane and pass (not unrolled: four at once would take the registers
        // of a second workgroup)
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            const int jl = jq + 4 * q;
            const int i = 16 * bi + il, j = 16 * bj + jl;
            const bool in = i < N && j < N && i >= j;
            double re = 0.0, im = 0.0, so[6];
            if (in) {
                const int gx = Gs[i] - Gs[j], gy = Gs[N + i] - Gs[N + j], gz = Gs[2 * N + i] - Gs[2 * N + j];
                local_V(P, gx, gy, gz, re, im, vtab);
                if (i == j) {
                    const double kx = S[i], ky = S[N + i], kz = S[2 * N + i];
                    re += P.kin * (kx * kx + ky * ky + kz * kz);
                }
                if (P.nl) {
                    double r, m;
                    nonlocal(P, L, S, i, j, r, m);
                    re += r;
                    im += m;
                }
                if constexpr (kSoc) soc_block(P, L, S, i, j, so);
            }
            if constexpr (F == HForm::kReal) {
                if (in) A[i + (size_t)j * ld] = Tw[jl][il] = re;
            } else if constexpr (F == HForm::kComplex) {
                if (in) A[i + (size_t)j * ld] = Tw[jl][il] = make_double2(re, im);
            } else {
                // the blocks in turn: element (row r0 + i, column c0 + j), and its conjugate at
                // (c0 + j, r0 + i) through four rows of the slot (runs of four elements); the
                // diagonal of an off-diagonal block has a transpose of its own
                auto put = [&](int r0, int c0, T h) {
                    if (in) A[(r0 + i) + (size_t)(c0 + j) * ld] = Tw[jq][il] = h;
                    wsync();
                    const int j2 = 16 * bj + 4 * q + (lane & 3), i2 = 16 * bi + (lane >> 2);
                    if (i2 < N && j2 < N && (i2 > j2 || (i2 == j2 && r0 != c0))) {
                        const T t = Tw[lane & 3][lane >> 2];
                        T& to = A[(c0 + j2) + (size_t)(r0 + i2) * ld];
                        if constexpr (F == HForm::kQuaternion) to = conj_if(t, true);
                        else to = make_double2(t.x, -t.y);
                    }
                    wsync();
                };
                if constexpr (F == HForm::kQuaternion) {
                    put(0, 0, T{re + so[0], im + so[1], so[4], so[5]});
                } else {
                    put(0, 0, make_double2(re + so[0], im + so[1]));
                    put(N, N, make_double2(re - so[0], im - so[1]));
                    put(N, 0, make_double2(so[4], so[5]));
                    put(0, N, make_double2(so[2], so[3]));
                }
            }
        }
        if constexpr (!kSoc) {
            wsync();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int il2 = jq + 4 * q;
                const int j = 16 * bj + il, i = 16 * bi + il2;  // consecutive lanes walk j
                if (i < N && j < N && i > j) {
                    const T h = Tw[il][il2];
                    if constexpr (F == HForm::kReal) A[j + (size_t)i * ld] = h;
                    else A[j + (size_t)i * ld] = make_double2(h.x, -h.y);
                }
            }
            wsync();
        }
    }
}

constexpr int kAsmBS = 256;

namespace {
template <HForm F>
hipError_t launch_assemble_form(const DevParams& P, const int32_t* dG, const double* dk, int64_t nk,
                                typename HElem<F>::T* dH, int ld, hipStream_t s) {
    // the per-vector arrays (at most 164 bytes a vector, 196 with spin-orbit) beside the
    // phase table and the transpose slots: 576 vectors take 117 of the 160 KB of a CU, 288
    // spinor ones 66
    const size_t shm = vec_bytes(P);
    const size_t fixed = sizeof(double2) * kVPhaseTab + (kAsmBS / 64) * (F == HForm::kSpinor || F == HForm::kQuaternion ? 4 : 16) * 17 * sizeof(typename HElem<F>::T);
    if (shm + fixed > 163840) return hipErrorInvalidValue;
    auto kern = assemble_kernel<kAsmBS, F>;
    hipError_t err = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(kern, dim3((unsigned)nk), dim3(kAsmBS), shm, s, P, dG, dk, dH, ld);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_assemble(const DevParams& P, const int32_t* dG, const double* dk, int64_t nk, double2* dH, int ld,
                           hipStream_t s) {
    if (P.soc) return launch_assemble_form<HForm::kSpinor>(P, dG, dk, nk, dH, ld, s);
    return launch_assemble_form<HForm::kComplex>(P, dG, dk, nk, dH, ld, s);
}

hipError_t launch_assemble_real(const DevParams& P, const int32_t* dG, const double* dk, int64_t nk, double* dH, int ld,
                                hipStream_t s) {
    if (P.soc) return hipErrorInvalidValue;
    return launch_assemble_form<HForm::kReal>(P, dG, dk, nk, dH, ld, s);
}

hipError_t launch_assemble_quaternion(const DevParams& P, const int32_t* dG, const double* dk, int64_t nk, q4<double>* dH,
                                      int ld, hipStream_t s) {
    if (!P.soc) return hipErrorInvalidValue;
    return launch_assemble_form<HForm::kQuaternion>(P, dG, dk, nk, dH, ld, s);
}

}  // namespace uepm
