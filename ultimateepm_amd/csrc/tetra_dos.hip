// Linear-tetrahedron density of states on a Brillouin-zone mesh.
//
// DOS(E) for one band = sum over tetrahedra of the iso-surface polygon area
// times the mean of 1/|grad E| at its corners, over (2 pi)^3
// (Tetra::compute_tetra_dos_energy_band, src/BZ_MESH/mesh_tetra.cpp:477-525,
// summed by MeshBZ::compute_dos_at_energy_and_band, src/BZ_MESH/bz_mesh.cpp:844-862,
// on the energy grid of compute_dos_band_at_band_auto, :889-916).
//
// Work split: one energy group of kEnergiesPerGroup samples x one slice of the
// tetrahedra per workgroup.  A per-band prepass stores each tetrahedron's energy
// range and sample-index window (24 bytes, read from L2 by every group).  A block
// of kBlock tetrahedra is first turned into the list of (energy, tetrahedron) pairs
// that cut, energy by energy in tetrahedron order, and the list is then worked off
// one pair per lane: about a tenth of the pairs cut, so a lane per tetrahedron left
// the waves to their slowest lane: 56k tetrahedra, 500 samples took 0.95 ms a band,
// with the lists 0.28, with the fewer divisions and no arc tangents of tetra_dos_at
// 0.21, bound by FP64 issue.  An energy's contributions are added in the order of its
// own list, and partial sums per (slice, energy) go to a workspace that a second
// kernel adds in slice order: the result depends neither on scheduling nor on the
// other energies of the grid.
//
// Every expression follows the reference's operation order with contraction
// off, so a tetrahedron's contribution rounds as the reference's does (the corners'
// angles only rank them, and are compared by a function that rises with the angle).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "solver.hpp"

#pragma clang fp contract(off)

namespace {

constexpr int kThreads = 256;
constexpr int kEnergiesPerGroup = 4;  // one wave each in the sums
constexpr int kBlock = 1024;          // tetrahedra per list: 4 per lane, 40 KB of LDS at worst

struct V3 {
    double x, y, z;
};
__device__ inline V3 sub(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ inline V3 add(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ inline V3 scale(double s, V3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ inline V3 divide(V3 a, double s) { return {a.x / s, a.y / s, a.z / s}; }
__device__ inline double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline V3 cross(V3 a, V3 b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
__device__ inline double norm(V3 a) { return sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ inline double triple(V3 a, V3 b, V3 c) { return dot(a, cross(b, c)); }
__device__ inline V3 load3(const double* p, int64_t i) { return {p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }

// (1/6) * (e1 . (e2 x e3)) scaled back by 6, as Tetra::compute_signed_volume
// (mesh_tetra.cpp:128-132) and compute_barycentric_coordinates (:173-191) do.
__global__ void tetra_det_kernel(const double* __restrict__ pos, const int32_t* __restrict__ tet, int64_t nt,
                                 double* __restrict__ det) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= nt) return;
    const V3 p0 = load3(pos, tet[4 * t]);
    const V3 e0 = sub(load3(pos, tet[4 * t + 1]), p0);
    const V3 e1 = sub(load3(pos, tet[4 * t + 2]), p0);
    const V3 e2 = sub(load3(pos, tet[4 * t + 3]), p0);
    const double signed_volume = (1.0 / 6.0) * triple(e0, e1, e2);
    det[t] = 6.0 * signed_volume;
}

// Vertex-major (nv x ld) energies and (nv x ld x 3) gradients -> band-major.
__global__ void bands_to_band_major_kernel(const double* __restrict__ E, const double* __restrict__ G, int64_t nv,
                                           int ld, int first, int nb, double* __restrict__ Eb,
                                           double* __restrict__ Gb) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= nv * nb) return;
    const int64_t v = i / nb;
    const int b = static_cast<int>(i - v * nb);
    Eb[b * nv + v] = E[v * ld + first + b];
    if (G) {
        const double* g = G + 3 * (v * ld + first + b);
        double* o = Gb + 3 * (b * nv + v);
        o[0] = g[0];
        o[1] = g[1];
        o[2] = g[2];
    }
}

// Energy range and sample-index window [lo, hi] of every tetrahedron for one band.
// The window is a filter (one sample of slack on each side) that keeps what is
// outside the wedge or has no energy at all out; the range is the exact test.
__global__ void tetra_window_kernel(const int32_t* __restrict__ tet, const uint8_t* __restrict__ in_wedge, int64_t nt,
                                    const double* __restrict__ Eb, double e0, double step, int n_points,
                                    uepm::TetraRange* __restrict__ range) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= nt) return;
    uepm::TetraRange w{0.0, 0.0, 1, 0};  // empty
    if (!in_wedge || in_wedge[t]) {
        const double e[4] = {Eb[tet[4 * t]], Eb[tet[4 * t + 1]], Eb[tet[4 * t + 2]], Eb[tet[4 * t + 3]]};
        const double mn = fmin(fmin(e[0], e[1]), fmin(e[2], e[3])), mx = fmax(fmax(e[0], e[1]), fmax(e[2], e[3]));
        w.emin = w.emax = e[0];
        for (int j = 1; j < 4; ++j) {
            if (e[j] < w.emin) w.emin = e[j];
            if (w.emax < e[j]) w.emax = e[j];
        }
        if (mn <= mx) {
            const double flo = floor((mn - e0) / step) - 1.0, fhi = ceil((mx - e0) / step) + 1.0;
            if (fhi >= 0.0 && flo <= static_cast<double>(n_points - 1)) {
                w.lo = flo < 0.0 ? 0 : static_cast<int>(flo);
                w.hi = fhi > static_cast<double>(n_points - 1) ? n_points - 1 : static_cast<int>(fhi);
            }
        }
    }
    range[t] = w;
}

struct TetraBand {
    int v[4];      // corners
    double emin, emax;
    double es[4];  // corner energies, ascending
    V3 ps[4];      // corners in that order (1/m)
};

__device__ __forceinline__ void load_tetra(TetraBand& T, const double* pos, const int32_t* tet, const double* Eb, int64_t t) {
    double v[4];
    V3 q[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        T.v[j] = tet[4 * t + j];
        q[j] = load3(pos, T.v[j]);
        v[j] = Eb[T.v[j]];
    }
    T.emin = v[0];
    T.emax = v[0];
#pragma unroll
    for (int j = 1; j < 4; ++j) {
        if (v[j] < T.emin) T.emin = v[j];
        if (T.emax < v[j]) T.emax = v[j];
    }
    // five-comparator network (Tetra::pre_compute_sorted_slots_per_band,
    // mesh_tetra.cpp:287-315); the corners move with their energies, so the
    // sorted data needs no dynamic indexing.
#define UEPM_CSWAP(a, b)                \
    if (v[a] > v[b]) {                  \
        const double tv = v[a];         \
        v[a] = v[b];                    \
        v[b] = tv;                      \
        const V3 tq = q[a];             \
        q[a] = q[b];                    \
        q[b] = tq;                      \
    }
    UEPM_CSWAP(0, 1)
    UEPM_CSWAP(2, 3)
    UEPM_CSWAP(0, 2)
    UEPM_CSWAP(1, 3)
    UEPM_CSWAP(1, 2)
#undef UEPM_CSWAP
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        T.es[j] = v[j];
        T.ps[j] = q[j];
    }
}

// Contribution of tetrahedron t at one energy (states / (eV m^3), before the
// mesh-level factors).  What the gradients need is loaded only after the polygon is
// done (its corners are in the caches): both at once take 215 registers.
__device__ __forceinline__ double tetra_dos_at(const TetraBand& T, const double* pos, const double* det, const double* Gb,
                                               int64_t t, double energy) {
    if (energy < T.emin || energy > T.emax) return 0.0;
    const double e_0 = T.es[0], e_1 = T.es[1], e_2 = T.es[2], e_3 = T.es[3];
    const V3 P0 = T.ps[0], P1 = T.ps[1], P2 = T.ps[2], P3 = T.ps[3];
    // iso-energy polygon (Tetra::compute_band_iso_energy_surface, mesh_tetra.cpp:339-395):
    // corner i at l of the way from A to B; the three cases differ in what goes in, so a
    // wave that has all three divides four times, not ten
    const bool low = energy < e_1 && energy >= e_0, mid = !low && energy < e_2 && energy >= e_1;
    const int n = mid ? 4 : 3;
    V3 iso[4];
    auto corner = [&](double num, double den, V3 A, V3 B) {
        const double l = num / den;
        return add(scale(1.0 - l, A), scale(l, B));
    };
    auto pick = [](bool b, V3 x, V3 y) { return V3{b ? x.x : y.x, b ? x.y : y.y, b ? x.z : y.z}; };
    const double up = energy - e_0, down = e_3 - energy;
    const V3 P = pick(low || mid, P0, P3);
    iso[0] = corner(low || mid ? up : down, low ? e_1 - e_0 : mid ? e_2 - e_0 : e_3 - e_2, P, pick(low, P1, P2));
    iso[1] = corner(low || mid ? up : down, low ? e_2 - e_0 : mid ? e_3 - e_0 : e_3 - e_1, P, pick(low, P2, pick(mid, P3, P1)));
    iso[2] = corner(low ? up : mid ? e_2 - energy : down, mid ? e_2 - e_1 : e_3 - e_0, pick(low, P0, pick(mid, P2, P3)),
                    pick(low, P3, pick(mid, P1, P0)));
    iso[3] = corner(energy - e_1, e_3 - e_1, P1, P3);  // n = 4 only
    // cyclic order around the centroid (order_cyclic, mesh_tetra.cpp:402-450).
    // Loops run to 4 with a guard so every array index is static (registers,
    // no scratch); the stable sort by angle becomes a stable rank.
    V3 c = {0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < n) c = add(c, iso[i]);
    c = divide(c, static_cast<double>(n));
    V3 nrm = cross(sub(iso[1], iso[0]), sub(iso[2], iso[0]));
    const double len = norm(nrm);
    if (len > 0.0) nrm = divide(nrm, len);
    V3 u = sub(iso[0], c);
    const double ulen = norm(u);
    if (ulen > 0.0) {
        u = divide(u, ulen);
    } else {
        u = {1.0, 0.0, 0.0};
    }
    const V3 v = cross(nrm, u);
    double ang[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const V3 d = sub(iso[i], c);
        // y / (|x| + |y|), continued over the four quadrants: increases with the angle of
        // (x, y) from -pi to pi, which is all that the ranks need
        const double y = dot(d, v), x = dot(d, u), s = fabs(x) + fabs(y);
        const double a = s > 0.0 ? y / s : 0.0;
        ang[i] = i >= n ? 0.0 : x < 0.0 ? copysign(2.0, y) - a : a;
    }
    int rank[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int r = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < n && j != i && (ang[j] < ang[i] || (j < i && !(ang[i] < ang[j])))) ++r;
        rank[i] = r;
    }
    V3 q[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        q[p] = iso[0];
#pragma unroll
        for (int i = 1; i < 4; ++i)
            if (i < n && rank[i] == p) q[p] = iso[i];
    }
    // polygon area (polygon_area, mesh_tetra.cpp:462-474)
    V3 sum = {0.0, 0.0, 0.0};
    sum = add(sum, cross(q[0], q[1]));
    sum = add(sum, cross(q[1], q[2]));
    if (n == 4) {
        sum = add(sum, cross(q[2], q[3]));
        sum = add(sum, cross(q[3], q[0]));
    } else {
        sum = add(sum, cross(q[2], q[0]));
    }
    const double A = 0.5 * norm(sum);
    if (!(A > 0.0)) return 0.0;
    // mean of 1/|grad E| at the polygon corners, gradients interpolated
    // barycentrically (interpolate_gradient_energy_at_band, mesh_tetra.cpp:214-230)
    int c0 = T.v[0], c1 = T.v[1], c2 = T.v[2], c3 = T.v[3];
    asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3));  // the corners again, not kept
    const V3 p0 = load3(pos, c0);
    const V3 edge[3] = {sub(load3(pos, c1), p0), sub(load3(pos, c2), p0), sub(load3(pos, c3), p0)};
    const V3 grad[4] = {load3(Gb, c0), load3(Gb, c1), load3(Gb, c2), load3(Gb, c3)};
    const double dt = det[t];
    double inv_grad_sum = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i >= n) break;
        const V3 v1 = sub(iso[i], p0);
        const double l2 = triple(v1, edge[1], edge[2]) / dt;
        const double l3 = triple(v1, edge[2], edge[0]) / dt;
        const double l4 = triple(v1, edge[0], edge[1]) / dt;
        const double l1 = 1.0 - l2 - l3 - l4;
        V3 g = {0.0, 0.0, 0.0};
        g = add(g, scale(l1, grad[0]));
        g = add(g, scale(l2, grad[1]));
        g = add(g, scale(l3, grad[2]));
        g = add(g, scale(l4, grad[3]));
        const double gn = norm(g);
        const double g_min = 1e-12;
        inv_grad_sum += 1.0 / (gn < g_min ? g_min : gn);
    }
    const double inv_grad_avg = inv_grad_sum / static_cast<double>(n);
    const double pref = 1.0 / (8.0 * M_PI * M_PI * M_PI);
    return pref * (A * inv_grad_avg);
}

__device__ inline double wave_sum(double x) {
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

__global__ void __launch_bounds__(kThreads) tetra_dos_kernel(
    const double* __restrict__ pos, const int32_t* __restrict__ tet, const double* __restrict__ det,
    const uepm::TetraRange* __restrict__ range, int64_t nt, int64_t per_slice, const double* __restrict__ Eb,
    const double* __restrict__ Gb, double e0, double step, int n_points, double* __restrict__ partial) {
    constexpr int NW = kThreads / 64, PT = kBlock / kThreads, NG = kEnergiesPerGroup;
    static_assert(NG == NW && NG * PT * NW == 64, "one wave scans the counts and each sums one energy");
    __shared__ double val[NG * kBlock];
    __shared__ uint16_t list[NG * kBlock];
    __shared__ int count[64];    // cutting tetrahedra by (energy, tetrahedron round, wave)
    __shared__ int offset[65];   // their exclusive sums: where each group of the list starts
    const int g0 = blockIdx.x * NG;
    const int64_t t_begin = blockIdx.y * per_slice;
    const int64_t t_end = min(nt, t_begin + per_slice);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double acc = 0.0;  // of energy g0 + wave, in lane 0
    for (int64_t t0 = t_begin; t0 < t_end; t0 += kBlock) {
        uint64_t cut[NG][PT];
#pragma unroll
        for (int k = 0; k < PT; ++k) {
            const int64_t t = t0 + k * kThreads + threadIdx.x;
            const uepm::TetraRange w = range[min(t, nt - 1)];
#pragma unroll
            for (int j = 0; j < NG; ++j) {
                const int i = g0 + j;
                const double energy = e0 + static_cast<double>(i) * step;
                cut[j][k] = __ballot(t < t_end && i < n_points && w.lo <= i && i <= w.hi &&
                                     !(energy < w.emin || energy > w.emax));
                if (lane == 0) count[(j * PT + k) * NW + wave] = __popcll(cut[j][k]);
            }
        }
        __syncthreads();
        if (wave == 0) {
            int s = count[lane];
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(s, o, 64);
                if (lane >= o) s += u;
            }
            offset[lane + 1] = s;
            if (lane == 0) offset[0] = 0;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PT; ++k)
#pragma unroll
            for (int j = 0; j < NG; ++j)
                if (cut[j][k] >> lane & 1)
                    list[offset[(j * PT + k) * NW + wave] + __popcll(cut[j][k] & ((1ull << lane) - 1))] =
                        static_cast<uint16_t>(k * kThreads + threadIdx.x);
        __syncthreads();
        const int total = offset[64];
        for (int q = threadIdx.x; q < total; q += kThreads) {
            int j = 0;
            for (int u = 1; u < NG; ++u) j += q >= offset[u * PT * NW];
            TetraBand T;
            const int64_t t = t0 + list[q];
            load_tetra(T, pos, tet, Eb, t);
            val[q] = tetra_dos_at(T, pos, det, Gb, t, e0 + static_cast<double>(g0 + j) * step);
        }
        __syncthreads();
        {
            double s = 0.0;
            const int q1 = offset[(wave + 1) * PT * NW];
            for (int q = offset[wave * PT * NW] + lane; q < q1; q += 64) s += val[q];
            acc += wave_sum(s);
        }
        // (the next block writes count before its first barrier, offset and list after it)
    }
    if (lane == 0 && g0 + wave < n_points) partial[blockIdx.y * (int64_t)n_points + g0 + wave] = acc;
}

// Adds the slices in order and applies the mesh factors in the reference's
// order (bz_mesh.cpp:855-860).
__global__ void tetra_dos_finish_kernel(const double* __restrict__ partial, int slices, int n_points, double e0,
                                        double step, double reduce_bz_factor, double spin_degeneracy,
                                        double wedge_factor, double* __restrict__ energies, double* __restrict__ dos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_points) return;
    double s = 0.0;
    for (int k = 0; k < slices; ++k) s += partial[(int64_t)k * n_points + i];
    s *= reduce_bz_factor;
    s *= spin_degeneracy;
    s *= wedge_factor;
    if (energies) energies[i] = e0 + static_cast<double>(i) * step;
    dos[i] = s;
}

}  // namespace

namespace uepm {

hipError_t launch_tetra_det(const double* pos, const int32_t* tet, int64_t nt, double* det, hipStream_t s) {
    if (nt <= 0) return hipSuccess;
    const unsigned blocks = static_cast<unsigned>((nt + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(tetra_det_kernel, dim3(blocks), dim3(kThreads), 0, s, pos, tet, nt, det);
    return hipGetLastError();
}

hipError_t launch_bands_to_band_major(const double* E, const double* G, int64_t nv, int ld, int first, int nb,
                                      double* Eb, double* Gb, hipStream_t s) {
    const int64_t n = nv * nb;
    if (n <= 0) return hipSuccess;
    const unsigned blocks = static_cast<unsigned>((n + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(bands_to_band_major_kernel, dim3(blocks), dim3(kThreads), 0, s, E, G, nv, ld, first, nb, Eb,
                       Gb);
    return hipGetLastError();
}

int tetra_dos_slices(int64_t nt, int n_points) {
    // 1024 tetrahedra per slice (at most 256 slices), from nt alone: the
    // order in which a sample's contributions are added then does not depend
    // on the energy grid, and one energy gives the same bits alone or in a grid.
    (void)n_points;
    int64_t slices = (nt + 1023) / 1024;
    if (slices < 1) slices = 1;
    if (slices > 256) slices = 256;
    return static_cast<int>(slices);
}

hipError_t launch_tetra_dos(const double* pos, const int32_t* tet, const double* det, const uint8_t* in_wedge,
                            int64_t nt, const double* Eb, const double* Gb, int n_points, double e_min, double e_max,
                            double reduce_bz_factor, double spin_degeneracy, double wedge_factor, TetraRange* range,
                            double* partial, double* energies, double* dos, hipStream_t s) {
    const double step = (e_max - e_min) / static_cast<double>(n_points - 1);
    const int slices = tetra_dos_slices(nt, n_points);
    if (nt > 0) {
        const unsigned tb = static_cast<unsigned>((nt + kThreads - 1) / kThreads);
        hipLaunchKernelGGL(tetra_window_kernel, dim3(tb), dim3(kThreads), 0, s, tet, in_wedge, nt, Eb, e_min, step,
                           n_points, range);
        const int64_t per_slice = (nt + slices - 1) / slices;
        const unsigned groups = static_cast<unsigned>((n_points + kEnergiesPerGroup - 1) / kEnergiesPerGroup);
        hipLaunchKernelGGL(tetra_dos_kernel, dim3(groups, slices), dim3(kThreads), 0, s, pos, tet, det, range, nt,
                           per_slice, Eb, Gb, e_min, step, n_points, partial);
    }
    const unsigned fb = static_cast<unsigned>((n_points + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(tetra_dos_finish_kernel, dim3(fb), dim3(kThreads), 0, s, partial, nt > 0 ? slices : 0,
                       n_points, e_min, step, reduce_bz_factor, spin_degeneracy, wedge_factor, energies, dos);
    return hipGetLastError();
}

}  // namespace uepm
