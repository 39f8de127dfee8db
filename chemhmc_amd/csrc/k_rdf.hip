// All-pairs kernels.
//  k_rdf: radial distribution histogram, the replacement of Tag_RDF (code/modules/identical_particles.cpp:739-776).
//    The reference runs one team per bin over all N^2 ordered pairs (O(bins * N^2)); here each pair is
//    visited once and counted twice, which equals the reference's ordered count exactly.  The bin of a
//    pair is the reference's (int)(r / size_bin) with its FP64 minimum image (min of (d-L)^2, d^2,
//    (d+L)^2) for every pair, but almost all of them are decided in FP32 (see below).
//  k_open_potential: code-carsten/potential_energy.hh:6-15, sum_{i<j} a/r^n - b/r^6 with open
//    boundaries, FP64, per-tile partial sums, added in a fixed order by k_open_sum.
#include "chmc_internal.hpp"

#include <algorithm>

#pragma clang fp contract(off)

namespace chmc {

// The exact bin of a pair, as the reference computes it (no contraction)
__device__ __forceinline__ int rdf_bin_exact(const ChainDev& C, double xi, double yi, double zi, double xj, double yj,
                                             double zj, double size_bin)
{
    double r = 0.0, dd, ri, si;
    dd = xj - xi;
    ri = (dd - C.L[0]) * (dd - C.L[0]); si = dd * dd; if (si < ri) ri = si;
    si = (dd + C.L[0]) * (dd + C.L[0]); if (si < ri) ri = si; r += ri;
    dd = yj - yi;
    ri = (dd - C.L[1]) * (dd - C.L[1]); si = dd * dd; if (si < ri) ri = si;
    si = (dd + C.L[1]) * (dd + C.L[1]); if (si < ri) ri = si; r += ri;
    dd = zj - zi;
    ri = (dd - C.L[2]) * (dd - C.L[2]); si = dd * dd; if (si < ri) ri = si;
    si = (dd + C.L[2]) * (dd + C.L[2]); if (si < ri) ri = si; r += ri;
    return (int)(sqrt(r) / size_bin);
}

// Coordinates as 32-bit fractions of the box, u = round(2^32 x / L): the minimum image of a difference is
// then the wrap of an integer subtraction.  w = 1 where a coordinate is outside [0, L] (or not a number):
// pairs of such an atom take the exact path.  The counts are cleared here too.
__global__ __launch_bounds__(256) void k_rdf_prep(DevView v, int chain, int nbins, uint4* __restrict__ u,
                                                  unsigned long long* __restrict__ counts)
{
    const ChainDev& C = v.chains[chain];
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nbins) counts[i] = 0ull;
    if (i >= C.natoms) return;
    unsigned q[3], bad = 0u;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double x = v.x[(size_t)d * v.Ntot + C.atom_off + i];
        const bool ok = x >= 0.0 && x <= C.L[d];
        bad |= ok ? 0u : 1u;
        q[d] = ok ? (unsigned)(unsigned long long)(x / C.L[d] * 4294967296.0 + 0.5) : 0u;
    }
    u[i] = make_uint4(q[0], q[1], q[2], bad);
}

constexpr int kRdfJ = 32;          // j atoms per step of a workgroup

// One thread per i atom (256 a workgroup, row blockIdx.y), j atoms in steps of kRdfJ along the row, read
// through scalar registers (the index is uniform), so that a pair costs no LDS read; one LDS histogram per
// workgroup, added to the global counters once at its end.
//   FP32 decision: with u exact to 2^-33 L, t = |d| / size_bin from three integer differences, converted,
// scaled and summed in FP32 is within 6.5 * 2^-24 t + 2^-32 |L| / size_bin of the exact quotient (3 roundings
// per component, 3 of the sum of squares, halved by the root, and 1 ulp of v_sqrt_f32; in a cube (CUBE) the root
// is scaled instead of the components: 2 roundings for 2).  A pair whose t is
// farther than eps from an integer, eps = (nbins + 1) 2^-21 + 2^-31 |L| / size_bin, therefore has the exact
// bin (int)t; the others (0.05 % at 500 bins) and any NaN are binned in FP64.  Pairs whose t is beyond nbins + 1 by
// the fixed-point part of eps (more than a bin where size_bin < 2^-31 |L|) are never counted and need no decision.
//   Bound: VALU issue, ~20 slots a pair (22 outside a cube).  N = 32768, 500 bins up to L / 2 (5.4e8 pairs): 271 us,
// against 308 us with the components scaled and the tests repeated as selects, and 1531 us with the FP64 root and
// division for every pair.
template <bool CUBE>
__global__ __launch_bounds__(256) void k_rdf(DevView v, int chain, int nbins, double size_bin,
                                             const uint4* __restrict__ u, unsigned long long* __restrict__ counts)
{
    extern __shared__ unsigned int hist[];     // [nbins]
    const ChainDev& C = v.chains[chain];
    const int n = C.natoms, off = C.atom_off, N = v.Ntot;
    const int tid = threadIdx.x, lane = tid & 63;
    const int i0 = blockIdx.y * 256, steps = (n + kRdfJ - 1) / kRdfJ;
    const int first = i0 / kRdfJ + blockIdx.x;
    if (first >= steps) return;
    for (int b = tid; b < nbins; b += 256) hist[b] = 0u;
    __syncthreads();
    const int i = i0 + tid;
    const bool ival = i < n;
    const uint4 ui = u[ival ? i : n - 1];
    const double xi = v.x[off + (ival ? i : n - 1)], yi = v.x[(size_t)N + off + (ival ? i : n - 1)],
                 zi = v.x[2 * (size_t)N + off + (ival ? i : n - 1)];
    const float sx = (float)(C.L[0] / 4294967296.0 / size_bin), sy = (float)(C.L[1] / 4294967296.0 / size_bin),
                sz = (float)(C.L[2] / 4294967296.0 / size_bin);
    const double diag = sqrt(C.L[0] * C.L[0] + C.L[1] * C.L[1] + C.L[2] * C.L[2]);
    const double fixed = diag / size_bin / 2147483648.0;
    const float half = (float)(0.5 - ((nbins + 1) / 2097152.0 + fixed) - 1e-7);
    const float edge = (float)((nbins + 1 + fixed) * (1.0 + 1e-6)), nb = (float)nbins;
    auto exact = [&](int j) {
        const int b = rdf_bin_exact(C, xi, yi, zi, v.x[off + j], v.x[(size_t)N + off + j], v.x[2 * (size_t)N + off + j], size_bin);
        if (b < nbins) atomicAdd(&hist[b], 1u);
    };
    // KB pairs (i, j0 ... j0 + KB - 1), those with j > i where check is set
    auto pairs = [&](int j0, auto kb, bool check) {
        constexpr int KB = decltype(kb)::value;
        float t[KB];
#pragma unroll
        for (int k = 0; k < KB; k++) {
            const uint4 uj = u[j0 + k];
            float dx = (float)(int)(uj.x - ui.x), dy = (float)(int)(uj.y - ui.y), dz = (float)(int)(uj.z - ui.z);
            if constexpr (!CUBE) {
                dx *= sx;
                dy *= sy;
                dz *= sz;
            }
            t[k] = __builtin_amdgcn_sqrtf(__builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)));
            if constexpr (CUBE) t[k] *= sx;
        }
        unsigned late = 0u;
#pragma unroll
        for (int k = 0; k < KB; k++) {
            // clearly inside a bin; a pair that is not, and not clearly beyond the last bin, is decided exactly
            // (a NaN is neither).  Whole waves; the masks of the compares themselves (5: ordered <=, 4: <, 3: >=)
            const float mid = fabsf(__builtin_amdgcn_fractf(t[k]) - 0.5f);
            const unsigned long long on = check ? __ballot(ival && j0 + k > i) : ~0ull;
            const unsigned long long sure = __builtin_amdgcn_fcmpf(mid, half, 5);
            if (__builtin_amdgcn_inverse_ballot_w64(sure & on & __builtin_amdgcn_fcmpf(t[k], nb, 4))) atomicAdd(&hist[(int)t[k]], 1u);
            const unsigned long long un = on & ~sure;
            if (un != 0ull) {                      // rare
                if (__builtin_amdgcn_inverse_ballot_w64(un & ~__builtin_amdgcn_fcmpf(t[k], edge, 3))) late |= 1u << k;
            }
        }
        if (__ballot(late != 0u) != 0ull)
            while (late != 0u) {
                const int k = __ffs(late) - 1;
                late &= late - 1u;
                exact(j0 + k);
            }
    };
    int done = 0;
    auto flush = [&]() {
        __syncthreads();
        for (int k = tid; k < nbins; k += 256) {
            int b = k + (int)(blockIdx.x + blockIdx.y) * 64 % nbins;      // workgroups start at different counters
            if (b >= nbins) b -= nbins;
            const unsigned s = hist[b];
            hist[b] = 0u;
            if (s) atomicAdd(&counts[b], 2ull * s);
        }
        __syncthreads();
    };
    for (int J = first; J < steps; J += gridDim.x) {
        const int j0 = J * kRdfJ, jn = min(kRdfJ, n - j0);
        const bool odd = __ballot(ui.w != 0u || u[j0 + min(lane & (kRdfJ - 1), jn - 1)].w != 0u) != 0ull;
        if (odd) {
            for (int jj = 0; jj < jn; jj++)
                if (ival && j0 + jj > i) exact(j0 + jj);
        } else if (j0 < i0 + 256 || i0 + 256 > n || jn < kRdfJ) {
            for (int jj = 0; jj < jn; jj++) pairs(j0 + jj, std::integral_constant<int, 1>{}, true);
        } else {
            for (int jj = 0; jj < kRdfJ; jj += 8) pairs(j0 + jj, std::integral_constant<int, 8>{}, false);
        }
        if (++done == (1 << 18)) {             // 2^31 pairs: before a 32-bit count can overflow
            done = 0;
            flush();
        }
    }
    flush();
}

// |n|-th power of r from q = r^2 by repeated squaring (n uniform); an odd power takes one factor sqrt(q)
__device__ __forceinline__ double pow_from_square(double q, int n)
{
    const unsigned m = n < 0 ? 0u - (unsigned)n : (unsigned)n;
    double p = (m & 1u) ? sqrt(q) : 1.0;
    for (unsigned e = m >> 1; e != 0u; e >>= 1) {
        if (e & 1u) p *= q;
        q *= q;
    }
    return n < 0 ? 1.0 / p : p;
}

// Tiles of E x E pairs (E = 64: four waves of 64 i atoms, each a quarter of the 64 j atoms; E = 256: one i
// atom per thread, all 256 j atoms); coordinate d of atom i is xyz[3 i + d].  The j atoms are uniform in a
// wave and come through scalar loads.  r^n and r^6 are powers of r^2 by multiplication: a call of pow cost
// ~150 instructions twice a pair and the root another 20.  Bound: latency below a few thousand atoms (the
// 64-tiles put 136 workgroups on N = 1000 where 256-tiles put 10), FP64 VALU beyond.  N = 1000, n = 12:
// 10.7 us against 225 us (pow, 256-tiles).
template <int E>
__global__ __launch_bounds__(256) void k_open_potential(const double* __restrict__ xyz, int n, int nexp, double a, double b,
                                                        double* __restrict__ partials)
{
    __shared__ double wpart[4];
    const int I = blockIdx.y, J = blockIdx.x;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t pid = (size_t)I * gridDim.x + J;
    if (J < I) {
        if (tid == 0) partials[pid] = 0.0;
        return;
    }
    constexpr int JN = E == 64 ? 16 : 256;
    const int i = I * E + (tid & (E - 1)), j0 = J * E + (E == 64 ? wave * JN : 0);
    double s = 0.0;
    if (i < n) {
        const double xi = xyz[3 * (size_t)i], yi = xyz[3 * (size_t)i + 1], zi = xyz[3 * (size_t)i + 2];
        const int jend = min(j0 + JN, n);
#pragma unroll 2
        for (int j = j0; j < jend; j++) {
            const double d0 = xi - xyz[3 * (size_t)j], d1 = yi - xyz[3 * (size_t)j + 1], d2 = zi - xyz[3 * (size_t)j + 2];
            const double q = d0 * d0 + d1 * d1 + d2 * d2;
            const double e = a / pow_from_square(q, nexp) - b / (q * q * q);     // lennardjones.hh:5-9
            s += j > i ? e : 0.0;
        }
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m, 64);
    if ((tid & 63) == 0) wpart[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) partials[pid] = ((wpart[0] + wpart[1]) + wpart[2]) + wpart[3];
}

// the sum of the tile partials in a fixed order: 1024 strided sums, then a tree
__global__ __launch_bounds__(1024) void k_open_sum(const double* __restrict__ partials, size_t count, double* __restrict__ result)
{
    __shared__ double wpart[16];
    double s = 0.0;
    for (size_t k = threadIdx.x; k < count; k += 1024) s += partials[k];
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m, 64);
    if ((threadIdx.x & 63) == 0) wpart[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x != 0) return;
    s = 0.0;
    for (int k = 0; k < 16; k++) s += wpart[k];
    *result = s;
}

// about 4096 workgroups, of which the half below the diagonal returns at once (8 a CU stay): few enough that adding
// their histograms to the counters stays small, rows in order, so that the long ones start first
hipError_t launch_rdf(const DevView& v, int chain, int natoms, bool cube, int nbins, double size_bin, uint4* u,
                      unsigned long long* counts, hipStream_t s)
{
    hipLaunchKernelGGL(k_rdf_prep, dim3((std::max(natoms, nbins) + 255) / 256), dim3(256), 0, s, v, chain, nbins, u, counts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || natoms == 0) return e;
    const int rows = (natoms + 255) / 256, steps = (natoms + kRdfJ - 1) / kRdfJ;
    const int gx = std::min(steps, std::max(1, 4096 / rows));
    const size_t lds = sizeof(unsigned int) * nbins;
    if (cube) hipLaunchKernelGGL(k_rdf<true>, dim3(gx, rows), dim3(256), lds, s, v, chain, nbins, size_bin, u, counts);
    else hipLaunchKernelGGL(k_rdf<false>, dim3(gx, rows), dim3(256), lds, s, v, chain, nbins, size_bin, u, counts);
    return hipGetLastError();
}

// 64-tiles while their count fits the partials of 65536 atoms in 256-tiles
int open_potential_tiles(int n)
{
    return n <= kOpenSmall ? (n + 63) / 64 : (n + 255) / 256;
}

size_t open_potential_partials(int n)
{
    const size_t T = (size_t)open_potential_tiles(n);
    return T * T;
}

hipError_t launch_open_potential(const double* xyz, int n, int nexp, double a, double b, double* partials, double* result,
                                 hipStream_t s)
{
    const int T = open_potential_tiles(n);
    if (T > 0) {
        if (n <= kOpenSmall)
            hipLaunchKernelGGL(k_open_potential<64>, dim3(T, T), dim3(256), 0, s, xyz, n, nexp, a, b, partials);
        else
            hipLaunchKernelGGL(k_open_potential<256>, dim3(T, T), dim3(256), 0, s, xyz, n, nexp, a, b, partials);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_open_sum, dim3(1), dim3(1024), 0, s, partials, open_potential_partials(n), result);
    return hipGetLastError();
}

}  // namespace chmc
