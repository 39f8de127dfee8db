// Cell binning: the replacement of parallel_binning (code/modules/identical_particles_binning.cpp:97-110,
// code/modules/binning.cpp:15-54) and of the discarded quicksort (code/modules/quick_sort.cpp:509-547).
//
// The reference's binning is, in effect, a stable counting sort of the previous permute_vector by
// cell id, computed with two O(N * cells) sweeps.  Here it is O(N):
//   k_count          : optional fused drift + wrap (identical_particles.cpp:651-669), cell id
//                      (particles.hpp:108-113) and arrival slot from an atomic per-cell counter; the count
//                      can also be done by the heat bath, or inside the FP32 force sweep right after the kick
//                      and the following drift of each atom
//   k_scan           : one workgroup scans the counts into the next offsets (and clears them)
//   k_scatter        : atom -> (cell offset + arrival slot), with its sort key (its previous sorted slot, or
//                      its id for in-cell order by atom id)
//   k_cell_rank      : 16 lanes per cell rank the cell's entries by key -> the stable order
//   k_bin_small      : all of it in one workgroup's LDS for small contexts
// The placement writes the next perm/offs buffers, invperm and the sorted coordinates (FP64, and FP32 relative
// to the cell); the
// host then flips the parity argument that selects the current buffers.
#include "chmc_internal.hpp"
#include "bin_device.hpp"

#pragma clang fp contract(off)   // drift and cell index must match the FP64 oracle bit for bit

namespace chmc {

// What the binning of one atom needs, read together before the first store: the compiler takes no load of the
// chain's constants ahead of a store, so that each dimension waited for its own loads after the one before it (an
// FP64 leapfrog step of N = 512 11.9 us, then 11.2; of 2,744 21.2, then 18.5)
struct BinAtom {
    double x[3], p[3], L[3], sizebin[3], coeff_x;
    int nbin[3], cell_off;
};
__device__ __forceinline__ BinAtom load_atom(const DevView& v, const ChainDev& C, int a, int do_drift)
{
    BinAtom b;
    const int N = v.Ntot;
    b.coeff_x = C.coeff_x;                             // compute_coeff_position, identical_particles.cpp:646-648
    b.cell_off = C.cell_off;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        b.x[d] = v.x[d * N + a];
        b.p[d] = do_drift ? v.p[d * N + a] : 0.0;
        b.L[d] = C.L[d];
        b.sizebin[d] = C.sizebin[d];
        b.nbin[d] = C.nbin[d];
    }
    return b;
}
// the drifted position in dimension d (written back), or the position itself
__device__ __forceinline__ double drift_dim(const DevView& v, const BinAtom& b, int a, int d, double drift_dt, int do_drift)
{
    double xv = b.x[d];
    if (do_drift) {
        xv += drift_dt * b.coeff_x * b.p[d];
        xv = lp_round(xv, v.lp_scale);
        xv = wrap_box(xv, b.L[d]);
        v.x[d * v.Ntot + a] = xv;
    }
    return xv;
}

__global__ __launch_bounds__(256) void k_count(DevView v, double drift_dt, int do_drift)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < v.Ntot) {
        const ChainDev& C = v.chains[v.atom_chain[a]];
        const BinAtom b = load_atom(v, C, a, do_drift);
        double x3[3];
#pragma unroll
        for (int d = 0; d < 3; d++) x3[d] = drift_dim(v, b, a, d, drift_dt, do_drift);
        int g[3];
        count_atom(v, cell_index(b, x3, g), a);
    }
}

__global__ __launch_bounds__(1024) void k_scan(DevView v)
{
    scan_counts_block(v);
}

__global__ __launch_bounds__(256) void k_drift(DevView v, double dt)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= v.Ntot) return;
    const ChainDev& C = v.chains[v.atom_chain[a]];
    const int N = v.Ntot;
    double coeff_x = C.coeff_x;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double xv = v.x[d * N + a];
        xv += dt * coeff_x * v.p[d * N + a];
        xv = lp_round(xv, v.lp_scale);
        xv = wrap_box(xv, C.L[d]);
        v.x[d * N + a] = xv;
    }
}

__global__ __launch_bounds__(256) void k_scatter(DevView v, int atom_id_order)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= v.Ntot) return;
    const int dest = offs_next(v)[v.cell_of[a]] + v.slot[a];
    v.skey[dest] = atom_id_order ? a : v.invperm[a];
    v.satom[dest] = a;
}

__device__ __forceinline__ void cell_origin(const ChainDev& C, int c, double o[3])
{
    const int lc = c - C.cell_off;
    int b[3];
    b[2] = lc / (C.nbin[0] * C.nbin[1]);
    b[1] = (lc - b[2] * C.nbin[0] * C.nbin[1]) / C.nbin[0];
    b[0] = lc - C.nbin[0] * (b[1] + b[2] * C.nbin[1]);
    for (int d = 0; d < 3; d++) o[d] = b[d] * C.sizebin[d];
}

__device__ __forceinline__ void place_atom(const DevView& v, int* perm_n, int pos, int atom, const double x3[3],
                                           const double o[3])
{
    perm_n[pos] = atom;
    v.invperm[atom] = pos;
#pragma unroll
    for (int d = 0; d < 3; d++) v.xs64[(size_t)d * v.Ntot + pos] = x3[d];
    v.xs[pos] = make_float4((float)(x3[0] - o[0]), (float)(x3[1] - o[1]), (float)(x3[2] - o[2]), __int_as_float(atom));
}

// 16 lanes per cell, each entry's position is its rank among the cell's (unique) keys
__global__ __launch_bounds__(256) void k_cell_rank(DevView v)
{
    const int c = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int sub = threadIdx.x & 15;
    if (c >= v.Ctot) return;
    const int N = v.Ntot;
    const int* offs = offs_next(v);
    int* perm_n = perm_next(v);
    const int beg = offs[c];
    const int n = offs[c + 1] - beg;
    const ChainDev& C = v.chains[v.cell_chain[c]];
    double o[3];
    cell_origin(C, c, o);
    for (int e = sub; e < n; e += 16) {
        const int key = v.skey[beg + e];
        const int atom = v.satom[beg + e];
        const double x3[3] = { v.x[atom], v.x[N + atom], v.x[2 * N + atom] };
        int rank = 0;
#pragma unroll 8
        for (int q = 0; q < n; q++) rank += (v.skey[beg + q] < key) ? 1 : 0;
        place_atom(v, perm_n, beg + rank, atom, x3, o);
    }
}

// The whole binning of a context of at most kBinSmall atoms and cells in one workgroup: counts, their scan and
// the sort keys stay in LDS, each thread keeps its (up to three) atoms.  Four launches of a few microseconds of
// latency each otherwise: N = 512, FP64 leapfrog, count + scan + placement took 21 us an evaluation, now
// 4.9.  Bound: latency (three global round trips, six barriers), and one CU's instructions from about 2000 atoms
// on: an FP64 leapfrog step of 2,744 atoms takes 18.5 us with it and 22.4 without, of 4,096 29.7 (before the loads
// were brought together) and 24.1.  512 threads where an atom each is enough: 11.2 -> 10.9 us a step of N = 512.
template <int T, int PT>
__global__ __launch_bounds__(T) void k_bin_small(DevView v, double drift_dt, int do_drift, int atom_id_order)
{
    constexpr int kMax = T * PT;
    __shared__ int cnt[kMax], key[kMax], wsum[T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int N = v.Ntot, nc = v.Ctot;
#pragma unroll
    for (int k = 0; k < PT; k++) cnt[k * T + tid] = 0;
    double x3[PT][3], o3[PT][3];
    int cell[PT], slot[PT], mykey[PT];
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int a = k * T + tid;
        if (a >= N) continue;
        const BinAtom b = load_atom(v, v.chains[v.atom_chain[a]], a, do_drift);
        mykey[k] = atom_id_order ? a : v.invperm[a];
#pragma unroll
        for (int d = 0; d < 3; d++) x3[k][d] = drift_dim(v, b, a, d, drift_dt, do_drift);
        int g[3];
        cell[k] = cell_index(b, x3[k], g);
#pragma unroll
        for (int d = 0; d < 3; d++) o3[k][d] = g[d] * b.sizebin[d];       // cell_origin
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PT; k++)
        if (k * T + tid < N) slot[k] = atomicAdd(&cnt[cell[k]], 1);
    __syncthreads();
    // exclusive scan of the counts, PT contiguous cells a thread
    int c4[PT], s = 0;
#pragma unroll
    for (int k = 0; k < PT; k++) {
        c4[k] = cnt[tid * PT + k];
        s += c4[k];
    }
    int incl = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    int run = incl - s;
    for (int w = 0; w < wid; w++) run += wsum[w];
    int* offs = offs_next(v);
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int c = tid * PT + k;
        cnt[c] = run;
        if (c <= nc) offs[c] = run;            // cells from nc on are empty: the end offset is N
        run += c4[k];
    }
    if (tid == 0 && nc == kMax) offs[nc] = N;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PT; k++)
        if (k * T + tid < N) key[cnt[cell[k]] + slot[k]] = mykey[k];
    __syncthreads();
    int* perm_n = perm_next(v);
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int a = k * T + tid;
        if (a >= N) continue;
        const int beg = cnt[cell[k]], end = cell[k] + 1 < kMax ? cnt[cell[k] + 1] : N;
        int rank = 0;
#pragma unroll 4
        for (int q = beg; q < end; q++) rank += key[q] < mykey[k] ? 1 : 0;
        place_atom(v, perm_n, beg + rank, a, x3[k], o3[k]);
    }
}

__global__ void k_fill_int(int* p, int value, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

hipError_t launch_fill_int(int* p, int value, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_int, dim3((n + 255) / 256), dim3(256), 0, s, p, value, n);
    return hipGetLastError();
}

hipError_t launch_count(const DevView& v, double drift_dt, hipStream_t s)
{
    hipLaunchKernelGGL(k_count, dim3((v.Ntot + 255) / 256), dim3(256), 0, s, v, drift_dt, drift_dt != 0.0 ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_scan(const DevView& v, hipStream_t s)
{
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, v);
    return hipGetLastError();
}

hipError_t launch_place(const DevView& v, bool atom_id_order, hipStream_t s)
{
    hipLaunchKernelGGL(k_scatter, dim3((v.Ntot + 255) / 256), dim3(256), 0, s, v, atom_id_order ? 1 : 0);
    hipLaunchKernelGGL(k_cell_rank, dim3((v.Ctot + 15) / 16), dim3(256), 0, s, v);
    return hipGetLastError();
}

hipError_t launch_bin_small(const DevView& v, double drift_dt, bool atom_id_order, hipStream_t s)
{
    const int drift = drift_dt != 0.0 ? 1 : 0, order = atom_id_order ? 1 : 0;
    if (v.Ntot <= 512 && v.Ctot <= 512) hipLaunchKernelGGL((k_bin_small<512, 1>), dim3(1), dim3(512), 0, s, v, drift_dt, drift, order);
    else hipLaunchKernelGGL((k_bin_small<1024, kBinSmall / 1024>), dim3(1), dim3(1024), 0, s, v, drift_dt, drift, order);
    return hipGetLastError();
}

hipError_t launch_drift(const DevView& v, double dt, hipStream_t s)
{
    hipLaunchKernelGGL(k_drift, dim3((v.Ntot + 255) / 256), dim3(256), 0, s, v, dt);
    return hipGetLastError();
}

}  // namespace chmc
