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

__global__ __launch_bounds__(256) void k_count(DevView v, double drift_dt, int do_drift)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < v.Ntot) {
        const ChainDev& C = v.chains[v.atom_chain[a]];
        const int N = v.Ntot;
        const double coeff_x = C.coeff_x;              // compute_coeff_position, identical_particles.cpp:646-648
        double x3[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double xv = v.x[d * N + a];
            if (do_drift) {
                xv += drift_dt * coeff_x * v.p[d * N + a];
                xv = lp_round(xv, v.lp_scale);
                xv = wrap_box(xv, C.L[d]);
                v.x[d * N + a] = xv;
            }
            x3[d] = xv;
        }
        count_atom(v, C, a, x3);
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
// 5.7.  Bound: latency (three global round trips, six barriers), and one CU's instructions from about 2000 atoms
// on: an FP64 leapfrog step of 2,744 atoms takes 21.6 us with it and 22.4 without, of 4,096 29.7 and 25.4.
__global__ __launch_bounds__(1024) void k_bin_small(DevView v, double drift_dt, int do_drift, int atom_id_order)
{
    constexpr int T = 1024, PT = kBinSmall / T;
    __shared__ int cnt[kBinSmall], key[kBinSmall], wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int N = v.Ntot, nc = v.Ctot;
#pragma unroll
    for (int k = 0; k < PT; k++) cnt[k * T + tid] = 0;
    double x3[PT][3];
    int cell[PT], slot[PT], mykey[PT], chain[PT];
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int a = k * T + tid;
        if (a >= N) continue;
        chain[k] = v.atom_chain[a];
        mykey[k] = atom_id_order ? a : v.invperm[a];
        const ChainDev& C = v.chains[chain[k]];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double xv = v.x[d * N + a];
            if (do_drift) {
                xv += drift_dt * C.coeff_x * v.p[d * N + a];
                xv = lp_round(xv, v.lp_scale);
                xv = wrap_box(xv, C.L[d]);
                v.x[d * N + a] = xv;
            }
            x3[k][d] = xv;
        }
        cell[k] = cell_index(C, x3[k]);
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
    if (tid == 0 && nc == kBinSmall) offs[nc] = N;
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
        const ChainDev& C = v.chains[chain[k]];
        double o[3];
        cell_origin(C, cell[k], o);
        const int beg = cnt[cell[k]], end = cell[k] + 1 < kBinSmall ? cnt[cell[k] + 1] : N;
        int rank = 0;
#pragma unroll 4
        for (int q = beg; q < end; q++) rank += key[q] < mykey[k] ? 1 : 0;
        place_atom(v, perm_n, beg + rank, a, x3[k], o);
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
    hipLaunchKernelGGL(k_bin_small, dim3(1), dim3(1024), 0, s, v, drift_dt, drift_dt != 0.0 ? 1 : 0, atom_id_order ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_drift(const DevView& v, double dt, hipStream_t s)
{
    hipLaunchKernelGGL(k_drift, dim3((v.Ntot + 255) / 256), dim3(256), 0, s, v, dt);
    return hipGetLastError();
}

}  // namespace chmc
