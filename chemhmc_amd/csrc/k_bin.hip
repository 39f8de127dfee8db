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
//   k_cell_rank      : 16 lanes per cell, or for a cell of many atoms a workgroup, rank its entries by key -> the
//                      stable order
//   k_bin_small      : all of it in one workgroup's LDS for small contexts
// The placement writes the next perm/offs buffers, invperm and the sorted coordinates (FP64, and FP32 relative
// to the cell); the host then flips the parity argument that selects the current buffers.
#include "chmc_internal.hpp"
#include "bin_device.hpp"

#include <climits>

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

// Ranks of a cell's n entries by a whole workgroup of 256 threads, where 16 lanes that compare every pair would
// take long (n^2 / 16 loads a lane: a binning of 100,000 atoms in 125 cells 1.3 ms, in 27 cells 19 ms, 5,000
// atoms of which 2,900 share a cell 8.4 ms; this way 33, 54 and 42 us, the launches of a sparse binning being 31).
// Up to kRankTile entries, the pairwise count from LDS, n^2 / 256 compares a thread; or a bit for each key in a
// window of kRankWindow keys, set, counted by prefix, the rank of an entry the bits below its own: linear in n and in
// the range of keys (the previous slots of a cell's atoms are near each other, so that one or two windows hold them;
// atom ids range over Ntot).  A window costs about the pairwise count of 362 entries (six barriers, 16 KB of LDS
// written and read).
constexpr int kRankWindow = 65536, kRankTile = 4096;
__device__ __forceinline__ void rank_dense(const DevView& v, int* perm_n, int beg, int n, const double o[3], int (&lds)[kRankTile],
                                           int (&part)[8])
{
    const int N = v.Ntot, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    auto place = [&](int e, int rank) {
        const int atom = v.satom[beg + e];
        const double x3[3] = { v.x[atom], v.x[N + atom], v.x[2 * N + atom] };
        place_atom(v, perm_n, beg + rank, atom, x3, o);
    };
    int lo = INT_MAX, hi = 0;
#pragma unroll 8
    for (int e = tid; e < n; e += 256) {
        const int k = v.skey[beg + e];
        lo = min(lo, k);
        hi = max(hi, k);
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        lo = min(lo, __shfl_xor(lo, m, 64));
        hi = max(hi, __shfl_xor(hi, m, 64));
    }
    __syncthreads();                                       // lds and part free
    if (lane == 0) {
        part[wid] = lo;
        part[4 + wid] = hi;
    }
    __syncthreads();
    lo = min(min(part[0], part[1]), min(part[2], part[3]));
    hi = max(max(part[4], part[5]), max(part[6], part[7]));
    const int windows = (hi - lo) / kRankWindow + 1;
    if (n <= kRankTile && n * n / 131072 < windows) {
        for (int t = tid; t < (n + 3) / 4 * 4; t += 256) lds[t] = t < n ? v.skey[beg + t] : INT_MAX;
        __syncthreads();
        for (int e = tid; e < n; e += 256) {
            const int key = lds[e];
            int rank = 0;
            for (int q = 0; q < n; q += 4) {
                const int4 k4 = *reinterpret_cast<const int4*>(&lds[q]);
                rank += (k4.x < key ? 1 : 0) + (k4.y < key ? 1 : 0) + (k4.z < key ? 1 : 0) + (k4.w < key ? 1 : 0);
            }
            place(e, rank);
        }
        return;
    }
    static_assert(kRankWindow / 32 == 8 * 256 && kRankTile >= kRankWindow / 16, "8 words a thread");
    unsigned* bits = reinterpret_cast<unsigned*>(lds);     // the bits, then for each word the ranks before it
    int* pre = lds + kRankWindow / 32;
    int before = 0;
    for (int w = 0; w < windows; w++) {
        const int base = lo + w * kRankWindow;
        __syncthreads();                                   // lds and part free
#pragma unroll
        for (int u = 0; u < 8; u++) bits[u * 256 + tid] = 0u;
        __syncthreads();
#pragma unroll 8
        for (int e = tid; e < n; e += 256) {
            const unsigned k = (unsigned)(v.skey[beg + e] - base);
            if (k < (unsigned)kRankWindow) atomicOr(&bits[k >> 5], 1u << (k & 31u));
        }
        __syncthreads();
        int s = 0, c8[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            c8[u] = s;
            s += __popc(bits[8 * tid + u]);
        }
        int incl = s;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const int t = __shfl_up(incl, m, 64);
            if (lane >= m) incl += t;
        }
        if (lane == 63) part[wid] = incl;
        __syncthreads();
        int run = before + incl - s;
        for (int k = 0; k < wid; k++) run += part[k];
#pragma unroll
        for (int u = 0; u < 8; u++) pre[8 * tid + u] = run + c8[u];
        before += part[0] + part[1] + part[2] + part[3];
        __syncthreads();
        // two entries a thread together: the loads of the second ahead of the first one's stores
        constexpr int U = 2;
        for (int e0 = tid; e0 < n; e0 += 256 * U) {
            unsigned k[U];
            int atom[U];
            double x[U][3];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = beg + min(e0 + 256 * u, n - 1);
                k[u] = (unsigned)(v.skey[e] - base);
                atom[u] = v.satom[e];
            }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int d = 0; d < 3; d++) x[u][d] = v.x[(size_t)d * N + atom[u]];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (e0 + 256 * u < n && k[u] < (unsigned)kRankWindow)
                    place_atom(v, perm_n, beg + pre[k[u] >> 5] + __popc(bits[k[u] >> 5] & ((1u << (k[u] & 31u)) - 1u)), atom[u], x[u], o);
        }
    }
}

// 16 lanes per cell, each entry's position is its rank among the cell's (unique) keys; cells of more than
// kDenseCell atoms by the whole workgroup (rank_dense).  A workgroup has 16 cells, or PER = 1 in contexts of
// kDenseMean atoms a cell and more, whose dense cells would otherwise wait for each other.
constexpr int kDenseCell = 64, kDenseMean = 32;
template <int PER>
__global__ __launch_bounds__(256, 8) void k_cell_rank(DevView v)
{
    __shared__ alignas(16) int lds[kRankTile];
    __shared__ int part[8];
    const int c = blockIdx.x * PER + (PER == 1 ? 0 : threadIdx.x >> 4);
    const int sub = PER == 1 ? threadIdx.x : threadIdx.x & 15;
    const int N = v.Ntot;
    const int* offs = offs_next(v);
    int* perm_n = perm_next(v);
    bool dense = false;
    if (c < v.Ctot) {
        const int beg = offs[c];
        const int n = offs[c + 1] - beg;
        dense = n > kDenseCell;
        const ChainDev& C = v.chains[v.cell_chain[c]];
        double o[3];
        cell_origin(C, c, o);
        for (int e = dense ? n : sub; e < n; e += 256 / PER) {
            const int key = v.skey[beg + e];
            const int atom = v.satom[beg + e];
            const double x3[3] = { v.x[atom], v.x[N + atom], v.x[2 * N + atom] };
            int rank = 0;
#pragma unroll 8
            for (int q = 0; q < n; q++) rank += (v.skey[beg + q] < key) ? 1 : 0;
            place_atom(v, perm_n, beg + rank, atom, x3, o);
        }
    }
    if (__syncthreads_or(dense) == 0) return;
    for (int k = 0; k < PER; k++) {
        const int c = blockIdx.x * PER + k;
        if (c >= v.Ctot) break;
        const int beg = offs[c];
        const int n = offs[c + 1] - beg;
        if (n <= kDenseCell) continue;
        double o[3];
        cell_origin(v.chains[v.cell_chain[c]], c, o);
        rank_dense(v, perm_n, beg, n, o, lds, part);
    }
}

// The whole binning of a context of at most kBinSmall atoms and cells in one workgroup: counts, their scan and
// the sort keys stay in LDS, each thread keeps its (up to three) atoms.  Four launches of a few microseconds of
// latency each otherwise: N = 512, FP64 leapfrog, count + scan + placement took 21 us an evaluation, now
// 4.9.  Bound: latency (three global round trips, six barriers), and one CU's instructions from about 2000 atoms
// on: an FP64 leapfrog step of 2,744 atoms takes 18.5 us with it and 22.4 without, of 4,096 29.7 (before the loads
// were brought together) and 24.1.  Up to 512 atoms and cells, 512 threads with an atom each: 11.2 -> 10.9 us a step
// of N = 512; contexts beyond take 1024 threads with up to three atoms each, also those of 513 to 1024, for which an
// instance of one atom a thread has not been measured.
// Cells of more than kSmallDense atoms (clustered systems, or those of few cells) follow at the end and rank their
// keys by a bit for each, in the cell's own part of key[] (16 KB more LDS made a step of 2,744 atoms 1 % longer):
// 3000 atoms in one cell, pairwise 217 us a binning, now 26.  The test for them costs 0.2 of the 20 us a step of
// 2,744 atoms takes.  Contexts of up to 512 atoms go without: all of them in one cell, ranked pairwise, take 24 us a
// binning against 15 spread out, and the test would cost each step 0.1 of 10.9 us.
constexpr int kSmallDense = 160;
template <int T, int PT>
__global__ __launch_bounds__(T) void k_bin_small(DevView v, double drift_dt, int do_drift, int atom_id_order)
{
    constexpr int kMax = T * PT, kWords = kMax / 32;
    constexpr bool kDenseToo = PT > 1;
    static_assert(kWords + kWords / 2 <= kSmallDense, "the bits and their counts before each word, in 16 bits");
    __shared__ int cnt[kMax], key[kMax], wsum[T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
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
    int c4[PT], s = 0, most = 0;
#pragma unroll
    for (int k = 0; k < PT; k++) {
        c4[k] = cnt[tid * PT + k];
        s += c4[k];
        most = max(most, c4[k]);
    }
    const bool dense_wave = kDenseToo && __ballot(most > kSmallDense) != 0ull;
    int incl = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    if (lane == 63) wsum[wid] = incl | (dense_wave ? 1 << 16 : 0);
    __syncthreads();
    bool dense = false;                    // in any wave
    int run = incl - s;
    if constexpr (kDenseToo) {
        const int ws = wsum[lane & (T / 64 - 1)];
        dense = __ballot(ws >> 16 != 0) != 0ull;
        for (int w = 0; w < wid; w++) run += __builtin_amdgcn_readlane(ws, w) & 0xffff;
    } else {
        for (int w = 0; w < wid; w++) run += wsum[w];
    }
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
    auto end_of = [&](int k) { return cell[k] + 1 < kMax ? cnt[cell[k] + 1] : N; };
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int a = k * T + tid;
        if (a >= N) continue;
        const int beg = cnt[cell[k]], end = end_of(k);
        if (kDenseToo && end - beg > kSmallDense) continue;
        int rank = 0;
#pragma unroll 4
        for (int q = beg; q < end; q++) rank += key[q] < mykey[k] ? 1 : 0;
        place_atom(v, perm_n, beg + rank, a, x3[k], o3[k]);
    }
    if (!kDenseToo || !dense) return;
    // f(begin) for every dense cell, by the wave of the thread that scanned it
    auto dense_cells = [&](auto f) {
#pragma unroll
        for (int k = 0; k < PT; k++)
            for (unsigned long long m = __ballot(c4[k] > kSmallDense); m != 0ull; m &= m - 1ull)
                f(__shfl(cnt[tid * PT + k], __ffsll((long long)m) - 1, 64));
    };
    dense_cells([&](int beg) {
        for (int w = lane; w < kWords; w += 64) key[beg + w] = 0;
    });
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PT; k++) {
        if (k * T + tid >= N) continue;
        const int beg = cnt[cell[k]];
        if (end_of(k) - beg > kSmallDense) atomicOr(&key[beg + (mykey[k] >> 5)], (int)(1u << (mykey[k] & 31)));
    }
    __syncthreads();
    dense_cells([&](int beg) {
        int before = 0;
        for (int w0 = 0; w0 < kWords; w0 += 64) {
            const int n = w0 + lane < kWords ? __popc((unsigned)key[beg + w0 + lane]) : 0;
            int incl = n;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int t = __shfl_up(incl, o, 64);
                if (lane >= o) incl += t;
            }
            if (w0 + lane < kWords) reinterpret_cast<unsigned short*>(key + beg + kWords)[w0 + lane] = (unsigned short)(before + incl - n);
            before += __shfl(incl, 63, 64);
        }
    });
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int a = k * T + tid;
        if (a >= N) continue;
        const int beg = cnt[cell[k]], w = mykey[k] >> 5;
        if (end_of(k) - beg <= kSmallDense) continue;
        const int rank = reinterpret_cast<const unsigned short*>(key + beg + kWords)[w] +
                         __popc((unsigned)key[beg + w] & ((1u << (mykey[k] & 31)) - 1u));
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
    if (v.Ntot / kDenseMean >= v.Ctot) hipLaunchKernelGGL(k_cell_rank<1>, dim3(v.Ctot), dim3(256), 0, s, v);
    else hipLaunchKernelGGL(k_cell_rank<16>, dim3((v.Ctot + 15) / 16), dim3(256), 0, s, v);
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
