// Device helpers shared by the kernels that bin atoms (k_bin.hip, and the fused drift + count of the
// FP32 force sweep and of the heat bath): cell index with the reference's floor(x / sizebin)
// (particles.hpp:108-113) clamped to the grid, the count phase of one atom and the one-workgroup exclusive scan of
// the per-cell counts.
#pragma once
#include "chmc_internal.hpp"

namespace chmc {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Exclusive scan of the per-cell counts into the next offsets (and the counts cleared), by one
// workgroup of 1024 threads: rounds of 8192 counts are loaded into LDS with coalesced reads, each thread
// scans 8 contiguous ones, a block scan over the threads and a running carry join the rounds, and the
// offsets go back with coalesced writes.
__device__ inline void scan_counts_block(const DevView& v)
{
    constexpr int T = 1024, PT = 8;
    __shared__ int buf[T * PT];
    __shared__ int wsum[16];
    __shared__ int carry;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int n = v.Ctot;
    int* count = v.count;
    int* offs = offs_next(v);
    if (tid == 0) carry = 0;
    for (int r0 = 0; r0 < n; r0 += T * PT) {
#pragma unroll
        for (int k = 0; k < PT; k++) {
            const int c = r0 + k * T + tid;
            buf[k * T + tid] = c < n ? count[c] : 0;
        }
        __syncthreads();
        int vals[PT];
        int s = 0;
#pragma unroll
        for (int k = 0; k < PT; k++) {
            vals[k] = buf[tid * PT + k];
            s += vals[k];
        }
        int incl = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        if (wid == 0) {
            int w = lane < 16 ? wsum[lane] : 0;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                const int t = __shfl_up(w, o, 64);
                if (lane >= o) w += t;
            }
            if (lane < 16) wsum[lane] = w;
        }
        __syncthreads();
        int run = carry + incl - s + (wid > 0 ? wsum[wid - 1] : 0);
#pragma unroll
        for (int k = 0; k < PT; k++) {
            buf[tid * PT + k] = run;
            run += vals[k];
        }
        __syncthreads();                      // every thread has read carry; buf holds the round's scan
        if (tid == T - 1) carry = run;
#pragma unroll
        for (int k = 0; k < PT; k++) {
            const int c = r0 + k * T + tid;
            if (c < n) {
                offs[c] = buf[k * T + tid];
                count[c] = 0;
            }
        }
        __syncthreads();                      // buf free, carry final
    }
    if (tid == 0) offs[n] = carry;
}

// cell of a position, and its grid coordinates b (C: the chain, or the members of it that are used here)
template <typename Grid>
__device__ __forceinline__ int cell_index(const Grid& C, const double x3[3], int b[3])
{
#pragma unroll
    for (int d = 0; d < 3; d++) b[d] = clampi((int)floor(x3[d] / C.sizebin[d]), 0, C.nbin[d] - 1);
    return C.cell_off + b[0] + C.nbin[0] * (b[1] + b[2] * C.nbin[1]);
}

// Count phase of one atom at its current position (any drift already applied): its cell and its arrival slot
// there.  One atomic per distinct cell among the wave's active lanes, all issued together (one after another,
// each waiting for the last, they made the count of 250,047 atoms 23.6 us; with the rest of its loads now 11.6).  The
// arrival slot only has to be unique within the cell: the placement ranks the cell's entries by key.
__device__ __forceinline__ void count_atom(const DevView& v, int cell, int a)
{
    v.cell_of[a] = cell;
    const int lane = threadIdx.x & 63;
    unsigned long long left = __ballot(1);
    int lead = lane, rank = 0, size = 1;
    while (left) {
        const int l = __ffsll((long long)left) - 1;
        const unsigned long long m = __ballot(cell == __builtin_amdgcn_readlane(cell, l)) & left;
        if ((m >> lane) & 1ull) {
            lead = l;
            rank = __popcll(m & ((1ull << lane) - 1ull));
            size = __popcll(m);
        }
        left &= ~m;
    }
    int base = 0;
    if (lane == lead) base = atomicAdd(&v.count[cell], size);
    v.slot[a] = __shfl(base, lead, 64) + rank;
}
__device__ __forceinline__ void count_atom(const DevView& v, const ChainDev& C, int a, const double x3[3])
{
    int b[3];
    count_atom(v, cell_index(C, x3, b), a);
}

}  // namespace chmc
