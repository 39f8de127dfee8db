// Lennard-Jones sweep over the 27 neighbour cells: the replacement of Tag_force_binning
// (code/modules/identical_particles.cpp:567-639), Tag_potential_binning (:395-454) and the kick of
// update_momenta (:676-694), with a pair virial the reference does not have.
//
// Both sweeps run one workgroup per i-cell: lanes 0..26 of wave 0 resolve the 27 neighbour cells (with the
// reference's explicit image shift when the neighbour index wraps, :584-600), a prefix sum gives the
// concatenated j-list, and all threads stage it into LDS at once (binary search of the segment, one load
// each, all in flight together), with the image shift folded into the staged coordinates.
// FP32 sweep (k_lj): inside a wave, lanes are IS i-slots x (64/IS) j-groups (lane = g*IS + ii): i-atom ii of
//   the wave's current i-chunk against every (64/IS)-th j entry, one broadcast LDS read per pair; waves
//   take i-chunks round-robin; a butterfly over the j-groups sums the partials.  Coordinates relative to the
//   cell origin (|d| < 2 cell sides), per-atom FP32 sums, +grad U stored and/or the FP64 momenta kicked in
//   place (p -= (dt*beta)*f).  LJ_DRIFT: right after its kick each atom also takes the integrator's next
//   drift and is counted into its new cell (the count phase of the next binning).
//   Self-exclusion is r^2 > 0: the staged copy of atom i is bitwise equal to its own coordinates.
// FP64 sweep (k_lj64): see there.
#include "chmc_internal.hpp"
#include "bin_device.hpp"

#pragma clang fp contract(off)   // the kick must round like the oracle's p -= dt*c*f

namespace chmc {

__device__ __forceinline__ int xcd_remap(int b, int nblocks)
{
    // blocks are dispatched round-robin over the 8 XCDs; give each XCD a contiguous range of cells
    // so that neighbouring cells share one L2.
    const int per = nblocks >> 3;
    return (b & 7) * per + (b >> 3);
}

__device__ __forceinline__ double rcp64(double r2)
{
    double y = __builtin_amdgcn_rcp(r2);
    double e = __builtin_fma(-r2, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-r2, y, 1.0);
    return __builtin_fma(y, e, y);
}
template <int IS, int kWaves, int MODE>
__global__ __launch_bounds__(64 * kWaves) void k_lj(DevView v, double kick_dt, double drift_dt, int nblocks)
{
    constexpr int JG = 64 / IS;
    constexpr int NT = 64 * kWaves;
    __shared__ float4 sj[kMaxJ];
    __shared__ int seg_beg[27];
    __shared__ int seg_pref[28];
    __shared__ float seg_sh[27][3];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int c = xcd_remap(blockIdx.x, nblocks);
    if (c < v.Ctot) {
    const int ch = v.cell_chain[c];
    const ChainDev& C = v.chains[ch];
    const int nx = C.nbin[0], ny = C.nbin[1], nz = C.nbin[2];
    const int lc = c - C.cell_off;
    const int bz = lc / (nx * ny);
    const int by = (lc - bz * nx * ny) / nx;
    const int bx = lc - nx * (by + bz * ny);
    const int* offs = offs_cur(v);
    const int ibeg = offs[c];
    const int ni = offs[c + 1] - ibeg;
    const int N = v.Ntot;

    if (ni > 0) {
        // ---- 1. neighbour segments -----------------------------------------------------------
        if (wave == 0) {
            int cnt = 0;
            if (lane < 27) {
                const int dd[3] = { lane % 3 - 1, (lane / 3) % 3 - 1, lane / 9 - 1 };
                const int b3[3] = { bx, by, bz };
                const int n3[3] = { nx, ny, nz };
                int j3[3];
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    j3[d] = b3[d] + dd[d];
                    if (j3[d] < 0 || j3[d] >= n3[d]) j3[d] = (b3[d] + n3[d] + dd[d]) % n3[d];
                    // staged = (x_j - o_j) + dd*s: the j cell's origin seen from the i cell's origin
                    seg_sh[lane][d] = (float)dd[d] * C.sizebin_f[d];
                }
                const int jc = C.cell_off + j3[0] + nx * (j3[1] + j3[2] * ny);
                const int o0 = offs[jc];
                seg_beg[lane] = o0;
                cnt = offs[jc + 1] - o0;
            }
            int incl = cnt;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                int t = __shfl_up(incl, o, 64);
                if (lane >= o) incl += t;
            }
            if (lane < 27) seg_pref[lane + 1] = incl;
            if (lane == 0) seg_pref[0] = 0;
        }
        __syncthreads();
        const int nj = seg_pref[27];

        // ---- 2. staging of j-list entries [jlo, jhi): every thread, binary search of its segment ----
        auto stage = [&](int jlo, int jhi) {
            for (int t = jlo + tid; t < jhi; t += NT) {
                int k = 0;
#pragma unroll
                for (int step = 16; step > 0; step >>= 1)
                    if (k + step < 27 && seg_pref[k + step] <= t) k += step;
                const int src = seg_beg[k] + (t - seg_pref[k]);
                const float4 q = v.xs[src];
                sj[t - jlo] = make_float4(q.x + seg_sh[k][0], q.y + seg_sh[k][1], q.z + seg_sh[k][2], 0.f);
            }
        };
        const bool single = nj <= kMaxJ;
        if (single) {
            stage(0, nj);
            __syncthreads();
        }

        // ---- 3. i-chunks (round-robin over waves) x j-groups ----------------------------------------
        const int ii = lane % IS, g = lane / IS;
        const float rc2 = C.rc2_f, sig2 = C.sigma2_f;
        const int nchunk = (ni + IS - 1) / IS;
        // every wave runs the same number of chunk iterations so that the multi-pass staging barriers match
        const int rounds = (nchunk + kWaves - 1) / kWaves;
        for (int rnd = 0; rnd < rounds; rnd++) {
            const int chunk = rnd * kWaves + wave;
            const int i = chunk * IS + ii;
            const bool ival = i < ni;
            const int ic = ival ? i : ni - 1;
            const float4 xi = v.xs[ibeg + ic];
            const int atom = __float_as_int(xi.w);
            float ax = 0.f, ay = 0.f, az = 0.f;
            for (int jlo = 0; jlo < nj; jlo += kMaxJ) {
                const int jhi = min(nj, jlo + kMaxJ);
                if (!single) {
                    __syncthreads();
                    stage(jlo, jhi);
                    __syncthreads();
                }
                const int jn = (chunk < nchunk) ? jhi - jlo : 0;
#pragma unroll 4
                for (int j = g; j < jn; j += JG) {
                    const float4 q = sj[j];
                    const float dx = xi.x - q.x, dy = xi.y - q.y, dz = xi.z - q.z;
                    const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                    const bool in = (r2 < rc2) && (r2 > 0.f);
                    const float inv = __builtin_amdgcn_rcpf(r2);
                    const float s2 = sig2 * inv;
                    const float s6 = s2 * s2 * s2;
                    float gq = s6 * (0.5f - s6) * inv;           // sr6 (0.5 - sr6) / r^2, :611-613
                    gq = in ? gq : 0.f;
                    ax = __builtin_fmaf(gq, dx, ax);
                    ay = __builtin_fmaf(gq, dy, ay);
                    az = __builtin_fmaf(gq, dz, az);
                }
            }
            if (chunk >= nchunk) continue;   // wave-uniform
            // butterfly over the j-groups (lanes ii, ii+IS, ...): every lane ends with the i-atom total
#pragma unroll
            for (int m = IS; m < 64; m <<= 1) {
                ax += __shfl_xor(ax, m, 64);
                ay += __shfl_xor(ay, m, 64);
                az += __shfl_xor(az, m, 64);
            }
            {
                if (g == 0 && ival) {
                    const float f3[3] = { C.eps48_f * ax, C.eps48_f * ay, C.eps48_f * az };
                    const double kdt = kick_dt * C.beta;     // dt * coeff_p, coeff_p = beta (:642-644)
                    double pn[3];
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        if constexpr ((MODE & LJ_STOREF) != 0) v.f32[d * N + atom] = f3[d];
                        if constexpr ((MODE & LJ_KICK) != 0) {
                            const double fd = (double)f3[d];
                            pn[d] = lp_round(v.p[d * N + atom] - kdt * fd, v.lp_scale);
                            v.p[d * N + atom] = pn[d];
                        }
                    }
                    if constexpr ((MODE & LJ_DRIFT) != 0) {
                        // the following update_positions (identical_particles.cpp:651-669) of this atom,
                        // then the count phase of the next binning at its new position
                        const double coeff_x = C.coeff_x;
                        double x3[3];
#pragma unroll
                        for (int d = 0; d < 3; d++) {
                            double xv = v.x[d * N + atom];
                            xv += drift_dt * coeff_x * pn[d];
                            xv = lp_round(xv, v.lp_scale);
                            xv = wrap_box(xv, C.L[d]);
                            v.x[d * N + atom] = xv;
                            x3[d] = xv;
                        }
                        count_atom(v, C, atom, x3);
                    }
                }
            }
        }
    }
    }   // c < Ctot
}

// ---- FP64 sweep ------------------------------------------------------------------------------------
// One workgroup of W wavefronts per i-cell, or `parts` of them (forces), one wave per i-atom.  The 64 lanes test 64
// staged j entries a step (FP64 coordinates relative to the i-cell origin, r^2 < rc^2), and the pairs inside (14 % of the candidates
// at liquid density) are appended by ballot prefix to the wave's LDS list; whenever 64 are pending, and at the
// end, the lanes take one each and evaluate it: reciprocal from v_rcp_f64 with two Newton steps, per-lane sums.
//   LJ_FORCE: a butterfly over the wave sums the three components per atom; lanes 0..2 store and kick.
//   LJ_ENERGY: per-lane energy, virial and pair sums run on over the wave's atoms (and the kinetic energy over
//   the cell's atoms); reduced once in a fixed order into per-cell partials that the chain reduction sums.
// Self-exclusion is r^2 > 0: the i-atom is its own staged copy.
// Bound: VALU issue of the tests (12 instructions per 64 candidates, the next step's entries loaded ahead; r^2 > 0 is
// tested with the pairs inside only, entries are LDS byte offsets) and the workgroups' start at large N, latency at
// small N.  Evaluating every candidate, 8 i-slots x 8 j-groups a wave, took 23.4 us at N = 512 (27 cells: chains
// of 128 dependent iterations) and 169 us for the energy at N = 250,047; one wave per atom 8.7 us (kick) and 110 us;
// the tests' shorter steps (16 instructions before) 106 us there, and 0.5 us of a leapfrog step at N = 512.
// An FP32 copy of the entries for the tests cost more in LDS (6 instead of 8 workgroups a CU) than its narrower
// reads saved (118 us there).
// Forces of up to kWideCells cells: workgroups of 8 waves, and so many per cell that a wave has one atom (1.3 times
// the mean occupancy), as long as the launch stays within kForceGroups, two rounds of 2 a CU: 16 waves for each of
// 27 cells used a tenth of the CUs, and most waves ran a second atom after the first.  A leapfrog step of the FP64
// path (with its binning): N = 256 23.2 -> 13.7 us, 512 14.1 -> 12.4, 800 24.4 -> 15.6; 8,000 (512 cells, two each
// instead of one of four waves) 30.2 -> 26.4, 16,384 36.0 -> 32.4.  From 2,197 cells on the chip is full and four
// waves are as fast (42.8 against 42.2 us), from 4,096 faster (58.1 against 61.5).
// Energies need a cell's sums in one workgroup: 16 waves below kSmallCells cells, else 4.
constexpr int kWideCells = 2048, kForceGroups = 1024;
constexpr int kSmallCells = 512;
constexpr int kMaxJ64 = 512;          // j entries per LDS pass, 17 KB: nine workgroups of four waves fit a CU, its wave slots take eight

template <int W, int MODE>
__global__ __launch_bounds__(64 * W) void k_lj64(DevView v, double kick_dt, int parts)
{
    constexpr int NT = 64 * W, PEND = 128;
    constexpr double kFar2 = 1.0e300;     // its twelfth power underflows: no contribution
    auto at8 = [](const double* a, unsigned j8) { return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(a) + j8); };
    __shared__ double sx[kMaxJ64 + 128], sy[kMaxJ64 + 128], sz[kMaxJ64 + 128];     // padded with far entries
    __shared__ unsigned short pend[W][PEND];
    __shared__ int seg_beg[27], seg_pref[28];
    __shared__ double seg_sh[27][3];
    __shared__ double wsum[W][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int item = xcd_block(blockIdx.x, v.Ctot * parts), c = item / parts, first = (item - c * parts) * W, step = W * parts;
    const ChainDev& C = v.chains[v.cell_chain[c]];
    const int nx = C.nbin[0], ny = C.nbin[1], nz = C.nbin[2];
    const int lc = c - C.cell_off;
    const int bz = lc / (nx * ny), by = (lc - bz * nx * ny) / nx, bx = lc - nx * (by + bz * ny);
    const int* offs = offs_cur(v);
    const int ibeg = offs[c];
    const int ni = offs[c + 1] - ibeg;
    const int N = v.Ntot;
    double au = 0.0, aw = 0.0, ak = 0.0;
    int an = 0;
    if (ni > first) {
        if (wave == 0) {
            int cnt = 0;
            if (lane < 27) {
                const int dd[3] = { lane % 3 - 1, (lane / 3) % 3 - 1, lane / 9 - 1 };
                const int b3[3] = { bx, by, bz }, n3[3] = { nx, ny, nz };
                int j3[3];
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    j3[d] = b3[d] + dd[d];
                    const bool wrapped = j3[d] < 0 || j3[d] >= n3[d];
                    if (wrapped) j3[d] = (b3[d] + n3[d] + dd[d]) % n3[d];
                    // FP64: x_j + wrap - o_i, wrap = dd*L only when the index wrapped
                    seg_sh[lane][d] = (wrapped ? dd[d] * C.L[d] : 0.0) - b3[d] * C.sizebin[d];
                }
                const int jc = C.cell_off + j3[0] + nx * (j3[1] + j3[2] * ny);
                seg_beg[lane] = offs[jc];
                cnt = offs[jc + 1] - offs[jc];
            }
            int incl = cnt;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const int t = __shfl_up(incl, o, 64);
                if (lane >= o) incl += t;
            }
            if (lane < 27) seg_pref[lane + 1] = incl;
            if (lane == 0) seg_pref[0] = 0;
        }
        __syncthreads();
        const int nj = seg_pref[27];
        auto stage = [&](int jlo, int jhi) {
            for (int t = jlo + tid; t < jhi; t += NT) {
                int k = 0;
#pragma unroll
                for (int step = 16; step > 0; step >>= 1)
                    if (k + step < 27 && seg_pref[k + step] <= t) k += step;
                const int src = seg_beg[k] + (t - seg_pref[k]);
                sx[t - jlo] = v.xs64[src] + seg_sh[k][0];
                sy[t - jlo] = v.xs64[(size_t)N + src] + seg_sh[k][1];
                sz[t - jlo] = v.xs64[2 * (size_t)N + src] + seg_sh[k][2];
            }
            if (tid < 128) sx[jhi - jlo + tid] = sy[jhi - jlo + tid] = sz[jhi - jlo + tid] = (double)kFarShift;
        };
        const bool single = nj <= kMaxJ64;
        if (single) {
            stage(0, nj);
            __syncthreads();
        }
        const double rc2 = C.rc2, sig2 = C.sigma2;
        const double kdt = kick_dt * C.beta;              // dt * coeff_p, coeff_p = beta (:642-644)
        // every wave runs the same number of rounds so that the multi-pass staging barriers match
        const int rounds = (ni - first + step - 1) / step;
        for (int rnd = 0; rnd < rounds; rnd++) {
            const int i = rnd * step + first + wave;
            const bool ival = i < ni;                     // wave-uniform
            // the i-atom: its own staged copy (segment 13) where the whole j-list is staged
            double xi, yi, zi;
            if (single) {
                const int own = seg_pref[13] + (ival ? i : 0);
                xi = sx[own];
                yi = sy[own];
                zi = sz[own];
            } else {
                const int slot = ibeg + (ival ? i : 0);
                xi = v.xs64[slot] + seg_sh[13][0];
                yi = v.xs64[(size_t)N + slot] + seg_sh[13][1];
                zi = v.xs64[2 * (size_t)N + slot] + seg_sh[13][2];
            }
            int atom = 0;
            if constexpr ((MODE & LJ_FORCE) != 0) atom = perm_cur(v)[ibeg + (ival ? i : 0)];
            double p_d = 0.0;
            if constexpr ((MODE & LJ_KICK) != 0) p_d = v.p[(size_t)min(lane, 2) * N + atom];
            double ax = 0.0, ay = 0.0, az = 0.0;
            // the pending pair of this lane; the i-atom itself and coincident ones (r^2 = 0) count as far away
            auto evaluate = [&](bool on) {
                const unsigned j8 = pend[wave][on ? lane : 0];
                const double dx = xi - at8(sx, j8), dy = yi - at8(sy, j8), dz = zi - at8(sz, j8);
                double r2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
                on = on && r2 > 0.0;
                r2 = on ? r2 : kFar2;
                const double inv = rcp64(r2);
                const double s2 = sig2 * inv;
                const double s6 = s2 * s2 * s2;
                if constexpr ((MODE & LJ_FORCE) != 0) {
                    const double gq = s6 * (0.5 - s6) * inv;                 // sr6 (0.5 - sr6) / r^2, :611-613
                    ax = __builtin_fma(gq, dx, ax);
                    ay = __builtin_fma(gq, dy, ay);
                    az = __builtin_fma(gq, dz, az);
                }
                if constexpr ((MODE & LJ_ENERGY) != 0) {
                    au += s6 * (s6 - 1.0);
                    aw += s6 * (s6 - 0.5);
                    an += on ? 1 : 0;
                }
            };
            auto lds_sync = [&]() {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            };
            for (int jlo = 0; jlo < nj; jlo += kMaxJ64) {
                const int jn = min(nj, jlo + kMaxJ64) - jlo;
                if (!single) {
                    __syncthreads();
                    stage(jlo, jlo + jn);
                    __syncthreads();
                }
                if (!ival) continue;
                int np = 0;
                unsigned j8 = 8u * (unsigned)lane;
                double px = at8(sx, j8), py = at8(sy, j8), pz = at8(sz, j8);
                for (int j0 = 0; j0 < jn; j0 += 64) {
                    const double dx = xi - px, dy = yi - py, dz = zi - pz;
                    const unsigned t8 = j8;
                    j8 += 512u;                           // the next step's entries (the padding after the last)
                    px = at8(sx, j8);
                    py = at8(sy, j8);
                    pz = at8(sz, j8);
                    const double r2 = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
                    const unsigned long long m = __builtin_amdgcn_fcmp(r2, rc2, 4);            // ordered less
                    const unsigned pos = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                    if (r2 < rc2) (pend[wave] + np)[pos] = (unsigned short)t8;
                    np += __popcll(m);
                    if (np >= 64) {                       // np - 64 < 64 stay pending
                        lds_sync();
                        evaluate(true);
                        const unsigned short rest = pend[wave][64 + lane];
                        lds_sync();
                        pend[wave][lane] = rest;
                        np -= 64;
                    }
                }
                lds_sync();
                if (np > 0) evaluate(lane < np);
                lds_sync();                               // read before the next atom's candidates replace them
            }
            if constexpr ((MODE & LJ_FORCE) != 0) {
                if (!ival) continue;
                auto wave_sum = [](double s) {
                    s = group_sum<16>(s);
                    s += __shfl_xor(s, 16, 64);
                    return s + __shfl_xor(s, 32, 64);
                };
                ax = wave_sum(ax);
                ay = wave_sum(ay);
                az = wave_sum(az);
                if (lane < 3) {
                    const double fd = (lane == 0 ? ax : (lane == 1 ? ay : az)) * (48 * C.eps);
                    if constexpr ((MODE & LJ_STOREF) != 0) v.f64[(size_t)lane * N + atom] = fd;
                    if constexpr ((MODE & LJ_KICK) != 0) v.p[(size_t)lane * N + atom] = lp_round(p_d - kdt * fd, v.lp_scale);
                }
            }
        }
        if constexpr ((MODE & LJ_ENERGY) != 0) {
            // kinetic energy: every atom is an i-atom exactly once (K_f, HMC.cpp:90)
            for (int i = tid; i < ni; i += NT) {
                const int atom = perm_cur(v)[ibeg + i];
                const double px = v.p[atom], py = v.p[(size_t)N + atom], pz = v.p[2 * (size_t)N + atom];
                ak += (px * px + py * py + pz * pz) / (2 * C.mass);
            }
        }
    }
    if constexpr ((MODE & LJ_ENERGY) != 0) {
        // per-lane sums through LDS (the staged positions are done with): wave k sums value k over the waves
        // and then its lanes (a butterfly of all four in every wave was a sixth of the kernel's instructions)
        __syncthreads();
        if constexpr (W != 4) {
            const double s4[4] = { au, aw, (double)an, ak };
#pragma unroll
            for (int k = 0; k < 4; k++) {
                double t = group_sum<16>(s4[k]);
                t += __shfl_xor(t, 16, 64);
                t += __shfl_xor(t, 32, 64);
                if (lane == 0) wsum[wave][k] = t;
            }
            __syncthreads();
            if (tid < 4) {
                double t = 0.0;
                for (int w = 0; w < W; w++) t += wsum[w][tid];
                v.cell_part[4 * (size_t)c + tid] = t;
            }
        } else {
            sx[tid] = au;
            sx[256 + tid] = aw;
            sy[tid] = (double)an;
            sy[256 + tid] = ak;
            __syncthreads();
            const double* q = (wave < 2 ? sx : sy) + (wave & 1) * 256 + lane;
            double t = ((q[0] + q[64]) + q[128]) + q[192];
            t = group_sum<16>(t);
            t += __shfl_xor(t, 16, 64);
            t += __shfl_xor(t, 32, 64);
            if (lane == 0) v.cell_part[4 * (size_t)c + wave] = t;
        }
    }
}

template <int MODE>
static hipError_t launch_lj64(const DevView& v, double kick_dt, hipStream_t s)
{
    if constexpr ((MODE & LJ_ENERGY) != 0) {
        if (v.Ctot < kSmallCells) hipLaunchKernelGGL((k_lj64<16, MODE>), dim3(v.Ctot), dim3(1024), 0, s, v, kick_dt, 1);
        else hipLaunchKernelGGL((k_lj64<4, MODE>), dim3(v.Ctot), dim3(256), 0, s, v, kick_dt, 1);
    } else if (v.Ctot <= kWideCells) {
        const int need = (int)((13LL * v.Ntot + 80LL * v.Ctot - 1) / (80LL * v.Ctot));     // waves for 1.3 x the mean, in eights
        const int parts = std::min(need, std::max(1, kForceGroups / v.Ctot));
        hipLaunchKernelGGL((k_lj64<8, MODE>), dim3(v.Ctot * parts), dim3(512), 0, s, v, kick_dt, parts);
    } else {
        hipLaunchKernelGGL((k_lj64<4, MODE>), dim3(v.Ctot), dim3(256), 0, s, v, kick_dt, 1);
    }
    return hipGetLastError();
}

template <int IS, int W, int MODE>
static void launch_one(const DevView& v, double kick_dt, double drift_dt, hipStream_t s)
{
    const int nblocks = ((v.Ctot + 7) / 8) * 8;
    hipLaunchKernelGGL((k_lj<IS, W, MODE>), dim3(nblocks), dim3(64 * W), 0, s, v, kick_dt, drift_dt, nblocks);
}

template <int MODE>
static hipError_t launch_tiled(const DevView& v, int tiling, double kick_dt, double drift_dt, hipStream_t s)
{
    switch (tiling) {
    case 41: launch_one<4, 1, MODE>(v, kick_dt, drift_dt, s); break;
    case 42: launch_one<4, 2, MODE>(v, kick_dt, drift_dt, s); break;
    case 44: launch_one<4, 4, MODE>(v, kick_dt, drift_dt, s); break;
    case 81: launch_one<8, 1, MODE>(v, kick_dt, drift_dt, s); break;
    case 84: launch_one<8, 4, MODE>(v, kick_dt, drift_dt, s); break;
    case 161: launch_one<16, 1, MODE>(v, kick_dt, drift_dt, s); break;
    case 162: launch_one<16, 2, MODE>(v, kick_dt, drift_dt, s); break;
    default: launch_one<8, 2, MODE>(v, kick_dt, drift_dt, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_lj(const DevView& v, int mode, bool fp64, int tiling, double kick_dt, double drift_dt, hipStream_t s)
{
    constexpr int FK = LJ_FORCE | LJ_KICK;
    if (!fp64) {
        switch (mode) {
        case FK: return launch_tiled<FK>(v, tiling, kick_dt, drift_dt, s);
        case LJ_FORCE | LJ_STOREF: return launch_tiled<LJ_FORCE | LJ_STOREF>(v, tiling, kick_dt, drift_dt, s);
        case FK | LJ_STOREF: return launch_tiled<FK | LJ_STOREF>(v, tiling, kick_dt, drift_dt, s);
        case FK | LJ_DRIFT: return launch_tiled<FK | LJ_DRIFT>(v, tiling, kick_dt, drift_dt, s);
        case FK | LJ_STOREF | LJ_DRIFT: return launch_tiled<FK | LJ_STOREF | LJ_DRIFT>(v, tiling, kick_dt, drift_dt, s);
        default: return hipErrorInvalidValue;
        }
    }
    switch (mode) {
    case FK: return launch_lj64<FK>(v, kick_dt, s);
    case LJ_FORCE | LJ_STOREF: return launch_lj64<LJ_FORCE | LJ_STOREF>(v, kick_dt, s);
    case FK | LJ_STOREF: return launch_lj64<FK | LJ_STOREF>(v, kick_dt, s);
    default: return hipErrorInvalidValue;
    }
}

// the sorted FP64 positions of atoms that moved since the binning, in their old cells
__global__ __launch_bounds__(256) void k_resort(DevView v)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int N = v.Ntot;
    if (s >= N) return;
    const int a = perm_cur(v)[s];
    for (int d = 0; d < 3; d++) v.xs64[(size_t)d * N + s] = v.x[(size_t)d * N + a];
}

hipError_t launch_energy(const DevView& v, bool stale, hipStream_t s)
{
    if (stale) {
        hipLaunchKernelGGL(k_resort, dim3((v.Ntot + 255) / 256), dim3(256), 0, s, v);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return launch_lj64<LJ_ENERGY>(v, 0.0, s);
}

}  // namespace chmc
