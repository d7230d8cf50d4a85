// Self-gravity and black-hole accretion of the collapsar model: the parts of
// CUSTOM_UPDATE (model/collapsar/src/custom.f90:416-658) that run after
// FINDPRESSURE in UPDATE(p).
//
//   k_mdot            mass accretion rate through the inner face from the x
//                     sweep's density flux at face 0 (GETFLUX_X, :222-245)
//   k_mbh<STAGE>      the RK update of m_bh, r_sh and the horizon check
//   k_sor_red         the red half of one SOR sweep pair (and the decision
//                     of the pair before it)
//   k_sor_black       the black half and the blocks' error partials
//   k_sor_decide      the decision of a batch's last pair
//   k_sor_bc          the boundary values of the final potential
//
// FP64 only.  The sweeps are bit-identical to the serial loop: a red cell
// ((-1)**(j+k+l) > 0) reads only black neighbours and vice versa, so the order
// within a sweep does not matter.  During a solve the potential lives split
// by colour (every cell of one colour in a dense array, like rho_in) and
// ping-pongs: a sweep pair reads the red and black values at its
// start and writes both colours anew; red cells read the start values, black
// cells the new red ones.  The boundary values a pair reads are those the
// reference's previous pair set (custom.f90:601-631), formed on the fly from
// the start values: phi(0) = phi(1), phi(nx+1) = -1, zero theta gradient,
// periodic in phi -- and 0 on the first pair after the zero guess of
// UPDATE(0) (:497-505), which had set no boundary values yet.  k_sor_copy
// moves phi into the split arrays at the start and back at the end, and
// k_sor_bc writes the boundary values for the gravity source.
// The error is the OpenMP MAX reduction of :588-598 as the reference's
// one-thread CPU build evaluates it: a private fold of
// MAX(abserror, |dphi/phi_old|) in l, k, j order with flang's MAX
// (a > b ? a : b) -- a NaN term replaces the running value and the next term
// replaces the NaN -- then a combine with the shared 1e-50 that drops a NaN.
// So the result is 1e-50 when the last term is NaN (0/0 where phi stays 0,
// as on the first sweep from the zero guess), else the larger of 1e-50 and
// the maximum of the terms after the last NaN.  k_sor_black leaves per-block
// partials (the last NaN index of the block and the maximum of the terms
// after it) and one block of the next kernel combines them exactly.  The
// host runs sweep pairs in batches and reads the end flag between batches;
// pairs queued after the solve ended return at once.
#pragma once
#include "kernels.hpp"

namespace cumc3d {

// colour-split slots of each colour per plane of a block, one per thread
constexpr int SOR_SLOTS = 256;

// Per-cell SOR data are split by colour so that each sweep reads its cells
// densely: colour c (0 red, 1 black) holds, for row (k, l), the cells
// j = j0 + 2i with j0 = 1 when (1 + k + l) % 2 == c, else 2, at
// c*hx*ny*nz + i + hx*((k-1) + ny*(l-1)), hx = (nx+1)/2 (a padded slot when
// j > nx).  Per cell only rho_in, the density above the atmosphere
// (custom.f90:544-546), refreshed per solve.  poisson_coef's azimuthal
// coefficients (poisson.f90:52-63) are formed in the kernel from a (j, k)
// factor and the cell's phi spacings with the same divisions in the same
// order, so they are the values the reference stores:
//   clp1 = ((2/xc^2/sin^2) / (zp1-zm1)) / (zp1-zc)
//   clm1 = ((2/xc^2/sin^2) / (zp1-zm1)) / (zc-zm1)
//   epsc = (radial + polar terms) - ((2/xc^2/sin^2) / (zp1-zc)) / (zc-zm1)

struct SorArgs {
    int nx, ny, nz;
    long NX, NY;
    // phi during a solve, split by colour like rho_in (index
    // i + hx((k-1) + ny(l-1)) within a colour): the red and black values at
    // the start of the sweep pair and after it
    const double *rin, *bin;
    double *rout, *bout;
    const double *rho_in;               // per cell, split by colour (see above)
    const double *ajp1, *ajm1;          // [j], j = 1..nx
    const double *bkp1, *bkm1;          // [k(nx+1) + j]
    const double *a2, *e2;              // [k(nx+1) + j]: 2/xc^2/sin^2 and epsc's radial + polar terms
    const double *z[3], *iz[3];         // [l]: zp1-zm1, zp1-zc, zc-zm1 and their rounded reciprocals
    long long *part_nan;                // per run of SOR_SLOTS slots of a plane: q of its last NaN term, -1 if none
    double *part_max;                   // per run: max of the terms after it, -1 if none
    int runs, items;                    // runs per plane; runs times plane pairs (the blocks' work)
    int nblk;                           // runs: ceil(hx ny / SOR_SLOTS) per plane, times nz
    int relax_max;
    int zero_ghosts;                    // the first pair after the zero guess: boundary values 0
    int combine;                        // red kernel: block 0 first decides the previous pair's exit
    double pa, omega, tol, pi4;         // prim_a(irho), omega_weight, tolerance, 4 pi
    DevScalars *S;
};

// r_sh from m_bh and the horizon check of custom.f90:481-484 (STOP: the
// stage kernels of every later stage return at once)
__device__ __forceinline__ void grav_horizon(DevScalars *S, double c_code, double xF0) {
    S->r_sh = 2.0 * S->m_bh / (c_code * c_code);
    if (S->r_sh >= xF0) {
        S->grav_stop = 1;
        S->active = 0;
    }
}

// custom.f90:450-465: mdot = sum over l, k (serial order) of
// -mflux_x(k,l) xF(0)^2 dcose(k) dz(l), clipped at 0, from the x sweep's
// density flux at face 0.  256 threads form up to 4096 terms at a time into
// LDS (all loads in flight together); one wave then adds them in the serial
// order, reading ahead of the dependent add chain, which is the cost.  Runs
// on a second stream beside the stage's later kernels.
constexpr int ACC_CHUNK = 4096;
__global__ __launch_bounds__(256) void k_mdot(ArgsT<double> a) {
    if (!a.S->active) return;
    __shared__ double term[ACC_CHUNK];
    const int nk = a.ny * a.nz;
    const double xf0 = a.ax[0].xF[3];
    double mdot = 0.0;
    for (int base = 0; base < nk; base += ACC_CHUNK) {
        const int m = nk - base < ACC_CHUNK ? nk - base : ACC_CHUNK;
        for (int i = threadIdx.x; i < m; i += blockDim.x) {
            const int t = base + i;
            const int k = 1 + t % a.ny, l = 1 + t / a.ny;
            const double mf = a.F[0][0][cidx(a, 0, k, l)];
            term[i] = (-mf) * xf0 * xf0 * a.dcose[k + 3] * a.ax[2].d[l + 3];
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            int i = 0;
            for (; i + 8 <= m; i += 8) {
                double r[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) r[u] = term[i + u];
#pragma unroll
                for (int u = 0; u < 8; ++u) mdot = mdot + r[u];
            }
            for (; i < m; ++i) mdot = mdot + term[i];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) a.S->mdot = fmax2(mdot, 0.0);
}

// custom.f90:467-484 for p = STAGE: the RK combine of m_bh with the stage's
// mdot, then r_sh and the horizon check
template <int STAGE> __global__ void k_mbh(DevScalars *S, double c_code, double xF0) {
    if (!S->active) return;
    const double dt = S->dt, mdot = S->mdot;
    if constexpr (STAGE == 1) {
        S->mbh_old = S->m_bh;
        S->m_bh = S->mbh_old + dt * mdot;
    } else if constexpr (STAGE == 2) {
        S->m_bh = (3.0 / 4.0) * S->mbh_old + (1.0 / 4.0) * S->m_bh + (1.0 / 4.0) * dt * mdot;
    } else {
        S->m_bh = (1.0 / 3.0) * S->mbh_old + (2.0 / 3.0) * S->m_bh + (2.0 / 3.0) * dt * mdot;
    }
    grav_horizon(S, c_code, xF0);
}

// UPDATE(0): m_bh as the initial model left it, then r_sh and the check
__global__ void k_grav_start(DevScalars *S, double m_bh, double c_code, double xF0) {
    S->m_bh = m_bh;
    S->mbh_old = m_bh;
    S->grav_stop = 0;
    grav_horizon(S, c_code, xF0);
}

// Start of a solve: the iteration state (k_fill0 writes the zero guess phi = 0
// of p = 0, custom.f90:491-507, over the whole box; the outer layers are
// never read).  An inactive run (finished or stopped) skips the solve.
__global__ void k_sor_begin(DevScalars *S) {
    S->sor_n = 0;
    S->sor_nan = 0;
    if (!S->active) {
        S->sor_state = 1;
        S->sor_iter = 0;
        return;
    }
    S->sor_state = 0;
}

__global__ __launch_bounds__(256) void k_fill0(double *p, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

__device__ __forceinline__ long sor_c(const SorArgs &a, int j, int k, int l) {
    return (long)(j + 2) + a.NX * ((long)(k + 2) + a.NY * (long)(l + 2));
}

// index of cell (j, k, l) within its colour's arrays
__device__ __forceinline__ long sor_i(const SorArgs &a, int j, int k, int l) {
    const long hx = (a.nx + 1) >> 1;
    return (long)((j - 1) >> 1) + hx * ((long)(k - 1) + (long)a.ny * (l - 1));
}

// The neighbour values the update of a cell of colour C reads
// (custom.f90:548-550), for the cell at split index c = sor_i(j, k, l) in a
// plane l that the block shares: cells of the other colour from `other` (the
// black start values for a red cell, the new red values for a black one), the
// boundary values from the start values of the pair: phi(0) = phi(1) and the
// theta ends copy the cell itself (`own`, its start value), phi(nx+1) = -1,
// periodic in phi.  In the split order the neighbours sit at fixed offsets:
// along x at c or c +- 1 by j's parity, along theta at c +- hx, along phi at
// c +- hx ny.  Every load is unconditional, from a clamped index.
template <int C>
__device__ __forceinline__ void sor_neigh(const SorArgs &a, const double *other, int j, int k, int l, int c, double own,
                                          double nb[6]) {
    const bool z0 = a.zero_ghosts;
    const int hx = (a.nx + 1) >> 1, nh = hx * a.ny, odd = j & 1, wrap = nh * (a.nz - 1);
    // j + k + l = C modulo 2, so the cell across the periodic boundary has
    // the colour C + 1 - l, or C + nz - l
    const double *up = l < a.nz ? other + nh : (((C + 1 - l) & 1) ? a.bin : a.rin) - wrap;
    const double *dn = l > 1 ? other - nh : (((C + a.nz - l) & 1) ? a.bin : a.rin) + wrap;
    const double xp = other[j < a.nx ? c + 1 - odd : c], xm = other[j > 1 ? c - odd : c];
    const double yp = other[k < a.ny ? c + hx : c], ym = other[k > 1 ? c - hx : c];
    const double zp = up[c], zm = dn[c];
    nb[0] = j < a.nx ? xp : (z0 ? 0.0 : -1.0);
    nb[1] = j > 1 ? xm : (z0 ? 0.0 : own);
    nb[2] = k < a.ny ? yp : (z0 ? 0.0 : own);
    nb[3] = k > 1 ? ym : (z0 ? 0.0 : own);
    nb[4] = l == a.nz && z0 ? 0.0 : zp;
    nb[5] = l == 1 && z0 ? 0.0 : zm;
}

// The coefficients of a (j, k) column that do not depend on the plane
struct SorColumn {
    double A, e2, ajp1, ajm1, bkp1, bkm1;
};
__device__ __forceinline__ SorColumn sor_column(const SorArgs &a, int j, int k) {
    const int jk = k * (a.nx + 1) + j;
    return {a.a2[jk], a.e2[jk], a.ajp1[j], a.ajm1[j], a.bkp1[jk], a.bkm1[jk]};
}

// one cell's relaxation (custom.f90:544-551); returns the new value.  The five
// quotients by the plane's phi spacings take their reciprocals from the table.
__device__ __forceinline__ double sor_cell(const SorArgs &a, const SorColumn &q, int l, double rho_in,
                                           const double nb[6], double old) {
    const Den<double> dpm(a.z[0][l], a.iz[0][l]), dpc(a.z[1][l], a.iz[1][l]), dcm(a.z[2][l], a.iz[2][l]);
    const double t = dpm(q.A);
    const double clp1 = dpc(t), clm1 = dcm(t);
    const double epsc = q.e2 - dcm(dpc(q.A));
    const double s = q.ajp1 * nb[0] + q.ajm1 * nb[1] + q.bkp1 * nb[2] + q.bkm1 * nb[3] + clp1 * nb[4] + clm1 * nb[5];
    const double rhs = Den<double>(epsc).tiny(a.pi4 * rho_in - s);
    return (1.0 - a.omega) * old + a.omega * rhs;
}

// The run and the first plane of a block.  Block row y covers plane l and plane
// l + 2, whose cells of one colour share (j, k) and with it the column's six
// coefficients and the plane between them.  Blocks are dealt to the 8 XCDs
// round-robin; each XCD takes one contiguous eighth of the (row, run) items,
// the same in both kernels, so that most of what it reads is what it wrote.
// False for a padding block.
__device__ __forceinline__ bool sor_item(const SorArgs &a, int block, int &run, int &l0) {
    const int per = (a.items + 7) >> 3, w = (block & 7) * per + (block >> 3);
    const int y = w / a.runs;
    run = w - y * a.runs;
    l0 = 4 * (y >> 1) + 1 + (y & 1);
    return (block >> 3) < per && w < a.items && l0 <= a.nz;
}

// Holds v where it is: a value loaded before a branch is not sunk behind it.
__device__ __forceinline__ void pin(double &v) { __asm__ volatile("" : "+v"(v)); }

// position of cell i of row (k, l) of a colour in the colour-split rho_in
__device__ __forceinline__ long sor_rec(const SorArgs &a, int colour, int i, int k, int l) {
    const long hx = (a.nx + 1) >> 1;
    return (long)colour * hx * a.ny * a.nz + i + hx * ((long)(k - 1) + (long)a.ny * (l - 1));
}

// Start of a solve: rho_in of every cell, split by colour
// (custom.f90:544-546: MERGE(1, 0, rho - prim_a(irho) > 0) * rho).
__global__ __launch_bounds__(256) void k_sor_rho(SorArgs a, const double *rho, double *rho_in) {
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (unsigned)(a.nx * a.ny)) return;
    const int l = 1 + blockIdx.y;
    const int k = 1 + (int)(t / (unsigned)a.nx), j = 1 + (int)(t - (unsigned)(k - 1) * a.nx);
    const double r = rho[sor_c(a, j, k, l)];
    const double diff = r - a.pa;
    const double factor = diff > 0.0 ? 1.0 : 0.0;
    const int colour = (j + k + l) & 1;
    const int j0 = ((1 + k + l) & 1) == colour ? 1 : 2;
    rho_in[sor_rec(a, colour, (j - j0) >> 1, k, l)] = factor * r;
}

__device__ __forceinline__ long long block_max_ll(long long v) {
    __shared__ long long red[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        long long o = __shfl_down(v, off, 64);
        v = o > v ? o : v;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    long long m = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = red[w] > m ? red[w] : m;
    __syncthreads();
    return m;
}

// max of non-NaN values >= -1 (the terms are >= 0; -1 marks none)
__device__ __forceinline__ double block_max_d(double v) {
    __shared__ double red[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_down(v, off, 64);
        v = o > v ? o : v;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double m = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = red[w] > m ? red[w] : m;
    __syncthreads();
    return m;
}

// Maximum over the wave, in lane 63 (values >= -1, no NaN): DPP moves within
// rows of 16, then the row broadcasts.
template <int CTRL> __device__ __forceinline__ double dpp_max(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
    const double o = __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
    return o > v ? o : v;
}
__device__ __forceinline__ double wave_max_d(double v) {
    v = dpp_max<0x111>(v);   // row_shr:1
    v = dpp_max<0x112>(v);   // row_shr:2
    v = dpp_max<0x114>(v);   // row_shr:4
    v = dpp_max<0x118>(v);   // row_shr:8
    v = dpp_max<0x142>(v);   // row_bcast:15
    return dpp_max<0x143>(v);   // row_bcast:31
}

// Two partials of consecutive q ranges, the right one folded into the left:
// the last NaN of the right range supersedes everything before it.
__device__ __forceinline__ void fold_partial(long long &L, double &M, long long L2, double M2) {
    if (L2 >= 0) {
        L = L2;
        M = M2;
    } else {
        M = M2 > M ? M2 : M;
    }
}

// The previous pair's abserror from the black blocks' partials and the exit
// decision (custom.f90:638, :644), by one block of 256 threads.  Most pairs
// have no NaN term (a block that has one sets sor_nan): then abserror is the
// maximum of the runs' maxima in any order, and each thread takes every 256th
// run, its loads in flight together.
// Else the partials are folded left to right (they are in q order: the last
// NaN q, and the maximum of the terms after it): each thread folds a
// contiguous run of them, then the threads' results are folded in thread
// order (lane i takes lane i + off at each level of the tree).
__device__ void sor_decide(const SorArgs &a) {
    DevScalars *S = a.S;
    __shared__ double wm[4];
    __shared__ long long wl[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nan = S->sor_nan;
    double M = -1.0;
    for (int i0 = threadIdx.x; i0 < a.nblk; i0 += 16 * 256) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = i0 + 256 * u < a.nblk ? a.part_max[i0 + 256 * u] : -1.0;
#pragma unroll
        for (int u = 0; u < 16; ++u) M = v[u] > M ? v[u] : M;
    }
    long long L = -1;
    if (nan) {
        const int per = (a.nblk + 255) >> 8;
        const int i0 = (int)threadIdx.x * per, i1 = i0 + per < a.nblk ? i0 + per : a.nblk;
        M = -1.0;
        for (int i = i0; i < i1; ++i) fold_partial(L, M, a.part_nan[i], a.part_max[i]);
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const long long L2 = __shfl_down(L, off, 64);
            const double M2 = __shfl_down(M, off, 64);
            if (lane + off < 64) fold_partial(L, M, L2, M2);
        }
        if (lane == 0) {
            wl[wv] = L;
            wm[wv] = M;
        }
    } else {
        M = wave_max_d(M);
        if (lane == 63) {
            wl[wv] = -1;
            wm[wv] = M;
        }
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    L = wl[0];
    M = wm[0];
    for (int w = 1; w < 4; ++w) fold_partial(L, M, wl[w], wm[w]);
    S->sor_nan = 0;
    const long long N = (long long)a.nx * a.ny * a.nz;
    double err;
    if (L == N - 1) err = 1.0e-50;   // the private result is NaN: the combine keeps 1e-50
    else err = M > 1.0e-50 ? M : 1.0e-50;
    S->sor_err = err;
    const int n = S->sor_n + 1;
    S->sor_n = n;
    if (err <= a.tol) {
        S->sor_state = 1;
        S->sor_iter = n;
    } else if (n == a.relax_max) {
        S->sor_state = 1;
        S->sor_iter = n + 1;   // the DO loop ran out: n = relax_max + 1 after it
    }
}

// Red cells ((j + k + l) even).  With `combine`, block 0 decides the previous
// pair's exit (the work items start at block 8); the others do not wait for it:
// a pair begun after the solve ended only writes the buffer that is not the
// result, and the black kernel and every later kernel see the decision and
// return.  At the sizes of a progenitor grid (156 x 44 x 128) the arrays sit in
// the Infinity Cache and both kernels are bound by its latency and the launch
// (fewer instructions no longer help): each thread takes two cells that share
// their column, loads everything before it looks at the end flag, divides by
// reciprocals, and finds its planes on the XCD that wrote them.  A solve of
// 10496 pairs took 196 ms (18.7 us a pair); two planes a thread with
// reciprocals 172, fixed neighbour offsets and the order-free fold 164, the
// XCD order 157 ms (15.0 us).
__global__ __launch_bounds__(256) void k_sor_red(SorArgs a) {
    if (blockIdx.x < 8) {
        if (a.combine && blockIdx.x == 0 && !a.S->sor_state && a.S->active) sor_decide(a);
        return;
    }
    const bool stop = a.S->sor_state || !a.S->active;
    const int hx = (a.nx + 1) >> 1, nh = hx * a.ny;
    int run, l0;
    if (!sor_item(a, blockIdx.x - 8, run, l0)) return;
    const int s = run * SOR_SLOTS + (int)threadIdx.x;
    if (s >= nh) return;
    const int k = 1 + s / hx, i = s - (k - 1) * hx;
    const int j = (((1 + k + l0) & 1) == 0 ? 1 : 2) + 2 * i;
    if (j > a.nx) return;
    const bool two = l0 + 2 <= a.nz;
    const SorColumn q = sor_column(a, j, k);
    double rho_in[2], old[2], nb[2][6];
    int ic[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int l = p && two ? l0 + 2 : l0;
        ic[p] = s + nh * (l - 1);   // sor_i(a, j, k, l)
        rho_in[p] = a.rho_in[ic[p]];
        old[p] = a.rin[ic[p]];
        sor_neigh<0>(a, a.bin, j, k, l, ic[p], old[p], nb[p]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        pin(rho_in[p]);
        for (int v = 0; v < 6; ++v) pin(nb[p][v]);
    }
    if (stop) return;
    const double n0 = sor_cell(a, q, l0, rho_in[0], nb[0], old[0]);
    a.rout[ic[0]] = n0;
    if (two) a.rout[ic[1]] = sor_cell(a, q, l0 + 2, rho_in[1], nb[1], old[1]);
}

// Every interior cell, in the colour-split order: a block takes one run of
// SOR_SLOTS split indices of both colours in each of its two planes; in a plane
// those are the cells (k, j = 2i+1, 2i+2), one contiguous range of q.  A thread
// relaxes the black cell of its slot from the new red values and forms the
// error terms |dphi/phi_old| (custom.f90:593) of its black and red cell from
// the pair's start and end values; the run's partial is their fold.  Without a
// NaN in the block (its waves vote) that is one maximum per plane.
__global__ __launch_bounds__(256) void k_sor_black(SorArgs a) {
    const bool stop = a.S->sor_state || !a.S->active;
    const int hx = (a.nx + 1) >> 1, nh = hx * a.ny, nxy = a.nx * a.ny;
    int run, l0;
    if (!sor_item(a, blockIdx.x, run, l0)) return;
    const bool two = l0 + 2 <= a.nz;
    const int s = run * SOR_SLOTS + (int)threadIdx.x;
    const int sc = s < nh ? s : nh - 1;
    const int k = 1 + sc / hx, i = sc - (k - 1) * hx;
    const int jb = (((1 + k + l0) & 1) == 1 ? 1 : 2) + 2 * i, jr = (((1 + k + l0) & 1) == 0 ? 1 : 2) + 2 * i;
    // the padded slot of an odd row holds no cell; its thread reads the row's last one
    const bool lb = s < nh && jb <= a.nx, lr = s < nh && jr <= a.nx;
    const int j = jb <= a.nx ? jb : a.nx;
    const SorColumn q = sor_column(a, j, k);
    double rho_in[2], bold[2], rold[2], rnew[2], nb[2][6];
    int ic[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int l = p && two ? l0 + 2 : l0;
        ic[p] = sc + nh * (l - 1);   // sor_i of both cells
        rho_in[p] = (a.rho_in + nh * a.nz)[ic[p]];
        bold[p] = a.bin[ic[p]];
        rold[p] = a.rin[ic[p]];
        rnew[p] = a.rout[ic[p]];
        sor_neigh<1>(a, a.rout, j, k, l, ic[p], bold[p], nb[p]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        pin(rho_in[p]);
        pin(rold[p]);
        pin(rnew[p]);
        for (int v = 0; v < 6; ++v) pin(nb[p][v]);
    }
    if (stop) return;
    double eb[2], er[2];
    bool bad = false;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const bool on = p == 0 || two;
        eb[p] = er[p] = -1.0;
        if (lb && on) {
            const double nw = sor_cell(a, q, p ? l0 + 2 : l0, rho_in[p], nb[p], bold[p]);
            a.bout[ic[p]] = nw;
            eb[p] = fabs((nw - bold[p]) / bold[p]);
        }
        if (lr && on) er[p] = fabs((rnew[p] - rold[p]) / rold[p]);
        bad = bad || eb[p] != eb[p] || er[p] != er[p];
    }
    __shared__ double wm[2][4];
    __shared__ int wbad[4];
    const int w = threadIdx.x >> 6;
    const int vote = __ballot(bad) != 0;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const double m = wave_max_d(eb[p] > er[p] ? eb[p] : er[p]);
        if ((threadIdx.x & 63) == 63) wm[p][w] = m;
    }
    if ((threadIdx.x & 63) == 63) wbad[w] = vote;
    __syncthreads();
    const bool any = wbad[0] | wbad[1] | wbad[2] | wbad[3];
    const int b = (l0 - 1) * a.runs + run;
    if (!any) {
        if (threadIdx.x < (two ? 2 : 1)) {
            const double *v = wm[threadIdx.x];
            double m = v[0];
            for (int u = 1; u < 4; ++u) m = v[u] > m ? v[u] : m;
            a.part_nan[b + threadIdx.x * 2 * a.runs] = -1;
            a.part_max[b + threadIdx.x * 2 * a.runs] = m;
        }
        return;
    }
    for (int p = 0; p < (two ? 2 : 1); ++p) {
        const long long q0 = (long long)(l0 + 2 * p - 1) * nxy + (long long)(k - 1) * a.nx - 1;
        long long last = -1;
        if (er[p] != er[p]) last = q0 + jr;
        if (eb[p] != eb[p]) last = q0 + jb > last ? q0 + jb : last;
        last = block_max_ll(last);
        double m = -1.0;
        if (q0 + jb > last && eb[p] == eb[p]) m = eb[p];
        if (q0 + jr > last && er[p] == er[p]) m = er[p] > m ? er[p] : m;
        m = block_max_d(m);
        if (threadIdx.x == 0) {
            a.part_nan[b + 2 * p * a.runs] = last;
            a.part_max[b + 2 * p * a.runs] = m;
            a.S->sor_nan = 1;
        }
    }
}

// The decision of a solve's last pair when no red kernel follows it.
__global__ __launch_bounds__(256) void k_sor_decide(SorArgs a) {
    if (!a.S->sor_state && a.S->active) sor_decide(a);
}

// phi over the interior between the ghosted box and the colour-split
// arrays: to_split at the start of a solve, back at its end.
__global__ __launch_bounds__(256) void k_sor_copy(SorArgs a, double *phi, double *red, double *black, int to_split) {
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (unsigned)(a.nx * a.ny)) return;
    const int l = 1 + blockIdx.y;
    const int k = 1 + (int)(t / (unsigned)a.nx), j = 1 + (int)(t - (unsigned)(k - 1) * a.nx);
    double *s = ((j + k + l) & 1) ? black : red;
    const long c = sor_c(a, j, k, l), ic = sor_i(a, j, k, l);
    if (to_split) s[ic] = phi[c];
    else phi[c] = s[ic];
}

// The boundary values of the final potential (custom.f90:601-631), written
// once a solve has ended: phi(0) = phi(1), phi(nx+1) = -1 over the interior
// (k, l); theta ends copy their neighbours over (j, l); phi is periodic over
// (j, k).
__global__ __launch_bounds__(256) void k_sor_bc(double *phi, int nx, int ny, int nz, long NX, long NY) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long sy = NX, sz = NX * NY;
    auto ci = [&](int j, int k, int l) { return (long)(j + 2) + NX * ((long)(k + 2) + NY * (long)(l + 2)); };
    if (t < (long)ny * nz) {
        const int k = 1 + (int)(t % ny), l = 1 + (int)(t / ny);
        const long c = ci(1, k, l);
        phi[c - 1] = phi[c];
        phi[ci(nx + 1, k, l)] = -1.0;
        return;
    }
    t -= (long)ny * nz;
    if (t < (long)nx * nz) {
        const int j = 1 + (int)(t % nx), l = 1 + (int)(t / nx);
        const long c1 = ci(j, 1, l), cn = ci(j, ny, l);
        phi[c1 - sy] = phi[c1];
        phi[cn + sy] = phi[cn];
        return;
    }
    t -= (long)nx * nz;
    if (t < (long)nx * ny) {
        const int j = 1 + (int)(t % nx), k = 1 + (int)(t / nx);
        const long c1 = ci(j, k, 1), cn = ci(j, k, nz);
        phi[c1 - sz] = phi[cn];
        phi[cn + sz] = phi[c1];
    }
}

}  // namespace cumc3d
