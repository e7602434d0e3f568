// Device functions shared by the CA step kernels and the adjoint kernels.
// Arithmetic follows the reference's operation order; everything that
// includes this file is compiled with -ffp-contract=off.
#pragma once

#include <hip/hip_runtime.h>

#include "mmca_exp.h"
#include "mmca_internal.h"

namespace mmca {

// Device buffers reached through the domain table are generic pointers to
// the compiler, whose loads and stores are then FLAT instructions: 64-bit
// per-lane addresses, and a wait for LDS results also waits for them.  G(p)
// states that p points to global memory, so that global (and, for uniform
// addresses, scalar) loads and stores are used.
#define MMCA_GLOBAL __attribute__((address_space(1)))

template <typename T>
__device__ __forceinline__ MMCA_GLOBAL T *G(T *p)
{
    return (MMCA_GLOBAL T *) p;
}

// MIN(x,y) of globals.h:19
__device__ __forceinline__ double ref_min(double x, double y) { return (x < y) ? x : y; }

// Sum over a workgroup of nt threads, whole waves (result valid in thread 0).
__device__ __forceinline__ double
block_sum(double v, double *s_red, int nt)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
        v += __shfl_xor(v, d, 64);
    const int tid = threadIdx.x + threadIdx.y * blockDim.x;
    if ((tid & 63) == 0)
        s_red[tid >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (tid == 0)
        for (int i = 0; i < nt / 64; ++i)
            s += s_red[i];
    return s;
}

template <int NT>
__device__ __forceinline__ double
block_sum(double v, double *s_red)
{
    return block_sum(v, s_red, NT);
}

// Values handed from the workgroups of a launch to the one that finishes last
// (last_workgroup): stores and loads at agent scope go past the L2s, of which
// every XCD has its own.
template <typename T>
__device__ __forceinline__ void
st_agent(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
__device__ __forceinline__ T
ld_agent(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// True in the workgroup, of n, that gets here last; all of its threads call it.
// Every thread first waits until its st_agent stores have arrived, so that the
// last workgroup's ld_agent loads see all of them.  Only such values may be
// handed on: a plain store may still be in the L2 of its XCD, and a plain load
// may find an old line there.  (A __threadfence() instead would write back and
// invalidate the whole L2 in every workgroup: it took k_list_count of a 256 x
// 256 x 512 block from 7 to 150 us.)  *done is 0 before and after.
__device__ __forceinline__ bool
last_workgroup(int *done, int n)
{
    __shared__ int s_last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
    {
        s_last = __hip_atomic_fetch_add(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
        if (s_last)
            *done = 0;
    }
    __syncthreads();
    return s_last != 0;
}

// direct_temp_calc (temperature.c:24-126); x,y,z are padded indices.  AM
// selects the Gaussian-beam model at compile time, so that kernels of the
// other models do not carry its registers.
template <bool AM>
__device__ __forceinline__ double
temp_model(const Consts &c, double sim_time, int x, int y, int z)
{
    if (!AM && c.gradient == 0)
        return c.t_init - sim_time * c.cool_rate;
    double rx = c.origin[0] + ((c.off[0] + x) + 0.5) * c.cell_size;
    double ry = c.origin[1] + ((c.off[1] + y) + 0.5) * c.cell_size;
    double rz = c.origin[2] + ((c.off[2] + z) + 0.5) * c.cell_size;
    if (!AM)
    {
        double axis = ((c.gdimz == 1) ? ry : rz) - c.cell_size * 0.5;
        double tgrad = c.gradient + c.grad_coef * sim_time;
        double v = c.velocity + c.velo_coef * sim_time;
        double vt = 0.5 * (v + c.velocity) * sim_time;
        return c.t_init + tgrad * (axis - vt);
    }
    double lv = c.lv;
    double invlv = 1. / lv;
    double ls = c.lsd / (2. * 1.414);
    double xlen = c.gnsbx * c.nx * c.cell_size;
    xlen = xlen + c.lsd;
    double tline = xlen * invlv;
    double tpause = 1.5e-4 * invlv;
    tline = tline + tpause;
    double trackno = 0;
    if (c.am_tracks > 1)
        trackno = floor(sim_time / tline);
    double xnow = c.x0 + (sim_time - trackno * tline) * lv;
    double ynow = c.y0 + trackno * c.lhs;
    double znow = c.z0;
    double lpow = c.lpow;
    double lx = rx - xnow;
    double ly = ry - ynow;
    double lz = rz - znow;
    if (!(rz <= znow + c.cell_size))
        return 0.0;
    const int nt = 400;
    double Tinteg = 0.0;
    double pi15 = 5.568328;
    double lalpha = c.lthcon / (c.rho * c.lcp);
    double tsteady = 20 * lalpha * invlv * invlv;
    double ldt = tsteady / nt;
    if (sim_time < 1e-4)
        lpow = 0;
    for (int i = 0; i < nt; i++)
    {
        double lt = (0.5 + i) * ldt;
        double Tlocal = sqrt(lalpha * lt) * (ls * ls + 4. * lalpha * lt);
        Tinteg += ldt *
            exp_glibc(-((lx + lv * lt) * (lx + lv * lt) + ly * ly) / (ls * ls + 4. * lalpha * lt) -
                          (lz * lz / (4. * lalpha * lt)),
                      exp_tab) /
            Tlocal;
    }
    double Tfront = c.lab * lpow * lalpha / (pi15 * c.lthcon);
    return c.liniT + Tfront * Tinteg;
}

__device__ __forceinline__ double beam_lalpha(const Consts &c) { return c.lthcon / (c.rho * c.lcp); }

__device__ __forceinline__ double
beam_ldt(const Consts &c)
{
    const double invlv = 1. / c.lv;
    const double tsteady = 20 * beam_lalpha(c) * invlv * invlv;
    return tsteady / BEAM_NT;
}

// beam position and amplitude at sim_time (temperature.c:62-103)
struct BeamNow {
    double xnow, ynow, znow, Tfront;
};

__device__ __forceinline__ BeamNow
beam_now(const Consts &c, double sim_time)
{
    const double invlv = 1. / c.lv;
    double xlen = c.gnsbx * c.nx * c.cell_size;
    xlen = xlen + c.lsd;
    double tline = xlen * invlv;
    const double tpause = 1.5e-4 * invlv;
    tline = tline + tpause;
    double trackno = 0;
    if (c.am_tracks > 1)
        trackno = floor(sim_time / tline);
    BeamNow n;
    n.xnow = c.x0 + (sim_time - trackno * tline) * c.lv;
    n.ynow = c.y0 + trackno * c.lhs;
    n.znow = c.z0;
    const double lpow = (sim_time < 1e-4) ? 0.0 : c.lpow;
    n.Tfront = c.lab * lpow * beam_lalpha(c) / (5.568328 * c.lthcon);
    return n;
}

// The Gaussian-beam quadrature of temp_model<true> with the factors of its
// 400 terms that do not depend on the cell tabulated (same operations and
// order as temp_model<true>, so the same values):
//   vlt[i] = lv * lt,  A[i] = ls*ls + 4.*lalpha*lt,
//   Tl[i] = sqrt(lalpha*lt) * (ls*ls + 4.*lalpha*lt),
// the correctly rounded reciprocals of A and Tl, and a copy of the exp table,
// so that its lookups are LDS reads.  k_beam_nodes computes the tables once
// per block into DevBufs::beam_nodes (BEAM_NODE_ROWS x BEAM_NT), and
//   Zq[z][i] = lz*lz / (4.*lalpha*lt)
// per padded plane into DevBufs::beam_zq.
enum { BN_VLT, BN_A, BN_RA, BN_TL, BN_RTL, BEAM_NODE_ROWS };

struct BeamTab {
    double node[BEAM_NODE_ROWS][BEAM_NT];
    uint64_t exp_tab[EXP_TAB_WORDS];
};

__device__ __forceinline__ void
beam_tab_load(const DevBufs &b, BeamTab &t, int tid, int nthreads)
{
    for (int i = tid; i < BEAM_NODE_ROWS * BEAM_NT; i += nthreads)
        (&t.node[0][0])[i] = G(b.beam_nodes)[i];
    for (int i = tid; i < EXP_TAB_WORDS; i += nthreads)
        t.exp_tab[i] = exp_tab[i];
}

// a / b, correctly rounded, from rb = 1 / b correctly rounded: a product and
// two corrections with exact remainders.  The first brings the quotient
// within one unit of its last place, the second then rounds it correctly
// (Markstein's theorem: q + (a - b q) rb rounds to a / b when q is that close
// and rb is the rounded reciprocal).  Needs a and b so far from the limits of
// the exponent range that no intermediate leaves it; 5 operations where the
// division sequence takes 11 and a quarter-rate reciprocal.
__device__ __forceinline__ double
div_by(double a, double b, double rb)
{
    double q = a * rb;
    q = fma(fma(-b, q, a), rb, q);
    return fma(fma(-b, q, a), rb, q);
}

// lane Q of every group of LANES (2 or 4) lanes, to all of the group
template <int LANES, int Q>
__device__ __forceinline__ double
group_lane(double v)
{
    constexpr int ctrl = LANES == 4 ? Q | Q << 2 | Q << 4 | Q << 6                       // DPP quad_perm
                                    : Q | Q << 2 | (2 + Q) << 4 | (2 + Q) << 6;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// temp_model<true> on the tables, one cell per LANES lanes (1, 2 or 4): lane g
// of a group computes the terms LANES m + g and every lane adds all of them in
// node order.  All lanes of a group pass the same cell.
//
// Four terms at a time, so that their chains overlap.  Where c.beam_fast holds
// and every exponent of the wave is in exp's normal range (then ldt * exp is
// above 1e-250, far from where a division by a reciprocal could go wrong) the
// terms are straight-line code, 28 FP64 operations each.
//
// The node factors are the same for every lane of a wave with one lane per
// cell: they come as scalar loads, because reading them from LDS (20 of the 44
// clocks of LDS time a term took) held the four SIMDs of a CU to two thirds of
// their FP64 rate.  With more lanes per cell they are LDS reads.
template <int LANES>
__device__ __forceinline__ double
beam_quad(const Consts &c, const DevBufs &b, const BeamTab &t, const MMCA_GLOBAL double *Z, const BeamNow &bn, int x, int y, int z, int g)
{
    constexpr int U = 4;
    static_assert(BEAM_NT % (4 * U) == 0, "whole rounds of four terms per lane");
    const double rx = c.origin[0] + ((c.off[0] + x) + 0.5) * c.cell_size;
    const double ry = c.origin[1] + ((c.off[1] + y) + 0.5) * c.cell_size;
    const double rz = c.origin[2] + ((c.off[2] + z) + 0.5) * c.cell_size;
    if (!(rz <= bn.znow + c.cell_size))
        return 0.0;
    if (bn.Tfront == 0.0)
        return c.liniT + bn.Tfront * 0.0;         // every term is finite, so Tfront * Tinteg is this
    const double lx = rx - bn.xnow;
    const double ly = ry - bn.ynow;
    const double ly2 = ly * ly;
    const double ldt = beam_ldt(c);
    auto node = [&](int row, int i) -> double {
        if constexpr (LANES == 1)
            return ((const __attribute__((address_space(4))) double *) (unsigned long long) b.beam_nodes)[row * BEAM_NT + i];
        else
            return t.node[row][i];
    };
    double Tinteg = 0.0;
    for (int m = 0; m < BEAM_NT / LANES; m += U)
    {
        double term[U], e[U];
        bool normal = c.beam_fast;
        if (c.beam_fast)
        {
#pragma unroll
            for (int k = 0; k < U; ++k)
            {
                const int i = LANES * (m + k) + g;
                const double u = lx + node(BN_VLT, i);
                const double a = u * u + ly2;
                e[k] = -div_by(a, node(BN_A, i), node(BN_RA, i)) - Z[i];
                normal = normal && e[k] > -512.0 && e[k] < -0x1p-54;
            }
        }
        if (__all(normal))
        {
#pragma unroll
            for (int k = 0; k < U; ++k)
            {
                const int i = LANES * (m + k) + g;
                term[k] = div_by(ldt * exp_normal(e[k], t.exp_tab), node(BN_TL, i), node(BN_RTL, i));
            }
        }
        else
        {
#pragma unroll 1
            for (int k = 0; k < U; ++k)
            {
                const int i = LANES * (m + k) + g;
                const double u = lx + node(BN_VLT, i);
                const double v = ldt * exp_glibc(-(u * u + ly2) / node(BN_A, i) - Z[i], t.exp_tab) / node(BN_TL, i);
                term[0] = k == 0 ? v : term[0];
                term[1] = k == 1 ? v : term[1];
                term[2] = k == 2 ? v : term[2];
                term[3] = k == 3 ? v : term[3];
            }
        }
#pragma unroll
        for (int k = 0; k < U; ++k)
        {
            if constexpr (LANES == 1)
                Tinteg += term[k];
            else
            {
                Tinteg += group_lane<LANES, 0>(term[k]);
                Tinteg += group_lane<LANES, 1>(term[k]);
                if constexpr (LANES == 4)
                {
                    Tinteg += group_lane<LANES, 2>(term[k]);
                    Tinteg += group_lane<LANES, 3>(term[k]);
                }
            }
        }
    }
    return c.liniT + bn.Tfront * Tinteg;
}

// Half-width of the interval around an approximate beam temperature T
// (DevBufs::temp32) that holds the quadrature's value: its FP32 storage and
// rounding (far below 1e-5 relative to the terms it is the sum of) and the
// interpolation's error (c.beam_tol times the largest sum of terms).
__device__ __forceinline__ double
beam_margin(const Consts &c, double T)
{
    return 1e-5 * (fabs(T) + fabs(c.liniT)) + c.beam_tol;
}

// Octahedron half-diagonal of a solid cell (grow_octahedra, growth.c:392-403)
// from its centre offset, fs and grain g.
__device__ __forceinline__ double
octa_d(const Consts &c, const DevBufs &b, long long i, int g, double fs)
{
    const MMCA_GLOBAL double *R = G(b.g_rot) + 9 * (long long) g;
    double rx0 = 0.0 - G(b.dc)[3 * i];
    double ry0 = 0.0 - G(b.dc)[3 * i + 1];
    double rz0 = 0.0 - G(b.dc)[3 * i + 2];
    double gx0 = R[0] * rx0 + R[3] * ry0 + R[6] * rz0;
    double gy0 = R[1] * rx0 + R[4] * ry0 + R[7] * rz0;
    double gz0 = R[2] * rx0 + R[5] * ry0 + R[8] * rz0;
    double ds1 = fabs(gx0) + fabs(gy0) + fabs(gz0);
    ds1 = ref_min(ds1, 1.5);
    return ds1 + fs * c.rev_fsgrow;
}

// With track_d: a cell that stops being solid keeps, in the reference's d
// array, the half-diagonal of its last step as a solid cell (grow_octahedra
// writes solid cells only).  That value follows from the state the
// partitioning step starts from: the cell's dc and fs are the ones of its
// last growth step (capture writes only liquid cells).
__device__ __forceinline__ void
keep_stale_d(const Consts &c, const DevBufs &b, long long i, int g_old, int g_new, double fs_old)
{
    if (c.track_d && g_old > 0 && g_new <= 0 && g_old < c.max_total_grains)
        G(b.d)[i] = octa_d(c, b, i, g_old, fs_old);
}

// 64-bit words of one step's branch record
__host__ __device__ inline long long
rec_words(const Consts &c)
{
    return 3ll * c.w64 * (c.ny + 2) * (c.nz + 2);
}

// Branch record of one step: per padded row (j, k) and 64-cell segment of x,
// three 64-bit planes; bit (x - 1) % 64 of plane p is bit p of the
// MMCA_BRANCH_* code of cell x (3 bits per interior cell).
__device__ __forceinline__ long long
rec_word(const Consts &c, int seg, int j, int k)
{
    return (((long long) k * (c.ny + 2) + j) * c.w64 + seg) * 3;
}

__device__ __forceinline__ int
rec_code(const Consts &c, const unsigned char *rec, int x, int j, int k)
{
    const unsigned long long *w = reinterpret_cast<const unsigned long long *>(rec) + rec_word(c, (x - 1) >> 6, j, k);
    const int bit = (x - 1) & 63;
    return (int) ((w[0] >> bit) & 1ull) | (int) (((w[1] >> bit) & 1ull) << 1) | (int) (((w[2] >> bit) & 1ull) << 2);
}

// ---------------------------------------------------------------------------
// Diffusion (growth.c:85-113, order +x,-x,+y,-y,+z,-z) of one cell, from the
// neighbours' cl and fs and their mold flags.
__device__ __forceinline__ double
diffuse_cell(const Consts &c, double ce_old, double conc, double lspfs, const double *cln,
             const double *fsn, const int *mo)
{
    double nbsum = 0;
#pragma unroll
    for (int n = 0; n < 6; ++n)
    {
        double fs_av = 0.5 * (lspfs + fsn[n]);
        double r = (c.rs * fs_av + c.rl * (1 - fs_av)) * (1 - mo[n]);
        nbsum += r * (cln[n] - conc);
    }
    return ce_old + nbsum;
}

}  // namespace mmca
