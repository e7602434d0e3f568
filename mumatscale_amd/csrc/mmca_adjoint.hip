// Frozen-branch replay of diffusion + partitioning and its adjoint, for
// gfx950.
//
// A forward run records the MMCA_BRANCH_* code that fs_change_diffuse
// (growth.c:221-273) took at every cell and step.  With those codes fixed,
// one step is a smooth map of the FP64 state (ce, cl, fs):
//   ce' = ce + sum_n r_n (cl_n - cl),  r_n = (rs f_n + rl (1 - f_n)) (1 - mold_n),
//         f_n = (fs + fs_n) / 2                     (growth.c:85-113, +x,-x,+y,-y,+z,-z)
//   LIQUID, REMELT: cl' = ce', fs' = 0
//   SOLID:          cl' = ce' k_inv, fs' = fs
//   GROW:           cl' = cl + dcl, fs' = fs + dfs
//   FULL:           cl' = cl + dcl, fs' = 1
//   dcl = (c_int - cl) D_xt 2 + dce / A,  dfs = (dcl A - dce) km_inv / cl,
//   A = 1 - km fs,  dce = ce' - ce,  c_int = c0 + m_inv (T - T_liq)
// k_replay evaluates it with the forward kernel's expressions (bit-identical
// with the recorded run at the recorded parameters).  The adjoint of one
// step back-propagates the branch of each cell to lam = dL/dce' and to the
// direct dependence on (ce, cl, fs), gathers lam of the 6 neighbours through
// the diffusion stencil, and sums the parameter partials in fixed order, so
// that the gradients are reproducible run to run:
//   k_adj_fused            all of it in one pass, outputs apart from inputs
//   k_adj_part, _diff, _sum  the same in place, and for beams and thin boxes

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <initializer_list>
#include <mutex>

#include "host_init.h"
#include "mmca_device.h"
#include "mmca_internal.h"

// Workspace of mmca_adjoint_step_noalloc, for callers that cannot allocate:
// lam over the padded cells, then the per-workgroup partial sums.  Each GPU
// holds its own copy of this array until the process ends; every call on
// that GPU uses it, so calls that overlap on one GPU race.
constexpr long long ADJ_SCRATCH_DOUBLES = 1ll << 22;     // 32 MiB
static __device__ __align__(256) double scratch[ADJ_SCRATCH_DOUBLES];

namespace mmca {
namespace {

// Device address of `scratch` on the current device.  The host-side name of
// the array is not a device address: it is looked up once per device with
// that device current, and only the looked-up address is passed to kernels.
constexpr int ADJ_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double *g_scratch_dev[ADJ_MAX_DEVICES] = {};

int adj_scratch_ptr(double **out)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess)
        return MMCA_ERR_HIP;
    if (dev < 0 || dev >= ADJ_MAX_DEVICES)
        return MMCA_ERR_ARG;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev])
    {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
            return MMCA_ERR_HIP;
        g_scratch_dev[dev] = (double *) p;
    }
    *out = g_scratch_dev[dev];
    return MMCA_OK;
}

constexpr int ADJ_BX = 64;
constexpr int ADJ_BY = 4;
constexpr int ADJ_BS = ADJ_BX * ADJ_BY;
constexpr int SUM_BS = 256;

// Derivatives of the folded constants with respect to the parameters:
// rs = d_sol * dtx, rl = d_liq * dtx (growth.c:38-40), D_xt = d_liq / dx / dx * dt
// (growth.c:185-186), km = 1 - k, km_inv = 1 / km, k_inv = 1 / k.
struct Deriv {
    double dtx;       // d rl / d d_liq = d rs / d d_sol
    double dDxt;      // d D_xt / d d_liq
};

long long adj_blocks(const Consts &c)
{
    return (long long) ((c.nx + ADJ_BX - 1) / ADJ_BX) * ((c.ny + ADJ_BY - 1) / ADJ_BY) * c.nz;
}

struct Cell {
    int x, j, k;
    long long idx;
    bool active;
};

// Tile of this workgroup: the hardware places workgroup w on XCD w % 8, so each
// XCD takes one contiguous eighth of the tiles, whose work is equal, and tiles
// that share halo cells share an L2 (128 x 120 x 104: replay 23.7 us with tiles
// dealt one by one, 22.1 with eighths, and no less with two to four planes per
// thread on top of that; the adjoint step in place 66 and 52).  Of a beam block
// the tiles where cells grow evaluate the quadrature, 400 terms a cell, and lie
// side by side: its tiles are dealt one by one (replay of a 128 x 120 x 104 melt
// pool 730 us, 1270 with eighths).
__device__ __forceinline__ int
xcd_eighth()
{
    const int per = gridDim.x / 8;
    return (int) blockIdx.x < 8 * per ? (blockIdx.x % 8) * per + blockIdx.x / 8 : blockIdx.x;
}

template <bool AM = false>
__device__ __forceinline__ Cell
cell_of(const Consts &c)
{
    const int gbx = (c.nx + ADJ_BX - 1) / ADJ_BX, gby = (c.ny + ADJ_BY - 1) / ADJ_BY;
    const long long blk = AM ? (int) blockIdx.x : xcd_eighth();
    Cell q;
    q.x = (int) (blk % gbx) * ADJ_BX + threadIdx.x + 1;
    q.j = (int) ((blk / gbx) % gby) * ADJ_BY + threadIdx.y + 1;
    q.k = (int) (blk / ((long long) gbx * gby)) + 1;
    q.active = (q.x <= c.nx) && (q.j <= c.ny);
    q.idx = q.k * c.sxy + (long long) q.j * c.sx + q.x;
    return q;
}

// neighbours in the diffusion order +x,-x,+y,-y,+z,-z and their mold flags
// (only the padded faces of the box can be mold)
__device__ __forceinline__ void
stencil(const Consts &c, const Cell &q, long long nb[6], int mo[6])
{
    nb[0] = q.idx + 1;
    nb[1] = q.idx - 1;
    nb[2] = q.idx + c.sx;
    nb[3] = q.idx - c.sx;
    nb[4] = q.idx + c.sxy;
    nb[5] = q.idx - c.sxy;
    mo[0] = (q.x == c.nx) ? c.pad_hi[0] : 0;
    mo[1] = (q.x == 1) ? c.pad_lo[0] : 0;
    mo[2] = (q.j == c.ny) ? c.pad_hi[1] : 0;
    mo[3] = (q.j == 1) ? c.pad_lo[1] : 0;
    mo[4] = (q.k == c.nz) ? c.pad_hi[2] : 0;
    mo[5] = (q.k == 1) ? c.pad_lo[2] : 0;
}

template <bool AM>
__global__ void __launch_bounds__(ADJ_BS)
k_replay(Consts c, const unsigned char *code, double sim_time, const double *ce, const double *cl,
         const double *fs, double *ce_o, double *cl_o, double *fs_o)
{
    const Cell q = cell_of<AM>(c);
    if (!q.active)
        return;
    long long nb[6];
    int mo[6];
    stencil(c, q, nb, mo);
    double cln[6], fsn[6];
#pragma unroll
    for (int n = 0; n < 6; ++n)
    {
        cln[n] = cl[nb[n]];
        fsn[n] = fs[nb[n]];
    }
    const double ce_old = ce[q.idx], conc = cl[q.idx], lspfs = fs[q.idx];
    const double ce_new = diffuse_cell(c, ce_old, conc, lspfs, cln, fsn, mo);
    const int br = rec_code(c, code, q.x, q.j, q.k);
    double clv, fsv;
    if (br == MMCA_BRANCH_SOLID)
    {
        clv = ce_new * c.k_inv;
        fsv = lspfs;
    }
    else if (br == MMCA_BRANCH_GROW || br == MMCA_BRANCH_FULL)
    {
        const double Tcell = temp_model<AM>(c, sim_time, q.x, q.j, q.k);
        const double c_int = c.cinit + c.m_inv * (Tcell - c.Tliq);
        const double dce = ce_new - ce_old;
        const double dcl = (c_int - conc) * c.D_xt * 2 + dce / (1 - c.km * lspfs);
        const double dfs = (dcl * (1. - c.km * lspfs) - dce) * c.km_inv / conc;
        clv = conc + dcl;
        fsv = (br == MMCA_BRANCH_GROW) ? lspfs + dfs : 1.0;
    }
    else
    {
        clv = ce_new;
        fsv = 0.0;
    }
    ce_o[q.idx] = ce_new;
    cl_o[q.idx] = clv;
    fs_o[q.idx] = fsv;
}

// What the branch of a cell passes back: lam = dL/dce', the direct
// derivatives with respect to its own (ce, cl, fs), and its terms of the
// derivatives with respect to d_liq and part_coef.
struct BranchAdj {
    double lam, ce, cl, fs, dl, k;
};

// `diffused` gives ce': most waves are in the liquid throughout, where
// nothing depends on it, and a cell for which only lam is wanted (!own) needs
// it where the cell grows.
template <bool AM, typename Diffused>
__device__ __forceinline__ BranchAdj
branch_adjoint(const Consts &c, const Deriv &dv, int br, double sim_time, int x, int j, int k, double ce_old,
               double conc, double lspfs, Diffused diffused, bool own, double ga, double gb, double ge)
{
    BranchAdj r = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    if (br == MMCA_BRANCH_SOLID)
    {
        // cl' = ce' k_inv, fs' = fs
        r.lam = ga + gb * c.k_inv;
        r.fs = ge;
        if (own)
            r.k = -gb * diffused() * c.k_inv * c.k_inv;
    }
    else if (br == MMCA_BRANCH_GROW || br == MMCA_BRANCH_FULL)
    {
        const double Tcell = temp_model<AM>(c, sim_time, x, j, k);
        const double c_int = c.cinit + c.m_inv * (Tcell - c.Tliq);
        const double A = 1 - c.km * lspfs;
        const double dce = diffused() - ce_old;
        const double D2 = c.D_xt * 2;
        const double dcl = (c_int - conc) * D2 + dce / A;
        const double u = dcl * A - dce;
        const double gdfs = (br == MMCA_BRANCH_GROW) ? ge : 0.0;   // FULL: fs' = 1
        // dfs = u km_inv / cl
        const double gu = gdfs * c.km_inv / conc;
        double gq = -gdfs * u * c.km_inv / (conc * conc);
        const double gkminv = gdfs * u / conc;
        // u = dcl A - dce ; cl' = cl + dcl
        const double gdcl = gb + gu * A;
        const double gA = gu * dcl - gdcl * dce / (A * A);
        const double gdce = -gu + gdcl / A;
        // dcl = (c_int - cl) D2 + dce / A
        gq += gb - gdcl * D2;
        const double gD2 = gdcl * (c_int - conc);
        // A = 1 - km fs ; fs' = fs + dfs
        const double gs = gdfs - gA * c.km;
        const double gkm = -gA * lspfs - gkminv * c.km_inv * c.km_inv;
        r.lam = ga + gdce;
        r.ce = -gdce;           // dce = ce' - ce
        r.cl = gq;
        r.fs = gs;
        r.k = -gkm;             // km = 1 - k
        r.dl = gD2 * 2 * dv.dDxt;
    }
    else
    {
        // LIQUID, REMELT: cl' = ce', fs' = 0
        r.lam = ga + gb;
    }
    return r;
}

// The sums of N values over the workgroup, valid in thread 0; s_red holds
// N * (BS / 64) doubles.
template <int BS, int N>
__device__ __forceinline__ void
block_sums(double *t, double *s_red)
{
#pragma unroll
    for (int n = 0; n < N; ++n)
        for (int d = 32; d > 0; d >>= 1)
            t[n] += __shfl_xor(t[n], d, 64);
    const int tid = threadIdx.x;
    if ((tid & 63) == 0)
#pragma unroll
        for (int n = 0; n < N; ++n)
            s_red[n * (BS / 64) + (tid >> 6)] = t[n];
    __syncthreads();
    if (tid == 0)
#pragma unroll
        for (int n = 0; n < N; ++n)
        {
            t[n] = 0.0;
            for (int i = 0; i < BS / 64; ++i)
                t[n] += s_red[n * (BS / 64) + i];
        }
    __syncthreads();
}

// lam's pull-back through a cell's diffusion stencil, as sums over its
// neighbours of r (lam_n - lam), of d (lam_n - lam), of f d and of (1 - f) d,
// with d = cl_n - cl, f = (fs + fs_n) / 2 and r = rs f + rl (1 - f): the
// factors that do not depend on the neighbour stay outside, 11 FP64 operations
// a neighbour (22 with each of the four derivatives formed term by term).  r
// as rl + (rs - rl) f would take one less, but in the solid, where r = rs =
// rl / 3000, it loses 3 digits (9.6e-15 instead of 1e-15 of error in the
// derivatives with respect to the diffusivities over 81 steps).
struct DiffSums {
    double rl, dl, fd, gd;
};

__device__ __forceinline__ void
diff_term(const Consts &c, double lc, double clc, double fsc, double ln, double cln, double fsn, int mo, DiffSums &q)
{
    const double f = 0.5 * (fsc + fsn), g = 1.0 - f;
    const double r = mo ? 0.0 : __builtin_fma(c.rs, f, c.rl * g);
    const double d = mo ? 0.0 : cln - clc;
    const double l = ln - lc;
    q.rl = __builtin_fma(r, l, q.rl);
    q.dl = __builtin_fma(d, l, q.dl);
    q.fd = __builtin_fma(f, d, q.fd);
    q.gd = __builtin_fma(g, d, q.gd);
}

// The derivatives with respect to cl, fs, rl and rs from the sums.
struct DiffAdj {
    double cl, fs, rl, rs;
};

__device__ __forceinline__ DiffAdj
diff_adjoint(const Consts &c, double lc, const DiffSums &q)
{
    return { q.rl, -0.5 * (c.rs - c.rl) * q.dl, lc * q.gd, lc * q.fd };
}

// One adjoint step in one pass over the fields.  A workgroup walks a tile of
// ADJ_TX x TY cells up its planes: at plane kk it forms lam there, for the
// tile and the ring of cells around it (their lam is formed again by the
// neighbouring tiles, by waves of their own), and finishes plane kk - 1, whose
// neighbours' lam are then known.  cl, fs and lam of the planes at hand are in
// LDS, and the loads of a plane are issued a plane ahead.  lam and the direct
// derivatives, 7 of the 19 passes over a field that two kernels make, stay out
// of memory.  The outputs must not overlap the inputs: neighbouring tiles read
// the inputs again.
// Partials of (d_liq, d_sol, part_coef) go to part[3 * blk]; the workgroup
// that finishes last adds their sums, in fixed order, to g_param.
// 128 x 120 x 104 along a trajectory: 51 us against 31 + 33 + 10 of the two
// passes and their sum (before xcd_eighth).  A liquid block stepped again and
// again, in one pass and in two: 24 x 20 x 22 12.0 and 12.4 us, 48 x 41 x 56
// 14.4 and 13.7, 64^3 16.3 and 16.1, 128 x 120 x 104 30 and 52, 256^3 283 and
// 692.  It is bound by
// memory latency: the rings and the planes at the ends of the walks bring the
// 121 MB to some 200, and LDS and registers hold one workgroup per CU (tiles
// of 4, 5, 12 and 13 rows, two workgroups per CU: 49 to 53 us).
constexpr int ADJ_TX = 64;
using u32x2 = unsigned __attribute__((ext_vector_type(2)));

// threads of a workgroup: the tile's, and whole waves for the ring and its corners
constexpr int adj_threads(int ty) { return ADJ_TX * ty + (2 * ADJ_TX + 2 * ty + 4 + 63) / 64 * 64; }

template <int TY>
__global__ void __launch_bounds__(adj_threads(TY))
k_adj_fused(Consts c, Deriv dv, int kz, const unsigned char *code, double sim_time, const double *ce,
            const double *cl, const double *fs, const double *g_ce, const double *g_cl, const double *g_fs,
            double *o_ce, double *o_cl, double *o_fs, double *part, int *done, double *g_param)
{
    constexpr int BS = adj_threads(TY);
    constexpr int CW = ADJ_TX + 4, CN = CW * (TY + 4);    // cl, fs: two cells around the tile
    constexpr int LW = ADJ_TX + 2, LN = LW * (TY + 2);    // lam: one cell around it
    constexpr int RING = 2 * ADJ_TX + 2 * TY, OUTER = RING + 4;
    static_assert(OUTER <= BS - ADJ_TX * TY, "one ring and one outer cell per thread");
    __shared__ double s_cl[4][CN], s_fs[4][CN], s_lam[2][LN];
    __shared__ double s_red[3 * (BS / 64)];

    const int tid = threadIdx.x;
    const int gbx = (c.nx + ADJ_TX - 1) / ADJ_TX, gby = (c.ny + TY - 1) / TY;
    const int w = xcd_eighth();
    const int x0 = (w % gbx) * ADJ_TX + 1, j0 = ((w / gbx) % gby) * TY + 1, z0 = (w / (gbx * gby)) * kz + 1;
    const int z1 = min(z0 + kz - 1, c.nz);

    // Cell t of the cells at distance d around the tile, in tile coordinates:
    // the row below, the row above, the columns left and right.
    auto around = [&](int t, int d, int &ex, int &ey) {
        if (t < 2 * ADJ_TX)
        {
            ex = t & (ADJ_TX - 1);
            ey = (t < ADJ_TX) ? -d : TY - 1 + d;
        }
        else
        {
            t -= 2 * ADJ_TX;
            ex = (t < TY) ? -d : ADJ_TX - 1 + d;
            ey = (t < TY) ? t : t - TY;
        }
    };
    // The first ADJ_TX * TY threads have a cell of the tile, the others one of
    // the ring and load one of the cells around it (cl and fs only).
    const bool tile = tid < ADJ_TX * TY;
    const int r = tid - ADJ_TX * TY;
    int ex = tid & (ADJ_TX - 1), ey = tid / ADJ_TX, ox = 0, oy = 0;
    if (!tile)
    {
        around(min(r, RING - 1), 1, ex, ey);
        if (r < RING)
            around(r, 2, ox, oy);
        else
        {
            ox = (r & 1) ? ADJ_TX : -1;                  // the corners of the ring
            oy = (r & 2) ? TY : -1;
        }
    }
    auto inside = [&](int x, int j, int h) { return x >= 1 - h && x <= c.nx + h && j >= 1 - h && j <= c.ny + h; };
    const int x = x0 + ex, j = j0 + ey;
    const bool used = tile || r < RING, outer = !tile && r < OUTER;
    const bool in = used && inside(x, j, 0);
    // Byte offsets in a plane, whose address stays in scalar registers.  Every
    // lane loads at every plane, lanes and planes outside the box from its
    // edge (no cell inside reads what they get), and stores go through a
    // buffer descriptor that drops the lanes without a cell: with no branch
    // around a memory access the compiler knows how many are in flight and
    // waits for the oldest ones only.
    const unsigned po = used && inside(x, j, 1) ? 8u * (unsigned) (j * c.sx + x) : 0u;
    const unsigned pq = outer && inside(x0 + ox, j0 + oy, 1) ? 8u * (unsigned) ((j0 + oy) * c.sx + x0 + ox) : 0u;
    const unsigned co = in ? 4u * (unsigned) (6 * (j * c.w64 + ((x - 1) >> 6)) + (((x - 1) >> 5) & 1)) : 0u;
    const unsigned ps = tile && in ? po : ~0u;
    const int so = (ey + 2) * CW + ex + 2, sq = (oy + 2) * CW + ox + 2, lo = (ey + 1) * LW + ex + 1;
    const long long cpitch = 24ll * c.w64 * (c.ny + 2);  // bytes of a plane's codes
    auto ld = [](const double *plane, unsigned off) { return *(const double *) ((const char *) plane + off); };
    auto st = [&](double *plane, unsigned off, double v) {
        auto d = __builtin_amdgcn_make_buffer_rsrc(plane, 0, (int) (8u * (unsigned) c.sxy), 0x00027000);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), d, off, 0, 0);
    };
    // loads under way: cl and fs of a plane, for the thread's cell and for the
    // one around the ring; ce, the incoming derivatives and the branch code
    // (the half word of each bit plane that holds the cell's bit)
    double cl_n, fs_n, ocl_n, ofs_n, ce_n, gce_n, gcl_n, gfs_n;
    unsigned w0, w1, w2;
    auto ld_plane = [&](int k) {
        const long long p = min(max(k, 0), c.nz + 1) * c.sxy;
        cl_n = ld(cl + p, po);
        fs_n = ld(fs + p, po);
        ocl_n = ld(cl + p, pq);
        ofs_n = ld(fs + p, pq);
    };
    auto ld_cell = [&](int k) {
        const int kc = min(max(k, 1), c.nz);
        const long long p = kc * c.sxy;
        ce_n = ld(ce + p, po);
        gce_n = ld(g_ce + p, po);
        gcl_n = ld(g_cl + p, po);
        gfs_n = ld(g_fs + p, po);
        const unsigned char *q = code + kc * cpitch;
        w0 = *(const unsigned *) (q + co);
        w1 = *(const unsigned *) (q + (co + 8u));
        w2 = *(const unsigned *) (q + (co + 16u));
    };
    auto put_plane = [&](int k) {
        if (used)
        {
            s_cl[k & 3][so] = cl_n;
            s_fs[k & 3][so] = fs_n;
        }
        if (outer)
        {
            s_cl[k & 3][sq] = ocl_n;
            s_fs[k & 3][sq] = ofs_n;
        }
    };
    const int mx1 = (x == c.nx) ? c.pad_hi[0] : 0, mx0 = (x == 1) ? c.pad_lo[0] : 0;
    const int my1 = (j == c.ny) ? c.pad_hi[1] : 0, my0 = (j == 1) ? c.pad_lo[1] : 0;

    double lam2 = 0.0, lam1 = 0.0;                       // own lam of kk-2 and kk-1
    double dce = 0.0, dcl = 0.0, dfs = 0.0;              // direct derivatives of kk-1
    double p_dl = 0.0, p_ds = 0.0, p_k = 0.0;
    ld_plane(z0 - 2);
    put_plane(z0 - 2);
    ld_plane(z0 - 1);
    put_plane(z0 - 1);
    __builtin_amdgcn_sched_barrier(0);
    ld_plane(z0);
    __builtin_amdgcn_sched_barrier(0);
    ld_cell(z0 - 1);
    __builtin_amdgcn_sched_barrier(0);
    // as many stores in flight behind the loads as in every later turn (no
    // lane takes part), for the count that the loop waits for
    st(o_ce + c.sxy, ~0u, 0.0);
    st(o_cl + c.sxy, ~0u, 0.0);
    st(o_fs + c.sxy, ~0u, 0.0);
    for (int kk = z0 - 1; kk <= z1 + 1; ++kk)
    {
        put_plane(kk + 1);                               // over plane kk - 3
        __builtin_amdgcn_sched_barrier(0);
        ld_plane(kk + 2);
        __syncthreads();

        // of planes kk - 2 and kk + 1 only the thread's own words are read
        const double *C = s_cl[kk & 3] + so, *F = s_fs[kk & 3] + so;
        const double *Cu = s_cl[(kk + 1) & 3] + so, *Fu = s_fs[(kk + 1) & 3] + so;
        const double *Cd = s_cl[(kk + 3) & 3] + so, *Fd = s_fs[(kk + 3) & 3] + so;
        double lam0 = 0.0, ece = 0.0, ecl = 0.0, efs = 0.0;
        const bool here = kk >= z0 && kk <= z1;
        if (in && (here || (tile && kk >= 1 && kk <= c.nz)))
        {
            auto diffused = [&]() {
                const int mo[6] = { mx1, mx0, my1, my0, (kk == c.nz) ? c.pad_hi[2] : 0, (kk == 1) ? c.pad_lo[2] : 0 };
                const double cn[6] = { C[1], C[-1], C[CW], C[-CW], Cu[0], Cd[0] };
                const double fn[6] = { F[1], F[-1], F[CW], F[-CW], Fu[0], Fd[0] };
                return diffuse_cell(c, ce_n, C[0], F[0], cn, fn, mo);
            };
            const int bit = (x - 1) & 31;
            const int br = (int) ((w0 >> bit) & 1u) | (int) (((w1 >> bit) & 1u) << 1) | (int) (((w2 >> bit) & 1u) << 2);
            const BranchAdj d = branch_adjoint<false>(c, dv, br, sim_time, x, j, kk, ce_n, C[0], F[0], diffused,
                                                   here && tile, gce_n, gcl_n, gfs_n);
            lam0 = d.lam;
            ece = d.ce;
            ecl = d.cl;
            efs = d.fs;
            if (here && tile)
            {
                p_dl += d.dl;
                p_k += d.k;
            }
        }
        if (used)
            s_lam[kk & 1][lo] = lam0;
        __builtin_amdgcn_sched_barrier(0);
        ld_cell(kk + 1);
        __builtin_amdgcn_sched_barrier(0);

        const int m = kk - 1;
        double vce = 0.0, vcl = 0.0, vfs = 0.0;
        if (m >= z0 && tile && in)
        {
            const double *L = s_lam[m & 1] + lo;
            const double clc = Cd[0], fsc = Fd[0];
            DiffSums u = { 0.0, 0.0, 0.0, 0.0 };
            diff_term(c, lam1, clc, fsc, L[1], Cd[1], Fd[1], mx1, u);
            diff_term(c, lam1, clc, fsc, L[-1], Cd[-1], Fd[-1], mx0, u);
            diff_term(c, lam1, clc, fsc, L[LW], Cd[CW], Fd[CW], my1, u);
            diff_term(c, lam1, clc, fsc, L[-LW], Cd[-CW], Fd[-CW], my0, u);
            diff_term(c, lam1, clc, fsc, lam0, C[0], F[0], (m == c.nz) ? c.pad_hi[2] : 0, u);
            diff_term(c, lam1, clc, fsc, lam2, s_cl[(kk + 2) & 3][so], s_fs[(kk + 2) & 3][so], (m == 1) ? c.pad_lo[2] : 0, u);
            const DiffAdj q = diff_adjoint(c, lam1, u);
            vce = dce + lam1;
            vcl = dcl + q.cl;
            vfs = dfs + q.fs;
            p_dl += q.rl * dv.dtx;
            p_ds += q.rs * dv.dtx;
        }
        const long long p = max(m, 1) * c.sxy;
        const unsigned off = m >= z0 ? ps : ~0u;
        st(o_ce + p, off, vce);
        st(o_cl + p, off, vcl);
        st(o_fs + p, off, vfs);

        lam2 = lam1, lam1 = lam0;
        dce = ece, dcl = ecl, dfs = efs;
    }

    double t[3] = { p_dl, p_ds, p_k };
    block_sums<BS, 3>(t, s_red);
    if (tid == 0)
#pragma unroll
        for (int n = 0; n < 3; ++n)
            st_agent(&part[3 * (long long) blockIdx.x + n], t[n]);
    const int nblk = gridDim.x;
    if (!last_workgroup(done, nblk))
        return;
    t[0] = t[1] = t[2] = 0.0;
    for (int i = tid; i < nblk; i += BS)
#pragma unroll
        for (int n = 0; n < 3; ++n)
            t[n] += ld_agent(&part[3 * (long long) i + n]);
    block_sums<BS, 3>(t, s_red);
    if (tid == 0)
#pragma unroll
        for (int n = 0; n < 3; ++n)
            g_param[n] += t[n];
}

// The same step in two passes: the outputs may be the incoming derivatives,
// which only the cell itself reads in each pass.  Also the way of beam blocks
// and thin boxes (adj_one_pass).
// First the branch: lam, and the direct derivatives; partials of (d_liq,
// part_coef) per workgroup into part[2 * blk].
template <bool AM>
__global__ void __launch_bounds__(ADJ_BS)
k_adj_part(Consts c, Deriv dv, const unsigned char *code, double sim_time, const double *ce,
           const double *cl, const double *fs, const double *g_ce, const double *g_cl, const double *g_fs,
           double *lam, double *gce_in, double *gcl_in, double *gfs_in, double *part)
{
    __shared__ double s_red[ADJ_BS / 64];
    const Cell q = cell_of<AM>(c);
    double p_dl = 0.0, p_k = 0.0;
    if (q.active)
    {
        const double ce_old = ce[q.idx], conc = cl[q.idx], lspfs = fs[q.idx];
        auto diffused = [&]() {
            long long nb[6];
            int mo[6];
            stencil(c, q, nb, mo);
            double cln[6], fsn[6];
#pragma unroll
            for (int n = 0; n < 6; ++n)
            {
                cln[n] = cl[nb[n]];
                fsn[n] = fs[nb[n]];
            }
            return diffuse_cell(c, ce_old, conc, lspfs, cln, fsn, mo);
        };
        const int br = rec_code(c, code, q.x, q.j, q.k);
        const BranchAdj r = branch_adjoint<AM>(c, dv, br, sim_time, q.x, q.j, q.k, ce_old, conc, lspfs, diffused, true,
                                               g_ce[q.idx], g_cl[q.idx], g_fs[q.idx]);
        lam[q.idx] = r.lam;
        gce_in[q.idx] = r.ce;
        gcl_in[q.idx] = r.cl;
        gfs_in[q.idx] = r.fs;
        p_dl = r.dl;
        p_k = r.k;
    }
    const double s_dl = block_sum<ADJ_BS>(p_dl, s_red);
    __syncthreads();
    const double s_k = block_sum<ADJ_BS>(p_k, s_red);
    if (threadIdx.x == 0 && threadIdx.y == 0)
    {
        part[2 * (long long) blockIdx.x] = s_dl;
        part[2 * (long long) blockIdx.x + 1] = s_k;
    }
}

// Then the stencil: adds lam's pull-back to (ce, cl, fs); partials of (d_liq,
// d_sol) per workgroup into part[2 * blk].  lam is zero on the halo (halo
// cells are never updated).
__global__ void __launch_bounds__(ADJ_BS)
k_adj_diff(Consts c, Deriv dv, const double *cl, const double *fs, const double *lam, double *gce_in,
           double *gcl_in, double *gfs_in, double *part)
{
    __shared__ double s_red[ADJ_BS / 64];
    const Cell q = cell_of(c);
    double p_dl = 0.0, p_ds = 0.0;
    if (q.active)
    {
        long long nb[6];
        int mo[6];
        stencil(c, q, nb, mo);
        double ln[6], cln[6], fsn[6];
#pragma unroll
        for (int n = 0; n < 6; ++n)
        {
            ln[n] = lam[nb[n]];
            cln[n] = cl[nb[n]];
            fsn[n] = fs[nb[n]];
        }
        const double lc = lam[q.idx];
        const double clc = cl[q.idx], fsc = fs[q.idx];
        DiffSums u = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
        for (int n = 0; n < 6; ++n)
            diff_term(c, lc, clc, fsc, ln[n], cln[n], fsn[n], mo[n], u);
        const DiffAdj r = diff_adjoint(c, lc, u);
        gce_in[q.idx] += lc;
        gcl_in[q.idx] += r.cl;
        gfs_in[q.idx] += r.fs;
        p_dl = r.rl * dv.dtx;
        p_ds = r.rs * dv.dtx;
    }
    const double s_dl = block_sum<ADJ_BS>(p_dl, s_red);
    __syncthreads();
    const double s_ds = block_sum<ADJ_BS>(p_ds, s_red);
    if (threadIdx.x == 0 && threadIdx.y == 0)
    {
        part[2 * (long long) blockIdx.x] = s_dl;
        part[2 * (long long) blockIdx.x + 1] = s_ds;
    }
}

// g_param[0..2] += sums of the partials: (d_liq, part_coef) from pa,
// (d_liq, d_sol) from pb.  One workgroup; fixed summation order.
__global__ void __launch_bounds__(SUM_BS)
k_adj_sum(const double *pa, const double *pb, long long nblk, double *g_param)
{
    __shared__ double s_red[SUM_BS / 64];
    double v[4] = { 0.0, 0.0, 0.0, 0.0 };
    for (long long i = threadIdx.x; i < nblk; i += SUM_BS)
    {
        v[0] += pa[2 * i];
        v[1] += pa[2 * i + 1];
        v[2] += pb[2 * i];
        v[3] += pb[2 * i + 1];
    }
    double t[4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
    {
        t[m] = block_sum<SUM_BS>(v[m], s_red);
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        g_param[0] += t[0] + t[2];
        g_param[1] += t[3];
        g_param[2] += t[1];
    }
}

// lam = 0 on the halo cells of the padded box (the stencil reads them; they
// are never written by k_adj_part)
__global__ void __launch_bounds__(256)
k_zero_halo(Consts c, double *lam)
{
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.P)
        return;
    const int x = (int) (i % c.sx);
    const long long r = i / c.sx;
    const int j = (int) (r % (c.ny + 2));
    const int k = (int) (r / (c.ny + 2));
    if (x == 0 || x > c.nx || j == 0 || j > c.ny || k == 0 || k > c.nz)
        lam[i] = 0.0;
}

constexpr int ADJ_TY = 8;

long long adj_tiles(const Consts &c)
{
    return (long long) ((c.nx + ADJ_TX - 1) / ADJ_TX) * ((c.ny + ADJ_TY - 1) / ADJ_TY);
}

// Planes that a workgroup of k_adj_fused walks.  One workgroup fits a CU, and
// a walk takes two planes more than it finishes: the fewest rounds of the
// chip's 256 CUs times the planes of a walk.  128 x 120 x 104 (30 tiles): 13
// planes (240 workgroups) 50 us, 7 (450) 59, 15 (210) 55, 4 (780) 68.
// *cost: that product.
int adj_planes(const Consts &c, long long *cost)
{
    const long long t = adj_tiles(c);
    int best = 1;
    *cost = -1;
    for (int kz = 1; kz <= std::min(64, c.nz); ++kz)
    {
        const long long rounds = (t * ((c.nz + kz - 1) / kz) + 255) / 256;
        if (*cost < 0 || rounds * (kz + 2) < *cost)
        {
            best = kz;
            *cost = rounds * (kz + 2);
        }
    }
    return best;
}

// True where one pass is the faster way.  Not in boxes of one or two rows or
// planes, where the walks' rows are idle or two of three planes walked are not
// finished, unless the walks are so short that one launch less decides: one pass
// and two take 74 and 40 us for 1000 x 1000 x 1 (cost 24), 85 and 69 for 1000 x
// 1000 x 2 (32), 18.5 and 16.6 for 300 x 1 x 300 (8), 16.3 and 14.8 for 64 x 1 x
// 1000 (6), 19.6 and 18.7 for 1000 x 2 x 100 (9); but 13.4 and 15.2 for 300 x 300 x
// 1 (3), 14.9 and 17.1 for 300 x 300 x 2 (4), 12.0 and 14.4 for 128 x 1 x 64 (3);
// and 97 and 100 for 1000 x 1000 x 3, 19.1 and 19.9 for 300 x 3 x 300.
// Not for beam blocks either: the quadratures of growing cells in successive
// planes of a walk follow one another (128 x 120 x 104 melt pool: 9350 us in one
// pass, 700 in two).
bool adj_one_pass(const Consts &c, long long cost)
{
    return !c.am && ((c.ny >= 3 && c.nz >= 3) || cost <= 4);
}

// True when none of the outputs overlaps an input or another output.
bool adj_separate(const Consts &c, std::initializer_list<const double *> out, std::initializer_list<const double *> in)
{
    const uintptr_t n = (uintptr_t) c.P * sizeof(double);
    auto apart = [&](const double *a, const double *b) {
        const uintptr_t p = (uintptr_t) a, q = (uintptr_t) b;
        return p + n <= q || q + n <= p;
    };
    for (auto o = out.begin(); o != out.end(); ++o)
    {
        for (const double *i : in)
            if (!apart(*o, i))
                return false;
        for (auto p = o + 1; p != out.end(); ++p)
            if (!apart(*o, *p))
                return false;
    }
    return true;
}

// The launches of one adjoint step; lam holds P doubles, pa and pb 2 * nblk each.
hipError_t
adjoint_launch(const Consts &c, const Deriv &dv, uint64_t timestep, const uint8_t *codes, const double *ce,
               const double *cl, const double *fs, const double *g_ce, const double *g_cl, const double *g_fs,
               double *g_ce_in, double *g_cl_in, double *g_fs_in, double *g_param, double *lam, double *pa,
               double *pb, hipStream_t s)
{
    const long long nblk = adj_blocks(c);
    const double sim_time = timestep * c.dt;
    // one pass needs outputs apart from the inputs, and a plane's byte offsets in 31 bits
    long long cost = 0;
    const int kz = adj_planes(c, &cost);
    if (adj_one_pass(c, cost) && c.sxy <= (1ll << 28) - 1 &&
        adj_separate(c, { g_ce_in, g_cl_in, g_fs_in }, { ce, cl, fs, g_ce, g_cl, g_fs }))
    {
        const dim3 fgrid((unsigned) (adj_tiles(c) * ((c.nz + kz - 1) / kz)));
        // the first cell of lam is a halo cell, 0 between the calls
        int *done = (int *) lam;
        hipLaunchKernelGGL(k_adj_fused<ADJ_TY>, fgrid, dim3(adj_threads(ADJ_TY)), 0, s, c, dv, kz, codes, sim_time, ce,
                           cl, fs, g_ce, g_cl, g_fs, g_ce_in, g_cl_in, g_fs_in, pa, done, g_param);
        return hipGetLastError();
    }
    const dim3 grid((unsigned) nblk), blk(ADJ_BX, ADJ_BY);
    if (c.am)
        hipLaunchKernelGGL(k_adj_part<true>, grid, blk, 0, s, c, dv, codes, sim_time, ce, cl, fs, g_ce, g_cl, g_fs,
                           lam, g_ce_in, g_cl_in, g_fs_in, pa);
    else
        hipLaunchKernelGGL(k_adj_part<false>, grid, blk, 0, s, c, dv, codes, sim_time, ce, cl, fs, g_ce, g_cl,
                           g_fs, lam, g_ce_in, g_cl_in, g_fs_in, pa);
    hipLaunchKernelGGL(k_adj_diff, grid, blk, 0, s, c, dv, cl, fs, lam, g_ce_in, g_cl_in, g_fs_in, pb);
    hipLaunchKernelGGL(k_adj_sum, dim3(1), dim3(SUM_BS), 0, s, pa, pb, nblk, g_param);
    return hipGetLastError();
}

int adj_consts(const mmca_params *p, Consts &c, Deriv &dv)
{
    if (!p)
        return MMCA_ERR_ARG;
    mmca_params q = *p;
    q.precision = MMCA_PREC_FP64;
    const int st = build_consts(q, c);
    if (st != MMCA_OK)
        return st;
    dv.dtx = p->dt / (p->cell_size * p->cell_size);
    dv.dDxt = 1.0 / p->cell_size / p->cell_size * p->dt;
    return MMCA_OK;
}

}  // namespace
}  // namespace mmca

extern "C" {

int mmca_replay_step(const mmca_params *params, uint64_t timestep, const uint8_t *codes, const double *ce,
                     const double *cl, const double *fs, double *ce_out, double *cl_out, double *fs_out,
                     void *stream)
{
    using namespace mmca;
    Consts c;
    Deriv dv;
    int st = adj_consts(params, c, dv);
    if (st != MMCA_OK)
        return st;
    if (!codes || !ce || !cl || !fs || !ce_out || !cl_out || !fs_out)
        return MMCA_ERR_ARG;
    if (ce_out == ce || cl_out == cl || fs_out == fs || cl_out == fs || fs_out == cl)
        return MMCA_ERR_ARG;     // the stencil reads neighbours of the inputs
    hipStream_t s = (hipStream_t) stream;
    const double sim_time = timestep * c.dt;
    const dim3 grid((unsigned) adj_blocks(c)), blk(ADJ_BX, ADJ_BY);
    if (c.am)
        hipLaunchKernelGGL(k_replay<true>, grid, blk, 0, s, c, codes, sim_time, ce, cl, fs, ce_out, cl_out, fs_out);
    else
        hipLaunchKernelGGL(k_replay<false>, grid, blk, 0, s, c, codes, sim_time, ce, cl, fs, ce_out, cl_out,
                           fs_out);
    return hipGetLastError() == hipSuccess ? MMCA_OK : MMCA_ERR_HIP;
}

int mmca_record_bytes(const mmca_params *params, int64_t *bytes_per_step)
{
    using namespace mmca;
    Consts c;
    Deriv dv;
    int st = adj_consts(params, c, dv);
    if (st != MMCA_OK)
        return st;
    if (!bytes_per_step)
        return MMCA_ERR_ARG;
    *bytes_per_step = (int64_t) sizeof(unsigned long long) * rec_words(c);
    return MMCA_OK;
}

int mmca_adjoint_workspace_bytes(const mmca_params *params, int64_t *bytes)
{
    using namespace mmca;
    Consts c;
    Deriv dv;
    int st = adj_consts(params, c, dv);
    if (st != MMCA_OK)
        return st;
    if (!bytes)
        return MMCA_ERR_ARG;
    *bytes = (int64_t) sizeof(double) * (c.P + 4 * adj_blocks(c));
    return MMCA_OK;
}

int mmca_adjoint_step(const mmca_params *params, uint64_t timestep, const uint8_t *codes, const double *ce,
                      const double *cl, const double *fs, const double *g_ce, const double *g_cl,
                      const double *g_fs, double *g_ce_in, double *g_cl_in, double *g_fs_in, double *g_param,
                      void *workspace, void *stream)
{
    using namespace mmca;
    Consts c;
    Deriv dv;
    int st = adj_consts(params, c, dv);
    if (st != MMCA_OK)
        return st;
    if (!codes || !ce || !cl || !fs || !g_ce || !g_cl || !g_fs || !g_ce_in || !g_cl_in || !g_fs_in ||
        !g_param || !workspace)
        return MMCA_ERR_ARG;
    const long long nblk = adj_blocks(c);
    double *lam = (double *) workspace;
    double *pa = lam + c.P;
    double *pb = pa + 2 * nblk;
    return adjoint_launch(c, dv, timestep, codes, ce, cl, fs, g_ce, g_cl, g_fs, g_ce_in, g_cl_in, g_fs_in, g_param,
                          lam, pa, pb, (hipStream_t) stream) == hipSuccess
               ? MMCA_OK
               : MMCA_ERR_HIP;
}

int mmca_adjoint_step_noalloc(const mmca_params *params, uint64_t timestep, const uint8_t *codes,
                              const double *ce, const double *cl, const double *fs, const double *g_ce,
                              const double *g_cl, const double *g_fs, double *g_ce_in, double *g_cl_in,
                              double *g_fs_in, double *g_param, void *stream)
{
    using namespace mmca;
    Consts c;
    Deriv dv;
    int st = adj_consts(params, c, dv);
    if (st != MMCA_OK)
        return st;
    if (!codes || !ce || !cl || !fs || !g_ce || !g_cl || !g_fs || !g_ce_in || !g_cl_in || !g_fs_in || !g_param)
        return MMCA_ERR_ARG;
    const long long nblk = adj_blocks(c);
    if (c.P + 4 * nblk > ADJ_SCRATCH_DOUBLES)
    {
        fprintf(stderr, "mmca_adjoint_step_noalloc: %lld padded cells need %lld bytes of workspace, above the "
                        "%lld of its fixed device array\n",
                (long long) c.P, (long long) sizeof(double) * (c.P + 4 * nblk),
                (long long) sizeof(double) * ADJ_SCRATCH_DOUBLES);
        return MMCA_ERR_ARG;
    }
    double *lam = nullptr;
    st = adj_scratch_ptr(&lam);
    if (st != MMCA_OK)
        return st;
    double *pa = lam + c.P;
    double *pb = pa + 2 * nblk;
    hipStream_t s = (hipStream_t) stream;
    // a previous call (another shape) may have left values where this shape's halo lies
    hipLaunchKernelGGL(k_zero_halo, dim3((unsigned) ((c.P + 255) / 256)), dim3(256), 0, s, c, lam);
    return adjoint_launch(c, dv, timestep, codes, ce, cl, fs, g_ce, g_cl, g_fs, g_ce_in, g_cl_in, g_fs_in, g_param,
                          lam, pa, pb, s) == hipSuccess
               ? MMCA_OK
               : MMCA_ERR_HIP;
}

}  // extern "C"
