// HIP kernels of the CA step for gfx950 (CDNA4, wave64).
//
// One step (doiteration, calculate.c:193-352) on one subblock is five
// launches on the context's stream:
//   k_nuc_detect    cell_nucleation (grain.c:1222-1318) over the sorted site list
//                   and, in the workgroup that finishes last, activateNewGrains
//                   (grain.c:841-916): ids in site order
//   k_solute_rw     diffusion + partitioning (growth.c:30-170, 177-276),
//                   fused, and a 1-bit "solid" mask of gr > 0
//   k_list_count    interface-list membership counts from the mask
//                   (grow_cell_reduction, growth.c:461-538) and, in the
//                   workgroup that finishes last, their exclusive scan ->
//                   raster-order slots
//   k_list_write    the list itself (diff_id) in raster order
//   k_capture       capture_octahedra_diffuse (growth.c:574-807) over the
//                   list slots, dealt evenly over the whole grid, with the
//                   octahedron half-diagonal of each candidate neighbour
//                   computed on the fly (grow_octahedra, growth.c:339-407)
// A Gaussian-beam block adds the approximate beam temperature before them
// (k_beam_ax, k_beam_field) and k_beam_finish after the solute kernel.
//
// Arithmetic follows the reference's operation order and is compiled with
// -ffp-contract=off: FP64 results are bit-identical with the reference CPU
// build.  The Gaussian-beam temperature's exp is a restatement of the host C
// library's (mmca_exp.h).

#include <hip/hip_runtime.h>

#include <algorithm>

#include "mmca_device.h"
#include "mmca_internal.h"

namespace mmca {

// Ping-pong buffer `buf` (0/1) of a field, chosen with a select rather than an
// indexed load, so that a private copy of DevBufs stays in registers.
__device__ __forceinline__ MMCA_GLOBAL double *fs_buf(const DevBufs &b, int buf) { return G(buf ? b.fs[1] : b.fs[0]); }
__device__ __forceinline__ MMCA_GLOBAL double *cl_buf(const DevBufs &b, int buf) { return G(buf ? b.cl[1] : b.cl[0]); }
__device__ __forceinline__ MMCA_GLOBAL float *cl32_buf(const DevBufs &b, int buf) { return G(buf ? b.cl32[1] : b.cl32[0]); }

// Solute storage: FP64 values, or FP32 deviations from c0 (F32).  Arithmetic
// is FP64 in both cases.
template <bool F32>
__device__ __forceinline__ double
ld_ce(const DevBufs &b, const Consts &c, long long i)
{
    return F32 ? c.cinit + (double) G(b.ce32)[i] : G(b.ce)[i];
}

template <bool F32>
__device__ __forceinline__ double
ld_cl(const DevBufs &b, const Consts &c, int buf, long long i)
{
    return F32 ? c.cinit + (double) cl32_buf(b, buf)[i] : cl_buf(b, buf)[i];
}

// The solute kernel writes each cell of ce, cl and fs once per step and the
// later kernels of the step read few of them back (capture), so these stores
// are non-temporal: streamed past the caches, coherent at the kernel's end.
template <typename T>
__device__ __forceinline__ void
st_stream(MMCA_GLOBAL T *p, long long i, T v)
{
    __builtin_nontemporal_store(v, &p[i]);
}

// store ce; returns the FP64 solute lost to the FP32 rounding (0 for FP64)
template <bool F32>
__device__ __forceinline__ double
st_ce(const DevBufs &b, const Consts &c, long long i, double v)
{
    if (F32)
    {
        const double dev = v - c.cinit;
        const float f = (float) dev;
        st_stream(G(b.ce32), i, f);
        return dev - (double) f;
    }
    st_stream(G(b.ce), i, v);
    return 0.0;
}

template <bool F32>
__device__ __forceinline__ void
st_cl(const DevBufs &b, const Consts &c, int buf, long long i, double v)
{
    if (F32)
        st_stream(cl32_buf(b, buf), i, (float) (v - c.cinit));
    else
        st_stream(cl_buf(b, buf), i, v);
}

// Compensated (Kahan) addition of a workgroup's residual into its ledger slot.
__device__ __forceinline__ void
ledger_add(const DevBufs &b, long long slot, double v)
{
    double s = G(b.ledger)[2 * slot], comp = G(b.ledger)[2 * slot + 1];
    double y = v - comp;
    double t = s + y;
    comp = (t - s) - y;
    G(b.ledger)[2 * slot] = t;
    G(b.ledger)[2 * slot + 1] = comp;
}

// ---------------------------------------------------------------------------
// Block-wide exclusive scan of 0/1 flags with wave ballots.  NW = waves/block.
template <int NW>
__device__ __forceinline__ int
block_exscan_flag(int flag, int *total, int *s_w)
{
    unsigned long long bal = __ballot(flag);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int r = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0)
        s_w[w] = __popcll(bal);
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i)
    {
        int v = s_w[i];
        off += (i < w) ? v : 0;
        tot += v;
    }
    __syncthreads();
    *total = tot;
    return off + r;
}

// Block-wide exclusive scan of small non-negative ints.
template <int NW>
__device__ __forceinline__ int
block_exscan_int(int v, int *total, int *s_w)
{
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
    {
        int t = __shfl_up(incl, d, 64);
        if (lane >= d)
            incl += t;
    }
    if (lane == 63)
        s_w[w] = incl;
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i)
    {
        int x = s_w[i];
        off += (i < w) ? x : 0;
        tot += x;
    }
    __syncthreads();
    *total = tot;
    return off + incl - v;
}

// Domain of workgroup w: the last d with off[d] <= w (domains without work
// share their offset with the next domain).
__device__ __forceinline__ int
find_dom(const long long *off, int ndom, long long w)
{
    int lo = 0, hi = ndom - 1;
    while (lo < hi)
    {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= w)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
constexpr int NUC_BS = 256;

// A cell that becomes solid between lean steps: from the next step on its ce
// is read, which for a liquid cell equals cl and need not have been written.
__device__ __forceinline__ void
put_ce_of_liquid(const DevBufs &b, int buf, long long idx)
{
    G(b.ce)[idx] = cl_buf(b, buf)[idx];
}

// Event ordering and activateNewGrains/createGrains on one rank
// (grain.c:841-916, 348-425), one workgroup.
// mode: 1 = order the detected events, 2 = activate, 4 = advance the timestep
// (k_nuc_detect: 8 = detect at the next timestep without advancing).
// nev1 >= 0: the number of events of a domain with one detecting workgroup,
// already in order in `events`.
__device__ __forceinline__ void
nuc_activate(const DevBufs &b, const Consts &c, int mode, int nev1, int lean, int cur)
{
    __shared__ int s_w[NUC_BS / 64];
    __shared__ int s_nev;
    const int nblk = (b.nsites + NUC_BS - 1) / NUC_BS;
    Counters *cnt = b.cnt;
    const int tid = threadIdx.x;
    const unsigned long long ts = cnt->timestep + ((mode & 4) ? 1ull : 0ull);
    if (nev1 >= 0)
    {
        if (tid == 0)
        {
            s_nev = nev1;
            cnt->n_events = nev1;
        }
    }
    else if (mode & 1)
    {
        // exclusive scan of the per-workgroup counts, then concatenate
        int carry = 0;
        for (int base = 0; base < nblk; base += NUC_BS)
        {
            int blk = base + tid;
            int v = (blk < nblk) ? ld_agent(&b.ev_cnt[blk]) : 0;
            int tot;
            int off = carry + block_exscan_int<NUC_BS / 64>(v, &tot, s_w);
            for (int i = 0; i < v; ++i)
                G(b.events)[off + i] = ld_agent(&b.ev_blk[blk * NUC_BS + i]);
            carry += tot;
        }
        if (tid == 0)
        {
            s_nev = carry;
            cnt->n_events = carry;
        }
    }
    else if (tid == 0)
        s_nev = cnt->n_events;
    __syncthreads();
    const int nev = s_nev;
    if ((mode & 2) && nev > 0)
    {
        const int base_id = cnt->num_grains;
        const int rnd0 = cnt->random_used;
        const long long maxg = c.max_total_grains;
        int rused = 0;
        for (int base = 0; base < nev; base += NUC_BS)
        {
            int e = base + tid;
            int isev = e < nev;
            int s = isev ? G(b.events)[e] : 0;
            int fixed = isev ? G(b.site_fixed)[s] : -1;
            int israndom = isev && fixed < 0;
            int rtot;
            int rrank = block_exscan_flag<NUC_BS / 64>(israndom, &rtot, s_w);
            if (isev)
            {
                long long id = (long long) base_id + e;
                if (id <= maxg)
                {
                    int idx = G(b.site_idx)[s];
                    if (lean == 1 || lean == 2)
                        put_ce_of_liquid(b, cur, idx);
                    G(b.gr)[idx] = (int) id;
                    const double *rot;
                    int src;
                    if (fixed >= 0)
                    {
                        rot = b.fixed_rot + 9 * (long long) fixed;
                        src = fixed;
                    }
                    else
                    {
                        int k = rnd0 + rused + rrank;
                        rot = b.rand_rot + 9 * (long long) k;
                        src = -(k + 1);
                    }
                    for (int q = 0; q < 9; ++q)
                        b.g_rot[9 * id + q] = rot[q];
                    G(b.g_cell)[id] = idx;
                    G(b.g_step)[id] = ts;
                    G(b.g_src)[id] = src;
                }
            }
            rused += rtot;
        }
        __syncthreads();
        if (tid == 0)
        {
            long long total = (long long) base_id + nev;
            if (total > maxg + 1)
            {
                // grain.c:868-888: with every slot taken nothing is activated;
                // otherwise createGrains runs past MaxTotGrains and aborts
                // (grain.c:361-366) after creating the grains that fit.
                if ((long long) base_id != maxg + 1)
                {
                    cnt->status = MMCA_ERR_GRAIN_CAPACITY;
                    cnt->failed_step = ts;
                }
            }
            else
            {
                cnt->num_grains = (int) total;
                cnt->random_used = rnd0 + rused;
                cnt->new_grains += nev;
            }
        }
    }
    if ((mode & 4) && tid == 0)
        cnt->timestep = ts;
}

// activation on its own (mmca_activate_new_grains)
__global__ void __launch_bounds__(NUC_BS)
k_nuc_activate(View V, int mode)
{
    const DevBufs b = V.dom[blockIdx.x].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[blockIdx.x].c;
    if (b.cnt->status != MMCA_OK)
        return;
    nuc_activate(b, c, mode, -1, 0, 0);
}

// cell_nucleation (grain.c:1222-1318): one thread per site, sites sorted by
// padded index; each workgroup compacts its events in site order.  The
// workgroup of a domain that finishes last orders them and, by `mode`,
// activates the grains (nuc_activate): one launch where detection and
// activation took two of 4.6 us each, nearly all of it launch latency.
__global__ void __launch_bounds__(NUC_BS)
k_nuc_detect(View V, int mode, int cur)
{
    __shared__ int s_w[NUC_BS / 64];
    const int d = find_dom(V.off_nuc, V.ndom, blockIdx.x);
    const long long blk = blockIdx.x - V.off_nuc[d];
    const DevBufs b = V.dom[d].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[d].c;
    const MMCA_GLOBAL Counters *cnt = G(b.cnt);
    if (cnt->status != MMCA_OK)
        return;
    const unsigned long long ts = cnt->timestep + ((mode & 12) ? 1ull : 0ull);
    const double sim_time = ts * c.dt;
    const int s = (int) blk * NUC_BS + threadIdx.x;
    int flag = 0;
    if (s < b.nsites)
    {
        int idx = G(b.site_idx)[s];
        int z = (int) (idx / c.sxy);
        int rem = (int) (idx - z * c.sxy);
        int y = rem / c.sx;
        int x = rem - y * c.sx;
        double T;
        if (c.am)
        {
            // The tests below read T only through comparisons (undercooling
            // falls with T where the slope m is constant): where they all come
            // out the same at both ends of the approximate temperature's
            // interval, it will do.
            T = (double) G(b.temp32)[idx];
            const double d = beam_margin(c, T);
            const double lo = T - d, hi = T + d;
            const double cl = c.f32 ? ld_cl<true>(b, c, cur, idx) : ld_cl<false>(b, c, cur, idx);
            const double add = c.mc * (cl - c.cinit), thr = (double) G(b.site_thr)[s];
            const bool same = (lo > c.Tliq || hi <= c.Tliq) && (lo >= c.Tsol || hi < c.Tsol) &&
                              ((c.Tliq - hi) + add > thr || (c.Tliq - lo) + add <= thr);
            if (!(c.ma == 0.0 && c.mb == 0.0 && same))
                T = temp_model<true>(c, sim_time, x, y, z);
        }
        else
            T = temp_model<false>(c, sim_time, x, y, z);
        int layerno = 1, initnuc = 1;
        if (c.am)
        {
            // tempUpdateSB_int sets lsindex before nucleation (temperature.c:256-259)
            if (T > c.Tliq)
                G(b.site_ls)[s] = 1;
            if (c.am_layers == 1)
                layerno = 1;
            else if (c.am_layers > 1 && G(b.site_ls)[s] == 1)
                layerno = 1;
            else
                layerno = 0;
            if (sim_time <= 1e-4)
                initnuc = 1;
            else if (T >= c.Tsol)
                initnuc = 1;
            else
                initnuc = 0;
        }
        if (G(b.gr)[idx] <= 0 && layerno && initnuc)
        {
            double Tunder = c.Tliq - T;
            double m_solute0 = c.ma * T * T + c.mb * T + c.mc;
            Tunder += m_solute0 * ((c.f32 ? ld_cl<true>(b, c, cur, idx) : ld_cl<false>(b, c, cur, idx)) - c.cinit);
            if (Tunder > (double) G(b.site_thr)[s])
                flag = 1;
        }
    }
    int tot;
    int r = block_exscan_flag<NUC_BS / 64>(flag, &tot, s_w);
    const int nwg = (int) (V.off_nuc[d + 1] - V.off_nuc[d]);
    if (nwg == 1)
    {
        // nothing to wait for or to order
        if (flag)
            G(b.events)[r] = s;
        nuc_activate(b, c, mode, tot, V.lean, cur);
        return;
    }
    if (flag)
        st_agent(&b.ev_blk[blk * NUC_BS + r], s);
    if (threadIdx.x == 0)
        st_agent(&b.ev_cnt[blk], tot);
    if (last_workgroup(b.nuc_done, nwg))
        nuc_activate(b, c, mode, -1, V.lean, cur);
}


// activateNewGrains over the ranks of a coupled batch (grain.c:841-916), one
// workgroup: each domain's ordered events (k_nuc_activate mode 1) get ids
// in rank order after the grains existing so far (the displacements of
// grain.c:893-898), orientations from the domain's own stream (its fixed
// entries or its next random draws), in the one grain table the domains
// share.  Every domain advances its timestep; running past MaxTotGrains
// stops all of them, as createGrains' error() stops every rank.
__global__ void __launch_bounds__(NUC_BS)
k_nuc_activate_coupled(View V, int cur)
{
    __shared__ int s_w[NUC_BS / 64];
    const int tid = threadIdx.x;
    // The counters of all domains at once.  Most steps create no grain, and
    // then only the timesteps move on: 4.3 us on average with 8 ranks, where a
    // walk over the domains, each a chain of loads, took 10.2.
    const Counters *c0 = V.dom[0].b.cnt;
    const unsigned long long ts = c0->timestep + 1ull;
    const int base_id = c0->num_grains;
    int stopped = 0, events = 0;
    for (int d = tid; d < V.ndom; d += NUC_BS)
    {
        const Counters *cnt = V.dom[d].b.cnt;
        stopped |= cnt->status != MMCA_OK;
        events |= cnt->n_events;
    }
    if (__syncthreads_or(stopped))
        return;                                   // all domains stop together
    if (!__syncthreads_or(events))
    {
        for (int d = tid; d < V.ndom; d += NUC_BS)
            V.dom[d].b.cnt->timestep = ts;
        return;
    }
    const long long maxg = V.dom[0].c.max_total_grains;
    long long total = base_id;
    for (int d = 0; d < V.ndom; ++d)
        total += V.dom[d].b.cnt->n_events;
    const bool over = total > maxg + 1;
    int next = base_id;
    for (int d = 0; d < V.ndom && !over; ++d)
    {
        const DevBufs b = V.dom[d].b;    // private copy: stores cannot alias it
        const int nev = b.cnt->n_events;
        const int rnd0 = b.cnt->random_used;
        int rused = 0;
        for (int base = 0; base < nev; base += NUC_BS)
        {
            int e = base + tid;
            int isev = e < nev;
            int s = isev ? G(b.events)[e] : 0;
            int fixed = isev ? G(b.site_fixed)[s] : -1;
            int israndom = isev && fixed < 0;
            int rtot;
            int rrank = block_exscan_flag<NUC_BS / 64>(israndom, &rtot, s_w);
            if (isev)
            {
                const long long id = (long long) next + e;
                int idx = G(b.site_idx)[s];
                if (V.lean == 1 || V.lean == 2)
                    put_ce_of_liquid(b, cur, idx);
                G(b.gr)[idx] = (int) id;
                const double *rot;
                int src;
                if (fixed >= 0)
                {
                    rot = b.fixed_rot + 9 * (long long) fixed;
                    src = fixed;
                }
                else
                {
                    int k = rnd0 + rused + rrank;
                    rot = b.rand_rot + 9 * (long long) k;
                    src = -(k + 1);
                }
                for (int q = 0; q < 9; ++q)
                    b.g_rot[9 * id + q] = rot[q];
                G(b.g_cell)[id] = idx;
                G(b.g_step)[id] = ts;
                G(b.g_src)[id] = src;
                G(b.g_dom)[id] = d;
            }
            rused += rtot;
        }
        __syncthreads();
        if (tid == 0)
        {
            b.cnt->random_used = rnd0 + rused;
            b.cnt->new_grains += nev;
        }
        next += nev;
    }
    __syncthreads();
    if (tid == 0)
        for (int d = 0; d < V.ndom; ++d)
        {
            Counters *cnt = V.dom[d].b.cnt;
            if (over)
            {
                // grain.c:868-888, 361-366: with every slot taken nothing is
                // activated; otherwise createGrains stops the run
                if ((long long) base_id != maxg + 1)
                {
                    cnt->status = MMCA_ERR_GRAIN_CAPACITY;
                    cnt->failed_step = ts;
                }
            }
            else
                cnt->num_grains = (int) total;
            cnt->timestep = ts;
        }
}

// Halo exchange between the subblocks of a coupled batch (ExchangeFacesForVar
// / FinishExchangeForVar, calculate.c:227-330): the interior layer of each
// neighbouring subblock is copied into this subblock's halo layer, face by
// face.  Phase 0 (start of the step): cl and fs of buffer `cb` and dc.  Phase
// 1 (after partitioning): gr, fs of buffer `cb`, and the solid bits of the
// halo cells (mask words of the y/z halo rows, x-halo bytes).  Only face
// cells are exchanged: the step reads no edge or corner halo cell.
// grid.y = domain * 6 + face (face 2a: low side of axis a, 2a+1: high side).
__global__ void __launch_bounds__(256)
k_halo_exchange(View V, int phase, int cb)
{
    const int d = blockIdx.y / 6, f = blockIdx.y % 6;
    const int ax = f / 2, hi = f % 2;
    const DevBufs b = V.dom[d].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[d].c;
    if (c.nsub[0] == 0 || G(b.cnt)->status != MMCA_OK)
        return;                                   // a stopped batch keeps its halos
    // Everything indexed by the face's axis is picked with selects, not array
    // subscripts: a runtime subscript would put the descriptor in private
    // (scratch) memory for every thread.
    const int ns0 = c.nsub[0], ns1 = c.nsub[1], ns2 = c.nsub[2];
    int cx = c.off[0] / c.nx, cy = c.off[1] / c.ny, cz = c.off[2] / c.nz;
    const int na = ax == 0 ? c.nx : (ax == 1 ? c.ny : c.nz);     // cells along the axis
    const int nsa = ax == 0 ? ns0 : (ax == 1 ? ns1 : ns2);
    int ca = (ax == 0 ? cx : (ax == 1 ? cy : cz)) + (hi ? 1 : -1);
    if (ca < 0 || ca >= nsa)
    {
        // a face of the global domain: a mold wall, or a wrapped face whose
        // neighbour is the subblock at the other end of the axis
        // (sbID_from_sbcoords, functions.c:272-311); with one subblock along
        // the axis that is the subblock itself, which exchanges nothing
        // (face_util.c:128, 217) and keeps its halo
        const int wall = hi ? (ax == 0 ? c.pad_hi[0] : (ax == 1 ? c.pad_hi[1] : c.pad_hi[2]))
                            : (ax == 0 ? c.pad_lo[0] : (ax == 1 ? c.pad_lo[1] : c.pad_lo[2]));
        if (wall || nsa < 2)
            return;
        ca = (ca + nsa) % nsa;
    }
    if (ax == 0)
        cx = ca;
    else if (ax == 1)
        cy = ca;
    else
        cz = ca;
    const int r = (cz * ns1 + cy) * ns0 + cx;     // MPI Cart rank (z, y, x)
    const DevBufs nb = V.dom[r].b;
    // the two axes along the face, u (faster) and v, with their strides
    const int nu = ax == 0 ? c.ny : c.nx, nv = ax == 2 ? c.ny : c.nz;
    const long long su = ax == 0 ? c.sx : 1, sv = ax == 2 ? c.sx : c.sxy;
    const long long sa = ax == 0 ? 1 : (ax == 1 ? c.sx : c.sxy);
    const long long nface = (long long) nu * nv;
    const long long t = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    const int hal = hi ? na + 1 : 0;              // halo layer of this subblock
    const int src = hi ? 1 : na;                  // the neighbour's interior layer
    if (t < nface)
    {
        const int qu = (int) (t % nu) + 1, qv = (int) (t / nu) + 1;
        const long long base = qu * su + qv * sv;
        const long long dst = base + hal * sa;
        const long long from = base + src * sa;
        if (phase == 0)
        {
            if (c.f32)
                cl32_buf(b, cb)[dst] = cl32_buf(nb, cb)[from];
            else
                cl_buf(b, cb)[dst] = cl_buf(nb, cb)[from];
            fs_buf(b, cb)[dst] = fs_buf(nb, cb)[from];
            for (int e = 0; e < 3; ++e)
                G(b.dc)[3 * dst + e] = G(nb.dc)[3 * from + e];
        }
        else
        {
            const int g = G(nb.gr)[from];
            G(b.gr)[dst] = g;
            fs_buf(b, cb)[dst] = fs_buf(nb, cb)[from];
            if (ax == 0)
            {
                const long long row = (long long) qv * (c.ny + 2) + qu;   // x face: u = y, v = z
                G(b.xhalo)[2 * row + hi] = (unsigned char) (g > 0);
            }
        }
    }
    if (phase == 1 && ax > 0)
    {
        // mask words of the halo rows: y faces, rows (hal, k) for k = 1..nz;
        // z faces, rows (j, hal) for j = 1..ny
        const int nrow = (ax == 1) ? c.nz : c.ny;
        if (t < (long long) nrow * c.w64)
        {
            const int w = (int) (t % c.w64), i = (int) (t / c.w64) + 1;
            const long long rd = (ax == 1) ? ((long long) i * (c.ny + 2) + hal) : ((long long) hal * (c.ny + 2) + i);
            const long long rs = (ax == 1) ? ((long long) i * (c.ny + 2) + src) : ((long long) src * (c.ny + 2) + i);
            G(b.mask)[rd * c.w64 + w] = G(nb.mask)[rs * c.w64 + w];
        }
    }
}

// Partitioning of one cell (fs_change_diffuse, growth.c:221-273).  The
// temperature, temp(), is only evaluated for cells with gr > 0.  *branch
// receives the MMCA_BRANCH_* code of the branch taken.
template <typename TempFn>
__device__ __forceinline__ void
partition_cell(const Consts &c, TempFn temp, double ce_new, double ce_prev, double conc, double lspfs,
               int g_old, double *cl_out, double *fs_out, int *g_out, int *branch)
{
    int g = g_old;
    *branch = MMCA_BRANCH_LIQUID;
    if (g <= 0)
    {
        *cl_out = ce_new;
        *g_out = 0;
        *fs_out = 0;
        return;
    }
    const double Tcell = temp();
    double c_int = c.cinit + c.m_inv * (Tcell - c.Tliq);
    double Tunder = c.Tliq - Tcell;
    Tunder += c.liq_slope * (conc - c.cinit);
    if (Tcell < 1.0 || Tcell > c.Tliq)
    {
        *cl_out = ce_new;
        *g_out = 0;
        *fs_out = 0;
        return;
    }
    if (lspfs == 1.0 && (Tunder >= 0.0))
    {
        *cl_out = ce_new * c.k_inv;
        *fs_out = lspfs;
        *g_out = g;
        *branch = MMCA_BRANCH_SOLID;
        return;
    }
    double dce = ce_new - ce_prev;
    double dcl = (c_int - conc) * c.D_xt * 2 + dce / (1 - c.km * lspfs);
    double dfs = (dcl * (1. - c.km * lspfs) - dce) * c.km_inv / conc;
    double cl = conc + dcl;
    double fs = lspfs + dfs;
    *branch = (1.0 < fs) ? MMCA_BRANCH_FULL : MMCA_BRANCH_GROW;
    fs = ref_min(1.0, fs);
    if (fs < 0.)
    {
        fs = 0.;
        g = 0;
        cl = ce_new;
        *branch = MMCA_BRANCH_REMELT;
    }
    *cl_out = cl;
    *fs_out = fs;
    *g_out = g;
}

// What a solid cell's partitioning does at every temperature in [T - d, T + d]
// (fs_change_diffuse's tests, growth.c:228-241, which read T only through
// comparisons that hold or fail for the whole interval): true if it is the
// same branch, LIQUID or SOLID, so that an approximate T gives the cell's
// result to the bit.  Tunder falls with T, in floating point too.  A growing
// or remelting cell needs the exact T (false), and so does a NaN.
__device__ __forceinline__ bool
branch_decided(const Consts &c, double T, double d, double conc, double lspfs)
{
    if (T - d > c.Tliq || T + d < 1.0)
        return true;
    return lspfs == 1.0 && T - d >= 1.0 && T + d <= c.Tliq &&
           (c.Tliq - (T + d)) + c.liq_slope * (conc - c.cinit) >= 0.0;
}

// Appends the padded indices of the lanes with `flag` to the block's list of
// waiting cells: one atomic per wave.  All lanes call it.
__device__ __forceinline__ void
und_append(const DevBufs &b, bool flag, int idx)
{
    const unsigned long long m = __ballot(flag);
    if (!m)
        return;
    const int lane = threadIdx.x & 63;
    int base = 0;
    if (lane == (int) __ffsll(m) - 1)
        base = atomicAdd(b.und_n, __popcll(m));
    base = __shfl(base, (int) __ffsll(m) - 1, 64);
    if (flag)
        G(b.und)[base + __popcll(m & ((1ull << lane) - 1ull))] = idx;
}

// A cell whose partitioning waits for the exact temperature (k_beam_finish)
// keeps what that needs in its output slots: FP64 storage, the ce before
// diffusion in fs (the new one is in ce); FP32 storage, the new ce unrounded in
// fs and the stored ce before diffusion in cl.
template <bool F32>
__device__ __forceinline__ void
defer_cell(const DevBufs &b, const Consts &c, int nxt, long long idx, double ce_new, double ce_prev)
{
    fs_buf(b, nxt)[idx] = F32 ? ce_new : ce_prev;
    if (F32)
        cl32_buf(b, nxt)[idx] = (float) (ce_prev - c.cinit);
}

// growth.c:163-165: error() ends every rank.  In a coupled batch the status
// goes to every domain of the view, so that each rank's later kernels (and
// the halo exchange) stop at the same point; the ranks share one timestep.
__device__ __forceinline__ void
flag_negative_ce(const View &V, const Consts &c, Counters *cnt)
{
    if (c.nsub[0] == 0)
    {
        if (atomicCAS(&cnt->status, MMCA_OK, MMCA_ERR_NEGATIVE_CE) == MMCA_OK)
            cnt->failed_step = cnt->timestep;
        return;
    }
    for (int d = 0; d < V.ndom; ++d)
    {
        Counters *o = V.dom[d].b.cnt;
        if (atomicCAS(&o->status, MMCA_OK, MMCA_ERR_NEGATIVE_CE) == MMCA_OK)
            o->failed_step = o->timestep;
    }
}

// Cell-parallel kernel.  DIFF && FSC: fused step reading buffers `cur`,
// writing `nxt`.  DIFF only: ce += nbsum (the caller copies ce to oce
// beforehand).  FSC only: in place on `cur` with ce_old = oce.  FSC writes
// the solid mask (gr > 0).  REC also writes each cell's partitioning branch
// into the domain's branch record.
constexpr int SOL_BX = 64;
constexpr int SOL_BY = 4;
constexpr int SOL_BZ = 8;    // planes per workgroup: spreads the per-workgroup set-up over 8 x 256 cells

template <bool DIFF, bool FSC, bool AM, bool F32, bool REC = false>
__global__ void __launch_bounds__(SOL_BX *SOL_BY)
k_solute(View V, int cur, int nxt)
{
    // the fused step of a beam block works from the approximate temperature
    // and leaves the cells that need the exact one to k_beam_finish; the single
    // operators and the recorded step evaluate the quadrature in place
    constexpr bool DEFER = AM && DIFF && FSC && !REC;
    __shared__ double s_red[SOL_BX * SOL_BY / 64];
    __shared__ int s_stop;
    const int dm = find_dom(V.off_cell, V.ndom, blockIdx.x);
    const DevBufs b = V.dom[dm].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[dm].c;
    // workgroup -> 64 x 4 tile and SOL_BZ planes (32-bit index arithmetic:
    // a domain has fewer than 2^31 cells)
    const unsigned blk = (unsigned) (blockIdx.x - V.off_cell[dm]);
    const unsigned gbx = (unsigned) (c.nx + SOL_BX - 1) / SOL_BX, gby = (unsigned) (c.ny + SOL_BY - 1) / SOL_BY;
    const unsigned rest = blk / gbx;
    const int bx = (int) (blk - rest * gbx);
    const int by = (int) (rest % gby);
    const int bz = (int) (rest / gby);
    Counters *cnt = b.cnt;
    // this kernel itself may raise the status: read it once per workgroup so
    // that every wave takes the same branch before the barrier of block_sum
    if (threadIdx.x == 0 && threadIdx.y == 0)
        s_stop = (G(b.cnt)->status != MMCA_OK);
    __syncthreads();
    if (s_stop)
        return;
    const int x = bx * SOL_BX + threadIdx.x + 1;   // interior x
    const int j = by * SOL_BY + threadIdx.y + 1;
    const int k0 = bz * SOL_BZ + 1;
    const int k1 = min(c.nz, k0 + SOL_BZ - 1);
    const bool rowok = (j <= c.ny);
    const bool active = rowok && (x <= c.nx);
    const double sim_time = G(b.cnt)->timestep * c.dt;
    double lost = 0.0;                                   // FP32 storage rounding of ce
    for (int k = k0; k <= k1; ++k)
    {
        int g_new = 0;
        int br_rec = 0;
        bool wait = false;
        if (active)
        {
            const long long idx = k * c.sxy + (long long) j * c.sx + x;
            const MMCA_GLOBAL double *fsc = fs_buf(b, cur);
            const double ce_old = ld_ce<F32>(b, c, idx);
            const double conc = ld_cl<F32>(b, c, cur, idx);
            const double lspfs = fsc[idx];
            double ce_new = ce_old;
            if (DIFF)
            {
                const long long nb[6] = { idx + 1, idx - 1, idx + c.sx, idx - c.sx, idx + c.sxy, idx - c.sxy };
                // mold of a neighbour: a padded face of the box (interior cells are never mold)
                const int mo[6] = { (x == c.nx) ? c.pad_hi[0] : 0, (x == 1) ? c.pad_lo[0] : 0,
                                    (j == c.ny) ? c.pad_hi[1] : 0, (j == 1) ? c.pad_lo[1] : 0,
                                    (k == c.nz) ? c.pad_hi[2] : 0, (k == 1) ? c.pad_lo[2] : 0 };
                double cln[6], fsn[6];
#pragma unroll
                for (int n = 0; n < 6; ++n)
                {
                    cln[n] = ld_cl<F32>(b, c, cur, nb[n]);
                    fsn[n] = fsc[nb[n]];
                }
                ce_new = diffuse_cell(c, ce_old, conc, lspfs, cln, fsn, mo);
                if (c.check_neg && ce_new < 0)
                    flag_negative_ce(V, c, cnt);
                lost += st_ce<F32>(b, c, idx, ce_new);
            }
            if (FSC)
            {
                const double ce_prev = DIFF ? ce_old : G(b.oce)[idx];
                const int g_old = G(b.gr)[idx];
                if constexpr (DEFER)
                    if (g_old > 0)
                    {
                        const double T = (double) G(b.temp32)[idx];
                        wait = !branch_decided(c, T, beam_margin(c, T), conc, lspfs);
                    }
                double cl_out, fs_out;
                int g = g_old, branch;
                if (wait)
                    defer_cell<F32>(b, c, nxt, idx, ce_new, ce_prev);
                else
                {
                    partition_cell(
                        c,
                        [&]() {
                            if constexpr (DEFER)
                                return (double) G(b.temp32)[idx];
                            else
                                return temp_model<AM>(c, sim_time, x, j, k);
                        },
                        ce_new, ce_prev, conc, lspfs, g_old, &cl_out, &fs_out, &g, &branch);
                    br_rec = branch;
                    st_cl<F32>(b, c, nxt, idx, cl_out);
                    st_stream(fs_buf(b, nxt), idx, fs_out);
                    if (g != g_old)
                        G(b.gr)[idx] = g;
                    keep_stale_d(c, b, idx, g_old, g, lspfs);
                }
                g_new = g;
            }
        }
        if (FSC)
        {
            if (DEFER)
                und_append(b, wait, (int) (k * c.sxy + (long long) j * c.sx + x));
            const unsigned long long bits = __ballot(active && g_new > 0 && !wait);
            if (threadIdx.x == 0 && rowok)
                G(b.mask)[((long long) k * (c.ny + 2) + j) * c.w64 + bx] = bits;
        }
        if (REC)
        {
            // branch record of this step, three bit planes per 64-cell segment
            // (bounds: set by the host, checked here too)
            const unsigned long long p0 = __ballot(active && (br_rec & 1));
            const unsigned long long p1 = __ballot(active && (br_rec & 2));
            const unsigned long long p2 = __ballot(active && (br_rec & 4));
            const long long rs = (long long) (G(b.cnt)->timestep - b.rec_t0) - 1;
            if (threadIdx.x == 0 && rowok && rs >= 0 && rs < b.rec_steps)
            {
                MMCA_GLOBAL unsigned long long *w = (MMCA_GLOBAL unsigned long long *) b.rec +
                                                    rs * rec_words(c) + rec_word(c, bx, j, k);
                w[0] = p0;
                w[1] = p1;
                w[2] = p2;
            }
        }
    }
    if (F32)
    {
        const double tot = block_sum<SOL_BX * SOL_BY>(lost, s_red);
        if (threadIdx.x == 0 && threadIdx.y == 0 && tot != 0.0)
            ledger_add(b, blk, tot);
    }
}

// Tile of this workgroup.  The hardware places workgroup w on XCD w % 8; runs
// of V.xcd_run consecutive tiles (x fastest, then y, then z, then domain) go
// to one XCD, run q to XCD q % 8, so that tiles sharing halo rows share an L2
// while all XCDs work on the same planes.  Runs of 8 were the fastest on
// blocks of every size (256 x 256 x 512 FP64: 403 us, against 425 us with
// tiles dealt one by one and 440 us with one contiguous eighth per XCD).
// At or past V.tot_zm: no tile (the grid is rounded up to whole rounds).
__device__ __forceinline__ long long
xcd_tile(const View &V)
{
    const unsigned m = (unsigned) V.xcd_run, i = blockIdx.x / 8;
    return ((long long) (i / m) * 8 + blockIdx.x % 8) * m + i % m;
}

// Raw storage of ce and cl (FP64 values, or FP32 deviations from c0), kept
// unconverted while a load is in flight, so that a prefetched value is only
// waited for where it is used.
template <bool F32> struct Store { using T = double; };
template <> struct Store<true> { using T = float; };

template <bool F32>
__device__ __forceinline__ typename Store<F32>::T
raw_ce(const DevBufs &b, long long i)
{
    if constexpr (F32)
        return G(b.ce32)[i];
    else
        return G(b.ce)[i];
}

template <bool F32>
__device__ __forceinline__ typename Store<F32>::T
raw_cl(const DevBufs &b, int buf, long long i)
{
    if constexpr (F32)
        return cl32_buf(b, buf)[i];
    else
        return cl_buf(b, buf)[i];
}

template <bool F32>
__device__ __forceinline__ double
from_raw(const Consts &c, typename Store<F32>::T r)
{
    if constexpr (F32)
        return c.cinit + (double) r;
    else
        return r;
}

// Lane shifts of a double by one over the whole wave (DPP wave_shl / wave_shr,
// which CDNA has): lane l gets lane l + 1 (up) or l - 1 (down); the last
// (first) lane, which has no such lane, gets `edge`.
__device__ __forceinline__ double
from_lane_up(double v, double edge)
{
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x130, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double
from_lane_down(double v, double edge)
{
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x138, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// What a wave loads of one plane: cl and fs of rows -1 .. RY of its tile, ce
// and gr of its own rows, the x neighbours across the tile's edges (lane 63:
// x + 1, the others: x - 1 of lane 0) and, in beam blocks (TF), the
// approximate temperature.
template <int RY, bool F32, bool TF>
struct RwPlane {
    using S = typename Store<F32>::T;
    S cl[RY + 2], ce[RY], ecl[RY];
    double fs[RY + 2], efs[RY];
    float t[TF ? RY : 1];
    int g[RY];
    unsigned long long w;            // act words of buffer nxt: lane r has row r
};

__device__ __forceinline__ unsigned long long
lane_word(unsigned long long v, int lane)
{
    return (unsigned long long) (unsigned) __builtin_amdgcn_readlane((int) v, lane) |
           (unsigned long long) (unsigned) __builtin_amdgcn_readlane((int) (v >> 32), lane) << 32;
}

// base + byte offset: a scalar base and a 32-bit lane offset, the addressing
// form of a global load or store that needs no 64-bit lane arithmetic
template <typename T>
__device__ __forceinline__ MMCA_GLOBAL T *
at_byte(MMCA_GLOBAL T *base, unsigned off)
{
    return (MMCA_GLOBAL T *) ((MMCA_GLOBAL char *) base + off);
}

// Fused diffusion + partitioning, rows in registers.  A wave owns 64 cells x
// RY rows and walks `zm_planes` planes upward; the four waves of a workgroup
// take neighbouring rows (4 RY of them) and share nothing but the caches: no
// barrier in the walk.
//
// The solute that crosses a face is the same number, with the other sign, for
// the two cells on its sides: r (growth.c:95-99) is symmetric in them and
// IEEE subtraction is antisymmetric.  So each face is computed once: the x
// face towards x + 1 in each lane and handed to the next lane, the y faces
// between the rows of a wave in registers, the z face towards k + 1 kept for
// the next plane.  A cell then costs 3 face terms instead of 6, and the sums
// run in the reference's order, so results keep its bits.
//
// The loads of plane k + 1 are issued before plane k is worked on, in two
// register sets used in turn.  A cell is finished one plane late: its z terms
// come last in the sum, so its x and y terms wait in a register until the
// plane above has landed.
//
// Where the steps of a call are lean (V.lean), what stays as it is isn't
// written: in a row of 64 liquid cells fs and the mask, zero in both buffers,
// and ce, which is cl again after the partitioning (cl = ce, fs = 0).  Such a
// row writes 8 bytes a cell instead of 24.  What decides it are gr, read
// anyway, and one word a row, the cells that were solid when buffer nxt was
// last written (act).  Leaving out the loads as well (of rows with no solid
// cell in sight, from act words two planes ahead) made the kernel issue-bound
// by the tests for it: 323 us for 256 x 256 x 512, and 55 instead of 36 for 150
// x 140 x 165.
//
// Bound by memory: with the arithmetic taken out (a timing copy) the walk over
// 256 x 256 x 512 takes the same time.  Two rows per wave and 16 planes read
// the fewest halo rows that still leave two waves per SIMD in registers.
// FP64, 256 x 256 x 512: 403 us (447 us with planes staged in LDS, 4.2 TB/s
// of 56 B per cell), 336 us lean with 2/3 of the rows liquid; 128 x 128 x 256:
// 48 us (142), 45 lean; 40 x 36 x 44: 8.3 us (93).  FP32-deviation storage,
// 256 x 256 x 512: 293 us (337).
constexpr int RW_LATE = 2048;                    // waiting cells of a tile buffered in LDS

template <int RY, bool F32, bool TF, bool LEAN>
__global__ void __launch_bounds__(512, RY == 1 ? 4 : 2)
k_solute_rw(View V, int cur, int nxt)
{
    using S = typename Store<F32>::T;
    constexpr unsigned E = sizeof(S);
    __shared__ double s_red[8];
    __shared__ int s_stop;
    // the non-beam temperatures depend on z only (on y in 2-D runs): one value
    // per plane of the tile (per row); dynamic LDS
    extern __shared__ double s_T[];
    // beam blocks: the tile's waiting cells (s_late: their number, and where
    // the buffer ended), appended to the block's list with one atomic; cells
    // past the buffer go to the list directly
    __shared__ int s_cell[TF ? RW_LATE : 1], s_late[TF ? 3 : 1];
    const long long gtile = xcd_tile(V);
    if (gtile >= V.tot_zm)
        return;                                   // uniform over the workgroup
    const int dm = find_dom(V.off_zm, V.ndom, gtile);
    const unsigned tile = (unsigned) (gtile - V.off_zm[dm]);
    const DomainDesc *dd = &V.dom[dm];
    const Consts c = dd->c;           // private copies: stores cannot alias them
    MMCA_GLOBAL S *clc, *cln, *ceb;
    if constexpr (F32)
    {
        clc = cl32_buf(dd->b, cur);
        cln = cl32_buf(dd->b, nxt);
        ceb = G(dd->b.ce32);
    }
    else
    {
        clc = cl_buf(dd->b, cur);
        cln = cl_buf(dd->b, nxt);
        ceb = G(dd->b.ce);
    }
    const MMCA_GLOBAL double *fsc = fs_buf(dd->b, cur);
    MMCA_GLOBAL double *fsn = fs_buf(dd->b, nxt);
    MMCA_GLOBAL int *grb = G(dd->b.gr);
    const MMCA_GLOBAL float *tb = G(dd->b.temp32);
    MMCA_GLOBAL unsigned long long *mask = G(dd->b.mask);
    const int lean = LEAN ? V.lean : 0;
    MMCA_GLOBAL unsigned long long *actn = G(dd->b.act[nxt]);
    const int lane = threadIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int rows = blockDim.y * RY;
    const unsigned ntx = (unsigned) (c.nx + 63) / 64, nty = (unsigned) (c.ny + rows - 1) / rows;
    const unsigned trow = tile / ntx;
    const int bx = (int) (tile - trow * ntx);
    const int bz = (int) (trow / nty);
    const int by = (int) (trow - bz * nty);
    const int x = bx * 64 + lane + 1;
    const int j0 = by * rows + wv * RY + 1;
    const int k0 = bz * c.zm_planes + 1;
    const int k1 = min(c.nz, k0 + c.zm_planes - 1);
    // this kernel itself may raise the status: read it once per workgroup so
    // that every wave takes the same branch before the barrier of block_sum
    if (lane == 0 && threadIdx.y == 0)
    {
        s_stop = (G(dd->b.cnt)->status != MMCA_OK);
        if constexpr (TF)
            s_late[0] = 0, s_late[1] = RW_LATE;
    }
    const bool two_d = (c.gdimz == 1);
    if constexpr (!TF)
    {
        const double sim_time = G(dd->b.cnt)->timestep * c.dt;
        const int nT = two_d ? rows : k1 - k0 + 1;
        for (int e = wv * 64 + lane; e < nT; e += 64 * blockDim.y)
            s_T[e] = temp_model<false>(c, sim_time, 1, two_d ? by * rows + 1 + e : 1, two_d ? 1 : k0 + e);
    }
    __syncthreads();
    if (s_stop)
        return;
    double lost = 0.0;
    bool neg = false;
    if (j0 <= c.ny)
    {
        // every lane issues every load, at an address clamped into the padded box
        const unsigned xc = (unsigned) min(x, c.nx + 1);
        const unsigned xe = lane == 63 ? (unsigned) min(x + 1, c.nx + 1) : (unsigned) (bx * 64);
        const double wxr = (x == c.nx) ? (double) (1 - c.pad_hi[0]) : 1.0;
        const double wxl = (x == 1) ? (double) (1 - c.pad_lo[0]) : 1.0;
        // rows relative to row j0 - 1: the padding row is the last one loaded
        const int rmax = c.ny + 2 - j0;
        const long long row0 = (long long) (j0 - 1) * c.sx;
        const MMCA_GLOBAL unsigned long long *wsrc =
            actn + (long long) (j0 - 1 + min(lane < RY ? lane + 1 : 1, rmax)) * c.w64 + bx;
        const long long wplane = (long long) (c.ny + 2) * c.w64;
        auto load = [&](RwPlane<RY, F32, TF> &p, int k) {
            const long long at = k * c.sxy + row0;
            if constexpr (LEAN)
                p.w = wsrc[k * wplane];
#pragma unroll
            for (int r = 0; r < RY + 2; ++r)
            {
                const unsigned o = (unsigned) (min(r, rmax) * c.sx) + xc;
                p.cl[r] = *at_byte(clc + at, o * E);
                p.fs[r] = *at_byte(fsc + at, o * 8);
            }
#pragma unroll
            for (int r = 0; r < RY; ++r)
            {
                const unsigned rb = (unsigned) (min(r + 1, rmax) * c.sx);
                p.ecl[r] = *at_byte(clc + at, (rb + xe) * E);
                p.efs[r] = *at_byte(fsc + at, (rb + xe) * 8);
                p.ce[r] = *at_byte(ceb + at, (rb + xc) * E);
                p.g[r] = *at_byte(grb + at, (rb + xc) * 4);
                if constexpr (TF)
                    p.t[r] = *at_byte(tb + at, (rb + xc) * 4);
            }
        };
        // solute through the face from cell a to cell b (growth.c:95-99)
        auto face = [&](double cla, double fsa, double clb, double fsb, double w) -> double {
            const double f = 0.5 * (fsa + fsb);
            const double r = (c.rs * f + c.rl * (1 - f)) * w;
            return r * (clb - cla);
        };
        // the plane below, not finished yet: x and y terms, own values, and
        // the z face below it
        double psum[RY], pcl[RY], pfs[RY], pce[RY], pfz[RY];
        float pt[TF ? RY : 1];
        int pg[RY];
        unsigned long long pw = 0;
        RwPlane<RY, F32, TF> P0, P1;
        load(P0, k0);
        {
            const long long at = (k0 - 1) * c.sxy + row0;
#pragma unroll
            for (int r = 0; r < RY; ++r)
            {
                const unsigned o = (unsigned) (min(r + 1, rmax) * c.sx) + xc;
                pcl[r] = from_raw<F32>(c, *at_byte(clc + at, o * E));
                pfs[r] = *at_byte(fsc + at, o * 8);
                psum[r] = pce[r] = pfz[r] = 0.0;
                pg[r] = 0;
            }
        }
        // plane k in A (landed); plane k + 1 goes to N
        auto plane = [&](int k, RwPlane<RY, F32, TF> &A, RwPlane<RY, F32, TF> &N) {
            load(N, min(k + 1, k1 + 1));
            const double wz = (k == 1) ? (double) (1 - c.pad_lo[2])
                                       : (k == c.nz + 1) ? (double) (1 - c.pad_hi[2]) : 1.0;
            double cl = from_raw<F32>(c, A.cl[1]);
            double fy = face(from_raw<F32>(c, A.cl[0]), A.fs[0], cl, A.fs[1],
                             (j0 == 1) ? (double) (1 - c.pad_lo[1]) : 1.0);
#pragma unroll
            for (int r = 0; r < RY; ++r)
            {
                const int j = j0 + r;
                const double fs = A.fs[r + 1];
                const double fz = face(pcl[r], pfs[r], cl, fs, wz);
                if (k > k0)
                {
                    // finish plane k - 1
                    double sum = psum[r];
                    sum += fz;
                    sum -= pfz[r];
                    const double ce_new = pce[r] + sum;
                    int g_new = 0;
                    bool wait = false;
                    const unsigned long long solid = __ballot(pg[r] > 0 && x <= c.nx);
                    const bool put_fs = !LEAN || (solid | lane_word(pw, r)) != 0, put_ce = !LEAN || lean != 1 || solid != 0;
                    if (j <= c.ny && x <= c.nx)
                    {
                        const long long at = (k - 1) * c.sxy + row0;
                        const unsigned o = (unsigned) ((r + 1) * c.sx) + (unsigned) x;
                        neg |= (ce_new < 0);
                        if constexpr (F32)
                        {
                            const double dev = ce_new - c.cinit;
                            const float f = (float) dev;
                            lost += dev - (double) f;
                            if (put_ce)
                                *at_byte(ceb + at, o * E) = f;
                        }
                        else if (put_ce)
                            *at_byte(ceb + at, o * E) = ce_new;
                        if constexpr (TF)
                            wait = pg[r] > 0 && !branch_decided(c, (double) pt[r], beam_margin(c, (double) pt[r]),
                                                                pcl[r], pfs[r]);
                        if (wait)
                        {
                            // as defer_cell
                            *at_byte(fsn + at, o * 8) = F32 ? ce_new : pce[r];
                            if constexpr (F32)
                                *at_byte(cln + at, o * E) = (float) (pce[r] - c.cinit);
                        }
                        else
                        {
                            double cl_out, fs_out;
                            int branch;
                            partition_cell(
                                c,
                                [&]() {
                                    if constexpr (TF)
                                        return (double) pt[r];
                                    else
                                        return s_T[two_d ? wv * RY + r : k - 1 - k0];
                                },
                                ce_new, pce[r], pcl[r], pfs[r], pg[r], &cl_out, &fs_out, &g_new, &branch);
                            if constexpr (F32)
                                *at_byte(cln + at, o * E) = (float) (cl_out - c.cinit);
                            else
                                *at_byte(cln + at, o * E) = cl_out;
                            if (put_fs)
                                *at_byte(fsn + at, o * 8) = fs_out;
                            if (g_new != pg[r])
                            {
                                *at_byte(grb + at, o * 4) = g_new;
                                if (c.track_d)
                                    keep_stale_d(c, dd->b, at + o, pg[r], g_new, pfs[r]);
                            }
                        }
                    }
                    if (put_fs)
                    {
                        const unsigned long long bits = __ballot(g_new > 0);
                        if (lane == 0 && j <= c.ny)
                        {
                            const long long w = ((long long) (k - 1) * (c.ny + 2) + j) * c.w64 + bx;
                            mask[w] = bits;
                            if constexpr (LEAN)
                                actn[w] = solid;
                        }
                    }
                    if constexpr (TF)
                    {
                        const unsigned long long late = __ballot(wait);
                        if (late)
                        {
                            const int cell = (int) ((k - 1) * c.sxy + (long long) j * c.sx + x);
                            int base = 0;
                            if (lane == 0)
                            {
                                base = atomicAdd(&s_late[0], __popcll(late));
                                if (base + __popcll(late) > RW_LATE)
                                    atomicMin(&s_late[1], base);
                            }
                            base = __builtin_amdgcn_readfirstlane(base);
                            if (base + __popcll(late) > RW_LATE)
                                und_append(dd->b, wait, cell);
                            else if (wait)
                                s_cell[base + __popcll(late & ((1ull << lane) - 1ull))] = cell;
                        }
                    }
                }
                // x and y terms of plane k
                const double ecl = from_raw<F32>(c, A.ecl[r]);
                const double fx = face(cl, fs, from_lane_up(cl, ecl), from_lane_up(fs, A.efs[r]), wxr);
                const double fe = face(ecl, A.efs[r], cl, fs, wxl);  // lane 0: from x - 1
                const double clu = from_raw<F32>(c, A.cl[r + 2]);
                const double fyu = face(cl, fs, clu, A.fs[r + 2], (j == c.ny) ? (double) (1 - c.pad_hi[1]) : 1.0);
                double sum = 0.0 + fx;
                sum -= from_lane_down(fx, fe);
                sum += fyu;
                sum -= fy;
                psum[r] = sum;
                pcl[r] = cl;
                pfs[r] = fs;
                pce[r] = (!LEAN || lean == 3 || A.g[r] > 0) ? from_raw<F32>(c, A.ce[r]) : cl;
                pg[r] = A.g[r];
                pfz[r] = fz;
                if constexpr (TF)
                    pt[r] = A.t[r];
                fy = fyu;
                cl = clu;
            }
            if constexpr (LEAN)
                pw = A.w;
        };
        // the loop starts with nothing in flight, so that its waits are the
        // steady-state ones
        __builtin_amdgcn_s_waitcnt(0);
        for (int k = k0;;)
        {
            plane(k, P0, P1);
            if (++k > k1 + 1)
                break;
            plane(k, P1, P0);
            if (++k > k1 + 1)
                break;
        }
    }
    if (c.check_neg && neg)
        flag_negative_ce(V, c, dd->b.cnt);
    if (LEAN && lane == 0 && threadIdx.y == 0)
        G(dd->b.stamp)[tile] = (unsigned) G(dd->b.cnt)->timestep;
    if constexpr (TF)
    {
        __syncthreads();
        const int n = min(s_late[0], s_late[1]);
        if (n > 0)                                // uniform over the workgroup
        {
            if (lane == 0 && threadIdx.y == 0)
                s_late[2] = atomicAdd(dd->b.und_n, n);
            __syncthreads();
            for (int e = wv * 64 + lane; e < n; e += 64 * blockDim.y)
                G(dd->b.und)[s_late[2] + e] = s_cell[e];
        }
    }
    if (F32)
    {
        const double tot = block_sum(lost, s_red, 64 * blockDim.y);
        if (lane == 0 && threadIdx.y == 0 && tot != 0.0)
            ledger_add(dd->b, tile, tot);
    }
}

// upper bound of a block's solute tiles, of whatever shape
__host__ __device__ __forceinline__ long long
tile_slots_d(const Consts &c)
{
    return (long long) ((c.nx + 63) / 64) * ((c.ny + 3) / 4) * c.nz;
}

// Start of a call of lean steps: nothing is known of any cell.
__global__ void __launch_bounds__(256)
k_wake_all(View V)
{
    const DevBufs b = V.dom[blockIdx.y].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[blockIdx.y].c;
    const long long n = (long long) (c.nz + 2) * (c.ny + 2) * c.w64;
    const long long nt = tile_slots_d(c);
    for (long long i = (long long) blockIdx.x * 256 + threadIdx.x; i < max(n, nt); i += 256ll * gridDim.x)
    {
        if (i < n)
            G(b.act[0])[i] = G(b.act[1])[i] = ~0ull;
        if (i < nt)
            G(b.stamp)[i] = ~0u;
    }
}

// After lean steps that stopped on an error at the timestep `failed` (not the
// first of the call): ce of the liquid cells, which need not have been
// written.  The tiles that finished that step left it as cl in the buffer
// `cur`, the others in the one before.
__global__ void __launch_bounds__(256)
k_settle(const DomainDesc *dom, int cur, unsigned failed)
{
    const DevBufs b = dom->b;         // private copies: stores cannot alias them
    const Consts c = dom->c;          // the tiles of the steps, whatever was set on the context since
    const unsigned ntx = (unsigned) (c.nx + 63) / 64, nty = (unsigned) (c.ny + c.zm_by - 1) / c.zm_by;
    const long long N = (long long) c.nx * c.ny * c.nz;
    for (long long i = (long long) blockIdx.x * 256 + threadIdx.x; i < N; i += 256ll * gridDim.x)
    {
        const int x = (int) (i % c.nx) + 1, j = (int) (i / c.nx % c.ny) + 1, k = (int) (i / c.nx / c.ny) + 1;
        const unsigned tile = ((unsigned) (k - 1) / c.zm_planes * nty + (unsigned) (j - 1) / c.zm_by) * ntx +
                              (unsigned) (x - 1) / 64;
        const int buf = G(b.stamp)[tile] == failed ? cur : cur ^ 1;
        const long long idx = k * c.sxy + (long long) j * c.sx + x;
        if (G(b.gr)[idx] <= 0)
            put_ce_of_liquid(b, buf, idx);
    }
}

// Solid mask from gr (used when the list is built outside the fused step).
// Mask layout: per padded row (j,k), w64 words; bit b of word w is interior
// x = 64 w + b + 1.
__global__ void
k_mask_from_gr(DevBufs b, Consts c)
{
    const int x = blockIdx.x * 64 + threadIdx.x + 1;
    const int j = blockIdx.y;
    const int k = blockIdx.z;
    bool solid = false;
    if (x <= c.nx)
        solid = G(b.gr)[k * c.sxy + (long long) j * c.sx + x] > 0;
    unsigned long long bits = __ballot(solid);
    if (threadIdx.x == 0)
        G(b.mask)[((long long) k * (c.ny + 2) + j) * c.w64 + blockIdx.x] = bits;
}

// ---------------------------------------------------------------------------
// Interface list: interior cells with gr <= 0 and a neighbour with gr > 0
// (growth.c:496-513), in raster order.  One thread per 64-bit mask word.
constexpr int LIST_BS = 256;

__host__ __device__ __forceinline__ long long
list_words_d(const Consts &c)
{
    return (long long) c.nz * c.ny * c.w64;
}

// workgroups of the list writer: list_w mask words each
__host__ __device__ __forceinline__ int
list_blocks_d(const Consts &c)
{
    return (int) ((list_words_d(c) + c.list_w - 1) / c.list_w);
}

__device__ __forceinline__ unsigned long long
mask_word(const DevBufs &b, const Consts &c, int k, int j, int w)
{
    return G(b.mask)[((long long) k * (c.ny + 2) + j) * c.w64 + w];
}

// mask word wi (< nz * ny * w64 < 2^31) -> padded plane k, row j, word w;
// 32-bit arithmetic (64-bit division is a long instruction sequence)
__device__ __forceinline__ void
word_pos(const Consts &c, long long wi, int *k, int *j, int *w)
{
    const unsigned u = (unsigned) wi, w64 = (unsigned) c.w64, ny = (unsigned) c.ny;
    const unsigned nrow = u / w64;
    *w = (int) (u - nrow * w64);
    const unsigned kk = nrow / ny;
    *j = (int) (nrow - kk * ny) + 1;
    *k = (int) kk + 1;
}

// Solid bits of the x-1 (left) and x+1 (right) neighbours of the cells of
// mask word w; the halo cells x = 0 and x = nx+1 come from the row's x-halo
// bytes (solid only where another subblock of a coupled batch lies there).
__device__ __forceinline__ void
x_neighbour_bits(const DevBufs &b, const Consts &c, int k, int j, int w, unsigned long long own,
                 unsigned long long *left, unsigned long long *right)
{
    *left = own << 1;
    *right = own >> 1;
    const long long row = (long long) k * (c.ny + 2) + j;
    if (w > 0)
        *left |= mask_word(b, c, k, j, w - 1) >> 63;
    else
        *left |= (unsigned long long) (G(b.xhalo)[2 * row] != 0);
    if (w + 1 < c.w64)
        *right |= mask_word(b, c, k, j, w + 1) << 63;
    else
        *right |= (unsigned long long) (G(b.xhalo)[2 * row + 1] != 0) << (c.nx - 1 - 64 * w);
}

__device__ __forceinline__ unsigned long long
member_bits(const DevBufs &b, const Consts &c, long long wi, int *pk, int *pj, int *pw)
{
    int k, j, w;
    word_pos(c, wi, &k, &j, &w);
    *pk = k;
    *pj = j;
    *pw = w;
    unsigned long long own = mask_word(b, c, k, j, w);
    unsigned long long left, right;
    x_neighbour_bits(b, c, k, j, w, own, &left, &right);
    unsigned long long yz = mask_word(b, c, k, j - 1, w) | mask_word(b, c, k, j + 1, w) |
                            mask_word(b, c, k - 1, j, w) | mask_word(b, c, k + 1, j, w);
    // bit b of word w is interior x = 64 w + b + 1 <= nx
    const int hi = c.nx - w * 64;
    const unsigned long long inter = (hi >= 64) ? ~0ull : ((1ull << hi) - 1ull);
    return ~own & (left | right | yz) & inter;
}

// Offsets of the list workgroups from their counts, by one workgroup of BS
// threads, and, when decide_realloc is set, the dc_tmp growth rule of
// growth.c:644-660.  AGENT: the counts come from workgroups of this launch.
template <int BS, bool AGENT>
__device__ __forceinline__ void
list_scan(const DevBufs &b, const Consts &c, int decide_realloc)
{
    __shared__ int s_w[BS / 64];
    const int tid = threadIdx.x, nblk = list_blocks_d(c);
    int tot = 0;
    for (int base = 0; base < nblk; base += BS)
    {
        const int i = base + tid;
        int v = 0, n;
        if (i < nblk)
            v = AGENT ? ld_agent(&b.blk_count[i]) : G(b.blk_count)[i];
        const int ex = block_exscan_int<BS / 64>(v, &n, s_w);
        if (i < nblk)
            G(b.blk_count)[i] = tot + ex;
        tot += n;
    }
    if (tid == 0)
    {
        Counters *cnt = b.cnt;
        cnt->gindex = tot;
        if (decide_realloc)
        {
            if (tot > cnt->dc_tmp_size)
            {
                cnt->realloc_old = cnt->dc_tmp_size;
                cnt->dc_tmp_size = tot + 100;
            }
            else
                cnt->realloc_old = -1;
        }
    }
}

// Counts the members of every list workgroup (c.list_w words of k_list_write).
// FUSED: the workgroup of a domain that finishes last also scans the counts,
// which takes k_list_scan's launch (4.7 us) out of the step of small blocks.
template <bool FUSED>
__global__ void __launch_bounds__(LIST_BS)
k_list_count(View V, int decide_realloc)
{
    __shared__ int s_w[LIST_BS / 64];
    const int dm = find_dom(V.off_count, V.ndom, blockIdx.x);
    const long long blk = blockIdx.x - V.off_count[dm];
    const DevBufs b = V.dom[dm].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[dm].c;
    const long long nwords = list_words_d(c);
    if (G(b.cnt)->status != MMCA_OK)
        return;
    const int tid = threadIdx.x;
    const long long wi = blk * LIST_BS + tid;
    int v = 0;
    if (wi < nwords)
    {
        int k, j, w;
        v = __popcll(member_bits(b, c, wi, &k, &j, &w));
    }
    if (c.list_w == 64)
    {
        // one count per wave
        for (int d = 32; d > 0; d >>= 1)
            v += __shfl_xor(v, d, 64);
        const long long q = blk * (LIST_BS / 64) + (tid >> 6);
        if ((tid & 63) == 0 && q < list_blocks_d(c))
        {
            if (FUSED)
                st_agent(&b.blk_count[q], v);
            else
                G(b.blk_count)[q] = v;
        }
    }
    else
    {
        int tot;
        block_exscan_int<LIST_BS / 64>(v, &tot, s_w);
        if (tid == 0)
        {
            if (FUSED)
                st_agent(&b.blk_count[blk], tot);
            else
                G(b.blk_count)[blk] = tot;
        }
    }
    if constexpr (FUSED)
        if (last_workgroup(b.list_done, (int) (V.off_count[dm + 1] - V.off_count[dm])))
            list_scan<LIST_BS, true>(b, c, decide_realloc);
}

constexpr int SCAN_BS = 1024;

__global__ void __launch_bounds__(SCAN_BS)
k_list_scan(View V, int decide_realloc)
{
    const DevBufs b = V.dom[blockIdx.x].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[blockIdx.x].c;
    if (b.cnt->status != MMCA_OK)
        return;
    list_scan<SCAN_BS, false>(b, c, decide_realloc);
}

__global__ void
k_realloc_decide(DevBufs b)
{
    Counters *cnt = b.cnt;
    if (cnt->status != MMCA_OK)
        return;
    if (cnt->gindex > cnt->dc_tmp_size)
    {
        cnt->realloc_old = cnt->dc_tmp_size;
        cnt->dc_tmp_size = cnt->gindex + 100;
    }
    else
        cnt->realloc_old = -1;
}

// Interface list writer (grow_cell_reduction, growth.c:496-513): slot
// base+i+1 of diff_id gets the padded index of the workgroup's member i, in
// raster order.  The members of a workgroup's 256 mask words are spread
// evenly over its threads: member i is found by a binary search over the
// per-word prefix counts in LDS.
__device__ __forceinline__ int
nth_set_bit(unsigned long long m, int r)
{
    int pos = 0;
#pragma unroll
    for (int half = 32; half > 0; half >>= 1)
    {
        const unsigned long long lo = m & ((1ull << half) - 1ull);
        const int c = __popcll(lo);
        if (r >= c)
        {
            r -= c;
            m >>= half;
            pos += half;
        }
        else
            m = lo;
    }
    return pos;
}

__global__ void __launch_bounds__(LIST_BS)
k_list_write(View V)
{
    __shared__ int s_w[LIST_BS / 64];
    __shared__ unsigned long long s_mem[LIST_BS];
    __shared__ unsigned long long s_nb[6][LIST_BS];   // solid bits of the 6 neighbours, per word
    __shared__ int s_ex[LIST_BS];
    const int dm = find_dom(V.off_list, V.ndom, blockIdx.x);
    const long long blk = blockIdx.x - V.off_list[dm];
    const DevBufs b = V.dom[dm].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[dm].c;
    const long long nwords = list_words_d(c);
    if (G(b.cnt)->status != MMCA_OK)
        return;
    const int base = G(b.blk_count)[blk];            // members before this workgroup
    const int next = blk + 1 < list_blocks_d(c) ? G(b.blk_count)[blk + 1] : G(b.cnt)->gindex;
    if (next == base && c.capture_band == 0)
        return;                                      // no members (the bands need every row's slot)
    const int W = c.list_w;                          // words of a workgroup: 64 or LIST_BS
    const long long wi0 = blk * W;
    const long long wi = wi0 + threadIdx.x;
    const bool mine = (int) threadIdx.x < W && wi < nwords;
    unsigned long long mem = 0;
    unsigned long long nb[6] = { 0, 0, 0, 0, 0, 0 };
    if (mine)
    {
        int k, j, w;
        word_pos(c, wi, &k, &j, &w);
        const unsigned long long own = mask_word(b, c, k, j, w);
        // bit b of each word: the neighbour of interior x = 64 w + b + 1 in the
        // capture order +x, +y, -x, -y, +z, -z (growth.c:604-610)
        x_neighbour_bits(b, c, k, j, w, own, &nb[2], &nb[0]);
        nb[1] = mask_word(b, c, k, j + 1, w);
        nb[3] = mask_word(b, c, k, j - 1, w);
        nb[4] = mask_word(b, c, k + 1, j, w);
        nb[5] = mask_word(b, c, k - 1, j, w);
        const int hi = c.nx - w * 64;
        const unsigned long long inter = (hi >= 64) ? ~0ull : ((1ull << hi) - 1ull);
        mem = ~own & (nb[0] | nb[1] | nb[2] | nb[3] | nb[4] | nb[5]) & inter;
    }
    int tot;
    int ex = block_exscan_int<LIST_BS / 64>(__popcll(mem), &tot, s_w);
    s_mem[threadIdx.x] = mem;
#pragma unroll
    for (int n = 0; n < 6; ++n)
        s_nb[n][threadIdx.x] = nb[n];
    s_ex[threadIdx.x] = ex;
    __syncthreads();
    if (mine)
    {
        // slot of the first member of each row (of the next member after the
        // row's start when the row has none), for capture's row bands
        int k, j, w;
        word_pos(c, wi, &k, &j, &w);
        if (w == 0)
            G(b.row_first)[(long long) (k - 1) * c.ny + (j - 1)] = base + ex + 1;
    }
    for (int i = threadIdx.x; i < tot; i += LIST_BS)
    {
        // word of member i: the last word whose prefix count is <= i
        int lo = 0, hi = W - 1;
        while (lo < hi)
        {
            int mid = (lo + hi + 1) >> 1;
            if (s_ex[mid] <= i)
                lo = mid;
            else
                hi = mid - 1;
        }
        const int bit = nth_set_bit(s_mem[lo], i - s_ex[lo]);
        int k, j, w;
        word_pos(c, wi0 + lo, &k, &j, &w);
        const int x = w * 64 + bit + 1;
        unsigned int pattern = 0;
#pragma unroll
        for (int n = 0; n < 6; ++n)
            pattern |= (unsigned int) ((s_nb[n][lo] >> bit) & 1ull) << n;
        G(b.diff_id)[base + i + 1] = (int) (k * c.sxy + (long long) j * c.sx + x);   // slots start at 1
        G(b.nbr)[base + i + 1] = (unsigned char) pattern;
    }
}

// capture_octahedra_diffuse, INDEX_SEP branch (growth.c:640-807), over the
// slots 1..gindex of the list.  Every member is independent: it reads only
// solid neighbours (through the pre-capture mask) and writes only itself and
// its slot, so the slots may be dealt to the threads in any order.  `cb` is
// the buffer holding fs/cl after fs_change; `rows` is 1 when the list writer
// of the same list has filled row_first (the row bands need it).
// Bound by the latency of its loads (slot, then neighbours, then rotation
// matrix; 2.3 TB/s), so by the waves in flight: 128 registers, for four waves
// per SIMD instead of three.
__global__ void __launch_bounds__(LIST_BS, 4)
k_capture(View V, int cb, int rows)
{
    const int dm = find_dom(V.off_cap, V.ndom, blockIdx.x);
    const long long blk = blockIdx.x - V.off_cap[dm];
    const long long nwg = V.off_cap[dm + 1] - V.off_cap[dm];
    const long long nthr = nwg * LIST_BS;
    const DevBufs b = V.dom[dm].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[dm].c;
    const MMCA_GLOBAL Counters *cnt = G(b.cnt);
    if (cnt->status != MMCA_OK)
        return;
    const int nmem = cnt->gindex;
    const bool realloc = cnt->realloc_old >= 0;
    const long long maxg = c.max_total_grains;
    MMCA_GLOBAL double *fsb = fs_buf(b, cb);
    MMCA_GLOBAL double *clb = cl_buf(b, cb);
    auto member = [&](long long t) {
        const int slot = (int) t + 1;
        const int idx = G(b.diff_id)[slot];
        double tx, ty, tz;
        if (realloc)
            tx = ty = tz = 0.0;
        else
        {
            tx = G(b.dtx)[slot];
            ty = G(b.dty)[slot];
            tz = G(b.dtz)[slot];
        }
        // neighbour order +x, +y, -x, -y, +z, -z (growth.c:686-700)
        const int nnx[6] = { 1, 0, -1, 0, 0, 0 };
        const int nny[6] = { 0, 1, 0, -1, 0, 0 };
        const int nnz[6] = { 0, 0, 0, 0, 1, -1 };
        const int sxy = (int) c.sxy;                     // padded cells < 2^31
        const int ndxs[6] = { idx + 1, idx + c.sx, idx - 1, idx - c.sx, idx + sxy, idx - sxy };
        // solid neighbours before capture (recorded by the list writer); their
        // grain ids, centres and fs are independent loads issued together
        const unsigned int sol = G(b.nbr)[slot];
        int gids[6];
        double pdc[6][3], pfs[6];
#pragma unroll
        for (int n = 0; n < 6; ++n)
        {
            gids[n] = 0;
            pdc[n][0] = pdc[n][1] = pdc[n][2] = pfs[n] = 0.0;
            if ((sol >> n) & 1u)
            {
                gids[n] = G(b.gr)[ndxs[n]];
                const MMCA_GLOBAL double *p = G(b.dc) + 3 * (long long) ndxs[n];
                pdc[n][0] = p[0];
                pdc[n][1] = p[1];
                pdc[n][2] = p[2];
                pfs[n] = fsb[ndxs[n]];
            }
        }
        int found = -1;
        int gfound = 0;
        double g00 = 0, g10 = 0, g20 = 0, g01 = 0, g11 = 0, g21 = 0, g02 = 0, g12 = 0, g22 = 0;
        double dx = 0, dy = 0, dz = 0, dn = 0, ddx = 0, ddy = 0, ddz = 0;
#pragma unroll
        for (int n = 0; n < 6; ++n)
        {
            const int gid = gids[n];
            if (found >= 0 || !(gid > 0 && gid < maxg))
                continue;
            const MMCA_GLOBAL double *R = G(b.g_rot) + 9 * (long long) gid;
            g00 = R[0]; g01 = R[1]; g02 = R[2];
            g10 = R[3]; g11 = R[4]; g12 = R[5];
            g20 = R[6]; g21 = R[7]; g22 = R[8];
            ddx = pdc[n][0];
            ddy = pdc[n][1];
            ddz = pdc[n][2];
            // grow_octahedra (growth.c:392-403)
            double rx0 = 0.0 - ddx;
            double ry0 = 0.0 - ddy;
            double rz0 = 0.0 - ddz;
            double gx0 = g00 * rx0 + g10 * ry0 + g20 * rz0;
            double gy0 = g01 * rx0 + g11 * ry0 + g21 * rz0;
            double gz0 = g02 * rx0 + g12 * ry0 + g22 * rz0;
            double ds1 = fabs(gx0) + fabs(gy0) + fabs(gz0);
            ds1 = ref_min(ds1, 1.5);
            dn = ds1 + pfs[n] * c.rev_fsgrow;
            // growth.c:717-735
            double rx1 = -1.0 * nnx[n] - ddx;
            double ry1 = -1.0 * nny[n] - ddy;
            double rz1 = -1.0 * nnz[n] - ddz;
            dx = g00 * rx1 + g10 * ry1 + g20 * rz1;
            dy = g01 * rx1 + g11 * ry1 + g21 * rz1;
            dz = g02 * rx1 + g12 * ry1 + g22 * rz1;
            double dfs = dn - (fabs(dx) + fabs(dy) + fabs(dz));
            if (dfs > 0)
            {
                found = n;
                gfound = gid;
            }
        }
        if (found > -1)
        {
            double ncx = 0., ncz = 0., ncy = 0.;
            double ncd = ref_min(dn, 1.0);
            double dd = dn - ncd;
            if (dx + dy >= 0 && dx - dy > 0 && dx + dz > 0 && dx - dz >= 0)
                ncx = dd;
            else if (dx + dy <= 0 && dx - dy < 0 && dx + dz < 0 && dx - dz <= 0)
                ncx = -1. * dd;
            else if (dy + dx > 0 && dy - dx >= 0 && dy + dz >= 0 && dy - dz > 0)
                ncy = dd;
            else if (dy + dx < 0 && dy - dx <= 0 && dy + dz <= 0 && dy - dz < 0)
                ncy = -1. * dd;
            else if (dz + dx >= 0 && dz - dx > 0 && dz + dy > 0 && dz - dy >= 0)
                ncz = dd;
            else
                ncz = -1. * dd;
            tx = ddx + nnx[found] + g00 * ncx + g01 * ncy + g02 * ncz;
            ty = ddy + nny[found] + g10 * ncx + g11 * ncy + g12 * ncz;
            tz = ddz + nnz[found] + g20 * ncx + g21 * ncy + g22 * ncz;
            G(b.gr)[idx] = gfound;
            fsb[idx] = 0.;
            if (V.lean)
                put_ce_of_liquid(b, cb, idx);         // cl = ce already
            else if (c.f32)
                cl32_buf(b, cb)[idx] = G(b.ce32)[idx];
            else
                clb[idx] = G(b.ce)[idx];
        }
        if (found > -1 || realloc)
        {
            G(b.dtx)[slot] = tx;
            G(b.dty)[slot] = ty;
            G(b.dtz)[slot] = tz;
        }
        G(b.dc)[3 * (long long) idx] = tx;
        G(b.dc)[3 * (long long) idx + 1] = ty;
        G(b.dc)[3 * (long long) idx + 2] = tz;
    };
    const int band = c.capture_band;
    const int nband = band > 0 ? (c.ny + band - 1) / band : 0;
    const int chunk = c.capture_chunk;
    if (rows && nband >= 8 && nwg >= 8)
    {
        // Units of `band` rows of one plane.  Band q of every plane belongs
        // to the XCD q % 8 (the hardware places workgroup w on XCD w % 8), and
        // the workgroups of this domain on one XCD take its units plane by
        // plane, one unit per workgroup at a time.  A member's solid
        // neighbours lie in its own row, in the rows next to it (mostly in
        // the same unit: one workgroup, one L1) and in the planes next to it
        // (units of the same XCD in flight together: one L2).
        const long long o = V.off_cap[dm];
        const int xcd = (int) (blockIdx.x % 8);
        const long long first = o + ((xcd - (int) (o % 8)) + 8) % 8;
        const long long rank = (blockIdx.x - first) / 8;
        const long long nxcd = (o + nwg - 1 - first) / 8 + 1;
        const int mine = (nband - 1 - xcd) / 8 + 1;            // bands of this XCD in a plane
        const long long nunit = (long long) c.nz * mine;
        const long long nrow = (long long) c.nz * c.ny;
        for (long long u = rank; u < nunit; u += nxcd)
        {
            const int k = (int) (u / mine);                    // plane k + 1
            const int q = xcd + 8 * (int) (u - (long long) k * mine);
            const long long r0 = (long long) k * c.ny + (long long) q * band;
            const long long r1 = (long long) k * c.ny + min((q + 1) * band, c.ny);
            const int s0 = max(1, min(G(b.row_first)[r0], nmem + 1));
            const int s1 = r1 < nrow ? max(s0, min(G(b.row_first)[r1], nmem + 1)) : nmem + 1;
            for (int t = s0 - 1 + (int) threadIdx.x; t < s1 - 1; t += LIST_BS)
                member(t);
        }
    }
    else if (chunk > 0 && nwg >= 8)
    {
        // Contiguous chunks of `chunk` slots, chunk q on the XCD q % 8: the
        // members of one chunk (about chunk / (nx * ny) planes of the
        // interface) share most of their solid neighbours, whose lines then
        // stay in that XCD's L2.  The hardware places workgroup w on XCD
        // w % 8; the workgroups of this domain on one XCD stride over the
        // 256-slot groups of that XCD's chunks.
        const int S = chunk / LIST_BS;
        const long long o = V.off_cap[dm];
        const int xcd = (int) (blockIdx.x % 8);
        const long long first = o + ((xcd - (int) (o % 8)) + 8) % 8;
        const long long rank = (blockIdx.x - first) / 8;
        const long long nxcd = (o + nwg - 1 - first) / 8 + 1;
        const long long nchunk = (nmem + chunk - 1) / chunk;
        const long long mine = (nchunk > xcd) ? (nchunk - 1 - xcd) / 8 + 1 : 0;
        for (long long u = rank; u < mine * S; u += nxcd)
        {
            const long long t = (xcd + 8 * (u / S)) * (long long) chunk + (u % S) * LIST_BS + threadIdx.x;
            if (t < nmem)
                member(t);
        }
    }
    else
        for (long long t = blk * LIST_BS + threadIdx.x; t < nmem; t += nthr)
            member(t);
}

// ---------------------------------------------------------------------------
// Sum of min(1,fs) (reduce_fs, growth.c:541-566) and of ce over the interior.
constexpr int RED_BS = 256;

__global__ void __launch_bounds__(RED_BS)
k_reduce_partial(DevBufs b, Consts c, int cb)
{
    __shared__ double s_a[RED_BS], s_b[RED_BS];
    double a = 0.0, s = 0.0;
    const long long N = (long long) c.nx * c.ny * c.nz;
    const MMCA_GLOBAL double *fs = fs_buf(b, cb);
    for (long long i = (long long) blockIdx.x * RED_BS + threadIdx.x; i < N;
         i += (long long) gridDim.x * RED_BS)
    {
        const unsigned ui = (unsigned) i, unx = (unsigned) c.nx, uny = (unsigned) c.ny;   // N < 2^31
        const unsigned row = ui / unx;
        int x = (int) (ui - row * unx) + 1;
        const unsigned kk = row / uny;
        int j = (int) (row - kk * uny) + 1;
        int k = (int) kk + 1;
        long long idx = k * c.sxy + (long long) j * c.sx + x;
        a += ref_min(1.0, fs[idx]);
        s += c.f32 ? (double) G(b.ce32)[idx] : G(b.ce)[idx];     // FP32: deviation from c0
    }
    s_a[threadIdx.x] = a;
    s_b[threadIdx.x] = s;
    __syncthreads();
    for (int d = RED_BS / 2; d > 0; d >>= 1)
    {
        if (threadIdx.x < d)
        {
            s_a[threadIdx.x] += s_a[threadIdx.x + d];
            s_b[threadIdx.x] += s_b[threadIdx.x + d];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        G(b.red_part)[2 * blockIdx.x] = s_a[0];
        G(b.red_part)[2 * blockIdx.x + 1] = s_b[0];
    }
}

__global__ void __launch_bounds__(RED_BS)
k_reduce_final(DevBufs b, int nblk, double *out)
{
    __shared__ double s_a[RED_BS], s_b[RED_BS];
    double a = 0.0, s = 0.0;
    for (int i = threadIdx.x; i < nblk; i += RED_BS)
    {
        a += G(b.red_part)[2 * i];
        s += G(b.red_part)[2 * i + 1];
    }
    s_a[threadIdx.x] = a;
    s_b[threadIdx.x] = s;
    __syncthreads();
    for (int d = RED_BS / 2; d > 0; d >>= 1)
    {
        if (threadIdx.x < d)
        {
            s_a[threadIdx.x] += s_a[threadIdx.x + d];
            s_b[threadIdx.x] += s_b[threadIdx.x + d];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        out[0] = s_a[0];
        out[1] = s_b[0];
    }
}

// ---------------------------------------------------------------------------
// Gaussian beam in the step.  The reference evaluates a 400-term quadrature at
// every solid cell; its value matters only where a cell grows or remelts.  So
// a step computes an approximate temperature of the whole block (k_beam_field,
// a few multiply-adds per cell), the solute kernel finishes every cell whose
// branch is the same over the approximation's whole error interval
// (branch_decided) and marks the others, and k_beam_finish evaluates the
// quadrature for the marked ones, bit for bit the reference's.
//
// The approximation: as functions of the time node t, the x factors
// exp(-(lx + v t)^2 / A(t)) are smooth over the quadrature's short range, so
// they are interpolated between beam_rank Chebyshev points tau_j (chosen on
// the host so that the error is below 1e-9).  With w_i(y, z) = ldt / Tl_i *
// exp(-ly^2 / A_i - lz^2 / (4 alpha t_i)) and interpolation weights C[i][j],
//   T = liniT + Tfront * sum_j X_j(x) (sum_i C[i][j] w_i(y, z)),
// where the inner sums change only with the track.

// With beam_sep (FP32-deviation storage) the temperature outputs of the block's
// interior come from the same product with all 400 nodes as points (then the
// weights are the unit matrix), in double: the quadrature's sum of products of
// separately rounded factors, within 1e-13 of it.

// Table shapes: x factors, one row per interpolation point, of beam_x_pitch
// columns (zero past nx); row factors, one row per (z, y) row of the block, of
// beam_rank values, beam_w_rows of them (zero past ny nz).
constexpr int BF_COLS = 128;                      // columns per workgroup of k_beam_field
constexpr int BF_ROWS = 64;                       // rows per workgroup
__host__ __device__ __forceinline__ int beam_x_pitch(const Consts &c) { return (c.nx + BF_COLS - 1) / BF_COLS * BF_COLS; }
__host__ __device__ __forceinline__ long long
beam_w_rows(const Consts &c)
{
    return ((long long) c.ny * c.nz + BF_ROWS - 1) / BF_ROWS * BF_ROWS;
}

// node factors (BeamTab) and plane factors of the quadrature
__global__ void __launch_bounds__(256)
k_beam_nodes(DevBufs b, Consts c)
{
    const double ls = c.lsd / (2. * 1.414);
    const double lalpha = beam_lalpha(c);
    const double ldt = beam_ldt(c);
    for (long long e = (long long) blockIdx.x * 256 + threadIdx.x; e < (long long) BEAM_NT * (c.nz + 3);
         e += 256ll * gridDim.x)
    {
        const int z = (int) (e / BEAM_NT) - 1, i = (int) (e % BEAM_NT);
        const double lt = (0.5 + i) * ldt;
        if (z < 0)
        {
            const double A = ls * ls + 4. * lalpha * lt;
            const double Tl = sqrt(lalpha * lt) * (ls * ls + 4. * lalpha * lt);
            G(b.beam_nodes)[BN_VLT * BEAM_NT + i] = c.lv * lt;
            G(b.beam_nodes)[BN_A * BEAM_NT + i] = A;
            G(b.beam_nodes)[BN_RA * BEAM_NT + i] = 1.0 / A;
            G(b.beam_nodes)[BN_TL * BEAM_NT + i] = Tl;
            G(b.beam_nodes)[BN_RTL * BEAM_NT + i] = 1.0 / Tl;
        }
        else
        {
            const double rz = c.origin[2] + ((c.off[2] + z) + 0.5) * c.cell_size;
            const double lz = rz - c.z0;
            G(b.beam_zq)[(long long) z * BEAM_NT + i] = lz * lz / (4. * lalpha * lt);
        }
    }
}

// The next three kernels take all domains of a view in one launch: a step of 64
// blocks of 20 x 18 x 16 cells takes 62 us, and took 920 with launches for each
// domain (256 blocks of 12^3: 98 and 3020).  A step uses the points of each
// domain's description; an output (OUT) of one block the points `out`.
//
// x factors at the interpolation points for timestep cnt->timestep + adv; says
// in BeamSet::key[1] whether the row factors have to be built for a new track,
// and empties the list of waiting cells
template <bool OUT>
__global__ void __launch_bounds__(256)
k_beam_ax(BeamView V, BeamSet out, int adv)
{
    const int dm = OUT ? 0 : find_dom(V.off_ax, V.ndom, blockIdx.x);
    const int blk = (int) blockIdx.x - (OUT ? 0 : (int) V.off_ax[dm]);
    const DevBufs b = V.dom[dm].b;    // private copies: stores cannot alias them
    const Consts c = V.dom[dm].c;
    const BeamSet p = OUT ? out : V.dom[dm].beam;
    const double sim_time = (G(b.cnt)->timestep + (unsigned long long) adv) * c.dt;
    const BeamNow bn = beam_now(c, sim_time);
    if (blk == 0 && threadIdx.x == 0)
    {
        const double held = G(p.key)[0];
        G(p.key)[1] = __double_as_longlong(held) == __double_as_longlong(bn.ynow) ? 0.0 : 1.0;
        G(p.key)[0] = bn.ynow;
        *b.und_n = 0;
    }
    const double ls = c.lsd / (2. * 1.414);
    const double lalpha = beam_lalpha(c);
    const int e = blk * 256 + threadIdx.x, xp = beam_x_pitch(c);
    const int j = e / xp, q = e - j * xp;
    if (j >= p.rank)
        return;
    const double t = G(p.tau)[j];
    const double rx = c.origin[0] + ((c.off[0] + q + 1) + 0.5) * c.cell_size;
    const double u = (rx - bn.xnow) + c.lv * t;
    G(p.ax)[e] = q < c.nx ? exp(-(u * u) / (ls * ls + 4. * lalpha * t)) : 0.0;   // columns past nx pad the row
}

// row factors: one workgroup per (z, y) row at a time; 16 groups of 16 threads
// share the nodes, each thread sums for one interpolation point at a time
template <bool OUT>
__global__ void __launch_bounds__(256)
k_beam_aw(BeamView V, BeamSet out)
{
    __shared__ double s_w[BEAM_NT];
    __shared__ double s_p[16][17];
    const int jj = threadIdx.x & 15, g = threadIdx.x >> 4;
    for (long long w = blockIdx.x; w < V.tot_aw; w += gridDim.x)
    {
        const int dm = OUT ? 0 : find_dom(V.off_aw, V.ndom, w);
        const long long row = w - (OUT ? 0 : V.off_aw[dm]);
        const DevBufs b = V.dom[dm].b;
        const Consts c = V.dom[dm].c;
        const BeamSet p = OUT ? out : V.dom[dm].beam;
        if (G(p.key)[1] == 0.0)
            continue;                             // uniform over the workgroup
        const int z = (int) (row / c.ny), y = (int) (row - (long long) z * c.ny);
        const double ldt = beam_ldt(c);
        const double ry = c.origin[1] + ((c.off[1] + y + 1) + 0.5) * c.cell_size;
        const double ly = ry - G(p.key)[0];
        const MMCA_GLOBAL double *node = G(b.beam_nodes), *zq = G(b.beam_zq) + (long long) (z + 1) * BEAM_NT;
        __syncthreads();                          // the row before has been read
        for (int i = threadIdx.x; i < BEAM_NT; i += 256)
            s_w[i] = ldt / node[BN_TL * BEAM_NT + i] * exp(-(ly * ly) / node[BN_A * BEAM_NT + i] - zq[i]);
        __syncthreads();
        if (!p.weights)
        {
            for (int i = threadIdx.x; i < BEAM_NT; i += 256)
                G(p.aw)[row * BEAM_NT + i] = s_w[i];
            continue;
        }
        for (int j0 = 0; j0 < p.rank; j0 += 16)
        {
            double v = 0.0;
            for (int i = g; i < BEAM_NT; i += 16)
                v += s_w[i] * G(p.weights)[(long long) i * p.rank + j0 + jj];
            s_p[g][jj] = v;
            __syncthreads();
            if (g == 0)
            {
                double t = 0.0;
                for (int q = 0; q < 16; ++q)
                    t += s_p[q][jj];
                G(p.aw)[row * p.rank + j0 + jj] = t;
            }
            __syncthreads();
        }
    }
}

// T over the interior (padded indexing; 49 us for 500 x 256 x 128 cells and 32
// points, where 400 points took 230): the product of the row factors (rows
// q = (z-1) ny + y-1) and the x factors on the matrix cores, in double into
// b.temp (OUT), or rounded to float into b.temp32.  v_mfma_f64_16x16x4f64 multiplies a 16 x 4
// tile of W (lane l: row l % 16, node slot l / 16) by a 4 x 16 tile of X
// (lane l: node slot l / 16, column l % 16) into a 16 x 16 tile held as four
// doubles per lane (lane l, register r: row l / 16 + 4 r, column l % 16).
// The sum over the nodes may take them in any order, so the node slot k of
// step s in a block of 16 nodes 16 t is node 16 t + 4 k + s % 4: each lane
// then loads four consecutive W values of its row at once.  A wave owns 64
// rows x 32 columns (4 x 2 tiles, 32 accumulators per lane); the four waves
// of a workgroup share its 64 rows and take 32 columns each.
typedef double dvec4 __attribute__((ext_vector_type(4)));

template <bool OUT>
__global__ void __launch_bounds__(256)
k_beam_field(BeamView V, BeamSet out, int adv)
{
    const int dm = OUT ? 0 : find_dom(V.off_field, V.ndom, blockIdx.x);
    const unsigned blk = blockIdx.x - (OUT ? 0u : (unsigned) V.off_field[dm]);
    const DevBufs b = V.dom[dm].b;
    const Consts c = V.dom[dm].c;
    const BeamSet p = OUT ? out : V.dom[dm].beam;
    const MMCA_GLOBAL Counters *cnt = G(b.cnt);
    if (!OUT && cnt->status != MMCA_OK)
        return;                                   // uniform over the workgroup; an output is one of a stopped block too
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int xp = beam_x_pitch(c), K = p.rank;
    const unsigned ntx = (unsigned) (xp / BF_COLS), slab = blk / ntx;
    const long long q0 = (long long) slab * BF_ROWS;
    const int x0 = (int) (blk - slab * ntx) * BF_COLS + wave * 32;      // 0-based interior column
    const int kk = lane >> 4, lr = lane & 15;
    const double sim_time = (cnt->timestep + (unsigned long long) adv) * c.dt;
    const BeamNow bn = beam_now(c, sim_time);
    const long long nq = (long long) c.ny * c.nz;
    // stores tile (a, bb) register r: row q0 + 16 a + kk + 4 r, column x0 + 16 bb + lr
    const unsigned uy = (unsigned) c.ny;
    const int z0 = (int) (q0 / uy), y0 = (int) (q0 - (long long) z0 * uy);       // 0-based plane and row of q0
    auto store = [&](int a, int bb, int r, double sum, bool sep) {
        const int d = 16 * a + kk + 4 * r, x = x0 + 16 * bb + lr;
        if (q0 + d >= nq || x >= c.nx)
            return;
        // 32-bit arithmetic: a 64-bit division per value cost more than the product
        const unsigned t0 = (unsigned) (y0 + d), dz = uy >= BF_ROWS ? (t0 >= uy ? 1u : 0u) : t0 / uy;
        const int z = z0 + (int) dz + 1, y = (int) (t0 - dz * uy) + 1;
        const double rz = c.origin[2] + ((c.off[2] + z) + 0.5) * c.cell_size;
        double t;
        if (!(rz <= bn.znow + c.cell_size))
            t = 0.0;
        else if (!sep)
            t = c.liniT + bn.Tfront * 0.0;        // every term is finite: liniT + 0
        else
            t = c.liniT + bn.Tfront * sum;
        const long long at = (long long) z * c.sxy + (long long) y * c.sx + x + 1;
        if (OUT)
            G(b.temp)[at] = t;
        else
            G(b.temp32)[at] = (float) t;
    };
    if (bn.Tfront == 0.0)
    {
        for (int a = 0; a < 4; ++a)
            for (int bb = 0; bb < 2; ++bb)
                for (int r = 0; r < 4; ++r)
                    store(a, bb, r, 0.0, false);
        return;
    }
    // this lane's W rows (one per row tile) and X columns (one per column tile)
    const MMCA_GLOBAL double *Wr[4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
        Wr[a] = G(p.aw) + (q0 + 16 * a + lr) * K + 4 * kk;
    const MMCA_GLOBAL double *Xc = G(p.ax) + x0 + lr + (long long) (4 * kk) * xp;
    dvec4 acc[4][2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
        for (int bb = 0; bb < 2; ++bb)
            acc[a][bb] = dvec4{0.0, 0.0, 0.0, 0.0};
    // one block of 16 nodes: loads, then 4 steps of 8 MFMAs
    dvec4 wa[4];
    double xb[2][4];
    auto load = [&](int t) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
            wa[a] = *reinterpret_cast<const MMCA_GLOBAL dvec4 *>(Wr[a] + 16 * t);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int bb = 0; bb < 2; ++bb)
                xb[bb][m] = Xc[(long long) (16 * t + m) * xp + 16 * bb];
    };
    load(0);
    for (int t = 0; t < K / 16; ++t)
    {
        const dvec4 ca[4] = { wa[0], wa[1], wa[2], wa[3] };
        const double cb[2][4] = { { xb[0][0], xb[0][1], xb[0][2], xb[0][3] },
                                  { xb[1][0], xb[1][1], xb[1][2], xb[1][3] } };
        if (t + 1 < K / 16)
            load(t + 1);                          // the next block's loads overlap this block's MFMAs
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int bb = 0; bb < 2; ++bb)
                    acc[a][bb] = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[a][m], cb[bb][m], acc[a][bb], 0, 0, 0);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int bb = 0; bb < 2; ++bb)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                store(a, bb, r, acc[a][bb][r], true);
}

// The cells the solute kernel left (DevBufs::und): the quadrature, then the
// partitioning from what defer_cell kept.  The listed cells are dealt evenly to
// the grid's threads: one thread per cell, or two or four while the grid has
// that many, so that the 400-term chains stay short.
//
// A step that the solute kernel stopped on a negative ce is finished too: its
// waiting cells hold what defer_cell kept, and its buffers stay current.  The
// steps issued after it leave the list empty (k_beam_ax).
//
// Bound by the FP64 VALU of the quadrature, about 40 instructions per term.
// About 120 000 waiting cells of a 250 x 190 x 94 block: 85 us; a kernel that
// evaluated every solid cell in place took 10 ms a step.
template <bool F32>
__global__ void __launch_bounds__(256)
k_beam_finish(View V, int cur, int nxt)
{
    __shared__ BeamTab s_tab;
    const DevBufs b = V.dom[blockIdx.y].b;    // private copy: stores cannot alias it
    const Consts c = V.dom[blockIdx.y].c;
    const MMCA_GLOBAL Counters *cnt = G(b.cnt);
    if (cnt->status != MMCA_OK && !(cnt->status == MMCA_ERR_NEGATIVE_CE && cnt->failed_step == cnt->timestep))
        return;
    const int tid = threadIdx.x;
    const int n = *G(b.und_n);
    const long long nthr = 256ll * gridDim.x;
    // log2 of the threads per cell: up to about one wave on each of the 1024 SIMDs
    const int sh = n <= 16384 ? 2 : n <= 32768 ? 1 : 0;
    if (256ll * blockIdx.x >= (long long) n << sh)
        return;                                   // uniform over the workgroup
    beam_tab_load(b, s_tab, tid, 256);
    __syncthreads();
    const BeamNow bn = beam_now(c, G(b.cnt)->timestep * c.dt);
    const int g = tid & ((1 << sh) - 1);
    for (long long i = (256ll * blockIdx.x + tid) >> sh; i < n; i += nthr >> sh)
    {
        const int idx = G(b.und)[i];
        const int k = (int) (idx / c.sxy), rem = (int) (idx - k * c.sxy), j = rem / c.sx, x = rem - j * c.sx;
        const MMCA_GLOBAL double *Z = G(b.beam_zq) + (long long) k * BEAM_NT;
        const double T = sh == 2   ? beam_quad<4>(c, b, s_tab, Z, bn, x, j, k, g)
                         : sh == 1 ? beam_quad<2>(c, b, s_tab, Z, bn, x, j, k, g)
                                   : beam_quad<1>(c, b, s_tab, Z, bn, x, j, k, 0);
        const double kept = fs_buf(b, nxt)[idx];
        const double ce_new = F32 ? kept : G(b.ce)[idx];
        const double ce_prev = F32 ? c.cinit + (double) cl32_buf(b, nxt)[idx] : kept;
        const double conc = ld_cl<F32>(b, c, cur, idx), lspfs = fs_buf(b, cur)[idx];
        const int g_old = G(b.gr)[idx];
        double cl_out, fs_out;
        int g_new, branch;
        partition_cell(c, [&]() { return T; }, ce_new, ce_prev, conc, lspfs, g_old, &cl_out, &fs_out, &g_new, &branch);
        if (g == 0)
        {
            st_cl<F32>(b, c, nxt, idx, cl_out);
            st_stream(fs_buf(b, nxt), idx, fs_out);
            if (g_new != g_old)
                G(b.gr)[idx] = g_new;
            if (g_new > 0)
                atomicOr(&b.mask[((long long) k * (c.ny + 2) + j) * c.w64 + (x - 1) / 64], 1ull << ((x - 1) & 63));
            keep_stale_d(c, b, idx, g_old, g_new, lspfs);
        }
    }
}

// The quadrature over the padded box, or over its halo cells only
__global__ void __launch_bounds__(256)
k_beam_fill(DevBufs b, Consts c, int halo, double *out)
{
    __shared__ BeamTab s_tab;
    beam_tab_load(b, s_tab, threadIdx.x, 256);
    __syncthreads();
    const BeamNow bn = beam_now(c, G(b.cnt)->timestep * c.dt);
    const long long nA = 2 * c.sxy, nB = 2ll * c.nz * c.sx, nC = 2ll * c.ny * c.nz;
    const long long n = halo ? nA + nB + nC : c.P;
    for (long long e = (long long) blockIdx.x * 256 + threadIdx.x; e < n; e += 256ll * gridDim.x)
    {
        int x, y, z;
        if (!halo || e < nA)
        {
            z = (int) (e / c.sxy);
            const long long rem = e - z * c.sxy;
            y = (int) (rem / c.sx);
            x = (int) (rem - (long long) y * c.sx);
            if (halo && z == 1)
                z = c.nz + 1;
        }
        else if (e < nA + nB)
        {
            const long long f = e - nA, row = f / c.sx;
            x = (int) (f - row * c.sx);
            z = (int) (row >> 1) + 1;
            y = (row & 1) ? c.ny + 1 : 0;
        }
        else
        {
            const long long f = e - nA - nB, row = f >> 1;
            x = (f & 1) ? c.nx + 1 : 0;
            z = (int) (row / c.ny) + 1;
            y = (int) (row - (long long) (z - 1) * c.ny) + 1;
        }
        out[z * c.sxy + (long long) y * c.sx + x] =
            beam_quad<1>(c, b, s_tab, G(b.beam_zq) + (long long) z * BEAM_NT, bn, x, y, z, 0);
    }
}

hipError_t launch_beam_nodes(const DevBufs &b, const Consts &c, hipStream_t s)
{
    const long long n = (long long) BEAM_NT * (c.nz + 3);
    hipLaunchKernelGGL(k_beam_nodes, dim3((unsigned) std::min<long long>((n + 255) / 256, 1024)), dim3(256), 0, s, b, c);
    return hipGetLastError();
}

long long beam_x_blocks(const Consts &c, int rank) { return ((long long) rank * beam_x_pitch(c) + 255) / 256; }
long long beam_rows(const Consts &c) { return (long long) c.ny * c.nz; }
long long beam_field_blocks(const Consts &c) { return beam_x_pitch(c) / BF_COLS * (beam_w_rows(c) / BF_ROWS); }

// a launch takes less than 2^32 threads; a block of 2^24 rows would need more
static dim3 aw_grid(const BeamView &v) { return dim3((unsigned) std::min<long long>(v.tot_aw, 65536)); }

// The approximate beam temperature of timestep cnt->timestep + adv into b.temp32
// of every domain; the row factors too when `rows` (they may be stale)
hipError_t launch_beam_field(const BeamView &v, int adv, int rows, hipStream_t s)
{
    const BeamSet none = {};
    hipLaunchKernelGGL(k_beam_ax<false>, dim3((unsigned) v.tot_ax), dim3(256), 0, s, v, none, adv);
    if (rows)
        hipLaunchKernelGGL(k_beam_aw<false>, aw_grid(v), dim3(256), 0, s, v, none);
    hipLaunchKernelGGL(k_beam_field<false>, dim3((unsigned) v.tot_field), dim3(256), 0, s, v, none, adv);
    return hipGetLastError();
}

// The temperature of timestep cnt->timestep into b.temp of a view's only domain,
// from the point set p
hipError_t launch_beam_output(const BeamView &v, const Consts &c, const BeamSet &p, hipStream_t s)
{
    hipLaunchKernelGGL(k_beam_ax<true>, dim3((unsigned) beam_x_blocks(c, p.rank)), dim3(256), 0, s, v, p, 0);
    hipLaunchKernelGGL(k_beam_aw<true>, aw_grid(v), dim3(256), 0, s, v, p);
    hipLaunchKernelGGL(k_beam_field<true>, dim3((unsigned) beam_field_blocks(c)), dim3(256), 0, s, v, p, 0);
    return hipGetLastError();
}

// at most 1024 workgroups per domain: four waves per SIMD of the whole chip
hipError_t launch_beam_finish(const View &v, int f32, int cur, int nxt, hipStream_t s)
{
    const long long per = (v.tot_count * LIST_BS * 64 / v.ndom + 1023) / 1024;     // cells per domain / 1024, about
    const dim3 grid((unsigned) std::max<long long>(1, std::min<long long>(1024, per)), (unsigned) v.ndom);
    if (f32)
        hipLaunchKernelGGL(k_beam_finish<true>, grid, dim3(256), 0, s, v, cur, nxt);
    else
        hipLaunchKernelGGL(k_beam_finish<false>, grid, dim3(256), 0, s, v, cur, nxt);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Derived fields for download: the temperature of the other models (the
// beam's comes from k_beam_fill and, with beam_sep, k_beam_field).
__global__ void
k_fill_temp(DevBufs b, Consts c, double *out)
{
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.P)
        return;
    int z = (int) (i / c.sxy);
    long long rem = i - z * c.sxy;
    int y = (int) (rem / c.sx);
    int x = (int) (rem - (long long) y * c.sx);
    out[i] = temp_model<false>(c, G(b.cnt)->timestep * c.dt, x, y, z);
}

// cache_io_data (loop.c:74-113): FP32 copies of fs, ce and the temperature
// and a copy of gr over the padded box, for the output writers.  A null
// output is skipped; a beam's temperature is in b.temp.
template <bool F32>
__global__ void
k_io_fields(DevBufs b, Consts c, int cur, float *fs_io, float *ce_io, float *t_io, int *gr_io)
{
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.P)
        return;
    if (fs_io)
        fs_io[i] = (float) fs_buf(b, cur)[i];
    if (ce_io)
        ce_io[i] = (float) ld_ce<F32>(b, c, i);
    if (gr_io)
        gr_io[i] = G(b.gr)[i];
    if (t_io && c.am)
        t_io[i] = (float) G(b.temp)[i];
    else if (t_io)
    {
        int z = (int) (i / c.sxy);
        long long rem = i - z * c.sxy;
        int y = (int) (rem / c.sx);
        int x = (int) (rem - (long long) y * c.sx);
        t_io[i] = (float) temp_model<false>(c, G(b.cnt)->timestep * c.dt, x, y, z);
    }
}

hipError_t launch_io_fields(const DevBufs &b, const Consts &c, int cur, float *fs_io, float *ce_io, float *t_io,
                            int *gr_io, hipStream_t s)
{
    const dim3 grid((unsigned) ((c.P + 255) / 256));
    if (c.f32)
        hipLaunchKernelGGL(k_io_fields<true>, grid, dim3(256), 0, s, b, c, cur, fs_io, ce_io, t_io, gr_io);
    else
        hipLaunchKernelGGL(k_io_fields<false>, grid, dim3(256), 0, s, b, c, cur, fs_io, ce_io, t_io, gr_io);
    return hipGetLastError();
}

// grow_octahedra (growth.c:339-407) into the d buffer
__global__ void
k_grow_octahedra(DevBufs b, Consts c, int cb)
{
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= c.P || b.cnt->status != MMCA_OK)
        return;
    int z = (int) (i / c.sxy);
    long long rem = i - z * c.sxy;
    int y = (int) (rem / c.sx);
    int x = (int) (rem - (long long) y * c.sx);
    if (x < 1 || x > c.nx || y < 1 || y > c.ny || z < 1 || z > c.nz)
        return;
    int grid = G(b.gr)[i];
    // with track_d the solid set is the one of the last growth step (the
    // mask the solute kernel wrote, before capture), as in the reference
    const bool solid = c.track_d
        ? ((G(b.mask)[((long long) z * (c.ny + 2) + y) * c.w64 + (x - 1) / 64] >> ((x - 1) % 64)) & 1ull) != 0
        : grid > 0;
    if (solid && grid > 0 && grid < c.max_total_grains)
        G(b.d)[i] = octa_d(c, b, i, grid, fs_buf(b, cb)[i]);
}

// ---------------------------------------------------------------------------
// Launch wrappers (host side).
hipError_t launch_nucleate(const View &v, int mode, int cur, hipStream_t s)
{
    if (mode & 1)
        hipLaunchKernelGGL(k_nuc_detect, dim3((unsigned) v.tot_nuc), dim3(NUC_BS), 0, s, v, mode, cur);
    else
        hipLaunchKernelGGL(k_nuc_activate, dim3(v.ndom), dim3(NUC_BS), 0, s, v, mode);
    return hipGetLastError();
}

// Nucleation of a coupled batch: detection and event order per domain, then
// activation across the domains in rank order (which advances the timestep:
// detection works at the next one).
hipError_t launch_nucleate_coupled(const View &v, int cur, hipStream_t s)
{
    hipLaunchKernelGGL(k_nuc_detect, dim3((unsigned) v.tot_nuc), dim3(NUC_BS), 0, s, v, 1 | 8, cur);
    hipLaunchKernelGGL(k_nuc_activate_coupled, dim3(1), dim3(NUC_BS), 0, s, v, cur);
    return hipGetLastError();
}

// `max_face`: the largest face (cells) or halo-row word count of any domain
hipError_t launch_halo_exchange(const View &v, int phase, int cb, long long max_face, hipStream_t s)
{
    const unsigned gx = (unsigned) ((max_face + 255) / 256);
    hipLaunchKernelGGL(k_halo_exchange, dim3(gx, (unsigned) (6 * v.ndom)), dim3(256), 0, s, v, phase, cb);
    return hipGetLastError();
}

// zm_by: rows of the z-marching kernel (all domains of a view share it); 0
// selects the cell-parallel kernel.
template <bool AM, bool F32>
static void launch_solute_t(const View &v, int zm_by, int diff, int fsc, int rec, int cur, int nxt, hipStream_t s)
{
    dim3 blk(SOL_BX, SOL_BY);
    if (rec)
    {
        // branch recording: FP64 storage, fused cell-parallel kernel (the caller checks)
        if (diff && fsc && !F32)
            hipLaunchKernelGGL((k_solute<true, true, AM, false, true>), dim3((unsigned) v.tot_cell), blk, 0, s, v,
                               cur, nxt);
        return;
    }
    if (diff && fsc && zm_by > 0)
    {
        const long long run = 8ll * v.xcd_run;
        const dim3 grid((unsigned) ((v.tot_zm + run - 1) / run * run));
        const size_t tlds = AM ? 0 : (size_t) std::max(v.zm_planes_max, 16) * sizeof(double);   // per plane or row
        const dim3 wg(64, zm_by == 16 ? 8 : 4);      // waves of 2 rows (of 1 row for 4-row tiles)
        if constexpr (!F32 && !AM)
            if (v.lean)
            {
                if (zm_by == 4)
                    hipLaunchKernelGGL((k_solute_rw<1, F32, AM, true>), grid, wg, tlds, s, v, cur, nxt);
                else
                    hipLaunchKernelGGL((k_solute_rw<2, F32, AM, true>), grid, wg, tlds, s, v, cur, nxt);
                return;
            }
        if (zm_by == 4)
            hipLaunchKernelGGL((k_solute_rw<1, F32, AM, false>), grid, wg, tlds, s, v, cur, nxt);
        else
            hipLaunchKernelGGL((k_solute_rw<2, F32, AM, false>), grid, wg, tlds, s, v, cur, nxt);
    }
    else if (diff && fsc)
        hipLaunchKernelGGL((k_solute<true, true, AM, F32>), dim3((unsigned) v.tot_cell), blk, 0, s, v, cur, nxt);
    else if (F32)
        return;     // single operators run on FP64 storage only (the caller checks)
    else if (diff)
        hipLaunchKernelGGL((k_solute<true, false, AM, false>), dim3((unsigned) v.tot_cell), blk, 0, s, v, cur,
                           nxt);
    else
        hipLaunchKernelGGL((k_solute<false, true, AM, false>), dim3((unsigned) v.tot_cell), blk, 0, s, v, cur,
                           nxt);
}

hipError_t launch_solute(const View &v, int am, int f32, int zm_by, int diff, int fsc, int rec, int cur,
                         int nxt, hipStream_t s)
{
    if (am)
    {
        if (f32)
            launch_solute_t<true, true>(v, zm_by, diff, fsc, rec, cur, nxt, s);
        else
            launch_solute_t<true, false>(v, zm_by, diff, fsc, rec, cur, nxt, s);
    }
    else
    {
        if (f32)
            launch_solute_t<false, true>(v, zm_by, diff, fsc, rec, cur, nxt, s);
        else
            launch_solute_t<false, false>(v, zm_by, diff, fsc, rec, cur, nxt, s);
    }
    return hipGetLastError();
}

hipError_t launch_mask_from_gr(const DevBufs &b, const Consts &c, hipStream_t s)
{
    hipLaunchKernelGGL(k_mask_from_gr, dim3(c.w64, c.ny + 2, c.nz + 2), dim3(64), 0, s, b, c);
    return hipGetLastError();
}

long long list_words(const Consts &c) { return list_words_d(c); }
int list_blocks(const Consts &c) { return list_blocks_d(c); }
int count_blocks(const Consts &c) { return (int) ((list_words(c) + LIST_BS - 1) / LIST_BS); }
// The list writer takes 64 words per workgroup while that gives at most 2048
// workgroups (15.4 -> 7.7 us for the 65536 words and 450 000 members of 128 x
// 128 x 256, which gave 256 workgroups), and 256 in larger blocks: with 8192
// workgroups of 64 words, 256 x 256 x 512 takes 22.6 us to write and 10.3 to
// scan, against 16.5 and 4.7.
int list_unit(const Consts &c) { return list_words(c) <= 64 * 2048 ? 64 : LIST_BS; }
// Capture's workgroups: the list's slots are dealt to their threads, so a small
// block needs more of them than its mask has words (40 x 36 x 44: 7 workgroups
// took 19.5 us for 13 000 slots, 62 take 6.5).
int capture_blocks(const Consts &c)
{
    const long long cells = (long long) c.nx * c.ny * c.nz;
    return (int) std::max<long long>((list_words(c) + LIST_BS - 1) / LIST_BS, std::min<long long>(1024, (cells + 1023) / 1024));
}
int nuc_blocks(int nsites) { return std::max(1, (nsites + NUC_BS - 1) / NUC_BS); }   // at least the one that activates
long long cell_blocks(const Consts &c)
{
    return (long long) ((c.nx + SOL_BX - 1) / SOL_BX) * ((c.ny + SOL_BY - 1) / SOL_BY) *
           ((c.nz + SOL_BZ - 1) / SOL_BZ);
}
long long zm_tiles(const Consts &c, int by)
{
    return (long long) ((c.nx + 63) / 64) * ((c.ny + by - 1) / by) * ((c.nz + c.zm_planes - 1) / c.zm_planes);
}

// Up to this many list-count workgroups the scan runs in their launch: a 40 x
// 36 x 44 block (7 workgroups) steps in 28.3 instead of 29.4 us, a 99 x 130 x
// 121 one (123) in 47.8 instead of 48.2; 150 x 140 x 165 (271) takes 65.9 against
// 63.8 us with a launch of its own, 256 x 256 x 512 (8192) 603 against 571: the
// counter that orders the workgroups is one address for all XCDs.
constexpr long long LIST_FUSED = 192;

long long tile_slots(const Consts &c) { return tile_slots_d(c); }


hipError_t launch_wake_all(const View &v, hipStream_t s)
{
    hipLaunchKernelGGL(k_wake_all, dim3(64, (unsigned) v.ndom), dim3(256), 0, s, v);
    return hipGetLastError();
}

hipError_t launch_settle(const DomainDesc *dom, int cur, unsigned failed, hipStream_t s)
{
    hipLaunchKernelGGL(k_settle, dim3(1024), dim3(256), 0, s, dom, cur, failed);
    return hipGetLastError();
}

hipError_t launch_list(const View &v, int cb, int capture, int decide_realloc, hipStream_t s)
{
    const dim3 grid((unsigned) v.tot_count);
    if (v.tot_count <= LIST_FUSED)
        hipLaunchKernelGGL(k_list_count<true>, grid, dim3(LIST_BS), 0, s, v, decide_realloc);
    else
    {
        hipLaunchKernelGGL(k_list_count<false>, grid, dim3(LIST_BS), 0, s, v, decide_realloc);
        hipLaunchKernelGGL(k_list_scan, dim3(v.ndom), dim3(SCAN_BS), 0, s, v, decide_realloc);
    }
    if (capture >= 0)
        hipLaunchKernelGGL(k_list_write, dim3((unsigned) v.tot_list), dim3(LIST_BS), 0, s, v);
    if (capture > 0)
        hipLaunchKernelGGL(k_capture, dim3((unsigned) v.tot_cap), dim3(LIST_BS), 0, s, v, cb, 1);
    return hipGetLastError();
}

hipError_t launch_capture_only(const View &v, const DevBufs &b, int cb, hipStream_t s)
{
    hipLaunchKernelGGL(k_realloc_decide, dim3(1), dim3(1), 0, s, b);
    // the list may come from a state image, which holds no row_first
    hipLaunchKernelGGL(k_capture, dim3((unsigned) v.tot_cap), dim3(LIST_BS), 0, s, v, cb, 0);
    return hipGetLastError();
}

// the counters of every domain of a view, side by side
__global__ void __launch_bounds__(64)
k_gather_counters(View V, Counters *out)
{
    for (int d = blockIdx.x * 64 + threadIdx.x; d < V.ndom; d += 64 * gridDim.x)
        out[d] = *V.dom[d].b.cnt;
}

hipError_t launch_gather_counters(const View &v, Counters *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_gather_counters, dim3((unsigned) std::min(1024, (v.ndom + 63) / 64)), dim3(64), 0, s, v, out);
    return hipGetLastError();
}

__global__ void __launch_bounds__(64)
k_reset_new_grains(View V)
{
    for (int d = blockIdx.x * 64 + threadIdx.x; d < V.ndom; d += 64 * gridDim.x)
        V.dom[d].b.cnt->new_grains = 0;
}

hipError_t launch_reset_new_grains(const View &v, hipStream_t s)
{
    hipLaunchKernelGGL(k_reset_new_grains, dim3((unsigned) std::min(1024, (v.ndom + 63) / 64)), dim3(64), 0, s, v);
    return hipGetLastError();
}

int reduce_blocks(const Consts &c)
{
    long long N = (long long) c.nx * c.ny * c.nz;
    long long nb = (N + RED_BS * 8 - 1) / (RED_BS * 8);
    if (nb > 2048)
        nb = 2048;
    if (nb < 1)
        nb = 1;
    return (int) nb;
}

hipError_t launch_reduce(const DevBufs &b, const Consts &c, int cb, double *out2, hipStream_t s)
{
    hipLaunchKernelGGL(k_reduce_partial, dim3(b.nblk_red), dim3(RED_BS), 0, s, b, c, cb);
    hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(RED_BS), 0, s, b, b.nblk_red, out2);
    return hipGetLastError();
}

// temperature over the padded box (with beam_sep: of the halo cells, the
// interior is the separable field)
hipError_t launch_fill_temp(const DevBufs &b, const Consts &c, double *out, hipStream_t s)
{
    if (c.am)
    {
        const long long n = c.beam_sep ? 2 * c.sxy + 2ll * c.nz * c.sx + 2ll * c.ny * c.nz : c.P;
        hipLaunchKernelGGL(k_beam_fill, dim3((unsigned) std::min<long long>((n + 255) / 256, 8192)), dim3(256), 0, s,
                           b, c, c.beam_sep, out);
    }
    else
        hipLaunchKernelGGL(k_fill_temp, dim3((unsigned) ((c.P + 255) / 256)), dim3(256), 0, s, b, c, out);
    return hipGetLastError();
}

hipError_t launch_grow_octahedra(const DevBufs &b, const Consts &c, int cb, hipStream_t s)
{
    hipLaunchKernelGGL(k_grow_octahedra, dim3((unsigned) ((c.P + 255) / 256)), dim3(256), 0, s, b, c, cb);
    return hipGetLastError();
}

}  // namespace mmca

namespace mmca {

__global__ void
k_fill_f64(double *p, long long n, double v)
{
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

hipError_t launch_fill_f64(double *p, long long n, double v, hipStream_t s)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_fill_f64, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

// FP32 deviations to values and back, for fields on their way to and from the
// host: bound by the copy over PCIe next to it (a loop on one host core took
// 1.4 ns per cell and field: 22 ms for 205 x 251 x 303 cells, now 2.2).
__global__ void __launch_bounds__(256)
k_widen(const float *in, double *out, double c0, long long n)
{
    const long long i = (long long) blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        out[i] = c0 + (double) in[i];
}

__global__ void __launch_bounds__(256)
k_narrow(const double *in, float *out, float *out2, double c0, long long n)
{
    const long long i = (long long) blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    const float f = (float) (in[i] - c0);
    out[i] = f;
    if (out2)
        out2[i] = f;
}

hipError_t launch_widen(const float *in, double *out, double c0, long long n, hipStream_t s)
{
    hipLaunchKernelGGL(k_widen, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, in, out, c0, n);
    return hipGetLastError();
}

hipError_t launch_narrow(const double *in, float *out, float *out2, double c0, long long n, hipStream_t s)
{
    hipLaunchKernelGGL(k_narrow, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, in, out, out2, c0, n);
    return hipGetLastError();
}

// Streaming probes of the bandwidth a kernel with the solute kernel's field
// mix can reach: no arithmetic beyond a dependency that keeps every load
// live.  Each workgroup streams one contiguous run of PROBE_RUN cells: every
// thread issues the loads of PROBE_UNROLL cells 256 apart, then their stores.
// Short contiguous runs on many workgroups stream faster here than a grid
// stride over the whole array (about 5.3 against 4.3-5.2 TB/s for mix 1,
// depending on the grid).
//   mix 0: copy          read a f64, write b f64                         16 B/cell
//   mix 1: FP64 fields   read ce, cl, fs f64 and gr i32; write ce, cl, fs 52 B/cell
//   mix 2: FP32 fields   read ce, cl f32, fs f64, gr i32; write ce, cl, fs 36 B/cell
constexpr int PROBE_UNROLL = 4;
constexpr int PROBE_RUN = 256 * PROBE_UNROLL;

template <int MIX>
__global__ void __launch_bounds__(256)
k_probe(long long n, double *a, double *b, double *f, float *ea, float *eb, int *g)
{
    const long long i0 = (long long) blockIdx.x * PROBE_RUN + threadIdx.x;
    double v0[PROBE_UNROLL], v1[PROBE_UNROLL], v2[PROBE_UNROLL];
    int gv[PROBE_UNROLL];
#pragma unroll
    for (int u = 0; u < PROBE_UNROLL; ++u)
    {
        const long long i = min(i0 + u * 256, n - 1);
        if constexpr (MIX == 0)
            v0[u] = G(a)[i];
        else if constexpr (MIX == 1)
        {
            v0[u] = G(a)[i];
            v1[u] = G(b)[i];
            v2[u] = G(f)[i];
            gv[u] = G(g)[i];
        }
        else
        {
            v0[u] = G(ea)[i];
            v1[u] = G(eb)[i];
            v2[u] = G(f)[i];
            gv[u] = G(g)[i];
        }
    }
#pragma unroll
    for (int u = 0; u < PROBE_UNROLL; ++u)
    {
        const long long i = i0 + u * 256;
        if (i >= n)
            break;
        if constexpr (MIX == 0)
            G(b)[i] = v0[u];
        else if constexpr (MIX == 1)
        {
            G(a)[i] = v0[u] + gv[u];
            G(b)[i] = v1[u];
            G(f)[i] = v2[u];
        }
        else
        {
            G(ea)[i] = (float) v0[u] + gv[u];
            G(eb)[i] = (float) v1[u];
            G(f)[i] = v2[u];
        }
    }
}

hipError_t launch_probe(int mix, long long n, double *a, double *b, double *f, float *ea, float *eb, int *g,
                        hipStream_t s)
{
    const unsigned grid = (unsigned) ((n + PROBE_RUN - 1) / PROBE_RUN);
    if (mix == 0)
        hipLaunchKernelGGL(k_probe<0>, dim3(grid), dim3(256), 0, s, n, a, b, f, ea, eb, g);
    else if (mix == 1)
        hipLaunchKernelGGL(k_probe<1>, dim3(grid), dim3(256), 0, s, n, a, b, f, ea, eb, g);
    else
        hipLaunchKernelGGL(k_probe<2>, dim3(grid), dim3(256), 0, s, n, a, b, f, ea, eb, g);
    return hipGetLastError();
}

// y[i] = exp(x[i]) through the beam quadrature's exp (mmca_exp.h), with the
// table read from constant memory as temp_model<true> reads it
__global__ void
k_eval_exp(const double *x, double *y, long long n)
{
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        y[i] = exp_glibc(x[i], exp_tab);
}

hipError_t launch_eval_exp(const double *x, double *y, long long n, hipStream_t s)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_eval_exp, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, x, y, n);
    return hipGetLastError();
}

}  // namespace mmca
