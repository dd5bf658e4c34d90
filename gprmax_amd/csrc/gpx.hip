// MI355X (gfx950) FDTD solve path: Yee E/H updates with fused CFS-PML slab
// corrections, dispersive multipole A/B, point sources, receivers and
// snapshots.  C ABI declared in include/gpx.h.
//
// Kernels.  gpx_rows.h has the row kernels, which run almost every model, and
// gpx_plane.h the one of 2-D models.  Here are the general passes, for models that
// those cannot place (rows_ok) and for single sub-steps (gpx_part), and the host code.
//
// Work mapping of the general passes.  Field arrays are [nx+1][ny+1][kp], z fastest,
// kp floats a row (nz+1, padded), so one x-plane is a contiguous run of (ny+1) kp
// floats.  A block owns `block` consecutive
// points of that plane and marches along x over a chunk of planes; each thread
// owns one (j, k) column.  Every load of a plane is therefore one coalesced
// stream, the x-neighbour is carried in registers from the previous plane (a
// register queue), and the y/z neighbours are the same stream shifted by
// kp or 1 elements and are served by L1/L2.  Blocks are remapped so that
// consecutive plane segments land on the same XCD and share its L2.
//
// Fusion.  The H pass applies, per cell and in the reference order: receiver
// store (old values), main H update, each H-PML slab in slab order, magnetic
// dipoles.  The E pass applies: main E update or dispersive part A, each E-PML
// slab in slab order, voltage sources, Hertzian dipoles, dispersive part B.
// Every correction of a cell is made by the thread that owns it, so no atomics
// are needed and the float32 rounding sequence is the CPU path's.
//
// Rounding.  Built with -ffp-contract=off and IEEE division, every expression
// rounds as written, in the reference's association order, so results are
// comparable bit for bit with a CPU run built the same way.

#include <hip/hip_runtime.h>

#include <limits.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <map>
#include <string>
#include <utility>
#include <algorithm>
#include <vector>

#include "gpx.h"
#include "gpx_step.h"
#include "gpx_rows.h"

namespace gpx {

struct StepArgs {
    int nx, ny, nz;
    int kp, plane;       // floats per row of a field array; (ny+1)*kp
    int nseg, nitems, per_xcd, xc;  // work items: nseg plane segments x x-chunks of xc planes
    float *Ex, *Ey, *Ez, *Hx, *Hy, *Hz;
    const void *ID;      // [6][ntot] of the compact index type
    long long ntot;
    const float *coef;   // [nmat][5]
    const float *R;      // all slabs' R tables for this field, concatenated
    int nR;
    const float *disp;   // [nmat][3P] (real) or [nmat][3P][2] (complex)
    const uint8_t *dispflag;
    TArgs T;             // compacted auxiliary values
    int nmat;
    int form;            // 0 HORIPML, 1 MRIPML
    int nslab;
    SlabArgs slab[MAX_SLABS];
    int flags;
    int it, iterations;
    SrcArgs src0, src1;  // H: src0 magnetic; E: src0 voltage, src1 Hertzian
    int nrx;
    const int *rxc;      // [nrx][3]
    float *rxbuf;        // [6][iterations][nrx]
    // Per x-plane flags: bit 0 a receiver, bit 1 a magnetic source, bit 2 an
    // electric source on the plane; bits 8..13 slabs whose E box holds the
    // plane, bits 16..21 the same for H.
    const uint32_t *planeflag;
    // Cell split.  The interior box [ix0,ix1) x [iy0,iy1) x [iz0,iz1) holds
    // cells with every neighbour inside the grid, every update applying and no
    // PML slab; the interior kernel covers it.  The boundary kernel covers
    // the rest: full planes for x outside [ix0, ix1) (items_a1 items below
    // ix0, items_a2 above), and for x inside, the plane cells of the frame
    // list (plane offsets j*kp+k outside the interior rectangle).
    int box[6];
    int nseg_a, nseg_b, items_a1, items_a2;
    const int *frame;
    int nframe;
};


// Slabs whose box, for one field, contains lane (j, k) in y and z; the x part
// comes per plane from the plane flags.
__device__ __forceinline__ uint32_t lane_slab_mask(const StepArgs &a, int j, int k)
{
    uint32_t m = 0;
    for (int s = 0; s < a.nslab; ++s) {
        const SlabArgs &sl = a.slab[s];
        if (j >= sl.lo[1] && j < sl.hi[1] && k >= sl.lo[2] && k < sl.hi[2]) m |= 1u << s;
    }
    return m;
}


// ---------------------------------------------------------------- work items
struct Cell {
    int xa, xb;   // x range of the item
    int j, k;     // the lane's cell in the plane
    bool live;
};

// Map (item, lane) to an x range and a plane cell; see StepArgs for the split.
template <bool BND>
__device__ __forceinline__ Cell item_cell(const StepArgs &a, int item)
{
    Cell c;
    const int lane = threadIdx.x, B = blockDim.x;
    if (!BND) {
        const int Kin = a.box[5] - a.box[4];
        const int ncell = (a.box[3] - a.box[2]) * Kin;
        const int seg = item % a.nseg, chunk = item / a.nseg;
        const int t = seg * B + lane;
        c.xa = a.box[0] + chunk * a.xc;
        c.xb = min(c.xa + a.xc, a.box[1]);
        c.live = t < ncell;
        const int q = c.live ? t : 0;
        c.j = a.box[2] + q / Kin;
        c.k = a.box[4] + q % Kin;
        return c;
    }
    int t;
    if (item < a.items_a1 + a.items_a2) {
        const bool lower = item < a.items_a1;
        const int r = lower ? item : item - a.items_a1;
        const int seg = r % a.nseg_a, chunk = r / a.nseg_a;
        c.xa = (lower ? 0 : a.box[1]) + chunk * a.xc;
        c.xb = min(c.xa + a.xc, lower ? a.box[0] : a.nx + 1);
        t = seg * B + lane;
        c.live = t < a.plane;
        if (!c.live) t = 0;
    } else {
        const int r = item - a.items_a1 - a.items_a2;
        const int seg = r % a.nseg_b, chunk = r / a.nseg_b;
        c.xa = a.box[0] + chunk * a.xc;
        c.xb = min(c.xa + a.xc, a.box[1]);
        const int q = seg * B + lane;
        c.live = q < a.nframe;
        t = c.live ? a.frame[q] : 0;
    }
    c.j = t / a.kp;
    c.k = t - c.j * a.kp;
    if (c.k > a.nz) {  // padding of the row
        c.live = false;
        c.k = a.nz;
    }
    return c;
}


// ---------------------------------------------------------------- H pass
struct HLoad {
    float ex, ey1, ez1, hx, hy, hz, ezj, exj, eyk, exk;
    uint32_t m3, m4, m5;
};
struct ELoad {
    float hx, hy, hz, ex, ey, ez, hzj, hxj, hyk, hxk;
    uint32_t m0, m1, m2;
    uint32_t s0, s1, s2;   // auxiliary-value slots of the three edges (dispersive models)
};

// update_magnetic (gprMax/fields_updates_ext.pyx:404-412), then each H-PML
// slab in order, then magnetic dipoles; receivers sample the state at the
// start of the iteration.
// The pass bodies run items first, first + stride, ... of the model `a`; `it`
// is the iteration.  k_*_pass hold one model's arguments by value; the
// k_*_pass_many kernels find theirs, one item per block, in a device table of
// several models (a batch of B-scan traces).
template <class IDT, bool BND>
__device__ __forceinline__ void h_pass_run(const StepArgs &a, int first, int stride, int it)
{
    extern __shared__ float4 lds4[];
    __shared__ SlabArgs lslab[MAX_SLABS];
    const int nm = a.nmat;
    const float4 *lc = lds4;
    const float *ls = reinterpret_cast<const float *>(lds4 + nm);
    const float *lR = ls + nm;
    stage_coef(lds4, const_cast<float *>(ls), a.coef, nm);
    if (BND) {
        stage(const_cast<float *>(lR), a.R, a.nR);
        stage_slabs(lslab, a.slab, a.nslab);
    }
    __syncthreads();

    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int NZ1 = a.kp;
    const size_t N = a.ntot;
    const int flags = a.flags;
    const IDT *ID = static_cast<const IDT *>(a.ID);
    const rsrc_t rEx = rsrc(a.Ex), rEy = rsrc(a.Ey), rEz = rsrc(a.Ez);
    const rsrc_t rHx = rsrc(a.Hx), rHy = rsrc(a.Hy), rHz = rsrc(a.Hz);
    const rsrc_t rI3 = rsrc(ID + 3 * N), rI4 = rsrc(ID + 4 * N), rI5 = rsrc(ID + 5 * N);
    const uint32_t P4 = (uint32_t)a.plane * 4u, Pid = (uint32_t)a.plane * (uint32_t)sizeof(IDT);

    for (int item = first; item < a.nitems; item += stride) {
        const Cell c = item_cell<BND>(a, item);
        if (!c.live) continue;
        const int j = c.j, k = c.k;
        const uint32_t off = (uint32_t)(j * NZ1 + k);
        const uint32_t to = off * 4u;
        const uint32_t tid = off * (uint32_t)sizeof(IDT);
        // A neighbour past the grid edge is clamped to the cell itself, which
        // makes the difference exactly +0, the value the reference's loop
        // bounds leave there.  Interior cells always have their neighbours.
        const uint32_t toj = (!BND || j < ny) ? to + 4u * NZ1 : to;
        const uint32_t tok = (!BND || k < nz) ? to + 4u : to;
        const uint32_t jkmask = (BND && (flags & F_PML_ALL)) ? lane_slab_mask(a, j, k) & ((uint32_t)flags >> 4) : 0u;

        // One plane's loads.  The interior variant issues the next plane's
        // loads before computing the current one (its register budget allows
        // two sets in flight); the boundary variant loads as it goes.
        auto load = [&](int ip, HLoad &L) {
            const uint32_t so = (uint32_t)ip * P4;
            const uint32_t sn = (!BND || ip < nx) ? so + P4 : so;  // plane ip+1, or ip itself at the edge
            const uint32_t si = (uint32_t)ip * Pid;
            L.ex = bld(rEx, to, so);
            L.ey1 = bld(rEy, to, sn);
            L.ez1 = bld(rEz, to, sn);
            L.hx = bld(rHx, to, so);
            L.hy = bld(rHy, to, so);
            L.hz = bld(rHz, to, so);
            L.ezj = bld(rEz, toj, so);
            L.exj = bld(rEx, toj, so);
            L.eyk = bld(rEy, tok, so);
            L.exk = bld(rEx, tok, so);
            L.m3 = bld_id<IDT>(rI3, tid, si);
            L.m4 = bld_id<IDT>(rI4, tid, si);
            L.m5 = bld_id<IDT>(rI5, tid, si);
        };
        float ey = bld(rEy, to, (uint32_t)c.xa * P4), ez = bld(rEz, to, (uint32_t)c.xa * P4);
        HLoad cur, nxt;
        if (!BND) load(c.xa, cur);
        for (int i = c.xa; i < c.xb; ++i) {
            const uint32_t so = (uint32_t)i * P4;
            const uint32_t pf = ld(a.planeflag, 4u * (uint32_t)i);
            if (BND) load(i, cur);
            else load(i + 1 < c.xb ? i + 1 : i, nxt);
            PhiPre pre;
            pre.s = -1;
            if (BND) phi_preload(lslab, jkmask & (pf >> PF_SLAB_H), i, j, k, pre);
            const float ex = cur.ex, ey1 = cur.ey1, ez1 = cur.ez1;
            const float hx0 = cur.hx, hy0 = cur.hy, hz0 = cur.hz;
            const float ezj = cur.ezj, exj = cur.exj, eyk = cur.eyk, exk = cur.exk;
            const uint32_t m3 = cur.m3, m4 = cur.m4, m5 = cur.m5;

            // Differences of E used by the H update and the H-PML (forward).
            const float dEz_y = ezj - ez, dEy_z = eyk - ey, dEx_z = exk - ex;
            const float dEz_x = ez1 - ez, dEy_x = ey1 - ey, dEx_y = exj - ex;
            float hx = hx0, hy = hy0, hz = hz0;

            if (flags & F_MAIN) {
                if (!BND || (i >= 1 && j < ny && k < nz)) {
                    const float4 q = lc[m3];
                    hx = q.x * hx - q.z * dEz_y + q.w * dEy_z;
                }
                if (!BND || (i < nx && j >= 1 && k < nz)) {
                    const float4 q = lc[m4];
                    hy = q.x * hy - q.w * dEx_z + q.y * dEz_x;
                }
                if (!BND || (i < nx && j < ny && k >= 1)) {
                    const float4 q = lc[m5];
                    hz = q.x * hz - q.y * dEy_x + q.z * dEx_y;
                }
            }

            if (BND) {
                const uint32_t smask = jkmask & (pf >> PF_SLAB_H);
                if (smask) {
                    for (int s = 0; s < a.nslab; ++s) {
                        if (!(smask & (1u << s))) continue;
                        const SlabArgs &sl = lslab[s];
                        int p;
                        uint32_t q;
                        float a1, b1, a2, b2;
                        phi_get(sl, s, pre, i, j, k, p, q, a1, b1, a2, b2);
                        const float *R = lR + sl.roff;
                        if (sl.axis == 0) {
                            hy = pml_correct_pre(a.form, sl, R, p, hy, true, ls[m4], dEz_x / sl.d, a1, b1, sl.phi1, q, sl.ostep);
                            hz = pml_correct_pre(a.form, sl, R, p, hz, false, ls[m5], dEy_x / sl.d, a2, b2, sl.phi2, q, sl.ostep);
                        } else if (sl.axis == 1) {
                            hx = pml_correct_pre(a.form, sl, R, p, hx, false, ls[m3], dEz_y / sl.d, a1, b1, sl.phi1, q, sl.ostep);
                            hz = pml_correct_pre(a.form, sl, R, p, hz, true, ls[m5], dEx_y / sl.d, a2, b2, sl.phi2, q, sl.ostep);
                        } else {
                            hx = pml_correct_pre(a.form, sl, R, p, hx, true, ls[m3], dEy_z / sl.d, a1, b1, sl.phi1, q, sl.ostep);
                            hy = pml_correct_pre(a.form, sl, R, p, hy, false, ls[m4], dEx_z / sl.d, a2, b2, sl.phi2, q, sl.ostep);
                        }
                    }
                }
            }

            if ((flags & F_SRC) && (pf & PF_SRCH)) {  // magnetic dipoles, gprMax/sources.py:202-232
                for (int s = 0; s < a.src0.n; ++s) {
                    const int *in = a.src0.info + 6 * s;
                    if (in[0] != i || it < in[4] || it > in[5]) continue;
                    if (in[1] == j && in[2] == k) {
                        const int pol = in[3];
                        const uint32_t m = pol == 0 ? m3 : (pol == 1 ? m4 : m5);
                        const float w = a.src0.waves[(size_t)s * a.iterations + it];
                        const float v = ls[m] * w * a.src0.fac[2 * s];
                        if (pol == 0) hx = hx - v;
                        else if (pol == 1) hy = hy - v;
                        else hz = hz - v;
                    }
                }
            }

            if (flags & (F_MAIN | F_PML_ALL | F_SRC)) {
                bst(rHx, to, so, hx);
                bst(rHy, to, so, hy);
                bst(rHz, to, so, hz);
            }

            if ((flags & F_RX) && (pf & PF_RX)) {  // the state at the start of the iteration
                for (int r = 0; r < a.nrx; ++r) {
                    if (a.rxc[3 * r] != i) continue;
                    if (a.rxc[3 * r + 1] == j && a.rxc[3 * r + 2] == k) {
                        float *o = a.rxbuf + (size_t)it * a.nrx + r;
                        const size_t cs = (size_t)a.iterations * a.nrx;
                        o[0] = ex; o[cs] = ey; o[2 * cs] = ez;
                        o[3 * cs] = hx0; o[4 * cs] = hy0; o[5 * cs] = hz0;
                    }
                }
            }
            ey = ey1;
            ez = ez1;
            if (!BND) cur = nxt;
        }
    }
}

template <class IDT, bool BND>
__global__ void k_h_pass(StepArgs a)
{
    h_pass_run<IDT, BND>(a, logical_block(a.per_xcd), gridDim.x, a.it);
}

struct PassMany {
    const int *item0;      // [ntr + 1], first item of each model
    int ntr, nitems, per_xcd, it;
};

__device__ __forceinline__ int model_of(const PassMany &m, int item)
{
    int lo = 0, hi = m.ntr - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (m.item0[mid] <= item) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// `args` is a kernel parameter of its own, read-only and unaliased, so that
// the model's arguments are read with scalar loads as by-value ones are.
template <class IDT, bool BND>
__global__ void k_h_pass_many(const StepArgs *__restrict__ args, PassMany m)
{
    const int item = logical_block(m.per_xcd);
    if (item >= m.nitems) return;
    const int t = model_of(m, item);
    const StepArgs &a = args[t];
    const int local = item - m.item0[t];
    h_pass_run<IDT, BND>(a, local, a.nitems, m.it);
}


// ---------------------------------------------------------------- E pass

// update_electric or dispersive part A (gprMax/fields_updates_ext.pyx:81-107,
// 146-179), each E-PML slab in order, voltage sources, Hertzian dipoles and
// dispersive part B, all on the cell's own thread.
template <class IDT, int P, bool CPLX, bool BND>
__device__ __forceinline__ void e_pass_run(const StepArgs &a, int first, int stride, int it)
{
    extern __shared__ float4 lds4[];
    __shared__ SlabArgs lslab[MAX_SLABS];
    const int nm = a.nmat;
    const int nd = P > 0 ? nm * 3 * P * (CPLX ? 2 : 1) : 0;
    const float4 *lc = lds4;
    const float *ls = reinterpret_cast<const float *>(lds4 + nm);
    const float *lR = ls + nm;
    const float *ldisp = lR + a.nR;
    stage_coef(lds4, const_cast<float *>(ls), a.coef, nm);
    if (BND) {
        stage(const_cast<float *>(lR), a.R, a.nR);
        stage_slabs(lslab, a.slab, a.nslab);
    }
    if (P > 0) stage(const_cast<float *>(ldisp), a.disp, nd);
    __syncthreads();

    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int NZ1 = a.kp;
    const size_t Pl = a.plane, N = a.ntot;
    const int flags = a.flags;
    const IDT *ID = static_cast<const IDT *>(a.ID);
    const rsrc_t rEx = rsrc(a.Ex), rEy = rsrc(a.Ey), rEz = rsrc(a.Ez);
    const rsrc_t rHx = rsrc(a.Hx), rHy = rsrc(a.Hy), rHz = rsrc(a.Hz);
    const rsrc_t rI0 = rsrc(ID), rI1 = rsrc(ID + N), rI2 = rsrc(ID + 2 * N);
    const uint32_t P4 = (uint32_t)Pl * 4u, Pid = (uint32_t)Pl * (uint32_t)sizeof(IDT);

    for (int item = first; item < a.nitems; item += stride) {
        const Cell c = item_cell<BND>(a, item);
        if (!c.live) continue;
        const int j = c.j, k = c.k;
        const uint32_t off = (uint32_t)(j * NZ1 + k);
        const uint32_t to = off * 4u;
        const uint32_t tid = off * (uint32_t)sizeof(IDT);
        const uint32_t toj = (!BND || j >= 1) ? to - 4u * NZ1 : to;
        const uint32_t tok = (!BND || k >= 1) ? to - 4u : to;
        const uint32_t jkmask = (BND && (flags & F_PML_ALL)) ? lane_slab_mask(a, j, k) & ((uint32_t)flags >> 4) : 0u;

        // Hy, Hz of plane i-1 (the plane itself at i = 0, giving a +0 difference)
        const uint32_t sm = (uint32_t)(c.xa >= 1 ? c.xa - 1 : c.xa) * P4;
        float hy_m = bld(rHy, to, sm), hz_m = bld(rHz, to, sm);
        auto load = [&](int ip, ELoad &L) {
            const uint32_t so = (uint32_t)ip * P4, si = (uint32_t)ip * Pid;
            L.hx = bld(rHx, to, so);
            L.hy = bld(rHy, to, so);
            L.hz = bld(rHz, to, so);
            L.ex = bld(rEx, to, so);
            L.ey = bld(rEy, to, so);
            L.ez = bld(rEz, to, so);
            L.hzj = bld(rHz, toj, so);
            L.hxj = bld(rHx, toj, so);
            L.hyk = bld(rHy, tok, so);
            L.hxk = bld(rHx, tok, so);
            L.m0 = bld_id<IDT>(rI0, tid, si);
            L.m1 = bld_id<IDT>(rI1, tid, si);
            L.m2 = bld_id<IDT>(rI2, tid, si);
            if (P > 0 && (flags & (F_MAIN | F_DISPB))) {
                const size_t pe = (size_t)ip * Pl;
                L.s0 = ld(a.T.slot[0] + pe, to);
                L.s1 = ld(a.T.slot[1] + pe, to);
                L.s2 = ld(a.T.slot[2] + pe, to);
            }
        };
        ELoad cur, nxt;
        if (!BND && P == 0) load(c.xa, cur);
        for (int i = c.xa; i < c.xb; ++i) {
            const uint32_t so = (uint32_t)i * P4;
            const size_t po = (size_t)i * Pl;
            const uint32_t pf = ld(a.planeflag, 4u * (uint32_t)i);
            if (BND || P > 0) load(i, cur);
            else load(i + 1 < c.xb ? i + 1 : i, nxt);
            PhiPre pre;
            pre.s = -1;
            if (BND) phi_preload(lslab, jkmask & (pf >> PF_SLAB_E), i, j, k, pre);
            const float hx = cur.hx, hy = cur.hy, hz = cur.hz;
            float ex = cur.ex, ey = cur.ey, ez = cur.ez;
            const float hzj = cur.hzj, hxj = cur.hxj, hyk = cur.hyk, hxk = cur.hxk;
            const uint32_t m0 = cur.m0, m1 = cur.m1, m2 = cur.m2;
            const bool rx_ = !BND || (i < nx && j >= 1 && j < ny && k >= 1 && k < nz);
            const bool ry_ = !BND || (i >= 1 && i < nx && j < ny && k >= 1 && k < nz);
            const bool rz_ = !BND || (i >= 1 && i < nx && j >= 1 && j < ny && k < nz);
            // Auxiliary values change only on edges of materials with poles,
            // so only those edges read and write them.  Such an edge has a
            // slot (T_NOSLOT otherwise): the slots load with the plane, not
            // after the indices, so the auxiliary values follow one round
            // trip later instead of two.
            const bool td = P > 0 && (flags & (F_MAIN | F_DISPB));
            const uint32_t sx = td ? cur.s0 : T_NOSLOT, sy = td ? cur.s1 : T_NOSLOT, sz = td ? cur.s2 : T_NOSLOT;
            const bool dx_ = P > 0 && rx_ && sx != T_NOSLOT;
            const bool dy_ = P > 0 && ry_ && sy != T_NOSLOT;
            const bool dz_ = P > 0 && rz_ && sz != T_NOSLOT;
            float txr[P > 0 ? P : 1], txi[P > 0 ? P : 1];
            float tyr[P > 0 ? P : 1], tyi[P > 0 ? P : 1];
            float tzr[P > 0 ? P : 1], tzi[P > 0 ? P : 1];
            if (td) {
                if (dx_) t_load_at<P, CPLX>(a.T, 0, sx, txr, txi);
                if (dy_) t_load_at<P, CPLX>(a.T, 1, sy, tyr, tyi);
                if (dz_) t_load_at<P, CPLX>(a.T, 2, sz, tzr, tzi);
            }
            // Differences of H used by the E update and the E-PML (backward).
            const float dHz_y = hz - hzj, dHy_z = hy - hyk, dHx_z = hx - hxk;
            const float dHz_x = hz - hz_m, dHy_x = hy - hy_m, dHx_y = hx - hxj;

            if (flags & F_MAIN) {
                if (rx_) {
                    const float4 q = lc[m0];
                    float v = q.x * ex + q.z * dHz_y - q.w * dHy_z;
                    if (P > 0) {
                        const float phi = dx_ ? disp_a<P, CPLX>(ldisp, m0, txr, txi, ex) : 0.f;
                        v = v - ls[m0] * phi;
                    }
                    ex = v;
                }
                if (ry_) {
                    const float4 q = lc[m1];
                    float v = q.x * ey + q.w * dHx_z - q.y * dHz_x;
                    if (P > 0) {
                        const float phi = dy_ ? disp_a<P, CPLX>(ldisp, m1, tyr, tyi, ey) : 0.f;
                        v = v - ls[m1] * phi;
                    }
                    ey = v;
                }
                if (rz_) {
                    const float4 q = lc[m2];
                    float v = q.x * ez + q.y * dHy_x - q.z * dHx_y;
                    if (P > 0) {
                        const float phi = dz_ ? disp_a<P, CPLX>(ldisp, m2, tzr, tzi, ez) : 0.f;
                        v = v - ls[m2] * phi;
                    }
                    ez = v;
                }
            }

            if (BND) {
                const uint32_t smask = jkmask & (pf >> PF_SLAB_E);
                if (smask) {
                    for (int s = 0; s < a.nslab; ++s) {
                        if (!(smask & (1u << s))) continue;
                        const SlabArgs &sl = lslab[s];
                        int p;
                        uint32_t q;
                        float a1, b1, a2, b2;
                        phi_get(sl, s, pre, i, j, k, p, q, a1, b1, a2, b2);
                        const float *R = lR + sl.roff;
                        if (sl.axis == 0) {
                            ey = pml_correct_pre(a.form, sl, R, p, ey, false, ls[m1], dHz_x / sl.d, a1, b1, sl.phi1, q, sl.ostep);
                            ez = pml_correct_pre(a.form, sl, R, p, ez, true, ls[m2], dHy_x / sl.d, a2, b2, sl.phi2, q, sl.ostep);
                        } else if (sl.axis == 1) {
                            ex = pml_correct_pre(a.form, sl, R, p, ex, true, ls[m0], dHz_y / sl.d, a1, b1, sl.phi1, q, sl.ostep);
                            ez = pml_correct_pre(a.form, sl, R, p, ez, false, ls[m2], dHx_y / sl.d, a2, b2, sl.phi2, q, sl.ostep);
                        } else {
                            ex = pml_correct_pre(a.form, sl, R, p, ex, false, ls[m0], dHy_z / sl.d, a1, b1, sl.phi1, q, sl.ostep);
                            ey = pml_correct_pre(a.form, sl, R, p, ey, true, ls[m1], dHx_z / sl.d, a2, b2, sl.phi2, q, sl.ostep);
                        }
                    }
                }
            }

            if ((flags & F_SRC) && (pf & PF_SRCE)) {
                // Voltage sources, then Hertzian dipoles (gprMax/model_build_run.py:458-461).
                for (int s = 0; s < a.src0.n; ++s) {  // gprMax/sources.py:81-120
                    const int *in = a.src0.info + 6 * s;
                    if (in[0] != i || it < in[4] || it > in[5]) continue;
                    if (in[1] == j && in[2] == k) {
                        const int pol = in[3] & 3;
                        const bool hard = in[3] >= 4;
                        const uint32_t m = pol == 0 ? m0 : (pol == 1 ? m1 : m2);
                        const float w = a.src0.waves[(size_t)s * a.iterations + it];
                        float *F = pol == 0 ? &ex : (pol == 1 ? &ey : &ez);
                        if (hard) *F = -w / a.src0.fac[2 * s];
                        else *F = *F - ls[m] * w * a.src0.fac[2 * s];
                    }
                }
                for (int s = 0; s < a.src1.n; ++s) {  // gprMax/sources.py:163-193
                    const int *in = a.src1.info + 6 * s;
                    if (in[0] != i || it < in[4] || it > in[5]) continue;
                    if (in[1] == j && in[2] == k) {
                        const int pol = in[3];
                        const uint32_t m = pol == 0 ? m0 : (pol == 1 ? m1 : m2);
                        const float w = a.src1.waves[(size_t)s * a.iterations + it];
                        const float v = ls[m] * w * a.src1.fac[2 * s] * a.src1.fac[2 * s + 1];
                        if (pol == 0) ex = ex - v;
                        else if (pol == 1) ey = ey - v;
                        else ez = ez - v;
                    }
                }
            }

            if (P > 0 && (flags & F_DISPB)) {
                if (dx_) disp_b<P, CPLX>(ldisp, m0, txr, txi, ex);
                if (dy_) disp_b<P, CPLX>(ldisp, m1, tyr, tyi, ey);
                if (dz_) disp_b<P, CPLX>(ldisp, m2, tzr, tzi, ez);
            }
            if (P > 0 && (flags & (F_MAIN | F_DISPB))) {
                if (dx_) t_store<P, CPLX>(a.T, 0, sx, txr, txi);
                if (dy_) t_store<P, CPLX>(a.T, 1, sy, tyr, tyi);
                if (dz_) t_store<P, CPLX>(a.T, 2, sz, tzr, tzi);
            }
            if (flags & (F_MAIN | F_PML_ALL | F_SRC)) {
                bst(rEx, to, so, ex);
                bst(rEy, to, so, ey);
                bst(rEz, to, so, ez);
            }
            hy_m = hy;
            hz_m = hz;
            if (!BND && P == 0) cur = nxt;
        }
    }
}

template <class IDT, int P, bool CPLX, bool BND>
__global__ void k_e_pass(StepArgs a)
{
    e_pass_run<IDT, P, CPLX, BND>(a, logical_block(a.per_xcd), gridDim.x, a.it);
}

template <class IDT, int P, bool CPLX, bool BND>
__global__ void k_e_pass_many(const StepArgs *__restrict__ args, PassMany m)
{
    const int item = logical_block(m.per_xcd);
    if (item >= m.nitems) return;
    const int t = model_of(m, item);
    const StepArgs &a = args[t];
    const int local = item - m.item0[t];
    e_pass_run<IDT, P, CPLX, BND>(a, local, a.nitems, m.it);
}


// ---------------------------------------------------------------- snapshots
// Cell averages of gprMax/snapshots_ext.pyx:58-71 over the slices of
// gprMax/snapshots.py:78-80; one thread per output cell.
__global__ void k_snapshot(int ny, int kp, int xs, int ys, int zs, int sdx, int sdy, int sdz,
                           int snx, int sny, int snz, const float *Ex, const float *Ey,
                           const float *Ez, const float *Hx, const float *Hy, const float *Hz,
                           float *out)
{
    const long long n = (long long)snx * sny * snz;
    const long long o = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n) return;
    const int k = (int)(o % snz);
    const int j = (int)((o / snz) % sny);
    const int i = (int)(o / ((long long)snz * sny));
    const long long NY1 = ny + 1, NZ1 = kp;
    auto at = [&](int a, int b, int c) {
        return ((long long)(xs + a * sdx) * NY1 + (ys + b * sdy)) * NZ1 + (zs + c * sdz);
    };
    out[o] = (Ex[at(i, j, k)] + Ex[at(i, j + 1, k)] + Ex[at(i, j, k + 1)] + Ex[at(i, j + 1, k + 1)]) / 4.0f;
    out[n + o] = (Ey[at(i, j, k)] + Ey[at(i + 1, j, k)] + Ey[at(i, j, k + 1)] + Ey[at(i + 1, j, k + 1)]) / 4.0f;
    out[2 * n + o] = (Ez[at(i, j, k)] + Ez[at(i + 1, j, k)] + Ez[at(i, j + 1, k)] + Ez[at(i + 1, j + 1, k)]) / 4.0f;
    out[3 * n + o] = (Hx[at(i, j, k)] + Hx[at(i + 1, j, k)]) / 2.0f;
    out[4 * n + o] = (Hy[at(i, j, k)] + Hy[at(i, j + 1, k)]) / 2.0f;
    out[5 * n + o] = (Hz[at(i, j, k)] + Hz[at(i, j, k + 1)]) / 2.0f;
}


// ---------------------------------------------------------------- transmission lines
// A one-dimensional line attached to the E edge at (i, j, k)
// (gprMax/sources.py:286-451).  Line arithmetic follows NumPy 2 promotion
// of the reference's expressions: the line coefficients are float64
// scalars, so each update is a float64 product on float32 differences,
// rounded to float32 when stored; the cell sizes of the current loop and of
// the E assignment are Python floats, so those are float32 operations.
struct TLDev {
    int i, j, k, pol, first, last, nl, srcpos, antpos;
    double cV, cI, cW, h;   // R (c dt / dl), (1/R)(c dt / dl), c dt / dl, ABC factor
    float dpol, da, db;     // cell size along pol; the two sizes of the current loop
    float *V, *I, *abc;     // line voltage [nl], current [nl], ABC memory (abcv0, abcv1)
    const float *whole, *half;  // waveform on whole and half steps [iterations]
    float *vt, *itot;       // voltage and current at the antenna end per iteration
};

// After the H pass: the line state at the start of the iteration goes to the
// outputs (gprMax/fields_outputs.py:65-67); in the active window the line
// current is updated and its antenna end takes the current of the H loop
// around the edge (update_magnetic, gprMax/sources.py:428-451, and
// Ix/Iy/Iz, gprMax/grid.py:413-461).  One thread per line.
__global__ void k_tl_h(const TLDev *tl, int n, int it, int ny, int kp, const float *Hx, const float *Hy,
                       const float *Hz)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const TLDev &L = tl[s];
    L.vt[it] = L.V[L.antpos];
    L.itot[it] = L.I[L.antpos];
    if (it < L.first || it > L.last) return;
    for (int m = 0; m + 1 < L.nl; ++m) {
        const float d = L.V[m + 1] - L.V[m];
        L.I[m] = (float)((double)L.I[m] - L.cI * (double)d);
    }
    L.I[L.srcpos - 1] = (float)((double)L.I[L.srcpos - 1] + L.cI * (double)L.half[it]);
    const long long NY1 = ny + 1, NZ1 = kp;
    auto at = [&](int a, int b, int c) { return ((long long)a * NY1 + b) * NZ1 + c; };
    const int x = L.i, y = L.j, z = L.k;
    float cur = 0.f;
    if (L.pol == 0) {
        if (y != 0 && z != 0)
            cur = L.da * (Hy[at(x, y, z - 1)] - Hy[at(x, y, z)]) + L.db * (Hz[at(x, y, z)] - Hz[at(x, y - 1, z)]);
    } else if (L.pol == 1) {
        if (x != 0 && z != 0)
            cur = L.da * (Hx[at(x, y, z)] - Hx[at(x, y, z - 1)]) + L.db * (Hz[at(x - 1, y, z)] - Hz[at(x, y, z)]);
    } else {
        if (x != 0 && y != 0)
            cur = L.da * (Hx[at(x, y - 1, z)] - Hx[at(x, y, z)]) + L.db * (Hy[at(x, y, z)] - Hy[at(x - 1, y, z)]);
    }
    L.I[L.antpos] = cur;
}

// After the E pass, in the active window: line voltage, the one-way
// injector, the absorbing end, then the edge's E from the antenna voltage
// (update_electric, gprMax/sources.py:361-426).
__global__ void k_tl_e(const TLDev *tl, int n, int it, int ny, int kp, float *Ex, float *Ey, float *Ez)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const TLDev &L = tl[s];
    if (it < L.first || it > L.last) return;
    for (int m = L.nl - 1; m >= 1; --m) {
        const float d = L.I[m] - L.I[m - 1];
        L.V[m] = (float)((double)L.V[m] - L.cV * (double)d);
    }
    L.V[L.srcpos] = (float)((double)L.V[L.srcpos] + L.cW * (double)L.whole[it]);
    const float a0 = L.abc[0], a1 = L.abc[1];
    L.V[0] = (float)(L.h * (double)(L.V[1] - a0) + (double)a1);
    L.abc[0] = L.V[0];
    L.abc[1] = L.V[1];
    const long long at = ((long long)L.i * (ny + 1) + L.j) * kp + L.k;
    float *E = L.pol == 0 ? Ex : (L.pol == 1 ? Ey : Ez);
    E[at] = -L.V[L.antpos] / L.dpol;
}

}  // namespace gpx

using namespace gpx;

// ====================================================================== ctx
struct Slab {
    int dir, xs, xf, ys, yf, zs, zf, order, t, roff = 0;
    float d;
    long long dims[4][3];  // reference shapes of EPhi1, EPhi2, HPhi1, HPhi2, without the order axis
    // Phi on the device: all slabs of a field in one array, per order and term
    // (1, 2) the slabs one after the other, each [ni][nj][nkp] in ascending
    // cell order (the reference runs the profile axis of the minus slabs
    // backwards), rows padded so that cell k sits at k mod 4 as in the fields.
    long long base = -1;   // of the slab within a block of one order and term (-1: not laid out yet)
    int ni, nj, nkp;
    std::vector<float> R[2];  // E, H profile tables RA, RB, RE, RF, each [order][t]
};

struct Snap {
    int xs, ys, zs, dx, dy, dz, snx, sny, snz, time;
    float *out = nullptr;  // [6][snx][sny][snz]
};

struct TLine {
    TLDev d;                // device pointers into `mem`
    float *mem = nullptr;   // V, I, abc, whole, half, vt, itot
};

struct SrcSet {
    int n = 0;
    std::vector<int> host;  // info rows, for the plane flags
    int *info = nullptr;
    float *fac = nullptr, *waves = nullptr;
};

struct gpx_ctx {
    gpx_desc desc;
    long long ntot = 0;
    int kp = 0, plane = 0;    // floats per field row (nz + 1, padded: see gpx_create); (ny + 1) kp
    hipStream_t stream = nullptr;
    // The state: fields and H Phi, twice for the kernels that write the next state
    // beside the current one (the one-launch step and the 2-D kernel; the second copy
    // is allocated when one first runs), `cur` the current one; E Phi twice for the
    // 2-D kernel.  ntot counts padded points.
    float *Fmem[2] = {nullptr, nullptr};    // 6 x fstride floats: Ex, Ey, Ez, Hx, Hy, Hz
    float *phiH[2] = {nullptr, nullptr}, *phiE[2] = {nullptr, nullptr};
    int cur = 0, curE = 0;    // current copy of the fields and H Phi, of E Phi
    float *field(int c) const { return Fmem[cur] + c * fstride; }
    long long np = 0;         // floats of one (order, term) block of Phi
    int phi_orders = 0;       // orders the Phi arrays hold
    bool phi_dirty = false;   // slabs were added since the Phi arrays were laid out
    size_t next_bytes = 0;    // bytes of the second state and of the second Phi
    long long fstride = 0;    // floats between components: ntot rounded up to 64, and a row more
    uint16_t *ID = nullptr;   // [6][ntot] (nmat < 2^16, see gpx_create)
    std::vector<float> hostE, hostH, hostdisp;  // coefficients and pole tables, for the row kernels' tables
    float *img = nullptr;     // those tables (row_stage), nimg floats
    int nimg = 0;
    RowModel *row = nullptr;  // the model as the row kernels see it
    RowModel rowh;            // its host copy
    bool state_given = false; // fields or Phi have been uploaded, or see note_state
    bool row_dirty = true;    // something in it changed
    bool planes_dirty = true; // slabs, sources or receivers changed since the planes' flags went up
    bool hu = false;          // every material has the same H coefficients
    int row_block = 0;        // threads per block of the one-launch step
    float *cE = nullptr, *cH = nullptr;
    float *Rall[2] = {nullptr, nullptr};  // E, H: all slabs' R tables back to back
    std::vector<float> Rhost[2];
    int disp_complex = 0;
    float *disp = nullptr;    // real [nmat][3P] or complex [nmat][3P][2]
    uint8_t *dispflag = nullptr;
    float *T[3] = {nullptr, nullptr, nullptr};  // compacted: [P][tn[c]] (x2 complex)
    uint32_t *tslot[3] = {nullptr, nullptr, nullptr};  // [ntot]: place of an edge with poles
    uint32_t *tmasks = nullptr;      // the same as the row passes read it
    long long tn[3] = {0, 0, 0};     // edges with poles per component
    bool tslot_dirty = true;         // ID or dispersive tables changed since the slots were built
    bool have_id = false, have_coeffs = false, have_disp = false;
    std::vector<Slab> slabs;
    SrcSet src[3];
    int nrx = 0;
    std::vector<int> rxhost;
    int *rxc = nullptr;
    float *rxbuf = nullptr;
    std::vector<Snap> snaps;
    std::vector<TLine> tls;          // transmission lines
    TLDev *tldev = nullptr;          // device copy of their descriptions
    uint32_t *planeflag = nullptr;  // [2][nx+1]: slab bits by slab, by direction
    StepRare *rare = nullptr;        // device copy of the source/receiver tables of the row kernels
    bool rare_dirty = true;
    int box[6] = {0, 0, 0, 0, 0, 0}; // interior box (see StepArgs)
    int *frame = nullptr;            // plane offsets outside the interior rectangle
    int nframe = 0;
    bool deep = false;               // the interior box has at least two cells on every axis
    int xchunk = 0, block = 0;
    int fused = 4;                   // step form, see gpx_set_step
    int choice = -1;                 // form 4, as reported: -1 open, 4 form 6, 5 form 7
    hipStream_t stream2 = nullptr;   // second stream of form 2
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    int tile_cells = 0;              // cells per block of the one-launch step (0 = auto)
    int cus = 0;                     // compute units of the device
    mutable std::map<std::pair<const void *, size_t>, int> occupancy;
    float *stage = nullptr;          // dense values on their way between the host and padded rows
    size_t nstage = 0;               // its floats, at most STAGE_FLOATS
    size_t bytes = 0;
    std::string err;
};
constexpr size_t STAGE_FLOATS = (size_t)8 << 20;

// Of the last failure without a context, per thread: models are made on several at a time.
static thread_local std::string g_err;
static int update_planeflags(gpx_ctx *ctx);
static int ensure_planes(gpx_ctx *ctx);

#define GPX_TRY(call)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) return fail_hip(ctx, e_, #call);                                 \
    } while (0)

static int fail(gpx_ctx *ctx, int code, const std::string &msg)
{
    if (ctx) ctx->err = msg;
    else g_err = msg;
    return code;
}

static int fail_hip(gpx_ctx *ctx, hipError_t e, const char *what)
{
    std::string msg = std::string(what) + ": " + hipGetErrorString(e);
    return fail(ctx, (int)e, msg);
}

static hipError_t dalloc(gpx_ctx *ctx, void **p, size_t bytes, bool zero = true)
{
    hipError_t e = hipMalloc(p, bytes ? bytes : 4);
    if (e != hipSuccess) return e;
    ctx->bytes += bytes;
    if (zero) e = hipMemsetAsync(*p, 0, bytes ? bytes : 4, ctx->stream);
    return e;
}

extern "C" const char *gpx_last_error(const gpx_ctx *ctx)
{
    return ctx ? ctx->err.c_str() : g_err.c_str();
}

// Whether a whole state of so many points a component passes 32-bit byte offsets
// (the indices, half as many bytes, then may not).
static bool past_offsets(double points) { return points * 24.0 >= 4294967295.0; }

extern "C" int gpx_create(const gpx_desc *d, gpx_ctx **out)
{
    gpx_ctx *ctx = nullptr;
    if (!d || !out) return fail(nullptr, GPX_EARG, "gpx_create: null argument");
    *out = nullptr;
    // One axis of one cell is a 2-D model (TMx, TMy, TMz).  The 3-D update
    // ranges then give the results of the reference's 2-D branches
    // (gprMax/fields_updates_ext.pyx:55-77, 376-400): the E components the
    // 2-D branch skips have empty 3-D ranges, and the H cells only the 3-D
    // ranges add lie on outer faces whose E never leaves zero.
    if (d->nx < 1 || d->ny < 1 || d->nz < 1 || (d->nx == 1) + (d->ny == 1) + (d->nz == 1) > 1)
        return fail(nullptr, GPX_EARG, "gpx_create: a grid needs at least 2 cells on two axes and 1 on the third");
    if (d->iterations < 1 || d->nmat < 1)
        return fail(nullptr, GPX_EARG, "gpx_create: iterations and nmat must be positive");
    if (d->maxpoles < 0 || d->maxpoles > MAX_POLES)
        return fail(nullptr, GPX_ELIMIT, "gpx_create: at most " + std::to_string(MAX_POLES) + " dispersive poles are supported");
    if (d->pml_formulation != 0 && d->pml_formulation != 1)
        return fail(nullptr, GPX_EARG, "gpx_create: pml_formulation must be 0 (HORIPML) or 1 (MRIPML)");
    {
        // The kernels address a field array with 32-bit byte offsets (buffer
        // instructions: plane offset plus lane offset), so a component may
        // hold at most 2^30 - 1 points; larger grids are refused here rather
        // than wrapping.
        const unsigned long long pts = (unsigned long long)(d->nx + 1) * (d->ny + 1) * (d->nz + 1);
        if (pts * 4ull > 0xFFFFFFFFull)
            return fail(nullptr, GPX_ELIMIT,
                        "gpx_create: " + std::to_string(pts) + " points per field component exceed the limit of " +
                            std::to_string(0xFFFFFFFFull / 4) + " (32-bit byte offsets)");
    }
    size_t lds = (size_t)d->nmat * 5 * 4 + (size_t)d->nmat * 3 * d->maxpoles * 2 * 4 + d->nmat;
    if (lds > (size_t)MAX_LDS_BYTES)
        return fail(nullptr, GPX_ELIMIT, "gpx_create: too many materials for the LDS coefficient table");
    hipError_t e = hipSetDevice(d->device);
    if (e != hipSuccess) return fail(nullptr, (int)e, std::string("hipSetDevice: ") + hipGetErrorString(e));
    ctx = new gpx_ctx();
    ctx->desc = *d;
    {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, d->device);
        if (e != hipSuccess) {
            delete ctx;
            return fail(nullptr, (int)e, std::string("hipGetDeviceProperties: ") + hipGetErrorString(e));
        }
        ctx->cus = prop.multiProcessorCount;
    }
    // Rows padded to four floats, so that the row kernels load and store whole
    // lanes.  Not rows of two floats, a 2-D model's, which are a lane as they are
    // and would be twice as long (1500x1500 with a pole, us an iteration: 134
    // padded, 68 not); nor where the row kernels cannot run the model: past the
    // 32-bit offsets by the padding alone, or with poles by the whole state.
    ctx->kp = d->nz == 1 ? 2 : (d->nz + 1 + 3) / 4 * 4;
    {
        const double points = (double)(d->nx + 1) * (d->ny + 1) * ctx->kp;
        if (points * 4.0 > 4294967295.0 || (d->maxpoles > 0 && past_offsets(points + 128))) ctx->kp = d->nz + 1;
    }
    ctx->plane = (d->ny + 1) * ctx->kp;
    ctx->ntot = (long long)(d->nx + 1) * ctx->plane;
    e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        int rc = fail(nullptr, (int)e, std::string("hipStreamCreate: ") + hipGetErrorString(e));
        delete ctx;
        return rc;
    }
    ctx->fstride = (ctx->ntot + 16 + 63) / 64 * 64;
    e = dalloc(ctx, (void **)&ctx->Fmem[0], (size_t)6 * ctx->fstride * 4);
    if (e != hipSuccess) goto fail_alloc;
    // The coefficient tables must fit LDS (as the reference's must fit 64 KB
    // of constant memory, gprMax/model_build_run.py:512-516), which bounds
    // nmat far below 2^16: every material index fits 16 bits.
    e = dalloc(ctx, (void **)&ctx->ID, (6 * (size_t)ctx->ntot + 16) * 2, false);
    if (e != hipSuccess) goto fail_alloc;
    e = dalloc(ctx, (void **)&ctx->cE, (size_t)d->nmat * 5 * 4);
    if (e != hipSuccess) goto fail_alloc;
    e = dalloc(ctx, (void **)&ctx->cH, (size_t)d->nmat * 5 * 4);
    if (e != hipSuccess) goto fail_alloc;
    e = dalloc(ctx, (void **)&ctx->planeflag, (size_t)(d->nx + 1) * 8);
    if (e != hipSuccess) goto fail_alloc;
    if (int rc = update_planeflags(ctx)) {
        gpx_destroy(ctx);
        return fail(nullptr, rc, "gpx_create: layout set-up failed");
    }
    *out = ctx;
    return 0;
fail_alloc : {
    int rc = fail(nullptr, (int)e, std::string("hipMalloc: ") + hipGetErrorString(e));
    gpx_destroy(ctx);
    return rc;
}
}

extern "C" int gpx_destroy(gpx_ctx *ctx)
{
    if (!ctx) return 0;
    hipSetDevice(ctx->desc.device);
    if (ctx->stream) hipStreamSynchronize(ctx->stream);
    for (auto &p : ctx->Fmem) if (p) hipFree(p);
    for (auto &p : ctx->T) if (p) hipFree(p);
    for (auto &p : ctx->tslot) if (p) hipFree(p);
    if (ctx->tmasks) hipFree(ctx->tmasks);
    if (ctx->ID) hipFree(ctx->ID);
    if (ctx->cE) hipFree(ctx->cE);
    if (ctx->cH) hipFree(ctx->cH);
    for (auto &p : ctx->Rall) if (p) hipFree(p);
    if (ctx->disp) hipFree(ctx->disp);
    if (ctx->dispflag) hipFree(ctx->dispflag);
    for (auto &p : ctx->phiH) if (p) hipFree(p);
    for (float *m : ctx->phiE)
        if (m) hipFree(m);
    if (ctx->img) hipFree(ctx->img);
    if (ctx->stage) hipFree(ctx->stage);
    if (ctx->row) hipFree(ctx->row);
    for (auto &s : ctx->src) {
        if (s.info) hipFree(s.info);
        if (s.fac) hipFree(s.fac);
        if (s.waves) hipFree(s.waves);
    }
    if (ctx->rxc) hipFree(ctx->rxc);
    if (ctx->rxbuf) hipFree(ctx->rxbuf);
    if (ctx->planeflag) hipFree(ctx->planeflag);
    if (ctx->rare) hipFree(ctx->rare);
    if (ctx->frame) hipFree(ctx->frame);
    for (auto &s : ctx->snaps) if (s.out) hipFree(s.out);
    for (auto &t : ctx->tls) if (t.mem) hipFree(t.mem);
    if (ctx->tldev) hipFree(ctx->tldev);
    if (ctx->stream2) hipStreamSynchronize(ctx->stream2);
    if (ctx->ev_fork) hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_join) hipEventDestroy(ctx->ev_join);
    if (ctx->stream2) hipStreamDestroy(ctx->stream2);
    if (ctx->stream) hipStreamDestroy(ctx->stream);
    delete ctx;
    return 0;
}

static int copy_in(gpx_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    GPX_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    GPX_TRY(hipStreamSynchronize(ctx->stream));
    return 0;
}

static int copy_out(gpx_ctx *ctx, void *dst, const void *src, size_t bytes)
{
    GPX_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    GPX_TRY(hipStreamSynchronize(ctx->stream));
    return 0;
}

// ---------------------------------------------------------------- Phi arrays
static size_t phi_bytes(const gpx_ctx *ctx) { return (size_t)ctx->phi_orders * 2 * ctx->np * 4 + 16; }

// Several arrays, all of them or none.
static int dalloc_all(gpx_ctx *ctx, int n, float **p, const size_t *bytes, bool zero)
{
    for (int q = 0; q < n; ++q) p[q] = nullptr;
    for (int q = 0; q < n; ++q) {
        const hipError_t e = dalloc(ctx, (void **)&p[q], bytes[q], zero);
        if (e == hipSuccess) continue;
        for (int f = 0; f <= q; ++f) {
            if (!p[f]) continue;
            hipFree(p[f]);
            ctx->bytes -= bytes[f];
            p[f] = nullptr;
        }
        return fail_hip(ctx, e, "hipMalloc");
    }
    return 0;
}

// Lays the Phi arrays out once slabs are there; slabs added later keep the
// values of the ones before.
static int ensure_phi(gpx_ctx *ctx)
{
    if (!ctx->phi_dirty) return 0;
    hipSetDevice(ctx->desc.device);
    long long np = 0;
    int orders = 0;
    std::vector<long long> base;
    for (const Slab &S : ctx->slabs) {
        base.push_back(np);
        np += (long long)S.ni * S.nj * S.nkp;
        if (S.order > orders) orders = S.order;
    }
    const size_t nb = (size_t)orders * 2 * np * 4 + 16, bytes[3] = {nb, nb, nb};
    const bool two = ctx->Fmem[1] != nullptr;
    float *p[3];   // E, H and H of the second state
    if (int rc = dalloc_all(ctx, two ? 3 : 2, p, bytes, true)) return rc;
    if (ctx->phiE[ctx->curE]) {  // values of the slabs that were there, laid out the same in themselves
        for (size_t s = 0; s < ctx->slabs.size() && ctx->slabs[s].base >= 0; ++s) {
            const Slab &S = ctx->slabs[s];
            for (int q = 0; q < 2 * S.order; ++q)
                for (int f = 0; f < (two ? 3 : 2); ++f) {
                    const float *old = (f ? ctx->phiH[ctx->cur] : ctx->phiE[ctx->curE]) + (size_t)q * ctx->np + S.base;
                    GPX_TRY(hipMemcpyAsync(p[f] + (size_t)q * np + base[s], old, (size_t)S.ni * S.nj * S.nkp * 4,
                                           hipMemcpyDeviceToDevice, ctx->stream));
                }
        }
        GPX_TRY(hipStreamSynchronize(ctx->stream));
        const int next = (ctx->phiH[1] != nullptr) + (ctx->phiE[1] != nullptr);
        ctx->bytes -= phi_bytes(ctx) * (2 + next);
        ctx->next_bytes -= phi_bytes(ctx) * next;
        for (float **q : {&ctx->phiE[0], &ctx->phiE[1], &ctx->phiH[0], &ctx->phiH[1]}) {
            if (*q) hipFree(*q);
            *q = nullptr;
        }
    }
    ctx->np = np;
    ctx->phi_orders = orders;
    for (size_t s = 0; s < base.size(); ++s) ctx->slabs[s].base = base[s];
    ctx->curE = 0;
    ctx->phiE[0] = p[0];
    ctx->phiH[0] = p[1];
    if (two) {
        ctx->phiH[1] = p[2];
        ctx->next_bytes += nb;
    }
    ctx->phi_dirty = false;
    ctx->row_dirty = true;
    return 0;
}

// ---------------------------------------------------------------- second state
// The one-launch step writes the next state, fields and H Phi, into second
// copies.  They are made on first use, equal to the current ones, so a model
// that only ever updates in place (dispersive models, models with
// transmission lines) holds one state.
static int ensure_next_state(gpx_ctx *ctx)
{
    if (ctx->Fmem[1]) return 0;
    // Without a second state the current one is Fmem[0].
    const size_t bytes[2] = {(size_t)6 * ctx->fstride * 4, phi_bytes(ctx)};
    const int n = ctx->phiH[0] ? 2 : 1;
    float *p[2];
    if (int rc = dalloc_all(ctx, n, p, bytes, false)) return rc;
    ctx->Fmem[1] = p[0];
    ctx->next_bytes += bytes[0];
    if (n == 2) {
        ctx->phiH[1] = p[1];
        ctx->next_bytes += bytes[1];
    }
    ctx->row_dirty = true;
    GPX_TRY(hipMemcpyAsync(p[0], ctx->Fmem[0], bytes[0], hipMemcpyDeviceToDevice, ctx->stream));
    if (n == 2) GPX_TRY(hipMemcpyAsync(p[1], ctx->phiH[0], bytes[1], hipMemcpyDeviceToDevice, ctx->stream));
    return 0;
}

// The 2-D kernel writes the next E Phi into a second copy too.
static int ensure_next_plane(gpx_ctx *ctx)
{
    if (int rc = ensure_next_state(ctx)) return rc;
    if (!ctx->phiE[0] || ctx->phiE[1]) return 0;
    const size_t b = phi_bytes(ctx);   // the current one is phiE[0]
    float *p;
    if (int rc = dalloc_all(ctx, 1, &p, &b, false)) return rc;
    ctx->phiE[1] = p;
    ctx->next_bytes += b;
    ctx->row_dirty = true;
    GPX_TRY(hipMemcpyAsync(p, ctx->phiE[0], b, hipMemcpyDeviceToDevice, ctx->stream));
    return 0;
}

// ---------------------------------------------------------------- auxiliary-value slots
// Edges of one component whose material has poles, per block of 1024 cells.
template <class IDT>
__global__ void k_tslot_count(const IDT *ID, const uint8_t *flag, long long ntot, uint32_t *bsum)
{
    __shared__ int tot;
    if (threadIdx.x == 0) tot = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * 1024;
    int cnt = 0;
    for (int q = threadIdx.x; q < 1024; q += blockDim.x) {
        const long long e = base + q;
        if (e < ntot && flag[ID[e]]) ++cnt;
    }
    atomicAdd(&tot, cnt);
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = (uint32_t)tot;
}

// The slot of every such edge: the block's offset plus the edges before it
// in the block (wave ballots, then the waves before it).  1024 threads.
template <class IDT>
__global__ void __launch_bounds__(1024) k_tslot_fill(const IDT *ID, const uint8_t *flag, long long ntot,
                                                     const uint32_t *boff, uint32_t *slot)
{
    __shared__ int wsum[16];
    const long long e = (long long)blockIdx.x * 1024 + threadIdx.x;
    const bool f = e < ntot && flag[ID[e]];
    const unsigned long long m = __ballot(f);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) wsum[w] = __popcll(m);
    __syncthreads();
    int off = 0;
    for (int q = 0; q < w; ++q) off += wsum[q];
    const int before = __popcll(m & ((1ull << lane) - 1ull));
    if (e < ntot) slot[e] = f ? boff[blockIdx.x] + (uint32_t)(off + before) : 0xffffffffu;
}

// The slots as the passes read them (row_slots_of): a wave for each group of
// 64 lanes of a plane (128 cells of `plane`, fewer at its end) and each component.
__global__ void k_tslot_masks(const uint32_t *slot, uint32_t *masks, int c, int plane, int groups, int n)
{
    const int g = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (g >= n) return;
    const int i = g / groups, q = (g - i * groups) * 128 + 2 * lane;
    const uint32_t *s = slot + (size_t)i * plane;
    const uint32_t s0 = q < plane ? s[q] : T_NOSLOT, s1 = q + 1 < plane ? s[q + 1] : T_NOSLOT;
    const unsigned long long even = __ballot(s0 != T_NOSLOT), odd = __ballot(s1 != T_NOSLOT), any = even | odd;
    const uint32_t mine = s0 != T_NOSLOT ? s0 : s1;
    const uint32_t first = any ? __shfl(mine, __ffsll(any) - 1) : 0u;
    if (lane == 0) {
        uint32_t *m = masks + (size_t)g * 16;
        m[4 * c] = (uint32_t)even;
        m[4 * c + 1] = (uint32_t)(even >> 32);
        m[4 * c + 2] = (uint32_t)odd;
        m[4 * c + 3] = (uint32_t)(odd >> 32);
        m[12 + c] = first;
    }
}
static int tslot_groups(const gpx_ctx *ctx) { return (ctx->plane + 127) / 128; }

static int ensure_tslots(gpx_ctx *ctx);

static void fill_targs(const gpx_ctx *ctx, TArgs &t)
{
    for (int c = 0; c < 3; ++c) {
        t.T[c] = ctx->T[c];
        t.slot[c] = ctx->tslot[c];
        t.n[c] = ctx->tn[c];
    }
    t.masks = ctx->tmasks;
    t.groups = tslot_groups(ctx);
}

// Builds the slots and the compacted auxiliary arrays (zeroed) once the
// indices and the dispersive tables are on the device.  A new upload of
// either starts the auxiliary values again from zero.
static int ensure_tslots(gpx_ctx *ctx)
{
    const int P = ctx->desc.maxpoles;
    if (P == 0 || !ctx->tslot_dirty || !ctx->have_id || !ctx->have_disp) return 0;
    const long long N = ctx->ntot;
    if (N >= 0xffffffffLL) return fail(ctx, GPX_ELIMIT, "dispersive models need fewer than 2^32 points");
    hipSetDevice(ctx->desc.device);
    const int nb = (int)((N + 1023) / 1024);
    const int ng = (ctx->desc.nx + 1) * tslot_groups(ctx);
    if (!ctx->tmasks) GPX_TRY(dalloc(ctx, (void **)&ctx->tmasks, (size_t)ng * 64, false));
    uint32_t *boff = nullptr;
    GPX_TRY(dalloc(ctx, (void **)&boff, (size_t)nb * 4, false));
    std::vector<uint32_t> h(nb);
    int rc = 0;
    for (int c = 0; c < 3 && !rc; ++c) {
        if (!ctx->tslot[c]) {
            hipError_t e = dalloc(ctx, (void **)&ctx->tslot[c], (size_t)N * 4, false);
            if (e != hipSuccess) { rc = fail_hip(ctx, e, "slot array"); break; }
        }
        hipLaunchKernelGGL(k_tslot_count<uint16_t>, dim3(nb), dim3(256), 0, ctx->stream,
                           ctx->ID + (size_t)c * N, ctx->dispflag, N, boff);
        if ((rc = copy_out(ctx, h.data(), boff, (size_t)nb * 4))) break;
        unsigned long long acc = 0;
        for (int b = 0; b < nb; ++b) {
            const uint32_t v = h[b];
            h[b] = (uint32_t)acc;
            acc += v;
        }
        if ((rc = copy_in(ctx, boff, h.data(), (size_t)nb * 4))) break;
        hipLaunchKernelGGL(k_tslot_fill<uint16_t>, dim3(nb), dim3(1024), 0, ctx->stream,
                           ctx->ID + (size_t)c * N, ctx->dispflag, N, boff, ctx->tslot[c]);
        hipLaunchKernelGGL(k_tslot_masks, dim3((ng + 3) / 4), dim3(256), 0, ctx->stream, ctx->tslot[c], ctx->tmasks, c,
                           ctx->plane, tslot_groups(ctx), ng);
        hipError_t e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) { rc = fail_hip(ctx, e, "slot build"); break; }
        ctx->tn[c] = (long long)acc;
        if (ctx->T[c]) { hipFree(ctx->T[c]); ctx->T[c] = nullptr; }
        ctx->row_dirty = true;
        // a pair's load at the last slot goes one value further
        const size_t tb = ((size_t)P * (size_t)(acc > 0 ? acc : 1) + 1) * 4 * (ctx->disp_complex ? 2 : 1);
        e = dalloc(ctx, (void **)&ctx->T[c], tb);
        if (e != hipSuccess) { rc = fail_hip(ctx, e, "auxiliary values"); break; }
    }
    hipFree(boff);
    if (!rc) {
        GPX_TRY(hipStreamSynchronize(ctx->stream));
        ctx->tslot_dirty = false;
    }
    return rc;
}

// Material indices of n rows of nk: to 16 bits (every index < nmat < 2^16), rows of kp,
// the padding material 0; *bad: the least place, counted from `first`, of an
// index that is not below nmat.  Four cells a thread, a copy's work.
__global__ void k_narrow_id(const uint32_t *src, uint16_t *dst, long long n, int nk, int kp, uint32_t nmat,
                            unsigned long long first, unsigned long long *bad)
{
    const long long cells = n * kp, q0 = (long long)blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long long q = q0 + u * 256;
        if (q >= cells) return;
        const long long r = q / kp;
        const int k = (int)(q - r * kp);
        uint32_t m = 0;
        if (k < nk) {
            m = src[r * nk + k];
            if (m >= nmat) {
                atomicMin(bad, first + (unsigned long long)(r * nk + k));
                m = 0;
            }
        }
        dst[q] = (uint16_t)m;
    }
}
constexpr size_t ID_PIECE = (size_t)64 << 20;   // bytes of indices in flight to the device

extern "C" int gpx_upload_id(gpx_ctx *ctx, const uint32_t *ID)
{
    if (!ctx || !ID) return fail(ctx, GPX_EARG, "gpx_upload_id: null argument");
    const uint32_t nmat = (uint32_t)ctx->desc.nmat;
    const gpx_desc &g = ctx->desc;
    const size_t nk = (size_t)g.nz + 1, rows = 6 * (size_t)(g.nx + 1) * (g.ny + 1);
    auto refuse = [&](size_t q) {
        return fail(ctx, GPX_EARG, "gpx_upload_id: material index " + std::to_string(ID[q]) + " >= nmat " + std::to_string(nmat));
    };
    hipSetDevice(g.device);
    // Every ID indexes the coefficient tables; out-of-range values are refused
    // so no kernel can read outside them.  A model that has indices keeps them
    // then, so new ones are looked through here first.
    for (size_t q = 0; q < rows * nk && ctx->have_id; ++q)
        if (ID[q] >= nmat) return refuse(q);
    // 32-bit indices go up in pieces and are checked, narrowed and padded there:
    // one pass of the host over them, the copy's, instead of four (300x300x200,
    // 437 MB: 86 ms before, 20 now).
    const size_t piece = std::max<size_t>(1, std::min(rows, ID_PIECE / (nk * 4)));
    uint32_t *d = nullptr;
    unsigned long long *bad = nullptr, first = ~0ull;
    const size_t words = (piece * nk + 1) / 2 * 2;
    hipError_t e = hipMalloc((void **)&d, words * 4 + 8);
    bad = reinterpret_cast<unsigned long long *>(d + words);
    int rc = 0;
    if (e == hipSuccess) e = hipMemsetAsync(bad, 0xff, 8, ctx->stream);
    for (size_t r = 0; r < rows && e == hipSuccess; r += piece) {
        const size_t n = std::min(piece, rows - r);
        e = hipMemcpyAsync(d, ID + r * nk, n * nk * 4, hipMemcpyHostToDevice, ctx->stream);
        if (e != hipSuccess) break;
        const size_t cells = n * (size_t)ctx->kp;
        hipLaunchKernelGGL(k_narrow_id, dim3((unsigned)((cells + 1023) / 1024)), dim3(256), 0, ctx->stream, d,
                           ctx->ID + r * ctx->kp, (long long)n, (int)nk, ctx->kp, nmat, (unsigned long long)(r * nk), bad);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&first, bad, 8, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (d) hipFree(d);
    if (e != hipSuccess) return fail_hip(ctx, e, "gpx_upload_id");
    if (first != ~0ull) return refuse((size_t)first);
    if (!rc) {
        ctx->have_id = true;
        ctx->tslot_dirty = true;
        rc = ensure_tslots(ctx);
    }
    return rc;
}

extern "C" int gpx_upload_coeffs(gpx_ctx *ctx, const float *cE, const float *cH)
{
    if (!ctx || !cE || !cH) return fail(ctx, GPX_EARG, "gpx_upload_coeffs: null argument");
    hipSetDevice(ctx->desc.device);
    const size_t b = (size_t)ctx->desc.nmat * 5 * 4;
    int rc = copy_in(ctx, ctx->cE, cE, b);
    if (!rc) rc = copy_in(ctx, ctx->cH, cH, b);
    if (!rc) ctx->have_coeffs = true;
    // Non-magnetic models (mu_r and sigma* the same everywhere, the rule in
    // ground-penetrating radar) have one row of H coefficients: the row
    // kernels then read no H index and look nothing up, 6 bytes a cell and
    // step less.
    ctx->hu = true;
    for (int m = 1; m < ctx->desc.nmat; ++m)
        if (memcmp(cH, cH + 5 * (size_t)m, 20) != 0) ctx->hu = false;
    ctx->hostE.assign(cE, cE + 5 * (size_t)ctx->desc.nmat);
    ctx->hostH.assign(cH, cH + 5 * (size_t)ctx->desc.nmat);
    ctx->row_dirty = true;
    return rc;
}

extern "C" int gpx_upload_dispersive(gpx_ctx *ctx, const float *dc)
{
    if (!ctx || !dc) return fail(ctx, GPX_EARG, "gpx_upload_dispersive: null argument");
    const int P = ctx->desc.maxpoles, nm = ctx->desc.nmat;
    if (P == 0) return fail(ctx, GPX_ESTATE, "gpx_upload_dispersive: model has no poles");
    hipSetDevice(ctx->desc.device);
    // Keep complex arithmetic only where an imaginary part is non-zero
    // (Lorentz); Debye and Drude poles are real.
    int cplx = 0;
    for (size_t q = 0; q < (size_t)nm * 3 * P; ++q)
        if (dc[2 * q + 1] != 0.0f) cplx = 1;
    std::vector<float> host;
    std::vector<uint8_t> flag(nm, 0);
    for (int m = 0; m < nm; ++m)
        for (int q = 0; q < 3 * P; ++q)
            if (dc[((size_t)m * 3 * P + q) * 2] != 0.0f || dc[((size_t)m * 3 * P + q) * 2 + 1] != 0.0f) flag[m] = 1;
    if (cplx) host.assign(dc, dc + (size_t)nm * 3 * P * 2);
    else {
        host.resize((size_t)nm * 3 * P);
        for (size_t q = 0; q < host.size(); ++q) host[q] = dc[2 * q];
    }
    if (ctx->have_disp && cplx != ctx->disp_complex)
        return fail(ctx, GPX_ESTATE, "gpx_upload_dispersive: real/complex kind cannot change after upload");
    if (!ctx->disp) {
        GPX_TRY(dalloc(ctx, (void **)&ctx->disp, host.size() * 4));
        GPX_TRY(dalloc(ctx, (void **)&ctx->dispflag, nm));
    }
    ctx->disp_complex = cplx;
    int rc = copy_in(ctx, ctx->disp, host.data(), host.size() * 4);
    if (!rc) rc = copy_in(ctx, ctx->dispflag, flag.data(), nm);
    if (!rc) {
        ctx->have_disp = true;
        ctx->tslot_dirty = ctx->row_dirty = true;
        ctx->hostdisp.swap(host);
        rc = ensure_tslots(ctx);
    }
    return rc;
}

static void phi_dims(int field, int axis, int snx, int sny, int snz, long long d1[3], long long d2[3])
{
    // gprMax/pml.py:202-219
    long long a[3], b[3];
    if (field == 0) {
        if (axis == 0) { a[0] = snx + 1; a[1] = sny; a[2] = snz + 1; b[0] = snx + 1; b[1] = sny + 1; b[2] = snz; }
        else if (axis == 1) { a[0] = snx; a[1] = sny + 1; a[2] = snz + 1; b[0] = snx + 1; b[1] = sny + 1; b[2] = snz; }
        else { a[0] = snx; a[1] = sny + 1; a[2] = snz + 1; b[0] = snx + 1; b[1] = sny; b[2] = snz + 1; }
    } else {
        if (axis == 0) { a[0] = snx; a[1] = sny + 1; a[2] = snz; b[0] = snx; b[1] = sny; b[2] = snz + 1; }
        else if (axis == 1) { a[0] = snx + 1; a[1] = sny; a[2] = snz; b[0] = snx; b[1] = sny; b[2] = snz + 1; }
        else { a[0] = snx + 1; a[1] = sny; a[2] = snz; b[0] = snx; b[1] = sny + 1; b[2] = snz; }
    }
    for (int n = 0; n < 3; ++n) { d1[n] = a[n]; d2[n] = b[n]; }
}

extern "C" int gpx_add_pml(gpx_ctx *ctx, int dir, int xs, int xf, int ys, int yf, int zs, int zf,
                           int order, float d, const float *eR, const float *hR, int *slab)
{
    if (!ctx || !eR || !hR) return fail(ctx, GPX_EARG, "gpx_add_pml: null argument");
    if ((int)ctx->slabs.size() >= MAX_SLABS) return fail(ctx, GPX_ELIMIT, "gpx_add_pml: at most 6 slabs");
    if (dir < 0 || dir > 5 || (order != 1 && order != 2))
        return fail(ctx, GPX_EARG, "gpx_add_pml: direction must be 0..5 and order 1 or 2");
    const gpx_desc &g = ctx->desc;
    if (xs < 0 || ys < 0 || zs < 0 || xf > g.nx || yf > g.ny || zf > g.nz || xs >= xf || ys >= yf || zs >= zf)
        return fail(ctx, GPX_EARG, "gpx_add_pml: slab box outside the grid");
    const int axis = dir % 3;
    const int t = axis == 0 ? xf - xs : (axis == 1 ? yf - ys : zf - zs);
    // The corrected cells reach one cell beyond the box on the minus side
    // (E) and one cell inside it (H); both must have their neighbours.
    const int lo = axis == 0 ? xs : (axis == 1 ? ys : zs);
    const int hi = axis == 0 ? xf : (axis == 1 ? yf : zf);
    const int n = axis == 0 ? g.nx : (axis == 1 ? g.ny : g.nz);
    if (dir < 3 && (hi - t + 1 < 1 || hi >= n + 1)) return fail(ctx, GPX_EARG, "gpx_add_pml: minus slab out of range");
    if (dir >= 3 && (lo < 1 || lo + t > n)) return fail(ctx, GPX_EARG, "gpx_add_pml: plus slab out of range");
    hipSetDevice(g.device);
    Slab s;
    s.dir = dir; s.xs = xs; s.xf = xf; s.ys = ys; s.yf = yf; s.zs = zs; s.zf = zf;
    s.order = order; s.t = t; s.d = d;
    phi_dims(0, axis, xf - xs, yf - ys, zf - zs, s.dims[0], s.dims[1]);
    phi_dims(1, axis, xf - xs, yf - ys, zf - zs, s.dims[2], s.dims[3]);
    s.ni = s.nj = 0;
    int nk = 0;
    for (auto &q : s.dims) {
        s.ni = s.ni > q[0] ? s.ni : (int)q[0];
        s.nj = s.nj > q[1] ? s.nj : (int)q[1];
        nk = nk > q[2] ? nk : (int)q[2];
    }
    s.nkp = (nk + 3 + 3) / 4 * 4;  // up to three floats before the first cell
    const size_t rb = (size_t)4 * order * t * 4;
    s.roff = (int)ctx->Rhost[0].size();
    const size_t need = (size_t)g.nmat * 5 * 4 + (ctx->Rhost[0].size() + rb / 4) * 4 +
                        (size_t)g.nmat * 3 * g.maxpoles * 2 * 4 + g.nmat;
    if (need > (size_t)MAX_LDS_BYTES)
        return fail(ctx, GPX_ELIMIT, "gpx_add_pml: coefficient tables exceed the LDS budget");
    s.R[0].assign(eR, eR + rb / 4);
    s.R[1].assign(hR, hR + rb / 4);
    ctx->slabs.push_back(s);
    ctx->phi_dirty = ctx->row_dirty = true;
    ctx->Rhost[0].insert(ctx->Rhost[0].end(), eR, eR + rb / 4);
    ctx->Rhost[1].insert(ctx->Rhost[1].end(), hR, hR + rb / 4);
    if (slab) *slab = (int)ctx->slabs.size() - 1;
    return update_planeflags(ctx);
}

extern "C" int gpx_set_sources(gpx_ctx *ctx, int kind, int n, const int32_t *info,
                               const float *factors, const float *waves)
{
    if (!ctx || kind < 0 || kind > 2 || n < 0) return fail(ctx, GPX_EARG, "gpx_set_sources: bad argument");
    if (n > 0 && (!info || !factors || !waves)) return fail(ctx, GPX_EARG, "gpx_set_sources: null array");
    const gpx_desc &g = ctx->desc;
    for (int s = 0; s < n; ++s) {
        const int32_t *in = info + 6 * s;
        const int pol = in[3] & 3;
        if (in[0] < 0 || in[0] > g.nx || in[1] < 0 || in[1] > g.ny || in[2] < 0 || in[2] > g.nz || pol > 2 ||
            (in[3] >= 4 && kind != GPX_SRC_VOLTAGE) || in[3] < 0 || in[3] > 6)
            return fail(ctx, GPX_EARG, "gpx_set_sources: source " + std::to_string(s) + " has a bad cell or polarisation");
    }
    hipSetDevice(g.device);
    SrcSet &S = ctx->src[kind];
    if (S.info) { hipFree(S.info); S.info = nullptr; }
    if (S.fac) { hipFree(S.fac); S.fac = nullptr; }
    if (S.waves) { hipFree(S.waves); S.waves = nullptr; }
    S.n = n;
    S.host.clear();
    if (n == 0) return update_planeflags(ctx);
    GPX_TRY(dalloc(ctx, (void **)&S.info, (size_t)n * 6 * 4, false));
    GPX_TRY(dalloc(ctx, (void **)&S.fac, (size_t)n * 2 * 4, false));
    GPX_TRY(dalloc(ctx, (void **)&S.waves, (size_t)n * g.iterations * 4, false));
    S.host.assign(info, info + (size_t)n * 6);
    int rc = copy_in(ctx, S.info, info, (size_t)n * 6 * 4);
    if (!rc) rc = copy_in(ctx, S.fac, factors, (size_t)n * 2 * 4);
    if (!rc) rc = copy_in(ctx, S.waves, waves, (size_t)n * g.iterations * 4);
    if (!rc) rc = update_planeflags(ctx);
    return rc;
}

extern "C" int gpx_add_transmission_line(gpx_ctx *ctx, const int32_t *info, const double *coef,
                                         const float *sizes, const float *whole, const float *half,
                                         const float *voltage, const float *current, const float *abc,
                                         int *index)
{
    if (!ctx || !info || !coef || !sizes || !whole || !half || !voltage || !current || !abc)
        return fail(ctx, GPX_EARG, "gpx_add_transmission_line: null argument");
    const gpx_desc &g = ctx->desc;
    const int i = info[0], j = info[1], k = info[2], pol = info[3], nl = info[6], srcpos = info[7],
              antpos = info[8];
    if (i < 0 || i > g.nx || j < 0 || j > g.ny || k < 0 || k > g.nz || pol < 0 || pol > 2)
        return fail(ctx, GPX_EARG, "gpx_add_transmission_line: bad cell or polarisation");
    if (nl < 2 || srcpos < 1 || srcpos >= nl || antpos < 0 || antpos >= nl)
        return fail(ctx, GPX_EARG, "gpx_add_transmission_line: bad line length or positions");
    hipSetDevice(g.device);
    TLine t;
    TLDev &d = t.d;
    d.i = i; d.j = j; d.k = k; d.pol = pol; d.first = info[4]; d.last = info[5];
    d.nl = nl; d.srcpos = srcpos; d.antpos = antpos;
    d.cV = coef[0]; d.cI = coef[1]; d.cW = coef[2]; d.h = coef[3];
    d.dpol = sizes[0]; d.da = sizes[1]; d.db = sizes[2];
    const size_t its = (size_t)g.iterations;
    const size_t nf = 2 * (size_t)nl + 2 + 4 * its;
    GPX_TRY(dalloc(ctx, (void **)&t.mem, nf * 4));
    d.V = t.mem;
    d.I = d.V + nl;
    d.abc = d.I + nl;
    d.whole = d.abc + 2;
    d.half = d.whole + its;
    d.vt = const_cast<float *>(d.half) + its;
    d.itot = d.vt + its;
    int rc = copy_in(ctx, d.V, voltage, (size_t)nl * 4);
    if (!rc) rc = copy_in(ctx, d.I, current, (size_t)nl * 4);
    if (!rc) rc = copy_in(ctx, d.abc, abc, 8);
    if (!rc) rc = copy_in(ctx, const_cast<float *>(d.whole), whole, its * 4);
    if (!rc) rc = copy_in(ctx, const_cast<float *>(d.half), half, its * 4);
    if (rc) {
        hipFree(t.mem);
        return rc;
    }
    ctx->tls.push_back(t);
    if (ctx->tldev) { hipFree(ctx->tldev); ctx->tldev = nullptr; }
    GPX_TRY(dalloc(ctx, (void **)&ctx->tldev, ctx->tls.size() * sizeof(TLDev), false));
    std::vector<TLDev> all;
    for (const TLine &x : ctx->tls) all.push_back(x.d);
    rc = copy_in(ctx, ctx->tldev, all.data(), all.size() * sizeof(TLDev));
    if (index) *index = (int)ctx->tls.size() - 1;
    return rc;
}

extern "C" int gpx_download_transmission_line(gpx_ctx *ctx, int index, float *vtotal, float *itotal,
                                              float *voltage, float *current)
{
    if (!ctx || index < 0 || index >= (int)ctx->tls.size())
        return fail(ctx, GPX_EARG, "gpx_download_transmission_line: bad index");
    hipSetDevice(ctx->desc.device);
    const TLDev &d = ctx->tls[index].d;
    const size_t its = (size_t)ctx->desc.iterations;
    GPX_TRY(hipStreamSynchronize(ctx->stream));
    if (vtotal) GPX_TRY(hipMemcpy(vtotal, d.vt, its * 4, hipMemcpyDeviceToHost));
    if (itotal) GPX_TRY(hipMemcpy(itotal, d.itot, its * 4, hipMemcpyDeviceToHost));
    if (voltage) GPX_TRY(hipMemcpy(voltage, d.V, (size_t)d.nl * 4, hipMemcpyDeviceToHost));
    if (current) GPX_TRY(hipMemcpy(current, d.I, (size_t)d.nl * 4, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int gpx_set_receivers(gpx_ctx *ctx, int n, const int32_t *coords)
{
    if (!ctx || n < 0 || (n > 0 && !coords)) return fail(ctx, GPX_EARG, "gpx_set_receivers: bad argument");
    const gpx_desc &g = ctx->desc;
    for (int r = 0; r < n; ++r)
        if (coords[3 * r] < 0 || coords[3 * r] > g.nx || coords[3 * r + 1] < 0 || coords[3 * r + 1] > g.ny ||
            coords[3 * r + 2] < 0 || coords[3 * r + 2] > g.nz)
            return fail(ctx, GPX_EARG, "gpx_set_receivers: receiver outside the grid");
    hipSetDevice(g.device);
    if (ctx->rxc) { hipFree(ctx->rxc); ctx->rxc = nullptr; }
    if (ctx->rxbuf) { hipFree(ctx->rxbuf); ctx->rxbuf = nullptr; }
    ctx->nrx = n;
    ctx->rxhost.assign(coords, coords + (size_t)n * 3);
    if (n == 0) return update_planeflags(ctx);
    GPX_TRY(dalloc(ctx, (void **)&ctx->rxc, (size_t)n * 3 * 4, false));
    GPX_TRY(dalloc(ctx, (void **)&ctx->rxbuf, (size_t)6 * g.iterations * n * 4));
    int rc = copy_in(ctx, ctx->rxc, coords, (size_t)n * 3 * 4);
    return rc ? rc : update_planeflags(ctx);
}

extern "C" int gpx_add_snapshot(gpx_ctx *ctx, int xs, int ys, int zs, int dx, int dy, int dz,
                                int snx, int sny, int snz, int time, int *index)
{
    if (!ctx || dx < 1 || dy < 1 || dz < 1 || snx < 1 || sny < 1 || snz < 1 || xs < 0 || ys < 0 || zs < 0)
        return fail(ctx, GPX_EARG, "gpx_add_snapshot: bad argument");
    const gpx_desc &g = ctx->desc;
    // The averages read slice points up to index snx (one past the last cell).
    if (xs + (long long)snx * dx > g.nx || ys + (long long)sny * dy > g.ny || zs + (long long)snz * dz > g.nz)
        return fail(ctx, GPX_EARG, "gpx_add_snapshot: snapshot volume outside the grid");
    hipSetDevice(g.device);
    Snap s;
    s.xs = xs; s.ys = ys; s.zs = zs; s.dx = dx; s.dy = dy; s.dz = dz;
    s.snx = snx; s.sny = sny; s.snz = snz; s.time = time;
    GPX_TRY(dalloc(ctx, (void **)&s.out, (size_t)6 * snx * sny * snz * 4));
    ctx->snaps.push_back(s);
    if (index) *index = (int)ctx->snaps.size() - 1;
    return 0;
}

extern "C" int gpx_set_step(gpx_ctx *ctx, int fused, int tile_cells)
{
    if (!ctx || fused < 0 || fused > 7 ||
        !(tile_cells == 0 || tile_cells == 256 || tile_cells == 512 || tile_cells == 1024))
        return fail(ctx, GPX_EARG, "gpx_set_step: bad argument");
    ctx->fused = fused;
    ctx->tile_cells = tile_cells;
    ctx->choice = -1;
    ctx->row_dirty = true;
    return 0;
}

extern "C" int gpx_set_launch(gpx_ctx *ctx, int xchunk, int block)
{
    if (!ctx || xchunk < 0 || !(block == 0 || block == 64 || block == 128 || block == 256 || block == 512 || block == 1024))
        return fail(ctx, GPX_EARG, "gpx_set_launch: bad argument");
    ctx->xchunk = xchunk;
    ctx->block = block;
    ctx->row_dirty = true;
    return 0;
}

// ---------------------------------------------------------------- launching
// Work split of one pass.  Items are (cell segment, x chunk), one block each:
// the grid holds every item (rounded up to a multiple of 8) and the hardware
// dispatcher balances them.  Chunks are short (6 planes for the interior, 4
// for the boundary, unless fixed by gpx_set_launch): on the 300x300x200
// half-space these beat both longer chunks and a persistent grid of resident
// blocks by 11 %, since fewer planes are streamed at once.  Grids too small
// to fill the GPU with such items take shorter chunks.
static long long count_items(const gpx_ctx *ctx, bool bnd, int block, int xc, StepArgs *a)
{
    const int *b = ctx->box;
    const int nframe = ctx->nframe;
    auto ch = [&](int len) { return len > 0 ? (len + xc - 1) / xc : 0; };
    if (!bnd) {
        const long long cells = (long long)(b[3] - b[2]) * (b[5] - b[4]);
        const int nseg = (int)((cells + block - 1) / block);
        const long long items = cells > 0 ? (long long)nseg * ch(b[1] - b[0]) : 0;
        if (a) { a->nseg = nseg; a->nitems = (int)items; }
        return items;
    }
    const int nseg_a = (ctx->plane + block - 1) / block;
    const int nseg_b = (nframe + block - 1) / block;
    const long long a1 = (long long)nseg_a * ch(b[0]);
    const long long a2 = (long long)nseg_a * ch(ctx->desc.nx + 1 - b[1]);
    const long long bb = (long long)nseg_b * ch(b[1] - b[0]);
    if (a) {
        a->nseg_a = nseg_a; a->nseg_b = nseg_b;
        a->items_a1 = (int)a1; a->items_a2 = (int)a2;
        a->nitems = (int)(a1 + a2 + bb);
    }
    return a1 + a2 + bb;
}

static void plan(const gpx_ctx *ctx, bool bnd, int block, StepArgs &a, int &grid, int fill = 0)
{
    const int NX1 = ctx->desc.nx + 1;
    int xc = ctx->xchunk ? ctx->xchunk : (bnd ? 4 : 6);
    if (xc > NX1) xc = NX1;
    // Small grids: shorter chunks, down to 2 planes, until the items fill the
    // `fill` blocks the GPU holds at once (on the 100^3 grid 2 planes beat 1:
    // each chunk loads one neighbour plane more).
    if (!ctx->xchunk)
        while (xc > 2 && count_items(ctx, bnd, block, xc, nullptr) < fill) --xc;
    a.xc = xc;
    long long g = count_items(ctx, bnd, block, xc, &a);
    g = (g + 7) / 8 * 8;
    if (g < 8) g = 8;
    a.per_xcd = (int)(g / 8);
    grid = (int)g;
}

static int resident_blocks(const gpx_ctx *ctx, const void *kernel, int block, size_t lds)
{
    auto key = std::make_pair(kernel, lds * 4096 + (size_t)block);
    auto it = ctx->occupancy.find(key);
    if (it != ctx->occupancy.end()) return it->second;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, block, lds) != hipSuccess || nb < 1) nb = 1;
    const int r = nb * (ctx->cus > 0 ? ctx->cus : 256);
    ctx->occupancy[key] = r;
    return r;
}

// Box of corrected cells, profile direction and Phi strides of slab s.
static void fill_slab_args(const gpx_ctx *ctx, int field, int s, SlabArgs &a)
{
    const Slab &S = ctx->slabs[s];
    const int axis = S.dir % 3, minus = S.dir < 3;
    const int st[3] = {S.xs, S.ys, S.zs}, en[3] = {S.xf, S.yf, S.zf};
    a.axis = axis;
    a.minus = minus;
    for (int n = 0; n < 3; ++n) {
        a.lo[n] = st[n];
        a.hi[n] = en[n];
    }
    if (minus) {
        if (field == 0) {  // cells f - p, p in [0, t)
            a.lo[axis] = en[axis] - S.t + 1;
            a.hi[axis] = en[axis] + 1;
            a.pend = en[axis];
        } else {           // cells f - (p + 1)
            a.lo[axis] = en[axis] - S.t;
            a.hi[axis] = en[axis];
            a.pend = en[axis] - 1;
        }
    } else {
        a.lo[axis] = st[axis];
        a.hi[axis] = st[axis] + S.t;
        a.pend = st[axis];
    }
    a.sx = S.nj * S.nkp;
    a.sy = S.nkp;
    a.off = (int)(S.base - (long long)a.lo[0] * a.sx - (long long)a.lo[1] * a.sy - a.lo[2] + (a.lo[2] & 3));
    a.ostep = (uint32_t)(2 * ctx->np);
    a.t = S.t;
    a.order = S.order;
    a.d = S.d;
    a.phi1 = field == 0 ? ctx->phiE[ctx->curE] : ctx->phiH[ctx->cur];
    a.phi2 = a.phi1 ? a.phi1 + ctx->np : nullptr;
    a.roff = S.roff;
}

static int update_planeflags(gpx_ctx *ctx)
{
    ctx->rare_dirty = ctx->planes_dirty = true;  // sources, receivers or slabs may have changed
    // Interior box: cells 1..n-1 on every axis (all neighbours and all updates
    // present), shrunk past every slab box that spans the cross-section.
    const gpx_desc &g = ctx->desc;
    const int n[3] = {g.nx, g.ny, g.nz};
    int lo[3] = {1, 1, 1}, hi[3] = {g.nx, g.ny, g.nz};
    bool empty = false;
    for (size_t s = 0; s < ctx->slabs.size() && !empty; ++s) {
        for (int field = 0; field < 2; ++field) {
            SlabArgs b;
            fill_slab_args(ctx, field, (int)s, b);
            const int ax = b.axis;
            bool spans = true;
            for (int o = 0; o < 3; ++o)
                if (o != ax && (b.lo[o] > 1 || b.hi[o] < n[o])) spans = false;
            if (!spans) { empty = true; break; }
            if (b.minus) lo[ax] = lo[ax] > b.hi[ax] ? lo[ax] : b.hi[ax];
            else hi[ax] = hi[ax] < b.lo[ax] ? hi[ax] : b.lo[ax];
        }
    }
    for (int o = 0; o < 3; ++o)
        if (lo[o] >= hi[o]) empty = true;
    if (empty) {
        const int b[6] = {g.nx + 1, g.nx + 1, 0, 0, 0, 0};
        memcpy(ctx->box, b, sizeof(b));
    } else {
        const int b[6] = {lo[0], hi[0], lo[1], hi[1], lo[2], hi[2]};
        memcpy(ctx->box, b, sizeof(b));
    }
    const int *b = ctx->box;
    ctx->deep = !empty && b[0] + 1 < b[1] && b[2] + 1 < b[3] && b[4] + 1 < b[5];
    ctx->row_dirty = true;
    return 0;
}

// Brings the planes' flags, the general passes' frame of the interior box and
// their profile tables up to date: once before a run, not with every slab,
// source and receiver set.
static int ensure_planes(gpx_ctx *ctx)
{
    if (!ctx->planes_dirty) return 0;
    hipSetDevice(ctx->desc.device);
    const int NX1 = ctx->desc.nx + 1;
    std::vector<uint32_t> pf(2 * NX1, 0);
    for (int r = 0; r < ctx->nrx; ++r) pf[ctx->rxhost[3 * r]] |= PF_RX;
    for (int s = 0; s < ctx->src[GPX_SRC_MAGNETIC].n; ++s) pf[ctx->src[GPX_SRC_MAGNETIC].host[6 * s]] |= PF_SRCH;
    for (int kind : {GPX_SRC_HERTZIAN, GPX_SRC_VOLTAGE})
        for (int s = 0; s < ctx->src[kind].n; ++s) pf[ctx->src[kind].host[6 * s]] |= PF_SRCE;
    for (size_t s = 0; s < ctx->slabs.size(); ++s) {
        SlabArgs e, h;
        fill_slab_args(ctx, 0, (int)s, e);
        fill_slab_args(ctx, 1, (int)s, h);
        const int dir = ctx->slabs[s].dir;
        for (int i = 0; i < NX1; ++i) {
            if (i >= e.lo[0] && i < e.hi[0]) pf[i] |= 1u << (PF_SLAB_E + s), pf[NX1 + i] |= 1u << (PF_SLAB_E + dir);
            if (i >= h.lo[0] && i < h.hi[0]) pf[i] |= 1u << (PF_SLAB_H + s), pf[NX1 + i] |= 1u << (PF_SLAB_H + dir);
        }
    }
    for (int i = 0; i < NX1; ++i) pf[NX1 + i] |= pf[i] & (PF_RX | PF_SRCH | PF_SRCE);
    int rc = copy_in(ctx, ctx->planeflag, pf.data(), pf.size() * 4);
    if (rc) return rc;
    for (int f = 0; f < 2; ++f) {
        if (ctx->Rall[f]) hipFree(ctx->Rall[f]);
        ctx->Rall[f] = nullptr;
        if (ctx->Rhost[f].empty()) continue;
        GPX_TRY(dalloc(ctx, (void **)&ctx->Rall[f], ctx->Rhost[f].size() * 4, false));
        if ((rc = copy_in(ctx, ctx->Rall[f], ctx->Rhost[f].data(), ctx->Rhost[f].size() * 4))) return rc;
    }
    const int *lo = ctx->box, *hi = ctx->box + 1;
    std::vector<int> fr;
    if (lo[0] < hi[0]) {
        for (int j = 0; j <= ctx->desc.ny; ++j)
            for (int k = 0; k <= ctx->desc.nz; ++k)
                if (!(j >= lo[2] && j < hi[2] && k >= lo[4] && k < hi[4])) fr.push_back(j * ctx->kp + k);
    }
    if (ctx->frame) { hipFree(ctx->frame); ctx->frame = nullptr; }
    ctx->nframe = (int)fr.size();
    if (!fr.empty()) {
        GPX_TRY(dalloc(ctx, (void **)&ctx->frame, fr.size() * 4, false));
        rc = copy_in(ctx, ctx->frame, fr.data(), fr.size() * 4);
        if (rc) return rc;
    }
    ctx->planes_dirty = false;
    return 0;
}

static void base_args(const gpx_ctx *ctx, int field, StepArgs &a, int &block, size_t &lds)
{
    block = ctx->block ? ctx->block : 256;
    memset(&a, 0, sizeof(a));
    const gpx_desc &g = ctx->desc;
    a.nx = g.nx; a.ny = g.ny; a.nz = g.nz;
    a.kp = ctx->kp;
    a.plane = ctx->plane;
    a.Ex = ctx->field(0); a.Ey = ctx->field(1); a.Ez = ctx->field(2);
    a.Hx = ctx->field(3); a.Hy = ctx->field(4); a.Hz = ctx->field(5);
    a.ID = ctx->ID;
    a.ntot = ctx->ntot;
    a.nmat = g.nmat;
    a.coef = field == 0 ? ctx->cE : ctx->cH;
    a.R = ctx->Rall[field == 0 ? 0 : 1];
    a.nR = (int)ctx->Rhost[0].size();
    a.form = g.pml_formulation;
    a.planeflag = ctx->planeflag;
    memcpy(a.box, ctx->box, sizeof(a.box));
    a.frame = ctx->frame;
    a.nframe = ctx->nframe;
    a.iterations = g.iterations;
    a.nslab = (int)ctx->slabs.size();
    for (int s = 0; s < a.nslab; ++s) fill_slab_args(ctx, field, s, a.slab[s]);
    lds = (size_t)g.nmat * 20 + (size_t)a.nR * 4;
    if (field == 0) {
        a.src0 = {ctx->src[GPX_SRC_VOLTAGE].n, ctx->src[GPX_SRC_VOLTAGE].info, ctx->src[GPX_SRC_VOLTAGE].fac, ctx->src[GPX_SRC_VOLTAGE].waves};
        a.src1 = {ctx->src[GPX_SRC_HERTZIAN].n, ctx->src[GPX_SRC_HERTZIAN].info, ctx->src[GPX_SRC_HERTZIAN].fac, ctx->src[GPX_SRC_HERTZIAN].waves};
        const int P = g.maxpoles;
        if (P > 0) {
            a.disp = ctx->disp;
            a.dispflag = ctx->dispflag;
            fill_targs(ctx, a.T);
            lds += (size_t)g.nmat * 3 * P * 4 * (ctx->disp_complex ? 2 : 1) + g.nmat;
        }
    } else {
        a.src0 = {ctx->src[GPX_SRC_MAGNETIC].n, ctx->src[GPX_SRC_MAGNETIC].info, ctx->src[GPX_SRC_MAGNETIC].fac, ctx->src[GPX_SRC_MAGNETIC].waves};
        a.nrx = ctx->nrx;
        a.rxc = ctx->rxc;
        a.rxbuf = ctx->rxbuf;
    }
}

typedef void (*pass_kernel)(StepArgs);

static hipError_t launch_kernel(const gpx_ctx *ctx, pass_kernel kernel, bool bnd, int field, int flags, int it,
                                hipStream_t stream = nullptr)
{
    StepArgs a;
    int block, grid;
    size_t lds;
    base_args(ctx, field, a, block, lds);
    if (count_items(ctx, bnd, block, 1, nullptr) <= 0) return hipSuccess;
    const int fill = resident_blocks(ctx, (const void *)kernel, block, lds);
    plan(ctx, bnd, block, a, grid, fill);   // one block per item
    a.flags = flags;
    a.it = it;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), lds, stream ? stream : ctx->stream, a);
    return hipGetLastError();
}

template <class IDT, bool BND>
static pass_kernel e_kernel(int P, bool C)
{
    switch (P) {
    case 0: return k_e_pass<IDT, 0, false, BND>;
    case 1: return C ? k_e_pass<IDT, 1, true, BND> : k_e_pass<IDT, 1, false, BND>;
    case 2: return C ? k_e_pass<IDT, 2, true, BND> : k_e_pass<IDT, 2, false, BND>;
    case 3: return C ? k_e_pass<IDT, 3, true, BND> : k_e_pass<IDT, 3, false, BND>;
    default: return C ? k_e_pass<IDT, 4, true, BND> : k_e_pass<IDT, 4, false, BND>;
    }
}

template <bool BND>
static pass_kernel pick_kernel(const gpx_ctx *ctx, int field)
{
    if (field == 1)
        return k_h_pass<uint16_t, BND>;
    const int P = ctx->desc.maxpoles;
    const bool C = ctx->disp_complex != 0;
    return e_kernel<uint16_t, BND>(P, C);
}

typedef void (*many_kernel)(const StepArgs *, PassMany);

template <class IDT, bool BND>
static many_kernel e_many(int P, bool C)
{
    switch (P) {
    case 0: return k_e_pass_many<IDT, 0, false, BND>;
    case 1: return C ? k_e_pass_many<IDT, 1, true, BND> : k_e_pass_many<IDT, 1, false, BND>;
    case 2: return C ? k_e_pass_many<IDT, 2, true, BND> : k_e_pass_many<IDT, 2, false, BND>;
    case 3: return C ? k_e_pass_many<IDT, 3, true, BND> : k_e_pass_many<IDT, 3, false, BND>;
    default: return C ? k_e_pass_many<IDT, 4, true, BND> : k_e_pass_many<IDT, 4, false, BND>;
    }
}

template <bool BND>
static many_kernel pick_many(const gpx_ctx *ctx, int field)
{
    if (field == 1)
        return k_h_pass_many<uint16_t, BND>;
    const int P = ctx->desc.maxpoles;
    const bool C = ctx->disp_complex != 0;
    return e_many<uint16_t, BND>(P, C);
}

// One pass = interior kernel (skipped when only PML work is asked for) then
// boundary kernel; they touch disjoint cells.  With `ev`, an event is recorded
// before, between and after the two launches.
static hipError_t launch_pass(const gpx_ctx *ctx, int field, int flags, int it, hipEvent_t *ev = nullptr)
{
    hipError_t e;
    if (ev && (e = hipEventRecord(ev[0], ctx->stream)) != hipSuccess) return e;
    if (flags & ~F_PML_ALL) {
        e = launch_kernel(ctx, pick_kernel<false>(ctx, field), false, field, flags & ~F_PML_ALL, it);
        if (e != hipSuccess) return e;
    }
    if (ev && (e = hipEventRecord(ev[1], ctx->stream)) != hipSuccess) return e;
    e = launch_kernel(ctx, pick_kernel<true>(ctx, field), true, field, flags, it);
    if (e != hipSuccess) return e;
    if (ev) e = hipEventRecord(ev[2], ctx->stream);
    return e;
}

// The second stream and its fork and join events, made on first use.
static hipError_t ensure_stream2(gpx_ctx *ctx)
{
    hipError_t e;
    if (!ctx->stream2 && (e = hipStreamCreateWithFlags(&ctx->stream2, hipStreamNonBlocking)) != hipSuccess) return e;
    if (!ctx->ev_fork && (e = hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming)) != hipSuccess) return e;
    if (!ctx->ev_join && (e = hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming)) != hipSuccess) return e;
    return hipSuccess;
}

// The same pass with the interior and boundary kernels running side by side,
// the boundary kernel on the second stream, each with one block per item.
// Both read only the other field and write disjoint cells of their own.
static hipError_t launch_pass_overlap(gpx_ctx *ctx, int field, int flags, int it)
{
    hipError_t e;
    if ((e = ensure_stream2(ctx)) != hipSuccess) return e;
    const bool interior = ctx->box[0] < ctx->box[1] && ctx->box[2] < ctx->box[3] && ctx->box[4] < ctx->box[5];
    if ((e = hipEventRecord(ctx->ev_fork, ctx->stream)) != hipSuccess) return e;
    if ((e = hipStreamWaitEvent(ctx->stream2, ctx->ev_fork, 0)) != hipSuccess) return e;
    if (interior && flags) {
        e = launch_kernel(ctx, pick_kernel<false>(ctx, field), false, field, flags & ~F_PML_ALL, it, ctx->stream);
        if (e != hipSuccess) return e;
    }
    e = launch_kernel(ctx, pick_kernel<true>(ctx, field), true, field, flags, it, ctx->stream2);
    if (e != hipSuccess) return e;
    if ((e = hipEventRecord(ctx->ev_join, ctx->stream2)) != hipSuccess) return e;
    return hipStreamWaitEvent(ctx->stream, ctx->ev_join, 0);
}

// ---------------------------------------------------------------- row kernels
// The row kernels are compiled in step_*.hip, one file per PML form.
namespace gpx {
RowKernels row_kernel_plain(int P, bool C, bool hu, bool big);
RowKernels row_kernel_hori1(int P, bool C, bool hu, bool big);
RowKernels row_kernel_hori2(int P, bool C, bool hu, bool big);
RowKernels row_kernel_mri1(int P, bool C, bool hu, bool big);
RowKernels row_kernel_mri2(int P, bool C, bool hu, bool big);
}  // namespace gpx

static bool big_state(const gpx_ctx *ctx) { return past_offsets((double)ctx->fstride); }

// PML order shared by every slab, 0 without slabs, -1 when they differ.
static int slab_order(const gpx_ctx *ctx)
{
    int o = 0;
    for (const Slab &S : ctx->slabs) {
        if (o && S.order != o) return -1;
        o = S.order;
    }
    return o;
}

static RowKernels row_kernels(const gpx_ctx *ctx)
{
    const int P = ctx->desc.maxpoles;
    const bool C = ctx->disp_complex != 0, hu = ctx->hu, big = big_state(ctx);
    const int o = slab_order(ctx);
    if (o <= 0) return row_kernel_plain(P, C, hu, big);
    if (ctx->desc.pml_formulation == 0) return o == 1 ? row_kernel_hori1(P, C, hu, big) : row_kernel_hori2(P, C, hu, big);
    return o == 1 ? row_kernel_mri1(P, C, hu, big) : row_kernel_mri2(P, C, hu, big);
}

// Floats of dispersive coefficients and of one field's profile tables.
static int disp_floats(const gpx_ctx *ctx)
{
    return ctx->desc.maxpoles > 0 ? ctx->desc.nmat * 3 * ctx->desc.maxpoles * (ctx->disp_complex ? 2 : 1) : 0;
}
static int profile_floats(const gpx_ctx *ctx)
{
    int n = 0;
    const int o = slab_order(ctx);
    for (const Slab &S : ctx->slabs) n += S.t * row_entry(ctx->desc.pml_formulation, o);
    return n;
}

// Floats of a field's tables, and dynamic LDS of the one-launch step with
// blocks of B threads and of a pass.
static int image_floats(const gpx_ctx *ctx, int field)
{
    return field == 0 ? row_image(ctx->desc.nmat, profile_floats(ctx), disp_floats(ctx))
                      : row_image(ctx->hu ? 0 : ctx->desc.nmat, profile_floats(ctx), 0);
}
static size_t step_lds(const gpx_ctx *ctx, int B)
{
    return (size_t)(image_floats(ctx, 0) + image_floats(ctx, 1)) * 4 + (size_t)B * (NC * 16 + 8);
}
static size_t pass_lds(const gpx_ctx *ctx, int field) { return (size_t)image_floats(ctx, field) * 4 + 16; }

// Models the row kernels take: rows of whole lanes, one PML order for all
// slabs, slabs given in the order x0, y0, z0, xmax, ymax, zmax (the kernels
// apply them so; any may be missing) that do not overlap the one opposite, with
// cell sizes row_quot takes, 32-bit byte offsets into the Phi arrays and, with
// poles, into a whole state, and tables that leave room in LDS.  Others take
// the general passes.
static bool rows_ok(const gpx_ctx *ctx)
{
    const int o = slab_order(ctx);
    if (ctx->kp % NC != 0 || o < 0 || (big_state(ctx) && ctx->desc.maxpoles > 0)) return false;
    double np = 0;
    int before = -1, end[2][3];
    for (auto &f : end)
        for (int &e : f) e = -1;
    for (size_t s = 0; s < ctx->slabs.size(); ++s) {
        const Slab &S = ctx->slabs[s];
        if (S.dir <= before || !(S.d > 1e-12f && S.d < 1.6e7f)) return false;
        before = S.dir;
        np += (double)S.ni * S.nj * S.nkp;
        for (int f = 0; f < 2; ++f) {
            SlabArgs a;
            fill_slab_args(ctx, f, (int)s, a);
            const int u = a.axis == 2 ? NC : 1;   // nor share a lane
            int &e = end[f][a.axis];
            if (a.lo[a.axis] / u < e) return false;
            e = (a.hi[a.axis] + u - 1) / u;
        }
    }
    if (np * 8.0 * (o > 0 ? o : 1) >= 2147483647.0) return false;
    return pass_lds(ctx, 0) <= (size_t)MAX_LDS_BYTES && pass_lds(ctx, 1) <= (size_t)MAX_LDS_BYTES;
}

// Threads per block of the one-launch step: 0 when it cannot run.
static int step_block(const gpx_ctx *ctx)
{
    if (!rows_ok(ctx) || big_state(ctx) || !ctx->tls.empty()) return 0;
    auto ok = [&](int B) { return B >= 128 && B <= ROW_BLOCK_MAX && step_lds(ctx, B) <= (size_t)MAX_LDS_BYTES; };
    if (ctx->fused == 1 && ctx->tile_cells) return ok(ctx->tile_cells / NC) ? ctx->tile_cells / NC : 0;
    for (int B : {ROW_BLOCK_MAX, 256, 128})
        if (ok(B)) return B;
    return 0;
}

// Lanes at the start and at the end of a row with a cell in a z slab.
static void z_lanes(const gpx_ctx *ctx, int &za, int &zb)
{
    const int lpr = ctx->kp / NC;
    za = zb = 0;
    for (size_t s = 0; s < ctx->slabs.size(); ++s)
        for (int f = 0; f < 2; ++f) {
            SlabArgs a;
            fill_slab_args(ctx, f, (int)s, a);
            if (ctx->slabs[s].dir == 2) za = std::max(za, (a.hi[2] + NC - 1) / NC);
            if (ctx->slabs[s].dir == 5) zb = std::max(zb, lpr - a.lo[2] / NC);
        }
    if (za + zb > lpr) zb = lpr - za;
}

// Tiles and x chunks of the one-launch step with blocks of B threads.
static void row_tiles(const gpx_ctx *ctx, int B, int xchunk, RowModel &m)
{
    const int lpr = ctx->kp / NC, ny1 = ctx->desc.ny + 1, nx1 = ctx->desc.nx + 1;
    // Rows longer than ROW_LANES_MAX lanes are split, each part with one lane
    // of the part before it.
    // Short enough that two rows fit with the z lanes apart.
    const int most = std::min((B - 63) / 2, ROW_LANES_MAX);
    m.ntk = lpr <= most ? 1 : (lpr + most - 2) / (most - 1);
    m.hk = m.ntk > 1;
    m.LTo = (lpr + m.ntk - 1) / m.ntk;
    m.LT = m.LTo + m.hk;
    z_lanes(ctx, m.za, m.zb);
    // in lanes of the first and of the last part, the lanes past a row's start
    // and end among them
    const int last = lpr - (m.ntk - 1) * m.LTo + m.hk;
    m.za = std::min(m.za + m.hk, m.LT);
    m.zb = std::min(m.zb, last - m.hk) + m.LT - last;
    if (m.ntk == 1) m.zb = std::min(m.zb, m.LT - m.za);
    // rows: as many as fit with the z lanes from a whole wave on
    auto need = [&](int R) {
        int most_t = 0;
        for (int tk : {0, 1, m.ntk - 1}) {
            if (tk >= m.ntk) continue;
            const int z = (tk == 0 ? m.za : 0) + (tk == m.ntk - 1 ? m.zb : 0);
            most_t = std::max(most_t, (R * (m.LT - z) + 63) / 64 * 64 + R * z);
        }
        return most_t;
    };
    m.R = B / m.LT;
    while (m.R > 1 && need(m.R) > B) --m.R;
    if (m.R >= ny1) {  // the plane in one row of tiles
        m.R = m.Ro = ny1;
        m.hj = 0;
    } else {
        m.hj = 1;
        m.Ro = m.R - 1;
    }
    m.ntj = (ny1 + m.Ro - 1) / m.Ro;
    m.xc = xchunk < 1 ? 1 : (xchunk > nx1 ? nx1 : xchunk);
    m.nitems = m.ntk * m.ntj * ((nx1 + m.xc - 1) / m.xc);
    m.threads = (need(m.R) + 63) / 64 * 64;
}

static int resident_blocks(const gpx_ctx *ctx, const void *kernel, int block, size_t lds);

// The launch shape of the one-launch step.
static void plan_step(const gpx_ctx *ctx, RowModel &m, int &B)
{
    B = step_block(ctx);
    int xc = ctx->xchunk ? ctx->xchunk : 4;
    row_tiles(ctx, B, xc, m);
    // Small grids: shorter chunks (a chunk also computes H of the plane before
    // it) and smaller blocks, until the items fill the GPU.
    const int fill = 2 * (ctx->cus > 0 ? ctx->cus : 256);
    const bool fixed = ctx->fused == 1 && ctx->tile_cells;
    while (!fixed && B > 128 && m.nitems < fill && 2 * m.LT <= B / 2) row_tiles(ctx, B /= 2, xc, m);
    while (!ctx->xchunk && xc > 2 && m.nitems < fill) row_tiles(ctx, B, --xc, m);
    if (m.threads < B && !fixed) B = m.threads;  // no idle waves
}

// One slab for the row kernels, and its profile entries (row_corr's order).
static void row_slab_args(const gpx_ctx *ctx, int field, int s, RowSlab &r)
{
    SlabArgs a;
    fill_slab_args(ctx, field, s, a);
    r.pend = a.pend;
    r.sign = a.minus ? -1 : 1;
    r.t = a.t;
    memcpy(r.lo, a.lo, sizeof(r.lo));
    memcpy(r.hi, a.hi, sizeof(r.hi));
    r.off = a.off;
    r.sx = a.sx;
    r.sy = a.sy;
    r.d = a.d;
    r.rd = (float)(1.0 / (double)a.d);
    r.rl = (float)(1.0 / (double)a.d - (double)r.rd);
    r.rt = 0;
}

static void row_profile(const gpx_ctx *ctx, int field, int s, float *out)
{
    const Slab &S = ctx->slabs[s];
    const int t = S.t, form = ctx->desc.pml_formulation, ne = row_entry(form, S.order), ot = S.order * t;
    const float *R = S.R[field].data();
    for (int p = 0; p < t; ++p) {
        float *e = out + (size_t)p * ne;
        for (int n = 0; n < ne; ++n) e[n] = 0.f;
        const float A0 = R[p], B0 = R[ot + p], E0 = R[2 * ot + p], F0 = R[3 * ot + p];
        if (S.order == 1) {
            if (form == 0) {
                e[0] = A0 - 1.0f; e[1] = B0; e[2] = E0; e[3] = F0;
            } else {
                const float IRA = 1.0f / A0;
                e[0] = IRA - 1.0f; e[1] = IRA; e[2] = E0; e[3] = IRA * B0 * F0;
            }
            continue;
        }
        const float A1 = R[t + p], B1 = R[ot + t + p], E1 = R[2 * ot + t + p], F1 = R[3 * ot + t + p];
        if (form == 0) {
            e[0] = A0 * A1 - 1.0f; e[1] = A1 * B0; e[2] = B1; e[3] = A0; e[4] = B0; e[5] = E0; e[6] = F0; e[7] = E1; e[8] = F1;
        } else {
            const float IRA = 1.0f / (A0 + A1);
            e[0] = IRA - 1.0f; e[1] = IRA; e[2] = B0; e[3] = B1; e[4] = E0; e[5] = E1; e[6] = IRA * F0; e[7] = IRA * F1;
        }
    }
}

static hipError_t upload_rare(gpx_ctx *ctx);

// Threads per block of the row passes.
static int pass_block(const gpx_ctx *ctx)
{
    const int b = ctx->block ? ctx->block : 256;
    return b < ROW_PASS_MAX ? b : ROW_PASS_MAX;
}

// Items of the row passes: one lane per NC cells, blocks of B lanes of a plane,
// chunks of xc planes.  Chunks are short: a longer one re-reads fewer planes
// of the field it differences along x, but that plane is still in the
// last-level cache, and the longer the chunks the fewer blocks there are and the
// longer each one's chain of planes (300x300x200, HORIPML, us per iteration: 353
// in chunks of 1, 349 of 2, 350 of 4, 377 of 10; 100x100x100: 23.1, 22.5, 27.7).
// The dispersive E pass, with its auxiliary values, has more to wait for per
// plane and gains from keeping H of the plane before in registers (240x240x180,
// 3 poles: 360, 331, 326 in chunks of 1, 2, 4).
static void pass_items(const gpx_ctx *ctx, int B, int xc, RowModel &m)
{
    const int lanes = (ctx->desc.ny + 1) * (ctx->kp / NC), nx1 = ctx->desc.nx + 1;
    m.pxc = xc > nx1 ? nx1 : xc;
    m.pseg = (lanes + B - 1) / B;
    m.pitems = m.pseg * ((nx1 + m.pxc - 1) / m.pxc);
}
static int pass_chunk(const gpx_ctx *ctx) { return ctx->desc.maxpoles > 0 ? 4 : 2; }
// Below this many items shorter chunks: blocks for every compute unit four times over (a
// 120x105 2-D model: 8.6 us per iteration in chunks of 1, 11.4 of 2, 16.8 of 4).
static int pass_fill(const gpx_ctx *ctx) { return 4 * (ctx->cus > 0 ? ctx->cus : 256); }

// Brings the device's description of the model up to date (waits when it has
// changed).
static int ensure_row(gpx_ctx *ctx)
{
    if (ctx->phi_dirty) return fail(ctx, GPX_ESTATE, "slabs without Phi arrays");   // check_ready lays them out
    if (ctx->rare_dirty || !ctx->rare) GPX_TRY(upload_rare(ctx));
    if (!ctx->row_dirty) return 0;
    const gpx_desc &g = ctx->desc;
    const int o = slab_order(ctx);
    // the tables as they lie in LDS, and the slabs
    RowModel &m = ctx->rowh;
    memset(&m, 0, sizeof(m));
    const int nRT = profile_floats(ctx), nE = image_floats(ctx, 0), nH = image_floats(ctx, 1);
    std::vector<float> img((size_t)nE + nH, 0.f);
    for (int f = 0; f < 2; ++f) {
        const std::vector<float> &c = f ? ctx->hostH : ctx->hostE;
        const int nm = f && ctx->hu ? 0 : g.nmat;
        float *at = img.data() + (f ? nE : 0), *rt = at + 4 * nm, *sl = rt + nRT, *c5 = sl;
        if (nRT) c5 += 6 * sizeof(RowSlab) / 4;
        for (int n = 0; n < nm; ++n) {
            memcpy(at + 4 * n, &c[5 * (size_t)n], 16);
            c5[n] = c[5 * (size_t)n + 4];
        }
        if (!f && g.maxpoles > 0) memcpy(c5 + nm, ctx->hostdisp.data(), ctx->hostdisp.size() * 4);
        int first = 0;
        for (size_t s = 0; s < ctx->slabs.size(); ++s) {
            const int dir = ctx->slabs[s].dir;
            RowSlab d;
            row_slab_args(ctx, f, (int)s, d);
            d.rt = first;
            memcpy(sl + dir * (sizeof(RowSlab) / 4), &d, sizeof(d));
            const RowAt w = {d.lo[1], d.hi[1], d.lo[2], d.hi[2], d.off, d.sx, d.sy, 0};
            (f ? m.atH : m.atE)[dir] = w;
            row_profile(ctx, f, (int)s, rt + first);
            first += ctx->slabs[s].t * row_entry(g.pml_formulation, o);
        }
    }
    if (nE + nH > ctx->nimg) {
        if (ctx->img) hipFree(ctx->img);
        ctx->img = nullptr;
        ctx->nimg = 0;
        GPX_TRY(dalloc(ctx, (void **)&ctx->img, img.size() * 4, false));
        ctx->nimg = nE + nH;
    }
    if (int rc = copy_in(ctx, ctx->img, img.data(), img.size() * 4)) return rc;
    m.nx = g.nx; m.ny = g.ny; m.nz = g.nz;
    m.kp = ctx->kp;
    m.plane = ctx->plane;
    int B = 0;
    if (step_block(ctx)) plan_step(ctx, m, B);
    ctx->row_block = B;
    int xc = ctx->xchunk ? ctx->xchunk : pass_chunk(ctx);
    pass_items(ctx, pass_block(ctx), xc, m);
    while (!ctx->xchunk && xc > 1 && m.pitems < pass_fill(ctx)) pass_items(ctx, pass_block(ctx), --xc, m);
    m.F[0] = ctx->Fmem[0];
    m.F[1] = ctx->Fmem[1];
    m.cs = (uint32_t)(ctx->fstride * 4);
    m.ci = (uint32_t)(ctx->ntot * 2);
    m.csl = (size_t)ctx->fstride * 4;
    m.cil = (size_t)ctx->ntot * 2;
    m.ID = ctx->ID;
    m.img = reinterpret_cast<const float4 *>(ctx->img);
    m.n4E = nE / 4;
    m.n4H = nH / 4;
    m.nmat = g.nmat;
    for (int n = 0; n < 5 && ctx->hu; ++n) m.h[n] = ctx->hostH[n];
    m.nRT = nRT;
    m.phiE[0] = ctx->phiE[0];
    m.phiE[1] = ctx->phiE[1];
    m.phiH[0] = ctx->phiH[0];
    m.phiH[1] = ctx->phiH[1];
    m.np4 = (uint32_t)(ctx->np * 4);
    if (g.maxpoles > 0) fill_targs(ctx, m.T);
    m.iterations = g.iterations;
    m.rare = ctx->rare;
    m.planeflag = ctx->planeflag + g.nx + 1;
    if (!ctx->row) GPX_TRY(dalloc(ctx, (void **)&ctx->row, sizeof(RowModel), false));
    if (int rc = copy_in(ctx, ctx->row, &m, sizeof(m))) return rc;
    ctx->row_dirty = false;
    return 0;
}

static RowArgs row_args(const gpx_ctx *ctx, int nitems, int it)
{
    RowArgs b;
    b.item0 = nullptr;
    b.ntr = 1;
    b.nitems = nitems;
    b.per_xcd = (nitems + 7) / 8;
    b.flip = ctx->cur;
    b.flipE = ctx->curE;
    b.it = it;
    b.p0 = 0;
    b.p1 = ctx->desc.nx + 1;
    return b;
}

// One iteration in one launch; then the next state is the current one.
static hipError_t launch_row_step(gpx_ctx *ctx, int it)
{
    const RowArgs b = row_args(ctx, ctx->rowh.nitems, it);
    hipLaunchKernelGGL(row_kernels(ctx).step, dim3(8 * b.per_xcd), dim3(ctx->row_block), step_lds(ctx, ctx->row_block),
                       ctx->stream, ctx->row, b);
    ctx->cur ^= 1;
    return hipGetLastError();
}

// The H (field 1) or E pass over planes [p0, p1), in one launch.
static hipError_t launch_row_pass(const gpx_ctx *ctx, int field, int it, int p0, int p1)
{
    const RowModel &m = ctx->rowh;
    RowArgs b = row_args(ctx, m.pseg * ((p1 - p0 + m.pxc - 1) / m.pxc), it);
    b.p0 = p0;
    b.p1 = p1;
    const RowKernels k = row_kernels(ctx);
    hipLaunchKernelGGL(field == 1 ? k.h : k.e, dim3(8 * b.per_xcd), dim3(pass_block(ctx)), pass_lds(ctx, field),
                       ctx->stream, ctx->row, b);
    return hipGetLastError();
}

// ---------------------------------------------------------------- 2-D models
// Tiles of the 2-D kernel (gpx_plane.h); w: the axis of one cell, -1 when it
// cannot run the model.
struct PlaneShape {
    int w, tp, tq, halo;
};

// The axis of one cell, when the 2-D kernel can run the model: what it leaves out
// is zero and stays so.  No state has been uploaded, sources lie (and lay) on the
// plane's cells and drive its components, slabs lie across the two long axes
// and every coefficient is finite.  -1 otherwise.
static int plane_axis(const gpx_ctx *ctx)
{
    const gpx_desc &g = ctx->desc;
    const int dim[3] = {g.nx, g.ny, g.nz};
    int w = -1;
    for (int q = 0; q < 3; ++q)
        if (dim[q] == 1) {
            if (w >= 0) return -1;
            w = q;
        }
    if (w < 0 || g.maxpoles > 0 || ctx->state_given || !ctx->tls.empty() || !rows_ok(ctx) || big_state(ctx)) return -1;
    auto finite = [](const std::vector<float> &x) {
        return std::all_of(x.begin(), x.end(), [](float v) { return isfinite(v); });
    };
    if (!finite(ctx->hostE) || !finite(ctx->hostH)) return -1;
    for (const Slab &S : ctx->slabs)
        if (S.dir % 3 == w || !finite(S.R[0]) || !finite(S.R[1])) return -1;
    for (int kind : {GPX_SRC_MAGNETIC, GPX_SRC_VOLTAGE, GPX_SRC_HERTZIAN})
        for (int s = 0; s < ctx->src[kind].n; ++s) {
            const int *in = &ctx->src[kind].host[6 * s];
            if (in[w] != 0 || ((in[3] & 3) == w) != (kind != GPX_SRC_MAGNETIC)) return -1;
        }
    return w;
}

// Tiles for a run of n iterations: the shape that takes the least time by what
// launches of several shapes took, 5.5 us + 0.7 us for each wave a SIMD is
// given + for each iteration 0.25 us a wave, 0.5 at the least.  Measured, us per iteration
// (columns of a tile, halo): 120x105 1.98 (16x16, 4), 1.75 (16x32, 6), 1.90 (32x32,
// 8), the passes 9.0; 250x180 2.48, 2.93, 1.90, 9.0; 500x500 7.0, 8.6, 6.5, 4.8
// (32x32, 4), 11.8; 1200x1000 27, 35, 23, 17.0 (32x32, 4), 35.
static PlaneShape plane_shape(const gpx_ctx *ctx, int n)
{
    PlaneShape best = {plane_axis(ctx), 0, 0, 0};
    if (best.w < 0) return best;
    const gpx_desc &g = ctx->desc;
    const int np = best.w == 0 ? g.ny : g.nx, nq = best.w == 2 ? g.ny : g.nz, cus = ctx->cus > 0 ? ctx->cus : 256;
    const int tiles[3][2] = {{16, 16}, {16, 32}, {32, 32}};
    double least = 0;
    for (auto &t : tiles)
        for (int h = 1; 2 * h + 4 <= t[0] && (h <= n || h == 1); ++h) {
            const int op = t[0] - 2 * h, oq = t[1] - 2 * h;
            const double blocks = (double)((np + op) / op) * ((nq + oq) / oq);
            const double waves = ceil(blocks / cus) * t[0] * t[1] / 256;
            const double us = (5.5 + 0.7 * waves + h * std::max(0.5, 0.25 * waves)) / h;
            if (best.halo && us >= least) continue;
            least = us;
            best = {best.w, t[0], t[1], h};
        }
    return best;
}

// Iterations [it, it + n), n at most the halo, in one launch.
static hipError_t launch_plane(gpx_ctx *ctx, const PlaneShape &s, int it, int n)
{
    const gpx_desc &g = ctx->desc;
    PlaneArgs b;
    b.flip = ctx->cur;
    b.flipE = ctx->curE;
    b.it = it;
    b.n = n;
    b.w = s.w;
    b.tp = s.tp;
    b.tq = s.tq;
    b.halo = s.halo;
    b.hu = ctx->hu;
    const int op = s.tp - 2 * s.halo, oq = s.tq - 2 * s.halo;
    const int np = s.w == 0 ? g.ny : g.nx, nq = s.w == 2 ? g.ny : g.nz;
    b.ntq = (nq + oq) / oq;
    b.nitems = (np + op) / op * b.ntq;
    b.per_xcd = (b.nitems + 7) / 8;
    const int B = s.tp * s.tq;
    hipLaunchKernelGGL(row_kernels(ctx).plane, dim3(8 * b.per_xcd), dim3(B), (size_t)B * 12, ctx->stream, ctx->row, b);
    ctx->cur ^= 1;
    ctx->curE ^= ctx->slabs.empty() ? 0 : 1;
    return hipGetLastError();
}

// Copies the source and receiver tables of the row kernels to the device.
static hipError_t upload_rare(gpx_ctx *ctx)
{
    if (!ctx->rare) {
        hipError_t e = dalloc(ctx, (void **)&ctx->rare, sizeof(StepRare), false);
        if (e != hipSuccess) return e;
        ctx->row_dirty = true;
    }
    StepRare r;
    memset(&r, 0, sizeof(r));
    auto src = [&](int kind) {
        const SrcSet &S = ctx->src[kind];
        return SrcArgs{S.n, S.info, S.fac, S.waves};
    };
    r.srcM = src(GPX_SRC_MAGNETIC);
    r.srcV = src(GPX_SRC_VOLTAGE);
    r.srcD = src(GPX_SRC_HERTZIAN);
    r.nrx = ctx->nrx;
    r.rxc = ctx->rxc;
    r.rxbuf = ctx->rxbuf;
    hipError_t e = hipMemcpyAsync(ctx->rare, &r, sizeof(r), hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e == hipSuccess) ctx->rare_dirty = false;
    return e;
}

// ---------------------------------------------------------------- step forms
// Models forms 3, 5 and 7 are reported for: no dispersive poles, no lines, and
// a 3-D grid with an interior.
static bool split_eligible(const gpx_ctx *ctx)
{
    return ctx->desc.maxpoles == 0 && ctx->deep && step_block(ctx) > 0;
}

// The rule of form 4: models without slabs and poles take the one-launch step,
// which reads and writes 54 bytes a cell where the two passes take 78; in the
// slabs its chain of dependent work per plane (H, a barrier, E) costs more than
// that saves (300x300x200: 386 us an iteration against 349 with 10 cells of PML
// on each side, 285 against 300 without).
static bool one_launch(const gpx_ctx *ctx)
{
    return ctx->slabs.empty() && ctx->desc.maxpoles == 0 && step_block(ctx) > 0;
}

// What gpx_run does with the model: STEP (one launch), PASSES (two row
// passes), PLANE (several iterations of a 2-D model a launch), GENERAL (the
// general passes), BESIDE (form 2).
enum RunKind { RUN_STEP, RUN_PASSES, RUN_PLANE, RUN_GENERAL, RUN_BESIDE };

static RunKind run_kind(const gpx_ctx *ctx)
{
    const RunKind passes = rows_ok(ctx) ? RUN_PASSES : RUN_GENERAL;
    switch (ctx->fused) {
    case 1: return step_block(ctx) ? RUN_STEP : passes;
    case 2: return RUN_BESIDE;
    case 0: case 6: return passes;
    default: return plane_axis(ctx) >= 0 ? RUN_PLANE : (one_launch(ctx) ? RUN_STEP : passes);   // 3, 5, 7 and 4
    }
}

static hipError_t launch_snapshot(const gpx_ctx *ctx, int s)
{
    const Snap &S = ctx->snaps[s];
    const long long n = (long long)S.snx * S.sny * S.snz;
    const int block = 256;
    const int grid = (int)((n + block - 1) / block);
    hipLaunchKernelGGL(k_snapshot, dim3(grid), dim3(block), 0, ctx->stream, ctx->desc.ny, ctx->kp,
                       S.xs, S.ys, S.zs, S.dx, S.dy, S.dz, S.snx, S.sny, S.snz, ctx->field(0),
                       ctx->field(1), ctx->field(2), ctx->field(3), ctx->field(4), ctx->field(5), S.out);
    return hipGetLastError();
}

// The transmission-line kernel after the H pass (field 1) or the E pass.
static hipError_t launch_tl(const gpx_ctx *ctx, int field, int it)
{
    const int n = (int)ctx->tls.size();
    if (!n) return hipSuccess;
    const int B = 64, grid = (n + B - 1) / B;
    const gpx_desc &g = ctx->desc;
    if (field == 1)
        hipLaunchKernelGGL(k_tl_h, dim3(grid), dim3(B), 0, ctx->stream, ctx->tldev, n, it, g.ny, ctx->kp,
                           ctx->field(3), ctx->field(4), ctx->field(5));
    else
        hipLaunchKernelGGL(k_tl_e, dim3(grid), dim3(B), 0, ctx->stream, ctx->tldev, n, it, g.ny, ctx->kp,
                           ctx->field(0), ctx->field(1), ctx->field(2));
    return hipGetLastError();
}

// Cases the line kernels cannot order as the reference does: the line
// reads H after the PML and before magnetic dipoles, and sets E after
// voltage sources, before Hertzian dipoles and dispersive part B.
static int check_tls(gpx_ctx *ctx)
{
    if (ctx->tls.empty()) return 0;
    if (ctx->desc.maxpoles > 0)
        return fail(ctx, GPX_EARG, "transmission lines in a model with dispersive materials are not supported");
    for (const TLine &t : ctx->tls) {
        const TLDev &L = t.d;
        // (component 0..2 = Hx..Hz, cell) pairs the line's current reads
        int reads[4][4];
        if (L.pol == 0) {
            const int r[4][4] = {{1, L.i, L.j, L.k - 1}, {1, L.i, L.j, L.k}, {2, L.i, L.j, L.k}, {2, L.i, L.j - 1, L.k}};
            memcpy(reads, r, sizeof(r));
        } else if (L.pol == 1) {
            const int r[4][4] = {{0, L.i, L.j, L.k}, {0, L.i, L.j, L.k - 1}, {2, L.i - 1, L.j, L.k}, {2, L.i, L.j, L.k}};
            memcpy(reads, r, sizeof(r));
        } else {
            const int r[4][4] = {{0, L.i, L.j - 1, L.k}, {0, L.i, L.j, L.k}, {1, L.i, L.j, L.k}, {1, L.i - 1, L.j, L.k}};
            memcpy(reads, r, sizeof(r));
        }
        const SrcSet &M = ctx->src[GPX_SRC_MAGNETIC], &D = ctx->src[GPX_SRC_HERTZIAN];
        for (int s = 0; s < M.n; ++s) {
            const int *in = &M.host[6 * s];
            for (auto &r : reads)
                if (in[3] == r[0] && in[0] == r[1] && in[1] == r[2] && in[2] == r[3])
                    return fail(ctx, GPX_EARG, "a magnetic dipole on an H component a transmission line reads");
        }
        for (int s = 0; s < D.n; ++s) {
            const int *in = &D.host[6 * s];
            if (in[3] == L.pol && in[0] == L.i && in[1] == L.j && in[2] == L.k)
                return fail(ctx, GPX_EARG, "a Hertzian dipole on the edge of a transmission line");
        }
    }
    return 0;
}

static int plane_axis(const gpx_ctx *ctx);

// Called before anything steps a model: once a 2-D model is stepped with what the
// 2-D kernel leaves out (a source of another component, say), that may stay
// behind in the state, and later runs take the passes too.
static void note_state(gpx_ctx *ctx)
{
    if (plane_axis(ctx) < 0) ctx->state_given = true;
}

static int check_ready(gpx_ctx *ctx)
{
    if (!ctx->have_id || !ctx->have_coeffs)
        return fail(ctx, GPX_ESTATE, "ID and coefficient tables must be uploaded before stepping");
    if (ctx->desc.maxpoles > 0 && !ctx->have_disp)
        return fail(ctx, GPX_ESTATE, "dispersive coefficients must be uploaded before stepping");
    if (int rc = ensure_tslots(ctx)) return rc;
    if (int rc = ensure_planes(ctx)) return rc;
    if (int rc = ensure_phi(ctx)) return rc;
    note_state(ctx);
    return check_tls(ctx);
}

static int h_flags(const gpx_ctx *ctx)
{
    int f = F_MAIN | F_SRC | (ctx->nrx ? F_RX : 0);
    for (size_t s = 0; s < ctx->slabs.size(); ++s) f |= F_PML0 << s;
    return f;
}

static int e_flags(const gpx_ctx *ctx)
{
    int f = F_MAIN | F_SRC | (ctx->desc.maxpoles ? F_DISPB : 0);
    for (size_t s = 0; s < ctx->slabs.size(); ++s) f |= F_PML0 << s;
    return f;
}

// Bytes that an iteration of the row passes goes over, each array once.
static double pass_bytes(const gpx_ctx *ctx)
{
    double b = (double)ctx->fstride * 24.0 + (double)ctx->ntot * 2.0 * (ctx->hu ? 3 : 6);
    if (!ctx->slabs.empty()) b += 2.0 * (double)phi_bytes(ctx);
    if (ctx->desc.maxpoles > 0) {
        b += (double)ctx->ntot / 2;
        for (int c = 0; c < 3; ++c) b += (double)ctx->tn[c] * ctx->desc.maxpoles * (ctx->disp_complex ? 8 : 4);
    }
    return b;
}

// Blocks of planes of run_wave: as few as keep a block within WAVE_BYTES, every
// one more being a launch of 5 us per pass beside its bytes.  The last-level
// cache has 256 MB; a block moves through the planes, and past about 200 it evicts itself
// between the passes.  A grid that fits whole, up to WHOLE_BYTES, is not divided.  us per
// iteration in 1, 2, 3, ... blocks (MiB of a block in brackets where fastest):
// 300x300x200 348, 335, 296, 275 (at 3: 199), 283 ...; 250x220x180 179, 146 (168), 161;
// 611x407x45 247, 226, 200 (146), 209; 420x400x200 612, 629, 606, 604, 567, 519
// (182), 520 at 7, 570 at 13; 240x240x180 with 3 poles 320, 323, 294 (199), 299.
// Around the whole cache: 196 MiB 76, 91; 216 82, 96; 236 90, 105; 248 119, 109; 256
// 124, 110; 315 159, 132.
static const double WAVE_BYTES = 200.0 * 1024 * 1024, WHOLE_BYTES = 240.0 * 1024 * 1024;
// Iterations a block is taken through: 300x300x200 takes 357 us an iteration at
// 1, 316 at 2, 290 at 4, 280 at 8, 276 at 16 and 278 at 32.  At one iteration whole passes
// are the faster ones (347).
static const int WAVE_ITS = 16;
static int wave_blocks(const gpx_ctx *ctx)
{
    const double bytes = pass_bytes(ctx), n = bytes <= WHOLE_BYTES ? 1.0 : ceil(bytes / WAVE_BYTES);
    return n < (double)(ctx->desc.nx + 1) ? (int)n : ctx->desc.nx + 1;
}

// The row passes of iterations [it, it + n) in blocks of planes, each block
// taken through all of them before the next one is begun, so that what its
// first pass brings into the last-level cache serves the others too.  A block's
// planes move down by one with each iteration: iteration s of the block that
// begins at plane a covers planes [a - s, a - s + w).  New H at plane i needs E
// of the iteration before at i and i + 1, which the block has just made up to
// a - s + w; new E at i needs this iteration's H at i and i - 1, and the block
// before ended at a - s - 1.  Every cell sees the same values in the same order
// as in whole passes.  On grids past the cache whole passes run at the rate of
// the memory (4.7 of about 5 TB/s), the blocks at that of the cache (6.5 of 8).
static int run_wave(gpx_ctx *ctx, int it, int n, int blocks)
{
    const int nx1 = ctx->desc.nx + 1, w = (nx1 + n - 1 + blocks - 1) / blocks;
    for (int a = 0; a < nx1 + n - 1; a += w)
        for (int s = 0; s < n; ++s) {
            const int p0 = std::max(a - s, 0), p1 = std::min(a - s + w, nx1);
            if (p0 >= p1) continue;
            GPX_TRY(launch_row_pass(ctx, 1, it + s, p0, p1));
            GPX_TRY(launch_row_pass(ctx, 0, it + s, p0, p1));
        }
    return 0;
}

// Timing events, destroyed when the set goes out of scope.
struct EventSet {
    std::vector<hipEvent_t> e;
    ~EventSet()
    {
        for (hipEvent_t x : e)
            if (x) hipEventDestroy(x);
    }
};

// Runs iterations [it0, it0+n) in the step form set by gpx_set_step.  With
// `ms4`, events around every kernel give the mean duration of each kernel of
// an iteration over the run: the one-launch step in ms4[0] (the rest 0); the
// row passes in ms4[0] and ms4[2]; or H interior, H boundary, E interior and
// E boundary of the general passes.  Form 4 reports its rule's form from its
// first run of at least CHOOSE_ITS iterations on (gpx_step_choice).
static const int CHOOSE_ITS = 26;

static int run_steps(gpx_ctx *ctx, int it0, int n, float *ms4)
{
    if (!ms4 && ctx->fused == 4 && ctx->choice == -1 && n >= CHOOSE_ITS)
        ctx->choice = one_launch(ctx) ? 5 : 4;
    const int hf = h_flags(ctx), ef = e_flags(ctx);
    RunKind kind = run_kind(ctx);
    if (ms4 && kind == RUN_PLANE) kind = RUN_PASSES;   // the kernels of each iteration are timed
    const bool rows = kind == RUN_STEP || kind == RUN_PASSES || kind == RUN_PLANE;
    if (n > 0 && kind == RUN_STEP)
        if (int rc = ensure_next_state(ctx)) return rc;
    if (n > 0 && kind == RUN_PLANE)
        if (int rc = ensure_next_plane(ctx)) return rc;
    const PlaneShape shape = kind == RUN_PLANE ? plane_shape(ctx, n) : PlaneShape{-1, 0, 0, 0};
    if (n > 0 && rows)
        if (int rc = ensure_row(ctx)) return rc;
    const int waves = kind == RUN_PASSES && !ms4 && ctx->tls.empty() ? wave_blocks(ctx) : 1;
    // With ms4, six events per iteration are recorded around the kernels and
    // read once at the end, so the host never waits between iterations and
    // the gaps between events are the kernels' own.
    const int per = 6;
    EventSet evs;
    if (ms4) {
        evs.e.assign((size_t)(n > 0 ? n : 0) * per, nullptr);
        for (auto &e : evs.e) GPX_TRY(hipEventCreate(&e));
    }
    for (int it = it0; it < it0 + n; ++it) {
        hipEvent_t *ev = ms4 ? &evs.e[(size_t)(it - it0) * per] : nullptr;
        for (size_t s = 0; s < ctx->snaps.size(); ++s)
            if (ctx->snaps[s].time == it + 1) GPX_TRY(launch_snapshot(ctx, (int)s));
        if (kind == RUN_STEP) {
            if (ev) GPX_TRY(hipEventRecord(ev[0], ctx->stream));
            GPX_TRY(launch_row_step(ctx, it));
            if (ev) GPX_TRY(hipEventRecord(ev[1], ctx->stream));
            continue;
        }
        if (waves > 1 || kind == RUN_PLANE) {
            // up to the next iteration that a snapshot is taken before
            int end = std::min(it0 + n, it + (kind == RUN_PLANE ? shape.halo : WAVE_ITS));
            for (const Snap &S : ctx->snaps)
                if (S.time - 1 > it && S.time - 1 < end) end = S.time - 1;
            if (kind == RUN_PLANE) GPX_TRY(launch_plane(ctx, shape, it, end - it));
            else if (int rc = run_wave(ctx, it, end - it, end - it > 1 ? waves : 1)) return rc;
            it = end - 1;
            continue;
        }
        if (kind == RUN_PASSES) {
            // events: the H pass between ev[0] and ev[1], the E pass between
            // ev[3] and ev[4]
            if (ev) GPX_TRY(hipEventRecord(ev[0], ctx->stream));
            GPX_TRY(launch_row_pass(ctx, 1, it, 0, ctx->desc.nx + 1));
            if (ev) GPX_TRY(hipEventRecord(ev[1], ctx->stream));
            GPX_TRY(launch_tl(ctx, 1, it));
            if (ev) GPX_TRY(hipEventRecord(ev[3], ctx->stream));
            GPX_TRY(launch_row_pass(ctx, 0, it, 0, ctx->desc.nx + 1));
            if (ev) GPX_TRY(hipEventRecord(ev[4], ctx->stream));
            GPX_TRY(launch_tl(ctx, 0, it));
            continue;
        }
        if (kind == RUN_BESIDE && !ms4) {
            GPX_TRY(launch_pass_overlap(ctx, 1, hf, it));
            GPX_TRY(launch_tl(ctx, 1, it));
            GPX_TRY(launch_pass_overlap(ctx, 0, ef, it));
            GPX_TRY(launch_tl(ctx, 0, it));
            continue;
        }
        GPX_TRY(launch_pass(ctx, 1, hf, it, ev));
        GPX_TRY(launch_tl(ctx, 1, it));
        GPX_TRY(launch_pass(ctx, 0, ef, it, ev ? ev + 3 : nullptr));
        GPX_TRY(launch_tl(ctx, 0, it));
    }
    if (ms4) {
        double acc[4] = {0, 0, 0, 0};
        GPX_TRY(hipStreamSynchronize(ctx->stream));
        // (begin, end) event pairs of each kernel slot: the step; the row
        // passes; H interior, H boundary, E interior, E boundary
        static const int pairs[3][4][2] = {{{0, 1}, {-1, -1}, {-1, -1}, {-1, -1}},
                                           {{0, 1}, {-1, -1}, {3, 4}, {-1, -1}},
                                           {{0, 1}, {1, 2}, {3, 4}, {4, 5}}};
        const int form = kind == RUN_STEP ? 0 : (kind == RUN_PASSES ? 1 : 2);
        for (int i = 0; i < n; ++i) {
            hipEvent_t *ev = &evs.e[(size_t)i * per];
            for (int q = 0; q < 4; ++q) {
                const int a = pairs[form][q][0], b = pairs[form][q][1];
                if (a < 0) continue;
                float t;
                GPX_TRY(hipEventElapsedTime(&t, ev[a], ev[b]));
                acc[q] += t;
            }
        }
        for (int q = 0; q < 4; ++q) ms4[q] = (float)(acc[q] / (n > 0 ? n : 1));
    }
    return 0;
}

extern "C" int gpx_step_kind(const gpx_ctx *ctx)
{
    return ctx && ctx->fused == 1 ? step_block(ctx) * NC : 0;
}

extern "C" int gpx_step_form(const gpx_ctx *ctx)
{
    if (!ctx) return GPX_EARG;
    switch (ctx->fused) {
    case 1: return step_block(ctx) ? 1 : 0;
    case 2: case 6: return ctx->fused;
    case 3: case 5: case 7: return split_eligible(ctx) ? ctx->fused : 0;
    case 4: return ctx->choice == 5 ? 7 : (ctx->choice == 4 ? 6 : (split_eligible(ctx) ? 3 : 0));
    default: return 0;
    }
}

extern "C" int gpx_step_choice(const gpx_ctx *ctx)
{
    if (!ctx) return GPX_EARG;
    return ctx->choice;
}

extern "C" int gpx_run(gpx_ctx *ctx, int it0, int n)
{
    if (!ctx || it0 < 0 || n < 0 || it0 + n > ctx->desc.iterations)
        return fail(ctx, GPX_EARG, "gpx_run: iteration range outside [0, iterations)");
    if (int rc = check_ready(ctx)) return rc;
    hipSetDevice(ctx->desc.device);
    return run_steps(ctx, it0, n, nullptr);
}

extern "C" int gpx_run_timed(gpx_ctx *ctx, int it0, int n, int per_kernel, float *ms_total,
                             float *ms_h, float *ms_e)
{
    if (!ctx || it0 < 0 || n < 0 || it0 + n > ctx->desc.iterations)
        return fail(ctx, GPX_EARG, "gpx_run_timed: iteration range outside [0, iterations)");
    if (int rc = check_ready(ctx)) return rc;
    hipSetDevice(ctx->desc.device);
    hipEvent_t a, b;
    GPX_TRY(hipEventCreate(&a));
    GPX_TRY(hipEventCreate(&b));
    GPX_TRY(hipEventRecord(a, ctx->stream));
    float ms4[4] = {0, 0, 0, 0};
    int rc = run_steps(ctx, it0, n, per_kernel ? ms4 : nullptr);
    if (rc) return rc;
    if (per_kernel) {
        if (ms_h) *ms_h = ms4[0] + ms4[1];
        if (ms_e) *ms_e = ms4[2] + ms4[3];
    }
    GPX_TRY(hipEventRecord(b, ctx->stream));
    GPX_TRY(hipEventSynchronize(b));
    float ms = 0;
    GPX_TRY(hipEventElapsedTime(&ms, a, b));
    hipEventDestroy(a);
    hipEventDestroy(b);
    if (ms_total) *ms_total = ms;
    return 0;
}

extern "C" int gpx_run_profiled(gpx_ctx *ctx, int it0, int n, float *ms4)
{
    if (!ctx || !ms4 || it0 < 0 || n < 1 || it0 + n > ctx->desc.iterations)
        return fail(ctx, GPX_EARG, "gpx_run_profiled: bad argument");
    if (int rc = check_ready(ctx)) return rc;
    hipSetDevice(ctx->desc.device);
    return run_steps(ctx, it0, n, ms4);
}

extern "C" int gpx_part(gpx_ctx *ctx, int part, int arg, int it)
{
    if (!ctx) return fail(ctx, GPX_EARG, "gpx_part: null ctx");
    if (it < 0 || it >= ctx->desc.iterations) return fail(ctx, GPX_EARG, "gpx_part: iteration out of range");
    if (int rc = check_ready(ctx)) return rc;
    hipSetDevice(ctx->desc.device);
    const int ns = (int)ctx->slabs.size();
    switch (part) {
    case GPX_PART_STORE_RX:
        if (ctx->nrx) GPX_TRY(launch_pass(ctx, 1, F_RX, it));
        return 0;
    case GPX_PART_SNAPSHOT:
        if (arg < 0 || arg >= (int)ctx->snaps.size()) return fail(ctx, GPX_EARG, "gpx_part: bad snapshot index");
        GPX_TRY(launch_snapshot(ctx, arg));
        return 0;
    case GPX_PART_H_MAIN: GPX_TRY(launch_pass(ctx, 1, F_MAIN, it)); return 0;
    case GPX_PART_H_SRC: GPX_TRY(launch_pass(ctx, 1, F_SRC, it)); return 0;
    case GPX_PART_E_MAIN: GPX_TRY(launch_pass(ctx, 0, F_MAIN, it)); return 0;
    case GPX_PART_E_SRC: GPX_TRY(launch_pass(ctx, 0, F_SRC, it)); return 0;
    case GPX_PART_E_DISP_B:
        if (ctx->desc.maxpoles) GPX_TRY(launch_pass(ctx, 0, F_DISPB, it));
        return 0;
    case GPX_PART_H_PML:
    case GPX_PART_E_PML:
        if (arg < 0 || arg >= ns) return fail(ctx, GPX_EARG, "gpx_part: bad slab index");
        GPX_TRY(launch_pass(ctx, part == GPX_PART_H_PML ? 1 : 0, F_PML0 << arg, it));
        return 0;
    default: return fail(ctx, GPX_EARG, "gpx_part: unknown part");
    }
}

extern "C" int gpx_synchronize(gpx_ctx *ctx)
{
    if (!ctx) return fail(ctx, GPX_EARG, "gpx_synchronize: null ctx");
    GPX_TRY(hipStreamSynchronize(ctx->stream));
    return 0;
}

extern "C" int gpx_download_rx(gpx_ctx *ctx, float *out)
{
    if (!ctx || !out) return fail(ctx, GPX_EARG, "gpx_download_rx: null argument");
    if (!ctx->nrx) return 0;
    return copy_out(ctx, out, ctx->rxbuf, (size_t)6 * ctx->desc.iterations * ctx->nrx * 4);
}

// Fields and Phi go between the reference's layout on the host and the device's
// padded rows through dense pieces on the device, which a kernel packs or
// unpacks: with the rows copied one by one on the host the fields of 300x300x200
// took 139 ms down and 115 up, now 41 and 14, the copies of 437 MB alone about
// as long.  `work` launches the kernel for values [first, first + n) of `total`.
template <class Fn>
static int staged(gpx_ctx *ctx, float *host, size_t total, bool up, const Fn &work)
{
    hipSetDevice(ctx->desc.device);
    const size_t want = std::min(total, STAGE_FLOATS);
    if (ctx->nstage < want) {
        if (ctx->stage) hipFree(ctx->stage);
        ctx->stage = nullptr;
        ctx->nstage = 0;
        GPX_TRY(hipMalloc((void **)&ctx->stage, want * 4));
        ctx->nstage = want;
    }
    for (size_t q = 0; q < total; q += ctx->nstage) {
        const size_t n = std::min(total - q, ctx->nstage);
        if (up) GPX_TRY(hipMemcpyAsync(ctx->stage, host + q, n * 4, hipMemcpyHostToDevice, ctx->stream));
        work(q, n, dim3((unsigned)((n + 255) / 256)), dim3(256));
        GPX_TRY(hipGetLastError());
        if (!up) GPX_TRY(hipMemcpyAsync(host + q, ctx->stage, n * 4, hipMemcpyDeviceToHost, ctx->stream));
    }
    GPX_TRY(hipStreamSynchronize(ctx->stream));
    return 0;
}

// Values [first, first + n) of the six components, `rows` rows of nk each, to
// dense from a state (rows of kp, fstride floats a component), or (up) from there
// into one or two.
struct RowsPlace {
    size_t pts, fstride;
    uint32_t nk, kp;
};
__global__ void k_rows_dense(float *a, float *b, float *dense, size_t first, size_t n, RowsPlace p, bool up)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const size_t q = first + t, c = q / p.pts;
    const uint32_t e = (uint32_t)(q - c * p.pts), r = e / p.nk;   // fewer than 2^30 points
    const size_t at = c * p.fstride + (size_t)r * p.kp + (e - r * p.nk);
    if (up) {
        a[at] = dense[t];
        if (b) b[at] = dense[t];
    } else {
        dense[t] = a[at];
    }
}

// The fields down, or (up) into both states where there are two: cells that no
// update touches keep their value in either.
static int fields_transfer(gpx_ctx *ctx, float *host, bool up)
{
    const gpx_desc &g = ctx->desc;
    RowsPlace p;
    p.pts = (size_t)(g.nx + 1) * (g.ny + 1) * (g.nz + 1);
    p.fstride = (size_t)ctx->fstride;
    p.nk = (uint32_t)g.nz + 1;
    p.kp = (uint32_t)ctx->kp;
    float *one = ctx->Fmem[ctx->cur], *two = ctx->Fmem[ctx->cur ^ 1];
    if (p.nk == p.kp) {   // whole rows
        for (int c = 0; c < 6; ++c)
            for (float *m : {one, two}) {
                if (!m || (!up && m == two)) continue;
                float *dev = m + (size_t)c * p.fstride, *h = host + (size_t)c * p.pts;
                if (int rc = up ? copy_in(ctx, dev, h, p.pts * 4) : copy_out(ctx, h, dev, p.pts * 4)) return rc;
            }
        return 0;
    }
    return staged(ctx, host, 6 * p.pts, up, [&](size_t first, size_t n, dim3 G, dim3 B) {
        hipLaunchKernelGGL(k_rows_dense, G, B, 0, ctx->stream, one, two, ctx->stage, first, n, p, up);
    });
}

extern "C" int gpx_download_fields(gpx_ctx *ctx, float *out6)
{
    if (!ctx || !out6) return fail(ctx, GPX_EARG, "gpx_download_fields: null argument");
    return fields_transfer(ctx, out6, false);
}

extern "C" int gpx_upload_fields(gpx_ctx *ctx, const float *in6)
{
    if (!ctx || !in6) return fail(ctx, GPX_EARG, "gpx_upload_fields: null argument");
    ctx->state_given = true;
    return fields_transfer(ctx, const_cast<float *>(in6), true);
}

// Values [first, first + n) of a slab's Phi in the reference's layout,
// [order][d0][d1][d2], to dense or (up) from there into two arrays.  flip: the
// axis that the reference runs backwards (-1: none), of t cells.
struct PhiPlace {
    int d0, d1, d2, flip, t, nj, nkp, kofs;
    size_t at, ostep;        // of the slab's term of order 0, and from order to order
};
__global__ void k_phi_dense(float *a, float *b, float *dense, size_t first, size_t n, PhiPlace p, bool up)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    size_t q = first + t;
    int c[3];
    c[2] = (int)(q % p.d2);
    q /= p.d2;
    c[1] = (int)(q % p.d1);
    q /= p.d1;
    c[0] = (int)(q % p.d0);
    const size_t o = q / p.d0;
#pragma unroll
    for (int x = 0; x < 3; ++x)
        if (x == p.flip && c[x] < p.t) c[x] = p.t - 1 - c[x];
    const size_t at = p.at + o * p.ostep + ((size_t)c[0] * p.nj + c[1]) * p.nkp + c[2] + p.kofs;
    if (up) {
        a[at] = dense[t];
        if (b) b[at] = dense[t];
    } else {
        dense[t] = a[at];
    }
}

// Phi `which` (EPhi1, EPhi2, HPhi1, HPhi2) of a slab between the reference's
// layout on the host and the device's (see Slab); both copies go up.
static int phi_transfer(gpx_ctx *ctx, int slab, int which, float *host, bool up)
{
    const Slab &S = ctx->slabs[slab];
    const int field = which < 2 ? 0 : 1;
    SlabArgs a;
    fill_slab_args(ctx, field, slab, a);
    const long long *d = S.dims[which];
    PhiPlace p;
    p.d0 = (int)d[0]; p.d1 = (int)d[1]; p.d2 = (int)d[2];
    p.flip = S.dir < 3 ? S.dir : -1;
    p.t = S.t;
    p.nj = S.nj;
    p.nkp = S.nkp;
    p.kofs = a.lo[2] & 3;
    p.at = (size_t)(which & 1) * ctx->np + S.base;
    p.ostep = (size_t)2 * ctx->np;
    float *one = field == 0 ? ctx->phiE[ctx->curE] : ctx->phiH[ctx->cur],
          *two = field == 0 ? ctx->phiE[ctx->curE ^ 1] : ctx->phiH[ctx->cur ^ 1];
    return staged(ctx, host, (size_t)S.order * d[0] * d[1] * d[2], up, [&](size_t first, size_t n, dim3 G, dim3 B) {
        hipLaunchKernelGGL(k_phi_dense, G, B, 0, ctx->stream, one, two, ctx->stage, first, n, p, up);
    });
}

static int phi_check(gpx_ctx *ctx, int slab, int which)
{
    if (slab < 0 || slab >= (int)ctx->slabs.size() || which < 0 || which > 3)
        return fail(ctx, GPX_EARG, "bad slab or Phi index");
    return ensure_phi(ctx);
}

extern "C" int gpx_download_pml_phi(gpx_ctx *ctx, int slab, int which, float *out)
{
    if (!ctx || !out) return fail(ctx, GPX_EARG, "gpx_download_pml_phi: null argument");
    if (int rc = phi_check(ctx, slab, which)) return rc;
    return phi_transfer(ctx, slab, which, out, false);
}

extern "C" int gpx_upload_pml_phi(gpx_ctx *ctx, int slab, int which, const float *in)
{
    if (!ctx || !in) return fail(ctx, GPX_EARG, "gpx_upload_pml_phi: null argument");
    if (int rc = phi_check(ctx, slab, which)) return rc;
    ctx->state_given = true;
    return phi_transfer(ctx, slab, which, const_cast<float *>(in), true);
}

// T in the reference's layout, complex64 [3][P][ntot]; edges without poles
// hold no auxiliary values here and read back as zero.
extern "C" int gpx_download_dispersive_T(gpx_ctx *ctx, float *out)
{
    if (!ctx || !out) return fail(ctx, GPX_EARG, "gpx_download_dispersive_T: null argument");
    const int P = ctx->desc.maxpoles;
    if (!P) return fail(ctx, GPX_ESTATE, "gpx_download_dispersive_T: no dispersive state");
    if (int rc = ensure_tslots(ctx)) return rc;
    if (ctx->tslot_dirty || !ctx->T[0]) return fail(ctx, GPX_ESTATE, "gpx_download_dispersive_T: no dispersive state");
    const size_t N = (size_t)ctx->ntot, w = ctx->disp_complex ? 2 : 1;
    const size_t nk = (size_t)ctx->desc.nz + 1, kp = (size_t)ctx->kp, pts = N / kp * nk;
    std::fill(out, out + (size_t)3 * P * pts * 2, 0.0f);
    std::vector<uint32_t> slot(N);
    for (int c = 0; c < 3; ++c) {
        const size_t n = (size_t)ctx->tn[c];
        std::vector<float> t((size_t)P * (n ? n : 1) * w);
        if (int rc = copy_out(ctx, slot.data(), ctx->tslot[c], N * 4)) return rc;
        if (int rc = copy_out(ctx, t.data(), ctx->T[c], t.size() * 4)) return rc;
        for (size_t r = 0; r < N / kp; ++r)
            for (size_t k = 0; k < nk; ++k) {   // (a row's padding left out)
                const uint32_t s = slot[r * kp + k];
                if (s == 0xffffffffu) continue;  // no poles
                const size_t h = r * nk + k;
                for (int p = 0; p < P; ++p) {
                    float *o = out + (((size_t)c * P + p) * pts + h) * 2;
                    o[0] = t[((size_t)p * n + s) * w];
                    if (w == 2) o[1] = t[((size_t)p * n + s) * w + 1];
                }
            }
    }
    return 0;
}

extern "C" int gpx_upload_dispersive_T(gpx_ctx *ctx, const float *in)
{
    if (!ctx || !in) return fail(ctx, GPX_EARG, "gpx_upload_dispersive_T: null argument");
    const int P = ctx->desc.maxpoles;
    if (!P) return fail(ctx, GPX_ESTATE, "gpx_upload_dispersive_T: no dispersive state");
    if (int rc = ensure_tslots(ctx)) return rc;
    if (ctx->tslot_dirty || !ctx->T[0])
        return fail(ctx, GPX_ESTATE, "gpx_upload_dispersive_T: upload the indices and dispersive tables first");
    const size_t N = (size_t)ctx->ntot, w = ctx->disp_complex ? 2 : 1;
    const size_t nk = (size_t)ctx->desc.nz + 1, kp = (size_t)ctx->kp, pts = N / kp * nk;
    std::vector<uint32_t> slot(N);
    for (int c = 0; c < 3; ++c) {
        const size_t n = (size_t)ctx->tn[c];
        std::vector<float> t((size_t)P * (n ? n : 1) * w, 0.0f);
        if (int rc = copy_out(ctx, slot.data(), ctx->tslot[c], N * 4)) return rc;
        for (size_t r = 0; r < N / kp; ++r)
            for (size_t k = 0; k < nk; ++k) {
                const uint32_t s = slot[r * kp + k];
                if (s == 0xffffffffu) continue;
                const size_t h = r * nk + k;
                for (int p = 0; p < P; ++p) {
                    const float *v = in + (((size_t)c * P + p) * pts + h) * 2;
                    if (w == 1 && v[1] != 0.0f)
                        return fail(ctx, GPX_EARG, "gpx_upload_dispersive_T: imaginary part in a real-pole model");
                    t[((size_t)p * n + s) * w] = v[0];
                    if (w == 2) t[((size_t)p * n + s) * w + 1] = v[1];
                }
            }
        if (int rc = copy_in(ctx, ctx->T[c], t.data(), t.size() * 4)) return rc;
    }
    return 0;
}

extern "C" int gpx_download_snapshot(gpx_ctx *ctx, int index, float *out6)
{
    if (!ctx || !out6 || index < 0 || index >= (int)ctx->snaps.size())
        return fail(ctx, GPX_EARG, "gpx_download_snapshot: bad argument");
    const Snap &s = ctx->snaps[index];
    return copy_out(ctx, out6, s.out, (size_t)6 * s.snx * s.sny * s.snz * 4);
}

extern "C" int gpx_device_info(int device, char *name, int namelen, size_t *totalmem,
                               size_t *freemem, int *cus)
{
    hipDeviceProp_t prop;
    hipError_t e = hipGetDeviceProperties(&prop, device);
    if (e != hipSuccess) return fail(nullptr, (int)e, std::string("hipGetDeviceProperties: ") + hipGetErrorString(e));
    if (name && namelen > 0) {
        // Some runtimes leave the marketing name empty; the architecture and
        // the compute-unit count still name the part.
        if (prop.name[0])
            snprintf(name, (size_t)namelen, "%s (%s)", prop.name, prop.gcnArchName);
        else
            snprintf(name, (size_t)namelen, "AMD %s, %d CUs, %zu GiB", prop.gcnArchName, prop.multiProcessorCount,
                     (size_t)(prop.totalGlobalMem >> 30));
    }
    if (totalmem) *totalmem = prop.totalGlobalMem;
    if (cus) *cus = prop.multiProcessorCount;
    if (freemem) {
        size_t fr = 0, tot = 0;
        e = hipSetDevice(device);
        if (e == hipSuccess) e = hipMemGetInfo(&fr, &tot);
        if (e != hipSuccess) return fail(nullptr, (int)e, std::string("hipMemGetInfo: ") + hipGetErrorString(e));
        *freemem = fr;
    }
    return 0;
}

extern "C" int gpx_interior_box(const gpx_ctx *ctx, int *box6)
{
    if (!ctx || !box6) return GPX_EARG;
    memcpy(box6, ctx->box, sizeof(ctx->box));
    return 0;
}

extern "C" long long gpx_interior_cells(const gpx_ctx *ctx)
{
    if (!ctx) return 0;
    const int *b = ctx->box;
    if (b[1] <= b[0]) return 0;
    return (long long)(b[1] - b[0]) * (b[3] - b[2]) * (b[5] - b[4]);
}

extern "C" size_t gpx_memory_bytes(const gpx_ctx *ctx)
{
    return ctx ? ctx->bytes : 0;
}

// ====================================================================== batch
// Many models advanced together: each launch of an iteration (the two row passes or
// the one-launch step) covers the work items of every model of a group.  Each model
// keeps its own gpx_ctx (buffers, sources, receivers); the batch only holds the launch
// tables.
struct gpx_batch {
    std::vector<gpx_ctx *> ctx;
    int device = 0;
    hipStream_t stream = nullptr;
    int tile = 0, xchunk = 0;      // cells per block and chunk of the step; tile 0 = planned, in groups
    double group_bytes = 192.0 * 1024 * 1024;  // state bytes per group of models
    RowModel *dmodels = nullptr;   // [ntr]
    int *ditem0 = nullptr;         // each group's first item per model: [ntr + groups]
    StepArgs *dpass = nullptr;     // [4][ntr]: H interior, H boundary, E interior, E boundary
    int *dpitem = nullptr;         // [4][ntr + groups]: each group's first item per model
    std::string err;
};

static int bfail(gpx_batch *b, int code, const std::string &msg)
{
    if (b) b->err = msg;
    else g_err = msg;
    return code;
}

#define GPX_BTRY(call)                                                                         \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) return bfail(b, (int)e_, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

extern "C" const char *gpx_batch_last_error(const gpx_batch *b)
{
    return b ? b->err.c_str() : g_err.c_str();
}

// Whether models [g0, g0 + gn) all take the row passes with the same kernels.
static bool batch_passes(const gpx_batch *b, int g0, int gn)
{
    const RowKernels k = row_kernels(b->ctx[g0]);
    for (int t = g0; t < g0 + gn; ++t) {
        const RowKernels q = row_kernels(b->ctx[t]);
        if (!rows_ok(b->ctx[t]) || q.h != k.h || q.e != k.e) return false;
    }
    return true;
}

// Whether models [g0, g0 + gn) all take the one-launch step with one kernel.
static bool batch_rows(const gpx_batch *b, int g0, int gn)
{
    for (int t = g0; t < g0 + gn; ++t)
        if (!step_block(b->ctx[t]) || row_kernels(b->ctx[t]).step != row_kernels(b->ctx[g0]).step) return false;
    return true;
}

// Whether form 4 would take the one-launch step for all of them.
static bool batch_plain(const gpx_batch *b, int g0, int gn)
{
    for (int t = g0; t < g0 + gn; ++t)
        if (!one_launch(b->ctx[t])) return false;
    return true;
}

// Tile sizes every model of the batch accepts, smallest first.
static std::vector<int> batch_tiles(const gpx_batch *b)
{
    std::vector<int> out;
    if (!batch_rows(b, 0, (int)b->ctx.size())) return out;
    for (int tc : {256, 512, 1024}) {
        bool ok = tc / NC <= ROW_BLOCK_MAX;
        for (const gpx_ctx *c : b->ctx)
            if (step_lds(c, tc / NC) > (size_t)MAX_LDS_BYTES) ok = false;
        if (ok) out.push_back(tc);
    }
    return out;
}

extern "C" int gpx_batch_destroy(gpx_batch *b);

extern "C" int gpx_batch_create(gpx_ctx *const *ctxs, int n, gpx_batch **out)
{
    if (!ctxs || n < 1 || !out) return bfail(nullptr, GPX_EARG, "gpx_batch_create: bad argument");
    *out = nullptr;
    const gpx_ctx *c0 = ctxs[0];
    for (int t = 0; t < n; ++t) {
        gpx_ctx *c = ctxs[t];
        if (!c) return bfail(nullptr, GPX_EARG, "gpx_batch_create: null context");
        if (int rc = check_ready(c)) return bfail(nullptr, rc, "gpx_batch_create: model " + std::to_string(t) + ": " + c->err);
        if (!c->tls.empty())
            return bfail(nullptr, GPX_EARG, "gpx_batch_create: model " + std::to_string(t) + " has transmission lines");
        if (c->desc.device != c0->desc.device)
            return bfail(nullptr, GPX_EARG, "gpx_batch_create: all models must be on one device");
        if (c->desc.iterations != c0->desc.iterations)
            return bfail(nullptr, GPX_EARG, "gpx_batch_create: all models must have the same number of iterations");
        if (!c->snaps.empty())
            return bfail(nullptr, GPX_EARG, "gpx_batch_create: models with snapshots are stepped one by one");
        if (c->desc.maxpoles != c0->desc.maxpoles ||
            c->disp_complex != c0->disp_complex || c->desc.pml_formulation != c0->desc.pml_formulation)
            return bfail(nullptr, GPX_EARG, "gpx_batch_create: all models need the same kernel ("
                                            "poles and their kind, PML formulation)");
    }
    gpx_batch *b = new gpx_batch();
    b->ctx.assign(ctxs, ctxs + n);
    b->device = c0->desc.device;
    hipSetDevice(b->device);
    hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc((void **)&b->dmodels, sizeof(RowModel) * n);
    if (e == hipSuccess) e = hipMalloc((void **)&b->ditem0, sizeof(int) * 2 * n);
    if (e == hipSuccess) e = hipMalloc((void **)&b->dpass, sizeof(StepArgs) * 4 * n);
    if (e == hipSuccess) e = hipMalloc((void **)&b->dpitem, sizeof(int) * 4 * (2 * n));
    if (e != hipSuccess) {
        hipError_t e2 = e;
        gpx_batch_destroy(b);
        return bfail(nullptr, (int)e2, std::string("gpx_batch_create: ") + hipGetErrorString(e2));
    }
    *out = b;
    return 0;
}

extern "C" int gpx_batch_destroy(gpx_batch *b)
{
    if (!b) return 0;
    hipSetDevice(b->device);
    if (b->stream) hipStreamSynchronize(b->stream);
    if (b->dmodels) hipFree(b->dmodels);
    if (b->ditem0) hipFree(b->ditem0);
    if (b->dpass) hipFree(b->dpass);
    if (b->dpitem) hipFree(b->dpitem);
    if (b->stream) hipStreamDestroy(b->stream);
    delete b;
    return 0;
}

extern "C" int gpx_batch_set_shape(gpx_batch *b, int tile_cells, int xchunk)
{
    if (!b || xchunk < 0) return bfail(b, GPX_EARG, "gpx_batch_set_shape: bad argument");
    if (tile_cells) {  // 0 = planned
        const std::vector<int> ok = batch_tiles(b);
        bool found = false;
        for (int tc : ok) found = found || tc == tile_cells;
        if (!found) return bfail(b, GPX_EARG, "gpx_batch_set_shape: tile size not usable by every model");
    }
    b->tile = tile_cells;
    b->xchunk = xchunk;
    return 0;
}

// Groups.  Consecutive models whose state fits together in the 256 MB
// last-level cache (192 MB budget; a larger model is a group of its own); a
// group runs all its iterations before the next one starts, so that its state
// stays cached, as it does when the models run one by one.  A group whose
// models share their row kernels takes the two row passes, or the one-launch step
// where form 4 would; any other (different PML orders mixed, say) four general
// passes, H interior, H boundary, E interior, E boundary.  One block per item,
// the block finding its model in the table.
static const double GROUP_BYTES = 192.0 * 1024 * 1024;

extern "C" int gpx_batch_set_group_bytes(gpx_batch *b, double bytes)
{
    if (!b || !(bytes >= 0)) return bfail(b, GPX_EARG, "gpx_batch_set_group_bytes: bad argument");
    b->group_bytes = bytes > 0 ? bytes : GROUP_BYTES;
    return 0;
}

struct BatchGroup {
    int g0 = 0, gn = 0;
    enum { GENERAL, PASSES, STEP } kind = GENERAL;
    int B = 0, nitems_rows = 0;
    size_t lds_rows[2] = {0, 0};        // of the E pass or the step, of the H pass
    size_t off_rows = 0;                // of the group's item0 table in ditem0
    int nitems[4] = {0, 0, 0, 0}, grid[4] = {0, 0, 0, 0};
    size_t lds[4] = {0, 0, 0, 0};
    size_t item_off[4] = {0, 0, 0, 0};  // of the group's item0 table in dpitem
};

struct BatchPlan {
    many_kernel k[4] = {nullptr, nullptr, nullptr, nullptr};
    std::vector<BatchGroup> groups;
    int B = 256;
    int xc = 0;                          // of the last group with one launch per iteration
};

// A group of one model (a model larger than the group budget, or the last one
// left) shares its launches with nothing, so it runs as a plain solve of
// that model instead: run_steps with the model's own step form, on the
// model's stream, ordered after the batch stream's earlier work and before its
// later work.  The step forms give the same bits as the passes.
static bool group_alone(const BatchGroup &g) { return g.gn == 1; }

// Tiles and chunks of a group's models for the one-launch step (blocks of `tile`
// cells, 0: chosen) or the row passes, with chunks of xchunk planes (0: chosen).
static int batch_plan_rows(gpx_batch *b, int tile, int xchunk, BatchGroup &g, std::vector<RowModel> &models, int &xc)
{
    int cus = 256;
    for (int t = g.g0; t < g.g0 + g.gn; ++t) {
        gpx_ctx *c = b->ctx[t];
        if (g.kind == BatchGroup::STEP)
            if (int rc = ensure_next_state(c)) return bfail(b, rc, "gpx_batch: " + c->err);
        if (int rc = ensure_row(c)) return bfail(b, rc, "gpx_batch: " + c->err);
        models[t] = c->rowh;
        if (c->cur) {  // launch parity 0 reads the current state
            std::swap(models[t].F[0], models[t].F[1]);
            std::swap(models[t].phiH[0], models[t].phiH[1]);
        }
        if (c->curE) std::swap(models[t].phiE[0], models[t].phiE[1]);
        if (c->cus > 0) cus = c->cus;
    }
    if (g.kind == BatchGroup::PASSES) {
        g.B = 256;
        xc = xchunk ? xchunk : pass_chunk(b->ctx[g.g0]);
        for (;; --xc) {
            g.nitems_rows = 0;
            for (int t = g.g0; t < g.g0 + g.gn; ++t) {
                pass_items(b->ctx[t], g.B, xc, models[t]);
                g.nitems_rows += models[t].pitems;
            }
            if (xchunk || xc <= 1 || g.nitems_rows >= pass_fill(b->ctx[g.g0])) break;
        }
        for (int f = 0; f < 2; ++f)
            for (int t = g.g0; t < g.g0 + g.gn; ++t) g.lds_rows[f] = std::max(g.lds_rows[f], pass_lds(b->ctx[t], f));
        return 0;
    }
    int B = tile ? tile / NC : ROW_BLOCK_MAX;
    auto fits = [&](int block) {
        for (int t = g.g0; t < g.g0 + g.gn; ++t)
            if (step_lds(b->ctx[t], block) > (size_t)MAX_LDS_BYTES) return false;
        return true;
    };
    while (!tile && B > 128 && !fits(B)) B /= 2;
    auto items = [&](int block, int chunk) {
        int n = 0;
        for (int t = g.g0; t < g.g0 + g.gn; ++t) {
            row_tiles(b->ctx[t], block, chunk, models[t]);
            n += models[t].nitems;
        }
        return n;
    };
    xc = xchunk ? xchunk : 4;
    int n = items(B, xc);
    while (!tile && B > 128 && n < 2 * cus) n = items(B /= 2, xc);
    while (!xchunk && xc > 2 && n < 2 * cus) n = items(B, --xc);
    g.B = B;
    g.nitems_rows = n;
    for (int t = g.g0; t < g.g0 + g.gn; ++t) g.lds_rows[0] = std::max(g.lds_rows[0], step_lds(b->ctx[t], B));
    return 0;
}

// Launch tables.  tile 0: groups; else one group of every model with blocks
// of `tile` cells.
static int batch_prepare(gpx_batch *b, int tile, int xchunk, BatchPlan &p)
{
    const int n = (int)b->ctx.size();
    for (int kind = 0; kind < 4; ++kind)
        p.k[kind] = (kind & 1) ? pick_many<true>(b->ctx[0], kind < 2 ? 1 : 0)
                               : pick_many<false>(b->ctx[0], kind < 2 ? 1 : 0);
    // greedy groups in model order
    p.groups.clear();
    double acc = 0;
    for (int t = 0; t < n; ++t) {
        const gpx_ctx *c = b->ctx[t];
        const double bytes = (double)(c->bytes - c->next_bytes);
        if (p.groups.empty() || (!tile && acc + bytes > b->group_bytes)) {
            p.groups.push_back(BatchGroup());
            p.groups.back().g0 = t;
            acc = 0;
        }
        p.groups.back().gn++;
        acc += bytes;
    }
    const int G = (int)p.groups.size();
    std::vector<StepArgs> args(4 * (size_t)n);
    std::vector<RowModel> models(n);
    std::vector<int> item0(4 * (size_t)(n + G), 0), ritem0((size_t)n + G, 0);
    hipSetDevice(b->device);
    for (gpx_ctx *c : b->ctx)   // slabs, sources, receivers or tables may be new since the batch was made
        if (int rc = check_ready(c)) return bfail(b, rc, "gpx_batch: " + c->err);
    for (int gi = 0; gi < G; ++gi) {
        BatchGroup &g = p.groups[gi];
        if (!tile && group_alone(g)) continue;
        if (batch_rows(b, g.g0, g.gn) && (tile || batch_plain(b, g.g0, g.gn))) g.kind = BatchGroup::STEP;
        else if (batch_passes(b, g.g0, g.gn)) g.kind = BatchGroup::PASSES;
        if (g.kind != BatchGroup::GENERAL) {
            if (int rc = batch_plan_rows(b, tile, xchunk, g, models, p.xc)) return rc;
            g.off_rows = (size_t)g.g0 + gi;
            for (int t = 0; t < g.gn; ++t)
                ritem0[g.off_rows + t + 1] = ritem0[g.off_rows + t] + (g.kind == BatchGroup::STEP ? models[g.g0 + t].nitems
                                                                                                  : models[g.g0 + t].pitems);
            continue;
        }
        for (int kind = 0; kind < 4; ++kind) {
            const int field = kind < 2 ? 1 : 0;
            const bool bnd = kind & 1;
            g.item_off[kind] = (size_t)kind * (n + G) + g.g0 + gi;
            int *i0 = &item0[g.item_off[kind]];
            for (int t = 0; t < g.gn; ++t) {
                gpx_ctx *c = b->ctx[g.g0 + t];
                StepArgs &a = args[(size_t)kind * n + g.g0 + t];
                int block, grid;
                size_t lds;
                base_args(c, field, a, block, lds);
                plan(c, bnd, p.B, a, grid);
                const int f = field == 1 ? h_flags(c) : e_flags(c);
                a.flags = bnd ? f : f & ~F_PML_ALL;
                a.it = 0;
                if (lds > g.lds[kind]) g.lds[kind] = lds;
                i0[t + 1] = i0[t] + a.nitems;
            }
            g.nitems[kind] = i0[g.gn];
            g.grid[kind] = (g.nitems[kind] + 7) / 8 * 8;
        }
    }
    GPX_BTRY(hipMemcpyAsync(b->dpass, args.data(), args.size() * sizeof(StepArgs), hipMemcpyHostToDevice, b->stream));
    GPX_BTRY(hipMemcpyAsync(b->dpitem, item0.data(), item0.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
    GPX_BTRY(hipMemcpyAsync(b->dmodels, models.data(), models.size() * sizeof(RowModel), hipMemcpyHostToDevice, b->stream));
    GPX_BTRY(hipMemcpyAsync(b->ditem0, ritem0.data(), ritem0.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
    GPX_BTRY(hipStreamSynchronize(b->stream));
    return 0;
}

// Step s (0, 1, ...) of a run, iteration it, of one group.
static void batch_launch(const gpx_batch *b, const BatchPlan &p, const BatchGroup &g, int s, int it)
{
    const int n = (int)b->ctx.size();
    if (g.kind != BatchGroup::GENERAL) {
        const RowKernels k = row_kernels(b->ctx[g.g0]);
        RowArgs a;
        a.item0 = b->ditem0 + g.off_rows;
        a.ntr = g.gn;
        a.nitems = g.nitems_rows;
        a.per_xcd = (g.nitems_rows + 7) / 8;
        a.flip = g.kind == BatchGroup::STEP ? s & 1 : 0;
        a.flipE = 0;
        a.it = it;
        a.p0 = 0;
        a.p1 = INT_MAX;
        auto launch = [&](row_kernel f, size_t lds) {
            hipLaunchKernelGGL(f, dim3(8 * a.per_xcd), dim3(g.B), lds, b->stream, b->dmodels + g.g0, a);
        };
        if (g.kind == BatchGroup::STEP) return launch(k.step, g.lds_rows[0]);
        launch(k.h, g.lds_rows[1]);
        launch(k.e, g.lds_rows[0]);
        return;
    }
    for (int kind = 0; kind < 4; ++kind) {
        if (!g.nitems[kind]) continue;
        PassMany m;
        const StepArgs *args = b->dpass + (size_t)kind * n + g.g0;
        m.item0 = b->dpitem + g.item_off[kind];
        m.ntr = g.gn;
        m.nitems = g.nitems[kind];
        m.per_xcd = g.grid[kind] / 8;
        m.it = it;
        hipLaunchKernelGGL(p.k[kind], dim3(g.grid[kind]), dim3(p.B), g.lds[kind], b->stream, args, m);
    }
}

static int batch_steps(gpx_batch *b, const BatchPlan &p, int it0, int n, float *ms)
{
    // Work queued on the models' own streams (uploads) completes first.
    for (gpx_ctx *c : b->ctx) GPX_BTRY(hipStreamSynchronize(c->stream));
    hipEvent_t e0, e1, eb, ec;
    GPX_BTRY(hipEventCreate(&e0));
    GPX_BTRY(hipEventCreate(&e1));
    GPX_BTRY(hipEventCreateWithFlags(&eb, hipEventDisableTiming));
    GPX_BTRY(hipEventCreateWithFlags(&ec, hipEventDisableTiming));
    int rc = 0;
    auto alone = [&](const BatchGroup &g) { return group_alone(g) && g.kind == BatchGroup::GENERAL; };
    if (!rc) {
        hipError_t e = hipEventRecord(e0, b->stream);
        for (size_t gi = 0; e == hipSuccess && !rc && gi < p.groups.size(); ++gi) {
            const BatchGroup &g = p.groups[gi];
            if (alone(g)) {
                gpx_ctx *c = b->ctx[g.g0];
                e = hipEventRecord(eb, b->stream);
                if (e == hipSuccess) e = hipStreamWaitEvent(c->stream, eb, 0);
                if (e != hipSuccess) break;
                if (int r = run_steps(c, it0, n, nullptr)) {
                    rc = bfail(b, r, std::string("gpx_batch: ") + gpx_last_error(c));
                    break;
                }
                e = hipEventRecord(ec, c->stream);
                if (e == hipSuccess) e = hipStreamWaitEvent(b->stream, ec, 0);
                continue;
            }
            for (int s = 0; e == hipSuccess && s < n; ++s) {
                batch_launch(b, p, g, s, it0 + s);
                e = hipGetLastError();
            }
            if (g.kind == BatchGroup::STEP && (n & 1))
                for (int t = g.g0; t < g.g0 + g.gn; ++t) b->ctx[t]->cur ^= 1;
        }
        if (!rc) {
            if (e == hipSuccess) e = hipEventRecord(e1, b->stream);
            if (e == hipSuccess) e = hipEventSynchronize(e1);
            float t = 0;
            if (e == hipSuccess) e = hipEventElapsedTime(&t, e0, e1);
            if (e != hipSuccess) rc = bfail(b, (int)e, std::string("gpx_batch: ") + hipGetErrorString(e));
            else if (ms) *ms = t;
        }
    }
    for (gpx_ctx *c : b->ctx) hipStreamSynchronize(c->stream);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipEventDestroy(eb);
    hipEventDestroy(ec);
    return rc;
}

// `graph` is a caller's wish of old for one graph of the whole run.  A graph's
// iterations are its kernels' arguments, so it is launched once, and making it
// cost more than it saved: two models of 120x105 10.1 us an iteration on the device,
// 9.0 as a graph, two of 60^3 14.7 either way, and 7 us an iteration to make.
extern "C" int gpx_batch_run(gpx_batch *b, int it0, int n, int /*graph*/, float *ms)
{
    if (!b || it0 < 0 || n < 1 || it0 + n > b->ctx[0]->desc.iterations)
        return bfail(b, GPX_EARG, "gpx_batch_run: bad argument");
    hipSetDevice(b->device);
    BatchPlan p;
    if (int rc = batch_prepare(b, b->tile, b->xchunk, p)) return rc;
    return batch_steps(b, p, it0, n, ms);
}

// Zeroes the whole state of a model: both field copies, Phi, T and the
// receiver buffer.
static int zero_state(gpx_ctx *ctx)
{
    gpx_ctx *c = ctx;
    hipStream_t s = c->stream;
    for (float *m : c->Fmem)
        if (m) GPX_TRY(hipMemsetAsync(m, 0, (size_t)6 * c->fstride * 4, s));
    for (float *m : {c->phiE[0], c->phiE[1], c->phiH[0], c->phiH[1]})
        if (m) GPX_TRY(hipMemsetAsync(m, 0, phi_bytes(c), s));
    if (c->desc.maxpoles > 0)
        for (int q = 0; q < 3; ++q)
            if (c->T[q])
                GPX_TRY(hipMemsetAsync(c->T[q], 0, (size_t)c->desc.maxpoles * (size_t)(c->tn[q] > 0 ? c->tn[q] : 1) * 4 *
                                                       (c->disp_complex ? 2 : 1), s));
    if (c->rxbuf) GPX_TRY(hipMemsetAsync(c->rxbuf, 0, (size_t)6 * c->desc.iterations * c->nrx * 4, s));
    GPX_TRY(hipStreamSynchronize(s));
    return 0;
}

extern "C" int gpx_batch_tune(gpx_batch *b, int steps, int *tile_cells, int *xchunk, float *ms_per_step)
{
    if (!b || steps < 1 || steps > b->ctx[0]->desc.iterations) return bfail(b, GPX_EARG, "gpx_batch_tune: bad argument");
    hipSetDevice(b->device);
    float best = -1.f;
    int bt = 0, bx = 0;
    bool all_alone = true;
    {
        BatchPlan p;
        if (int rc = batch_prepare(b, 0, 0, p)) return rc;
        float ms = 0;
        if (int rc = batch_steps(b, p, 0, 1, nullptr)) return rc;  // first launch
        if (int rc = batch_prepare(b, 0, 0, p)) return rc;
        if (int rc = batch_steps(b, p, 0, steps, &ms)) return rc;
        best = ms / steps;
        for (const BatchGroup &g : p.groups) all_alone = all_alone && group_alone(g);
    }
    // Models too large to share a group each fill the GPU on their own and
    // run as plain solves; models that take the passes are slower in one launch
    // whatever its tiles (one_launch).
    for (int tc : all_alone || !batch_plain(b, 0, (int)b->ctx.size()) ? std::vector<int>() : batch_tiles(b)) {
        BatchPlan p;
        if (int rc = batch_prepare(b, tc, 0, p)) return rc;
        float ms = 0;
        if (int rc = batch_steps(b, p, 0, 1, nullptr)) return rc;  // first launch of a shape
        if (int rc = batch_prepare(b, tc, 0, p)) return rc;
        if (int rc = batch_steps(b, p, 0, steps, &ms)) return rc;
        ms /= steps;
        if (best < 0 || ms < best) {
            best = ms;
            bt = tc;
            bx = p.xc;
        }
    }
    for (gpx_ctx *c : b->ctx)
        if (int rc = zero_state(c)) return bfail(b, rc, "gpx_batch_tune: " + c->err);
    b->tile = bt;
    b->xchunk = bx;
    if (tile_cells) *tile_cells = bt;
    if (xchunk) *xchunk = bx;
    if (ms_per_step) *ms_per_step = best;
    return 0;
}
