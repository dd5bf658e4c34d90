// Row kernels of the differentiable solver: the H and E passes of its forward
// and the two halves of its adjoint (adjoint.hip states the scheme), every
// cell its own material.
//
// What bounds them.  160x160x120 (3.1 M points, 75 MB of fields) lies in the
// last-level cache apart from the stored states and the parameters: bytes set
// the time, 36 a point for H, 44 for E (56 when it stores the curl), 80 and 40
// for the adjoint's halves.  On 40^3 it is each launch's chain of accesses.
// So: two cells a lane as in gpx_rows.h, rows padded to four floats, every
// array in that layout (parameters and gradients too, 0 where a point is no
// cell), components apart; E^n is not copied to the store, the pass reads E
// there and writes E^{n+1} into the next slot; the adjoint's E half leaves lE
// alone and the H half multiplies it by CA in place, which also folds the poles'
// part of the next iteration in (k_inv_adj_h).
//
// The figures at each kernel are us per launch on 160x160x120 with 10 cells of
// PML; before, a thread had one point, lE and lH were float4 with CB and CA in
// w, and the points near a slab ran apart from the rest.  A gradient of 600
// iterations: 216 ms before, 141 now; on 40^3 with 3 poles, 150 iterations:
// 13.6 and 6.3 ms.
#ifndef GPX_INV_ROWS_H
#define GPX_INV_ROWS_H

#include "gpx_rows.h"

namespace gpx {

// One launch: arrays and the iteration.  All field arrays hold their three
// components RowModel::cs bytes apart.
struct InvStep {
    const float *E;          // forward: E^n; adjoint: the stored E^n
    float *En;               // forward: E^{n+1}
    float *H;                // H (adjoint: lH)
    float *lE;               // adjoint lE
    const float *mat;        // CA, CB, IEA
    float *curl;             // curl of H^{n+1}: stored by the forward (or null), read by the adjoint
    float *phi;              // phi^n of the poles, likewise
    const float *dc;         // ee, eqt, zt, each [P]
    float *T;                // T (adjoint: lT) of the three components, each [P]
    float *P, *Q;            // Phi of the pass's field; its adjoint read and written
    float *grad;             // dL/dCA, dL/dCB, dL/dIEA
    // Of the general kernels, receivers sorted by rows of points: [rows + 1], a row's
    // first in rxat; [receivers][2], k and number.  The row kernels': RowModel.
    const int *rxfirst, *rxat;
    const float *resid;      // [receivers][iterations]
    float *traces;
    int iterations, it;
    int si, sj, sk;
    float w, sfac;           // the source's waveform value and length factor
    float cH, DB;
    int nitems, per_xcd;
};

// Adds of one launch's slab terms in the adjoint: which slabs a lane's points
// and their neighbours (STEP +1: above, -1: below) lie in.
struct InvSlabs {
    RowSlabs own;
    uint32_t my, mz;         // y slabs of row j + STEP; z slabs of the lane's cells or the next one in STEP
    int qn;                  // Phi index of the y slab at row j + STEP, plane 0
    int sy;
};
template <int STEP>
__device__ __forceinline__ InvSlabs inv_slabs(const RowAt *at, int j, int kl, bool live)
{
    const RowAts r = row_ats(at);
    InvSlabs L;
    L.own.m = live ? row_mask(r, j, kl) : 0u;
    const uint32_t mj = live ? row_mask(r, j + STEP, kl) : 0u;
    const uint32_t mk = live ? row_mask(r, j, kl + STEP) : 0u;
    L.my = mj & ROW_Y;
    L.mz = (L.own.m | mk) & ROW_Z;
    const bool ylo = (L.own.m | L.my) & 2u, zlo = L.mz & 4u;
    const int offy = ylo ? r.s[1][4] : r.s[4][4], sy = ylo ? r.s[1][6] : r.s[4][6];
    L.own.qy = offy + j * sy + kl;
    L.qn = L.own.qy + STEP * sy;
    L.own.sy = ylo ? r.s[1][5] : r.s[4][5];
    L.own.qz = (zlo ? r.s[2][4] : r.s[5][4]) + j * (zlo ? r.s[2][6] : r.s[5][6]) + kl;
    L.own.sz = zlo ? r.s[2][5] : r.s[5][5];
    L.own.x0 = r.s[0];
    L.own.x1 = r.s[3];
    return L;
}

// a / d by the slab's row_quot, or the division itself.
__device__ __forceinline__ fN inv_quot(fN a, const RowSlab &S)
{
    fN q;
    RowOdd odd;
    row_quot(a, S, q, odd);
    if (odd.any()) {
#pragma unroll
        for (int u = 0; u < NC; ++u) q[u] = a[u] / S.d;
    }
    return q;
}

// dL/d(dd) of one slab term at a lane's cells: (f RA01) l - RF0 mu with f the
// signed coefficient, 0 outside `in`; e the cells' profile entries.
__device__ __forceinline__ float inv_ldd(float4 e, float f, float l, float mu, bool in)
{
    const float v = f * e.x * l - e.w * mu;
    return in ? v : 0.f;
}
// The adjoint of Phi one iteration back: RE mu + (f RB) l.
__device__ __forceinline__ float inv_mu(float4 e, float f, float l, float mu) { return e.z * mu + f * e.y * l; }

__device__ __forceinline__ float4 inv_entry(const RowSlab &S, const float *RT, int c)
{
    return *reinterpret_cast<const float4 *>(RT + S.rt + S.sign * (c - S.pend) * 4);
}

// Cells of a lane whose edge is updated (reference ranges of
// gprMax/fields_updates_ext.pyx): E component C at plane i, row j.
template <int C>
__device__ __forceinline__ bool inv_eupd(const RowModel &a, int i, int j, int k)
{
    const bool x = C == 0 ? i < a.nx : (i >= 1) & (i < a.nx);
    const bool y = C == 1 ? j < a.ny : (j >= 1) & (j < a.ny);
    const bool z = C == 2 ? k < a.nz : (k >= 1) & (k < a.nz);
    return x & y & z;
}
template <int C>
__device__ __forceinline__ bool inv_hupd(const RowModel &a, int i, int j, int k)
{
    const bool x = C == 0 ? (i >= 1) & (i <= a.nx) : (i >= 0) & (i < a.nx);
    const bool y = C == 1 ? (j >= 1) & (j <= a.ny) : (j >= 0) & (j < a.ny);
    const bool z = C == 2 ? (k >= 1) & (k <= a.nz) : (k >= 0) & (k < a.nz);
    return x & y & z;
}
template <int C>
__device__ __forceinline__ fN inv_emask(const RowModel &a, int i, int j, int kl, fN v)
{
#pragma unroll
    for (int u = 0; u < NC; ++u) v[u] = inv_eupd<C>(a, i, j, kl + u) ? v[u] : 0.f;
    return v;
}
template <int C>
__device__ __forceinline__ fN inv_hmask(const RowModel &a, int i, int j, int kl, fN v)
{
#pragma unroll
    for (int u = 0; u < NC; ++u) v[u] = inv_hupd<C>(a, i, j, kl + u) ? v[u] : 0.f;
    return v;
}

// Calls f(u, number) for the receivers on a lane's cells u, on planes that have any:
// those of the block's segment of the plane, one after the other, the same for all
// lanes, through the scalar cache.  With every receiver looked at by every lane of
// such a plane 400 on 40^3 took 45 to 76 us an iteration of the forward, now 14 to 19 (one:
// 11).  The tables' pointers are the model's, not the launch's: those stay in
// scalar registers throughout, of which the adjoint's H half had none left (91 reads of
// spilled ones; 60^3 with 6 receivers 28.2 us an iteration of the backward, now 27.9).
template <class Fn>
__device__ __forceinline__ void inv_receivers(const InvStep &b, const RowModel &a, uint32_t pf, int i, int seg, uint32_t to, const Fn &f)
{
    if (!(pf & PF_RX)) return;
    typedef __attribute__((address_space(4))) const int cint;
    typedef __attribute__((address_space(4))) const u32x2 cu32x2;
    const int at = i * a.pseg + seg, r1 = ((cint *)a.rxfirst)[at + 1];
    for (int r = ((cint *)a.rxfirst)[at]; r < r1; ++r) {
        const u32x2 x = ((cu32x2 *)a.rxat)[r];
        const uint32_t u = x[0] - to / 4u;
        if (u < NC) f((int)u, (int)x[1]);
    }
}

// H pass of the forward, receivers sampled before it.  38.0 + 4.6 us (the
// receivers a launch of their own) before, 24.2 now.
template <int ORDER>
__global__ void __launch_bounds__(ROW_PASS_MAX) ROW_PASS_WAVES(0, ORDER) k_inv_row_h(const RowModel *__restrict__ models, InvStep b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    const RowModel &a = *models;
    const RowLane q = row_lane(a, g, 0, a.nx + 1);
    const int j = q.j, kl = q.kl, lane = threadIdx.x & 63;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t toj = j < a.ny ? to + 4u * (uint32_t)a.kp : to;
    const rsrc_t rE = rsrc(b.E), rH = rsrc(b.H), rP = rsrc(b.P);
    const uint32_t P4 = (uint32_t)a.plane * 4u, cs = a.cs;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const bool patch = q.live && lane == 63 && kl + NC <= a.nz;
    RowSlabs L;
    if (ORDER > 0) L = row_slabs(a.atH, j, kl, q.live);
    fN ey = bldN(rE, to, (uint32_t)q.xa * P4 + cs), ez = bldN(rE, to, (uint32_t)q.xa * P4 + 2 * cs);
    fN ex, hx, hy, hz, ezj, exj, ey1, ez1;
    float ykn = 0.f, xkn = 0.f;
    RowPhis<ORDER> ph;
    uint32_t pf = 0, m = 0;
    auto load = [&](int i) {
        pf = plane_flags(a, i);
        const uint32_t so = (uint32_t)i * P4, sn = i < a.nx ? so + P4 : so;
        ex = bldN(rE, to, so);
        hx = bldN(rH, to, so);
        hy = bldN(rH, to, so + cs);
        hz = bldN(rH, to, so + 2 * cs);
        ezj = bldN(rE, toj, so + 2 * cs);
        exj = bldN(rE, toj, so);
        ey1 = bldN(rE, to, sn + cs);
        ez1 = bldN(rE, to, sn + 2 * cs);
        if (patch) {
            ykn = bld(rE, to + 4u * NC, so + cs);
            xkn = bld(rE, to + 4u * NC, so);
        }
        if (ORDER > 0) {
            m = L.m & (pf >> PF_SLAB_H);
            row_phis(ph, L, m, (pf >> PF_SLAB_H) & 1u, rP, np4, i, j, kl);
        }
    };
    load(q.xa);
    const RowLds S = row_stage<ORDER, true, false, true>(lds4, a);
    __syncthreads();
    for (int i = q.xa;;) {
        const uint32_t so = (uint32_t)i * P4;
        const fN eyk = shift_up(ey, from_next(ykn, ey.x)), exk = shift_up(ex, from_next(xkn, ex.x));
        if (q.live)
            inv_receivers(b, a, pf, i, q.seg, to, [&](int u, int r) {
                b.traces[(size_t)r * b.iterations + b.it] = u ? ez[1] : ez[0];
            });
        const idN none = 0u;
        row_h<0, ORDER, true>(a, S, pf, m, ph, i, j, kl, q.live, b.it, ex, ey, ez, ey1, ez1, exj, ezj, exk, eyk, none, none, none,
                              hx, hy, hz);
        if (ORDER > 0) row_phis_store(ph, m, rP, np4);
        if (q.live) {
            bstN(rH, to, so, hx);
            bstN(rH, to, so + cs, hy);
            bstN(rH, to, so + 2 * cs, hz);
        }
        if (++i == q.xb) break;
        ey = ey1;
        ez = ez1;
        load(i);
    }
}

// A lane's values of the poles: [pole], of one component or coefficient.
template <int P>
struct InvPoles {
    fN v[P > 0 ? P : 1];
};
template <int P>
__device__ __forceinline__ InvPoles<P> inv_poles(rsrc_t r, uint32_t to, uint32_t so, uint32_t cs, int first)
{
    InvPoles<P> p;
#pragma unroll
    for (int n = 0; n < P; ++n) p.v[n] = bldN(r, to, so + (uint32_t)(first + n) * cs);
    return p;
}

// E pass of the forward: E^{n+1} into b.En, with the poles, the slabs and the
// dipole; the curl (and phi^n) for the adjoint where they are kept.
// 43.6 us before (half of the launches storing), 30.4 now.
template <int P, int ORDER>
__global__ void __launch_bounds__(ROW_PASS_MAX) ROW_PASS_WAVES(P > 0 ? 2 : 0, ORDER) k_inv_row_e(const RowModel *__restrict__ models,
                                                                                                 InvStep b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    const RowModel &a = *models;
    const RowLane q = row_lane(a, g, 0, a.nx + 1);
    const int j = q.j, kl = q.kl, lane = threadIdx.x & 63;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t tob = j > 0 ? to - 4u * (uint32_t)a.kp : to;
    const rsrc_t rE = rsrc(b.E), wE = rsrc(b.En), rH = rsrc(b.H), rM = rsrc(b.mat), rP = rsrc(b.P);
    const uint32_t P4 = (uint32_t)a.plane * 4u, cs = a.cs;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const bool patch = q.live && lane == 0 && kl > 0;
    RowSlabs L;
    if (ORDER > 0) L = row_slabs(a.atE, j, kl, q.live);
    const uint32_t sm = (uint32_t)(q.xa > 0 ? q.xa - 1 : 0) * P4;
    fN hym = bldN(rH, to, sm + cs), hzm = bldN(rH, to, sm + 2 * cs);
    fN ex, ey, ez, hx, hy, hz, hxj, hzj, CA, CB, IEA = 0.f;
    float hxl = 0.f, hyl = 0.f;
    RowPhis<ORDER> ph;
    InvPoles<P> t[3], ee, eq, zt;
    uint32_t pf = 0, m = 0;
    auto load = [&](int i) {
        pf = plane_flags(a, i);
        const uint32_t so = (uint32_t)i * P4;
        hx = bldN(rH, to, so);
        hy = bldN(rH, to, so + cs);
        hz = bldN(rH, to, so + 2 * cs);
        ex = bldN(rE, to, so);
        ey = bldN(rE, to, so + cs);
        ez = bldN(rE, to, so + 2 * cs);
        CA = bldN(rM, to, so);
        CB = bldN(rM, to, so + cs);
        hxj = bldN(rH, tob, so);
        hzj = bldN(rH, tob, so + 2 * cs);
        if (patch) {
            hxl = bld(rH, to - 4u, so);
            hyl = bld(rH, to - 4u, so + cs);
        }
        if (ORDER > 0) {
            m = L.m & (pf >> PF_SLAB_E);
            row_phis(ph, L, m, (pf >> PF_SLAB_E) & 1u, rP, np4, i, j, kl);
        }
        if (P > 0 || m || i == b.si) IEA = bldN(rM, to, so + 2 * cs);
        if (P > 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) t[c] = inv_poles<P>(rsrc(b.T), to, so, cs, c * P);
            ee = inv_poles<P>(rsrc(b.dc), to, so, cs, 0);
            eq = inv_poles<P>(rsrc(b.dc), to, so, cs, P);
            zt = inv_poles<P>(rsrc(b.dc), to, so, cs, 2 * P);
        }
    };
    load(q.xa);
    const RowLds S = row_stage<ORDER, true, true, false>(lds4, a);
    __syncthreads();
    for (int i = q.xa;;) {
        const uint32_t so = (uint32_t)i * P4;
        const fN hxk = shift_down(hx, from_prev(hxl, hx[NC - 1])), hyk = shift_down(hy, from_prev(hyl, hy[NC - 1]));
        if (q.live) {
            const fN d2y = hz - hzj, d1z = hy - hyk, d0z = hx - hxk, d2x = hz - hzm, d1x = hy - hym, d0y = hx - hxj;
            fN p0 = 0.f, p1 = 0.f, p2 = 0.f;
            InvPoles<P> n[3];
            // dispersive part A (gprMax/fields_updates_ext.pyx:113-179)
            auto part_a = [&](const InvPoles<P> &t, fN e, fN &phi, InvPoles<P> &n) {
                fN s = 0.f;
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    s = s + ee.v[p] * t.v[p];
                    n.v[p] = eq.v[p] * t.v[p] + zt.v[p] * e;
                }
                phi = s;
            };
            if (P > 0) {
                part_a(t[0], ex, p0, n[0]);
                part_a(t[1], ey, p1, n[1]);
                part_a(t[2], ez, p2, n[2]);
            }
            fN vx = CA * ex + CB * d2y - CB * d1z, vy = CA * ey + CB * d0z - CB * d2x, vz = CA * ez + CB * d1x - CB * d0y;
            if (P > 0) {
                p0 = inv_emask<0>(a, i, j, kl, p0);
                p1 = inv_emask<1>(a, i, j, kl, p1);
                p2 = inv_emask<2>(a, i, j, kl, p2);
                vx = vx - IEA * p0;
                vy = vy - IEA * p1;
                vz = vz - IEA * p2;
            }
            const bool bx = i < a.nx && j >= 1 && j < a.ny, by = i >= 1 && i < a.nx && j < a.ny,
                       bz = i >= 1 && i < a.nx && j >= 1 && j < a.ny;
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const int k = kl + u;
                ex[u] = bx && k >= 1 && k < a.nz ? vx[u] : ex[u];
                ey[u] = by && k >= 1 && k < a.nz ? vy[u] : ey[u];
                ez[u] = bz && k < a.nz ? vz[u] : ez[u];
            }
            if (ORDER > 0 && m) {
                auto c = [&](int u) { return IEA[u]; };
                fN xy = -0.f, xz = -0.f, yx = -0.f, yz = -0.f, zx = -0.f, zy = -0.f;
                if (m & ROW_X)
                    row_slab<0, ORDER, false, false>(S.slE[(pf >> PF_SLAB_E) & 1u ? 0 : 3], S.RTE, i, kl, d2x, d1x, xy, xz, c, c, ph.x);
                if (m & ROW_Y)
                    row_slab<0, ORDER, true, false>(S.slE[m & 2u ? 1 : 4], S.RTE, j, kl, d2y, d0y, yx, yz, c, c, ph.y);
                if (m & ROW_Z)
                    row_slab<0, ORDER, false, true>(S.slE[m & 4u ? 2 : 5], S.RTE, 0, kl, d1z, d0z, zx, zy, c, c, ph.z);
                row_add(ex, yx, zx, (m & 20u) == 20u);
                row_add(ey, xy, zy, (m & 12u) == 12u);
                row_add(ez, xz, yz, (m & 10u) == 10u);
                row_phis_store(ph, m, rP, np4);
            }
            if (i == b.si && j == b.sj) {
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    const float v = ez[u] - IEA[u] * b.w * b.sfac;
                    ez[u] = kl + u == b.sk ? v : ez[u];
                }
            }
            if (P > 0) {  // dispersive part B; edges that are not updated keep T
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    const fN x = n[0].v[p] - zt.v[p] * ex, y = n[1].v[p] - zt.v[p] * ey, z = n[2].v[p] - zt.v[p] * ez;
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const int k = kl + u;
                        t[0].v[p][u] = bx && k >= 1 && k < a.nz ? x[u] : t[0].v[p][u];
                        t[1].v[p][u] = by && k >= 1 && k < a.nz ? y[u] : t[1].v[p][u];
                        t[2].v[p][u] = bz && k < a.nz ? z[u] : t[2].v[p][u];
                    }
#pragma unroll
                    for (int c = 0; c < 3; ++c) bstN(rsrc(b.T), to, so + (uint32_t)(c * P + p) * cs, t[c].v[p]);
                }
            }
            bstN(wE, to, so, ex);
            bstN(wE, to, so + cs, ey);
            bstN(wE, to, so + 2 * cs, ez);
            if (b.curl) {  // in the form dL/dCB reads it
                const rsrc_t w = rsrc(b.curl);
                bstN(w, to, so, d2y - d1z);
                bstN(w, to, so + cs, d0z - d2x);
                bstN(w, to, so + 2 * cs, d1x - d0y);
                if (P > 0) {
                    const rsrc_t s = rsrc(b.phi);
                    bstN(s, to, so, p0);
                    bstN(s, to, so + cs, p1);
                    bstN(s, to, so + 2 * cs, p2);
                }
            }
        }
        if (++i == q.xb) break;
        hym = hy;
        hzm = hz;
        load(i);
    }
}

// ------------------------------------------------------------------ adjoint
// A load of the stored states, which the sweep reads once, slots one after the
// other: not to be kept, so that lE, lH and the gradients, which every iteration
// goes over, stay in the last-level cache (the sweeps and their recompute on
// 160x160x120, 600 iterations: 93.3 ms with ordinary loads, 90.4).
__device__ __forceinline__ fN bld_stored(rsrc_t r, uint32_t voff, uint32_t soff)
{
    return bits<fN>(__builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 2));
}

// E half of iteration n: lH += (dE^{n+1}/dH^{n+1})^T lE*, the gradients from
// lE*, E^n and the curl, and the Phi adjoints into b.Q.  lE* (the poles' part B
// folded in) is left as it is.
// 95.4 us before, 53.2 now.
template <int P, int ORDER>
__global__ void __launch_bounds__(ROW_PASS_MAX) ROW_PASS_WAVES(2, ORDER) k_inv_adj_e(const RowModel *__restrict__ models, InvStep b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    const RowModel &a = *models;
    const RowLane q = row_lane(a, g, 0, a.nx + 1);
    const int j = q.j, kl = q.kl, lane = threadIdx.x & 63;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t toj = j < a.ny ? to + 4u * (uint32_t)a.kp : to;
    const rsrc_t rL = rsrc(b.lE), rH = rsrc(b.H), rM = rsrc(b.mat), rE = rsrc(b.E), rC = rsrc(b.curl), rG = rsrc(b.grad),
                 rP = rsrc(b.P), rQ = rsrc(b.Q);
    const uint32_t P4 = (uint32_t)a.plane * 4u, cs = a.cs;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const bool patch = q.live && lane == 63 && kl + NC <= a.nz;
    InvSlabs L;
    if (ORDER > 0) L = inv_slabs<1>(a.atE, j, kl, q.live);
    const uint32_t s0 = (uint32_t)q.xa * P4;
    fN ly = bldN(rL, to, s0 + cs), lz = bldN(rL, to, s0 + 2 * cs), CB = bldN(rM, to, s0 + cs);
    fN lx, lxj, lzj, CBj, ly1, lz1, CB1, hx, hy, hz, e0, e1, e2, c0, c1, c2, gA, gB;
    fN IEA = 0.f, IEA1 = 0.f, IEAj = 0.f;
    RowPhi<1> xo, xn, yo, yn, z;
    float lxk = 0.f, lyk = 0.f, CBk = 0.f, IEAk = 0.f, za = 0.f, zb = 0.f;
    uint32_t f = 0, fn = 0, mo = 0, mx = 0, my = 0, mz = 0;
    auto load = [&](int i) {
        const uint32_t so = (uint32_t)i * P4, sn = i < a.nx ? so + P4 : so;
        lx = bldN(rL, to, so);
        lxj = bldN(rL, toj, so);
        lzj = bldN(rL, toj, so + 2 * cs);
        CBj = bldN(rM, toj, so + cs);
        ly1 = bldN(rL, to, sn + cs);
        lz1 = bldN(rL, to, sn + 2 * cs);
        CB1 = bldN(rM, to, sn + cs);
        if (patch) {
            lxk = bld(rL, to + 4u * NC, so);
            lyk = bld(rL, to + 4u * NC, so + cs);
            CBk = bld(rM, to + 4u * NC, so + cs);
        }
        hx = bldN(rH, to, so);
        hy = bldN(rH, to, so + cs);
        hz = bldN(rH, to, so + 2 * cs);
        e0 = bld_stored(rE, to, so);
        e1 = bld_stored(rE, to, so + cs);
        e2 = bld_stored(rE, to, so + 2 * cs);
        c0 = bld_stored(rC, to, so);
        c1 = bld_stored(rC, to, so + cs);
        c2 = bld_stored(rC, to, so + 2 * cs);
        gA = bldN(rG, to, so);
        gB = bldN(rG, to, so + cs);
        if (ORDER > 0) {
            f = plane_flags(a, i) >> PF_SLAB_E;
            fn = i < a.nx ? plane_flags(a, i + 1) >> PF_SLAB_E : 0u;
            mo = L.own.m & f;
            mx = L.own.m & fn & ROW_X;
            my = L.my & f;
            mz = L.mz & f;
            if (mo | mx | my | mz) {
                IEA = bldN(rM, to, so + 2 * cs);
                if ((mo & ROW_X) | mx) {
                    const bool lo = (f | fn) & 1u;
                    const int off = lo ? L.own.x0[4] : L.own.x1[4], sx = lo ? L.own.x0[5] : L.own.x1[5];
                    const int at = off + i * sx + j * (lo ? L.own.x0[6] : L.own.x1[6]) + kl;
                    if (mo & ROW_X) row_phi_load(xo, at, rP, np4);
                    if (mx) {
                        row_phi_load(xn, at + sx, rP, np4);
                        IEA1 = bldN(rM, to, sn + 2 * cs);
                    }
                }
                if (mo & ROW_Y) row_phi_load(yo, L.own.qy + i * L.own.sy, rP, np4);
                if (my) {
                    row_phi_load(yn, L.qn + i * L.own.sy, rP, np4);
                    IEAj = bldN(rM, toj, so + 2 * cs);
                }
                if (mo & ROW_Z) row_phi_load(z, L.own.qz + i * L.own.sz, rP, np4);
                if (mz && patch) {
                    const uint32_t at = (uint32_t)(L.own.qz + i * L.own.sz + NC) * 4u;
                    za = bld(rP, at, 0u);
                    zb = bld(rP, at, np4);
                    IEAk = bld(rM, to + 4u * NC, so + 2 * cs);
                }
            }
        }
    };
    load(q.xa);
    const RowLds S = row_stage<ORDER, true, true, false>(lds4, a);
    __syncthreads();
    for (int i = q.xa;;) {
        const uint32_t so = (uint32_t)i * P4;
        // CB lE at the point and at its k+1, j+1 and i+1 neighbours, of updated edges
        const fN px = inv_emask<0>(a, i, j, kl, CB * lx), py = inv_emask<1>(a, i, j, kl, CB * ly),
                 pz = inv_emask<2>(a, i, j, kl, CB * lz);
        const fN pxj = inv_emask<0>(a, i, j + 1, kl, CBj * lxj), pzj = inv_emask<2>(a, i, j + 1, kl, CBj * lzj);
        const fN py1 = inv_emask<1>(a, i + 1, j, kl, CB1 * ly1), pz1 = inv_emask<2>(a, i + 1, j, kl, CB1 * lz1);
        const float nx_ = from_next(CBk * lxk, px.x), ny_ = from_next(CBk * lyk, py.x);
        const fN pxk = shift_up(px, inv_eupd<0>(a, i, j, kl + NC) ? nx_ : 0.f),
                 pyk = shift_up(py, inv_eupd<1>(a, i, j, kl + NC) ? ny_ : 0.f);
        fN d0 = py - pyk - pz + pzj, d1 = pz - pz1 - px + pxk, d2 = px - pxj - py + py1;
        if (ORDER > 0) {
            // z: what the next lane's first cell gives comes by a shift
            fN l0 = 0.f, l1 = 0.f, n0, n1;
            float k0 = 0.f, k1 = 0.f;
            if (mz) {
                const RowSlab &s = S.slE[mz & 4u ? 2 : 5];
                if (mo & ROW_Z) {
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const int k = kl + u;
                        const bool in = (k >= s.lo[2]) & (k < s.hi[2]);
                        const float4 e = inv_entry(s, S.RTE, in ? k : s.pend);
                        l0[u] = inv_ldd(e, -IEA[u], lx[u], z.a[0][u], in);
                        l1[u] = inv_ldd(e, IEA[u], ly[u], z.b[0][u], in);
                        z.a[0][u] = inv_mu(e, -IEA[u], lx[u], z.a[0][u]);
                        z.b[0][u] = inv_mu(e, IEA[u], ly[u], z.b[0][u]);
                    }
                }
                const int k = kl + NC;
                const bool in = patch & (k >= s.lo[2]) & (k < s.hi[2]);
                const float4 e = inv_entry(s, S.RTE, in ? k : s.pend);
                k0 = inv_ldd(e, -IEAk, lxk, za, in);
                k1 = inv_ldd(e, IEAk, lyk, zb, in);
            }
            const float p0 = from_next(k0, l0.x), p1 = from_next(k1, l1.x);
            n0 = shift_up(l0, kl + NC <= a.nz ? p0 : 0.f);
            n1 = shift_up(l1, kl + NC <= a.nz ? p1 : 0.f);
            if (mo | mx | my | mz) {
                fN x1 = -0.f, x2 = -0.f, y0 = -0.f, y2 = -0.f, z0 = -0.f, z1 = -0.f;
                if ((mo & ROW_X) | mx) {
                    const RowSlab &s = S.slE[(f | fn) & 1u ? 0 : 3];
                    const bool o = mo & ROW_X, w = mx;
                    const float4 eo = inv_entry(s, S.RTE, o ? i : s.pend), en = inv_entry(s, S.RTE, w ? i + 1 : s.pend);
                    fN v1, v2;
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const bool in = (kl + u >= s.lo[2]) & (kl + u < s.hi[2]);
                        v2[u] = inv_ldd(eo, -IEA[u], ly[u], xo.a[0][u], o & in) - inv_ldd(en, -IEA1[u], ly1[u], xn.a[0][u], w & in);
                        v1[u] = inv_ldd(eo, IEA[u], lz[u], xo.b[0][u], o & in) - inv_ldd(en, IEA1[u], lz1[u], xn.b[0][u], w & in);
                        xo.a[0][u] = inv_mu(eo, -IEA[u], ly[u], xo.a[0][u]);
                        xo.b[0][u] = inv_mu(eo, IEA[u], lz[u], xo.b[0][u]);
                    }
                    x2 = inv_quot(v2, s);
                    x1 = inv_quot(v1, s);
                }
                if ((mo & ROW_Y) | my) {
                    const RowSlab &s = S.slE[(mo | my) & 2u ? 1 : 4];
                    const bool o = mo & ROW_Y, w = my;
                    const float4 eo = inv_entry(s, S.RTE, o ? j : s.pend), en = inv_entry(s, S.RTE, w ? j + 1 : s.pend);
                    fN v0, v2;
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const bool in = (kl + u >= s.lo[2]) & (kl + u < s.hi[2]);
                        v2[u] = inv_ldd(eo, IEA[u], lx[u], yo.a[0][u], o & in) - inv_ldd(en, IEAj[u], lxj[u], yn.a[0][u], w & in);
                        v0[u] = inv_ldd(eo, -IEA[u], lz[u], yo.b[0][u], o & in) - inv_ldd(en, -IEAj[u], lzj[u], yn.b[0][u], w & in);
                        yo.a[0][u] = inv_mu(eo, IEA[u], lx[u], yo.a[0][u]);
                        yo.b[0][u] = inv_mu(eo, -IEA[u], lz[u], yo.b[0][u]);
                    }
                    y2 = inv_quot(v2, s);
                    y0 = inv_quot(v0, s);
                }
                if (mz) {
                    const RowSlab &s = S.slE[mz & 4u ? 2 : 5];
                    z1 = inv_quot(l0 - n0, s);
                    z0 = inv_quot(l1 - n1, s);
                }
                const uint32_t m = mo | mx | my | mz;
                row_add(d0, y0, z0, (m & 20u) == 20u);
                row_add(d1, x1, z1, (m & 12u) == 12u);
                row_add(d2, x2, y2, (m & 10u) == 10u);
            }
        }
        if (q.live) {
            const fN m0 = inv_emask<0>(a, i, j, kl, lx), m1 = inv_emask<1>(a, i, j, kl, ly), m2 = inv_emask<2>(a, i, j, kl, lz);
            fN ga = m0 * e0 + m1 * e1 + m2 * e2, gb = m0 * c0 + m1 * c1 + m2 * c2;
            bstN(rH, to, so, hx + d0);
            bstN(rH, to, so + cs, hy + d1);
            bstN(rH, to, so + 2 * cs, hz + d2);
            bstN(rG, to, so, gA + ga);
            bstN(rG, to, so + cs, gB + gb);
            if (P > 0 || (i == b.si && j == b.sj)) {
                fN gi = 0.f;
#pragma unroll
                for (int u = 0; u < NC; ++u)
                    if (i == b.si && j == b.sj && kl + u == b.sk) gi[u] = -lz[u] * b.w * b.sfac;
                if (P > 0) {
                    const rsrc_t rS = rsrc(b.phi);
                    gi = gi - m0 * bldN(rS, to, so);
                    gi = gi - m1 * bldN(rS, to, so + cs);
                    gi = gi - m2 * bldN(rS, to, so + 2 * cs);
                }
                bstN(rG, to, so + 2 * cs, bldN(rG, to, so + 2 * cs) + gi);
            }
            if (ORDER > 0) {
                if (mo & ROW_X) row_phi_store(xo, rQ, np4);
                if (mo & ROW_Y) row_phi_store(yo, rQ, np4);
                if (mo & ROW_Z) row_phi_store(z, rQ, np4);
            }
        }
        if (++i == q.xb) break;
        ly = ly1;
        lz = lz1;
        CB = CB1;
        load(i);
    }
}

// H half of iteration n: lE^n = CA lE* (+ the poles) + (dH^{n+1}/dE^n)^T lH on
// updated edges, plus the receivers' residuals, in place; lT one iteration
// back; then, with poles, lE* of iteration n-1 from both; and the Phi adjoints
// into b.Q.
// 56.9 us before (and 5.2 for lE* in a launch of its own on 40^3), 28.5 now.
template <int P, int ORDER>
__global__ void __launch_bounds__(ROW_PASS_MAX) ROW_PASS_WAVES(P > 0 ? 2 : 1, ORDER) k_inv_adj_h(const RowModel *__restrict__ models,
                                                                                                 InvStep b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    const RowModel &a = *models;
    const RowLane q = row_lane(a, g, 0, a.nx + 1);
    const int j = q.j, kl = q.kl, lane = threadIdx.x & 63;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t tob = j > 0 ? to - 4u * (uint32_t)a.kp : to;
    const rsrc_t rL = rsrc(b.lE), rH = rsrc(b.H), rM = rsrc(b.mat), rP = rsrc(b.P), rQ = rsrc(b.Q);
    const uint32_t P4 = (uint32_t)a.plane * 4u, cs = a.cs;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const bool patch = q.live && lane == 0 && kl > 0;
    InvSlabs L;
    if (ORDER > 0) L = inv_slabs<-1>(a.atH, j, kl, q.live);
    const uint32_t sm = (uint32_t)(q.xa > 0 ? q.xa - 1 : 0) * P4;
    fN hym = bldN(rH, to, sm + cs), hzm = bldN(rH, to, sm + 2 * cs);
    fN hx, hy, hz, hxj, hzj, lx, ly, lz, CA, IEA = 0.f;
    RowPhi<1> xo, xn, yo, yn, z;
    InvPoles<P> t[3], ee, eq, zt;
    float hxl = 0.f, hyl = 0.f, za = 0.f, zb = 0.f;
    uint32_t pf = 0, f = 0, fn = 0, mo = 0, mx = 0, my = 0, mz = 0;
    auto load = [&](int i) {
        const uint32_t so = (uint32_t)i * P4;
        pf = plane_flags(a, i);
        hx = bldN(rH, to, so);
        hy = bldN(rH, to, so + cs);
        hz = bldN(rH, to, so + 2 * cs);
        hxj = bldN(rH, tob, so);
        hzj = bldN(rH, tob, so + 2 * cs);
        if (patch) {
            hxl = bld(rH, to - 4u, so);
            hyl = bld(rH, to - 4u, so + cs);
        }
        lx = bldN(rL, to, so);
        ly = bldN(rL, to, so + cs);
        lz = bldN(rL, to, so + 2 * cs);
        CA = bldN(rM, to, so);
        if (ORDER > 0) {
            f = pf >> PF_SLAB_H;
            fn = i > 0 ? plane_flags(a, i - 1) >> PF_SLAB_H : 0u;
            mo = L.own.m & f;
            mx = L.own.m & fn & ROW_X;
            my = L.my & f;
            mz = L.mz & f;
            if ((mo & ROW_X) | mx) {
                const bool lo = (f | fn) & 1u;
                const int off = lo ? L.own.x0[4] : L.own.x1[4], sx = lo ? L.own.x0[5] : L.own.x1[5];
                const int at = off + i * sx + j * (lo ? L.own.x0[6] : L.own.x1[6]) + kl;
                if (mo & ROW_X) row_phi_load(xo, at, rP, np4);
                if (mx) row_phi_load(xn, at - sx, rP, np4);
            }
            if (mo & ROW_Y) row_phi_load(yo, L.own.qy + i * L.own.sy, rP, np4);
            if (my) row_phi_load(yn, L.qn + i * L.own.sy, rP, np4);
            if (mo & ROW_Z) row_phi_load(z, L.own.qz + i * L.own.sz, rP, np4);
            if (mz && patch) {
                const int before = L.own.qz + i * L.own.sz - 1;   // unused where the cell before is in no slab
                const uint32_t at = before > 0 ? (uint32_t)before * 4u : 0u;
                za = bld(rP, at, 0u);
                zb = bld(rP, at, np4);
            }
        }
        if (P > 0) {
            IEA = bldN(rM, to, so + 2 * cs);
#pragma unroll
            for (int c = 0; c < 3; ++c) t[c] = inv_poles<P>(rsrc(b.T), to, so, cs, c * P);
            ee = inv_poles<P>(rsrc(b.dc), to, so, cs, 0);
            eq = inv_poles<P>(rsrc(b.dc), to, so, cs, P);
            zt = inv_poles<P>(rsrc(b.dc), to, so, cs, 2 * P);
        }
    };
    load(q.xa);
    const RowLds S = row_stage<ORDER, true, false, true>(lds4, a);
    __syncthreads();
    for (int i = q.xa;;) {
        const uint32_t so = (uint32_t)i * P4;
        const float DB = b.DB;
        // DB lH at the point and at its k-1, j-1 and i-1 neighbours, of updated cells
        const fN px = inv_hmask<0>(a, i, j, kl, DB * hx), py = inv_hmask<1>(a, i, j, kl, DB * hy),
                 pz = inv_hmask<2>(a, i, j, kl, DB * hz);
        const fN pxj = inv_hmask<0>(a, i, j - 1, kl, DB * hxj), pzj = inv_hmask<2>(a, i, j - 1, kl, DB * hzj);
        const fN pym = inv_hmask<1>(a, i - 1, j, kl, DB * hym), pzm = inv_hmask<2>(a, i - 1, j, kl, DB * hzm);
        const float bx_ = from_prev(DB * hxl, px[NC - 1]), by_ = from_prev(DB * hyl, py[NC - 1]);
        const fN pxk = shift_down(px, inv_hupd<0>(a, i, j, kl - 1) ? bx_ : 0.f),
                 pyk = shift_down(py, inv_hupd<1>(a, i, j, kl - 1) ? by_ : 0.f);
        fN d0 = py - pyk - pz + pzj, d1 = pz - pzm - px + pxk, d2 = px - pxj - py + pym;
        if (ORDER > 0) {
            const float cH = b.cH;
            fN l0 = 0.f, l1 = 0.f, n0, n1;
            float k0 = 0.f, k1 = 0.f;
            if (mz) {
                const RowSlab &s = S.slH[mz & 4u ? 2 : 5];
                if (mo & ROW_Z) {
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const int k = kl + u;
                        const bool in = (k >= s.lo[2]) & (k < s.hi[2]);
                        const float4 e = inv_entry(s, S.RTH, in ? k : s.pend);
                        l0[u] = inv_ldd(e, cH, hx[u], z.a[0][u], in);
                        l1[u] = inv_ldd(e, -cH, hy[u], z.b[0][u], in);
                        z.a[0][u] = inv_mu(e, cH, hx[u], z.a[0][u]);
                        z.b[0][u] = inv_mu(e, -cH, hy[u], z.b[0][u]);
                    }
                }
                const int k = kl - 1;
                const bool in = patch & (k >= s.lo[2]) & (k < s.hi[2]);
                const float4 e = inv_entry(s, S.RTH, in ? k : s.pend);
                k0 = inv_ldd(e, cH, hxl, za, in);
                k1 = inv_ldd(e, -cH, hyl, zb, in);
            }
            const float p0 = from_prev(k0, l0[NC - 1]), p1 = from_prev(k1, l1[NC - 1]);
            n0 = shift_down(l0, kl > 0 ? p0 : 0.f);
            n1 = shift_down(l1, kl > 0 ? p1 : 0.f);
            if (mo | mx | my | mz) {
                fN x1 = -0.f, x2 = -0.f, y0 = -0.f, y2 = -0.f, z0 = -0.f, z1 = -0.f;
                if ((mo & ROW_X) | mx) {
                    const RowSlab &s = S.slH[(f | fn) & 1u ? 0 : 3];
                    const bool o = mo & ROW_X, w = mx;
                    const float4 eo = inv_entry(s, S.RTH, o ? i : s.pend), en = inv_entry(s, S.RTH, w ? i - 1 : s.pend);
                    fN v1, v2;
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const bool in = (kl + u >= s.lo[2]) & (kl + u < s.hi[2]);
                        v2[u] = inv_ldd(en, cH, hym[u], xn.a[0][u], w & in) - inv_ldd(eo, cH, hy[u], xo.a[0][u], o & in);
                        v1[u] = inv_ldd(en, -cH, hzm[u], xn.b[0][u], w & in) - inv_ldd(eo, -cH, hz[u], xo.b[0][u], o & in);
                        xo.a[0][u] = inv_mu(eo, cH, hy[u], xo.a[0][u]);
                        xo.b[0][u] = inv_mu(eo, -cH, hz[u], xo.b[0][u]);
                    }
                    x2 = inv_quot(v2, s);
                    x1 = inv_quot(v1, s);
                }
                if ((mo & ROW_Y) | my) {
                    const RowSlab &s = S.slH[(mo | my) & 2u ? 1 : 4];
                    const bool o = mo & ROW_Y, w = my;
                    const float4 eo = inv_entry(s, S.RTH, o ? j : s.pend), en = inv_entry(s, S.RTH, w ? j - 1 : s.pend);
                    fN v0, v2;
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        const bool in = (kl + u >= s.lo[2]) & (kl + u < s.hi[2]);
                        v2[u] = inv_ldd(en, -cH, hxj[u], yn.a[0][u], w & in) - inv_ldd(eo, -cH, hx[u], yo.a[0][u], o & in);
                        v0[u] = inv_ldd(en, cH, hzj[u], yn.b[0][u], w & in) - inv_ldd(eo, cH, hz[u], yo.b[0][u], o & in);
                        yo.a[0][u] = inv_mu(eo, -cH, hx[u], yo.a[0][u]);
                        yo.b[0][u] = inv_mu(eo, cH, hz[u], yo.b[0][u]);
                    }
                    y2 = inv_quot(v2, s);
                    y0 = inv_quot(v0, s);
                }
                if (mz) {
                    const RowSlab &s = S.slH[mz & 4u ? 2 : 5];
                    z1 = inv_quot(n0 - l0, s);
                    z0 = inv_quot(n1 - l1, s);
                }
                const uint32_t m = mo | mx | my | mz;
                row_add(d0, y0, z0, (m & 20u) == 20u);
                row_add(d1, x1, z1, (m & 12u) == 12u);
                row_add(d2, x2, y2, (m & 10u) == 10u);
            }
        }
        if (q.live) {
            fN o0 = CA * lx, o1 = CA * ly, o2 = CA * lz;
            if (P > 0) {
                auto back = [&](InvPoles<P> &t, fN l, fN &o) {
                    fN s = 0.f;
#pragma unroll
                    for (int p = 0; p < P; ++p) {
                        s = s + zt.v[p] * t.v[p];
                        t.v[p] = eq.v[p] * t.v[p] - IEA * ee.v[p] * l;
                    }
                    o = o + s;
                };
                back(t[0], lx, o0);
                back(t[1], ly, o1);
                back(t[2], lz, o2);
            }
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const int k = kl + u;
                lx[u] = (inv_eupd<0>(a, i, j, k) ? o0[u] : lx[u]) + d0[u];
                ly[u] = (inv_eupd<1>(a, i, j, k) ? o1[u] : ly[u]) + d1[u];
                lz[u] = (inv_eupd<2>(a, i, j, k) ? o2[u] : lz[u]) + d2[u];
            }
            inv_receivers(b, a, pf, i, q.seg, to, [&](int at, int r) {
                const float v = b.resid[(size_t)r * b.iterations + b.it];
#pragma unroll
                for (int u = 0; u < NC; ++u) lz[u] = at == u ? lz[u] + v : lz[u];
            });
            if (P > 0) {
                auto next = [&](const InvPoles<P> &t, fN l) {
#pragma unroll
                    for (int p = 0; p < P; ++p) l = l - zt.v[p] * t.v[p];
                    return l;
                };
                const fN s0 = next(t[0], lx), s1 = next(t[1], ly), s2 = next(t[2], lz);
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    const int k = kl + u;
                    lx[u] = inv_eupd<0>(a, i, j, k) ? s0[u] : lx[u];
                    ly[u] = inv_eupd<1>(a, i, j, k) ? s1[u] : ly[u];
                    lz[u] = inv_eupd<2>(a, i, j, k) ? s2[u] : lz[u];
                }
                // (where an edge is not updated zt or lT is never read)
#pragma unroll
                for (int c = 0; c < 3; ++c)
#pragma unroll
                    for (int p = 0; p < P; ++p) bstN(rsrc(b.T), to, so + (uint32_t)(c * P + p) * cs, t[c].v[p]);
            }
            bstN(rL, to, so, lx);
            bstN(rL, to, so + cs, ly);
            bstN(rL, to, so + 2 * cs, lz);
            if (ORDER > 0) {
                if (mo & ROW_X) row_phi_store(xo, rQ, np4);
                if (mo & ROW_Y) row_phi_store(yo, rQ, np4);
                if (mo & ROW_Z) row_phi_store(z, rQ, np4);
            }
        }
        if (++i == q.xb) break;
        hym = hy;
        hzm = hz;
        load(i);
    }
}

typedef void (*inv_kernel)(const RowModel *, InvStep);
struct InvKernels {
    inv_kernel h, e, adj_e, adj_h;
};
template <int ORDER>
InvKernels inv_kernels(int P)
{
#define GPX_IK(PP) InvKernels{k_inv_row_h<ORDER>, k_inv_row_e<PP, ORDER>, k_inv_adj_e<PP, ORDER>, k_inv_adj_h<PP, ORDER>}
    switch (P) {
    case 0: return GPX_IK(0);
    case 1: return GPX_IK(1);
    case 2: return GPX_IK(2);
    case 3: return GPX_IK(3);
    default: return GPX_IK(4);
    }
#undef GPX_IK
}

}  // namespace gpx

#endif  // GPX_INV_ROWS_H
