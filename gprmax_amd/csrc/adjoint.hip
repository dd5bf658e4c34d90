// Differentiable FDTD for per-cell permittivity and conductivity: a forward
// solve that keeps checkpoints, and the discrete adjoint (reverse mode) of it,
// which accumulates dL/dCA, dL/dCB and dL/dIEA per cell for a trace-misfit
// loss.  C ABI in include/gpx.h (gpx_inv_*).
//
// The forward scheme is the reference's solver loop (gprMax/model_build_run.py:
// 424-470) restricted to what a per-cell inversion needs: Yee updates
// (gprMax/fields_updates_ext.pyx:81-107, 404-412) with every cell its own
// material (E edge (c, i, j, k) takes cell (i, j, k), the reference's
// build_voxel without averaging), mu_r = 1 and no magnetic loss (DA = 1,
// DB = dt / (mu0 d)), HORIPML with one CFS term on any set of slabs
// (gprMax/pml_updates/pml_updates_*_HORIPML_ext.pyx, order1_*), optional
// Debye poles per cell with real auxiliary values (dispersive parts A and B,
// gprMax/fields_updates_ext.pyx:113-235; coefficients of
// gprMax/materials.py:92-143), one z-directed Hertzian dipole per solve
// (gprMax/sources.py:163-193), and Ez receivers sampled at the start of
// each iteration (gprMax/fields_outputs.py:40-67).
//
// With poles, an updated E edge of a cell with coefficients (ee, eqt, zt)
// per pole p does, around its E update:
//   A: phi = sum_p ee_p T_p;  T_p = eqt_p T_p + zt_p E^n;
//      E^{n+1} = CA E^n + CB curl H^{n+1} - IEA phi  (+ PML, source)
//   B: T_p = T_p - zt_p E^{n+1}
// so T^{n+1}_p = eqt_p T^n_p + zt_p (E^n - E^{n+1}).  Its reverse, with lT_p
// = dL/dT^{n+1}_p: the adjoint of E^{n+1} seen by the E update is
// lE* = lE - sum_p zt_p lT_p (which the gathers use); then lE^n = CA lE* + sum_p zt_p lT_p, lT^n_p = eqt_p lT_p -
// IEA ee_p lE*, and dL/dIEA gains -lE* phi^n (phi^n saved by the recompute).
//
// Iteration n maps the state s^n = (E^n, H^n, PhiE^n, PhiH^n) to s^{n+1}
// linearly.  Its adjoint, applied from n = N-1 down to 0 to the adjoint state
// (lE, lH, mE, mH) = dL/ds^{n+1}, is two gather kernels:
//   E half: lH += (dE^{n+1}/dH^{n+1})^T lE  (curl and E-PML terms); gradients
//           from lE and the stored E^n and curl H^{n+1}; mE = (dE/dPhiE)^T lE + RE mE;
//   H half: lE = CA lE + (dH^{n+1}/dE^n)^T lH  (curl and H-PML terms);
//           mH = (dH/dPhiH)^T lH + RE mH (lH = DA lH = lH); and the receiver
//           residual of iteration n is added to lEz at each receiver.
// Each half gathers from one field and updates the other in place; mE and mH are
// double-buffered (read one copy, write the other).  With poles the H half
// also leaves lE* of the next iteration down, so the array holds lE*.
// Forward states come from checkpoints every K iterations; each segment is
// recomputed forward, storing E^n and curl H^{n+1} for every iteration of it,
// before the adjoint sweeps back over it.  E^n is not copied: the E pass
// reads it from its slot of the store and writes E^{n+1} into the next.
//
// The row kernels (inv_rows.h) run models whose slabs they can place: at most one
// per direction, in the order x0, y0, z0, xmax, ymax, zmax, the ones of an
// axis apart; the kernels here, one point a thread and a loop over the slabs, run
// any other.

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <string.h>

#include <string>
#include <vector>

#include "gpx.h"
#include "inv_rows.h"

using namespace gpx;

namespace {

constexpr int INV_MAX_SLABS = 6;
constexpr int INV_MAX_POLES = 4;

// One PML slab of the inversion grid (order 1).  Boxes are the corrected
// cells of each field; the profile index along the normal is p = pend - c
// (minus slabs) or c - pend (plus slabs).
struct InvSlab {
    int axis, minus;
    int loE[3], hiE[3], loH[3], hiH[3];
    int pendE, pendH;
    int org[3];
    int dE1[3], dE2[3], dH1[3], dH2[3];  // Phi dims (without the order axis)
    const float *RE;                     // E: RA, RB, RE, RF, each [t]
    const float *RH;                     // H: the same
    int t;
    float *PE1, *PE2, *PH1, *PH2;        // Phi (forward) or their adjoints (read)
    float *QE1, *QE2, *QH1, *QH2;        // adjoint: the adjoints written
    // Points whose adjoint gathers see this slab: the E box and the box one
    // step down the normal (E), the H box and the box one step up (H).
    int gE_lo[3], gE_hi[3], gH_lo[3], gH_hi[3];
};

// Arrays hold one float per grid point, rows of kp floats (InvStep has them by
// component), parameters and gradients too (0 where a point is no cell).
struct InvArgs {
    int nx, ny, nz, kp;
    long long n;                         // floats of one component
    float d;
    InvStep b;
    int nslab;
    InvSlab slab[INV_MAX_SLABS];
    int P;                               // Debye poles (0: none)
    int all_gk, all_blocks, all_per_xcd; // all_gk blocks of 128 points along k per (j, i) row
};

// One-dimensional launches: the hardware deals block b to XCD b mod 8, so block
// b takes logical number (b mod 8) * per_xcd + b / 8 (per_xcd = launched blocks
// / 8).  Each XCD then works through a contiguous run of logical blocks, i.e.
// of neighbouring grid rows, and the rows a point's differences read (j +- 1,
// i +- 1) are in the same XCD's L2 instead of another's.
__device__ __forceinline__ int xcd_block(int per_xcd)
{
    const int b = blockIdx.x;
    return (b & 7) * per_xcd + (b >> 3);
}

// Point (i, j, k) of a launch over every grid point; false past the grid.
__device__ __forceinline__ bool all_point(const InvArgs &a, int &i, int &j, int &k)
{
    const int lb = xcd_block(a.all_per_xcd);
    if (lb >= a.all_blocks) return false;
    const int kb = lb % a.all_gk, r = lb / a.all_gk;
    k = kb * blockDim.x + threadIdx.x;
    j = r % (a.ny + 1);
    i = r / (a.ny + 1);
    return true;
}

// Grid offsets are 32-bit: gpx_inv_create requires fewer than 2^31 points.
__device__ __forceinline__ int fidx(const InvArgs &a, int i, int j, int k)
{
    return (i * (a.ny + 1) + j) * a.kp + k;
}
__device__ __forceinline__ bool in_box3(const int *lo, const int *hi, int i, int j, int k)
{
    return i >= lo[0] && i < hi[0] && j >= lo[1] && j < hi[1] && k >= lo[2] && k < hi[2];
}

// Reference update ranges (gprMax/fields_updates_ext.pyx): component c of E or H
// is updated at (i, j, k).
__device__ __forceinline__ bool e_upd(const InvArgs &a, int c, int i, int j, int k)
{
    if (i < 0 || j < 0 || k < 0) return false;
    if (c == 0) return i < a.nx && j >= 1 && j < a.ny && k >= 1 && k < a.nz;
    if (c == 1) return i >= 1 && i < a.nx && j < a.ny && k >= 1 && k < a.nz;
    return i >= 1 && i < a.nx && j >= 1 && j < a.ny && k < a.nz;
}
__device__ __forceinline__ bool h_upd(const InvArgs &a, int c, int i, int j, int k)
{
    if (i < 0 || j < 0 || k < 0) return false;
    if (c == 0) return i >= 1 && i <= a.nx && j < a.ny && k < a.nz;
    if (c == 1) return i < a.nx && j >= 1 && j <= a.ny && k < a.nz;
    return i < a.nx && j < a.ny && k >= 1 && k <= a.nz;
}

__device__ __forceinline__ bool in_e(const InvSlab &s, int i, int j, int k)
{
    return i >= s.loE[0] && i < s.hiE[0] && j >= s.loE[1] && j < s.hiE[1] && k >= s.loE[2] && k < s.hiE[2];
}
__device__ __forceinline__ bool in_h(const InvSlab &s, int i, int j, int k)
{
    return i >= s.loH[0] && i < s.hiH[0] && j >= s.loH[1] && j < s.hiH[1] && k >= s.loH[2] && k < s.hiH[2];
}

// Profile index and Phi index of cell (i, j, k) for the given field's box.
__device__ __forceinline__ void pidx(const InvSlab &s, bool efield, int i, int j, int k, int &p, int &q1,
                                     int &q2)
{
    int c[3] = {i - s.org[0], j - s.org[1], k - s.org[2]};
    const int along = s.axis == 0 ? i : (s.axis == 1 ? j : k);
    const int pend = efield ? s.pendE : s.pendH;
    p = s.minus ? pend - along : along - pend;
    c[s.axis] = p;
    const int *d1 = efield ? s.dE1 : s.dH1, *d2 = efield ? s.dE2 : s.dH2;
    q1 = (c[0] * d1[1] + c[1]) * d1[2] + c[2];
    q2 = (c[0] * d2[1] + c[1]) * d2[2] + c[2];
}

// E-PML pairs per axis: (corrected E component, source H component, sign) for
// Phi1 and Phi2; H-PML likewise (gprMax/pml_updates/*_HORIPML_ext.pyx).
__device__ __forceinline__ void e_pair(int axis, int w, int &comp, int &src, int &sign)
{
    const int tab[3][2][3] = {{{1, 2, -1}, {2, 1, +1}}, {{0, 2, +1}, {2, 0, -1}}, {{0, 1, -1}, {1, 0, +1}}};
    comp = tab[axis][w][0];
    src = tab[axis][w][1];
    sign = tab[axis][w][2];
}
__device__ __forceinline__ void h_pair(int axis, int w, int &comp, int &src, int &sign)
{
    const int tab[3][2][3] = {{{1, 2, +1}, {2, 1, -1}}, {{0, 2, -1}, {2, 0, +1}}, {{0, 1, +1}, {1, 0, -1}}};
    comp = tab[axis][w][0];
    src = tab[axis][w][1];
    sign = tab[axis][w][2];
}

__device__ __forceinline__ int axis_of(const InvSlab &s, int i, int j, int k)
{
    return s.axis == 0 ? i : (s.axis == 1 ? j : k);
}

// Component c of a point of an array.
__device__ __forceinline__ float at3(const InvArgs &a, const float *f, int c, int o) { return f[c * a.n + o]; }

// ------------------------------------------------------------------ forward
// Receiver samples, H update and H-PML of one iteration; one thread per grid point.
__global__ void k_inv_h(InvArgs a)
{
    int i, j, k;
    if (!all_point(a, i, j, k) || k > a.nz) return;
    const InvStep &b = a.b;
    const int o = fidx(a, i, j, k), oi = fidx(a, i + 1, j, k), oj = fidx(a, i, j + 1, k), ok = o + 1;
    const int row = i * (a.ny + 1) + j;
    for (int r = b.rxfirst[row]; r < b.rxfirst[row + 1]; ++r)
        if (b.rxat[2 * r] == k) b.traces[(long long)b.rxat[2 * r + 1] * b.iterations + b.it] = at3(a, b.E, 2, o);
    auto E = [&](int c, int at) { return at3(a, b.E, c, at); };
    float h[3] = {at3(a, b.H, 0, o), at3(a, b.H, 1, o), at3(a, b.H, 2, o)};
    if (h_upd(a, 0, i, j, k)) h[0] = 1.0f * h[0] - b.DB * (E(2, oj) - E(2, o)) + b.DB * (E(1, ok) - E(1, o));
    if (h_upd(a, 1, i, j, k)) h[1] = 1.0f * h[1] - b.DB * (E(0, ok) - E(0, o)) + b.DB * (E(2, oi) - E(2, o));
    if (h_upd(a, 2, i, j, k)) h[2] = 1.0f * h[2] - b.DB * (E(1, oi) - E(1, o)) + b.DB * (E(0, oj) - E(0, o));
    for (int s = 0; s < a.nslab; ++s) {
        const InvSlab &S = a.slab[s];
        if (!in_h(S, i, j, k)) continue;
        int p;
        int q[2];
        pidx(S, false, i, j, k, p, q[0], q[1]);
        const float RA01 = S.RH[p] - 1.0f, RB0 = S.RH[S.t + p], RE0 = S.RH[2 * S.t + p], RF0 = S.RH[3 * S.t + p];
        const int on = S.axis == 0 ? oi : (S.axis == 1 ? oj : ok);
        for (int w = 0; w < 2; ++w) {
            int comp, src, sign;
            h_pair(S.axis, w, comp, src, sign);
            float *Phi = w == 0 ? S.PH1 : S.PH2;
            const float dd = (E(src, on) - E(src, o)) / a.d;
            const float ph = Phi[q[w]];
            const float corr = b.cH * (RA01 * dd + RB0 * ph);
            Phi[q[w]] = RE0 * ph - RF0 * dd;
            h[comp] = sign > 0 ? h[comp] + corr : h[comp] - corr;
        }
    }
    for (int c = 0; c < 3; ++c) b.H[c * a.n + o] = h[c];
}

// E update with the poles, E-PML and the Hertzian dipole of one iteration.
__global__ void k_inv_e(InvArgs a)
{
    int i, j, k;
    if (!all_point(a, i, j, k) || k > a.nz) return;
    const InvStep &b = a.b;
    const int o = fidx(a, i, j, k);
    const int om[3] = {i > 0 ? fidx(a, i - 1, j, k) : o, j > 0 ? fidx(a, i, j - 1, k) : o, k > 0 ? o - 1 : o};
    auto dH = [&](int c, int axis) { return at3(a, b.H, c, o) - at3(a, b.H, c, om[axis]); };
    float e[3] = {at3(a, b.E, 0, o), at3(a, b.E, 1, o), at3(a, b.E, 2, o)};
    // (om clamps to the point itself at the low faces, so every load is inside
    // the grid)
    const float d2y = dH(2, 1), d1z = dH(1, 2), d0z = dH(0, 2), d2x = dH(2, 0), d1x = dH(1, 0), d0y = dH(0, 1);
    const bool cell = i < a.nx && j < a.ny && k < a.nz;
    const float CA = b.mat[o], CB = b.mat[a.n + o], IEA = b.mat[2 * a.n + o];
    const bool upd[3] = {e_upd(a, 0, i, j, k), e_upd(a, 1, i, j, k), e_upd(a, 2, i, j, k)};
    // dispersive part A: phi from T^n, then T advanced with E^n
    float phi[3] = {0.f, 0.f, 0.f}, tv[3][INV_MAX_POLES];
    const bool disp = a.P > 0 && cell;
    for (int c = 0; c < 3; ++c) {
        if (!disp || !upd[c]) continue;
        float ph = 0.f;
        for (int p = 0; p < a.P; ++p) {
            const float ee = b.dc[p * a.n + o], eq = b.dc[(a.P + p) * a.n + o], zt = b.dc[(2 * a.P + p) * a.n + o];
            const float t = b.T[(c * a.P + p) * a.n + o];
            ph = ph + ee * t;
            tv[c][p] = eq * t + zt * e[c];
        }
        phi[c] = ph;
    }
    if (upd[0]) e[0] = CA * e[0] + CB * d2y - CB * d1z;
    if (upd[1]) e[1] = CA * e[1] + CB * d0z - CB * d2x;
    if (upd[2]) e[2] = CA * e[2] + CB * d1x - CB * d0y;
    if (disp)
        for (int c = 0; c < 3; ++c)
            if (upd[c]) e[c] = e[c] - IEA * phi[c];
    for (int s = 0; s < a.nslab; ++s) {
        const InvSlab &S = a.slab[s];
        if (!in_e(S, i, j, k)) continue;
        int p;
        int q[2];
        pidx(S, true, i, j, k, p, q[0], q[1]);
        const float RA01 = S.RE[p] - 1.0f, RB0 = S.RE[S.t + p], RE0 = S.RE[2 * S.t + p], RF0 = S.RE[3 * S.t + p];
        for (int w = 0; w < 2; ++w) {
            int comp, src, sign;
            e_pair(S.axis, w, comp, src, sign);
            float *Phi = w == 0 ? S.PE1 : S.PE2;
            const float dd = dH(src, S.axis) / a.d;
            const float ph = Phi[q[w]];
            const float corr = IEA * (RA01 * dd + RB0 * ph);
            Phi[q[w]] = RE0 * ph - RF0 * dd;
            e[comp] = sign > 0 ? e[comp] + corr : e[comp] - corr;
        }
    }
    if (i == b.si && j == b.sj && k == b.sk) e[2] = e[2] - IEA * b.w * b.sfac;
    for (int c = 0; c < 3; ++c) {
        if (disp && upd[c])  // dispersive part B
            for (int p = 0; p < a.P; ++p)
                b.T[(c * a.P + p) * a.n + o] = tv[c][p] - b.dc[(2 * a.P + p) * a.n + o] * e[c];
        b.En[c * a.n + o] = e[c];
    }
    if (b.curl) {  // the curl of H^{n+1} in the form dL/dCB reads it, and phi^n
        b.curl[o] = d2y - d1z;
        b.curl[a.n + o] = d0z - d2x;
        b.curl[2 * a.n + o] = d1x - d0y;
        for (int c = 0; c < 3 && a.P; ++c) b.phi[c * a.n + o] = phi[c];
    }
}

// ------------------------------------------------------------------ adjoint
// dL/d(dd) of one E-PML term at E edge (comp of the pair w) of slab S; zero
// outside the slab's E box.
__device__ __forceinline__ float e_pml_ldd(const InvArgs &a, const InvSlab &S, int w, int i, int j, int k)
{
    if (i < 0 || j < 0 || k < 0 || i > a.nx || j > a.ny || k > a.nz || !in_e(S, i, j, k)) return 0.f;
    int comp, src, sign;
    e_pair(S.axis, w, comp, src, sign);
    int p;
    int q[2];
    pidx(S, true, i, j, k, p, q[0], q[1]);
    const float RA01 = S.RE[p] - 1.0f, RF0 = S.RE[3 * S.t + p];
    const int o = fidx(a, i, j, k);
    const float lF = at3(a, a.b.lE, comp, o);
    const float mu = (w == 0 ? S.PE1 : S.PE2)[q[w]];
    return (float)sign * at3(a, a.b.mat, 2, o) * RA01 * lF - RF0 * mu;
}

__device__ __forceinline__ float h_pml_ldd(const InvArgs &a, const InvSlab &S, int w, int i, int j, int k)
{
    if (i < 0 || j < 0 || k < 0 || i > a.nx || j > a.ny || k > a.nz || !in_h(S, i, j, k)) return 0.f;
    int comp, src, sign;
    h_pair(S.axis, w, comp, src, sign);
    int p;
    int q[2];
    pidx(S, false, i, j, k, p, q[0], q[1]);
    const float RA01 = S.RH[p] - 1.0f, RF0 = S.RH[3 * S.t + p];
    const float lF = at3(a, a.b.H, comp, fidx(a, i, j, k));
    const float mu = (w == 0 ? S.PH1 : S.PH2)[q[w]];
    return (float)sign * a.b.cH * RA01 * lF - RF0 * mu;
}

// CB of the cell of E edge (i, j, k) times lE_c there, when that edge is
// updated; DB times lH_c at H cell (i, j, k), likewise.
__device__ __forceinline__ float xi(const InvArgs &a, int c, int i, int j, int k)
{
    if (!e_upd(a, c, i, j, k)) return 0.f;
    const int o = fidx(a, i, j, k);
    return at3(a, a.b.mat, 1, o) * at3(a, a.b.lE, c, o);
}
__device__ __forceinline__ float eta(const InvArgs &a, int c, int i, int j, int k)
{
    if (!h_upd(a, c, i, j, k)) return 0.f;
    return a.b.DB * at3(a, a.b.H, c, fidx(a, i, j, k));
}

// Reverse of the E half of iteration n, one thread per grid point:
//   lH    += (dE^{n+1}/dH^{n+1})^T lE*      (curl and E-PML terms, a gather)
//   mE^n   = RE mE^{n+1} + (dE^{n+1}/dPhiE^n)^T lE*, into the Q arrays
//   gradients of the cell from lE*, the saved E^n and curl H^{n+1}.
__global__ void k_adj_e(InvArgs a)
{
    int i, j, k;
    if (!all_point(a, i, j, k) || k > a.nz) return;
    const InvStep &b = a.b;
    const int o = fidx(a, i, j, k);
    // Ex(i,j,k) = ... + CB (Hz(i,j,k) - Hz(i,j-1,k)) - CB (Hy(i,j,k) - Hy(i,j,k-1))
    // Ey(i,j,k) = ... + CB (Hx(i,j,k) - Hx(i,j,k-1)) - CB (Hz(i,j,k) - Hz(i-1,j,k))
    // Ez(i,j,k) = ... + CB (Hy(i,j,k) - Hy(i-1,j,k)) - CB (Hx(i,j,k) - Hx(i,j-1,k))
    float dh[3];
    dh[0] = xi(a, 1, i, j, k) - xi(a, 1, i, j, k + 1) - xi(a, 2, i, j, k) + xi(a, 2, i, j + 1, k);
    dh[1] = xi(a, 2, i, j, k) - xi(a, 2, i + 1, j, k) - xi(a, 0, i, j, k) + xi(a, 0, i, j, k + 1);
    dh[2] = xi(a, 0, i, j, k) - xi(a, 0, i, j + 1, k) - xi(a, 1, i, j, k) + xi(a, 1, i + 1, j, k);
    const float lE[3] = {at3(a, b.lE, 0, o), at3(a, b.lE, 1, o), at3(a, b.lE, 2, o)};
    const bool cell = i < a.nx && j < a.ny && k < a.nz;
    const float IEA = b.mat[2 * a.n + o];
    // E-PML: dd = (S(e) - S(e - axis)) / d uses H at the edge and at edge - axis,
    // so H here feeds the edge here (+) and the edge one step up the axis (-).
    for (int s = 0; s < a.nslab; ++s) {
        const InvSlab &S = a.slab[s];
        if (!in_box3(S.gE_lo, S.gE_hi, i, j, k)) continue;
        const bool own = in_e(S, i, j, k);
        int p = 0;
        int q[2] = {0, 0};
        if (own) pidx(S, true, i, j, k, p, q[0], q[1]);
        const int ip = i + (S.axis == 0), jp = j + (S.axis == 1), kp = k + (S.axis == 2);
        for (int w = 0; w < 2; ++w) {
            int comp, src, sign;
            e_pair(S.axis, w, comp, src, sign);
            dh[src] += (e_pml_ldd(a, S, w, i, j, k) - e_pml_ldd(a, S, w, ip, jp, kp)) / a.d;
            if (own && cell)
                (w == 0 ? S.QE1 : S.QE2)[q[w]] = S.RE[2 * S.t + p] * (w == 0 ? S.PE1 : S.PE2)[q[w]] +
                                                 (float)sign * IEA * S.RE[S.t + p] * lE[comp];
        }
    }
    for (int c = 0; c < 3; ++c) b.H[c * a.n + o] += dh[c];
    if (!cell) return;
    float gca = 0.f, gcb = 0.f, giea = 0.f;
    for (int c = 0; c < 3; ++c) {
        if (!e_upd(a, c, i, j, k)) continue;
        gca += lE[c] * at3(a, b.E, c, o);
        gcb += lE[c] * at3(a, b.curl, c, o);
    }
    if (i == b.si && j == b.sj && k == b.sk) giea += -lE[2] * b.w * b.sfac;
    for (int c = 0; c < 3 && a.P; ++c)
        if (e_upd(a, c, i, j, k)) giea += -lE[c] * at3(a, b.phi, c, o);
    b.grad[o] += gca;
    b.grad[a.n + o] += gcb;
    if (giea != 0.f) b.grad[2 * a.n + o] += giea;
}

// Reverse of the H half of iteration n (lH = dL/dH^{n+1}, complete):
//   lE^n   = CA lE* (+ the poles) on updated edges + (dH^{n+1}/dE^n)^T lH (a gather)
//   mH^n   = RE mH^{n+1} + (dH^{n+1}/dPhiH^n)^T lH, into the Q arrays
//   lT one iteration back, and lE* of iteration n-1 from it.
__global__ void k_adj_h(InvArgs a)
{
    int i, j, k;
    if (!all_point(a, i, j, k) || k > a.nz) return;
    const InvStep &b = a.b;
    const int o = fidx(a, i, j, k);
    // Hx(i,j,k) = Hx - DB (Ez(i,j+1,k) - Ez(i,j,k)) + DB (Ey(i,j,k+1) - Ey(i,j,k))
    // Hy(i,j,k) = Hy - DB (Ex(i,j,k+1) - Ex(i,j,k)) + DB (Ez(i+1,j,k) - Ez(i,j,k))
    // Hz(i,j,k) = Hz - DB (Ey(i+1,j,k) - Ey(i,j,k)) + DB (Ex(i,j+1,k) - Ex(i,j,k))
    float de[3];
    de[0] = eta(a, 1, i, j, k) - eta(a, 1, i, j, k - 1) - eta(a, 2, i, j, k) + eta(a, 2, i, j - 1, k);
    de[1] = eta(a, 2, i, j, k) - eta(a, 2, i - 1, j, k) - eta(a, 0, i, j, k) + eta(a, 0, i, j, k - 1);
    de[2] = eta(a, 0, i, j, k) - eta(a, 0, i, j - 1, k) - eta(a, 1, i, j, k) + eta(a, 1, i - 1, j, k);
    const float lH[3] = {at3(a, b.H, 0, o), at3(a, b.H, 1, o), at3(a, b.H, 2, o)};
    // H-PML: dd = (S(h + axis) - S(h)) / d, so E here feeds the cell here (-)
    // and the cell one step down the axis (+).
    for (int s = 0; s < a.nslab; ++s) {
        const InvSlab &S = a.slab[s];
        if (!in_box3(S.gH_lo, S.gH_hi, i, j, k)) continue;
        const bool own = in_h(S, i, j, k);
        int p = 0;
        int q[2] = {0, 0};
        if (own) pidx(S, false, i, j, k, p, q[0], q[1]);
        const int im = i - (S.axis == 0), jm = j - (S.axis == 1), km = k - (S.axis == 2);
        for (int w = 0; w < 2; ++w) {
            int comp, src, sign;
            h_pair(S.axis, w, comp, src, sign);
            de[src] += (h_pml_ldd(a, S, w, im, jm, km) - h_pml_ldd(a, S, w, i, j, k)) / a.d;
            if (own)
                (w == 0 ? S.QH1 : S.QH2)[q[w]] = S.RH[2 * S.t + p] * (w == 0 ? S.PH1 : S.PH2)[q[w]] +
                                                 (float)sign * b.cH * S.RH[S.t + p] * lH[comp];
        }
    }
    const float CA = b.mat[o], IEA = b.mat[2 * a.n + o];
    for (int c = 0; c < 3; ++c) {
        const float l = at3(a, b.lE, c, o);
        float out = l;
        const bool upd = e_upd(a, c, i, j, k);
        if (upd) {
            float add = 0.f;
            for (int p = 0; p < a.P; ++p) {
                const float ee = b.dc[p * a.n + o], eq = b.dc[(a.P + p) * a.n + o], zt = b.dc[(2 * a.P + p) * a.n + o];
                float *lt = b.T + (c * a.P + p) * a.n + o;
                add = add + zt * *lt;
                *lt = eq * *lt - IEA * ee * l;
            }
            out = CA * l;
            if (a.P) out = out + add;
        }
        out = out + de[c];
        const int row = i * (a.ny + 1) + j;
        for (int r = b.rxfirst[row]; c == 2 && r < b.rxfirst[row + 1]; ++r)
            if (b.rxat[2 * r] == k) out += b.resid[(long long)b.rxat[2 * r + 1] * b.iterations + b.it];
        for (int p = 0; p < a.P && upd; ++p)
            out = out - b.dc[(2 * a.P + p) * a.n + o] * b.T[(c * a.P + p) * a.n + o];
        b.lE[c * a.n + o] = out;
    }
}

// Cells [nx][ny][nz] of `count` dense arrays to points (0 where a point is no
// cell), and back.
__global__ void k_inv_to_points(InvArgs a, const float *cells, float *points, int count)
{
    int i, j, k;
    if (!all_point(a, i, j, k) || k >= a.kp) return;
    const bool cell = i < a.nx && j < a.ny && k < a.nz;
    const long long all = (long long)a.nx * a.ny * a.nz, at = ((long long)i * a.ny + j) * a.nz + k;
    for (int q = 0; q < count; ++q) points[q * a.n + fidx(a, i, j, k)] = cell ? cells[q * all + at] : 0.f;
}
__global__ void k_inv_to_cells(InvArgs a, const float *points, float *cells, int count)
{
    int i, j, k;
    if (!all_point(a, i, j, k) || i >= a.nx || j >= a.ny || k >= a.nz) return;
    const long long all = (long long)a.nx * a.ny * a.nz, at = ((long long)i * a.ny + j) * a.nz + k;
    for (int q = 0; q < count; ++q) cells[q * all + at] = points[q * a.n + fidx(a, i, j, k)];
}

}  // namespace

// ====================================================================== host
constexpr int INV_DENSE = 3;

struct gpx_inv {
    gpx_inv_desc desc;
    int kp = 0;                    // floats per row of points
    long long n = 0, ncell = 0;    // floats of one component (every row of points, rounded up to 64)
    hipStream_t stream = nullptr;
    float *F = nullptr;            // E, H: 6 n
    float *L = nullptr;            // adjoint lE, lH: 6 n
    float *ck = nullptr;           // checkpoints: nck x ck_stride
    float *seg = nullptr;          // segment store: K x seg_stride
    float *par = nullptr;          // CA, CB, IEA: 3 n
    float *grad = nullptr;         // gCA, gCB, gIEA: 3 n
    float *dense = nullptr;        // INV_DENSE x ncell: parameters or gradients as the caller has them
    int P = 0;                     // Debye poles
    float *dc = nullptr;           // ee, eqt, zt: 3 P n
    float *T = nullptr;            // T of Ex, Ey, Ez: 3 P n
    float *LT = nullptr;           // its adjoint
    std::vector<float> waves;
    int *rxtab = nullptr;          // InvStep's rxat, then rxfirst
    size_t nrxseg = 0;             // segments of rxfirst
    bool rowrx = false;            // the device's RowModel points to them
    float *traces = nullptr, *resid = nullptr;
    int nrx = 0, si = -1, sj = -1, sk = -1;
    float sfac = 0;
    bool have_model = false, have_forward = false;
    struct Slab {
        InvSlab s;
        int dir;
        std::vector<float> R[2];         // E, H profiles: RA, RB, RE, RF
        long long n[4] = {0, 0, 0, 0};   // Phi sizes
        float *phi[4] = {nullptr, nullptr, nullptr, nullptr};
        float *mu[4] = {nullptr, nullptr, nullptr, nullptr};
        float *mu2[4] = {nullptr, nullptr, nullptr, nullptr};  // second copies
        float *dR = nullptr;             // E then H tables, 8 t floats
    };
    std::vector<Slab> slabs;
    // Which kernels run the model, decided when its slabs or poles have changed
    // (prepare).  Row kernels: their description, and the Phi of all slabs, per
    // field 2 x np floats (term 1, term 2).
    bool dirty = true, rows = false;
    RowModel *row = nullptr;
    float *img = nullptr;          // its tables (row_stage)
    uint32_t *planeflag = nullptr; // [nx + 1]
    std::vector<uint32_t> slabflag;
    int items = 0;
    int pseg = 0;                  // segments of a plane
    size_t lds[2] = {0, 0};        // of the E and the H passes
    long long np = 0;
    float *phi[2] = {nullptr, nullptr}, *mu[2][2] = {{nullptr, nullptr}, {nullptr, nullptr}};  // [E, H], [copy]
    long long phi_total = 0;       // floats of the forward's Phi
    float ms_fwd = 0, ms_bwd = 0;
    // Segments whose stored states the forward keeps (gpx_inv_set_keep): the
    // last nkeep segments, each K x seg_stride floats, in `keep`; the backward
    // then skips their recompute.
    double keep_bytes = 0;
    float *keep = nullptr;
    long long keep_floats = 0;     // size of `keep`
    int nkeep = 0;                 // segments kept by the last forward
    std::string err;
};

static thread_local std::string g_inv_err;   // as g_err in gpx.hip

static int ifail(gpx_inv *v, int code, const std::string &m)
{
    if (v) v->err = m;
    else g_inv_err = m;
    return code;
}

#define INV_TRY(call)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) return ifail(v, (int)e_, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

extern "C" const char *gpx_inv_last_error(const gpx_inv *v)
{
    return v ? v->err.c_str() : g_inv_err.c_str();
}

template <class T>
static void ifree(T *&p)
{
    if (p) hipFree(p);
    p = nullptr;
}

extern "C" int gpx_inv_create(const gpx_inv_desc *d, gpx_inv **out)
{
    if (!d || !out) return ifail(nullptr, GPX_EARG, "gpx_inv_create: null argument");
    *out = nullptr;
    if (d->nx < 2 || d->ny < 2 || d->nz < 2 || d->iterations < 1 || d->K < 1 || !(d->d > 0) || !(d->dt > 0))
        return ifail(nullptr, GPX_EARG, "gpx_inv_create: bad descriptor");
    if (d->nx + 1 > 65535 || d->ny + 1 > 65535)
        return ifail(nullptr, GPX_ELIMIT, "gpx_inv_create: at most 65534 cells along x and y");
    const double rows = (double)(d->nx + 1) * (d->ny + 1);
    if (rows * (d->nz + 1) >= 2147483647.0)
        return ifail(nullptr, GPX_ELIMIT, "gpx_inv_create: at most 2^31 grid points");
    if (hipSetDevice(d->device) != hipSuccess) return ifail(nullptr, GPX_EARG, "gpx_inv_create: bad device");
    gpx_inv *v = new gpx_inv();
    v->desc = *d;
    v->kp = (d->nz + 4) & ~3;
    if (rows * v->kp >= 2147483647.0) v->kp = d->nz + 1;
    v->n = ((long long)(d->nx + 1) * (d->ny + 1) * v->kp + 63) / 64 * 64;
    v->ncell = (long long)d->nx * d->ny * d->nz;
    const size_t b = (size_t)v->n * 4;
    hipError_t e = hipStreamCreateWithFlags(&v->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc((void **)&v->F, 6 * b);
    if (e == hipSuccess) e = hipMalloc((void **)&v->L, 6 * b);
    if (e == hipSuccess) e = hipMalloc((void **)&v->seg, (size_t)d->K * 6 * b);
    if (e == hipSuccess) e = hipMalloc((void **)&v->par, 3 * b);
    if (e == hipSuccess) e = hipMalloc((void **)&v->grad, 3 * b);
    if (e == hipSuccess) e = hipMalloc((void **)&v->dense, INV_DENSE * v->ncell * 4);
    if (e != hipSuccess) {
        gpx_inv_destroy(v);
        return ifail(nullptr, (int)e, std::string("gpx_inv_create: ") + hipGetErrorString(e));
    }
    *out = v;
    return 0;
}

// Phi and its adjoints of both layouts.
static void free_phi(gpx_inv *v)
{
    for (auto &S : v->slabs)
        for (int q = 0; q < 4; ++q) {
            ifree(S.phi[q]);
            ifree(S.mu[q]);
            ifree(S.mu2[q]);
        }
    for (int f = 0; f < 2; ++f) {
        ifree(v->phi[f]);
        ifree(v->mu[f][0]);
        ifree(v->mu[f][1]);
    }
}

extern "C" int gpx_inv_destroy(gpx_inv *v)
{
    if (!v) return 0;
    hipSetDevice(v->desc.device);
    if (v->stream) hipStreamSynchronize(v->stream);
    for (float *p : {v->F, v->L, v->ck, v->seg, v->par, v->grad, v->dense, v->traces, v->resid, v->dc, v->T, v->LT,
                     v->keep, v->img})
        if (p) hipFree(p);
    ifree(v->rxtab);
    ifree(v->row);
    ifree(v->planeflag);
    free_phi(v);
    for (auto &S : v->slabs) ifree(S.dR);
    if (v->stream) hipStreamDestroy(v->stream);
    delete v;
    return 0;
}

extern "C" int gpx_inv_add_pml(gpx_inv *v, int dir, int xs, int xf, int ys, int yf, int zs, int zf,
                               const float *eR, const float *hR)
{
    if (!v || !eR || !hR || dir < 0 || dir > 5) return ifail(v, GPX_EARG, "gpx_inv_add_pml: bad argument");
    if ((int)v->slabs.size() >= INV_MAX_SLABS) return ifail(v, GPX_ELIMIT, "gpx_inv_add_pml: at most 6 slabs");
    const gpx_inv_desc &g = v->desc;
    if (xs < 0 || ys < 0 || zs < 0 || xf > g.nx || yf > g.ny || zf > g.nz || xs >= xf || ys >= yf || zs >= zf)
        return ifail(v, GPX_EARG, "gpx_inv_add_pml: slab box outside the grid");
    hipSetDevice(g.device);
    gpx_inv::Slab S;
    InvSlab &s = S.s;
    memset(&s, 0, sizeof(s));
    const int axis = dir % 3, minus = dir < 3;
    const int st[3] = {xs, ys, zs}, en[3] = {xf, yf, zf};
    const int t = en[axis] - st[axis];
    S.dir = dir;
    s.axis = axis;
    s.minus = minus;
    s.t = t;
    for (int n = 0; n < 3; ++n) {
        s.loE[n] = s.loH[n] = st[n];
        s.hiE[n] = s.hiH[n] = en[n];
        s.org[n] = st[n];
    }
    if (minus) {  // E cells f - p, H cells f - (p + 1)
        s.loE[axis] = en[axis] - t + 1;
        s.hiE[axis] = en[axis] + 1;
        s.pendE = en[axis];
        s.loH[axis] = en[axis] - t;
        s.hiH[axis] = en[axis];
        s.pendH = en[axis] - 1;
    } else {
        s.loE[axis] = s.loH[axis] = st[axis];
        s.hiE[axis] = s.hiH[axis] = st[axis] + t;
        s.pendE = s.pendH = st[axis];
    }
    for (int q = 0; q < 3; ++q) {
        s.gE_lo[q] = s.loE[q] - (q == axis);
        s.gE_hi[q] = s.hiE[q];
        s.gH_lo[q] = s.loH[q];
        s.gH_hi[q] = s.hiH[q] + (q == axis);
    }
    // Phi shapes of gprMax/pml.py:202-219 (order 1)
    const int nx = xf - xs, ny = yf - ys, nz = zf - zs;
    int dims[4][3];
    if (axis == 0) {
        const int d4[4][3] = {{nx + 1, ny, nz + 1}, {nx + 1, ny + 1, nz}, {nx, ny + 1, nz}, {nx, ny, nz + 1}};
        memcpy(dims, d4, sizeof(dims));
    } else if (axis == 1) {
        const int d4[4][3] = {{nx, ny + 1, nz + 1}, {nx + 1, ny + 1, nz}, {nx + 1, ny, nz}, {nx, ny, nz + 1}};
        memcpy(dims, d4, sizeof(dims));
    } else {
        const int d4[4][3] = {{nx, ny + 1, nz + 1}, {nx + 1, ny, nz + 1}, {nx + 1, ny, nz}, {nx, ny + 1, nz}};
        memcpy(dims, d4, sizeof(dims));
    }
    for (int n = 0; n < 3; ++n) {
        s.dE1[n] = dims[0][n];
        s.dE2[n] = dims[1][n];
        s.dH1[n] = dims[2][n];
        s.dH2[n] = dims[3][n];
    }
    for (int q = 0; q < 4; ++q) S.n[q] = (long long)dims[q][0] * dims[q][1] * dims[q][2];
    S.R[0].assign(eR, eR + 4 * t);
    S.R[1].assign(hR, hR + 4 * t);
    INV_TRY(hipMalloc((void **)&S.dR, (size_t)8 * t * 4));
    hipError_t e = hipMemcpy(S.dR, eR, (size_t)4 * t * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(S.dR + 4 * t, hR, (size_t)4 * t * 4, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        ifree(S.dR);
        return ifail(v, (int)e, std::string("gpx_inv_add_pml: ") + hipGetErrorString(e));
    }
    s.RE = S.dR;
    s.RH = S.dR + 4 * t;
    v->slabs.push_back(S);
    v->dirty = true;
    v->have_forward = false;
    return 0;
}

static InvArgs inv_args(const gpx_inv *v);
static dim3 grid_all(const gpx_inv *v)
{
    return dim3((unsigned)(8 * inv_args(v).all_per_xcd));
}

// `count` arrays of cells from the host to points (the caller waits).  All that
// `dense` holds go over in one launch.
static int upload_cells(gpx_inv *v, const float *const *src, int count, float *dst)
{
    for (int q = 0; q < count; q += INV_DENSE) {
        const int m = count - q < INV_DENSE ? count - q : INV_DENSE;
        for (int p = 0; p < m; ++p)
            INV_TRY(hipMemcpyAsync(v->dense + p * v->ncell, src[q + p], (size_t)v->ncell * 4, hipMemcpyHostToDevice, v->stream));
        hipLaunchKernelGGL(k_inv_to_points, grid_all(v), dim3(128), 0, v->stream, inv_args(v), v->dense, dst + q * v->n, m);
        INV_TRY(hipGetLastError());
    }
    return 0;
}

extern "C" int gpx_inv_set_model(gpx_inv *v, const float *CA, const float *CB, const float *IEA)
{
    if (!v || !CA || !CB || !IEA) return ifail(v, GPX_EARG, "gpx_inv_set_model: null argument");
    hipSetDevice(v->desc.device);
    const float *src[3] = {CA, CB, IEA};
    if (int rc = upload_cells(v, src, 3, v->par)) return rc;
    INV_TRY(hipStreamSynchronize(v->stream));
    v->have_model = true;
    v->have_forward = false;
    return 0;
}

extern "C" int gpx_inv_set_dispersive(gpx_inv *v, int P, const float *ee, const float *eqt, const float *zt)
{
    if (!v || P < 0 || P > INV_MAX_POLES || (P > 0 && (!ee || !eqt || !zt)))
        return ifail(v, GPX_EARG, "gpx_inv_set_dispersive: bad argument (at most 4 poles)");
    hipSetDevice(v->desc.device);
    const size_t b = (size_t)v->n * 4;
    v->have_forward = false;
    if (P != v->P || !v->seg) {
        auto drop = [&] {
            for (float **p : {&v->dc, &v->T, &v->LT, &v->ck, &v->seg}) ifree(*p);
        };
        drop();
        v->P = P;
        v->dirty = true;
        // the segment store keeps phi^n of the three E components beside E^n, curl H^{n+1}
        hipError_t e = hipMalloc((void **)&v->seg, (size_t)v->desc.K * (P ? 9 : 6) * b);
        for (float **p : {&v->dc, &v->T, &v->LT})
            if (e == hipSuccess && P) e = hipMalloc((void **)p, (size_t)3 * P * b);
        if (e != hipSuccess) {   // none of them: no forward until this has succeeded
            drop();
            return ifail(v, (int)e, std::string("gpx_inv_set_dispersive: ") + hipGetErrorString(e));
        }
    }
    const float *src[3 * INV_MAX_POLES];
    for (int q = 0; q < 3 * P; ++q) src[q] = (q < P ? ee : (q < 2 * P ? eqt : zt)) + q % P * v->ncell;
    if (int rc = upload_cells(v, src, 3 * P, v->dc)) return rc;
    INV_TRY(hipStreamSynchronize(v->stream));
    return 0;
}

static int n_checkpoints(const gpx_inv *v) { return (v->desc.iterations + v->desc.K - 1) / v->desc.K; }
static long long ck_stride(const gpx_inv *v) { return 6 * v->n + 3 * v->P * v->n + v->phi_total; }
// Floats per iteration in the segment store: E^n, curl H^{n+1} and, with poles,
// phi^n, three components each.
static long long seg_stride(const gpx_inv *v) { return (v->P ? 9 : 6) * v->n; }

// Floats of one field's tables (row_stage).
static int inv_image(const gpx_inv *v)
{
    int nRT = 0;
    for (const auto &S : v->slabs) nRT += 4 * S.s.t;
    return row_image(0, nRT, 0);
}
static size_t inv_lds(const gpx_inv *v) { return (size_t)inv_image(v) * 4 + 16; }

// Whether the row kernels can run the model: whole lanes, slabs in direction
// order with the two of an axis at least four cells apart (so that a lane and
// its neighbours see one of them), a cell size row_quot takes, 32-bit byte
// offsets into arrays of three components (three per pole) and into a Phi array,
// and profiles that fit the LDS.
static bool inv_rows_ok(const gpx_inv *v)
{
    const gpx_inv_desc &g = v->desc;
    if (v->kp % 4 != 0 || !(g.d > 1e-12f && g.d < 1.6e7f)) return false;
    if ((double)v->n * 12.0 * (v->P > 1 ? v->P : 1) >= 4294967295.0) return false;
    int before = -1, end[3] = {-4, -4, -4};
    double np = 0;
    for (const auto &S : v->slabs) {
        const InvSlab &s = S.s;
        const int ax = s.axis, lo = s.loE[ax] < s.loH[ax] ? s.loE[ax] : s.loH[ax];
        if (S.dir <= before || lo - end[ax] < 4) return false;
        before = S.dir;
        end[ax] = s.hiE[ax] > s.hiH[ax] ? s.hiE[ax] : s.hiH[ax];
        np += ((double)s.hiE[0] - s.loE[0]) * ((double)s.hiE[1] - s.loE[1]) * ((double)s.hiE[2] - s.loE[2] + 8);
    }
    return np * 8.0 < 2147483647.0 && inv_lds(v) <= (size_t)MAX_LDS_BYTES;
}

// Settles the kernels of a model whose slabs or poles have changed, and lays
// the Phi arrays out for them.
static int prepare(gpx_inv *v)
{
    if (!v->dirty) return 0;
    const gpx_inv_desc &g = v->desc;
    INV_TRY(hipStreamSynchronize(v->stream));
    free_phi(v);
    ifree(v->ck);
    v->rows = inv_rows_ok(v);
    v->phi_total = 0;
    if (!v->rows) {
        for (auto &S : v->slabs)
            for (int q = 0; q < 4; ++q) {
                for (float **p : {&S.phi[q], &S.mu[q], &S.mu2[q]}) INV_TRY(hipMalloc((void **)p, S.n[q] * 4));
                v->phi_total += S.n[q];
            }
        v->dirty = false;
        return 0;
    }
    RowModel m;
    memset(&m, 0, sizeof(m));
    m.nx = g.nx; m.ny = g.ny; m.nz = g.nz;
    m.kp = v->kp;
    m.plane = (g.ny + 1) * v->kp;
    m.cs = (uint32_t)(v->n * 4);
    const double mu0 = 1.25663706127e-6;
    m.h[0] = 1.0f;
    m.h[1] = m.h[2] = m.h[3] = (float)((1.0 / g.d) * (g.dt / mu0));
    m.h[4] = (float)(g.dt / mu0);
    const int nI = inv_image(v);
    int nRT = 0;
    for (const auto &S : v->slabs) nRT += 4 * S.s.t;
    std::vector<float> img((size_t)2 * nI + 4, 0.f);
    v->slabflag.assign(g.nx + 1, 0u);
    long long np = 0;
    int first = 0;
    for (const auto &S : v->slabs) {
        const InvSlab &s = S.s;
        int ext[3];
        for (int q = 0; q < 3; ++q) ext[q] = s.hiE[q] - s.loE[q];
        const int aE = s.loE[2] & ~3, aH = s.loH[2] & ~3;   // cell k at k mod 4
        const int nk = ((s.hiE[2] - aE > s.hiH[2] - aH ? s.hiE[2] - aE : s.hiH[2] - aH) + 3) & ~3;
        for (int f = 0; f < 2; ++f) {
            RowSlab d;
            memset(&d, 0, sizeof(d));
            d.t = s.t;
            d.pend = f ? s.pendH : s.pendE;
            d.sign = s.minus ? -1 : 1;
            for (int q = 0; q < 3; ++q) {
                d.lo[q] = f ? s.loH[q] : s.loE[q];
                d.hi[q] = f ? s.hiH[q] : s.hiE[q];
            }
            d.sy = nk;
            d.sx = ext[1] * nk;
            d.off = (int)(np - (long long)d.lo[0] * d.sx - (long long)d.lo[1] * d.sy - (d.lo[2] & ~3));
            d.rt = first;
            d.d = g.d;
            d.rd = (float)(1.0 / (double)g.d);
            d.rl = (float)(1.0 / (double)g.d - (double)d.rd);
            float *rt = img.data() + f * nI, *sl = rt + nRT;
            for (int p = 0; p < s.t; ++p) {
                float *e = rt + first + 4 * p;
                const float *R = S.R[f].data();
                e[0] = R[p] - 1.0f;
                e[1] = R[s.t + p];
                e[2] = R[2 * s.t + p];
                e[3] = R[3 * s.t + p];
            }
            memcpy(sl + S.dir * (sizeof(RowSlab) / 4), &d, sizeof(d));
            const RowAt w = {d.lo[1], d.hi[1], d.lo[2], d.hi[2], d.off, d.sx, d.sy, 0};
            (f ? m.atH : m.atE)[S.dir] = w;
            for (int i = d.lo[0]; i < d.hi[0] && i <= g.nx; ++i)
                v->slabflag[i] |= 1u << ((f ? PF_SLAB_H : PF_SLAB_E) + S.dir);
        }
        first += 4 * s.t;
        np += (long long)ext[0] * ext[1] * nk;
    }
    v->np = np;
    v->phi_total = 4 * np;
    for (int f = 0; f < 2 && np; ++f)
        for (float **p : {&v->phi[f], &v->mu[f][0], &v->mu[f][1]}) INV_TRY(hipMalloc((void **)p, (size_t)2 * np * 4 + 16));
    ifree(v->img);
    INV_TRY(hipMalloc((void **)&v->img, img.size() * 4));
    INV_TRY(hipMemcpy(v->img, img.data(), img.size() * 4, hipMemcpyHostToDevice));
    m.img = reinterpret_cast<const float4 *>(v->img);
    m.n4E = m.n4H = nI / 4;
    m.nRT = nRT;
    m.np4 = (uint32_t)(np * 4);
    if (!v->planeflag) INV_TRY(hipMalloc((void **)&v->planeflag, (size_t)(g.nx + 1) * 4));
    m.planeflag = v->planeflag;
    // launch shape, as the solver's row passes (pass_items there)
    const int lanes = (g.ny + 1) * (v->kp / NC);
    m.pseg = (lanes + 255) / 256;
    for (m.pxc = 2;; --m.pxc) {
        m.pitems = m.pseg * ((g.nx + m.pxc) / m.pxc);
        if (m.pxc == 1 || m.pitems >= 1024) break;
    }
    v->items = m.pitems;
    v->pseg = m.pseg;
    v->lds[0] = v->lds[1] = inv_lds(v);
    if (!v->row) INV_TRY(hipMalloc((void **)&v->row, sizeof(RowModel)));
    INV_TRY(hipMemcpy(v->row, &m, sizeof(m), hipMemcpyHostToDevice));
    v->rowrx = false;
    v->dirty = false;
    return 0;
}

// What every launch of a kernel has in common.
static InvArgs inv_args(const gpx_inv *v)
{
    InvArgs a;
    memset(&a, 0, sizeof(a));
    const gpx_inv_desc &g = v->desc;
    a.nx = g.nx; a.ny = g.ny; a.nz = g.nz;
    a.kp = v->kp;
    a.n = v->n;
    a.d = g.d;
    const double mu0 = 1.25663706127e-6;
    InvStep &b = a.b;
    b.DB = (float)((1.0 / g.d) * (g.dt / mu0));
    b.cH = (float)(g.dt / mu0);
    b.mat = v->par;
    b.dc = v->dc;
    b.grad = v->grad;
    b.rxat = v->rxtab;
    b.rxfirst = v->rxtab + 2 * (size_t)v->nrx;
    b.resid = v->resid;
    b.traces = v->traces;
    b.iterations = g.iterations;
    b.si = v->si; b.sj = v->sj; b.sk = v->sk;
    b.sfac = v->sfac;
    b.nitems = v->items;
    b.per_xcd = (v->items + 7) / 8;
    a.P = v->P;
    a.nslab = (int)v->slabs.size();
    for (int s = 0; s < a.nslab; ++s) a.slab[s] = v->slabs[s].s;
    a.all_gk = (g.nz + 1 + 127) / 128;
    a.all_blocks = a.all_gk * (g.ny + 1) * (g.nx + 1);
    a.all_per_xcd = (a.all_blocks + 7) / 8;
    return a;
}

// Copies the state (fields, T and Phi) to or from checkpoint c.
static int checkpoint(gpx_inv *v, int c, bool save)
{
    float *at = v->ck + (long long)c * ck_stride(v);
    auto cp = [&](float *live, long long n) {
        float *ckp = at;
        at += n;
        return save ? hipMemcpyAsync(ckp, live, n * 4, hipMemcpyDeviceToDevice, v->stream)
                    : hipMemcpyAsync(live, ckp, n * 4, hipMemcpyDeviceToDevice, v->stream);
    };
    INV_TRY(cp(v->F, 6 * v->n));
    if (v->P) INV_TRY(cp(v->T, 3 * v->P * v->n));
    for (int f = 0; f < 2 && v->rows && v->np; ++f) INV_TRY(cp(v->phi[f], 2 * v->np));
    for (auto &S : v->slabs)
        for (int q = 0; q < 4 && !v->rows; ++q) INV_TRY(cp(S.phi[q], S.n[q]));
    return 0;
}

static InvKernels inv_kernels_of(const gpx_inv *v)
{
    return v->slabs.empty() ? inv_kernels<0>(v->P) : inv_kernels<1>(v->P);
}

// Forward iterations [n0, n1), one segment or the head of one.  With `store`
// they leave E^n, curl H^{n+1} (and phi^n) of each in its slot there: E^n is in
// slot n (copied there for the first) and E^{n+1} goes to slot n+1, after the
// last one back to the fields.
static int forward_steps(gpx_inv *v, int n0, int n1, float *store)
{
    InvArgs a = inv_args(v);
    InvStep &b = a.b;
    const InvKernels k = inv_kernels_of(v);
    for (int s = 0; s < a.nslab; ++s) {
        float *const *P = v->slabs[s].phi;
        a.slab[s].PE1 = P[0];
        a.slab[s].PE2 = P[1];
        a.slab[s].PH1 = P[2];
        a.slab[s].PH2 = P[3];
    }
    b.E = b.En = v->F;
    b.H = v->F + 3 * v->n;
    b.T = v->T;
    if (store && n0 < n1) INV_TRY(hipMemcpyAsync(store, v->F, (size_t)3 * v->n * 4, hipMemcpyDeviceToDevice, v->stream));
    for (int it = n0; it < n1; ++it) {
        b.it = it;
        b.w = v->waves[it];
        if (store) {
            float *slot = store + (long long)(it - n0) * seg_stride(v);
            b.E = slot;
            b.En = it + 1 < n1 ? slot + seg_stride(v) : v->F;
            b.curl = slot + 3 * v->n;
            b.phi = slot + 6 * v->n;
        }
        if (v->rows) {
            const dim3 G(8 * b.per_xcd);
            b.P = v->phi[1];
            hipLaunchKernelGGL(k.h, G, dim3(256), v->lds[1], v->stream, v->row, b);
            b.P = v->phi[0];
            hipLaunchKernelGGL(k.e, G, dim3(256), v->lds[0], v->stream, v->row, b);
        } else {
            const dim3 G(8 * a.all_per_xcd);
            hipLaunchKernelGGL(k_inv_h, G, dim3(128), 0, v->stream, a);
            hipLaunchKernelGGL(k_inv_e, G, dim3(128), 0, v->stream, a);
        }
    }
    INV_TRY(hipGetLastError());
    return 0;
}

extern "C" int gpx_inv_forward(gpx_inv *v, int si, int sj, int sk, float sfac, const float *waves, int nrx,
                               const int *rx, float *traces)
{
    if (!v || !waves || nrx < 0 || (nrx > 0 && (!rx || !traces)))
        return ifail(v, GPX_EARG, "gpx_inv_forward: bad argument");
    if (!v->have_model) return ifail(v, GPX_ESTATE, "gpx_inv_forward: no model uploaded");
    if (!v->seg) return ifail(v, GPX_ESTATE, "gpx_inv_forward: the poles of the last gpx_inv_set_dispersive were not set");
    const gpx_inv_desc &g = v->desc;
    if (si < 1 || si >= g.nx || sj < 1 || sj >= g.ny || sk < 0 || sk >= g.nz)
        return ifail(v, GPX_EARG, "gpx_inv_forward: source edge outside the updated Ez range");
    for (int r = 0; r < nrx; ++r)
        if (rx[3 * r] < 0 || rx[3 * r] > g.nx || rx[3 * r + 1] < 0 || rx[3 * r + 1] > g.ny || rx[3 * r + 2] < 0 ||
            rx[3 * r + 2] > g.nz)
            return ifail(v, GPX_EARG, "gpx_inv_forward: receiver outside the grid");
    hipSetDevice(g.device);
    v->have_forward = false;
    v->si = si; v->sj = sj; v->sk = sk;
    v->sfac = sfac;
    v->waves.assign(waves, waves + g.iterations);
    if (int rc = prepare(v)) return rc;
    const size_t groups = (size_t)(g.nx + 1) * (v->rows ? v->pseg : g.ny + 1);
    if (nrx != v->nrx || groups != v->nrxseg || !v->rxtab) {
        auto drop = [&] {
            ifree(v->rxtab);
            ifree(v->traces);
            ifree(v->resid);
            v->rowrx = false;
        };
        drop();
        v->nrx = nrx;
        v->nrxseg = groups;
        const size_t tb = (size_t)(nrx > 0 ? nrx : 1) * g.iterations * 4;
        hipError_t e = hipMalloc((void **)&v->rxtab, (2 * (size_t)nrx + groups + 1) * 4);
        if (e == hipSuccess) e = hipMalloc((void **)&v->traces, tb);
        if (e == hipSuccess) e = hipMalloc((void **)&v->resid, tb);
        if (e != hipSuccess) {
            drop();
            return ifail(v, (int)e, std::string("gpx_inv_forward: ") + hipGetErrorString(e));
        }
    }
    {  // the receivers by segments, those of one in their order, and their planes
        std::vector<int> tab(2 * (size_t)nrx + groups + 1, 0);
        int *first = tab.data() + 2 * (size_t)nrx;
        auto place = [&](int r, size_t &seg) {
            const int *x = rx + 3 * r, cell = x[1] * v->kp + x[2];
            seg = v->rows ? (size_t)x[0] * v->pseg + cell / (256 * NC) : (size_t)x[0] * (g.ny + 1) + x[1];
            return v->rows ? cell : x[2];
        };
        size_t seg;
        for (int r = 0; r < nrx; ++r) place(r, seg), ++first[seg + 1];
        for (size_t q = 0; q < groups; ++q) first[q + 1] += first[q];
        std::vector<int> next(first, first + groups);
        for (int r = 0; r < nrx; ++r) {
            const int at = place(r, seg), n = next[seg]++;
            tab[2 * (size_t)n] = at;
            tab[2 * (size_t)n + 1] = r;
        }
        INV_TRY(hipMemcpy(v->rxtab, tab.data(), tab.size() * 4, hipMemcpyHostToDevice));
        if (v->rows && !v->rowrx) {
            const int *at[2] = {v->rxtab + 2 * (size_t)nrx, v->rxtab};
            static_assert(offsetof(RowModel, rxat) == offsetof(RowModel, rxfirst) + sizeof(at[0]), "both in one copy");
            INV_TRY(hipMemcpy(&v->row->rxfirst, at, sizeof(at), hipMemcpyHostToDevice));
            v->rowrx = true;
        }
        if (v->rows) {
            std::vector<uint32_t> pf(v->slabflag);
            for (int r = 0; r < nrx; ++r) pf[rx[3 * r]] |= PF_RX;
            INV_TRY(hipMemcpy(v->planeflag, pf.data(), pf.size() * 4, hipMemcpyHostToDevice));
        }
    }
    if (!v->ck) INV_TRY(hipMalloc((void **)&v->ck, (size_t)n_checkpoints(v) * ck_stride(v) * 4));
    // the segments whose states this forward keeps
    const int nseg = n_checkpoints(v);
    const long long seg_floats = (long long)g.K * seg_stride(v);
    const double fit = v->keep_bytes / ((double)seg_floats * 4.0);
    const int nkeep = fit >= nseg ? nseg : (int)fit;
    if ((long long)nkeep * seg_floats != v->keep_floats) {
        if (v->keep) hipFree(v->keep);
        v->keep = nullptr;
        v->keep_floats = 0;
        v->nkeep = 0;
        v->have_forward = false;
        if (nkeep > 0) {
            const hipError_t e = hipMalloc((void **)&v->keep, (size_t)nkeep * seg_floats * 4);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                v->keep = nullptr;
                return ifail(v, (int)e, "gpx_inv_forward: cannot allocate " +
                                              std::to_string((double)nkeep * seg_floats * 4 / 1e9) +
                                              " GB for the kept segments (gpx_inv_set_keep)");
            }
            v->keep_floats = (long long)nkeep * seg_floats;
        }
    }
    v->nkeep = nkeep;
    INV_TRY(hipMemsetAsync(v->F, 0, (size_t)6 * v->n * 4, v->stream));
    if (v->P) INV_TRY(hipMemsetAsync(v->T, 0, (size_t)3 * v->P * v->n * 4, v->stream));
    for (int f = 0; f < 2 && v->rows && v->np; ++f) INV_TRY(hipMemsetAsync(v->phi[f], 0, (size_t)2 * v->np * 4, v->stream));
    for (auto &S : v->slabs)
        for (int q = 0; q < 4 && !v->rows; ++q) INV_TRY(hipMemsetAsync(S.phi[q], 0, S.n[q] * 4, v->stream));
    hipEvent_t e0, e1;
    INV_TRY(hipEventCreate(&e0));
    INV_TRY(hipEventCreate(&e1));
    INV_TRY(hipEventRecord(e0, v->stream));
    for (int c = 0; c < nseg; ++c) {
        const int n0 = c * g.K, n1 = n0 + g.K < g.iterations ? n0 + g.K : g.iterations;
        const bool kept = c >= nseg - nkeep;  // its states, no checkpoint
        if (!kept)
            if (int rc = checkpoint(v, c, true)) return rc;
        if (int rc = forward_steps(v, n0, n1, kept ? v->keep + (long long)(c - (nseg - nkeep)) * seg_floats : nullptr)) return rc;
    }
    INV_TRY(hipEventRecord(e1, v->stream));
    INV_TRY(hipEventSynchronize(e1));
    INV_TRY(hipEventElapsedTime(&v->ms_fwd, e0, e1));
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (nrx) INV_TRY(hipMemcpy(traces, v->traces, (size_t)nrx * g.iterations * 4, hipMemcpyDeviceToHost));
    v->have_forward = true;
    return 0;
}

extern "C" int gpx_inv_backward(gpx_inv *v, const float *resid, float *gCA, float *gCB, float *gIEA)
{
    if (!v || !gCA || !gCB || !gIEA || (v->nrx > 0 && !resid)) return ifail(v, GPX_EARG, "gpx_inv_backward: bad argument");
    if (!v->have_forward) return ifail(v, GPX_ESTATE, "gpx_inv_backward: run gpx_inv_forward first");
    const gpx_inv_desc &g = v->desc;
    hipSetDevice(g.device);
    if (v->nrx) INV_TRY(hipMemcpy(v->resid, resid, (size_t)v->nrx * g.iterations * 4, hipMemcpyHostToDevice));
    INV_TRY(hipMemsetAsync(v->L, 0, (size_t)6 * v->n * 4, v->stream));
    INV_TRY(hipMemsetAsync(v->grad, 0, (size_t)3 * v->n * 4, v->stream));
    if (v->P) INV_TRY(hipMemsetAsync(v->LT, 0, (size_t)3 * v->P * v->n * 4, v->stream));
    for (int f = 0; f < 2 && v->rows && v->np; ++f)
        for (float *p : v->mu[f]) INV_TRY(hipMemsetAsync(p, 0, (size_t)2 * v->np * 4, v->stream));
    for (auto &S : v->slabs)
        for (int q = 0; q < 4 && !v->rows; ++q) {
            INV_TRY(hipMemsetAsync(S.mu[q], 0, S.n[q] * 4, v->stream));
            INV_TRY(hipMemsetAsync(S.mu2[q], 0, S.n[q] * 4, v->stream));
        }
    InvArgs a = inv_args(v);
    InvStep &b = a.b;
    const InvKernels k = inv_kernels_of(v);
    b.lE = v->L;
    b.H = v->L + 3 * v->n;
    b.T = v->LT;
    int cur = 0;
    hipEvent_t e0, e1;
    INV_TRY(hipEventCreate(&e0));
    INV_TRY(hipEventCreate(&e1));
    INV_TRY(hipEventRecord(e0, v->stream));
    const int nseg = n_checkpoints(v);
    for (int c = nseg - 1; c >= 0; --c) {
        const int n0 = c * g.K, n1 = n0 + g.K < g.iterations ? n0 + g.K : g.iterations;
        const bool kept = c >= nseg - v->nkeep;
        float *base = kept ? v->keep + (long long)(c - (nseg - v->nkeep)) * g.K * seg_stride(v) : v->seg;
        // recompute the segment, storing E^n and curl H^{n+1} (kept segments have them)
        if (!kept) {
            if (int rc = checkpoint(v, c, false)) return rc;
            if (int rc = forward_steps(v, n0, n1, base)) return rc;
        }
        // adjoint sweep over the segment
        for (int it = n1 - 1; it >= n0; --it, cur ^= 1) {
            float *slot = base + (long long)(it - n0) * seg_stride(v);
            b.it = it;
            b.w = v->waves[it];
            b.E = slot;
            b.curl = slot + 3 * v->n;
            b.phi = slot + 6 * v->n;
            if (v->rows) {
                const dim3 G(8 * b.per_xcd);
                b.P = v->mu[0][cur];
                b.Q = v->mu[0][cur ^ 1];
                hipLaunchKernelGGL(k.adj_e, G, dim3(256), v->lds[0], v->stream, v->row, b);
                b.P = v->mu[1][cur];
                b.Q = v->mu[1][cur ^ 1];
                hipLaunchKernelGGL(k.adj_h, G, dim3(256), v->lds[1], v->stream, v->row, b);
                continue;
            }
            for (int s = 0; s < a.nslab; ++s) {
                const auto &S = v->slabs[s];
                float *const *P = cur == 0 ? S.mu : S.mu2;
                float *const *Q = cur == 0 ? S.mu2 : S.mu;
                a.slab[s].PE1 = P[0]; a.slab[s].PE2 = P[1]; a.slab[s].PH1 = P[2]; a.slab[s].PH2 = P[3];
                a.slab[s].QE1 = Q[0]; a.slab[s].QE2 = Q[1]; a.slab[s].QH1 = Q[2]; a.slab[s].QH2 = Q[3];
            }
            const dim3 G(8 * a.all_per_xcd);
            hipLaunchKernelGGL(k_adj_e, G, dim3(128), 0, v->stream, a);
            hipLaunchKernelGGL(k_adj_h, G, dim3(128), 0, v->stream, a);
        }
        INV_TRY(hipGetLastError());
    }
    INV_TRY(hipEventRecord(e1, v->stream));
    INV_TRY(hipEventSynchronize(e1));
    INV_TRY(hipEventElapsedTime(&v->ms_bwd, e0, e1));
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    float *out[3] = {gCA, gCB, gIEA};
    hipLaunchKernelGGL(k_inv_to_cells, grid_all(v), dim3(128), 0, v->stream, a, v->grad, v->dense, 3);
    INV_TRY(hipGetLastError());
    for (int q = 0; q < 3; ++q)
        INV_TRY(hipMemcpyAsync(out[q], v->dense + q * v->ncell, (size_t)v->ncell * 4, hipMemcpyDeviceToHost, v->stream));
    INV_TRY(hipStreamSynchronize(v->stream));
    return 0;
}

extern "C" int gpx_inv_set_keep(gpx_inv *v, double bytes)
{
    if (!v || !(bytes >= 0)) return ifail(v, GPX_EARG, "gpx_inv_set_keep: bad argument");
    v->keep_bytes = bytes;
    return 0;
}

extern "C" int gpx_inv_timings(const gpx_inv *v, float *ms_forward, float *ms_backward)
{
    if (!v) return GPX_EARG;
    if (ms_forward) *ms_forward = v->ms_fwd;
    if (ms_backward) *ms_backward = v->ms_bwd;
    return 0;
}
