// Row kernels of the time loop: the H and E passes as one launch each over every
// cell, in place (k_row_h, k_row_e), and the whole step as one launch, the
// state double-buffered (k_row_step).
//
// What bounds them.  A step is a stencil of about 0.2 flop/B, so on grids past
// the last-level cache the bytes set the time: six float32 components read and
// written (E and H twice over two passes), three uint16 indices (six when the H
// coefficients differ between materials) and the slabs' Phi.  Within the cache
// it is the slabs' instructions, and on small grids the number of launches and
// each one's chain of dependent accesses: the model's description, then in one
// round the tables, the plane's fields and the Phi, then the stores.
//
// Lanes.  Field rows (fixed i, j; z fastest) are padded to a multiple of four
// floats (rows of two, a 2-D model's, are not), and a lane owns two consecutive cells of a row: half the loads,
// stores and address work of a cell per lane, and registers (under 96 with a
// slab of order 1) for five waves on a SIMD.  Four cells a lane, with twice the
// registers, took 367 us where two take 349 (300x300x200) and 38.8 where two
// take 30.4 (100x100x100).
//
// Neighbours.  k+1 (of E) and k-1 (of H) are the next and the previous lane's,
// by a shift of the wave; its last or first lane loads them.  The passes load
// j+1 (j-1) beside, which the row above or below brings into the cache too, and
// keep plane i+1 (i-1) in registers.
//
// The step.  A block holds R rows of LT lanes and marches x.  New H at j-1 comes
// through LDS from the row below in the block, at k-1 across waves too, so each
// block also holds the row below its own rows (and one lane before its own
// lanes where rows are split), and each x chunk begins one plane early: there
// it computes H only and writes nothing.  The next state and the next H Phi are
// other arrays than the current ones, so no block reads what another writes.  E
// Phi and the dispersive auxiliary values are touched only by the lane that
// owns the cell, in place.
//
// Slabs.  A lane lies in at most one slab along each axis; what the slab adds to
// the two components it corrects depends on the differences and its Phi only,
// not on the components, so a lane works its up to three slabs out one after the
// other and adds the results in the slabs' order.  All Phi are loaded with the
// plane and stored after its last use: a wait for a later slab's Phi would
// wait for the earlier slab's stores.  With a loop over the slabs, each
// loading, adding and storing in turn, 100x100x100 took 28.1 us an iteration,
// now 22.5.
//
// Rounding.  Every expression is the one of the general passes, in the same
// order; the slabs' profile terms that do not depend on the fields are tabled
// on the host with the same operations, and the division by the cell size is
// the correctly rounded quotient (row_quot).
//
// Grids past the last-level cache go through the passes in blocks of planes, several
// iterations a block (run_wave in gpx.hip).
//
// Measured, us per iteration, two passes here and four (interior and boundary
// apart, one cell per lane) or two with one merged step before:
//   120x105 (2-D)  8.6 from 16.7     100x100x100   22.5 from 40.8
//   157x131x97 MRIPML order 2  45 from 72        300x300x200  276 from 425
//   611x407x45  200 from 375      240x240x180, 3 poles  269 from 478
#ifndef GPX_ROWS_H
#define GPX_ROWS_H

#include "gpx_step.h"

namespace gpx {

constexpr int NC = 2;   // cells per lane
typedef float fN __attribute__((ext_vector_type(NC)));
typedef uint32_t uN __attribute__((ext_vector_type(NC)));
typedef uint32_t idN __attribute__((ext_vector_type(NC / 2)));

constexpr int ROW_BLOCK_MAX = 512;   // threads of a k_row_step block
constexpr int ROW_PASS_MAX = 512;    // threads of a pass block
constexpr int ROW_LANES_MAX = 64;    // longest row segment of a block, in lanes

// Waves per SIMD the passes' registers are kept to: without spilling, and six
// instead of five cost 300x300x200 11 % in spills.
#define ROW_PASS_WAVES(P, ORDER) __attribute__((amdgpu_waves_per_eu((P) > 1 ? 3 : (ORDER) == 2 || (P) == 1 ? 4 : 5)))

// One slab for one field, by direction (x0, y0, z0, xmax, ymax, zmax; t = 0:
// none).  Phi index of cell (i, j, k): off + i sx + j sy + k, in floats; Phi of
// (order o, term w) begins (2 o + w) * np floats further on.
struct RowSlab {
    int t, pend, sign;     // thickness; profile entry of cell c: sign (c - pend), sign -1 for the minus slabs
    int lo[3], hi[3];      // corrected cells
    int off, sx, sy;
    int rt;                // first profile entry of the slab, in floats of the table
    float d, rd, rl;       // cell size, its rounded reciprocal and what that lacks of it (64 bytes in all)
};
typedef int RowAt __attribute__((ext_vector_type(8)));  // of a slab: lo[1], hi[1], lo[2], hi[2], off, sx, sy (zeros: none)

// Floats per profile entry: HORIPML and MRIPML of order 1: 4, HORIPML of order
// 2: 12, MRIPML of order 2: 8 (row_profile in gpx.hip fills them).
constexpr int row_entry(int form, int order) { return order == 2 ? (form == 0 ? 12 : 8) : 4; }

// A model as the row kernels see it; in device memory, read through the scalar
// cache.  State and Phi twice: launch arguments `flip` (E Phi:
// `flipE`) say which is current.
struct RowModel {
    int nx, ny, nz, kp, plane;       // kp: floats per row; plane = (ny + 1) kp
    int LT, LTo, hk, R, Ro, hj;      // lanes of a tile (own: LTo, halo: hk), rows (own: Ro, halo: hj)
    int za, zb;                      // lanes at the start and the end of a row with a cell in a z slab
    int ntk, ntj, xc, nitems;        // tiles along k and j, planes per chunk, work items
    int threads;                     // threads of a block that have a lane, in whole waves
    int pitems, pxc, pseg;           // the passes' items, planes per chunk, segments per plane
    float *F[2];
    uint32_t cs, ci;                 // bytes between components of a state / of the indices
    const uint16_t *ID;
    const float4 *img;               // tables for LDS: n4E float4 for E, then n4H for H (row_stage)
    int n4E, n4H;
    int nmat;
    float h[5];                      // the H coefficients when every material has the same
    int nRT;                         // floats of a field's profile table
    RowAt atE[6], atH[6];            // the slabs by direction
    float *phiE[2], *phiH[2];
    uint32_t np4;                    // bytes of one (order, term) block of Phi
    TArgs T;
    int iterations;
    const StepRare *rare;
    const uint32_t *planeflag;       // [nx + 1], slab bits by direction
    size_t csl, cil;                 // cs and ci where they pass 32 bits (RowComps)
    // Of the differentiable solver (inv_rows.h), receivers sorted by segments of planes
    // (a block's lanes): [segments + 1], a segment's first in rxat; [receivers][2],
    // point of the plane and number.
    const int *rxfirst, *rxat;
};

struct RowArgs {
    const int *item0;                // [ntr + 1]: first item of each model (unused with one)
    int ntr, nitems, per_xcd;
    int flip, flipE, it;
    int p0, p1;                      // the passes' planes (p1 past the last one: to the model's end)
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <class To, class From>
__device__ __forceinline__ To bits(From v)
{
    return __builtin_bit_cast(To, v);
}
__device__ __forceinline__ fN bldN(rsrc_t r, uint32_t voff, uint32_t soff)
{
    return bits<fN>(__builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ idN bld_ids(rsrc_t r, uint32_t voff, uint32_t soff)
{
    return bits<idN>(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ void bstN(rsrc_t r, uint32_t voff, uint32_t soff, fN v)
{
    __builtin_amdgcn_raw_buffer_store_b64(bits<u32x2>(v), r, voff, soff, 0);
}
// Components of a state or of the indices.  Offsets are 32-bit, so a state of
// 4 GiB and more (BIG) has a resource for each component, any other one for all.
// 620x600x500, us an iteration: 4230 in the general passes, 3060 so.
template <bool BIG>
struct RowComps {
    rsrc_t r[BIG ? 6 : 1];
    uint32_t cs;
    __device__ __forceinline__ RowComps(const void *base, uint32_t cs_, size_t csl) : cs(cs_)
    {
#pragma unroll
        for (int c = 0; c < (BIG ? 6 : 1); ++c) r[c] = rsrc(static_cast<const char *>(base) + (size_t)c * csl);
    }
    __device__ __forceinline__ rsrc_t at(int c) const { return r[BIG ? c : 0]; }
    __device__ __forceinline__ uint32_t off(int c, uint32_t so) const { return BIG ? so : so + (uint32_t)c * cs; }
};
// Flags of plane i, as a scalar load: no kernel writes them, which the compiler
// cannot see behind the model's pointer; a vector load in its place would make
// every plane wait for all its loads before it knew its slabs.
__device__ __forceinline__ uint32_t plane_flags(const RowModel &a, int i)
{
    typedef __attribute__((address_space(4))) const uint32_t cu32;
    return ((cu32 *)a.planeflag)[i];
}
__device__ __forceinline__ uint32_t id_of(idN m, int u) { return (m[u >> 1] >> (16 * (u & 1))) & 0xffffu; }
// The lane's cells shifted by one: cells 1.. then the next lane's first; the
// previous lane's last, then cells 0..
__device__ __forceinline__ fN shift_up(fN v, float next)
{
    fN r;
#pragma unroll
    for (int u = 0; u + 1 < NC; ++u) r[u] = v[u + 1];
    r[NC - 1] = next;
    return r;
}
__device__ __forceinline__ fN shift_down(fN v, float before)
{
    fN r;
    r[0] = before;
#pragma unroll
    for (int u = 1; u < NC; ++u) r[u] = v[u - 1];
    return r;
}

// The value of the next (previous) lane of the wave; its last (first) lane
// gets `edge`.
__device__ __forceinline__ float from_next(float edge, float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v),
                                                                 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ float from_prev(float edge, float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v),
                                                                 0x138, 0xf, 0xf, false));
}

// q = x / d for a lane's cells, correctly rounded, with rd + rl = 1 / d, rd the
// rounded reciprocal: x rl + x rd, rounded, is within one unit in the last
// place, and from there one step with the exact remainder (fma) gives the
// rounded quotient (Markstein's theorem).  That holds while |x| is zero or at
// least 2^-100 (d being a cell size, 2^-40 < d < 2^24): no quotient is then
// subnormal and every remainder is exact; and while the quotient is finite: for an
// infinite x, or one whose quotient overflows, the remainder is the difference
// of two infinities and q comes out as NaN.  `odd` collects what a cell had of
// either, for which the division itself is needed.  Four operations instead of the
// division's twelve.
struct RowOdd {
    uint32_t least = ~0u;    // twice the bits of the least x but zero, less one
    bool nan = false;        // a q is NaN
    __device__ __forceinline__ bool any() const { return (least < 27u << 24) | nan; }  // exponent field below 27
};
__device__ __forceinline__ void row_quot(fN x, const RowSlab &S, fN &q, RowOdd &odd)
{
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const float v = __builtin_fmaf(x[u], S.rd, x[u] * S.rl);
        q[u] = __builtin_fmaf(__builtin_fmaf(-v, S.d, x[u]), S.rd, v);
        const float xu = x[u];  // bit_cast of the element itself reads element 0
        const uint32_t b = __builtin_bit_cast(uint32_t, xu) * 2u - 1u;  // zero wraps to the largest
        odd.least = b < odd.least ? b : odd.least;
    }
    static_assert(NC == 2, "one comparison for a lane's two cells");
    odd.nan |= __builtin_isunordered(q[0], q[1]);
}

// Makes the compiler forget how a value was computed, so that what is derived
// from it again later is computed again instead of being kept in registers.
__device__ __forceinline__ void forget(fN &v) { asm volatile("" : "+v"(v)); }

// Waits for loads here.  Loads and stores share one in-order counter, and past
// a branch that may or may not have stored the compiler can only wait for
// everything: a value first used after this plane's stores would wait for
// the stores to reach memory.
template <class V>
__device__ __forceinline__ void arrived(V v)
{
    asm volatile("" : : "v"(v));
}
template <class V, class... W>
__device__ __forceinline__ void arrived(V v, W... w)
{
    arrived(v);
    arrived(w...);
}

// Phi of one slab for a lane's cells: terms 1 and 2, orders 0 and 1.
template <int ORDER>
struct RowPhi {
    uint32_t q;             // byte offset of the cells in (order 0, term 1)
    fN a[ORDER > 0 ? ORDER : 1], b[ORDER > 0 ? ORDER : 1];
};
template <int ORDER>
__device__ __forceinline__ void row_phi_load(RowPhi<ORDER> &p, int q, rsrc_t r, uint32_t np4)
{
    p.q = (uint32_t)q * 4u;
#pragma unroll
    for (int o = 0; o < ORDER; ++o) {
        p.a[o] = bldN(r, p.q, (uint32_t)(2 * o) * np4);
        p.b[o] = bldN(r, p.q, (uint32_t)(2 * o + 1) * np4);
    }
}
template <int ORDER>
__device__ __forceinline__ void row_phi_store(const RowPhi<ORDER> &p, rsrc_t w, uint32_t np4)
{
#pragma unroll
    for (int o = 0; o < ORDER; ++o) {
        bstN(w, p.q, (uint32_t)(2 * o) * np4, p.a[o]);
        bstN(w, p.q, (uint32_t)(2 * o + 1) * np4, p.b[o]);
    }
}

// The slabs of a lane, one at most along each axis (rows_ok): `x`, `y`, `z`
// bits of a slab mask, both sides.
constexpr uint32_t ROW_X = 9u, ROW_Y = 18u, ROW_Z = 36u;
template <int ORDER>
struct RowPhis {
    RowPhi<ORDER> x, y, z;
};

// One corrected component of cell u (gprMax/pml_updates/*_ext.pyx): e is the
// profile entry, dd the difference over the cell size, c the cell's srce or
// srcm; ph are the cell's Phi values, replaced by the advanced ones.
template <int FORM, int ORDER>
__device__ __forceinline__ float row_corr(const float *e, float c, float dd, float &p0, float &p1)
{
    if (FORM == 0 && ORDER == 1) {         // RA - 1, RB, RE, RF
        const float corr = c * (e[0] * dd + e[1] * p0);
        p0 = e[2] * p0 - e[3] * dd;
        return corr;
    }
    if (FORM == 0) {                        // RA0 RA1 - 1, RA1 RB0, RB1, RA0 | RB0, RE0, RF0, RE1 | RF1
        const float corr = c * (e[0] * dd + e[1] * p0 + e[2] * p1);
        p1 = e[7] * p1 - e[8] * (e[3] * dd + e[4] * p0);
        p0 = e[5] * p0 - e[6] * dd;
        return corr;
    }
    if (ORDER == 1) {                       // IRA - 1, IRA, RE, RC
        const float corr = c * (e[0] * dd - e[1] * p0);
        p0 = e[2] * p0 + e[3] * dd - e[3] * p0;
        return corr;
    }
    // IRA - 1, IRA, RB0, RB1 | RE0, RE1, RC0, RC1
    const float psi = e[2] * p0 + e[3] * p1;
    const float corr = c * (e[0] * dd - e[1] * psi);
    p1 = e[5] * p1 + e[7] * (dd - psi);
    p0 = e[4] * p0 + e[6] * (dd - psi);
    return corr;
}

// What one slab adds to its two corrected components on a lane's cells: A1
// (the correction, negative unless PLUS1) from the differences D1, A2 (the
// other sign) from D2; -0, which changes nothing, on cells outside the slab.
// ALONGK: the profile runs along k, else cell `c` of the slab's axis holds for
// all.
template <int FORM, int ORDER, bool PLUS1, bool ALONGK, class C1, class C2>
__device__ __forceinline__ void row_slab(const RowSlab &S, const float *RT, int c, int kl, fN D1, fN D2, fN &A1, fN &A2,
                                         const C1 &c1, const C2 &c2, RowPhi<ORDER> &ph)
{
    constexpr int NE = row_entry(FORM, ORDER);
    const int klo = S.lo[2], khi = S.hi[2], at = S.rt + S.sign * ((ALONGK ? kl : c) - S.pend) * NE;
    const int step = ALONGK ? S.sign * NE : 0;
    fN Q1, Q2;
    RowOdd odd;
    row_quot(D1, S, Q1, odd);
    row_quot(D2, S, Q2, odd);
    if (odd.any()) {
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            Q1[u] = D1[u] / S.d;
            Q2[u] = D2[u] / S.d;
        }
    }
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int k = kl + u;
        const bool in = (k >= klo) & (k < khi);
        const float4 *t = reinterpret_cast<const float4 *>(RT + (ALONGK ? (in ? at + u * step : 0) : at));
        float e[NE];
#pragma unroll
        for (int n = 0; n < NE / 4; ++n) {
            const float4 v = t[n];
            e[4 * n] = v.x; e[4 * n + 1] = v.y; e[4 * n + 2] = v.z; e[4 * n + 3] = v.w;
        }
        float a0 = ph.a[0][u], b0 = ph.b[0][u];
        float a1 = ORDER == 2 ? ph.a[ORDER - 1][u] : 0.f, b1 = ORDER == 2 ? ph.b[ORDER - 1][u] : 0.f;
        const float q1 = row_corr<FORM, ORDER>(e, c1(u), Q1[u], a0, a1);
        const float q2 = row_corr<FORM, ORDER>(e, c2(u), Q2[u], b0, b1);
        A1[u] = in ? (PLUS1 ? q1 : -q1) : -0.f;
        A2[u] = in ? (PLUS1 ? -q2 : q2) : -0.f;
        if (ORDER == 2) {
            ph.a[ORDER - 1][u] = in ? a1 : ph.a[ORDER - 1][u];
            ph.b[ORDER - 1][u] = in ? b1 : ph.b[ORDER - 1][u];
        }
        ph.a[0][u] = in ? a0 : ph.a[0][u];
        ph.b[0][u] = in ? b0 : ph.b[0][u];
    }
}

// f + first + second, in that order; `swap`: the second first.
__device__ __forceinline__ void row_add(fN &f, fN first, fN second, bool swap)
{
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const float p = swap ? second[u] : first[u], q = swap ? first[u] : second[u];
        f[u] = f[u] + p + q;
    }
}

// Where the slabs lie: read once, through the scalar cache, all six together.
struct RowAts {
    RowAt s[6];
};
__device__ __forceinline__ RowAts row_ats(const RowAt *at)
{
    typedef __attribute__((address_space(4))) const RowAt cat;
    RowAts r;
#pragma unroll
    for (int d = 0; d < 6; ++d) r.s[d] = ((cat *)at)[d];
    return r;
}

// Slabs whose box holds one of the lane's cells in y and z.
__device__ __forceinline__ uint32_t row_mask(const RowAts &at, int j, int kl)
{
    uint32_t m = 0;
#pragma unroll
    for (int d = 0; d < 6; ++d) {
        const RowAt s = at.s[d];
        const bool in = (j >= s[0]) & (j < s[1]) & (kl + NC - 1 >= s[2]) & (kl < s[3]);
        m |= in ? 1u << d : 0u;
    }
    return m;
}

// What a lane keeps of its slabs from plane to plane.
struct RowSlabs {
    uint32_t m = 0;         // those whose y, z box holds one of its cells
    int qy, sy, qz, sz;     // Phi index of its y slab's and its z slab's cells at plane 0, and from plane to plane
    RowAt x0, x1;
};
__device__ __forceinline__ RowSlabs row_slabs(const RowAt *at, int j, int kl, bool live)
{
    const RowAts r = row_ats(at);
    RowSlabs L;
    L.m = live ? row_mask(r, j, kl) : 0u;
    const bool ylo = L.m & 2u, zlo = L.m & 4u;
    L.qy = (ylo ? r.s[1][4] : r.s[4][4]) + j * (ylo ? r.s[1][6] : r.s[4][6]) + kl;
    L.sy = ylo ? r.s[1][5] : r.s[4][5];
    L.qz = (zlo ? r.s[2][4] : r.s[5][4]) + j * (zlo ? r.s[2][6] : r.s[5][6]) + kl;
    L.sz = zlo ? r.s[2][5] : r.s[5][5];
    L.x0 = r.s[0];
    L.x1 = r.s[3];
    return L;
}

// Loads, with the rest of a plane, the Phi of the lane's slabs m at plane i; xlo:
// the plane lies in the lower x slab.
template <int ORDER>
__device__ __forceinline__ void row_phis(RowPhis<ORDER> &p, const RowSlabs &L, uint32_t m, bool xlo, rsrc_t r, uint32_t np4,
                                         int i, int j, int kl)
{
    if (m & ROW_X) {
        const int off = xlo ? L.x0[4] : L.x1[4], sx = xlo ? L.x0[5] : L.x1[5], sy = xlo ? L.x0[6] : L.x1[6];
        row_phi_load(p.x, off + i * sx + j * sy + kl, r, np4);
    }
    if (m & ROW_Y) row_phi_load(p.y, L.qy + i * L.sy, r, np4);
    if (m & ROW_Z) row_phi_load(p.z, L.qz + i * L.sz, r, np4);
}
template <int ORDER>
__device__ __forceinline__ void row_phis_store(const RowPhis<ORDER> &p, uint32_t m, rsrc_t w, uint32_t np4)
{
    if (m & ROW_X) row_phi_store(p.x, w, np4);
    if (m & ROW_Y) row_phi_store(p.y, w, np4);
    if (m & ROW_Z) row_phi_store(p.z, w, np4);
}

// Tables of one model in LDS.
struct RowLds {
    const float4 *cE, *cH;
    const float *sE, *sH, *RTE, *RTH, *disp;
    const RowSlab *slE, *slH;
    fN *lx, *lz;            // [2][B]: new Hx and Hz of the block, planes alternating
    float *ly;              // [2][B]: new Hy of every lane's last cell
};

// Floats of one field's tables: [nmat] coefficients 1 to 4, profile entries, the
// six slabs, [nmat] coefficient 5, [nd] pole coefficients.
__host__ __device__ constexpr int row_image(int nmat, int nRT, int nd)
{
    return (5 * nmat + nRT + (nRT ? 6 * (int)(sizeof(RowSlab) / 4) : 0) + nd + 3) & ~3;
}

// Copies the tables, which the host has laid out as they lie here, to dynamic
// LDS: one round of loads (the caller synchronises).  DOE, DOH: the fields
// whose tables are needed; HU: uniform H coefficients, which take no table.
template <int ORDER, bool HU, bool DOE, bool DOH>
__device__ __forceinline__ RowLds row_stage(float4 *lds4, const RowModel &a)
{
    RowLds S;
    const int n4E = a.n4E, n = DOE ? (DOH ? n4E + a.n4H : n4E) : a.n4H, B = blockDim.x;
    const float4 *src = DOE ? a.img : a.img + n4E;
    for (int q = threadIdx.x; q < n; q += 2 * B) {
        const float4 v = src[q];
        const bool two = q + B < n;
        float4 w = v;
        if (two) w = src[q + B];
        lds4[q] = v;
        if (two) lds4[q + B] = w;
    }
    const int nm = a.nmat, nRT = ORDER > 0 ? a.nRT : 0, ns = ORDER > 0 ? 6 * (int)(sizeof(RowSlab) / 4) : 0;
    const float *f = reinterpret_cast<float *>(lds4), *h = DOE ? f + 4 * n4E : f;
    const int nh = HU ? 0 : nm;
    S.cE = reinterpret_cast<const float4 *>(f);
    S.RTE = f + 4 * nm;
    S.slE = reinterpret_cast<const RowSlab *>(f + 4 * nm + nRT);
    S.sE = f + 4 * nm + nRT + ns;
    S.disp = S.sE + nm;
    S.cH = reinterpret_cast<const float4 *>(h);
    S.RTH = h + 4 * nh;
    S.slH = reinterpret_cast<const RowSlab *>(h + 4 * nh + nRT);
    S.sH = h + 4 * nh + nRT + ns;
    if (DOE && DOH) {
        S.lx = reinterpret_cast<fN *>(lds4 + n);
        S.lz = S.lx + 2 * B;
        S.ly = reinterpret_cast<float *>(S.lz + 2 * B);
    }
    return S;
}

// H of a lane's cells at plane i: update_magnetic
// (gprMax/fields_updates_ext.pyx:404-412), each H-PML slab in order, magnetic
// dipoles (gprMax/sources.py:202-232).  hx, hy, hz: old in, new out.
template <int FORM, int ORDER, bool HU>
__device__ __forceinline__ void row_h(const RowModel &a, const RowLds &S, uint32_t pf, uint32_t m, RowPhis<ORDER> &ph,
                                      int i, int j, int kl, bool live, int it, fN ex, fN ey,
                                      fN ez, fN ey1, fN ez1, fN exj, fN ezj, fN exk, fN eyk, idN m3, idN m4, idN m5,
                                      fN &hx, fN &hy, fN &hz)
{
    const fN dEz_y = ezj - ez, dEy_z = eyk - ey, dEx_z = exk - ex;
    const fN dEz_x = ez1 - ez, dEy_x = ey1 - ey, dEx_y = exj - ex;
    const int nx = a.nx, ny = a.ny, nz = a.nz;   // read once, and no branches
    const bool bx = (i >= 1) & (j < ny), by = (i < nx) & (j >= 1), bz = (i < nx) & (j < ny);
    float4 ux, uy, uz;
    if (HU) ux = uy = uz = make_float4(a.h[0], a.h[1], a.h[2], a.h[3]);
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int k = kl + u;
        if (!HU) {
            ux = S.cH[id_of(m3, u)];
            uy = S.cH[id_of(m4, u)];
            uz = S.cH[id_of(m5, u)];
        }
        const float nx_ = ux.x * hx[u] - ux.z * dEz_y[u] + ux.w * dEy_z[u];
        const float ny_ = uy.x * hy[u] - uy.w * dEx_z[u] + uy.y * dEz_x[u];
        const float nz_ = uz.x * hz[u] - uz.y * dEy_x[u] + uz.z * dEx_y[u];
        hx[u] = bx & (k < nz) ? nx_ : hx[u];
        hy[u] = by & (k < nz) ? ny_ : hy[u];
        hz[u] = bz & (k >= 1) & (k <= nz) ? nz_ : hz[u];
    }
    auto c3 = [&](int u) { return HU ? a.h[4] : S.sH[id_of(m3, u)]; };
    auto c4 = [&](int u) { return HU ? a.h[4] : S.sH[id_of(m4, u)]; };
    auto c5 = [&](int u) { return HU ? a.h[4] : S.sH[id_of(m5, u)]; };
    if (ORDER > 0) {
        forget(ex);
        forget(ey);
        forget(ez);
        const bool xlo = (pf >> PF_SLAB_H) & 1u;
        if (m) {
            fN xy = -0.f, xz = -0.f, yx = -0.f, yz = -0.f, zx = -0.f, zy = -0.f;
            if (m & ROW_X)
                row_slab<FORM, ORDER, true, false>(S.slH[xlo ? 0 : 3], S.RTH, i, kl, ez1 - ez, ey1 - ey, xy, xz, c4, c5, ph.x);
            if (m & ROW_Y)
                row_slab<FORM, ORDER, false, false>(S.slH[m & 2u ? 1 : 4], S.RTH, j, kl, ezj - ez, exj - ex, yx, yz, c3, c5, ph.y);
            if (m & ROW_Z)
                row_slab<FORM, ORDER, true, true>(S.slH[m & 4u ? 2 : 5], S.RTH, 0, kl, eyk - ey, exk - ex, zx, zy, c3, c4, ph.z);
            row_add(hx, yx, zx, (m & 20u) == 20u);
            row_add(hy, xy, zy, (m & 12u) == 12u);
            row_add(hz, xz, yz, (m & 10u) == 10u);
        }
    }
    if ((pf & PF_SRCH) && live) {
        const SrcArgs &M = a.rare->srcM;
        for (int s = 0; s < M.n; ++s) {
            const int *in = M.info + 6 * s;
            if (in[0] != i || in[1] != j || it < in[4] || it > in[5]) continue;
            const int pol = in[3];
            const float w = M.waves[(size_t)s * a.iterations + it];
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const bool at = in[2] == kl + u;
                const float c = pol == 0 ? c3(u) : (pol == 1 ? c4(u) : c5(u));
                const float v = c * w * M.fac[2 * s];
                hx[u] = at && pol == 0 ? hx[u] - v : hx[u];
                hy[u] = at && pol == 1 ? hy[u] - v : hy[u];
                hz[u] = at && pol == 2 ? hz[u] - v : hz[u];
            }
        }
    }
}

// Receivers on plane i sample the state at the start of the iteration.
__device__ __forceinline__ void row_rx(const RowModel &a, int i, int j, int kl, int it, fN ex, fN ey, fN ez, fN hx, fN hy,
                                       fN hz)
{
    const StepRare &Q = *a.rare;
    for (int r = 0; r < Q.nrx; ++r) {
        if (Q.rxc[3 * r] != i || Q.rxc[3 * r + 1] != j) continue;
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            if (Q.rxc[3 * r + 2] != kl + u) continue;
            float *o = Q.rxbuf + (size_t)it * Q.nrx + r;
            const size_t cs = (size_t)a.iterations * Q.nrx;
            o[0] = ex[u]; o[cs] = ey[u]; o[2 * cs] = ez[u];
            o[3 * cs] = hx[u]; o[4 * cs] = hy[u]; o[5 * cs] = hz[u];
        }
    }
}

// Auxiliary values of a lane's edges of one component.
template <int P, bool CPLX>
struct RowT {
    uN s;                // slots, T_NOSLOT for edges without poles or outside the range
    fN r[P > 0 ? P : 1], i[P > 0 && CPLX ? P : 1];   // of the lane's cells
};

// Calls f for poles (or cells) 0 to P - 1, each a constant (with a loop the values are
// indexed before it is unrolled and end up in scratch memory).
template <int P, class Fn>
__device__ __forceinline__ void row_poles(const Fn &f)
{
    if constexpr (P > 0) {
        row_poles<P - 1>(f);
        f(std::integral_constant<int, P - 1>{});
    }
}

// The values of pole p of component c.  A lane without any loads and stores at
// T_NONE, past the resource's end, where the hardware drops the access: no branch
// splits the plane's loads, which a wait for each component's would follow.
constexpr uint32_t T_NONE = 0xfffffff0u;
template <bool CPLX>
__device__ __forceinline__ rsrc_t row_t_at(const TArgs &T, int c, int p)
{
    return __builtin_amdgcn_make_buffer_rsrc(T.T[c] + (size_t)p * (size_t)T.n[c] * (CPLX ? 2 : 1), 0, 0xffffff00u, 0x00020000);
}

// Neighbouring edges with poles have neighbouring slots, so one load a pole
// brings both cells' values, or a value and what lies after it (after the
// last slot: the array's padding); row_t_settle gives the second cell its own
// where the values are first used.
template <int P, bool CPLX>
__device__ __forceinline__ void row_t_load(const TArgs &T, int c, RowT<P, CPLX> &t)
{
    const uint32_t q0 = t.s[0], q1 = t.s[1], s = q0 != T_NOSLOT ? q0 : q1;
    const uint32_t q = s != T_NOSLOT ? s * (CPLX ? 8u : 4u) : T_NONE;
    row_poles<P>([&](auto pole) {
        constexpr int p = decltype(pole)::value;
        const rsrc_t r = row_t_at<CPLX>(T, c, p);
        if constexpr (CPLX) {
            const float4 v = bits<float4>(__builtin_amdgcn_raw_buffer_load_b128(r, q, 0, 0));
            t.r[p] = (fN){v.x, v.z};
            t.i[p] = (fN){v.y, v.w};
        } else {
            t.r[p] = bldN(r, q, 0);
        }
    });
}
template <int P, bool CPLX>
__device__ __forceinline__ void row_t_settle(RowT<P, CPLX> &t)
{
    const bool both = t.s[0] != T_NOSLOT;
    row_poles<P>([&](auto pole) {
        constexpr int p = decltype(pole)::value;
        const float x = t.r[p][0], y = t.r[p][1];
        t.r[p][1] = both ? y : x;
        if constexpr (CPLX) {
            const float v = t.i[p][0], w = t.i[p][1];
            t.i[p][1] = both ? w : v;
        }
    });
}
template <int P, bool CPLX>
__device__ __forceinline__ void row_t_store(const TArgs &T, int c, const RowT<P, CPLX> &t)
{
    const uint32_t q0 = t.s[0], q1 = t.s[1], w = CPLX ? 8u : 4u;
    const bool in0 = q0 != T_NOSLOT, in1 = q1 != T_NOSLOT;
    const uint32_t two = in0 & in1 ? q0 * w : T_NONE, one = in0 != in1 ? (in0 ? q0 : q1) * w : T_NONE;
    if (__any(in0 & in1)) row_poles<P>([&](auto pole) {
        constexpr int p = decltype(pole)::value;
        const rsrc_t r = row_t_at<CPLX>(T, c, p);
        if constexpr (CPLX)
            __builtin_amdgcn_raw_buffer_store_b128(bits<u32x4>(make_float4(t.r[p][0], t.i[p][0], t.r[p][1], t.i[p][1])), r, two, 0, 0);
        else
            bstN(r, two, 0, t.r[p]);
    });
    if (!__any(in0 != in1)) return;
    row_poles<P>([&](auto pole) {
        constexpr int p = decltype(pole)::value;
        const rsrc_t r = row_t_at<CPLX>(T, c, p);
        const float r0 = t.r[p][0], r1 = t.r[p][1];
        if constexpr (CPLX) {
            const float i0 = t.i[p][0], i1 = t.i[p][1];
            __builtin_amdgcn_raw_buffer_store_b64(bits<u32x2>(make_float2(in0 ? r0 : r1, in0 ? i0 : i1)), r, one, 0, 0);
        } else {
            bst(r, one, 0, in0 ? r0 : r1);
        }
    });
}

// disp_a and disp_b for cell U of a lane.
template <int U, int P, bool CPLX>
__device__ __forceinline__ float row_disp_a(const float *D, uint32_t m, RowT<P, CPLX> &t, float e)
{
    float phi = 0.f;
    const float *c = D + (size_t)m * 3 * P * (CPLX ? 2 : 1);
    row_poles<P>([&](auto pole) {
        constexpr int p = decltype(pole)::value;
        const float r = t.r[p][U];
        if constexpr (CPLX) {
            const float *k = c + 6 * p;
            const float i = t.i[p][U];
            if constexpr (P == 1) phi = k[0] * r;
            else phi = phi + k[0] * r;
            t.r[p][U] = (k[2] * r - k[3] * i) + k[4] * e;
            t.i[p][U] = (k[2] * i + k[3] * r) + k[5] * e;
        } else {
            const float *k = c + 3 * p;
            if constexpr (P == 1) phi = k[0] * r;
            else phi = phi + k[0] * r;
            t.r[p][U] = k[1] * r + k[2] * e;
        }
    });
    return phi;
}
template <int U, int P, bool CPLX>
__device__ __forceinline__ void row_disp_b(const float *D, uint32_t m, RowT<P, CPLX> &t, float e)
{
    const float *c = D + (size_t)m * 3 * P * (CPLX ? 2 : 1);
    row_poles<P>([&](auto pole) {
        constexpr int p = decltype(pole)::value;
        if constexpr (CPLX) {
            t.r[p][U] = t.r[p][U] - c[6 * p + 4] * e;
            t.i[p][U] = t.i[p][U] - c[6 * p + 5] * e;
        } else {
            t.r[p][U] = t.r[p][U] - c[3 * p + 2] * e;
        }
    });
}

// E of a lane's cells at plane i: update_electric or dispersive part A
// (gprMax/fields_updates_ext.pyx:81-107, 146-179), each E-PML slab in order,
// voltage sources then Hertzian dipoles (gprMax/model_build_run.py:458-461),
// dispersive part B.  ex, ey, ez: old in, new out; H at the cell, at i-1 (hym,
// hzm), j-1 (hxj, hzj) and k-1 (hxk, hyk).
template <int P, bool CPLX, int FORM, int ORDER>
__device__ __forceinline__ void row_e(const RowModel &a, const RowLds &S, uint32_t pf, uint32_t m, RowPhis<ORDER> &ph,
                                      int i, int j, int kl, int it, fN hx, fN hy, fN hz, fN hym, fN hzm, fN hxj,
                                      fN hzj, fN hxk, fN hyk, idN m0, idN m1, idN m2, RowT<P, CPLX> &tx,
                                      RowT<P, CPLX> &ty, RowT<P, CPLX> &tz, fN &ex, fN &ey, fN &ez)
{
    const fN dHz_y = hz - hzj, dHy_z = hy - hyk, dHx_z = hx - hxk;
    const fN dHz_x = hz - hzm, dHy_x = hy - hym, dHx_y = hx - hxj;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const bool ji = (j >= 1) & (j < ny), ii = (i >= 1) & (i < nx);
    const bool bx = (i < nx) & ji, by = ii & (j < ny), bz = ii & ji;
    if constexpr (P > 0) {
        row_t_settle(tx);
        row_t_settle(ty);
        row_t_settle(tz);
    }
    row_poles<NC>([&](auto cell) {
        constexpr int u = decltype(cell)::value;
        const int k = kl + u;
        const uint32_t i0 = id_of(m0, u), i1 = id_of(m1, u), i2 = id_of(m2, u);
        const float4 q0 = S.cE[i0], q1 = S.cE[i1], q2 = S.cE[i2];
        const bool ki = (k >= 1) & (k < nz), rx_ = bx & ki, ry_ = by & ki, rz_ = bz & (k < nz);
        float vx = q0.x * ex[u] + q0.z * dHz_y[u] - q0.w * dHy_z[u];
        float vy = q1.x * ey[u] + q1.w * dHx_z[u] - q1.y * dHz_x[u];
        float vz = q2.x * ez[u] + q2.y * dHy_x[u] - q2.z * dHx_y[u];
        if (P > 0) {
            auto part_a = [&](RowT<P, CPLX> &t, uint32_t m, float e, float v) {
                const float phi = t.s[u] != T_NOSLOT ? row_disp_a<u, P, CPLX>(S.disp, m, t, e) : 0.f;
                return v - S.sE[m] * phi;
            };
            vx = part_a(tx, i0, ex[u], vx);
            vy = part_a(ty, i1, ey[u], vy);
            vz = part_a(tz, i2, ez[u], vz);
        }
        ex[u] = rx_ ? vx : ex[u];
        ey[u] = ry_ ? vy : ey[u];
        ez[u] = rz_ ? vz : ez[u];
    });
    auto c0 = [&](int u) { return S.sE[id_of(m0, u)]; };
    auto c1 = [&](int u) { return S.sE[id_of(m1, u)]; };
    auto c2 = [&](int u) { return S.sE[id_of(m2, u)]; };
    if (ORDER > 0) {
        forget(hx);
        forget(hy);
        forget(hz);
        const bool xlo = (pf >> PF_SLAB_E) & 1u;
        if (m) {
            fN xy = -0.f, xz = -0.f, yx = -0.f, yz = -0.f, zx = -0.f, zy = -0.f;
            if (m & ROW_X)
                row_slab<FORM, ORDER, false, false>(S.slE[xlo ? 0 : 3], S.RTE, i, kl, hz - hzm, hy - hym, xy, xz, c1, c2, ph.x);
            if (m & ROW_Y)
                row_slab<FORM, ORDER, true, false>(S.slE[m & 2u ? 1 : 4], S.RTE, j, kl, hz - hzj, hx - hxj, yx, yz, c0, c2, ph.y);
            if (m & ROW_Z)
                row_slab<FORM, ORDER, false, true>(S.slE[m & 4u ? 2 : 5], S.RTE, 0, kl, hy - hyk, hx - hxk, zx, zy, c0, c1, ph.z);
            row_add(ex, yx, zx, (m & 20u) == 20u);
            row_add(ey, xy, zy, (m & 12u) == 12u);
            row_add(ez, xz, yz, (m & 10u) == 10u);
        }
    }
    if (pf & PF_SRCE) {
        const SrcArgs &V = a.rare->srcV, &D = a.rare->srcD;
        for (int s = 0; s < V.n; ++s) {  // gprMax/sources.py:81-120
            const int *in = V.info + 6 * s;
            if (in[0] != i || in[1] != j || it < in[4] || it > in[5]) continue;
            const int pol = in[3] & 3;
            const bool hard = in[3] >= 4;
            const float w = V.waves[(size_t)s * a.iterations + it];
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const bool at = in[2] == kl + u;
                const float c = pol == 0 ? c0(u) : (pol == 1 ? c1(u) : c2(u));
                const float v = c * w * V.fac[2 * s], e = -w / V.fac[2 * s];
                ex[u] = at && pol == 0 ? (hard ? e : ex[u] - v) : ex[u];
                ey[u] = at && pol == 1 ? (hard ? e : ey[u] - v) : ey[u];
                ez[u] = at && pol == 2 ? (hard ? e : ez[u] - v) : ez[u];
            }
        }
        for (int s = 0; s < D.n; ++s) {  // gprMax/sources.py:163-193
            const int *in = D.info + 6 * s;
            if (in[0] != i || in[1] != j || it < in[4] || it > in[5]) continue;
            const int pol = in[3];
            const float w = D.waves[(size_t)s * a.iterations + it];
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const bool at = in[2] == kl + u;
                const float c = pol == 0 ? c0(u) : (pol == 1 ? c1(u) : c2(u));
                const float v = c * w * D.fac[2 * s] * D.fac[2 * s + 1];
                ex[u] = at && pol == 0 ? ex[u] - v : ex[u];
                ey[u] = at && pol == 1 ? ey[u] - v : ey[u];
                ez[u] = at && pol == 2 ? ez[u] - v : ez[u];
            }
        }
    }
    if constexpr (P > 0) {
        row_poles<NC>([&](auto cell) {
            constexpr int u = decltype(cell)::value;
            auto part_b = [&](RowT<P, CPLX> &t, uint32_t m, float e) {
                if (t.s[u] != T_NOSLOT) row_disp_b<u, P, CPLX>(S.disp, m, t, e);
            };
            part_b(tx, id_of(m0, u), ex[u]);
            part_b(ty, id_of(m1, u), ey[u]);
            part_b(tz, id_of(m2, u), ez[u]);
        });
        row_t_store(a.T, 0, tx);
        row_t_store(a.T, 1, ty);
        row_t_store(a.T, 2, tz);
    }
}

// Edges outside the update ranges (which hold no auxiliary values in use)
// count as without.
template <int P, bool CPLX>
__device__ __forceinline__ void row_slots_in(const RowModel &a, int i, int j, int kl, RowT<P, CPLX> &tx, RowT<P, CPLX> &ty,
                                             RowT<P, CPLX> &tz)
{
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const bool ji = (j >= 1) & (j < ny), ii = (i >= 1) & (i < nx);
    const bool bx = (i < nx) & ji, by = ii & (j < ny), bz = ii & ji;
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int k = kl + u;
        const bool ki = (k >= 1) & (k < nz);
        tx.s[u] = bx & ki ? tx.s[u] : T_NOSLOT;
        ty.s[u] = by & ki ? ty.s[u] : T_NOSLOT;
        tz.s[u] = bz & (k < nz) ? tz.s[u] : T_NOSLOT;
    }
}

// Slots of a lane's edges at plane i, from the arrays of every edge's slot.
template <int P, bool CPLX>
__device__ __forceinline__ void row_slots(const RowModel &a, int i, int j, int kl, uint32_t off, RowT<P, CPLX> &tx,
                                          RowT<P, CPLX> &ty, RowT<P, CPLX> &tz)
{
    if (P == 0) return;
    const size_t po = (size_t)i * a.plane * 4 + off;
    auto get = [&](int c) {
        typedef __attribute__((address_space(1))) const uN gu4;
        return *(gu4 *)(reinterpret_cast<const char *>(a.T.slot[c]) + po);
    };
    tx.s = get(0);
    ty.s = get(1);
    tz.s = get(2);
    row_slots_in(a, i, j, kl, tx, ty, tz);
}

// The same for a wave of a pass, whose lanes hold 128 edges one after the other
// (group `grp` of the plane): of each component the first slot among them and
// two masks of the edges with poles, one for each cell of a lane, 64 bytes in
// all through the scalar cache.  Slots read edge by edge are 12 bytes a cell more to
// fetch (the E pass of 240x240x180, 30 % of the cells with 3 poles, moves about
// 85); with a load for each value instead of each pair besides, us per iteration:
// that grid 296, now 269; 200x150x130 Drude 96, 76; 121x104x90 with two complex poles
// 44.9, 43.1; 150x140x100, 2 poles in 10 % of the cells, 55.1, 54.7.
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ u32x16 row_masks(const TArgs &T, int i, int grp)
{
    typedef __attribute__((address_space(4))) const u32x16 cu32x16;
    return ((cu32x16 *)T.masks)[(size_t)i * T.groups + grp];
}
template <int P, bool CPLX>
__device__ __forceinline__ void row_slots_of(const RowModel &a, int i, int j, int kl, u32x16 w, bool live, RowT<P, CPLX> &tx,
                                             RowT<P, CPLX> &ty, RowT<P, CPLX> &tz)
{
    const int lane = threadIdx.x & 63;
    auto get = [&](int c, RowT<P, CPLX> &t) {
        const uint32_t e0 = w[4 * c], e1 = w[4 * c + 1], o0 = w[4 * c + 2], o1 = w[4 * c + 3];
        uint32_t n = __builtin_amdgcn_mbcnt_hi(e1, __builtin_amdgcn_mbcnt_lo(e0, w[12 + c]));
        n = __builtin_amdgcn_mbcnt_hi(o1, __builtin_amdgcn_mbcnt_lo(o0, n));
        const uint32_t even = ((lane < 32 ? e0 : e1) >> (lane & 31)) & 1u, odd = ((lane < 32 ? o0 : o1) >> (lane & 31)) & 1u;
        t.s[0] = live && even ? n : T_NOSLOT;
        t.s[1] = live && odd ? n + even : T_NOSLOT;
    };
    get(0, tx);
    get(1, ty);
    get(2, tz);
    row_slots_in(a, i, j, kl, tx, ty, tz);
}

// ---------------------------------------------------------------- whole step
// Place of thread t in tile column tk: row r, lane c of the row.  The lanes
// with cells in a z slab (a at the start of a row, b at its end) come after
// all the others, from a whole wave on: along a row they are few (6 of 51 lanes
// of the 300x300x200 grid), and dealt with the row every wave would run the
// slab code for a tenth of its lanes.
struct RowPlace {
    int r, c;
    int row;    // threads between rows
    int prev;   // thread of the lane before
    bool end;   // the next thread is not the next lane of the row
};
__device__ __forceinline__ RowPlace row_place(const RowModel &a, int tk, int t)
{
    RowPlace q;
    const int za = tk == 0 ? a.za : 0, zb = tk == a.ntk - 1 ? a.zb : 0, z = za + zb, n = a.LT - z;
    const int z0 = (a.R * n + 63) & ~63;
    if (t < z0) {
        q.r = n > 0 ? t / n : a.R;
        const int x = t - q.r * n;
        q.c = za + x;
        q.row = n;
        q.end = x == n - 1;
        q.prev = x > 0 ? t - 1 : (za > 0 ? z0 + q.r * z + za - 1 : t);
    } else {
        const int y = t - z0;
        q.r = z > 0 ? y / z : a.R;
        const int x = y - q.r * z;
        q.c = x < za ? x : n + x;
        q.row = z;
        q.end = x == z - 1 || (x == za - 1 && n > 0);
        q.prev = x == za && n > 0 ? q.r * n + n - 1 : (x > 0 ? t - 1 : t);
    }
    if (q.r >= a.R) {  // a thread without a lane
        q.prev = t;
        q.row = 0;
    }
    return q;
}

template <int P, bool CPLX, int FORM, int ORDER, bool HU>
__device__ __forceinline__ void row_step_item(const RowModel &a, const RowLds &S, int item, int flip, int flipE, int it)
{
    const int tk = item % a.ntk, r1 = item / a.ntk;
    const int tj = r1 % a.ntj, ch = r1 / a.ntj;
    const int t = threadIdx.x, B = blockDim.x;
    const RowPlace q = row_place(a, tk, t);
    const int r = q.r, c = q.c;
    const int j_ = tj * a.Ro - a.hj + r, kl_ = NC * (tk * a.LTo - a.hk + c);
    const bool live = r < a.R && j_ >= 0 && j_ <= a.ny && kl_ >= 0 && kl_ < a.kp;
    const bool owner = live && r >= a.hj && c >= a.hk;
    const int j = live ? j_ : 0, kl = live ? kl_ : 0;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t toj = j < a.ny ? to + 4u * (uint32_t)a.kp : to;
    const uint32_t ti = to >> 1;
    const int xa = ch * a.xc, xb = min(xa + a.xc, a.nx + 1), xs = xa > 0 ? xa - 1 : 0;
    const rsrc_t rF = rsrc(a.F[flip]), wF = rsrc(a.F[flip ^ 1]), rI = rsrc(a.ID);
    const rsrc_t rP = rsrc(a.phiH[flip]), wP = rsrc(a.phiH[flip ^ 1]), rPE = rsrc(a.phiE[flipE]);
    const uint32_t P4 = (uint32_t)a.plane * 4u, Pi = (uint32_t)a.plane * 2u, cs = a.cs, ci = a.ci;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    // the next lane of the wave holds E at k+1, except where the row goes on
    // in another wave or group
    const bool end = q.end || (t & 63) == 63;
    const bool patch = live && end && kl + NC <= a.nz;
    RowSlabs LE, LH;
    if (ORDER > 0) {
        LE = row_slabs(a.atE, j, kl, live);
        LH = row_slabs(a.atH, j, kl, live);
    }
    fN ex, ey, ez, hym = 0.f, hzm = 0.f;
    {
        const uint32_t so = (uint32_t)xs * P4;
        ex = bldN(rF, to, so);
        ey = bldN(rF, to, so + cs);
        ez = bldN(rF, to, so + 2 * cs);
    }
    uint32_t pfn = plane_flags(a, xs);
    for (int i = xs; i < xb; ++i) {
        const bool own = owner && i >= xa;
        const uint32_t pf = pfn;
        pfn = plane_flags(a, i + 1 < xb ? i + 1 : i);
        const uint32_t so = (uint32_t)i * P4, sn = i < a.nx ? so + P4 : so, si = (uint32_t)i * Pi;
        fN hx = bldN(rF, to, so + 3 * cs), hy = bldN(rF, to, so + 4 * cs), hz = bldN(rF, to, so + 5 * cs);
        const fN ezj = bldN(rF, toj, so + 2 * cs), exj = bldN(rF, toj, so);
        const fN ex1 = bldN(rF, to, sn), ey1 = bldN(rF, to, sn + cs), ez1 = bldN(rF, to, sn + 2 * cs);
        float ykn = 0.f, xkn = 0.f;
        if (patch) {
            ykn = bld(rF, to + 4u * NC, so + cs);
            xkn = bld(rF, to + 4u * NC, so);
        }
        idN m3 = 0u, m4 = 0u, m5 = 0u;
        if (!HU) {
            m3 = bld_ids(rI, ti, si + 3 * ci);
            m4 = bld_ids(rI, ti, si + 4 * ci);
            m5 = bld_ids(rI, ti, si + 5 * ci);
        }
        const idN m0 = bld_ids(rI, ti, si), m1 = bld_ids(rI, ti, si + ci), m2 = bld_ids(rI, ti, si + 2 * ci);
        RowT<P, CPLX> tx, ty, tz;
        if (P > 0 && own) row_slots(a, i, j, kl, to, tx, ty, tz);
        RowPhis<ORDER> ph, pe;
        uint32_t mH = 0, mE = 0;
        if (ORDER > 0) {
            mH = LH.m & (pf >> PF_SLAB_H);
            mE = own ? LE.m & (pf >> PF_SLAB_E) : 0u;
            row_phis(ph, LH, mH, (pf >> PF_SLAB_H) & 1u, rP, np4, i, j, kl);
            row_phis(pe, LE, mE, (pf >> PF_SLAB_E) & 1u, rPE, np4, i, j, kl);
        }
        arrived(hx, hy, hz, ezj, exj, ex1, ey1, ez1, m0[0], m1[0], m2[0]);
        const float yn = from_next(ykn, ey.x), xn = from_next(xkn, ex.x);
        const fN eyk = shift_up(ey, end ? ykn : yn), exk = shift_up(ex, end ? xkn : xn);
        if (own && (pf & PF_RX)) row_rx(a, i, j, kl, it, ex, ey, ez, hx, hy, hz);
        row_h<FORM, ORDER, HU>(a, S, pf, mH, ph, i, j, kl, live, it, ex, ey, ez, ey1, ez1, exj, ezj, exk, eyk, m3, m4, m5, hx, hy,
                               hz);
        if (own) {
            if (ORDER > 0) row_phis_store(ph, mH, wP, np4);
            bstN(wF, to, so + 3 * cs, hx);
            bstN(wF, to, so + 4 * cs, hy);
            bstN(wF, to, so + 5 * cs, hz);
        }
        const int pb = (i & 1) * B;
        S.lx[pb + t] = hx;
        S.lz[pb + t] = hz;
        S.ly[pb + t] = hy[NC - 1];
        if (P > 0 && own) {
            row_t_load(a.T, 0, tx);
            row_t_load(a.T, 1, ty);
            row_t_load(a.T, 2, tz);
        }
        __syncthreads();
        if (own) {
            const int tb = pb + (j > 0 ? t - q.row : t);   // Hx, Hz at j-1 (unused at j = 0)
            const fN hxj = S.lx[tb], hzj = S.lz[tb];
            const fN hxk = shift_down(hx, S.lx[pb + q.prev][NC - 1]), hyk = shift_down(hy, S.ly[pb + q.prev]);
            row_e<P, CPLX, FORM, ORDER>(a, S, pf, mE, pe, i, j, kl, it, hx, hy, hz, hym, hzm, hxj, hzj, hxk, hyk, m0, m1, m2, tx,
                                        ty, tz, ex, ey, ez);
            if (ORDER > 0) row_phis_store(pe, mE, rPE, np4);
            bstN(wF, to, so, ex);
            bstN(wF, to, so + cs, ey);
            bstN(wF, to, so + 2 * cs, ez);
        }
        hym = hy;
        hzm = hz;
        ex = ex1;
        ey = ey1;
        ez = ez1;
    }
}

// The model of item g and its first item.
__device__ __forceinline__ int row_model_of(const RowArgs &b, int g, int &first)
{
    if (b.ntr == 1) {
        first = 0;
        return 0;
    }
    int lo = 0, hi = b.ntr - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (b.item0[mid] <= g) lo = mid;
        else hi = mid - 1;
    }
    first = b.item0[lo];
    return lo;
}

// One block per work item (tile, x chunk) of one or of several models.
template <int P, bool CPLX, int FORM, int ORDER, bool HU>
__global__ void __launch_bounds__(ROW_BLOCK_MAX) __attribute__((amdgpu_waves_per_eu(P > 0 ? 2 : (ORDER == 0 ? 5 : 4)))) k_row_step(const RowModel *__restrict__ models, RowArgs b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    int first;
    const RowModel &a = models[row_model_of(b, g, first)];
    const RowLds S = row_stage<ORDER, HU, true, true>(lds4, a);
    __syncthreads();
    row_step_item<P, CPLX, FORM, ORDER, HU>(a, S, g - first, b.flip, b.flipE, b.it);
}

// ---------------------------------------------------------------- passes
// The lane of pass item `item`: segment of the plane's lanes, x chunk of the
// launch's planes.
struct RowLane {
    int seg, j, kl, xa, xb;
    bool live;
};
__device__ __forceinline__ RowLane row_lane(const RowModel &a, int item, int p0, int p1)
{
    RowLane q;
    const int seg = q.seg = item % a.pseg, ch = item / a.pseg, lpr = a.kp / NC;
    const int t = seg * (int)blockDim.x + (int)threadIdx.x;
    q.live = t < (a.ny + 1) * lpr;
    q.j = q.live ? t / lpr : 0;
    q.kl = q.live ? NC * (t - q.j * lpr) : 0;
    q.xa = p0 + ch * a.pxc;
    q.xb = min(min(q.xa + a.pxc, p1), a.nx + 1);
    return q;
}

// H pass, in place: every lane reads E and its own H and writes its own H.
// The first plane's loads go out before the tables are staged, and the Phi
// loads with them: on small grids a pass is little more than its chain of
// dependent memory accesses.
template <int FORM, int ORDER, bool HU, bool BIG = false>
__global__ void __launch_bounds__(ROW_PASS_MAX) ROW_PASS_WAVES(0, ORDER) k_row_h(const RowModel *__restrict__ models, RowArgs b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    int first;
    const RowModel &a = models[row_model_of(b, g, first)];
    const RowLane q = row_lane(a, g - first, b.p0, b.p1);
    const int j = q.j, kl = q.kl, it = b.it, lane = threadIdx.x & 63;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t toj = j < a.ny ? to + 4u * (uint32_t)a.kp : to;
    const uint32_t ti = to >> 1;
    const RowComps<BIG> F(a.F[b.flip], a.cs, a.csl), I(a.ID, a.ci, a.cil);
    const rsrc_t rP = rsrc(a.phiH[b.flip]);
    const uint32_t P4 = (uint32_t)a.plane * 4u, Pi = (uint32_t)a.plane * 2u;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const bool patch = q.live && lane == 63 && kl + NC <= a.nz;
    RowSlabs L;
    if (ORDER > 0) L = row_slabs(a.atH, j, kl, q.live);
    fN ey = bldN(F.at(1), to, F.off(1, (uint32_t)q.xa * P4)), ez = bldN(F.at(2), to, F.off(2, (uint32_t)q.xa * P4));
    fN ex, hx, hy, hz, ezj, exj, ey1, ez1;
    float ykn = 0.f, xkn = 0.f;
    idN m3 = 0u, m4 = 0u, m5 = 0u;
    RowPhis<ORDER> ph;
    uint32_t pf = 0, m = 0;
    auto load = [&](int i) {
        pf = plane_flags(a, i);
        const uint32_t so = (uint32_t)i * P4, sn = i < a.nx ? so + P4 : so, si = (uint32_t)i * Pi;
        ex = bldN(F.at(0), to, F.off(0, so));
        hx = bldN(F.at(3), to, F.off(3, so));
        hy = bldN(F.at(4), to, F.off(4, so));
        hz = bldN(F.at(5), to, F.off(5, so));
        ezj = bldN(F.at(2), toj, F.off(2, so));
        exj = bldN(F.at(0), toj, F.off(0, so));
        ey1 = bldN(F.at(1), to, F.off(1, sn));
        ez1 = bldN(F.at(2), to, F.off(2, sn));
        if (patch) {
            ykn = bld(F.at(1), to + 4u * NC, F.off(1, so));
            xkn = bld(F.at(0), to + 4u * NC, F.off(0, so));
        }
        if (!HU) {
            m3 = bld_ids(I.at(3), ti, I.off(3, si));
            m4 = bld_ids(I.at(4), ti, I.off(4, si));
            m5 = bld_ids(I.at(5), ti, I.off(5, si));
        }
        if (ORDER > 0) {
            m = L.m & (pf >> PF_SLAB_H);
            row_phis(ph, L, m, (pf >> PF_SLAB_H) & 1u, rP, np4, i, j, kl);
        }
    };
    load(q.xa);
    const RowLds S = row_stage<ORDER, HU, false, true>(lds4, a);
    __syncthreads();
    for (int i = q.xa;;) {
        const uint32_t so = (uint32_t)i * P4;
        const fN eyk = shift_up(ey, from_next(ykn, ey.x)), exk = shift_up(ex, from_next(xkn, ex.x));
        if (q.live && (pf & PF_RX)) row_rx(a, i, j, kl, it, ex, ey, ez, hx, hy, hz);
        row_h<FORM, ORDER, HU>(a, S, pf, m, ph, i, j, kl, q.live, it, ex, ey, ez, ey1, ez1, exj, ezj, exk, eyk, m3, m4, m5, hx, hy,
                               hz);
        if (ORDER > 0) row_phis_store(ph, m, rP, np4);
        if (q.live) {
            bstN(F.at(3), to, F.off(3, so), hx);
            bstN(F.at(4), to, F.off(4, so), hy);
            bstN(F.at(5), to, F.off(5, so), hz);
        }
        if (++i == q.xb) break;
        ey = ey1;
        ez = ez1;
        load(i);
    }
}

// E pass, in place: every lane reads H and its own E and writes its own E.
template <int P, bool CPLX, int FORM, int ORDER, bool BIG = false>
__global__ void __launch_bounds__(ROW_PASS_MAX) ROW_PASS_WAVES(CPLX ? 2 : P, ORDER)
k_row_e(const RowModel *__restrict__ models, RowArgs b)
{
    extern __shared__ float4 lds4[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    int first;
    const RowModel &a = models[row_model_of(b, g, first)];
    const RowLane q = row_lane(a, g - first, b.p0, b.p1);
    const int j = q.j, kl = q.kl, it = b.it, lane = threadIdx.x & 63;
    const uint32_t to = (uint32_t)(j * a.kp + kl) * 4u;
    const uint32_t tob = j > 0 ? to - 4u * (uint32_t)a.kp : to;
    const uint32_t ti = to >> 1;
    const RowComps<BIG> F(a.F[b.flip], a.cs, a.csl), I(a.ID, a.ci, a.cil);
    const rsrc_t rP = rsrc(a.phiE[b.flipE]);
    const uint32_t P4 = (uint32_t)a.plane * 4u, Pi = (uint32_t)a.plane * 2u;
    const uint32_t np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const bool patch = q.live && lane == 0 && kl > 0;
    int grp = 0;    // the wave's place in the plane, in groups of 64 lanes; past the plane's end any
    if (P > 0) {
        grp = __builtin_amdgcn_readfirstlane(((g - first) % a.pseg * (int)blockDim.x + (int)threadIdx.x) >> 6);
        grp = min(grp, a.T.groups - 1);
    }
    RowSlabs L;
    if (ORDER > 0) L = row_slabs(a.atE, j, kl, q.live);
    const uint32_t sm = (uint32_t)(q.xa > 0 ? q.xa - 1 : 0) * P4;
    fN hym = bldN(F.at(4), to, F.off(4, sm)), hzm = bldN(F.at(5), to, F.off(5, sm));
    fN ex, ey, ez, hx, hy, hz, hxj, hzj;
    float hxl = 0.f, hyl = 0.f;
    idN m0, m1, m2;
    RowPhis<ORDER> ph;
    RowT<P, CPLX> tx, ty, tz;
    uint32_t pf = 0, m = 0;
    auto load = [&](int i) {
        pf = plane_flags(a, i);
        const uint32_t so = (uint32_t)i * P4, si = (uint32_t)i * Pi;
        u32x16 masks = 0u;
        if (P > 0) masks = row_masks(a.T, i, grp);
        hx = bldN(F.at(3), to, F.off(3, so));
        hy = bldN(F.at(4), to, F.off(4, so));
        hz = bldN(F.at(5), to, F.off(5, so));
        ex = bldN(F.at(0), to, F.off(0, so));
        ey = bldN(F.at(1), to, F.off(1, so));
        ez = bldN(F.at(2), to, F.off(2, so));
        hxj = bldN(F.at(3), tob, F.off(3, so));
        hzj = bldN(F.at(5), tob, F.off(5, so));
        if (patch) {
            hxl = bld(F.at(3), to - 4u, F.off(3, so));
            hyl = bld(F.at(4), to - 4u, F.off(4, so));
        }
        m0 = bld_ids(I.at(0), ti, I.off(0, si));
        m1 = bld_ids(I.at(1), ti, I.off(1, si));
        m2 = bld_ids(I.at(2), ti, I.off(2, si));
        if (ORDER > 0) {
            m = L.m & (pf >> PF_SLAB_E);
            row_phis(ph, L, m, (pf >> PF_SLAB_E) & 1u, rP, np4, i, j, kl);
        }
        if (P > 0) {
            row_slots_of(a, i, j, kl, masks, q.live, tx, ty, tz);
            row_t_load(a.T, 0, tx);
            row_t_load(a.T, 1, ty);
            row_t_load(a.T, 2, tz);
        }
    };
    load(q.xa);
    const RowLds S = row_stage<ORDER, true, true, false>(lds4, a);
    __syncthreads();
    for (int i = q.xa;;) {
        const uint32_t so = (uint32_t)i * P4;
        const fN hxk = shift_down(hx, from_prev(hxl, hx[NC - 1])), hyk = shift_down(hy, from_prev(hyl, hy[NC - 1]));
        if (q.live) {
            row_e<P, CPLX, FORM, ORDER>(a, S, pf, m, ph, i, j, kl, it, hx, hy, hz, hym, hzm, hxj, hzj, hxk, hyk, m0, m1, m2, tx,
                                        ty, tz, ex, ey, ez);
            if (ORDER > 0) row_phis_store(ph, m, rP, np4);
            bstN(F.at(0), to, F.off(0, so), ex);
            bstN(F.at(1), to, F.off(1, so), ey);
            bstN(F.at(2), to, F.off(2, so), ez);
        }
        if (++i == q.xb) break;
        hym = hy;
        hzm = hz;
        load(i);
    }
}

}  // namespace gpx

#include "gpx_plane.h"

namespace gpx {

typedef void (*row_kernel)(const RowModel *, RowArgs);
typedef void (*plane_kernel)(const RowModel *, PlaneArgs);

// The kernels of one model: the whole step, the H pass, the E pass, several
// iterations of a 2-D model (without poles).  big: a state of 4 GiB and more,
// which has the passes only, and those without poles.
struct RowKernels {
    row_kernel step, h, e;
    plane_kernel plane;
};

template <int FORM, int ORDER>
RowKernels row_kernel_table(int P, bool C, bool hu, bool big)
{
#define GPX_RK(PP, CC)                                                                                       \
    RowKernels{hu ? k_row_step<PP, CC, FORM, ORDER, true> : k_row_step<PP, CC, FORM, ORDER, false>,          \
               hu ? k_row_h<FORM, ORDER, true> : k_row_h<FORM, ORDER, false>, k_row_e<PP, CC, FORM, ORDER>, \
               PP == 0 ? k_plane<FORM, ORDER> : nullptr}
    if (big)
        return RowKernels{nullptr, hu ? k_row_h<FORM, ORDER, true, true> : k_row_h<FORM, ORDER, false, true>,
                          k_row_e<0, false, FORM, ORDER, true>, nullptr};
    switch (P) {
    case 0: return GPX_RK(0, false);
    case 1: return C ? GPX_RK(1, true) : GPX_RK(1, false);
    case 2: return C ? GPX_RK(2, true) : GPX_RK(2, false);
    case 3: return C ? GPX_RK(3, true) : GPX_RK(3, false);
    default: return C ? GPX_RK(4, true) : GPX_RK(4, false);
    }
#undef GPX_RK
}

}  // namespace gpx

#endif  // GPX_ROWS_H
