// Several iterations of a 2-D model in one launch (k_plane): one cell along
// axis w, u and v the next two axes in the order x, y, z, x.  Without poles, E
// along w and H along u and v on the plane's cells are all that ever differs
// from zero (plane_shape in gpx.hip sees to that), so a column is three values
// and the four Phi that go with them.
//
// What bounds it.  A plane has few cells: its two passes an iteration are two
// launches (2.4 us each) with a chain of dependent accesses apiece, and little
// else.  Here a block holds a tile of columns, one a lane, with their
// coefficients, profile entries and Phi in registers, `halo` columns more on
// every side, and takes it through up to `halo` iterations; neighbours' values
// go through LDS, E before the H half and H before the E half.  New H needs E at
// the next column and new E needs H at the one before, so with every iteration
// one column more at each edge of the tile is no longer the model's; after
// `halo` of them the columns inside the halo still are, and only those are
// written.  Halo columns are computed as their owners compute them, sources
// among them.  What is left is a launch's fixed time, 5.5 us with the chain model,
// indices, coefficients and Phi, and 0.5 us an iteration for two barriers and
// the chain between them (plane_shape in gpx.hip).  120x105 with HORIPML takes 1.75 us
// an iteration, 8.6 as passes; with all six components of a column in a lane it took 2.9,
// and with flat loads, the slabs' and receivers' descriptions read one after the other
// by every lane, 2.3.
//
// The next state (fields and both Phi) is another copy than the current one, as
// blocks read what others own.  Every lane reaches every barrier: the loop's
// bounds are the launch's.
#ifndef GPX_PLANE_H
#define GPX_PLANE_H

namespace gpx {

constexpr int PLANE_BLOCK_MAX = 1024;

struct PlaneArgs {
    int flip, flipE;        // current copies
    int it, n;              // first iteration, iterations (at most halo)
    int w;                  // the axis of one cell
    int tp, tq, halo;       // columns of a tile along p and q, halo included; q (lanes next to each other) is v, for w = y it is u
    int ntq, nitems, per_xcd;
    int hu;
};

// What many lanes read at one address goes through the scalar cache (no kernel
// writes these tables, which the compiler cannot see behind the model's pointer).
template <class V>
__device__ __forceinline__ V plane_uniform(const V *p, int n)
{
    typedef __attribute__((address_space(4))) const V cV;
    return ((cV *)p)[n];
}
__device__ __forceinline__ RowSlab plane_slab_at(const RowSlab *sl, int n)
{
    typedef int words __attribute__((ext_vector_type(16), aligned(4)));
    static_assert(sizeof(RowSlab) == sizeof(words), "a slab is read in one load");
    typedef __attribute__((address_space(4))) const words cwords;
    return bits<RowSlab>(((cwords *)sl)[n]);
}

// One slab's part in one component of a lane.
template <int FORM, int ORDER>
struct PlaneSlab {
    float e[ORDER > 0 ? row_entry(FORM, ORDER) : 1], p[ORDER > 0 ? ORDER : 1];
    uint32_t q;             // byte offset of its Phi (order 0)
    float d, rd, rl;
    bool in, hi;            // the lane lies in a slab; in the one at the far side
};

// The slab along `axis` that holds column c, and its Phi of term `term` (0 or
// 1); sl: byte offset of the field's slabs in the tables, rt: of its profiles.
template <int FORM, int ORDER>
__device__ __forceinline__ void plane_slab(PlaneSlab<FORM, ORDER> &s, const RowModel &a, const RowSlab *sl, rsrc_t rT,
                                           uint32_t rt, rsrc_t rP, int axis, int term, const int *c, int own, bool live)
{
    constexpr int NE = row_entry(FORM, ORDER);
    const RowSlab S0 = plane_slab_at(sl, axis), S1 = plane_slab_at(sl, axis + 3);
    auto holds = [&](const RowSlab &S) {
        bool in = live && S.t > 0;
#pragma unroll
        for (int q = 0; q < 3; ++q) in = in & (c[q] >= S.lo[q]) & (c[q] < S.hi[q]);
        return in;
    };
    const bool in0 = holds(S0), in1 = holds(S1);
    auto of = [&](int x0, int x1) { return in1 ? x1 : x0; };
    s.in = in0 | in1;
    s.hi = in1;
    s.d = in1 ? S1.d : S0.d;
    s.rd = in1 ? S1.rd : S0.rd;
    s.rl = in1 ? S1.rl : S0.rl;
    s.q = 4u * (uint32_t)(of(S0.off, S1.off) + c[0] * of(S0.sx, S1.sx) + c[1] * of(S0.sy, S1.sy) + c[2]) + (uint32_t)term * a.np4;
    if (!s.in) return;
    const uint32_t at = rt + 4u * (uint32_t)(of(S0.rt, S1.rt) + of(S0.sign, S1.sign) * (own - of(S0.pend, S1.pend)) * NE);
#pragma unroll
    for (int n = 0; n < NE / 4; ++n) {
        const float4 v = bits<float4>(__builtin_amdgcn_raw_buffer_load_b128(rT, at + 16u * n, 0, 0));
        s.e[4 * n] = v.x; s.e[4 * n + 1] = v.y; s.e[4 * n + 2] = v.z; s.e[4 * n + 3] = v.w;
    }
#pragma unroll
    for (int o = 0; o < ORDER; ++o) s.p[o] = bld(rP, s.q, (uint32_t)(2 * o) * a.np4);
}

// What the slab adds, its sign aside (row_slab for one cell and one component).
template <int FORM, int ORDER>
__device__ __forceinline__ float plane_corr(PlaneSlab<FORM, ORDER> &s, float c, float x)
{
    const float v = __builtin_fmaf(x, s.rd, x * s.rl);
    float q = __builtin_fmaf(__builtin_fmaf(-v, s.d, x), s.rd, v);
    const RowOdd odd = {__builtin_bit_cast(uint32_t, x) * 2u - 1u, q != q};
    if (odd.any()) q = x / s.d;
    float none = 0.f;
    return row_corr<FORM, ORDER>(s.e, c, q, s.p[0], ORDER == 2 ? s.p[ORDER - 1] : none);
}
template <int FORM, int ORDER>
__device__ __forceinline__ void plane_store(const PlaneSlab<FORM, ORDER> &s, rsrc_t w, uint32_t np4)
{
    if (!s.in) return;
#pragma unroll
    for (int o = 0; o < ORDER; ++o) bst(w, s.q, (uint32_t)(2 * o) * np4, s.p[o]);
}

// The sources of a kind on a lane's edge: those from s0 to before s1 (others may
// lie between), the first one's description beside, so that an iteration waits
// only for its sample, which is loaded at the iteration's start.
struct PlaneSrc {
    int s0 = 0, s1 = 0, pol, lo, hi;
    float f0, f1;
};
__device__ __forceinline__ PlaneSrc plane_src(const SrcArgs &A, const int *c, bool any)
{
    PlaneSrc r;
    if (!__any(any)) return r;
    const int n = A.n;
    for (int s = 0; s < n; ++s) {
        const int x = plane_uniform(A.info, 6 * s), y = plane_uniform(A.info, 6 * s + 1), z = plane_uniform(A.info, 6 * s + 2);
        const bool at = any & (x == c[0]) & (y == c[1]) & (z == c[2]);
        r.s0 = at && r.s1 == 0 ? s : r.s0;
        r.s1 = at ? s + 1 : r.s1;
    }
    if (r.s1) {
        const int *in = A.info + 6 * r.s0;
        r.pol = in[3]; r.lo = in[4]; r.hi = in[5];
        r.f0 = A.fac[2 * r.s0]; r.f1 = A.fac[2 * r.s0 + 1];
    }
    return r;
}
__device__ __forceinline__ float plane_sample(const PlaneSrc &r, const SrcArgs &A, int iterations, int it)
{
    return r.s1 ? A.waves[(size_t)r.s0 * iterations + it] : 0.f;
}
// Calls f(polarisation, sample, factors) for the sources of the edge at work in
// iteration it, in order.
template <class Fn>
__device__ __forceinline__ void plane_sources(const PlaneSrc &r, const SrcArgs &A, const int *c, int iterations, int it,
                                              float first, const Fn &f)
{
    if (!r.s1) return;
    if (it >= r.lo && it <= r.hi) f(r.pol, first, r.f0, r.f1);
    for (int s = r.s0 + 1; s < r.s1; ++s) {
        const int *in = A.info + 6 * s;
        if (in[0] != c[0] || in[1] != c[1] || in[2] != c[2] || it < in[4] || it > in[5]) continue;
        f(in[3], A.waves[(size_t)s * iterations + it], A.fac[2 * s], A.fac[2 * s + 1]);
    }
}

template <int FORM, int ORDER>
__global__ void __launch_bounds__(PLANE_BLOCK_MAX) k_plane(const RowModel *__restrict__ models, PlaneArgs b)
{
    extern __shared__ float lds[];
    const int g = logical_block(b.per_xcd);
    if (g >= b.nitems) return;
    const RowModel &a = *models;
    const int t = threadIdx.x, B = blockDim.x, tp = g / b.ntq, tq = g - tp * b.ntq;
    const int lp = t / b.tq, lq = t - lp * b.tq;
    const int cp = tp * (b.tp - 2 * b.halo) - b.halo + lp, cq = tq * (b.tq - 2 * b.halo) - b.halo + lq;
    const int w = b.w, u = w == 2 ? 0 : w + 1, v = w == 0 ? 2 : w - 1;
    const bool ufast = w == 1;
    const int cu_ = ufast ? cq : cp, cv_ = ufast ? cp : cq;
    const int dim[3] = {a.nx, a.ny, a.nz};
    const int nu = w == 0 ? dim[1] : (w == 1 ? dim[2] : dim[0]), nv = w == 0 ? dim[2] : (w == 1 ? dim[0] : dim[1]);
    const bool live = lp < b.tp && cu_ >= 0 && cu_ <= nu && cv_ >= 0 && cv_ <= nv;
    const bool own = live && lp >= b.halo && lp < b.tp - b.halo && lq >= b.halo && lq < b.tq - b.halo;
    const int cu = live ? cu_ : 0, cv = live ? cv_ : 0;
    const int c[3] = {w == 0 ? 0 : (w == 1 ? cv : cu), w == 0 ? cu : (w == 1 ? 0 : cv), w == 0 ? cv : (w == 1 ? cu : 0)};
    // lanes of the neighbours; at the tile's edges any lane, as what it gives is not used
    const int ds = ufast ? 1 : b.tq, dv = ufast ? b.tq : 1;
    const int up = t + ds < B ? t + ds : t, vp = t + dv < B ? t + dv : t;
    const int um = t >= ds ? t - ds : t, vm = t >= dv ? t - dv : t;
    const uint32_t cs = a.cs, ci = a.ci, np4 = __builtin_amdgcn_readfirstlane(a.np4);
    const uint32_t at = 4u * (uint32_t)(c[0] * a.plane + c[1] * a.kp + c[2]), ai = at >> 1;
    const rsrc_t rF = rsrc(a.F[b.flip]), rI = rsrc(a.ID), rT = rsrc(a.img);
    auto id = [&](uint32_t comp) {
        return 4u * (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rI, ai, comp * ci, 0);
    };
    const uint32_t iE = id(w);
    float E = bld(rF, at, w * cs), Hu = bld(rF, at, (3 + u) * cs), Hv = bld(rF, at, (3 + v) * cs);
    const uint32_t pf = live ? a.planeflag[c[0]] : 0u;
    const uint32_t nm = a.nmat, nh = b.hu ? 0 : nm, nRT = ORDER > 0 ? a.nRT : 0, ns = ORDER > 0 ? 6 * (sizeof(RowSlab) / 4) : 0;
    const uint32_t oH = 16u * a.n4E, tE = 16u * nm, tH = oH + 16u * nh, zE = tE + 4u * (nRT + ns), zH = tH + 4u * (nRT + ns);
    float kE[4], kU[4], kV[4];   // own, the two curl factors, srce or srcm
    kE[0] = bld(rT, 4u * iE, 0);
    kE[1] = bld(rT, 4u * iE, 4u + 4u * u);
    kE[2] = bld(rT, 4u * iE, 4u + 4u * v);
    kE[3] = bld(rT, iE, zE);
    if (b.hu) {
        kU[0] = kV[0] = a.h[0];
        kU[1] = a.h[1 + v]; kU[2] = a.h[1 + w] * 0.f;
        kV[1] = a.h[1 + w] * 0.f; kV[2] = a.h[1 + u];
        kU[3] = kV[3] = a.h[4];
    } else {
        const uint32_t iU = id(3 + u), iV = id(3 + v);
        kU[0] = bld(rT, 4u * iU, oH);
        kU[1] = bld(rT, 4u * iU, oH + 4u + 4u * v); kU[2] = bld(rT, 4u * iU, oH + 4u + 4u * w) * 0.f;
        kV[0] = bld(rT, 4u * iV, oH);
        kV[1] = bld(rT, 4u * iV, oH + 4u + 4u * w) * 0.f; kV[2] = bld(rT, 4u * iV, oH + 4u + 4u * u);
        kU[3] = bld(rT, iU, zH);
        kV[3] = bld(rT, iV, zH);
    }
    // E slabs along u and v, H slabs along u (for Hv) and v (for Hu)
    PlaneSlab<FORM, ORDER> eu, ev, su, sv;
    if constexpr (ORDER > 0) {
        const char *img = reinterpret_cast<const char *>(a.img);
        const RowSlab *slE = reinterpret_cast<const RowSlab *>(img + tE + 4u * nRT);
        const RowSlab *slH = reinterpret_cast<const RowSlab *>(img + tH + 4u * nRT);
        const rsrc_t rPE = rsrc(a.phiE[b.flipE]), rPH = rsrc(a.phiH[b.flip]);
        plane_slab(eu, a, slE, rT, tE, rPE, u, w == 0 ? 0 : 1, c, cu, live);
        plane_slab(ev, a, slE, rT, tE, rPE, v, w == 2 ? 1 : 0, c, cv, live);
        plane_slab(su, a, slH, rT, tH, rPH, u, w == 0 ? 1 : 0, c, cu, live);
        plane_slab(sv, a, slH, rT, tH, rPH, v, w == 2 ? 0 : 1, c, cv, live);
    }
    // the slabs' order is x0, y0, z0, xmax, ymax, zmax
    bool vfirst = false;
    if constexpr (ORDER > 0) vfirst = ev.hi == eu.hi ? v < u : eu.hi;
    const bool bE = cu >= 1 && cu < nu && cv >= 1 && cv < nv, bU = cu >= 1 && cv < nv, bV = cu < nu && cv >= 1;
    float *sE = lds, *sU = lds + B, *sV = lds + 2 * B;
    const StepRare &Q = *a.rare;
    const SrcArgs &M = Q.srcM, &V = Q.srcV, &D = Q.srcD;
    const PlaneSrc pM = plane_src(M, c, pf & PF_SRCH), pV = plane_src(V, c, pf & PF_SRCE), pD = plane_src(D, c, pf & PF_SRCE);
    int r0 = 0, r1 = 0;    // the lane's receivers are among these
    const bool rx = own && (pf & PF_RX);
    if (__any(rx)) {
        const int n = Q.nrx;
        const int *rxc = Q.rxc;
        for (int r = 0; r < n; ++r) {
            const int x = plane_uniform(rxc, 3 * r), y = plane_uniform(rxc, 3 * r + 1), z = plane_uniform(rxc, 3 * r + 2);
            const bool here = rx & (x == c[0]) & (y == c[1]) & (z == c[2]);
            r0 = here && r1 == 0 ? r : r0;
            r1 = here ? r + 1 : r1;
        }
    }
    for (int it = b.it; it < b.it + b.n; ++it) {
        const float xM = plane_sample(pM, M, a.iterations, it), xV = plane_sample(pV, V, a.iterations, it),
                    xD = plane_sample(pD, D, a.iterations, it);
        sE[t] = E;
        __syncthreads();
        for (int r = r0; r < r1; ++r) {    // the state at the start of the iteration
            const int *x = Q.rxc + 3 * r;
            if (r != r0 && (x[0] != c[0] || x[1] != c[1] || x[2] != c[2])) continue;
            float *o = Q.rxbuf + (size_t)it * Q.nrx + r;
            const size_t rs = (size_t)a.iterations * Q.nrx;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                o[q * rs] = q == w ? E : 0.f;
                o[(3 + q) * rs] = q == u ? Hu : (q == v ? Hv : 0.f);
            }
        }
        const float dU = sE[up] - E, dV = sE[vp] - E;
        float nU = kU[0] * Hu - kU[1] * dV + kU[2], nV = kV[0] * Hv - kV[1] + kV[2] * dU;
        Hu = bU ? nU : Hu;
        Hv = bV ? nV : Hv;
        if constexpr (ORDER > 0) {
            if (su.in) Hv += plane_corr(su, kV[3], dU);
            if (sv.in) Hu += -plane_corr(sv, kU[3], dV);
        }
        plane_sources(pM, M, c, a.iterations, it, xM, [&](int pol, float x, float f0, float) {
            if (pol == u) Hu = Hu - kU[3] * x * f0;
            if (pol == v) Hv = Hv - kV[3] * x * f0;
        });
        sU[t] = Hu;
        sV[t] = Hv;
        __syncthreads();
        const float gU = Hv - sV[um], gV = Hu - sU[vm];
        const float e = kE[0] * E + kE[1] * gU - kE[2] * gV;
        E = bE ? e : E;
        if constexpr (ORDER > 0) {
            if (eu.in || ev.in) {
                const float x = eu.in ? plane_corr(eu, kE[3], gU) : -0.f, y = ev.in ? -plane_corr(ev, kE[3], gV) : -0.f;
                E = vfirst ? E + y + x : E + x + y;
            }
        }
        plane_sources(pV, V, c, a.iterations, it, xV, [&](int pol, float x, float f0, float) {
            E = pol >= 4 ? -x / f0 : E - kE[3] * x * f0;
        });
        plane_sources(pD, D, c, a.iterations, it, xD, [&](int, float x, float f0, float f1) { E = E - kE[3] * x * f0 * f1; });
    }
    if (!own) return;
    const rsrc_t wF = rsrc(a.F[b.flip ^ 1]);
    bst(wF, at, w * cs, E);
    bst(wF, at, (3 + u) * cs, Hu);
    bst(wF, at, (3 + v) * cs, Hv);
    if constexpr (ORDER > 0) {
        const rsrc_t wPE = rsrc(a.phiE[b.flipE ^ 1]), wPH = rsrc(a.phiH[b.flip ^ 1]);
        plane_store(eu, wPE, np4);
        plane_store(ev, wPE, np4);
        plane_store(su, wPH, np4);
        plane_store(sv, wPH, np4);
    }
}

}  // namespace gpx

#endif  // GPX_PLANE_H
