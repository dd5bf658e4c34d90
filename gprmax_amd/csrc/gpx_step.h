// Device code shared by the translation units of libgprmax_hip.so: launch
// argument types, buffer-resource helpers, and the PML, dispersive and table
// helpers.  The row kernels (gpx_rows.h) and the general passes (gpx.hip) use
// them.
#ifndef GPX_STEP_H
#define GPX_STEP_H

#include <hip/hip_runtime.h>

#include <stddef.h>
#include <stdint.h>

#include <type_traits>

namespace gpx {

constexpr int MAX_SLABS = 6;
constexpr int MAX_POLES = 4;
constexpr int MAX_LDS_BYTES = 64 * 1024;

enum : int {
    F_MAIN = 1,
    F_SRC = 2,
    F_RX = 4,
    F_DISPB = 8,
    F_PML0 = 16,  // bits 4..9: one per slab
};
constexpr int F_PML_ALL = F_PML0 * ((1 << MAX_SLABS) - 1);

struct SlabArgs {
    int axis;        // 0 x, 1 y, 2 z
    int minus;       // 1 for xminus/yminus/zminus
    int lo[3], hi[3];// box of corrected cells for this field, [lo, hi)
    int pend;        // profile index p = pend - c (minus) or c - pend (plus)
    int off, sx, sy; // Phi index of cell (i, j, k): off + i sx + j sy + k
    uint32_t ostep;  // floats between the two orders of a Phi
    int t, order;
    int roff;        // offset of this slab's [4][order][t] table in the LDS R area
    float d;
    float *phi1, *phi2;
};

struct SrcArgs {
    int n;
    const int *info;     // [n][6]
    const float *fac;    // [n][2]
    const float *waves;  // [n][iterations]
};

constexpr uint32_t PF_RX = 1, PF_SRCH = 2, PF_SRCE = 4;
constexpr int PF_SLAB_E = 8, PF_SLAB_H = 16;

// Streamed arrays are read and written with buffer instructions: a scalar
// resource per array (base address in SGPRs), the lane's byte offset within
// the plane in a VGPR and the plane's byte offset in an SGPR, so no
// per-access vector address arithmetic is needed.  Offsets are 32-bit: an
// array holds fewer than 2^30 floats.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t rsrc(const void *p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, -1, 0x00020000);
}
// The b32 buffer builtins move raw 32-bit words; floats pass through as bits.
__device__ __forceinline__ float bld(rsrc_t r, uint32_t voff, uint32_t soff)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ void bst(rsrc_t r, uint32_t voff, uint32_t soff, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, 0);
}
template <class IDT>
__device__ __forceinline__ uint32_t bld_id(rsrc_t r, uint32_t voff, uint32_t soff)
{
    if (sizeof(IDT) == 1) return __builtin_amdgcn_raw_buffer_load_b8(r, voff, soff, 0);
    if (sizeof(IDT) == 2) return __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0);
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}

// Loads and stores at a uniform base pointer plus a 32-bit lane byte offset.
template <class T>
__device__ __forceinline__ T ld(const T *base, uint32_t boff)
{
    // Device memory: global, not flat, accesses (the pointer may have been
    // read from memory, which hides its address space from the compiler).
    // The value moves as a 4- or 8-byte word.
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4- or 8-byte values");
    typedef typename std::conditional<sizeof(T) == 4, uint32_t, unsigned long long>::type W;
    typedef __attribute__((address_space(1))) const W gW;
    const W w = *(gW *)(reinterpret_cast<const char *>(base) + boff);
    T v;
    __builtin_memcpy(&v, &w, sizeof(T));
    return v;
}
template <class T>
__device__ __forceinline__ void st(T *base, uint32_t boff, T v)
{
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4- or 8-byte values");
    typedef typename std::conditional<sizeof(T) == 4, uint32_t, unsigned long long>::type W;
    typedef __attribute__((address_space(1))) W gW;
    W w;
    __builtin_memcpy(&w, &v, sizeof(T));
    *(gW *)(reinterpret_cast<char *>(base) + boff) = w;
}

// ---------------------------------------------------------------- PML
// One corrected component (gprMax/pml_updates/*_ext.pyx) for formulation
// FORM (0 HORIPML, 1 MRIPML) and ORDER CFS terms.  R = [RA, RB, RE, RF] each
// [order][t] in LDS; i1/off index Phi order 0 and the order-1 offset.  Phi is
// read from `pin` and, when `wr`, the advanced values are written to `pout`
// (the same array for an in-place update).
// Phi pointers come from slab descriptions staged in LDS, so the compiler
// cannot tell their address space; Phi is always device memory, and global
// loads and stores avoid the flat path (which waits on both LDS and memory
// counters).
typedef __attribute__((address_space(1))) float gfloat_t;

// Phi values p0 (order 0) and p1 (order 1, ORDER 2 only) already loaded.
template <int FORM, int ORDER>
__device__ __forceinline__ float pml_v(const SlabArgs &s, const float *R, int p, float F,
                                       bool plus_sign, float c, float dd, float p0, float p1,
                                       float *pout_, bool wr, uint32_t i1, uint32_t off)
{
    gfloat_t *pout = (gfloat_t *)pout_;
    const int ot = ORDER * s.t;
    float corr;
    if (FORM == 0) {
        if (ORDER == 1) {  // pml_updates_*_HORIPML_ext.pyx, order1_*
            const float RA01 = R[p] - 1.0f;
            const float RB0 = R[ot + p], RE0 = R[2 * ot + p], RF0 = R[3 * ot + p];
            const float ph = p0;
            corr = c * (RA01 * dd + RB0 * ph);
            if (wr) pout[i1] = RE0 * ph - RF0 * dd;
        } else {           // order2_*
            const float RA0 = R[p], RA1 = R[s.t + p];
            const float RB0 = R[ot + p], RB1 = R[ot + s.t + p];
            const float RE0 = R[2 * ot + p], RE1 = R[2 * ot + s.t + p];
            const float RF0 = R[3 * ot + p], RF1 = R[3 * ot + s.t + p];
            const float RA01 = RA0 * RA1 - 1.0f;
            corr = c * (RA01 * dd + RA1 * RB0 * p0 + RB1 * p1);
            if (wr) {
                pout[i1 + off] = RE1 * p1 - RF1 * (RA0 * dd + RB0 * p0);
                pout[i1] = RE0 * p0 - RF0 * dd;
            }
        }
    } else {
        if (ORDER == 1) {  // pml_updates_*_MRIPML_ext.pyx, order1_*
            const float IRA = 1.0f / R[p];
            const float IRA1 = IRA - 1.0f;
            const float RB0 = R[ot + p], RE0 = R[2 * ot + p], RF0 = R[3 * ot + p];
            const float RC0 = IRA * RB0 * RF0;
            const float ph = p0;
            corr = c * (IRA1 * dd - IRA * ph);
            if (wr) pout[i1] = RE0 * ph + RC0 * dd - RC0 * ph;
        } else {           // order2_*
            const float IRA = 1.0f / (R[p] + R[s.t + p]);
            const float IRA1 = IRA - 1.0f;
            const float RB0 = R[ot + p], RB1 = R[ot + s.t + p];
            const float RE0 = R[2 * ot + p], RE1 = R[2 * ot + s.t + p];
            const float RC0 = IRA * R[3 * ot + p], RC1 = IRA * R[3 * ot + s.t + p];
            const float psi = RB0 * p0 + RB1 * p1;
            corr = c * (IRA1 * dd - IRA * psi);
            if (wr) {
                pout[i1 + off] = RE1 * p1 + RC1 * (dd - psi);
                pout[i1] = RE0 * p0 + RC0 * (dd - psi);
            }
        }
    }
    return plus_sign ? F + corr : F - corr;
}

// One in-place PML correction with the Phi values already loaded (phi_get).
__device__ __forceinline__ float pml_correct_pre(int form, const SlabArgs &s, const float *R, int p,
                                                 float F, bool plus_sign, float c, float dd, float p0,
                                                 float p1, float *phi, uint32_t i1, uint32_t off)
{
    if (form == 0)
        return s.order == 1 ? pml_v<0, 1>(s, R, p, F, plus_sign, c, dd, p0, p1, phi, true, i1, off)
                            : pml_v<0, 2>(s, R, p, F, plus_sign, c, dd, p0, p1, phi, true, i1, off);
    return s.order == 1 ? pml_v<1, 1>(s, R, p, F, plus_sign, c, dd, p0, p1, phi, true, i1, off)
                        : pml_v<1, 2>(s, R, p, F, plus_sign, c, dd, p0, p1, phi, true, i1, off);
}

// Profile index and Phi element index of cell (i, j, k).
__device__ __forceinline__ void slab_index(const SlabArgs &s, int i, int j, int k, int &p, uint32_t &q)
{
    const int along = s.axis == 0 ? i : (s.axis == 1 ? j : k);
    p = s.minus ? s.pend - along : along - s.pend;
    q = (uint32_t)(s.off + i * s.sx + j * s.sy + k);
}

// Phi of the first slab in `smask` for cell (i, j, k), loaded as soon as the
// cell's slabs are known: the loads then run beside the cell's field loads
// instead of after the main update that the correction follows.
struct PhiPre {
    int s;             // the slab, -1 when none
    int p;
    uint32_t q;
    float a1, b1, a2, b2;  // Phi1 orders 0 and 1, Phi2 orders 0 and 1
};

__device__ __forceinline__ void phi_preload(const SlabArgs *slab, uint32_t smask, int i, int j, int k, PhiPre &pp)
{
    pp.s = -1;
    pp.a1 = pp.b1 = pp.a2 = pp.b2 = 0.0f;
    if (!smask) return;
    const int s = __ffs(smask) - 1;
    const SlabArgs &sl = slab[s];
    slab_index(sl, i, j, k, pp.p, pp.q);
    pp.s = s;
    const gfloat_t *f1 = (const gfloat_t *)sl.phi1, *f2 = (const gfloat_t *)sl.phi2;
    pp.a1 = f1[pp.q];
    pp.a2 = f2[pp.q];
    if (sl.order == 2) {
        pp.b1 = f1[pp.q + sl.ostep];
        pp.b2 = f2[pp.q + sl.ostep];
    }
}

// Profile index, Phi index and Phi values of slab `s` for cell (i, j, k):
// from the preload when it holds that slab, else loaded here.
__device__ __forceinline__ void phi_get(const SlabArgs &sl, int s, const PhiPre &pre, int i, int j, int k, int &p,
                                        uint32_t &q, float &a1, float &b1, float &a2, float &b2)
{
    if (s == pre.s) {
        p = pre.p;
        q = pre.q;
        a1 = pre.a1; b1 = pre.b1; a2 = pre.a2; b2 = pre.b2;
        return;
    }
    slab_index(sl, i, j, k, p, q);
    const gfloat_t *f1 = (const gfloat_t *)sl.phi1, *f2 = (const gfloat_t *)sl.phi2;
    a1 = f1[q];
    a2 = f2[q];
    b1 = sl.order == 2 ? f1[q + sl.ostep] : 0.0f;
    b2 = sl.order == 2 ? f2[q + sl.ostep] : 0.0f;
}

// Blocks are dealt to the 8 XCDs round robin, so block b is renumbered
// (b mod 8) * per_xcd + b / 8; an XCD then works on a contiguous run of items, i.e. neighbouring plane segments that share rows
// through its L2.
__device__ __forceinline__ int logical_block(int per_xcd)
{
    const int b = blockIdx.x;
    return (b & 7) * per_xcd + (b >> 3);
}

// Copy a small table to LDS with four loads in flight per thread.
// Slab descriptions go to LDS so the PML branch reads them into VGPRs when a
// lane needs them instead of holding them in SGPRs for the whole loop.
__device__ __forceinline__ void stage_slabs(SlabArgs *dst, const SlabArgs *slab, int nslab)
{
    const int words = (int)(sizeof(SlabArgs) / 4) * nslab;
    const int *src = reinterpret_cast<const int *>(slab);
    int *d = reinterpret_cast<int *>(dst);
    for (int q = threadIdx.x; q < words; q += blockDim.x) d[q] = src[q];
}

__device__ __forceinline__ void stage(float *dst, const float *src, int n)
{
    const int B = blockDim.x;
    for (int q = threadIdx.x; q < n; q += 4 * B) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = q + u * B < n ? src[q + u * B] : 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (q + u * B < n) dst[q + u * B] = v[u];
    }
}

// Coefficients in LDS: (CA, CBx, CBy, CBz) or (DA, DBx, DBy, DBz) as one
// float4 per material, then srce/srcm as one float per material.
__device__ __forceinline__ void stage_coef(float4 *c4, float *c1, const float *src, int nmat)
{
    for (int m = threadIdx.x; m < nmat; m += blockDim.x) {
        const float *r = src + 5 * m;
        c4[m] = make_float4(r[0], r[1], r[2], r[3]);
        c1[m] = r[4];
    }
}

// Dispersive part A for one component (gprMax/fields_updates_ext.pyx:113-296):
// returns phi and advances the P auxiliary values from the old field e.
template <int P, bool CPLX>
__device__ __forceinline__ float disp_a(const float *D, uint32_t m, float *tr, float *ti, float e)
{
    float phi = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (CPLX) {
            const float *c = D + ((size_t)m * 3 * P + 3 * p) * 2;
            if (P == 1) phi = c[0] * tr[p];
            else phi = phi + c[0] * tr[p];
            const float er = c[2], ei = c[3], zr = c[4], zi = c[5];
            const float nr = (er * tr[p] - ei * ti[p]) + zr * e;
            const float ni = (er * ti[p] + ei * tr[p]) + zi * e;
            tr[p] = nr;
            ti[p] = ni;
        } else {
            const float *c = D + (size_t)m * 3 * P + 3 * p;
            if (P == 1) phi = c[0] * tr[p];
            else phi = phi + c[0] * tr[p];
            tr[p] = c[1] * tr[p] + c[2] * e;
        }
    }
    return phi;
}

// Dispersive part B (gprMax/fields_updates_ext.pyx:183-235, 299-346).
template <int P, bool CPLX>
__device__ __forceinline__ void disp_b(const float *D, uint32_t m, float *tr, float *ti, float e)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (CPLX) {
            const float *c = D + ((size_t)m * 3 * P + 3 * p) * 2;
            tr[p] = tr[p] - c[4] * e;
            ti[p] = ti[p] - c[5] * e;
        } else {
            tr[p] = tr[p] - D[(size_t)m * 3 * P + 3 * p + 2] * e;
        }
    }
}

// Dispersive auxiliary values, compacted: component c keeps its P poles
// only for the edges whose material has poles, in cell order,
// T[c][p * n[c] + slot], with slot[c][cell] the edge's place in that order
// (read only on such edges).
struct TArgs {
    float *T[3];
    const uint32_t *slot[3];
    long long n[3];
    const uint32_t *masks;    // [nx + 1][groups] entries of 64 bytes (row_slots_of)
    int groups;
};

// Slot of an edge whose material has no poles.
constexpr uint32_t T_NOSLOT = 0xffffffffu;

// Loads the P values of component c in slot s.
template <int P, bool CPLX>
__device__ __forceinline__ void t_load_at(const TArgs &t, int c, uint32_t s, float *tr, float *ti)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const size_t e = (size_t)p * (size_t)t.n[c] + s;
        if (CPLX) {
            const float2 v = ld(reinterpret_cast<const float2 *>(t.T[c]) + e, 0u);
            tr[p] = v.x;
            ti[p] = v.y;
        } else {
            tr[p] = ld((const float *)t.T[c] + e, 0u);
            ti[p] = 0.f;
        }
    }
}

template <int P, bool CPLX>
__device__ __forceinline__ void t_store(const TArgs &t, int c, uint32_t s, const float *tr, const float *ti)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const size_t e = (size_t)p * (size_t)t.n[c] + s;
        if (CPLX)
            st(reinterpret_cast<float2 *>(t.T[c]) + e, 0u, make_float2(tr[p], ti[p]));
        else
            st(t.T[c] + e, 0u, tr[p]);
    }
}

// Sources and receivers of the row kernels.  They are read only on planes that
// hold one, from device memory, so their addresses do not occupy registers
// for the whole kernel.
struct StepRare {
    SrcArgs srcM, srcV, srcD;    // magnetic dipoles, voltage sources, Hertzian dipoles
    int nrx;
    const int *rxc;              // [nrx][3]
    float *rxbuf;                // [6][iterations][nrx]
};

}  // namespace gpx

#endif  // GPX_STEP_H
