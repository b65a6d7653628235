// Per-quad whole-step updates shared by the slab engine and the batched engine: the E
// pass of one quad (core E + CPML-E + E sources + E probes) and the H pass (core H +
// CPML-H + H sources + H probes), with the same per-cell arithmetic as the in-place
// update_e/update_h + CPML + source kernels (bit for bit, masked lanes value*0).
#pragma once

#include "common.hpp"
#include "row_quads.hpp"

namespace mifdtd {

constexpr int SB = 256;
constexpr int kSMaxSrc = 4;
constexpr int kSMaxProbe = 8;

struct SCpml {
    int npml;
    int axes;                // bit a: CPML on both faces of axis a (x = 1, y = 2, z = 4)
    const float *bE, *aE, *bH, *aH;
    float *pe, *ph;          // packed psi E / psi H
    float *pe_out;           // where the E pass stores psi E (pe for in-place updates)
    size_t sX, sY, sZ;
    __host__ __device__ __forceinline__ size_t off(int f, int c) const
    {
        const int ax = f >> 1, sd = f & 1;
        if (ax == 0) return (size_t)(2 * sd + c) * sX;
        if (ax == 1) return 4 * sX + (size_t)(2 * sd + c) * sY;
        return 4 * sX + 4 * sY + (size_t)(2 * sd + c) * sZ;
    }
};

struct SSrc {
    int n;
    int comp[kSMaxSrc], i0[kSMaxSrc], i1[kSMaxSrc], j0[kSMaxSrc], j1[kSMaxSrc], k0[kSMaxSrc], k1[kSMaxSrc], ow[kSMaxSrc];
    float tval[kSMaxSrc], svs[kSMaxSrc];
    const float *sv[kSMaxSrc];
};

struct SProbe {
    int n;
    int comp[kSMaxProbe], i[kSMaxProbe], j[kSMaxProbe], k[kSMaxProbe], slot[kSMaxProbe];
    float *out;  // row of the probe series for this step; probe n writes out[slot[n]]
};

// A Drude box (auxiliary current; kuFDTD matter.py:104-221, drude_ade.c): on cells of the
// inclusive box [i0,i1] x [j0,j1] x [k0,k1], right after the core E update and before
// CPML-E and the sources, each component takes e' = e - CE J ; J' = CJA J + CJB e'.
// a/b: CJA/CJB, C-order box arrays (lj x lk per plane); J is read from jin and J' written
// to jout (the step's two current sets).
struct SDrude {
    int i0, i1, j0, j1, k0, k1;
    int lj, lk;
    const float *a[3], *b[3], *jin[3];
    float *jout[3];
    __device__ __forceinline__ bool row_in(int i, int j) const { return i >= i0 && i <= i1 && j >= j0 && j <= j1; }
};

// Drude update of component c on the quad (i, j, k0..k0+3) of a row inside the box (row_in):
// e: the core-updated values, ce: the quad's CE; returns J' in jn (stored by the caller
// for the cells it owns).
__device__ __forceinline__ void drude_quad(const SDrude &d, int c, int i, int j, int k0, const Q4 &ce, Q4 &e, Q4 &jn)
{
    const size_t rowb = ((size_t)(i - d.i0) * d.lj + (j - d.j0)) * d.lk;
    bool in[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) in[l] = k0 + l >= d.k0 && k0 + l <= d.k1;
    Q4 f, a, b;
    if (in[0] && in[3] && ((rowb + (size_t)(k0 - d.k0)) & 3u) == 0) {  // whole quad, 16-byte aligned
        const size_t n0 = rowb + (size_t)(k0 - d.k0);
        f = ld4(d.jin[c] + n0);
        a = ld4(d.a[c] + n0);
        b = ld4(d.b[c] + n0);
    } else {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const size_t n = in[l] ? rowb + (size_t)(k0 + l - d.k0) : rowb;
            f.v[l] = in[l] ? d.jin[c][n] : 0.f;
            a.v[l] = in[l] ? d.a[c][n] : 0.f;
            b.v[l] = in[l] ? d.b[c][n] : 0.f;
        }
    }
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        if (in[l]) {
            const float et = e.v[l] - ce.v[l] * f.v[l];
            e.v[l] = et;
            jn.v[l] = a.v[l] * f.v[l] + b.v[l] * et;
        }
    }
}

// Stores the J' of drude_quad for the quad's cells inside the box.
__device__ __forceinline__ void drude_store(const SDrude &d, int c, int i, int j, int k0, const Q4 &jn)
{
    const size_t rowb = ((size_t)(i - d.i0) * d.lj + (j - d.j0)) * d.lk;
    const size_t n0 = rowb + (size_t)(k0 - d.k0);
    if (k0 >= d.k0 && k0 + 3 <= d.k1 && (n0 & 3u) == 0) {
        st4(d.jout[c] + n0, jn);
        return;
    }
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int k = k0 + l;
        if (k >= d.k0 && k <= d.k1) d.jout[c][rowb + (size_t)(k - d.k0)] = jn.v[l];
    }
}

// TFSF face patches of one half step (kuFDTD tfsf.py:138-226 tables, normal incidence):
// patch p adds 0.5 * (coef * line[base + along]) to component comp on its inclusive box,
// along being the offset along the propagation axis from the box start; patches apply in
// table order after the sources.  line: the 1-D incident line of the other half (H for
// the E patches, E for the H patches).
constexpr int kTfMaxPatch = 12;
struct STfsf {
    int n, axis, line_n;
    int comp[kTfMaxPatch], box[kTfMaxPatch][6], base[kTfMaxPatch];
    float coef[kTfMaxPatch];
    const float *line;
};

__device__ __forceinline__ void tfsf_add(const STfsf &t, int p, int i, int j, int k0, Q4 &f)
{
    const int *b = t.box[p];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int k = k0 + l;
        if (k >= b[4] && k <= b[5]) {
            const int along = t.axis == 0 ? i - b[0] : t.axis == 1 ? j - b[2] : k - b[4];
            const float v = 0.5f * (t.coef[p] * t.line[t.base[p] + along]);
            f.v[l] = f.v[l] + v;
        }
    }
}

// The patches of one half step on the quad (i, j, k0..k0+3); c0: 0 for E, 3 for H; mask:
// the patches to consider (bit p; patches known not to touch the quad may be left out),
// applied in table order.
__device__ __forceinline__ void tfsf_quad(const STfsf &t, int c0, int i, int j, int k0, Q4 &f0, Q4 &f1, Q4 &f2,
                                          unsigned mask = ~0u)
{
    for (int p = 0; p < t.n; ++p) {
        if (!((mask >> p) & 1u)) continue;
        const int *b = t.box[p];
        if (i < b[0] || i > b[1] || j < b[2] || j > b[3]) continue;
        if (k0 + 3 < b[4] || k0 > b[5]) continue;  // the quad misses the patch (z-face patches: all lanes but one)
        const int c = t.comp[p] - c0;
        if (c == 0) tfsf_add(t, p, i, j, k0, f0);
        else if (c == 1) tfsf_add(t, p, i, j, k0, f1);
        else tfsf_add(t, p, i, j, k0, f2);
    }
}

// Bit p set for each patch of t whose box meets planes [ia, ib], row j and cells [ka, kb].
__device__ __forceinline__ unsigned tfsf_mask(const STfsf &t, int ia, int ib, int j, int ka, int kb)
{
    unsigned m = 0;
    for (int p = 0; p < t.n; ++p) {
        const int *b = t.box[p];
        if (b[0] <= ib && ia <= b[1] && j >= b[2] && j <= b[3] && b[4] <= kb && ka <= b[5]) m |= 1u << p;
    }
    return m;
}

// Design box of the adjoint: the curl of H (the factor of CE in the core E update) of its
// cells is stored component after component, C order, before the update changes E.
struct SCurl {
    int i0, j0, k0, di, dj, dk;
    float *out;
    __device__ __forceinline__ bool row_in(int i, int j) const
    {
        return i >= i0 && i < i0 + di && j >= j0 && j < j0 + dj;
    }
    __device__ __forceinline__ void store(int i, int j, int q0, const Q4 &x, const Q4 &y, const Q4 &z) const
    {
        const size_t s = (size_t)di * dj * dk;
        float *p = out + ((size_t)(i - i0) * dj + (j - j0)) * dk + (q0 - k0);
        if (q0 >= k0 && q0 + 4 <= k0 + dk && (((size_t)p | (s << 2)) & 15u) == 0) {
            st4(p, x);
            st4(p + s, y);
            st4(p + 2 * s, z);
            return;
        }
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            if (q0 + l < k0 || q0 + l >= k0 + dk) continue;
            p[l] = x.v[l];
            p[l + s] = y.v[l];
            p[l + 2 * s] = z.v[l];
        }
    }
};

struct SGeom {
    int nx, ny, nzp, nz;
    int i0;            // first plane of the slab
    RowQuads m;        // thread -> quad order over the slab's rows (whole-grid passes)
};

__host__ __device__ __forceinline__ int sslab_e(int q, int n_e, int npml, int &side, int &p)
{
    side = 0;
    p = 0;
    if (q < npml) { p = q; return p + 1; }
    if (q >= n_e - 1 - npml && q < n_e - 1) { side = 1; p = q - (n_e - 1 - npml); return npml + 1 + p; }
    return -1;
}
__host__ __device__ __forceinline__ int sslab_h(int q, int n_e, int npml, int &side, int &p)
{
    side = 0;
    p = 0;
    if (q < npml) { p = q; return p + 1; }
    if (q >= n_e - npml && q < n_e) { side = 1; p = q - (n_e - npml); return npml + 2 + p; }
    return -1;
}

// Source n's value of the step is s.tval[n], or tv_row[tv[n]] where tv_row is given.
__device__ __forceinline__ void sapply_src(const SSrc &s, int c, int i, int j, int k0, Q4 &v,
                                           const float *tv_row = nullptr, const int *tv = nullptr)
{
#pragma unroll 1
    for (int n = 0; n < s.n; ++n) {
        if (s.comp[n] == c && i >= s.i0[n] && i <= s.i1[n] && j >= s.j0[n] && j <= s.j1[n] &&
            k0 + 3 >= s.k0[n] && k0 <= s.k1[n]) {
            const int lj = s.j1[n] - s.j0[n] + 1, lk = s.k1[n] - s.k0[n] + 1;
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int k = k0 + l;
                if (k >= s.k0[n] && k <= s.k1[n]) {
                    const float w = s.sv[n] ? s.sv[n][((size_t)(i - s.i0[n]) * lj + (j - s.j0[n])) * lk + (k - s.k0[n])]
                                            : s.svs[n];
                    const float add = (tv_row ? tv_row[tv[n]] : s.tval[n]) * w;
                    v.v[l] = s.ow[n] ? add : v.v[l] + add;
                }
            }
        }
    }
}

// row: the step's probe row (p.out where it is null).
__device__ __forceinline__ void sprobe(const SProbe &p, int c, int i, int j, int k0, const Q4 &v, float *row = nullptr)
{
    float *out = row ? row : p.out;
#pragma unroll 1
    for (int n = 0; n < p.n; ++n) {
        if (p.comp[n] == c && p.i[n] == i && p.j[n] == j) {
#pragma unroll
            for (int l = 0; l < 4; ++l)
                if (p.k[n] == k0 + l) out[p.slot[n]] = v.v[l];
        }
    }
}

// The kernel's first argument, read where it is used: tables that few waves consult
// (sources, probes) passed as an ordinary argument are loaded into scalar registers at the
// kernel's start (54 of them spilled to vector lanes in the E pass).
template <class T>
__device__ __forceinline__ const T &first_kernel_arg()
{
    return *(const T *)__builtin_amdgcn_kernarg_segment_ptr();
}

// Both passes issue the quad's core loads (fields, neighbours, CE), the psi of its first x
// or y face and the psi of its z-slab cells together, then compute; the psi of a second face
// (the edges along z) follows after the core update.  92-104 and 96 VGPRs, 4 and 5 waves per
// SIMD.  Holding all six psi quads across the update took 120 and spilled scalars; loading the
// z faces after the update kept 6 waves and was slower (160^3 step 74 us against 64).

// How CE reaches the E update: the constant 0.5, three float arrays, or three uint8
// material-index arrays into a 3 x 256 float table (same float values, so the products
// are identical; 3 B per cell instead of 12).  The per-quad passes read the 3 KiB table
// from global memory, where it stays in L1/L2; the sweep kernels stage it in LDS.
enum CeMode { kCeConst = 0, kCeArrays = 1, kCeTable = 2, kCeTriple = 3 };  // kCeTriple: the fused sweep only

// CE of a quad as uint8 material indices m[0..3] into a 256-entry float table.
__device__ __forceinline__ Q4 ce_from_table(const unsigned char *__restrict__ m, const float *tab)
{
    const uchar4 t = *reinterpret_cast<const uchar4 *>(m);
    Q4 q;
    q.v[0] = tab[t.x];
    q.v[1] = tab[t.y];
    q.v[2] = tab[t.z];
    q.v[3] = tab[t.w];
    return q;
}

// Whole-wave lane shifts (DPP wave_shl:1 / wave_shr:1): lane i takes lane i+1's (next) or
// lane i-1's (prev) value; the lane at the end takes 0.
__device__ __forceinline__ float lane_next(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_prev(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, false));
}

// Sources and probes of one half step with the box [lo, hi] (quads: cells k rounded down
// and up) around all of them: waves outside the box skip the tables.
struct SAux {
    int i0, i1, j0, j1, k0, k1;  // i0 > i1: none
    SSrc src;
    SProbe prb;
    __device__ __forceinline__ bool near(int i, int j, int q0) const
    {
        return i >= i0 && i <= i1 && j >= j0 && j <= j1 && q0 + 3 >= k0 && q0 <= k1;
    }
};

inline void aux_cover(SAux &a, int i0, int i1, int j0, int j1, int k0, int k1)
{
    const bool first = a.i0 > a.i1;
    a.i0 = first || i0 < a.i0 ? i0 : a.i0;
    a.i1 = first || i1 > a.i1 ? i1 : a.i1;
    a.j0 = first || j0 < a.j0 ? j0 : a.j0;
    a.j1 = first || j1 > a.j1 ? j1 : a.j1;
    a.k0 = first || k0 < a.k0 ? k0 : a.k0;
    a.k1 = first || k1 > a.k1 ? k1 : a.k1;
}

// The box around src's and prb's cells.
inline void aux_box(SAux &a)
{
    a.i0 = 1;
    a.i1 = 0;
    for (int n = 0; n < a.src.n; ++n)
        aux_cover(a, a.src.i0[n], a.src.i1[n], a.src.j0[n], a.src.j1[n], a.src.k0[n], a.src.k1[n]);
    for (int n = 0; n < a.prb.n; ++n)
        aux_cover(a, a.prb.i[n], a.prb.i[n], a.prb.j[n], a.prb.j[n], a.prb.k[n], a.prb.k[n]);
}

// Table entry (t > 0: in a slab) and psi1 offset of cell k0+l of a z-slab quad; psi2 follows sZ
// later.  A cell in no slab takes the first cell of the row in the slab that the quad meets:
// its load, whose value is not used, stays inside the z faces, the only part of the buffer
// that a caller with CPML on z alone has to provide.
template <bool E>
__host__ __device__ __forceinline__ int zface_at(const SCpml &cp, int i, int j, int k0, int l, int ny, int nz, size_t &o)
{
    int zs, zp, t = E ? sslab_e(k0 + l, nz, cp.npml, zs, zp) : sslab_h(k0 + l, nz, cp.npml, zs, zp);
    if (!E && k0 + l == 0) t = -1;  // the wall
    if (t <= 0) {
        zs = k0 >= cp.npml;
        zp = 0;
    }
    o = cp.off(4 + zs, 0) + ((size_t)i * ny + j) * cp.npml + zp;
    return t;
}

// z-face psi and table entries of a quad's cells, loaded ahead of the update: loads that
// follow the previous cell's psi store are four memory round trips in a row.
struct ZFace {
    float q1[4], q2[4], b[4], a[4];
    __device__ __forceinline__ void load(int l, int t, const float *psi, size_t o, size_t s2, const float *tb,
                                         const float *ta)
    {
        const int e = t > 0 ? t : 0;
        q1[l] = psi[o];
        q2[l] = psi[o + s2];
        b[l] = tb[e];
        a[l] = ta[e];
    }
};

// E pass on the quad (i, j, k0..k0+3): reads E from exi.. and writes it to exo.. (the
// same arrays for an in-place update, the next-step buffers for a ping-pong one); psi E
// is read from cp.pe and written to cp.pe_out.  CE: CM = 0 the constant 0.5, 1 the float
// arrays cex.., 2 the uint8 material indices mx.. into tab ([3][256] floats, the same
// values as the arrays, so the products are identical).  next: the next lane holds the
// quad at k0+4 (else this lane loads its k0+4 neighbours itself).
constexpr int kFeatDrude = 1, kFeatTfsf = 2, kFeatCurl = 4;  // optional E-pass features (template bits)

template <int CM, bool PML, int FEAT = 0>
__device__ __forceinline__ void e_quad_at(
    const SGeom &g, int i, int j, int k0, bool next, const float *exi, const float *eyi, const float *ezi, float *exo,
    float *eyo, float *ezo, const float *__restrict__ hx, const float *__restrict__ hy, const float *__restrict__ hz,
    const float *__restrict__ cex, const float *__restrict__ cey, const float *__restrict__ cez,
    const SCpml &cp, const SAux &aux, const unsigned char *__restrict__ mx = nullptr,
    const unsigned char *__restrict__ my = nullptr, const unsigned char *__restrict__ mz = nullptr,
    const float *tab = nullptr, const SDrude *dr = nullptr, const STfsf *tf = nullptr, float *prow = nullptr,
    const float *tv_row = nullptr, const int *tv = nullptr, const SCurl *cu = nullptr)
{
    constexpr bool DR = (FEAT & kFeatDrude) != 0;
    constexpr bool TF = (FEAT & kFeatTfsf) != 0;
    const int nx = g.nx, ny = g.ny, nzp = g.nzp, nz = g.nz;
    const size_t id = ((size_t)i * ny + j) * nzp + k0;
    const size_t sx = (size_t)ny * nzp;
    const bool jy = j < ny - 1, ix = i < nx - 1;
    const Q4 z4 = splat4(0.f);

    // ---------------------------------------------------------------- loads
    const Q4 hx0 = ld4(hx + id), hy0 = ld4(hy + id), hz0 = ld4(hz + id);
    Q4 e0 = ld4(exi + id), e1 = ld4(eyi + id), e2 = ld4(ezi + id);
    const Q4 c0 = CM == 2 ? ce_from_table(mx + id, tab) : CM ? ld4(cex + id) : splat4(0.5f);
    const Q4 c1 = CM == 2 ? ce_from_table(my + id, tab + 256) : CM ? ld4(cey + id) : splat4(0.5f);
    const Q4 c2 = CM == 2 ? ce_from_table(mz + id, tab + 512) : CM ? ld4(cez + id) : splat4(0.5f);
    const Q4 hzU = jy ? ld4(hz + id + nzp) : z4;   // hz(j+1)
    const Q4 hxU = jy ? ld4(hx + id + nzp) : z4;   // hx(j+1)
    const Q4 hzN = ix ? ld4(hz + id + sx) : z4;    // hz(i+1)
    const Q4 hyN = ix ? ld4(hy + id + sx) : z4;    // hy(i+1)
    // hy, hx at k0+4: the next quad / next row's start
    float hyn = 0.f, hxn = 0.f;
    if (!next) {
        if (jy) hyn = hy[id + 4];
        if (ix) hxn = hx[id + 4];
    }

    const int npml = PML ? cp.npml : 0;
    int xs = 0, xp = 0, ys = 0, yp = 0, xt = -1, yt = -1;
    Q4 p1 = z4, p2 = z4;   // psi of the x face, or of the y face where there is no x face
    float pb = 0.f, pa = 0.f;
    size_t o1 = 0, o2 = 0;
    ZFace z;
    bool zq = false;
    if (PML) {
        xt = (cp.axes & 1) ? sslab_e(i, nx, npml, xs, xp) : -1;  // x slab planes are all < nx-1
        yt = (cp.axes & 2) ? sslab_e(j, ny, npml, ys, yp) : -1;  // y slab rows are all < ny-1
        if (xt > 0 || yt > 0) {
            const size_t o = xt > 0 ? ((size_t)xp * ny + j) * nzp + k0 : ((size_t)i * npml + yp) * nzp + k0;
            const int f = xt > 0 ? xs : 2 + ys;
            const int t = xt > 0 ? xt : yt;
            o1 = cp.off(f, 0) + o;
            o2 = cp.off(f, 1) + o;
            p1 = ld4(cp.pe + o1);
            p2 = ld4(cp.pe + o2);
            pb = cp.bE[t];
            pa = cp.aE[t];
        }
        zq = (cp.axes & 4) && (k0 < npml || (k0 + 3 >= nz - 1 - npml && k0 < nz - 1));
        if (zq) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                size_t o;
                const int t = zface_at<true>(cp, i, j, k0, l, ny, nz, o);
                z.load(l, t, cp.pe, o, cp.sZ, cp.bE, cp.aE);
            }
        }
    }

    // -------------------------------------------------------------- compute
    // ex: += cex*((hz[j+1]-hz) - (hy[k+1]-hy)) ; CPML + y psi2 (hz), - z psi1 (hy)
    // ey: += cey*((hx[k+1]-hx) - (hz[i+1]-hz)) ; CPML - x psi1 (hz), + z psi2 (hx)
    // ez: += cez*((hy[i+1]-hy) - (hx[j+1]-hx)) ; CPML + x psi2 (hy), - y psi1 (hx)
    const float y3 = lane_next(hy0.v[0]), x3 = lane_next(hx0.v[0]);  // every lane of the wave takes part
    if (next) {
        hyn = y3;
        hxn = x3;
    }
    // Drude box: J' of the three components (rows inside the box)
    const bool drow = DR && dr->row_in(i, j);
    Q4 jn0 = z4, jn1 = z4, jn2 = z4;
    float y1[4], x1[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        y1[l] = l < 3 ? hy0.v[l + 1] : hyn;
        x1[l] = l < 3 ? hx0.v[l + 1] : hxn;
    }
    if ((FEAT & kFeatCurl) && cu->row_in(i, j)) {
        Q4 w0, w1, w2;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            w0.v[l] = (hzU.v[l] - hz0.v[l]) - (y1[l] - hy0.v[l]);
            w1.v[l] = (x1[l] - hx0.v[l]) - (hzN.v[l] - hz0.v[l]);
            w2.v[l] = (hyN.v[l] - hy0.v[l]) - (hxU.v[l] - hx0.v[l]);
        }
        cu->store(i, j, k0, w0, w1, w2);
    }
    if (jy) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float v = e0.v[l] + c0.v[l] * ((hzU.v[l] - hz0.v[l]) - (y1[l] - hy0.v[l]));
            e0.v[l] = (k0 + l < nz - 1) ? v : v * 0.f;
        }
    }
    if (ix) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float v = e1.v[l] + c1.v[l] * ((x1[l] - hx0.v[l]) - (hzN.v[l] - hz0.v[l]));
            e1.v[l] = (k0 + l < nz - 1) ? v : v * 0.f;
        }
    }
    if (ix && jy) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float v = e2.v[l] + c2.v[l] * ((hyN.v[l] - hy0.v[l]) - (hxU.v[l] - hx0.v[l]));
            e2.v[l] = (k0 + l < nz) ? v : v * 0.f;
        }
    }
    if (drow) {
        drude_quad(*dr, 0, i, j, k0, c0, e0, jn0);
        drude_quad(*dr, 1, i, j, k0, c1, e1, jn1);
        drude_quad(*dr, 2, i, j, k0, c2, e2, jn2);
    }
    if (PML) {
        if (xt > 0) {  // psi1: ey, psi2: ez
            const float b = pb, a = pa;
#pragma unroll
            for (int l = 0; l < 4; ++l)
                if (k0 + l < nz - 1) {
                    const float tt = b * p1.v[l] + a * (hzN.v[l] - hz0.v[l]);
                    p1.v[l] = tt;
                    e1.v[l] = e1.v[l] - c1.v[l] * tt;
                }
            if (jy) {
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (k0 + l < nz) {
                        const float tt = b * p2.v[l] + a * (hyN.v[l] - hy0.v[l]);
                        p2.v[l] = tt;
                        e2.v[l] = e2.v[l] + c2.v[l] * tt;
                    }
            }
            st4(cp.pe_out + o1, p1);
            st4(cp.pe_out + o2, p2);
        }
        if (yt > 0) {  // psi1: ez, psi2: ex
            if (xt > 0) {
                const size_t o = ((size_t)i * npml + yp) * nzp + k0;
                o1 = cp.off(2 + ys, 0) + o;
                o2 = cp.off(2 + ys, 1) + o;
                p1 = ld4(cp.pe + o1);
                p2 = ld4(cp.pe + o2);
                pb = cp.bE[yt];
                pa = cp.aE[yt];
            }
            const float b = pb, a = pa;
#pragma unroll
            for (int l = 0; l < 4; ++l)
                if (k0 + l < nz - 1) {
                    const float tt = b * p2.v[l] + a * (hzU.v[l] - hz0.v[l]);
                    p2.v[l] = tt;
                    e0.v[l] = e0.v[l] + c0.v[l] * tt;
                }
            if (ix) {
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (k0 + l < nz) {
                        const float tt = b * p1.v[l] + a * (hxU.v[l] - hx0.v[l]);
                        p1.v[l] = tt;
                        e2.v[l] = e2.v[l] - c2.v[l] * tt;
                    }
            }
            st4(cp.pe_out + o1, p1);
            st4(cp.pe_out + o2, p2);
        }
        if (zq) {  // psi1: ex, psi2: ey
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                size_t o;
                const bool on = zface_at<true>(cp, i, j, k0, l, ny, nz, o) > 0;
                if (on && jy) {
                    const float tt = z.b[l] * z.q1[l] + z.a[l] * (y1[l] - hy0.v[l]);
                    cp.pe_out[o] = tt;
                    e0.v[l] = e0.v[l] - c0.v[l] * tt;
                }
                if (on && ix) {
                    const float tt = z.b[l] * z.q2[l] + z.a[l] * (x1[l] - hx0.v[l]);
                    cp.pe_out[o + cp.sZ] = tt;
                    e1.v[l] = e1.v[l] + c1.v[l] * tt;
                }
            }
        }
    }
    const bool near = aux.near(i, j, k0);
    if (near) {
        sapply_src(aux.src, 0, i, j, k0, e0, tv_row, tv);
        sapply_src(aux.src, 1, i, j, k0, e1, tv_row, tv);
        sapply_src(aux.src, 2, i, j, k0, e2, tv_row, tv);
    }
    if (TF) tfsf_quad(*tf, 0, i, j, k0, e0, e1, e2);

    // --------------------------------------------------------------- stores
    // (unchanged lanes store back the value they loaded; in place, a row or plane that nothing
    // updates is left alone, so that another stream may write it while the pass runs)
    const bool all = exo != exi || near || drow || TF;
    if (all || jy) st4(exo + id, e0);
    if (all || ix) st4(eyo + id, e1);
    if (all || (ix && jy)) st4(ezo + id, e2);
    if (drow) {
        drude_store(*dr, 0, i, j, k0, jn0);
        drude_store(*dr, 1, i, j, k0, jn1);
        drude_store(*dr, 2, i, j, k0, jn2);
    }
    if (near) {
        sprobe(aux.prb, 0, i, j, k0, e0, prow);
        sprobe(aux.prb, 1, i, j, k0, e1, prow);
        sprobe(aux.prb, 2, i, j, k0, e2, prow);
    }
}

// H pass on the quad (i, j, k0..k0+3): reads H from hxi.. and writes it to hxo.. (the
// same arrays for an in-place update); psi H is updated in place (cp.ph).  prev: the
// previous lane holds the quad at k0-4.
// CH: the coefficient arrays ch[0..2] in place of the constant 0.5.
template <bool PML, bool CH = false>
__device__ __forceinline__ void h_quad_at(
    const SGeom &g, int i, int j, int k0, bool prev, const float *__restrict__ ex, const float *__restrict__ ey,
    const float *__restrict__ ez, const float *hxi, const float *hyi, const float *hzi, float *hxo, float *hyo,
    float *hzo, const SCpml &cp, const SAux &aux, const STfsf *tf = nullptr, float *prow = nullptr,
    const float *tv_row = nullptr, const int *tv = nullptr, const float *const *ch = nullptr)
{
    const int nx = g.nx, ny = g.ny, nzp = g.nzp, nz = g.nz;
    (void)nx;
    const size_t id = ((size_t)i * ny + j) * nzp + k0;
    const size_t sx = (size_t)ny * nzp;
    const bool jp = j > 0, ip = i > 0;
    const Q4 z4 = splat4(0.f);

    // ---------------------------------------------------------------- loads
    const Q4 ex0 = ld4(ex + id), ey0 = ld4(ey + id), ez0 = ld4(ez + id);
    Q4 h0 = ld4(hxi + id), h1 = ld4(hyi + id), h2 = ld4(hzi + id);
    const Q4 c0 = CH ? ld4(ch[0] + id) : splat4(0.5f);
    const Q4 c1 = CH ? ld4(ch[1] + id) : splat4(0.5f);
    const Q4 c2 = CH ? ld4(ch[2] + id) : splat4(0.5f);
    const Q4 ezD = jp ? ld4(ez + id - nzp) : z4;   // ez(j-1)
    const Q4 exD = jp ? ld4(ex + id - nzp) : z4;   // ex(j-1)
    const Q4 ezB = ip ? ld4(ez + id - sx) : z4;    // ez(i-1)
    const Q4 eyB = ip ? ld4(ey + id - sx) : z4;    // ey(i-1)
    // ey, ex at k0-1: the previous quad / previous row's end
    float eyp = 0.f, exp_ = 0.f;
    if (!prev) {
        if (jp) eyp = ey[id - 1];
        if (ip) exp_ = ex[id - 1];
    }

    const int npml = PML ? cp.npml : 0;
    int xs = 0, xp = 0, ys = 0, yp = 0, xt = -1, yt = -1;
    Q4 p1 = z4, p2 = z4;   // psi of the x face, or of the y face where there is no x face
    float pb = 0.f, pa = 0.f;
    size_t o1 = 0, o2 = 0;
    ZFace z;
    bool zq = false;
    if (PML) {
        xt = ip && (cp.axes & 1) ? sslab_h(i, nx, npml, xs, xp) : -1;  // plane 0 is the wall
        yt = jp && (cp.axes & 2) ? sslab_h(j, ny, npml, ys, yp) : -1;  // row 0 is the wall
        if (xt > 0 || yt > 0) {
            const size_t o = xt > 0 ? ((size_t)xp * ny + j) * nzp + k0 : ((size_t)i * npml + yp) * nzp + k0;
            const int f = xt > 0 ? xs : 2 + ys;
            const int t = xt > 0 ? xt : yt;
            o1 = cp.off(f, 0) + o;
            o2 = cp.off(f, 1) + o;
            p1 = ld4(cp.ph + o1);
            p2 = ld4(cp.ph + o2);
            pb = cp.bH[t];
            pa = cp.aH[t];
        }
        zq = (cp.axes & 4) && (k0 < npml || (k0 + 3 >= nz - npml && k0 < nz));
        if (zq) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                size_t o;
                const int t = zface_at<false>(cp, i, j, k0, l, ny, nz, o);
                z.load(l, t, cp.ph, o, cp.sZ, cp.bH, cp.aH);
            }
        }
    }

    // -------------------------------------------------------------- compute
    // hx: j>0 ; -= 0.5*((ez - ez[j-1]) - (ey - ey[k-1])) ; CPML - y psi2 (ez), + z psi1 (ey)
    // hy: i>0 ; -= 0.5*((ex - ex[k-1]) - (ez - ez[i-1])) ; CPML + x psi1 (ez), - z psi2 (ex)
    // hz: i, j>0 ; -= 0.5*((ey - ey[i-1]) - (ex - ex[j-1])) ; CPML - x psi2 (ey), + y psi1 (ex)
    const float y3 = lane_prev(ey0.v[3]), x3 = lane_prev(ex0.v[3]);  // every lane of the wave takes part
    if (prev) {
        eyp = y3;
        exp_ = x3;
    }
    float ym[4], xm[4];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        ym[l] = l > 0 ? ey0.v[l - 1] : eyp;
        xm[l] = l > 0 ? ex0.v[l - 1] : exp_;
    }
    if (jp) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float v = h0.v[l] - c0.v[l] * ((ez0.v[l] - ezD.v[l]) - (ey0.v[l] - ym[l]));
            const int k = k0 + l;
            h0.v[l] = (k > 0 && k < nz) ? v : v * 0.f;
        }
    }
    if (ip) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float v = h1.v[l] - c1.v[l] * ((ex0.v[l] - xm[l]) - (ez0.v[l] - ezB.v[l]));
            const int k = k0 + l;
            h1.v[l] = (k > 0 && k < nz) ? v : v * 0.f;
        }
    }
    if (ip && jp) {
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float v = h2.v[l] - c2.v[l] * ((ey0.v[l] - eyB.v[l]) - (ex0.v[l] - exD.v[l]));
            h2.v[l] = (k0 + l < nz) ? v : v * 0.f;
        }
    }
    if (PML) {
        if (xt > 0) {  // psi1: hy, psi2: hz
            const float b = pb, a = pa;
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int k = k0 + l;
                if (k > 0 && k < nz) {
                    const float tt = b * p1.v[l] + a * (ez0.v[l] - ezB.v[l]);
                    p1.v[l] = tt;
                    h1.v[l] = h1.v[l] + c1.v[l] * tt;
                }
            }
            if (jp) {
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (k0 + l < nz) {
                        const float tt = b * p2.v[l] + a * (ey0.v[l] - eyB.v[l]);
                        p2.v[l] = tt;
                        h2.v[l] = h2.v[l] - c2.v[l] * tt;
                    }
            }
            st4(cp.ph + o1, p1);
            st4(cp.ph + o2, p2);
        }
        if (yt > 0) {  // psi1: hz, psi2: hx
            if (xt > 0) {
                const size_t o = ((size_t)i * npml + yp) * nzp + k0;
                o1 = cp.off(2 + ys, 0) + o;
                o2 = cp.off(2 + ys, 1) + o;
                p1 = ld4(cp.ph + o1);
                p2 = ld4(cp.ph + o2);
                pb = cp.bH[yt];
                pa = cp.aH[yt];
            }
            const float b = pb, a = pa;
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int k = k0 + l;
                if (k > 0 && k < nz) {
                    const float tt = b * p2.v[l] + a * (ez0.v[l] - ezD.v[l]);
                    p2.v[l] = tt;
                    h0.v[l] = h0.v[l] - c0.v[l] * tt;
                }
            }
            if (ip) {
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (k0 + l < nz) {
                        const float tt = b * p1.v[l] + a * (ex0.v[l] - exD.v[l]);
                        p1.v[l] = tt;
                        h2.v[l] = h2.v[l] + c2.v[l] * tt;
                    }
            }
            st4(cp.ph + o1, p1);
            st4(cp.ph + o2, p2);
        }
        if (zq) {  // psi1: hx, psi2: hy
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                size_t o;
                const bool on = zface_at<false>(cp, i, j, k0, l, ny, nz, o) > 0;
                if (on && jp) {
                    const float tt = z.b[l] * z.q1[l] + z.a[l] * (ey0.v[l] - ym[l]);
                    cp.ph[o] = tt;
                    h0.v[l] = h0.v[l] + c0.v[l] * tt;
                }
                if (on && ip) {
                    const float tt = z.b[l] * z.q2[l] + z.a[l] * (ex0.v[l] - xm[l]);
                    cp.ph[o + cp.sZ] = tt;
                    h1.v[l] = h1.v[l] - c1.v[l] * tt;
                }
            }
        }
    }
    const bool near = aux.near(i, j, k0);
    if (near) {
        sapply_src(aux.src, 3, i, j, k0, h0, tv_row, tv);
        sapply_src(aux.src, 4, i, j, k0, h1, tv_row, tv);
        sapply_src(aux.src, 5, i, j, k0, h2, tv_row, tv);
    }
    if (tf) tfsf_quad(*tf, 3, i, j, k0, h0, h1, h2);

    // --------------------------------------------------------------- stores
    const bool all = hxo != hxi || near || tf;
    if (all || jp) st4(hxo + id, h0);
    if (all || ip) st4(hyo + id, h1);
    if (all || (ip && jp)) st4(hzo + id, h2);
    if (near) {
        sprobe(aux.prb, 3, i, j, k0, h0, prow);
        sprobe(aux.prb, 4, i, j, k0, h1, prow);
        sprobe(aux.prb, 5, i, j, k0, h2, prow);
    }
}

// Cells of this thread in the whole-grid passes; false for an idle thread.
struct RowAt {
    int i, j, k0;
    bool next, prev;
};

__device__ __forceinline__ bool slab_quad(const SGeom &g, unsigned b, RowAt &r)
{
    const QuadAt a = row_quad(g.m, b, threadIdx.x);
    const int lane = threadIdx.x & 63;
    r.i = g.i0 + a.i;
    r.j = a.j;
    r.k0 = 4 * a.q;
    r.next = a.next && lane < 63;
    r.prev = a.prev && lane > 0;
    return a.active;
}

struct SFields {
    float *e[6];
    const float *ce[3];
    const unsigned char *cm[3];  // CE as material indices (kCeTable), else NULL
    const float *lut;            // their 3 x 256 table
};

}  // namespace mifdtd
