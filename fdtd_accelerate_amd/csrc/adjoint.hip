// Discrete adjoint of the in-place Yee + CPML step (update_e, CPML-E, sources,
// update_h, CPML-H on the KEMP layout), for gradients of an objective with respect to
// the CE coefficients of a design box.
//
// The forward step n maps (E, H, psiE, psiH) -> (E', H', psiE', psiH'):
//   E half:  Ec = E + CE*(K H) on valid E cells, 0 on masked lanes, E on walls;
//            psiE' = b_E psiE + a_E (D H);  E' = Ec -/+ CE psiE'   (+ sources)
//   H half:  Hc = H - 0.5*(Kt E') on valid H cells, 0 on masked lanes, H on walls;
//            psiH' = b_H psiH + a_H (Dt E');  H' = Hc +/- 0.5 psiH'
// with K the forward-difference curl of update_e and Kt = K^T the backward-difference
// curl of update_h.  Its transpose, run backward in time from the adjoint state
// (lE, lH, lpsiE, lpsiH) of the step's outputs, is four passes:
//   A  (E-like): lE += dJ/dE' - 0.5*K(lH restricted to valid H) + Dt^T(a_H t_H),
//                t_H = lpsiH +/- 0.5*lH on valid H slab cells;  lH = 0 on masked H lanes
//   B:           lpsiH = b_H * t_H
//   C  (H-like): lH += Kt(CE * lE restricted to valid E) + D^T(a_E t_E),
//                t_E = lpsiE -/+ CE*lE on valid E slab cells;  grad_CE += lE * (K H_prev)
//                on the design box;  lE = 0 on masked E lanes
//   D:           lpsiE = b_E * t_E
// A and C gather from neighbours (a lane per quad of z cells), so every pass reads only
// values no thread of the same pass writes.  B only touches the cell's own lH / lpsiH, so it runs
// inside C (before C changes lH of that cell); D only touches the cell's own lE / lpsiE,
// so it is deferred into A of the next (earlier) step, before A changes lE of that cell
// (on the zero initial state it is a no-op).  Two launches per step.  Sources do not
// depend on the state (no adjoint).

#include "row_quads.hpp"
#include "step_quad.hpp"

namespace mifdtd {

constexpr int AB = 256;

struct AGeom {
    int nx, ny, nzp, nz, npml;
    unsigned long long ncell;
    size_t sX, sY, sZ;  // packed psi face sizes
    __device__ __forceinline__ size_t off(int f, int c) const
    {
        const int ax = f >> 1, sd = f & 1;
        if (ax == 0) return (size_t)(2 * sd + c) * sX;
        if (ax == 1) return 4 * sX + (size_t)(2 * sd + c) * sY;
        return 4 * sX + 4 * sY + (size_t)(2 * sd + c) * sZ;
    }
};

// Which cells the forward core writes (valid), zeroes (masked lanes) or leaves (walls).
__device__ __forceinline__ bool e_row(int c, int i, int j, int nx, int ny)
{
    return c == 0 ? j < ny - 1 : c == 1 ? i < nx - 1 : (i < nx - 1 && j < ny - 1);
}
__device__ __forceinline__ bool e_lane(int c, int k, int nz) { return c == 2 ? k < nz : k < nz - 1; }
__device__ __forceinline__ bool h_row(int c, int i, int j)
{
    return c == 0 ? j > 0 : c == 1 ? i > 0 : (i > 0 && j > 0);
}
__device__ __forceinline__ bool h_lane(int c, int k, int nz) { return c == 2 ? k < nz : (k > 0 && k < nz); }

__device__ __forceinline__ bool in_grid(int i, int j, int k, const AGeom &g)
{
    return i >= 0 && i < g.nx && j >= 0 && j < g.ny && k >= 0 && k < g.nzp;
}
__device__ __forceinline__ size_t cidx(int i, int j, int k, const AGeom &g)
{
    return ((size_t)i * g.ny + j) * g.nzp + k;
}
__device__ __forceinline__ bool valid_e(int c, int i, int j, int k, const AGeom &g)
{
    return in_grid(i, j, k, g) && e_row(c, i, j, g.nx, g.ny) && e_lane(c, k, g.nz);
}
// CPML slab lookup along one axis: returns the table entry (>0) of coordinate q, or -1,
// and the slab side / depth p.  E planes: front p -> p+1, back n-1-npml+p -> npml+1+p;
// H planes: front p -> p+1, back n-npml+p -> npml+2+p.
__device__ __forceinline__ int tab_e(int q, int n, int npml, int &sd, int &p)
{
    sd = 0;
    p = 0;
    if (q >= 0 && q < npml) { p = q; return p + 1; }
    if (q >= n - 1 - npml && q < n - 1) { sd = 1; p = q - (n - 1 - npml); return npml + 1 + p; }
    return -1;
}
__device__ __forceinline__ int tab_h(int q, int n, int npml, int &sd, int &p)
{
    sd = 0;
    p = 0;
    if (q >= 0 && q < npml) { p = q; return p + 1; }
    if (q >= n - npml && q < n) { sd = 1; p = q - (n - npml); return npml + 2 + p; }
    return -1;
}

// Reach of the CPML adjoint terms along one axis (coordinate q of n): pass A adds
// Dt^T(a_H t_H) at an E cell when q or q+1 is an H slab plane (q < npml or
// q >= n-npml-1), and pass D (inside A) acts on E slab planes, a subset; pass C adds
// D^T(a_E t_E) at an H cell when q-1 or q is an E slab plane (q <= npml or
// q >= n-1-npml), and pass B (inside C) acts on H slab planes, a subset.  Elsewhere
// those terms are zero and are not formed.
__device__ __forceinline__ bool near_a(int q, int n, int npml) { return q < npml || q >= n - npml - 1; }
__device__ __forceinline__ bool near_c(int q, int n, int npml) { return q <= npml || q >= n - 1 - npml; }

// packed psi index of cell (i, j, k) on face (axis, side) at depth p
__device__ __forceinline__ size_t psi_at(const AGeom &g, int axis, int sd, int p, int c, int i, int j, int k)
{
    const int f = 2 * axis + sd;
    size_t r;
    if (axis == 0) r = ((size_t)p * g.ny + j) * g.nzp + k;
    else if (axis == 1) r = ((size_t)i * g.npml + p) * g.nzp + k;
    else r = ((size_t)i * g.ny + j) * g.npml + p;
    return g.off(f, c) + r;
}

// ------------------------------------------------------------------ the two passes
// One lane per quad of 4 z cells in the whole-grid passes' thread order (row_quads.hpp:
// a stripe of every plane per XCD, z-slab quads in waves of their own).  A quad's
// neighbour rows, planes and cells are loaded (or taken from the next lane) once and serve
// the curl and the CPML terms of all three axes; the psi of an axis is loaded only by the
// rows and quads it reaches.  With a thread per cell the passes ran 7 scalar gathers per
// component and re-derived every neighbour's validity: 160^3 cells, CPML 10, 75.5 + 110.6
// us; now 39.4 + 52.1 (84 B per cell and step and the psi, at 4.9-5.2 TB/s).
__device__ __forceinline__ Q4 keep_cells(const Q4 &q, int k0, int lo, int hi)  // lanes lo <= k < hi, else 0
{
    Q4 r;
#pragma unroll
    for (int l = 0; l < 4; ++l) r.v[l] = (k0 + l >= lo && k0 + l < hi) ? q.v[l] : 0.f;
    return r;
}

__device__ __forceinline__ Q4 scale4(const float *__restrict__ ce, size_t id, const Q4 &q)
{
    const Q4 c = ce ? ld4u(ce + id) : splat4(0.5f);
    Q4 r;
#pragma unroll
    for (int l = 0; l < 4; ++l) r.v[l] = c.v[l] * q.v[l];
    return r;
}

// H (E) slab entry and psi offset of coordinate q along an axis; t <= 0: not in a slab.
struct Entry {
    int t;
    size_t o1, o2;  // psi1, psi2 of cell (i, j, k) (x, y faces: of the quad's first cell)
};

template <bool E>
__device__ __forceinline__ Entry entry(const AGeom &g, int axis, int q, int i, int j, int k)
{
    const int n = axis == 0 ? g.nx : axis == 1 ? g.ny : g.nz;
    int sd, p;
    Entry e;
    e.t = E ? tab_e(q, n, g.npml, sd, p) : tab_h(q, n, g.npml, sd, p);
    e.o1 = e.o2 = 0;
    if (e.t > 0) {
        e.o1 = psi_at(g, axis, sd, p, 0, i, j, k);
        e.o2 = psi_at(g, axis, sd, p, 1, i, j, k);
    }
    return e;
}

// psi' = b * (psi + s) of one face's quad: s1, s2 the terms, c1, c2 the cells [lo, hi) they hold.
__device__ __forceinline__ void psi_step(float *lp, const Entry &e, float b, bool row1, const Q4 &s1, int lo1, int hi1,
                                         bool row2, const Q4 &s2, int lo2, int hi2, int k0, const Q4 &q1, const Q4 &q2)
{
    Q4 r1 = q1, r2 = q2;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int k = k0 + l;
        if (row1 && k >= lo1 && k < hi1) r1.v[l] = b * (q1.v[l] + s1.v[l]);
        if (row2 && k >= lo2 && k < hi2) r2.v[l] = b * (q2.v[l] + s2.v[l]);
    }
    st4u(lp + e.o1, r1);
    st4u(lp + e.o2, r2);
}

__device__ __forceinline__ Q4 neg4(const Q4 &q)
{
    return Q4{{-q.v[0], -q.v[1], -q.v[2], -q.v[3]}};
}
__device__ __forceinline__ Q4 half4(const Q4 &q, float s)
{
    return Q4{{s * q.v[0], s * q.v[1], s * q.v[2], s * q.v[3]}};
}

// a * (psi + s) on the cells [lo, hi) of a valid row in the slab, else 0.
__device__ __forceinline__ Q4 psi_term(bool on, float a, const Q4 &psi, const Q4 &s, int k0, int lo, int hi)
{
    Q4 r;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int k = k0 + l;
        r.v[l] = on && k >= lo && k < hi ? a * (psi.v[l] + s.v[l]) : 0.f;
    }
    return r;
}

__device__ __forceinline__ void add_diff(Q4 &v, const Q4 &p, const Q4 &m)
{
#pragma unroll
    for (int l = 0; l < 4; ++l) v.v[l] += p.v[l] - m.v[l];
}

__device__ __forceinline__ Q4 psi_ld(bool on, const float *lp, size_t o) { return on ? ld4u(lp + o) : splat4(0.f); }

// psi1, psi2 and the table entry of a z-face cell (entry e; what e.t <= 0 loads is not used).
// All cells' loads go ahead of the block's psi stores: a load that follows the previous
// cell's store is a memory round trip of its own, and at 160 cells a row 2 of 5 waves are
// z-slab waves (passes A + C 43.6 + 58.6 -> 39.4 + 52.1 us).  Pass A keeps 4 waves per SIMD
// at 12 bytes of spill (130 VGPRs without).
struct ZPsi {
    float q1, q2, c;
};
__device__ __forceinline__ ZPsi z_psi(const Entry &e, const float *lp, const float *tab)
{
    return ZPsi{lp[e.o1], lp[e.o2], tab[e.t > 0 ? e.t : 0]};
}

// Pass A (and D of the later step) on one quad.
__global__ __launch_bounds__(AB) __attribute__((amdgpu_waves_per_eu(4))) void k_adj_a(AGeom g, RowQuads m, float *__restrict__ lex, float *__restrict__ ley,
                                              float *__restrict__ lez, float *__restrict__ lhx,
                                              float *__restrict__ lhy, float *__restrict__ lhz,
                                              const float *__restrict__ lpH, const float *__restrict__ aH,
                                              const float *__restrict__ eplane, int iplane,
                                              const float *__restrict__ cex, const float *__restrict__ cey,
                                              const float *__restrict__ cez, float *__restrict__ lpE,
                                              const float *__restrict__ bE)
{
    const QuadAt at = row_quad(m, blockIdx.x, threadIdx.x);
    if (!at.active) return;
    const int i = at.i, j = at.j, k0 = 4 * at.q;
    const bool next = at.next && (threadIdx.x & 63) < 63;
    const int nz = g.nz;
    const size_t id = cidx(i, j, k0, g), sj = (size_t)g.nzp, si = (size_t)g.ny * g.nzp;
    const bool ip = i > 0, jp = j > 0, ix = i + 1 < g.nx, jy = j + 1 < g.ny;
    const Q4 z4 = splat4(0.f);
    // H valid cells: hx rows j > 0, hy planes i > 0 (0 < k < nz); hz i, j > 0 (k < nz)
    const Q4 hx0 = jp ? keep_cells(ld4u(lhx + id), k0, 1, nz) : z4;
    const Q4 hy0 = ip ? keep_cells(ld4u(lhy + id), k0, 1, nz) : z4;
    const Q4 hz0 = ip && jp ? keep_cells(ld4u(lhz + id), k0, 0, nz) : z4;
    const Q4 hxU = jy ? keep_cells(ld4u(lhx + id + sj), k0, 1, nz) : z4;
    const Q4 hzU = jy && ip ? keep_cells(ld4u(lhz + id + sj), k0, 0, nz) : z4;
    const Q4 hyN = ix ? keep_cells(ld4u(lhy + id + si), k0, 1, nz) : z4;
    const Q4 hzN = ix && jp ? keep_cells(ld4u(lhz + id + si), k0, 0, nz) : z4;
    Q4 vx = ld4u(lex + id), vy = ld4u(ley + id), vz = ld4u(lez + id);
    float hx4 = 0.f, hy4 = 0.f;  // at k0 + 4
    if (!next && k0 + 4 < nz) {
        if (jp) hx4 = lhx[id + 4];
        if (ip) hy4 = lhy[id + 4];
    }
    const float hxs = lane_next(hx0.v[0]), hys = lane_next(hy0.v[0]);  // every lane takes part
    if (next) {
        hx4 = hxs;
        hy4 = hys;
    }
    const bool nx_ = g.npml > 0 && near_a(i, g.nx, g.npml), ny_ = g.npml > 0 && near_a(j, g.ny, g.npml),
               nz_ = g.npml > 0 && (k0 < g.npml || k0 + 3 >= nz - g.npml - 1);
    const Q4 ex0 = vx, ey0 = vy, ez0 = vz;
    // -0.5*K(lH valid):  ex: (z[j+1]-z) - (y[k+1]-y);  ey: (x[k+1]-x) - (z[i+1]-z);
    //                     ez: (y[i+1]-y) - (x[j+1]-x)
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const float y1 = l < 3 ? hy0.v[l + 1] : hy4, x1 = l < 3 ? hx0.v[l + 1] : hx4;
        vx.v[l] = vx.v[l] - 0.5f * ((hzU.v[l] - hz0.v[l]) - (y1 - hy0.v[l]));
        vy.v[l] = vy.v[l] - 0.5f * ((x1 - hx0.v[l]) - (hzN.v[l] - hz0.v[l]));
        vz.v[l] = vz.v[l] - 0.5f * ((hyN.v[l] - hy0.v[l]) - (hxU.v[l] - hx0.v[l]));
    }
    if (nx_) {
        const Entry d = entry<true>(g, 0, i, i, j, k0), t0 = entry<false>(g, 0, i, i, j, k0),
                    t1 = entry<false>(g, 0, i + 1, i + 1, j, k0);
        const bool on0 = t0.t > 0 && ip, on1 = t1.t > 0 && ix;
        const Q4 q1 = psi_ld(d.t > 0, lpE, d.o1), q2 = psi_ld(d.t > 0, lpE, d.o2);
        const Q4 r1 = psi_ld(on0, lpH, t0.o1), r2 = psi_ld(on0, lpH, t0.o2);
        const Q4 s1 = psi_ld(on1, lpH, t1.o1), s2 = psi_ld(on1, lpH, t1.o2);
        if (d.t > 0)  // D: psi1 ey (-), psi2 ez (+)
            psi_step(lpE, d, bE[d.t], true, neg4(scale4(cey, id, ey0)), 0, nz - 1, jy, scale4(cez, id, ez0), 0, nz, k0,
                     q1, q2);
        const float a0 = on0 ? aH[t0.t] : 0.f, a1 = on1 ? aH[t1.t] : 0.f;
        // psi1 -> hy from ez (+), psi2 -> hz from ey (-)
        add_diff(vz, psi_term(on0, a0, r1, half4(hy0, 0.5f), k0, 1, nz), psi_term(on1, a1, s1, half4(hyN, 0.5f), k0, 1, nz));
        add_diff(vy, psi_term(on0 && jp, a0, r2, half4(hz0, -0.5f), k0, 0, nz),
                 psi_term(on1 && jp, a1, s2, half4(hzN, -0.5f), k0, 0, nz));
    }
    if (ny_) {
        const Entry d = entry<true>(g, 1, j, i, j, k0), t0 = entry<false>(g, 1, j, i, j, k0),
                    t1 = entry<false>(g, 1, j + 1, i, j + 1, k0);
        const bool on0 = t0.t > 0 && jp, on1 = t1.t > 0 && jy;
        const Q4 q1 = psi_ld(d.t > 0, lpE, d.o1), q2 = psi_ld(d.t > 0, lpE, d.o2);
        const Q4 r1 = psi_ld(on0, lpH, t0.o1), r2 = psi_ld(on0, lpH, t0.o2);
        const Q4 s1 = psi_ld(on1, lpH, t1.o1), s2 = psi_ld(on1, lpH, t1.o2);
        if (d.t > 0)  // D: psi1 ez (-), psi2 ex (+)
            psi_step(lpE, d, bE[d.t], ix, neg4(scale4(cez, id, ez0)), 0, nz, true, scale4(cex, id, ex0), 0, nz - 1, k0,
                     q1, q2);
        const float a0 = on0 ? aH[t0.t] : 0.f, a1 = on1 ? aH[t1.t] : 0.f;
        // psi1 -> hz from ex (+), psi2 -> hx from ez (-)
        add_diff(vx, psi_term(on0 && ip, a0, r1, half4(hz0, 0.5f), k0, 0, nz),
                 psi_term(on1 && ip, a1, s1, half4(hzU, 0.5f), k0, 0, nz));
        add_diff(vz, psi_term(on0, a0, r2, half4(hx0, -0.5f), k0, 1, nz), psi_term(on1, a1, s2, half4(hxU, -0.5f), k0, 1, nz));
    }
    if (nz_) {
        // D: psi1 ex (-), psi2 ey (+)
        ZPsi zd[4], zt[5];
#pragma unroll
        for (int l = 0; l < 4; ++l) zd[l] = z_psi(entry<true>(g, 2, k0 + l, i, j, k0 + l), lpE, bE);
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            const int kk = k0 + l < g.nzp ? k0 + l : 0;
            zt[l] = z_psi(entry<false>(g, 2, kk, i, j, kk), lpH, aH);
        }
        const Q4 gx = scale4(cex, id, ex0), gy = scale4(cey, id, ey0);
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const Entry d = entry<true>(g, 2, k0 + l, i, j, k0 + l);
            if (d.t > 0) {
                if (jy) lpE[d.o1] = zd[l].c * (zd[l].q1 - gx.v[l]);
                if (ix) lpE[d.o2] = zd[l].c * (zd[l].q2 + gy.v[l]);
            }
        }
        // a t of cells k0 .. k0+4: psi1 -> hx from ey (+), psi2 -> hy from ex (-)
        float t1[5], t2[5];
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            const int k = k0 + l;
            t1[l] = t2[l] = 0.f;
            const int kk = k < g.nzp ? k : 0;
            const Entry t = entry<false>(g, 2, kk, i, j, kk);
            if (k > 0 && k < nz && t.t > 0) {
                if (jp) t1[l] = zt[l].c * (zt[l].q1 + 0.5f * (l < 4 ? hx0.v[l & 3] : hx4));
                if (ip) t2[l] = zt[l].c * (zt[l].q2 - 0.5f * (l < 4 ? hy0.v[l & 3] : hy4));
            }
        }
#pragma unroll
        for (int l = 0; l < 4; ++l)
            if (near_a(k0 + l, nz, g.npml)) {
                vy.v[l] += t1[l] - t1[l + 1];
                vx.v[l] += t2[l] - t2[l + 1];
            }
    }
    if (eplane && i == iplane) {
        const size_t pid = (size_t)j * g.nzp + k0, ps = (size_t)g.ny * g.nzp;
        const Q4 px = ld4u(eplane + pid), py = ld4u(eplane + ps + pid), pz = ld4u(eplane + 2 * ps + pid);
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            vx.v[l] += 2.f * px.v[l];
            vy.v[l] += 2.f * py.v[l];
            vz.v[l] += 2.f * pz.v[l];
        }
    }
    st4u(lex + id, vx);
    st4u(ley + id, vy);
    st4u(lez + id, vz);
    // H masked lanes: H' does not depend on H there
    if (k0 == 0 || k0 + 3 >= nz) {
#pragma unroll
        for (int l = 0; l < 4; ++l)
            for (int c = 0; c < 3; ++c)
                if (h_row(c, i, j) && !h_lane(c, k0 + l, nz)) (c == 0 ? lhx : c == 1 ? lhy : lhz)[id + l] = 0.f;
    }
}

struct ADesign {
    int i0, j0, k0, di, dj, dk;  // box origin and extent
    const float *curl;           // (3, di, dj, dk) curl of H_prev for this step
    double *grad;                // (3, di, dj, dk) accumulated dJ/dCE
};

struct __attribute__((packed, aligned(8))) D2u {  // two doubles at any 8-byte aligned address
    double x, y;
};

// grad += lE * curl of one component on the quad's cells inside the box (q: box index of
// the quad's first cell).
__device__ __forceinline__ void grad_quad(const ADesign &dz, size_t q, int dk, const Q4 &e, int k0, int hi)
{
    if (dk >= 0 && dk + 3 < dz.dk && k0 + 3 < hi && (q & 3u) == 0) {
        const Q4 c = ld4u(dz.curl + q);
        D2u *p = reinterpret_cast<D2u *>(dz.grad + q);
        D2u a = p[0], b = p[1];
        a.x += (double)e.v[0] * (double)c.v[0];
        a.y += (double)e.v[1] * (double)c.v[1];
        b.x += (double)e.v[2] * (double)c.v[2];
        b.y += (double)e.v[3] * (double)c.v[3];
        p[0] = a;
        p[1] = b;
        return;
    }
#pragma unroll
    for (int l = 0; l < 4; ++l)
        if (dk + l >= 0 && dk + l < dz.dk && k0 + l < hi) dz.grad[q + l] += (double)e.v[l] * (double)dz.curl[q + l];
}

// Pass C (and B) on one quad.
__global__ __launch_bounds__(AB) void k_adj_c(AGeom g, RowQuads m, float *__restrict__ lex, float *__restrict__ ley,
                                              float *__restrict__ lez, float *__restrict__ lhx,
                                              float *__restrict__ lhy, float *__restrict__ lhz,
                                              const float *__restrict__ cex, const float *__restrict__ cey,
                                              const float *__restrict__ cez, const float *__restrict__ lpE,
                                              const float *__restrict__ aE, ADesign dz,
                                              float *__restrict__ lpH, const float *__restrict__ bH)
{
    const QuadAt at = row_quad(m, blockIdx.x, threadIdx.x);
    if (!at.active) return;
    const int i = at.i, j = at.j, k0 = 4 * at.q;
    const bool prev = at.prev && (threadIdx.x & 63) > 0;
    const int nz = g.nz;
    const size_t id = cidx(i, j, k0, g), sj = (size_t)g.nzp, si = (size_t)g.ny * g.nzp;
    const bool ip = i > 0, jp = j > 0, ix = i + 1 < g.nx, jy = j + 1 < g.ny;
    const Q4 z4 = splat4(0.f);
    const Q4 ex0 = ld4u(lex + id), ey0 = ld4u(ley + id), ez0 = ld4u(lez + id);
    Q4 vx = ld4u(lhx + id), vy = ld4u(lhy + id), vz = ld4u(lhz + id);
    // CE*lE on valid E cells: ex rows j < ny-1, ey planes i < nx-1 (k < nz-1); ez both (k < nz)
    const Q4 gx0 = jy ? keep_cells(scale4(cex, id, ex0), k0, 0, nz - 1) : z4;
    const Q4 gy0 = ix ? keep_cells(scale4(cey, id, ey0), k0, 0, nz - 1) : z4;
    const Q4 gz0 = ix && jy ? keep_cells(scale4(cez, id, ez0), k0, 0, nz) : z4;
    const Q4 gxD = jp ? keep_cells(scale4(cex, id - sj, ld4u(lex + id - sj)), k0, 0, nz - 1) : z4;
    const Q4 gzD = jp && ix ? keep_cells(scale4(cez, id - sj, ld4u(lez + id - sj)), k0, 0, nz) : z4;
    const Q4 gyB = ip ? keep_cells(scale4(cey, id - si, ld4u(ley + id - si)), k0, 0, nz - 1) : z4;
    const Q4 gzB = ip && jy ? keep_cells(scale4(cez, id - si, ld4u(lez + id - si)), k0, 0, nz) : z4;
    float gxm = 0.f, gym = 0.f;  // at k0 - 1
    if (!prev && k0 > 0 && k0 - 1 < nz - 1) {
        if (jy) gxm = (cex ? cex[id - 1] : 0.5f) * lex[id - 1];
        if (ix) gym = (cey ? cey[id - 1] : 0.5f) * ley[id - 1];
    }
    const float gxs = lane_prev(gx0.v[3]), gys = lane_prev(gy0.v[3]);  // every lane takes part
    if (prev) {
        gxm = gxs;
        gym = gys;
    }
    const bool nx_ = g.npml > 0 && near_c(i, g.nx, g.npml), ny_ = g.npml > 0 && near_c(j, g.ny, g.npml),
               nz_ = g.npml > 0 && (k0 <= g.npml || k0 + 3 >= nz - 1 - g.npml);
    const Q4 hx0 = vx, hy0 = vy, hz0 = vz;
    // Kt(CE*lE valid): hx: (z - z[j-1]) - (y - y[k-1]); hy: (x - x[k-1]) - (z - z[i-1]);
    //                  hz: (y - y[i-1]) - (x - x[j-1])
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const float xm = l > 0 ? gx0.v[l - 1] : gxm, ym = l > 0 ? gy0.v[l - 1] : gym;
        vx.v[l] = vx.v[l] + ((gz0.v[l] - gzD.v[l]) - (gy0.v[l] - ym));
        vy.v[l] = vy.v[l] + ((gx0.v[l] - xm) - (gz0.v[l] - gzB.v[l]));
        vz.v[l] = vz.v[l] + ((gy0.v[l] - gyB.v[l]) - (gx0.v[l] - gxD.v[l]));
    }
    if (nx_) {
        const Entry d = entry<false>(g, 0, i, i, j, k0), tm = entry<true>(g, 0, i - 1, i - 1, j, k0),
                    t0 = entry<true>(g, 0, i, i, j, k0);
        const bool on = d.t > 0 && ip, onm = tm.t > 0, on0 = t0.t > 0;
        const Q4 q1 = psi_ld(on, lpH, d.o1), q2 = psi_ld(on, lpH, d.o2);
        const Q4 r1 = psi_ld(onm, lpE, tm.o1), r2 = psi_ld(onm, lpE, tm.o2);
        const Q4 s1 = psi_ld(on0, lpE, t0.o1), s2 = psi_ld(on0, lpE, t0.o2);
        if (on)  // B: psi1 hy (+), psi2 hz (-)
            psi_step(lpH, d, bH[d.t], true, half4(hy0, 0.5f), 1, nz, jp, half4(hz0, -0.5f), 0, nz, k0, q1, q2);
        const float am = onm ? aE[tm.t] : 0.f, a0 = on0 ? aE[t0.t] : 0.f;
        // psi1 -> ey from hz (-CE), psi2 -> ez from hy (+CE)
        add_diff(vz, psi_term(onm, am, r1, neg4(gyB), k0, 0, nz - 1), psi_term(on0, a0, s1, neg4(gy0), k0, 0, nz - 1));
        add_diff(vy, psi_term(onm && jy, am, r2, gzB, k0, 0, nz), psi_term(on0 && jy, a0, s2, gz0, k0, 0, nz));
    }
    if (ny_) {
        const Entry d = entry<false>(g, 1, j, i, j, k0), tm = entry<true>(g, 1, j - 1, i, j - 1, k0),
                    t0 = entry<true>(g, 1, j, i, j, k0);
        const bool on = d.t > 0 && jp, onm = tm.t > 0, on0 = t0.t > 0;
        const Q4 q1 = psi_ld(on, lpH, d.o1), q2 = psi_ld(on, lpH, d.o2);
        const Q4 r1 = psi_ld(onm, lpE, tm.o1), r2 = psi_ld(onm, lpE, tm.o2);
        const Q4 s1 = psi_ld(on0, lpE, t0.o1), s2 = psi_ld(on0, lpE, t0.o2);
        if (on)  // B: psi1 hz (+), psi2 hx (-)
            psi_step(lpH, d, bH[d.t], ip, half4(hz0, 0.5f), 0, nz, true, half4(hx0, -0.5f), 1, nz, k0, q1, q2);
        const float am = onm ? aE[tm.t] : 0.f, a0 = on0 ? aE[t0.t] : 0.f;
        // psi1 -> ez from hx (-), psi2 -> ex from hz (+)
        add_diff(vx, psi_term(onm && ix, am, r1, neg4(gzD), k0, 0, nz), psi_term(on0 && ix, a0, s1, neg4(gz0), k0, 0, nz));
        add_diff(vz, psi_term(onm, am, r2, gxD, k0, 0, nz - 1), psi_term(on0, a0, s2, gx0, k0, 0, nz - 1));
    }
    if (nz_) {
        // B: psi1 hx (+), psi2 hy (-)
        ZPsi zd[4], zt[5];
#pragma unroll
        for (int l = 0; l < 4; ++l) zd[l] = z_psi(entry<false>(g, 2, k0 + l, i, j, k0 + l), lpH, bH);
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            const int kk = k0 - 1 + l > 0 ? k0 - 1 + l : 0;
            zt[l] = z_psi(entry<true>(g, 2, kk, i, j, kk), lpE, aE);
        }
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const int k = k0 + l;
            const Entry d = entry<false>(g, 2, k, i, j, k);
            if (d.t > 0 && k > 0) {
                if (jp) lpH[d.o1] = zd[l].c * (zd[l].q1 + 0.5f * hx0.v[l]);
                if (ip) lpH[d.o2] = zd[l].c * (zd[l].q2 - 0.5f * hy0.v[l]);
            }
        }
        // a t of cells k0-1 .. k0+3: psi1 -> ex from hy (-), psi2 -> ey from hx (+)
        float t1[5], t2[5];
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            const int k = k0 - 1 + l;
            t1[l] = t2[l] = 0.f;
            const int kk = k > 0 ? k : 0;
            const Entry t = entry<true>(g, 2, kk, i, j, kk);
            if (k >= 0 && k < nz - 1 && t.t > 0) {
                if (jy) t1[l] = zt[l].c * (zt[l].q1 - (l > 0 ? gx0.v[(l + 3) & 3] : gxm));
                if (ix) t2[l] = zt[l].c * (zt[l].q2 + (l > 0 ? gy0.v[(l + 3) & 3] : gym));
            }
        }
#pragma unroll
        for (int l = 0; l < 4; ++l)
            if (near_c(k0 + l, nz, g.npml)) {
                vy.v[l] += t1[l] - t1[l + 1];
                vx.v[l] += t2[l] - t2[l + 1];
            }
    }
    st4u(lhx + id, vx);
    st4u(lhy + id, vy);
    st4u(lhz + id, vz);
    // gradient of the CE of the design box: lE * (K H_prev)
    const int di = i - dz.i0, dj = j - dz.j0, dk = k0 - dz.k0;
    if (dz.grad && di >= 0 && di < dz.di && dj >= 0 && dj < dz.dj && dk + 3 >= 0 && dk < dz.dk) {
        const size_t q = (((size_t)di * dz.dj + dj) * dz.dk) + dk;  // dk may be -3..-1: cells before the box are skipped
        const size_t s = (size_t)dz.di * dz.dj * dz.dk;
        if (jy) grad_quad(dz, q, dk, ex0, k0, nz - 1);
        if (ix) grad_quad(dz, q + s, dk, ey0, k0, nz - 1);
        if (ix && jy) grad_quad(dz, q + 2 * s, dk, ez0, k0, nz);
    }
    // E masked lanes: E' does not depend on E there
    if (k0 + 3 >= nz - 1) {
#pragma unroll
        for (int l = 0; l < 4; ++l)
            for (int c = 0; c < 3; ++c)
                if (e_row(c, i, j, g.nx, g.ny) && !e_lane(c, k0 + l, nz)) (c == 0 ? lex : c == 1 ? ley : lez)[id + l] = 0.f;
    }
}

// curl of H at the E points of the design box, as update_e forms it:
//   ex: (hz[j+1]-hz) - (hy[k+1]-hy);  ey: (hx[k+1]-hx) - (hz[i+1]-hz);  ez: (hy[i+1]-hy) - (hx[j+1]-hx)
__global__ __launch_bounds__(AB) void k_design_curl(AGeom g, ADesign dz, const float *__restrict__ hx,
                                                    const float *__restrict__ hy, const float *__restrict__ hz,
                                                    float *__restrict__ out)
{
    const unsigned long long s = (unsigned long long)dz.di * dz.dj * dz.dk;
    const unsigned long long n = (unsigned long long)blockIdx.x * AB + threadIdx.x;
    if (n >= s) return;
    const int dk = (int)(n % (unsigned long long)dz.dk);
    const unsigned long long r = n / (unsigned long long)dz.dk;
    const int dj = (int)(r % (unsigned long long)dz.dj);
    const int di = (int)(r / (unsigned long long)dz.dj);
    const int i = dz.i0 + di, j = dz.j0 + dj, k = dz.k0 + dk;
    const size_t id = cidx(i, j, k, g), sj = (size_t)g.nzp, si = (size_t)g.ny * g.nzp;
    out[n] = valid_e(0, i, j, k, g) ? (hz[id + sj] - hz[id]) - (hy[id + 1] - hy[id]) : 0.f;
    out[s + n] = valid_e(1, i, j, k, g) ? (hx[id + 1] - hx[id]) - (hz[id + si] - hz[id]) : 0.f;
    out[2 * s + n] = valid_e(2, i, j, k, g) ? (hy[id + si] - hy[id]) - (hx[id + sj] - hx[id]) : 0.f;
}

static int adj_geom(AGeom &g, int nx, int ny, int nzp, int pad, int npml)
{
    if (int rc = check_grid(nx, ny, nzp, pad)) return rc;
    g.nx = nx;
    g.ny = ny;
    g.nzp = nzp;
    g.nz = nzp - pad;
    g.npml = npml;
    if (npml < 0 || npml > MIFDTD_MAX_NPML) return fail(MIFDTD_EINVAL, "npml %d", npml);
    if (npml && (nx < 2 * npml + 2 || ny < 2 * npml + 2 || g.nz < 2 * npml + 2))
        return fail(MIFDTD_EINVAL, "grid too small for npml %d", npml);
    g.ncell = (unsigned long long)nx * ny * nzp;
    g.sX = (size_t)npml * ny * nzp;
    g.sY = (size_t)nx * npml * nzp;
    g.sZ = (size_t)nx * ny * npml;
    return 0;
}

static int check_box(const AGeom &g, const mifdtd_design_box *d)
{
    if (!d) return fail(MIFDTD_ENULL, "design box is NULL");
    if (d->i0 < 0 || d->j0 < 0 || d->k0 < 0 || d->di < 1 || d->dj < 1 || d->dk < 1 || d->i0 + d->di > g.nx ||
        d->j0 + d->dj > g.ny || d->k0 + d->dk > g.nz)
        return fail(MIFDTD_EINVAL, "design box outside the grid");
    // The gradient accumulates dE'/dCE = K H only: an E cell of a CPML slab also carries
    // the -/+CE*psi term, whose derivative is not formed, so the box must keep off every
    // E slab plane (front [0, npml), back [n-1-npml, n-1) on each axis).
    if (g.npml > 0) {
        const int np_ = g.npml;
        if (d->i0 < np_ || d->j0 < np_ || d->k0 < np_ || d->i0 + d->di > g.nx - 1 - np_ ||
            d->j0 + d->dj > g.ny - 1 - np_ || d->k0 + d->dk > g.nz - 1 - np_)
            return fail(MIFDTD_EINVAL, "design box (%d,%d,%d)+(%d,%d,%d) overlaps a CPML slab (npml %d)", d->i0, d->j0,
                        d->k0, d->di, d->dj, d->dk, np_);
    }
    return 0;
}

}  // namespace mifdtd

using namespace mifdtd;

extern "C" {

int mifdtd_adjoint_step(int nx, int ny, int nz_pitch, int pad, float *const lam[6], const float *const ce[3],
                        int npml, float *lpsiE, float *lpsiH, const float *bE, const float *aE, const float *bH,
                        const float *aH, const float *eplane, int iplane, const mifdtd_design_box *box,
                        const float *curl, double *grad, mifdtd_stream_t stream)
{
    AGeom g;
    if (int rc = adj_geom(g, nx, ny, nz_pitch, pad, npml)) return rc;
    if (!lam) return fail(MIFDTD_ENULL, "adjoint fields NULL");
    for (int c = 0; c < 6; c++)
        if (!lam[c]) return fail(MIFDTD_ENULL, "adjoint field %d NULL", c);
    const float *c0 = ce ? ce[0] : nullptr, *c1 = ce ? ce[1] : nullptr, *c2 = ce ? ce[2] : nullptr;
    if ((c0 || c1 || c2) && !(c0 && c1 && c2)) return fail(MIFDTD_ENULL, "CE arrays all set or all NULL");
    if (npml && (!lpsiE || !lpsiH || !bE || !aE || !bH || !aH)) return fail(MIFDTD_ENULL, "CPML adjoint buffers NULL");
    if (eplane && (iplane < 0 || iplane >= nx)) return fail(MIFDTD_EINVAL, "monitor plane %d outside the grid", iplane);
    ADesign dz{};
    if (grad) {
        if (int rc = check_box(g, box)) return rc;
        if (!curl) return fail(MIFDTD_ENULL, "curl buffer NULL");
        dz.i0 = box->i0;
        dz.j0 = box->j0;
        dz.k0 = box->k0;
        dz.di = box->di;
        dz.dj = box->dj;
        dz.dk = box->dk;
        dz.curl = curl;
        dz.grad = grad;
    }
    if (g.ncell > 0xffffffffull - AB) return fail(MIFDTD_ERANGE, "grid of %llu cells: at most 2^32 - %d", g.ncell, AB);
    const RowQuads m = row_quads((unsigned)nx, (unsigned)ny, (unsigned)(nz_pitch / 4), g.nz, npml, npml + 1);
    const unsigned grid = (unsigned)row_quads_blocks(m);
    hipStream_t st = to_stream(stream);
    k_adj_a<<<grid, AB, 0, st>>>(g, m, lam[0], lam[1], lam[2], lam[3], lam[4], lam[5], lpsiH, aH, eplane, iplane, c0, c1,
                                 c2, lpsiE, bE);
    MIFDTD_CHECK_LAUNCH("adjoint pass A");
    k_adj_c<<<grid, AB, 0, st>>>(g, m, lam[0], lam[1], lam[2], lam[3], lam[4], lam[5], c0, c1, c2, lpsiE, aE, dz, lpsiH,
                                 bH);
    MIFDTD_CHECK_LAUNCH("adjoint pass C");
    return 0;
}

int mifdtd_design_curl(int nx, int ny, int nz_pitch, int pad, const float *hx, const float *hy, const float *hz,
                       const mifdtd_design_box *box, float *out, mifdtd_stream_t stream)
{
    AGeom g;
    if (int rc = adj_geom(g, nx, ny, nz_pitch, pad, 0)) return rc;
    if (int rc = check_box(g, box)) return rc;
    if (!hx || !hy || !hz || !out) return fail(MIFDTD_ENULL, "NULL pointer");
    // neighbours i+1, j+1, k+1 of the box must exist
    if (box->i0 + box->di >= nx || box->j0 + box->dj >= ny || box->k0 + box->dk >= nz_pitch)
        return fail(MIFDTD_EINVAL, "design box touches the upper grid edge");
    ADesign dz{};
    dz.i0 = box->i0;
    dz.j0 = box->j0;
    dz.k0 = box->k0;
    dz.di = box->di;
    dz.dj = box->dj;
    dz.dk = box->dk;
    const unsigned long long s = (unsigned long long)box->di * box->dj * box->dk;
    const unsigned grid = (unsigned)((s + AB - 1) / AB);
    k_design_curl<<<grid, AB, 0, to_stream(stream)>>>(g, dz, hx, hy, hz, out);
    MIFDTD_CHECK_LAUNCH("design curl");
    return 0;
}

}  // extern "C"
