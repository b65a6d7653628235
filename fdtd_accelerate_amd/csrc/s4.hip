// 4th-order symplectic FDTD: the stage updates of S4/Python-C/dielectric.c (H :5-49,
// E :52-96; the same arithmetic as the CUDA kernels of S4/PyCUDA/100-base.py:10-44) and
// a CPML for it, on the reference's layout: (nx, ny, nz) Fortran order, x contiguous,
// no padding.
//
// A lane per x-quad (4 consecutive x cells of one (j, k) row; nx must be a multiple of
// 4).  Per-cell arithmetic keeps the reference's
// evaluation order:
//   H: h -= (cl*ch) * (27*(((a0 - a1) - b0) + b1) - (((a2 - a3) - b2) + b3))
//   E: e += (dl*ce) * (27*(((a0 - a1) - b0) + b1) - (((a2 - a3) - b2) + b3))
// so that with -ffp-contract=off the result equals the reference C bit for bit.
// Guards (which cells each stage writes) follow dielectric.c:30-42,77-89 including its
// i < nx-1, j < ny-1, k < nz-1 loop bounds.

#include "row_quads.hpp"
#include "step_quad.hpp"

namespace mifdtd {

constexpr int S4B = 256;

// ------------------------------------------------------------------ stage kernels
// A lane per x-quad in the whole-grid thread order (row_quads.hpp with z as the planes and
// x as the cells: a stripe of every plane's rows per XCD, x-slab quads in waves of their
// own).  One pass updates E (or H) of a stage with its CPML, sources and probes, so each
// array is read and written once per stage; the y and z neighbour rows (three of each) are
// L2 hits of the stripe.  The bound is the traffic behind the L2s.  Against a marching
// work-group per 8 rows x 32 planes with separate CPML launches, called from Python (which
// left most of the chip idle on small grids: 36 work-groups at 132 x 90 x 75), a run's step
// with CPML 10: 64^3 620 -> 81 us, 132 x 90 x 75 726 -> 125, 200^3 971 -> 517, 400 x 300 x 200
// 2719 -> 1980, 512^3 10.76 -> 10.77 ms; without CPML 128^3 626 -> 130 us, 200^3 698 -> 367,
// 400^3 5542 -> 4294, 512^3 9.06 -> 8.78 ms; a bare stage H / E at 512^3 994 / 1035 -> 941 /
// 965 us, at 768 x 768 x 512 2322 / 2379 -> 2302 / 2300 (float CE, E 2825 -> 2877).
struct S4Geom {
    int nx, ny, nz;
    RowQuads m;
};

// CPML of one half: psi1/psi2 of face 2*axis + side (null: off), tables of the stage.
struct S4Cpml {
    int npml;
    float *psi1[6], *psi2[6];
    const float *b, *a;
};

// x neighbours of this lane's quad q of f (x = i0 .. i0+3): f[i0-2], f[i0-1], f[i0+4],
// f[i0+5], zero outside the row.  Called by every lane of the wave (lane shifts).
struct XN {
    float m2, m1, p4, p5;
};

__device__ __forceinline__ XN xneigh(const float *f, size_t id, const Q4 &q, int i0, int nx, bool prev, bool next)
{
    XN n;
    n.m2 = lane_prev(q.v[2]);
    n.m1 = lane_prev(q.v[3]);
    n.p4 = lane_next(q.v[0]);
    n.p5 = lane_next(q.v[1]);
    if (!prev) {
        const float2 t = i0 > 0 ? *reinterpret_cast<const float2 *>(f + id - 2) : make_float2(0.f, 0.f);
        n.m2 = t.x;
        n.m1 = t.y;
    }
    if (!next) {
        const float2 t = i0 + 4 < nx ? *reinterpret_cast<const float2 *>(f + id + 4) : make_float2(0.f, 0.f);
        n.p4 = t.x;
        n.p5 = t.y;
    }
    return n;
}

// CE of the E stage: the constant ce0, three float arrays, or three uint8 material-index
// arrays into a 3 x 256 table of the float values (the same products; the table stays in
// the caches).
enum S4Ce { kS4CeConst = 0, kS4CeArrays = 1, kS4CeTable = 2 };

template <int CEM>
__device__ __forceinline__ Q4 s4_ce(const float *c, const unsigned char *m, const float *tab, size_t id, float ce0)
{
    if (CEM == kS4CeConst) return splat4(ce0);
    if (CEM == kS4CeArrays) return ld4(c + id);
    return ce_from_table(m + id, tab);
}

// The 4th-order difference at one cell: 27 (p1 - p0) - (p2 - m1).
__device__ __forceinline__ float diff4(float m1, float p0, float p1, float p2) { return 27.f * (p1 - p0) - (p2 - m1); }

struct S4Half {
    float w;     // stage weight
    float b, a;  // table entry
};

// psi' = b psi + a d of one cell, and f -/+= w c psi'.
__device__ __forceinline__ void s4_psi_cell(const S4Half &h, float &psi, float d, float c, float &f, bool minus)
{
    const float tt = h.b * psi + h.a * d;
    psi = tt;
    if (minus) f -= h.w * c * tt;
    else f += h.w * c * tt;
}

// A quad's cells in an x face.  The slabs are more than a quad apart (nx >= 2 npml + 4), so
// a quad meets one side only: its cells' psi and table entries are consecutive.
struct S4FaceX {
    float *p1, *p2;  // psi1, psi2 of cell l = 0 (which may lie outside the slab)
    int t0;          // its table entry
    int lo, hi;      // cells l in [lo, hi) are in the slab and written by the stage
    float q1[4], q2[4], b[4], a[4];
    // slab planes [s0, s0+p) with entries from t; the stage writes [w0, w1); row = p*(j + ny*k)
    __device__ __forceinline__ void load(const S4Cpml &cp, int side, int i0, int s0, int t, int w0, int w1, size_t row)
    {
        float *f1 = side ? cp.psi1[1] : cp.psi1[0], *f2 = side ? cp.psi2[1] : cp.psi2[0];
        lo = max(max(s0, w0) - i0, 0);
        hi = f1 ? min(min(s0 + cp.npml, w1) - i0, 4) : 0;
        const ptrdiff_t o = (ptrdiff_t)row + (i0 - s0);
        p1 = f1 + o;
        p2 = f2 + o;
        t0 = t + (i0 - s0);
        const float *pb = cp.b + t0, *pa = cp.a + t0;
        // all loads before any store: a load that follows the previous cell's psi store is a
        // memory round trip of its own
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            q1[l] = q2[l] = b[l] = a[l] = 0.f;
            if (l >= lo && l < hi) {
                q1[l] = p1[l];
                q2[l] = p2[l];
                b[l] = pb[l];
                a[l] = pa[l];
            }
        }
    }
};

template <int CEM, bool PML>
__global__ __launch_bounds__(S4B) void k_s4_e(SAux, S4Geom g, S4Cpml cp, float dl, float *__restrict__ ex,
                                              float *__restrict__ ey, float *__restrict__ ez,
                                              const float *__restrict__ hx, const float *__restrict__ hy,
                                              const float *__restrict__ hz, const float *__restrict__ cx,
                                              const float *__restrict__ cy, const float *__restrict__ cz, float ce0,
                                              const unsigned char *__restrict__ mx, const unsigned char *__restrict__ my,
                                              const unsigned char *__restrict__ mz, const float *__restrict__ lut)
{
    const QuadAt at = row_quad(g.m, blockIdx.x, threadIdx.x);
    if (!at.active) return;
    const int k = at.i, j = at.j, i0 = 4 * at.q;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const int lane = threadIdx.x & 63;
    const size_t sy = (size_t)nx, sz = (size_t)nx * ny;
    const size_t id = (size_t)k * sz + (size_t)j * sy + i0;
    const Q4 z4 = splat4(0.f);
    // cells written: i, j, k <= n-2 and, off the component's own axis, 1 .. n-3
    const bool rows = j <= ny - 2 && k <= nz - 2;
    const bool jin = rows && j > 0 && j < ny - 2, kin = rows && k > 0 && k < nz - 2;
    const bool rx = jin && kin, ry = kin, rz = jin;

    const Q4 hx0 = ld4(hx + id), hy0 = ld4(hy + id), hz0 = ld4(hz + id);
    Q4 e0 = ld4(ex + id), e1 = ld4(ey + id), e2 = ld4(ez + id);
    const Q4 c0 = s4_ce<CEM>(cx, mx, lut, id, ce0);
    const Q4 c1 = s4_ce<CEM>(cy, my, lut + 256, id, ce0);
    const Q4 c2 = s4_ce<CEM>(cz, mz, lut + 512, id, ce0);
    Q4 hzm = z4, hzp = z4, hz2 = z4, hxm = z4, hxp = z4, hx2 = z4;  // rows j-1, j+1, j+2
    if (jin) {
        hzm = ld4(hz + id - sy);
        hzp = ld4(hz + id + sy);
        hz2 = ld4(hz + id + 2 * sy);
        hxm = ld4(hx + id - sy);
        hxp = ld4(hx + id + sy);
        hx2 = ld4(hx + id + 2 * sy);
    }
    Q4 hyM = z4, hyP = z4, hyQ = z4, hxM = z4, hxP = z4, hxQ = z4;  // planes k-1, k+1, k+2
    if (kin) {
        hyM = ld4(hy + id - sz);
        hyP = ld4(hy + id + sz);
        hyQ = ld4(hy + id + 2 * sz);
        hxM = ld4(hx + id - sz);
        hxP = ld4(hx + id + sz);
        hxQ = ld4(hx + id + 2 * sz);
    }
    const bool prev = at.prev && lane > 0, next = at.next && lane < 63;
    const XN nz_ = xneigh(hz, id, hz0, i0, nx, prev, next), ny_ = xneigh(hy, id, hy0, i0, nx, prev, next);
    // x windows f[i0-2 .. i0+5]
    const float wz[8] = {nz_.m2, nz_.m1, hz0.v[0], hz0.v[1], hz0.v[2], hz0.v[3], nz_.p4, nz_.p5};
    const float wy[8] = {ny_.m2, ny_.m1, hy0.v[0], hy0.v[1], hy0.v[2], hy0.v[3], ny_.p4, ny_.p5};
    const float c27 = 27.f;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int i = i0 + l;
        const bool in = i > 0 && i < nx - 2;
        if (rx && i <= nx - 2)
            e0.v[l] += dl * c0.v[l] * (c27 * (hzp.v[l] - hz0.v[l] - hyP.v[l] + hy0.v[l])
                                       - (hz2.v[l] - hzm.v[l] - hyQ.v[l] + hyM.v[l]));
        if (ry && in)
            e1.v[l] += dl * c1.v[l] * (c27 * (hxP.v[l] - hx0.v[l] - wz[l + 3] + hz0.v[l])
                                       - (hxQ.v[l] - hxM.v[l] - wz[l + 4] + wz[l + 1]));
        if (rz && in)
            e2.v[l] += dl * c2.v[l] * (c27 * (wy[l + 3] - hy0.v[l] - hxp.v[l] + hx0.v[l])
                                       - (wy[l + 4] - wy[l + 1] - hx2.v[l] + hxm.v[l]));
    }
    if (PML && rows) {
        const int p = cp.npml;
        int sdy, qy, sdz, qz;
        const int ty = jin ? sslab_e(j, ny, p, sdy, qy) : -1, tz = kin ? sslab_e(k, nz, p, sdz, qz) : -1;
        // the y and z faces' differences now: their rows and planes are not held any longer
        Q4 dy1 = z4, dy2 = z4, dz1 = z4, dz2 = z4;
        if (ty > 0) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                dy1.v[l] = diff4(hxm.v[l], hx0.v[l], hxp.v[l], hx2.v[l]);
                dy2.v[l] = diff4(hzm.v[l], hz0.v[l], hzp.v[l], hz2.v[l]);
            }
        }
        if (tz > 0) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                dz1.v[l] = diff4(hyM.v[l], hy0.v[l], hyP.v[l], hyQ.v[l]);
                dz2.v[l] = diff4(hxM.v[l], hx0.v[l], hxP.v[l], hxQ.v[l]);
            }
        }
        // psi of all faces together, when the rows' and planes' registers are free: face after
        // face, each one's loads wait for the stores before
        S4FaceX fx;
        const bool xf = i0 < p || i0 + 3 >= nx - 1 - p;
        if (xf) {
            const int side = i0 + 3 >= nx - 1 - p;
            fx.load(cp, side, i0, side ? nx - 1 - p : 0, side ? p + 1 : 1, 1, nx - 2, (size_t)p * ((size_t)j + (size_t)ny * k));
        }
        float *py1 = nullptr, *py2 = nullptr, *pz1 = nullptr, *pz2 = nullptr;
        Q4 sy1 = z4, sy2 = z4, sz1 = z4, sz2 = z4;
        if (ty > 0 && (sdy ? cp.psi1[3] : cp.psi1[2])) {
            const size_t n = (size_t)i0 + sy * ((size_t)qy + (size_t)p * k);
            py1 = (sdy ? cp.psi1[3] : cp.psi1[2]) + n;
            py2 = (sdy ? cp.psi2[3] : cp.psi2[2]) + n;
            sy1 = ld4u(py1);
            sy2 = ld4u(py2);
        }
        if (tz > 0 && (sdz ? cp.psi1[5] : cp.psi1[4])) {
            const size_t n = (size_t)i0 + sy * ((size_t)j + (size_t)ny * qz);
            pz1 = (sdz ? cp.psi1[5] : cp.psi1[4]) + n;
            pz2 = (sdz ? cp.psi2[5] : cp.psi2[4]) + n;
            sz1 = ld4u(pz1);
            sz2 = ld4u(pz2);
        }
        // x faces: psi1 -> ey from hz (-), psi2 -> ez from hy (+)
        if (xf) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                if (l < fx.lo || l >= fx.hi) continue;
                const S4Half h{dl, fx.b[l], fx.a[l]};
                if (ry) {
                    s4_psi_cell(h, fx.q1[l], diff4(wz[l + 1], wz[l + 2], wz[l + 3], wz[l + 4]), c1.v[l], e1.v[l], true);
                    fx.p1[l] = fx.q1[l];
                }
                if (rz) {
                    s4_psi_cell(h, fx.q2[l], diff4(wy[l + 1], wy[l + 2], wy[l + 3], wy[l + 4]), c2.v[l], e2.v[l], false);
                    fx.p2[l] = fx.q2[l];
                }
            }
        }
        // y faces: psi1 -> ez from hx (-), psi2 -> ex from hz (+)
        if (py1) {
            const S4Half h{dl, cp.b[ty], cp.a[ty]};
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int i = i0 + l;
                if (i > 0 && i < nx - 2) s4_psi_cell(h, sy1.v[l], dy1.v[l], c2.v[l], e2.v[l], true);
                if (rx && i <= nx - 2) s4_psi_cell(h, sy2.v[l], dy2.v[l], c0.v[l], e0.v[l], false);
            }
            st4u(py1, sy1);
            st4u(py2, sy2);
        }
        // z faces: psi1 -> ex from hy (-), psi2 -> ey from hx (+)
        if (pz1) {
            const S4Half h{dl, cp.b[tz], cp.a[tz]};
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int i = i0 + l;
                if (rx && i <= nx - 2) s4_psi_cell(h, sz1.v[l], dz1.v[l], c0.v[l], e0.v[l], true);
                if (i > 0 && i < nx - 2) s4_psi_cell(h, sz2.v[l], dz2.v[l], c1.v[l], e1.v[l], false);
            }
            st4u(pz1, sz1);
            st4u(pz2, sz2);
        }
    }
    const SAux &aux = first_kernel_arg<SAux>();
    const bool near = aux.near(k, j, i0);
    if (near) {
        sapply_src(aux.src, 0, k, j, i0, e0);
        sapply_src(aux.src, 1, k, j, i0, e1);
        sapply_src(aux.src, 2, k, j, i0, e2);
    }
    // (rows that the stage does not write are left alone, as in the passes of step_quad.hpp)
    if (rx || near) st4(ex + id, e0);
    if (ry || near) st4(ey + id, e1);
    if (rz || near) st4(ez + id, e2);
    if (near) {
        sprobe(aux.prb, 0, k, j, i0, e0);
        sprobe(aux.prb, 1, k, j, i0, e1);
        sprobe(aux.prb, 2, k, j, i0, e2);
    }
}

template <bool HC, bool PML>
__global__ __launch_bounds__(S4B) void k_s4_h(SAux, S4Geom g, S4Cpml cp, float cl, const float *__restrict__ ex,
                                              const float *__restrict__ ey, const float *__restrict__ ez,
                                              float *__restrict__ hx, float *__restrict__ hy, float *__restrict__ hz,
                                              const float *__restrict__ cx, const float *__restrict__ cy,
                                              const float *__restrict__ cz, float ch0)
{
    const QuadAt at = row_quad(g.m, blockIdx.x, threadIdx.x);
    if (!at.active) return;
    const int k = at.i, j = at.j, i0 = 4 * at.q;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const int lane = threadIdx.x & 63;
    const size_t sy = (size_t)nx, sz = (size_t)nx * ny;
    const size_t id = (size_t)k * sz + (size_t)j * sy + i0;
    const Q4 z4 = splat4(0.f);
    // cells written: i, j, k <= n-2 and, off the component's own axis, 2 .. n-2
    const bool rows = j <= ny - 2 && k <= nz - 2;
    const bool jin = rows && j > 1, kin = rows && k > 1;
    const bool rx = jin && kin, ry = kin, rz = jin;

    const Q4 ex0 = ld4(ex + id), ey0 = ld4(ey + id), ez0 = ld4(ez + id);
    Q4 h0 = ld4(hx + id), h1 = ld4(hy + id), h2 = ld4(hz + id);
    const Q4 c0 = HC ? ld4(cx + id) : splat4(ch0);
    const Q4 c1 = HC ? ld4(cy + id) : splat4(ch0);
    const Q4 c2 = HC ? ld4(cz + id) : splat4(ch0);
    Q4 ez2 = z4, ezm = z4, ezp = z4, ex2 = z4, exm = z4, exp = z4;  // rows j-2, j-1, j+1
    if (jin) {
        ez2 = ld4(ez + id - 2 * sy);
        ezm = ld4(ez + id - sy);
        ezp = ld4(ez + id + sy);
        ex2 = ld4(ex + id - 2 * sy);
        exm = ld4(ex + id - sy);
        exp = ld4(ex + id + sy);
    }
    Q4 eyQ = z4, eyM = z4, eyP = z4, exQ = z4, exM = z4, exP = z4;  // planes k-2, k-1, k+1
    if (kin) {
        eyQ = ld4(ey + id - 2 * sz);
        eyM = ld4(ey + id - sz);
        eyP = ld4(ey + id + sz);
        exQ = ld4(ex + id - 2 * sz);
        exM = ld4(ex + id - sz);
        exP = ld4(ex + id + sz);
    }
    const bool prev = at.prev && lane > 0, next = at.next && lane < 63;
    const XN nz_ = xneigh(ez, id, ez0, i0, nx, prev, next), ny_ = xneigh(ey, id, ey0, i0, nx, prev, next);
    const float wz[8] = {nz_.m2, nz_.m1, ez0.v[0], ez0.v[1], ez0.v[2], ez0.v[3], nz_.p4, nz_.p5};
    const float wy[8] = {ny_.m2, ny_.m1, ey0.v[0], ey0.v[1], ey0.v[2], ey0.v[3], ny_.p4, ny_.p5};
    const float c27 = 27.f;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const int i = i0 + l;
        const bool in = i > 1 && i <= nx - 2;
        if (rx && i <= nx - 2)
            h0.v[l] -= cl * c0.v[l] * (c27 * (ez0.v[l] - ezm.v[l] - ey0.v[l] + eyM.v[l])
                                       - (ezp.v[l] - ez2.v[l] - eyP.v[l] + eyQ.v[l]));
        if (ry && in)
            h1.v[l] -= cl * c1.v[l] * (c27 * (ex0.v[l] - exM.v[l] - ez0.v[l] + wz[l + 1])
                                       - (exP.v[l] - exQ.v[l] - wz[l + 3] + wz[l]));
        if (rz && in)
            h2.v[l] -= cl * c2.v[l] * (c27 * (ey0.v[l] - wy[l + 1] - ex0.v[l] + exm.v[l])
                                       - (wy[l + 3] - wy[l] - exp.v[l] + ex2.v[l]));
    }
    if (PML && rows) {
        const int p = cp.npml;
        int sdy, qy, sdz, qz;
        const int ty = jin ? sslab_h(j, ny, p, sdy, qy) : -1, tz = kin ? sslab_h(k, nz, p, sdz, qz) : -1;
        // the y and z faces' differences now: their rows and planes are not held any longer
        Q4 dy1 = z4, dy2 = z4, dz1 = z4, dz2 = z4;
        if (ty > 0) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                dy1.v[l] = diff4(ex2.v[l], exm.v[l], ex0.v[l], exp.v[l]);
                dy2.v[l] = diff4(ez2.v[l], ezm.v[l], ez0.v[l], ezp.v[l]);
            }
        }
        if (tz > 0) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                dz1.v[l] = diff4(eyQ.v[l], eyM.v[l], ey0.v[l], eyP.v[l]);
                dz2.v[l] = diff4(exQ.v[l], exM.v[l], ex0.v[l], exP.v[l]);
            }
        }
        // psi of all faces together, when the rows' and planes' registers are free: face after
        // face, each one's loads wait for the stores before
        S4FaceX fx;
        const bool xf = i0 < p || i0 + 3 >= nx - p;
        if (xf) {
            const int side = i0 + 3 >= nx - p;
            fx.load(cp, side, i0, side ? nx - p : 0, side ? p + 2 : 1, 2, nx - 1, (size_t)p * ((size_t)j + (size_t)ny * k));
        }
        float *py1 = nullptr, *py2 = nullptr, *pz1 = nullptr, *pz2 = nullptr;
        Q4 sy1 = z4, sy2 = z4, sz1 = z4, sz2 = z4;
        if (ty > 0 && (sdy ? cp.psi1[3] : cp.psi1[2])) {
            const size_t n = (size_t)i0 + sy * ((size_t)qy + (size_t)p * k);
            py1 = (sdy ? cp.psi1[3] : cp.psi1[2]) + n;
            py2 = (sdy ? cp.psi2[3] : cp.psi2[2]) + n;
            sy1 = ld4u(py1);
            sy2 = ld4u(py2);
        }
        if (tz > 0 && (sdz ? cp.psi1[5] : cp.psi1[4])) {
            const size_t n = (size_t)i0 + sy * ((size_t)j + (size_t)ny * qz);
            pz1 = (sdz ? cp.psi1[5] : cp.psi1[4]) + n;
            pz2 = (sdz ? cp.psi2[5] : cp.psi2[4]) + n;
            sz1 = ld4u(pz1);
            sz2 = ld4u(pz2);
        }
        // x faces: psi1 -> hy from ez (+), psi2 -> hz from ey (-)
        if (xf) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                if (l < fx.lo || l >= fx.hi) continue;
                const S4Half h{cl, fx.b[l], fx.a[l]};
                if (ry) {
                    s4_psi_cell(h, fx.q1[l], diff4(wz[l], wz[l + 1], wz[l + 2], wz[l + 3]), c1.v[l], h1.v[l], false);
                    fx.p1[l] = fx.q1[l];
                }
                if (rz) {
                    s4_psi_cell(h, fx.q2[l], diff4(wy[l], wy[l + 1], wy[l + 2], wy[l + 3]), c2.v[l], h2.v[l], true);
                    fx.p2[l] = fx.q2[l];
                }
            }
        }
        // y faces: psi1 -> hz from ex (+), psi2 -> hx from ez (-)
        if (py1) {
            const S4Half h{cl, cp.b[ty], cp.a[ty]};
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int i = i0 + l;
                if (i > 1 && i <= nx - 2) s4_psi_cell(h, sy1.v[l], dy1.v[l], c2.v[l], h2.v[l], false);
                if (rx && i <= nx - 2) s4_psi_cell(h, sy2.v[l], dy2.v[l], c0.v[l], h0.v[l], true);
            }
            st4u(py1, sy1);
            st4u(py2, sy2);
        }
        // z faces: psi1 -> hx from ey (+), psi2 -> hy from ex (-)
        if (pz1) {
            const S4Half h{cl, cp.b[tz], cp.a[tz]};
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const int i = i0 + l;
                if (rx && i <= nx - 2) s4_psi_cell(h, sz1.v[l], dz1.v[l], c0.v[l], h0.v[l], false);
                if (i > 1 && i <= nx - 2) s4_psi_cell(h, sz2.v[l], dz2.v[l], c1.v[l], h1.v[l], true);
            }
            st4u(pz1, sz1);
            st4u(pz2, sz2);
        }
    }
    const SAux &aux = first_kernel_arg<SAux>();
    const bool near = aux.near(k, j, i0);
    if (rx) st4(hx + id, h0);
    if (ry) st4(hy + id, h1);
    if (rz) st4(hz + id, h2);
    if (near) {
        sprobe(aux.prb, 3, k, j, i0, h0);
        sprobe(aux.prb, 4, k, j, i0, h1);
        sprobe(aux.prb, 5, k, j, i0, h2);
    }
}

// ------------------------------------------------------------------ CPML
// Thread per slab cell (both sides of one axis in one grid, side-major).  The face's
// two tangential components and the driving fields are picked by AXIS; see the header
// for the sign table.
__device__ __forceinline__ bool s4_valid_e(int c, int i, int j, int k, int nx, int ny, int nz)
{
    if (i > nx - 2 || j > ny - 2 || k > nz - 2) return false;
    if (c == 0) return j > 0 && j < ny - 2 && k > 0 && k < nz - 2;
    if (c == 1) return i > 0 && i < nx - 2 && k > 0 && k < nz - 2;
    return i > 0 && i < nx - 2 && j > 0 && j < ny - 2;
}
__device__ __forceinline__ bool s4_valid_h(int c, int i, int j, int k, int nx, int ny, int nz)
{
    if (i > nx - 2 || j > ny - 2 || k > nz - 2) return false;
    if (c == 0) return j > 1 && k > 1;
    if (c == 1) return i > 1 && k > 1;
    return i > 1 && j > 1;
}

struct S4Face {
    float *psi1[2], *psi2[2];
};

// Slab cell n of one side -> (i, j, k, psi index), psi layout x fastest:
// x face (npml, ny, nz), y face (nx, npml, nz), z face (nx, ny, npml).
template <int AXIS>
__device__ __forceinline__ void s4_slab_cell(unsigned n, int nx, int ny, int npml, int q, int &i, int &j, int &k)
{
    if (AXIS == 0) {
        const unsigned r = n / (unsigned)npml;  // j + ny*k
        j = (int)(r % (unsigned)ny);
        k = (int)(r / (unsigned)ny);
        i = q;
    } else if (AXIS == 1) {
        i = (int)(n % (unsigned)nx);
        const unsigned r = n / (unsigned)nx;  // p + npml*k
        k = (int)(r / (unsigned)npml);
        j = q;
    } else {
        i = (int)(n % (unsigned)nx);
        j = (int)((n / (unsigned)nx) % (unsigned)ny);
        k = q;
    }
}

template <int AXIS, bool HC>
__global__ __launch_bounds__(S4B) void k_s4_cpml_e(int nx, int ny, int nz, int npml, unsigned per_side, float w,
                                                   float *__restrict__ ex, float *__restrict__ ey, float *__restrict__ ez,
                                                   const float *__restrict__ hx, const float *__restrict__ hy,
                                                   const float *__restrict__ hz, const float *__restrict__ cx,
                                                   const float *__restrict__ cy, const float *__restrict__ cz, float ce0,
                                                   S4Face fs, const float *__restrict__ tb, const float *__restrict__ ta)
{
    unsigned n = blockIdx.x * S4B + threadIdx.x;
    if (n >= 2 * per_side) return;
    const int side = n >= per_side;
    if (side) n -= per_side;
    float *psi1 = fs.psi1[side], *psi2 = fs.psi2[side];
    if (!psi1) return;
    const int n_e = AXIS == 0 ? nx : AXIS == 1 ? ny : nz;
    int p;
    if (AXIS == 0) p = (int)(n % (unsigned)npml);
    else if (AXIS == 1) p = (int)((n / (unsigned)nx) % (unsigned)npml);
    else p = (int)(n / ((unsigned)nx * (unsigned)ny));
    const int q = side ? n_e - 1 - npml + p : p;
    const int t = side ? npml + 1 + p : p + 1;
    int i, j, k;
    s4_slab_cell<AXIS>(n, nx, ny, npml, q, i, j, k);
    const size_t id = ((size_t)k * ny + j) * nx + i;
    const size_t s = AXIS == 0 ? 1 : AXIS == 1 ? (size_t)nx : (size_t)nx * ny;
    // x: psi1 -> ey from hz (-), psi2 -> ez from hy (+); y: psi1 -> ez from hx (-),
    // psi2 -> ex from hz (+); z: psi1 -> ex from hy (-), psi2 -> ey from hx (+)
    float *e1 = AXIS == 0 ? ey : AXIS == 1 ? ez : ex;
    float *e2 = AXIS == 0 ? ez : AXIS == 1 ? ex : ey;
    const float *g1 = AXIS == 0 ? hz : AXIS == 1 ? hx : hy;
    const float *g2 = AXIS == 0 ? hy : AXIS == 1 ? hz : hx;
    const float *c1 = AXIS == 0 ? cy : AXIS == 1 ? cz : cx;
    const float *c2 = AXIS == 0 ? cz : AXIS == 1 ? cx : cy;
    const int comp1 = AXIS == 0 ? 1 : AXIS == 1 ? 2 : 0, comp2 = AXIS == 0 ? 2 : AXIS == 1 ? 0 : 1;
    const float b = tb[t], a = ta[t];
    const float c27 = 27.f;
    if (s4_valid_e(comp1, i, j, k, nx, ny, nz)) {
        const float d = c27 * (g1[id + s] - g1[id]) - (g1[id + 2 * s] - g1[id - s]);
        const float tt = b * psi1[n] + a * d;
        psi1[n] = tt;
        e1[id] -= w * (HC ? c1[id] : ce0) * tt;
    }
    if (s4_valid_e(comp2, i, j, k, nx, ny, nz)) {
        const float d = c27 * (g2[id + s] - g2[id]) - (g2[id + 2 * s] - g2[id - s]);
        const float tt = b * psi2[n] + a * d;
        psi2[n] = tt;
        e2[id] += w * (HC ? c2[id] : ce0) * tt;
    }
}

template <int AXIS, bool HC>
__global__ __launch_bounds__(S4B) void k_s4_cpml_h(int nx, int ny, int nz, int npml, unsigned per_side, float w,
                                                   const float *__restrict__ ex, const float *__restrict__ ey,
                                                   const float *__restrict__ ez, float *__restrict__ hx,
                                                   float *__restrict__ hy, float *__restrict__ hz,
                                                   const float *__restrict__ cx, const float *__restrict__ cy,
                                                   const float *__restrict__ cz, float ch0, S4Face fs,
                                                   const float *__restrict__ tb, const float *__restrict__ ta)
{
    unsigned n = blockIdx.x * S4B + threadIdx.x;
    if (n >= 2 * per_side) return;
    const int side = n >= per_side;
    if (side) n -= per_side;
    float *psi1 = fs.psi1[side], *psi2 = fs.psi2[side];
    if (!psi1) return;
    const int n_e = AXIS == 0 ? nx : AXIS == 1 ? ny : nz;
    int p;
    if (AXIS == 0) p = (int)(n % (unsigned)npml);
    else if (AXIS == 1) p = (int)((n / (unsigned)nx) % (unsigned)npml);
    else p = (int)(n / ((unsigned)nx * (unsigned)ny));
    const int q = side ? n_e - npml + p : p;
    const int t = side ? npml + 2 + p : p + 1;
    int i, j, k;
    s4_slab_cell<AXIS>(n, nx, ny, npml, q, i, j, k);
    const size_t id = ((size_t)k * ny + j) * nx + i;
    const size_t s = AXIS == 0 ? 1 : AXIS == 1 ? (size_t)nx : (size_t)nx * ny;
    // x: psi1 -> hy from ez (+), psi2 -> hz from ey (-); y: psi1 -> hz from ex (+),
    // psi2 -> hx from ez (-); z: psi1 -> hx from ey (+), psi2 -> hy from ex (-)
    float *h1 = AXIS == 0 ? hy : AXIS == 1 ? hz : hx;
    float *h2 = AXIS == 0 ? hz : AXIS == 1 ? hx : hy;
    const float *g1 = AXIS == 0 ? ez : AXIS == 1 ? ex : ey;
    const float *g2 = AXIS == 0 ? ey : AXIS == 1 ? ez : ex;
    const float *c1 = AXIS == 0 ? cy : AXIS == 1 ? cz : cx;
    const float *c2 = AXIS == 0 ? cz : AXIS == 1 ? cx : cy;
    const int comp1 = AXIS == 0 ? 1 : AXIS == 1 ? 2 : 0, comp2 = AXIS == 0 ? 2 : AXIS == 1 ? 0 : 1;
    const float b = tb[t], a = ta[t];
    const float c27 = 27.f;
    if (s4_valid_h(comp1, i, j, k, nx, ny, nz)) {
        const float d = c27 * (g1[id] - g1[id - s]) - (g1[id + s] - g1[id - 2 * s]);
        const float tt = b * psi1[n] + a * d;
        psi1[n] = tt;
        h1[id] += w * (HC ? c1[id] : ch0) * tt;
    }
    if (s4_valid_h(comp2, i, j, k, nx, ny, nz)) {
        const float d = c27 * (g2[id] - g2[id - s]) - (g2[id + s] - g2[id - 2 * s]);
        const float tt = b * psi2[n] + a * d;
        psi2[n] = tt;
        h2[id] -= w * (HC ? c2[id] : ch0) * tt;
    }
}

static int s4_check(int nx, int ny, int nz)
{
    if (nx < 4 || ny < 4 || nz < 4) return fail(MIFDTD_EINVAL, "4th-order grid (%d,%d,%d) smaller than 4", nx, ny, nz);
    if (nx % 4) return fail(MIFDTD_EALIGN, "4th-order nx %d is not a multiple of 4", nx);
    if ((unsigned long long)nx * ny * nz / 4 >= (1ull << 31)) return fail(MIFDTD_ERANGE, "4th-order grid too large");
    return 0;
}

static S4Geom s4_geom(int nx, int ny, int nz, int npml)
{
    return S4Geom{nx, ny, nz, row_quads((unsigned)nz, (unsigned)ny, (unsigned)(nx / 4), nx, npml)};
}

static int s4_check_fields(float *const e[6])
{
    for (int c = 0; c < 6; c++) {
        if (!e[c]) return fail(MIFDTD_ENULL, "field pointer is NULL");
        if (!aligned16(e[c])) return fail(MIFDTD_EALIGN, "field pointer not 16-byte aligned");
    }
    return 0;
}

static int s4_check_coef(const float *c0, const float *c1, const float *c2)
{
    if (!(c0 || c1 || c2)) return 0;
    if (!(c0 && c1 && c2)) return fail(MIFDTD_ENULL, "coefficient arrays must be all set or all NULL");
    if (!aligned16(c0) || !aligned16(c1) || !aligned16(c2))
        return fail(MIFDTD_EALIGN, "coefficient pointer not 16-byte aligned");
    return 0;
}

static int s4_check_mat(const unsigned char *const m[3], const float *lut)
{
    if (!m[0] || !m[1] || !m[2] || !lut) return fail(MIFDTD_ENULL, "material index or table is NULL");
    for (int c = 0; c < 3; c++)
        if (reinterpret_cast<uintptr_t>(m[c]) & 3u) return fail(MIFDTD_EALIGN, "material index array not 4-byte aligned");
    return 0;
}

static int s4_check_pml(int nx, int ny, int nz, const mifdtd_cpml_half *cp)
{
    const int npml = cp->npml;
    if (npml < 1 || npml > MIFDTD_MAX_NPML) return fail(MIFDTD_EINVAL, "npml %d outside [1,%d]", npml, MIFDTD_MAX_NPML);
    if (nx < 2 * npml + 4 || ny < 2 * npml + 4 || nz < 2 * npml + 4)
        return fail(MIFDTD_EINVAL, "4th-order grid (%d,%d,%d) too small for npml %d", nx, ny, nz, npml);
    if (!cp->b || !cp->a) return fail(MIFDTD_ENULL, "CPML tables are NULL");
    for (int f = 0; f < 6; f++)
        if ((cp->psi1[f] == nullptr) != (cp->psi2[f] == nullptr))
            return fail(MIFDTD_ENULL, "psi1/psi2 of face %d must both be set or both NULL", f);
    return 0;
}

static S4Cpml s4_pml(const mifdtd_cpml_half &h)
{
    S4Cpml c{};
    c.npml = h.npml;
    c.b = h.b;
    c.a = h.a;
    for (int f = 0; f < 6; f++) {
        c.psi1[f] = h.psi1[f];
        c.psi2[f] = h.psi2[f];
    }
    return c;
}

// One E (H) stage: pml null without CPML.
static int s4_stage_e(const S4Geom &g, const S4Cpml *pml, const SAux &aux, float dl, float *const e[6], int cem,
                      const float *const c[3], float ce0, const unsigned char *const m[3], const float *lut, hipStream_t st)
{
    const unsigned nb = (unsigned)row_quads_blocks(g.m);
    const S4Cpml cp = pml ? *pml : S4Cpml{};
#define MIFDTD_S4_E(CEM, P)                                                                                             \
    k_s4_e<CEM, P><<<nb, S4B, 0, st>>>(aux, g, cp, dl, e[0], e[1], e[2], e[3], e[4], e[5], c[0], c[1], c[2], ce0, m[0], m[1], \
                                       m[2], lut)
    if (cem == kS4CeTable) {
        if (pml) MIFDTD_S4_E(kS4CeTable, true);
        else MIFDTD_S4_E(kS4CeTable, false);
    } else if (cem == kS4CeArrays) {
        if (pml) MIFDTD_S4_E(kS4CeArrays, true);
        else MIFDTD_S4_E(kS4CeArrays, false);
    } else {
        if (pml) MIFDTD_S4_E(kS4CeConst, true);
        else MIFDTD_S4_E(kS4CeConst, false);
    }
#undef MIFDTD_S4_E
    MIFDTD_CHECK_LAUNCH("s4 update_e launch");
    return 0;
}

static int s4_stage_h(const S4Geom &g, const S4Cpml *pml, const SAux &aux, float cl, float *const e[6],
                      const float *const c[3], float ch0, hipStream_t st)
{
    const unsigned nb = (unsigned)row_quads_blocks(g.m);
    const S4Cpml cp = pml ? *pml : S4Cpml{};
#define MIFDTD_S4_H(HC, P) \
    k_s4_h<HC, P><<<nb, S4B, 0, st>>>(aux, g, cp, cl, e[0], e[1], e[2], e[3], e[4], e[5], c[0], c[1], c[2], ch0)
    if (c[0]) {
        if (pml) MIFDTD_S4_H(true, true);
        else MIFDTD_S4_H(true, false);
    } else {
        if (pml) MIFDTD_S4_H(false, true);
        else MIFDTD_S4_H(false, false);
    }
#undef MIFDTD_S4_H
    MIFDTD_CHECK_LAUNCH("s4 update_h launch");
    return 0;
}

static int s4_core(bool h_half, int nx, int ny, int nz, float w, float *ex, float *ey, float *ez, float *hx, float *hy,
                   float *hz, const float *c0, const float *c1, const float *c2, float cconst, hipStream_t st)
{
    if (int rc = s4_check(nx, ny, nz)) return rc;
    float *const e[6] = {ex, ey, ez, hx, hy, hz};
    if (int rc = s4_check_fields(e)) return rc;
    if (int rc = s4_check_coef(c0, c1, c2)) return rc;
    const float *const c[3] = {c0, c1, c2};
    const unsigned char *const m[3] = {nullptr, nullptr, nullptr};
    const S4Geom g = s4_geom(nx, ny, nz, 0);
    SAux aux{};
    aux_box(aux);
    if (h_half) return s4_stage_h(g, nullptr, aux, w, e, c, cconst, st);
    return s4_stage_e(g, nullptr, aux, w, e, c0 ? kS4CeArrays : kS4CeConst, c, cconst, m, nullptr, st);
}

template <int AXIS>
static int s4_cpml_axis(bool h_half, int nx, int ny, int nz, const mifdtd_cpml_half *cp, float w, float *ex, float *ey,
                        float *ez, float *hx, float *hy, float *hz, const float *c0, const float *c1, const float *c2,
                        float cconst, hipStream_t st)
{
    S4Face fs;
    bool any = false;
    for (int sd = 0; sd < 2; sd++) {
        fs.psi1[sd] = cp->psi1[2 * AXIS + sd];
        fs.psi2[sd] = cp->psi2[2 * AXIS + sd];
        if ((fs.psi1[sd] == nullptr) != (fs.psi2[sd] == nullptr))
            return fail(MIFDTD_ENULL, "psi1/psi2 of face %d must both be set or both NULL", 2 * AXIS + sd);
        any = any || fs.psi1[sd];
    }
    if (!any) return 0;
    const int npml = cp->npml;
    const unsigned per_side = AXIS == 0 ? (unsigned)npml * ny * nz
                            : AXIS == 1 ? (unsigned)nx * npml * nz
                                        : (unsigned)nx * ny * npml;
    const unsigned grid = (2 * per_side + S4B - 1) / S4B;
    const bool hc = c0 != nullptr;
    if (h_half) {
        if (hc) k_s4_cpml_h<AXIS, true><<<grid, S4B, 0, st>>>(nx, ny, nz, npml, per_side, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, fs, cp->b, cp->a);
        else k_s4_cpml_h<AXIS, false><<<grid, S4B, 0, st>>>(nx, ny, nz, npml, per_side, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, fs, cp->b, cp->a);
    } else {
        if (hc) k_s4_cpml_e<AXIS, true><<<grid, S4B, 0, st>>>(nx, ny, nz, npml, per_side, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, fs, cp->b, cp->a);
        else k_s4_cpml_e<AXIS, false><<<grid, S4B, 0, st>>>(nx, ny, nz, npml, per_side, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, fs, cp->b, cp->a);
    }
    MIFDTD_CHECK_LAUNCH("s4 cpml launch");
    return 0;
}

static int s4_cpml(bool h_half, int nx, int ny, int nz, const mifdtd_cpml_half *cp, float w, float *ex, float *ey,
                   float *ez, float *hx, float *hy, float *hz, const float *c0, const float *c1, const float *c2,
                   float cconst, hipStream_t st)
{
    if (int rc = s4_check(nx, ny, nz)) return rc;
    if (!cp) return fail(MIFDTD_ENULL, "CPML descriptor is NULL");
    if (int rc = s4_check_pml(nx, ny, nz, cp)) return rc;
    if ((c0 || c1 || c2) && !(c0 && c1 && c2)) return fail(MIFDTD_ENULL, "coefficient arrays must be all set or all NULL");
    if (int rc = s4_cpml_axis<0>(h_half, nx, ny, nz, cp, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, st)) return rc;
    if (int rc = s4_cpml_axis<1>(h_half, nx, ny, nz, cp, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, st)) return rc;
    return s4_cpml_axis<2>(h_half, nx, ny, nz, cp, w, ex, ey, ez, hx, hy, hz, c0, c1, c2, cconst, st);
}

}  // namespace mifdtd

using namespace mifdtd;

extern "C" {

void s4_update_h(int nx, int ny, int nz, float cl, float *ex, float *ey, float *ez, float *hx, float *hy, float *hz,
                 float *cx, float *cy, float *cz)
{
    if (!cx || !cy || !cz) {
        fail(MIFDTD_ENULL, "s4_update_h needs the three coefficient arrays");
        return;
    }
    s4_core(true, nx, ny, nz, cl, ex, ey, ez, hx, hy, hz, cx, cy, cz, 0.f, nullptr);
}

void s4_update_e(int nx, int ny, int nz, float dl, float *ex, float *ey, float *ez, float *hx, float *hy, float *hz,
                 float *cx, float *cy, float *cz)
{
    if (!cx || !cy || !cz) {
        fail(MIFDTD_ENULL, "s4_update_e needs the three coefficient arrays");
        return;
    }
    s4_core(false, nx, ny, nz, dl, ex, ey, ez, hx, hy, hz, cx, cy, cz, 0.f, nullptr);
}

int mifdtd_s4_update_h(int nx, int ny, int nz, float cl, const float *ex, const float *ey, const float *ez, float *hx,
                       float *hy, float *hz, const float *chx, const float *chy, const float *chz, float ch0,
                       mifdtd_stream_t stream)
{
    return s4_core(true, nx, ny, nz, cl, const_cast<float *>(ex), const_cast<float *>(ey), const_cast<float *>(ez), hx,
                   hy, hz, chx, chy, chz, ch0, to_stream(stream));
}

int mifdtd_s4_update_e(int nx, int ny, int nz, float dl, float *ex, float *ey, float *ez, const float *hx,
                       const float *hy, const float *hz, const float *cex, const float *cey, const float *cez, float ce0,
                       mifdtd_stream_t stream)
{
    return s4_core(false, nx, ny, nz, dl, ex, ey, ez, const_cast<float *>(hx), const_cast<float *>(hy),
                   const_cast<float *>(hz), cex, cey, cez, ce0, to_stream(stream));
}

int mifdtd_s4_update_e_lut(int nx, int ny, int nz, float dl, float *ex, float *ey, float *ez, const float *hx,
                           const float *hy, const float *hz, const unsigned char *mat_x, const unsigned char *mat_y,
                           const unsigned char *mat_z, const float *lut, mifdtd_stream_t stream)
{
    if (int rc = s4_check(nx, ny, nz)) return rc;
    float *const e[6] = {ex, ey, ez, const_cast<float *>(hx), const_cast<float *>(hy), const_cast<float *>(hz)};
    if (int rc = s4_check_fields(e)) return rc;
    const unsigned char *const m[3] = {mat_x, mat_y, mat_z};
    if (int rc = s4_check_mat(m, lut)) return rc;
    const float *const c[3] = {nullptr, nullptr, nullptr};
    SAux aux{};
    aux_box(aux);
    return s4_stage_e(s4_geom(nx, ny, nz, 0), nullptr, aux, dl, e, kS4CeTable, c, 0.f, m, lut, to_stream(stream));
}

int mifdtd_s4_run(const mifdtd_s4_desc *d, int nsteps, const float *tvals, float *probe_series, mifdtd_stream_t stream)
{
    if (!d) return fail(MIFDTD_ENULL, "step descriptor is NULL");
    const int nx = d->nx, ny = d->ny, nz = d->nz;
    if (int rc = s4_check(nx, ny, nz)) return rc;
    if (nsteps < 0) return fail(MIFDTD_EINVAL, "nsteps < 0");
    if (int rc = s4_check_fields(d->e)) return rc;
    if (int rc = s4_check_coef(d->ce[0], d->ce[1], d->ce[2])) return rc;
    if (int rc = s4_check_coef(d->ch[0], d->ch[1], d->ch[2])) return rc;
    const bool tbl = d->ce_mat[0] != nullptr;
    if (tbl)
        if (int rc = s4_check_mat(d->ce_mat, d->ce_lut)) return rc;
    const int cem = tbl ? kS4CeTable : d->ce[0] ? kS4CeArrays : kS4CeConst;
    const bool pml = d->cpml_e[0].npml > 0;
    S4Cpml pe[4], ph[5];
    if (pml) {
        for (int s = 0; s < 9; s++) {
            const mifdtd_cpml_half &h = s < 4 ? d->cpml_e[s] : d->cpml_h[s - 4];
            if (h.npml != d->cpml_e[0].npml) return fail(MIFDTD_EINVAL, "the stages' npml differ");
            if (int rc = s4_check_pml(nx, ny, nz, &h)) return rc;
            (s < 4 ? pe[s] : ph[s - 4]) = s4_pml(h);
        }
    }
    if (d->nsrc < 0 || d->nsrc > MIFDTD_FUSED_MAX_SRC) return fail(MIFDTD_EINVAL, "nsrc outside [0,%d]", MIFDTD_FUSED_MAX_SRC);
    if (d->nprobe < 0 || d->nprobe > MIFDTD_FUSED_MAX_PROBE)
        return fail(MIFDTD_EINVAL, "nprobe outside [0,%d]", MIFDTD_FUSED_MAX_PROBE);
    if (d->nsrc && !tvals) return fail(MIFDTD_ENULL, "tvals is NULL");
    if (d->nprobe && !probe_series) return fail(MIFDTD_ENULL, "probe_series is NULL");
    // the passes' planes are z and their cells x
    SSrc src{};
    src.n = d->nsrc;
    for (int n = 0; n < d->nsrc; n++) {
        const int *b = d->src_box[n];
        if (d->src_comp[n] < 0 || d->src_comp[n] > 2) return fail(MIFDTD_EINVAL, "source %d component %d", n, d->src_comp[n]);
        if (b[0] < 0 || b[2] < 0 || b[4] < 0 || b[1] >= nx || b[3] >= ny || b[5] >= nz || b[0] > b[1] || b[2] > b[3] ||
            b[4] > b[5])
            return fail(MIFDTD_EINVAL, "source box %d outside the grid", n);
        src.comp[n] = d->src_comp[n];
        src.i0[n] = b[4];
        src.i1[n] = b[5];
        src.j0[n] = b[2];
        src.j1[n] = b[3];
        src.k0[n] = b[0];
        src.k1[n] = b[1];
        src.sv[n] = d->src_sv[n];
        src.svs[n] = d->src_svs[n];
    }
    SProbe pbe{}, pbh{};
    for (int n = 0; n < d->nprobe; n++) {
        const int *p = d->probe_ijk[n], c = d->probe_comp[n];
        if (c < 0 || c > 5 || p[0] < 0 || p[0] >= nx || p[1] < 0 || p[1] >= ny || p[2] < 0 || p[2] >= nz)
            return fail(MIFDTD_EINVAL, "probe %d outside the grid", n);
        SProbe &P = c < 3 ? pbe : pbh;
        const int m = P.n++;
        P.comp[m] = c;
        P.i[m] = p[2];
        P.j[m] = p[1];
        P.k[m] = p[0];
        P.slot[m] = n;
    }
    const S4Geom g = s4_geom(nx, ny, nz, pml ? d->cpml_e[0].npml : 0);
    hipStream_t st = to_stream(stream);
    for (int t = 0; t < nsteps; t++) {
        float *row = d->nprobe ? probe_series + (size_t)t * d->nprobe : nullptr;
        for (int s = 0; s < 5; s++) {
            SAux ah{};
            if (s == 4) {  // the H components are final after the closing stage
                ah.prb = pbh;
                ah.prb.out = row;
            }
            aux_box(ah);
            if (int rc = s4_stage_h(g, pml ? &ph[s] : nullptr, ah, d->cl[s], d->e, d->ch, d->ch0, st)) return rc;
            if (s == 4) break;
            SAux ae{};
            ae.src = src;
            for (int n = 0; n < src.n; n++) ae.src.tval[n] = tvals[((size_t)t * 4 + s) * src.n + n];
            if (s == 3) {
                ae.prb = pbe;
                ae.prb.out = row;
            }
            aux_box(ae);
            if (int rc = s4_stage_e(g, pml ? &pe[s] : nullptr, ae, d->dl[s], d->e, cem, d->ce, d->ce0, d->ce_mat,
                                    d->ce_lut, st))
                return rc;
        }
    }
    return 0;
}

int mifdtd_s4_cpml_e(int nx, int ny, int nz, const mifdtd_cpml_half *cp, float dl, float *ex, float *ey, float *ez,
                     const float *hx, const float *hy, const float *hz, const float *cex, const float *cey,
                     const float *cez, float ce0, mifdtd_stream_t stream)
{
    return s4_cpml(false, nx, ny, nz, cp, dl, ex, ey, ez, const_cast<float *>(hx), const_cast<float *>(hy),
                   const_cast<float *>(hz), cex, cey, cez, ce0, to_stream(stream));
}

int mifdtd_s4_cpml_h(int nx, int ny, int nz, const mifdtd_cpml_half *cp, float cl, const float *ex, const float *ey,
                     const float *ez, float *hx, float *hy, float *hz, const float *chx, const float *chy,
                     const float *chz, float ch0, mifdtd_stream_t stream)
{
    return s4_cpml(true, nx, ny, nz, cp, cl, const_cast<float *>(ex), const_cast<float *>(ey), const_cast<float *>(ez),
                   hx, hy, hz, chx, chy, chz, ch0, to_stream(stream));
}

}  // extern "C"
