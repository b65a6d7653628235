// Double-precision KEMP core: update_e / update_h of the reference's 'double' programs
// (K7/cpu/src/core.c:11,59 substituted with DTYPE=double, INCRE=2 by K7/cpu/core.py:52-54;
// fields of K7/cpu/fields.py:25 with nz_pitch padded to 16 bytes = 2 doubles).
//
// Layout: C-order (nx, ny, nzp) float64, z contiguous, nzp even, pad lanes zero (the CPU
// programs pad nz to 2 doubles, pad 0 or 1; a 64-byte GPU pitch, K7/gpu/fields.py:45-50,
// gives pads up to 7 and the same masks by index).  One thread owns one
// aligned z-pair (16 bytes per array, the reference's SSE2 vector); consecutive lanes own
// consecutive pairs, so a wave streams 1 KiB per array.  Arithmetic order and masks are
// those of the float kernels (value*0 on masked lanes keeps the reference's signed zeros);
// compiled with -ffp-contract=off the results equal the reference's SSE2 code bit for bit.

#include "whole_pass.hpp"

namespace mifdtd {

namespace {

constexpr int kBlockD = 256;

struct D2 {
    double v[2];
};

__device__ __forceinline__ D2 ld2(const double *__restrict__ p)
{
    const double2 t = *reinterpret_cast<const double2 *>(p);
    return D2{{t.x, t.y}};
}

__device__ __forceinline__ void st2(double *__restrict__ p, const D2 &q)
{
    *reinterpret_cast<double2 *>(p) = make_double2(q.v[0], q.v[1]);
}

template <bool HC>
__device__ __forceinline__ D2 ldc(const double *__restrict__ c, size_t id)
{
    return HC ? ld2(c + id) : D2{{0.5, 0.5}};
}

// The next (previous) lane's value; the lane at the end takes 0.
__device__ __forceinline__ double lane_next_d(double x)
{
    return __hiloint2double(__float_as_int(lane_next(__int_as_float(__double2hiint(x)))),
                            __float_as_int(lane_next(__int_as_float(__double2loint(x)))));
}
__device__ __forceinline__ double lane_prev_d(double x)
{
    return __hiloint2double(__float_as_int(lane_prev(__int_as_float(__double2hiint(x)))),
                            __float_as_int(lane_prev(__int_as_float(__double2loint(x)))));
}

// The pair (i, j, k0..k0+1) of a thread, and whether the next / previous lane holds the next /
// previous pair in memory.
struct PairAt {
    int i, j, k0;
    bool next, prev;
};

struct GridF64 {
    int nx, ny, nzp, nz;
};

// Both updates issue all loads of the pair together (128 B without coefficients, of which 64
// are neighbours, and 48 B with them), as the bound is memory; rows and planes that an update
// does not reach keep the value loaded.
template <bool HC>
__device__ __forceinline__ void e_pair(const GridF64 &g, const PairAt &r, double *ex, double *ey, double *ez,
                                       const double *__restrict__ hx, const double *__restrict__ hy,
                                       const double *__restrict__ hz, const double *__restrict__ cex,
                                       const double *__restrict__ cey, const double *__restrict__ cez)
{
    const size_t id = ((size_t)r.i * g.ny + r.j) * g.nzp + r.k0;
    const size_t sx = (size_t)g.ny * g.nzp;
    const bool jy = r.j < g.ny - 1, ix = r.i < g.nx - 1;
    const D2 z2{{0.0, 0.0}};
    const D2 hx0 = ld2(hx + id), hy0 = ld2(hy + id), hz0 = ld2(hz + id);
    D2 e0 = ld2(ex + id), e1 = ld2(ey + id), e2 = ld2(ez + id);
    const D2 c0 = ldc<HC>(cex, id), c1 = ldc<HC>(cey, id), c2 = ldc<HC>(cez, id);
    const D2 hzU = jy ? ld2(hz + id + g.nzp) : z2, hxU = jy ? ld2(hx + id + g.nzp) : z2;
    const D2 hzN = ix ? ld2(hz + id + sx) : z2, hyN = ix ? ld2(hy + id + sx) : z2;
    double hyn = 0.0, hxn = 0.0;  // hy, hx at k0+2 (next row's first element on the last pair)
    if (!r.next) {
        if (jy) hyn = hy[id + 2];
        if (ix) hxn = hx[id + 2];
    }
    const double yl = lane_next_d(hy0.v[0]), xl = lane_next_d(hx0.v[0]);  // every lane of the wave takes part
    if (r.next) {
        hyn = yl;
        hxn = xl;
    }
#pragma unroll
    for (int l = 0; l < 2; l++) {
        const double y1 = l < 1 ? hy0.v[1] : hyn, x1 = l < 1 ? hx0.v[1] : hxn;
        const bool in = r.k0 + l < g.nz - 1;
        if (jy) {
            const double v = e0.v[l] + c0.v[l] * ((hzU.v[l] - hz0.v[l]) - (y1 - hy0.v[l]));
            e0.v[l] = in ? v : v * 0.0;
        }
        if (ix) {
            const double v = e1.v[l] + c1.v[l] * ((x1 - hx0.v[l]) - (hzN.v[l] - hz0.v[l]));
            e1.v[l] = in ? v : v * 0.0;
        }
        if (ix && jy) {
            const double v = e2.v[l] + c2.v[l] * ((hyN.v[l] - hy0.v[l]) - (hxU.v[l] - hx0.v[l]));
            e2.v[l] = (r.k0 + l < g.nz) ? v : v * 0.0;
        }
    }
    if (jy) st2(ex + id, e0);
    if (ix) st2(ey + id, e1);
    if (ix && jy) st2(ez + id, e2);
}

template <bool HC>
__device__ __forceinline__ void h_pair(const GridF64 &g, const PairAt &r, const double *__restrict__ ex,
                                       const double *__restrict__ ey, const double *__restrict__ ez, double *hx,
                                       double *hy, double *hz, const double *__restrict__ chx,
                                       const double *__restrict__ chy, const double *__restrict__ chz)
{
    const size_t id = ((size_t)r.i * g.ny + r.j) * g.nzp + r.k0;
    const size_t sx = (size_t)g.ny * g.nzp;
    const bool jp = r.j > 0, ip = r.i > 0;
    const D2 z2{{0.0, 0.0}};
    const D2 ex0 = ld2(ex + id), ey0 = ld2(ey + id), ez0 = ld2(ez + id);
    D2 h0 = ld2(hx + id), h1 = ld2(hy + id), h2 = ld2(hz + id);
    const D2 c0 = ldc<HC>(chx, id), c1 = ldc<HC>(chy, id), c2 = ldc<HC>(chz, id);
    const D2 ezD = jp ? ld2(ez + id - g.nzp) : z2, exD = jp ? ld2(ex + id - g.nzp) : z2;
    const D2 ezB = ip ? ld2(ez + id - sx) : z2, eyB = ip ? ld2(ey + id - sx) : z2;
    double eyp = 0.0, exp_ = 0.0;  // ey, ex at k0-1 (previous row's last element when k0 == 0)
    if (!r.prev) {
        if (jp) eyp = ey[id - 1];
        if (ip) exp_ = ex[id - 1];
    }
    const double yl = lane_prev_d(ey0.v[1]), xl = lane_prev_d(ex0.v[1]);  // every lane of the wave takes part
    if (r.prev) {
        eyp = yl;
        exp_ = xl;
    }
#pragma unroll
    for (int l = 0; l < 2; l++) {
        const double ym = l > 0 ? ey0.v[0] : eyp, xm = l > 0 ? ex0.v[0] : exp_;
        const int k = r.k0 + l;
        const bool in = k > 0 && k < g.nz;
        if (jp) {
            const double v = h0.v[l] - c0.v[l] * ((ez0.v[l] - ezD.v[l]) - (ey0.v[l] - ym));
            h0.v[l] = in ? v : v * 0.0;
        }
        if (ip) {
            const double v = h1.v[l] - c1.v[l] * ((ex0.v[l] - xm) - (ez0.v[l] - ezB.v[l]));
            h1.v[l] = in ? v : v * 0.0;
        }
        if (ip && jp) {
            const double v = h2.v[l] - c2.v[l] * ((ey0.v[l] - eyB.v[l]) - (ex0.v[l] - exD.v[l]));
            h2.v[l] = (k < g.nz) ? v : v * 0.0;
        }
    }
    if (jp) st2(hx + id, h0);
    if (ip) st2(hy + id, h1);
    if (ip && jp) st2(hz + id, h2);
}

// Thread -> pair: the whole grid in the order of row_quads.hpp (a stripe of every plane per
// XCD, so that the neighbour rows and planes are hits of its L2).
__device__ __forceinline__ bool pair_at(const RowQuads &m, PairAt &r)
{
    const int lane = threadIdx.x & 63;
    const QuadAt a = row_quad(m, blockIdx.x, threadIdx.x);
    r.i = a.i;
    r.j = a.j;
    r.k0 = 2 * a.q;
    r.next = a.next && lane < 63;
    r.prev = a.prev && lane > 0;
    return a.active;
}

template <bool HC>
__global__ __launch_bounds__(kBlockD) void k_update_e_f64(GridF64 g, RowQuads m, double *ex, double *ey, double *ez,
                                                          const double *__restrict__ hx, const double *__restrict__ hy,
                                                          const double *__restrict__ hz, const double *__restrict__ cx,
                                                          const double *__restrict__ cy, const double *__restrict__ cz)
{
    PairAt r;
    if (pair_at(m, r)) e_pair<HC>(g, r, ex, ey, ez, hx, hy, hz, cx, cy, cz);
}

template <bool HC>
__global__ __launch_bounds__(kBlockD) void k_update_h_f64(GridF64 g, RowQuads m, const double *__restrict__ ex,
                                                          const double *__restrict__ ey, const double *__restrict__ ez,
                                                          double *hx, double *hy, double *hz,
                                                          const double *__restrict__ cx, const double *__restrict__ cy,
                                                          const double *__restrict__ cz)
{
    PairAt r;
    if (pair_at(m, r)) h_pair<HC>(g, r, ex, ey, ez, hx, hy, hz, cx, cy, cz);
}

// Coefficients of the memory-order kernels: the arrays, or 0.5 where c is null.
__device__ __forceinline__ D2 ldc_opt(const double *__restrict__ c, size_t id)
{
    return c ? ld2(c + id) : D2{{0.5, 0.5}};
}

// Memory order: the pairs [p0, p1), component after component (the split form, and the whole
// grid where its planes have too few rows for stripes).  There the stripes' order gains no
// cache hits, and holding a pair's 12 to 15 loads at once costs waves in flight: E + H, this /
// e_pair and h_pair in the whole-grid order / in memory order, 62x42x250 with CE 20.1 / 23.8 /
// 23.0 us, 120x64x128 23.8 / 26.0 / 25.4, 300x48x300 118 / 145 / 123; from 72 rows on the
// whole-grid order wins: 72x72x72 12.8 / 9.8, 201x150x123 99 / 81, 320^3 873 / 844.
__global__ __launch_bounds__(kBlockD) void k_range_e_f64(
    int nx, int ny, int nzp, int nz, unsigned p0, unsigned p1, unsigned P,
    double *__restrict__ ex, double *__restrict__ ey, double *__restrict__ ez,
    const double *__restrict__ hx, const double *__restrict__ hy, const double *__restrict__ hz,
    const double *__restrict__ cex, const double *__restrict__ cey, const double *__restrict__ cez)
{
    const unsigned f = p0 + blockIdx.x * kBlockD + threadIdx.x;  // pairs [p0, p1) of the grid
    if (f >= p1) return;
    const unsigned row = f / P;
    const int k0 = (int)(f - row * P) * 2;
    const int i = (int)(row / (unsigned)ny);
    const int j = (int)row - i * ny;
    const size_t id = (size_t)row * nzp + k0;
    const size_t sx = (size_t)ny * nzp;

    const D2 hx0 = ld2(hx + id), hy0 = ld2(hy + id), hz0 = ld2(hz + id);
    if (j < ny - 1) {
        const D2 e = ld2(ex + id), c = ldc_opt(cex, id), h1 = ld2(hz + id + nzp);
        const double hyn = hy[id + 2];  // next row's first element on the last pair (row j+1 exists)
        D2 r;
#pragma unroll
        for (int l = 0; l < 2; l++) {
            const double h2 = l < 1 ? hy0.v[l + 1] : hyn;
            const double v = e.v[l] + c.v[l] * ((h1.v[l] - hz0.v[l]) - (h2 - hy0.v[l]));
            r.v[l] = (k0 + l < nz - 1) ? v : v * 0.0;
        }
        st2(ex + id, r);
    }
    if (i < nx - 1) {
        const D2 e = ld2(ey + id), c = ldc_opt(cey, id), h2 = ld2(hz + id + sx);
        const double hxn = hx[id + 2];
        D2 r;
#pragma unroll
        for (int l = 0; l < 2; l++) {
            const double h1 = l < 1 ? hx0.v[l + 1] : hxn;
            const double v = e.v[l] + c.v[l] * ((h1 - hx0.v[l]) - (h2.v[l] - hz0.v[l]));
            r.v[l] = (k0 + l < nz - 1) ? v : v * 0.0;
        }
        st2(ey + id, r);
        if (j < ny - 1) {
            const D2 e3 = ld2(ez + id), c3 = ldc_opt(cez, id), g1 = ld2(hy + id + sx), g2 = ld2(hx + id + nzp);
            D2 r3;
#pragma unroll
            for (int l = 0; l < 2; l++) {
                const double v = e3.v[l] + c3.v[l] * ((g1.v[l] - hy0.v[l]) - (g2.v[l] - hx0.v[l]));
                r3.v[l] = (k0 + l < nz) ? v : v * 0.0;
            }
            st2(ez + id, r3);
        }
    }
}

__global__ __launch_bounds__(kBlockD) void k_range_h_f64(
    int ny, int nzp, int nz, unsigned p0, unsigned p1, unsigned P,
    const double *__restrict__ ex, const double *__restrict__ ey, const double *__restrict__ ez,
    double *__restrict__ hx, double *__restrict__ hy, double *__restrict__ hz,
    const double *__restrict__ chx, const double *__restrict__ chy, const double *__restrict__ chz)
{
    const unsigned f = p0 + blockIdx.x * kBlockD + threadIdx.x;  // pairs [p0, p1) of the grid
    if (f >= p1) return;
    const unsigned row = f / P;
    const int k0 = (int)(f - row * P) * 2;
    const int i = (int)(row / (unsigned)ny);
    const int j = (int)row - i * ny;
    const size_t id = (size_t)row * nzp + k0;
    const size_t sx = (size_t)ny * nzp;

    const D2 ex0 = ld2(ex + id), ey0 = ld2(ey + id), ez0 = ld2(ez + id);
    if (j > 0) {
        const D2 h = ld2(hx + id), c = ldc_opt(chx, id), e1 = ld2(ez + id - nzp);
        const double eyp = ey[id - 1];  // previous row's last element when k0 == 0 (row j-1 exists)
        D2 r;
#pragma unroll
        for (int l = 0; l < 2; l++) {
            const double e2 = l > 0 ? ey0.v[l - 1] : eyp;
            const double v = h.v[l] - c.v[l] * ((ez0.v[l] - e1.v[l]) - (ey0.v[l] - e2));
            const int k = k0 + l;
            r.v[l] = (k > 0 && k < nz) ? v : v * 0.0;
        }
        st2(hx + id, r);
    }
    if (i > 0) {
        const D2 h = ld2(hy + id), c = ldc_opt(chy, id), e2 = ld2(ez + id - sx);
        const double exp_ = ex[id - 1];
        D2 r;
#pragma unroll
        for (int l = 0; l < 2; l++) {
            const double e1 = l > 0 ? ex0.v[l - 1] : exp_;
            const double v = h.v[l] - c.v[l] * ((ex0.v[l] - e1) - (ez0.v[l] - e2.v[l]));
            const int k = k0 + l;
            r.v[l] = (k > 0 && k < nz) ? v : v * 0.0;
        }
        st2(hy + id, r);
        if (j > 0) {
            const D2 h3 = ld2(hz + id), c3 = ldc_opt(chz, id), g1 = ld2(ey + id - sx), g2 = ld2(ex + id - nzp);
            D2 r3;
#pragma unroll
            for (int l = 0; l < 2; l++) {
                const double v = h3.v[l] - c3.v[l] * ((ey0.v[l] - g1.v[l]) - (ex0.v[l] - g2.v[l]));
                r3.v[l] = (k0 + l < nz) ? v : v * 0.0;
            }
            st2(hz + id, r3);
        }
    }
}

int check_grid_f64(int nx, int ny, int nzp, int pad)
{
    if (nx < 2 || ny < 2 || nzp < 2) return fail(MIFDTD_EINVAL, "grid (%d,%d,%d) too small", nx, ny, nzp);
    if (nzp % 2) return fail(MIFDTD_EALIGN, "nz_pitch %d is not a multiple of 2 (16-byte rows of doubles)", nzp);
    if (pad < 0 || pad > nzp - 2) return fail(MIFDTD_EINVAL, "pad %d invalid for nz_pitch %d", pad, nzp);
    const unsigned long long pairs = (unsigned long long)nx * ny * (nzp / 2);
    if (pairs >= (1ull << 31)) return fail(MIFDTD_ERANGE, "grid (%d,%d,%d) exceeds 2^31 pairs", nx, ny, nzp);
    return 0;
}

int launch_core_f64(bool e_half, int nx, int ny, int nzp, int pad, double *ex, double *ey, double *ez, double *hx,
                    double *hy, double *hz, const double *c0, const double *c1, const double *c2, hipStream_t st,
                    long long idx0 = 0, long long nmax = -1)
{
    if (int rc = check_grid_f64(nx, ny, nzp, pad)) return rc;
    const double *ptrs[6] = {ex, ey, ez, hx, hy, hz};
    for (const double *p : ptrs) {
        if (!p) return fail(MIFDTD_ENULL, "field pointer is NULL");
        if (!aligned16(p)) return fail(MIFDTD_EALIGN, "field pointer %p is not 16-byte aligned", (const void *)p);
    }
    if (c0 || c1 || c2) {
        if (!(c0 && c1 && c2)) return fail(MIFDTD_ENULL, "coefficient arrays must be all set or all NULL");
        if (!aligned16(c0) || !aligned16(c1) || !aligned16(c2))
            return fail(MIFDTD_EALIGN, "coefficient pointer is not 16-byte aligned");
    }
    const unsigned P = (unsigned)(nzp / 2);
    const unsigned npairs = (unsigned)nx * ny * P;
    const int nz = nzp - pad;
    const GridF64 g{nx, ny, nzp, nz};
    const bool hc = c0 != nullptr;
    unsigned p0 = 0, p1 = npairs;
    if (nmax >= 0) {  // the split form's element range, a pair per 2-element vector
        const long long n = 2ll * npairs;
        if (idx0 < 0 || idx0 > nmax || nmax > n)
            return fail(MIFDTD_EINVAL, "element range [%lld, %lld) outside the grid's %lld", idx0, nmax, n);
        if (idx0 % 2) return fail(MIFDTD_EALIGN, "idx0 %lld does not start a 2-element vector", idx0);
        p0 = (unsigned)(idx0 / 2);
        p1 = (unsigned)((nmax + 1) / 2);
        if (p1 == p0) return 0;
    }
    if (nmax >= 0 || ny < (int)kStripeMinRows) {
        const unsigned grid = (p1 - p0 + kBlockD - 1) / kBlockD;
        if (e_half) k_range_e_f64<<<grid, kBlockD, 0, st>>>(nx, ny, nzp, nz, p0, p1, P, ex, ey, ez, hx, hy, hz, c0, c1, c2);
        else k_range_h_f64<<<grid, kBlockD, 0, st>>>(ny, nzp, nz, p0, p1, P, ex, ey, ez, hx, hy, hz, c0, c1, c2);
        MIFDTD_CHECK_LAUNCH("update (double, memory order) launch");
        return 0;
    }
    const RowQuads m = grid_order(nx, ny, (int)P, nz, 0, 0);
    const unsigned grid = (unsigned)row_quads_blocks(m);
    if (e_half) {
        if (hc) k_update_e_f64<true><<<grid, kBlockD, 0, st>>>(g, m, ex, ey, ez, hx, hy, hz, c0, c1, c2);
        else k_update_e_f64<false><<<grid, kBlockD, 0, st>>>(g, m, ex, ey, ez, hx, hy, hz, c0, c1, c2);
    } else {
        if (hc) k_update_h_f64<true><<<grid, kBlockD, 0, st>>>(g, m, ex, ey, ez, hx, hy, hz, c0, c1, c2);
        else k_update_h_f64<false><<<grid, kBlockD, 0, st>>>(g, m, ex, ey, ez, hx, hy, hz, c0, c1, c2);
    }
    MIFDTD_CHECK_LAUNCH("update (double) launch");
    return 0;
}

}  // namespace

}  // namespace mifdtd

using namespace mifdtd;

extern "C" {

int mifdtd_update_e_f64(int nx, int ny, int nz_pitch, int pad, double *ex, double *ey, double *ez,
                        const double *hx, const double *hy, const double *hz,
                        const double *cex, const double *cey, const double *cez, mifdtd_stream_t stream)
{
    return launch_core_f64(true, nx, ny, nz_pitch, pad, ex, ey, ez, const_cast<double *>(hx), const_cast<double *>(hy),
                           const_cast<double *>(hz), cex, cey, cez, to_stream(stream));
}

int mifdtd_update_h_f64(int nx, int ny, int nz_pitch, int pad, const double *ex, const double *ey, const double *ez,
                        double *hx, double *hy, double *hz,
                        const double *chx, const double *chy, const double *chz, mifdtd_stream_t stream)
{
    return launch_core_f64(false, nx, ny, nz_pitch, pad, const_cast<double *>(ex), const_cast<double *>(ey),
                           const_cast<double *>(ez), hx, hy, hz, chx, chy, chz, to_stream(stream));
}

int mifdtd_update_e_f64_range(int nx, int ny, int nz_pitch, int pad, long long idx0, long long nmax, double *ex,
                              double *ey, double *ez, const double *hx, const double *hy, const double *hz,
                              const double *cex, const double *cey, const double *cez, mifdtd_stream_t stream)
{
    if (nmax < 0) return fail(MIFDTD_EINVAL, "nmax %lld < 0", nmax);
    return launch_core_f64(true, nx, ny, nz_pitch, pad, ex, ey, ez, const_cast<double *>(hx), const_cast<double *>(hy),
                           const_cast<double *>(hz), cex, cey, cez, to_stream(stream), idx0, nmax);
}

int mifdtd_update_h_f64_range(int nx, int ny, int nz_pitch, int pad, long long idx0, long long nmax,
                              const double *ex, const double *ey, const double *ez, double *hx, double *hy,
                              double *hz, const double *chx, const double *chy, const double *chz,
                              mifdtd_stream_t stream)
{
    if (nmax < 0) return fail(MIFDTD_EINVAL, "nmax %lld < 0", nmax);
    return launch_core_f64(false, nx, ny, nz_pitch, pad, const_cast<double *>(ex), const_cast<double *>(ey),
                           const_cast<double *>(ez), hx, hy, hz, chx, chy, chz, to_stream(stream), idx0, nmax);
}

}  // extern "C"
