// The whole-grid passes (whole_pass.hpp) and the slab-ordered step: per time step, for each
// slab of consecutive x planes, one E pass (core E + CPML-E + E sources + E probes) then one
// H pass (core H + CPML-H + H sources + H probes) over that slab, in place; by default the
// slab is the whole grid (two launches per step).  Smaller slabs keep a slab's E/H planes in the last-level cache
// between its two passes, which on MI355X was measured to gain less than the extra
// launches cost.
//
// Ordering is the reference's (E of the slab before H of the slab; slabs in increasing
// x): H of plane i needs E_new of planes i and i-1 (done by this or the previous slab's
// E pass) and E of plane i needs H_old of planes i and i+1 (not yet touched: the slab's
// H pass runs after its E pass, the next slab's later).

#include "whole_pass.hpp"

namespace mifdtd {

// The tables of a half step that few waves read, as the kernel's first argument.
struct SExtra {
    SAux aux;
    SDrude dr;
    STfsf tf;
};

// CM: CeMode (kCeTable: CE from the material indices and the 3 x 256 table).  The
// sources and probes (first argument) are read only by the waves near them.  LDS: the table
// staged in LDS, for the core alone on arrays of many materials (200 of them, E pass alone:
// 208^3 60.2 -> 52.2 us, 433x380x56 60.2 -> 54.0, 266x169x245 81.5 -> 72.7); where most cells
// are one material it costs 0-5% (192^3 40.9 -> 41.5), with the CPML in the pass 1-3.5%.
template <int CM, bool PML, bool LDS = false>
__global__ __launch_bounds__(SB) void k_slab_e(SAux, SGeom g, SFields F, SCpml cp)
{
    __shared__ float tab[LDS ? 768 : 1];
    if (LDS) {
        for (int t = threadIdx.x; t < 768; t += SB) tab[t] = F.lut[t];
        __syncthreads();
    }
    RowAt r;
    if (!slab_quad(g, blockIdx.x, r)) return;
    e_quad_at<CM, PML>(g, r.i, r.j, r.k0, r.next, F.e[0], F.e[1], F.e[2], F.e[0], F.e[1], F.e[2], F.e[3], F.e[4],
                       F.e[5], F.ce[0], F.ce[1], F.ce[2], cp, first_kernel_arg<SAux>(), F.cm[0], F.cm[1], F.cm[2],
                       LDS ? tab : F.lut);
}

// With a Drude box and / or TFSF patches (FEAT; a grid without CPML has cp.axes 0).
template <int CM, int FEAT>
__global__ __launch_bounds__(SB) void k_slab_e_feat(SExtra, SGeom g, SFields F, SCpml cp)
{
    RowAt r;
    if (!slab_quad(g, blockIdx.x, r)) return;
    const SExtra &x = first_kernel_arg<SExtra>();
    e_quad_at<CM, true, FEAT>(g, r.i, r.j, r.k0, r.next, F.e[0], F.e[1], F.e[2], F.e[0], F.e[1], F.e[2], F.e[3], F.e[4],
                              F.e[5], F.ce[0], F.ce[1], F.ce[2], cp, x.aux, F.cm[0], F.cm[1], F.cm[2], F.lut, &x.dr,
                              &x.tf);
}

// With the curl of H on a design box stored: 160^3 cells with a box of 64^3 35.7 us, against
// 35.0 without and 5.1 for a pass of its own (mifdtd_design_curl).
struct SCurlArg {
    SAux aux;
    SCurl cu;
};
template <int CM, bool PML>
__global__ __launch_bounds__(SB) void k_slab_e_curl(SCurlArg, SGeom g, SFields F, SCpml cp)
{
    RowAt r;
    if (!slab_quad(g, blockIdx.x, r)) return;
    const SCurlArg &x = first_kernel_arg<SCurlArg>();
    e_quad_at<CM, PML, kFeatCurl>(g, r.i, r.j, r.k0, r.next, F.e[0], F.e[1], F.e[2], F.e[0], F.e[1], F.e[2], F.e[3],
                                  F.e[4], F.e[5], F.ce[0], F.ce[1], F.ce[2], cp, x.aux, F.cm[0], F.cm[1], F.cm[2], F.lut,
                                  nullptr, nullptr, nullptr, nullptr, nullptr, &x.cu);
}

// CH: F.ce holds the three CH arrays.
template <bool PML, bool CH>
__global__ __launch_bounds__(SB) void k_slab_h(SAux, SGeom g, SFields F, SCpml cp)
{
    RowAt r;
    if (!slab_quad(g, blockIdx.x, r)) return;
    h_quad_at<PML, CH>(g, r.i, r.j, r.k0, r.prev, F.e[0], F.e[1], F.e[2], F.e[3], F.e[4], F.e[5], F.e[3], F.e[4], F.e[5],
                       cp, first_kernel_arg<SAux>(), nullptr, nullptr, nullptr, nullptr, F.ce);
}

__global__ __launch_bounds__(SB) void k_slab_h_tfsf(SExtra, SGeom g, SFields F, SCpml cp)
{
    RowAt r;
    if (!slab_quad(g, blockIdx.x, r)) return;
    const SExtra &x = first_kernel_arg<SExtra>();
    h_quad_at<true>(g, r.i, r.j, r.k0, r.prev, F.e[0], F.e[1], F.e[2], F.e[3], F.e[4], F.e[5], F.e[3], F.e[4], F.e[5],
                    cp, x.aux, &x.tf);
}

template <int CM>
static void launch_e(const WholeGrid &w, unsigned grid, const SAux &a, const SDrude *dr, const STfsf *tf,
                     const SCurl *cu)
{
    if (cu) {
        const SCurlArg x{a, *cu};
        if (w.cp.npml > 0) k_slab_e_curl<CM, true><<<grid, SB, 0, w.st>>>(x, w.g, w.F, w.cp);
        else k_slab_e_curl<CM, false><<<grid, SB, 0, w.st>>>(x, w.g, w.F, w.cp);
        return;
    }
    if (!dr && !tf) {
        if (w.cp.npml > 0) k_slab_e<CM, true><<<grid, SB, 0, w.st>>>(a, w.g, w.F, w.cp);
        else if (CM == kCeTable && w.lds_table) k_slab_e<CM, false, CM == kCeTable><<<grid, SB, 0, w.st>>>(a, w.g, w.F, w.cp);
        else k_slab_e<CM, false><<<grid, SB, 0, w.st>>>(a, w.g, w.F, w.cp);
        return;
    }
    SExtra x{};
    x.aux = a;
    if (dr) x.dr = *dr;
    if (tf) x.tf = *tf;
    if (dr && tf) k_slab_e_feat<CM, kFeatDrude | kFeatTfsf><<<grid, SB, 0, w.st>>>(x, w.g, w.F, w.cp);
    else if (dr) k_slab_e_feat<CM, kFeatDrude><<<grid, SB, 0, w.st>>>(x, w.g, w.F, w.cp);
    else k_slab_e_feat<CM, kFeatTfsf><<<grid, SB, 0, w.st>>>(x, w.g, w.F, w.cp);
}

int whole_e(const WholeGrid &w, const SAux &a, const SDrude *dr, const STfsf *tf, const SCurl *cu)
{
    const unsigned grid = (unsigned)row_quads_blocks(w.g.m);
    if (w.cem == kCeTable) launch_e<kCeTable>(w, grid, a, dr, tf, cu);
    else if (w.cem == kCeArrays) launch_e<kCeArrays>(w, grid, a, dr, tf, cu);
    else launch_e<kCeConst>(w, grid, a, dr, tf, cu);
    MIFDTD_CHECK_LAUNCH("whole-grid E launch");
    return 0;
}

int whole_h(const WholeGrid &w, const SAux &a, const STfsf *tf, const float *const *ch)
{
    const unsigned grid = (unsigned)row_quads_blocks(w.g.m);
    if (tf) {
        SExtra x{};
        x.aux = a;
        x.tf = *tf;
        k_slab_h_tfsf<<<grid, SB, 0, w.st>>>(x, w.g, w.F, w.cp);
    } else if (ch) {
        SFields F = w.F;
        for (int c = 0; c < 3; c++) F.ce[c] = ch[c];
        if (w.cp.npml > 0) k_slab_h<true, true><<<grid, SB, 0, w.st>>>(a, w.g, F, w.cp);
        else k_slab_h<false, true><<<grid, SB, 0, w.st>>>(a, w.g, F, w.cp);
    } else if (w.cp.npml > 0) {
        k_slab_h<true, false><<<grid, SB, 0, w.st>>>(a, w.g, w.F, w.cp);
    } else {
        k_slab_h<false, false><<<grid, SB, 0, w.st>>>(a, w.g, w.F, w.cp);
    }
    MIFDTD_CHECK_LAUNCH("whole-grid H launch");
    return 0;
}

RowQuads grid_order(int nx, int ny, int Q, int nz, int npml_y, int npml_z)
{
    thread_local int key[6] = {0, 0, 0, 0, 0, 0};
    thread_local RowQuads m;
    const int want[6] = {nx, ny, Q, nz, npml_y, npml_z};
    bool same = true;
    for (int n = 0; n < 6; n++) same = same && key[n] == want[n];
    if (!same) {
        m = yee_order((unsigned)nx, (unsigned)ny, (unsigned)Q, nz, npml_y, npml_z);
        for (int n = 0; n < 6; n++) key[n] = want[n];
    }
    return m;
}

}  // namespace mifdtd

// =========================================================================== C ABI
using namespace mifdtd;

extern "C" {

int mifdtd_slab_run(const mifdtd_fused_desc *d, int slab_planes, int nsteps, const float *tvals,
                    float *probe_series, mifdtd_stream_t stream)
{
    if (!d) return fail(MIFDTD_ENULL, "step descriptor is NULL");
    const int nx = d->nx, ny = d->ny, nzp = d->nz_pitch, pad = d->pad;
    if (int rc = check_grid(nx, ny, nzp, pad)) return rc;
    if (slab_planes < 1) return fail(MIFDTD_EINVAL, "slab_planes must be >= 1 : %d", slab_planes);
    if (nsteps < 0) return fail(MIFDTD_EINVAL, "nsteps < 0");
    for (int c = 0; c < 6; c++) {
        if (!d->e[c]) return fail(MIFDTD_ENULL, "field buffer is NULL");
        if (!aligned16(d->e[c])) return fail(MIFDTD_EALIGN, "field buffer not 16-byte aligned");
    }
    const bool hc = d->ce[0] != nullptr;
    if (hc && (!d->ce[1] || !d->ce[2])) return fail(MIFDTD_ENULL, "CE arrays must be all set or all NULL");
    if (hc && (!aligned16(d->ce[0]) || !aligned16(d->ce[1]) || !aligned16(d->ce[2])))
        return fail(MIFDTD_EALIGN, "CE arrays not 16-byte aligned");
    const bool tbl = d->ce_mat[0] != nullptr;
    if (tbl) {
        if (!d->ce_mat[1] || !d->ce_mat[2] || !d->ce_lut)
            return fail(MIFDTD_ENULL, "CE material indices need all three index arrays and the table");
        for (int q = 0; q < 3; q++)
            if (reinterpret_cast<uintptr_t>(d->ce_mat[q]) & 3u)
                return fail(MIFDTD_EALIGN, "CE material index arrays not 4-byte aligned");
    }
    const int cem = tbl ? kCeTable : hc ? kCeArrays : kCeConst;
    const int nz = nzp - pad;
    if (d->nsrc < 0 || d->nsrc > MIFDTD_FUSED_MAX_SRC) return fail(MIFDTD_EINVAL, "nsrc outside [0,%d]", MIFDTD_FUSED_MAX_SRC);
    if (d->nprobe < 0 || d->nprobe > MIFDTD_FUSED_MAX_PROBE)
        return fail(MIFDTD_EINVAL, "nprobe outside [0,%d]", MIFDTD_FUSED_MAX_PROBE);
    if (d->nprobe && !probe_series) return fail(MIFDTD_ENULL, "probe_series is NULL");
    if (d->nsrc && !tvals) return fail(MIFDTD_ENULL, "tvals is NULL");

    SCpml cp{};
    const bool pml = d->npml > 0;
    if (pml) {
        const int np_ = d->npml;
        if (np_ > MIFDTD_MAX_NPML) return fail(MIFDTD_EINVAL, "npml %d > %d", np_, MIFDTD_MAX_NPML);
        if (nx < 2 * np_ + 2 || ny < 2 * np_ + 2 || nz < 2 * np_ + 2)
            return fail(MIFDTD_EINVAL, "grid (%d,%d,%d) too small for npml %d", nx, ny, nz, np_);
        if (!d->bE || !d->aE || !d->bH || !d->aH) return fail(MIFDTD_ENULL, "CPML tables are NULL");
        if (!d->psiE || !d->psiH) return fail(MIFDTD_ENULL, "packed psi buffers are NULL");
        if (!aligned16(d->psiE) || !aligned16(d->psiH))
            return fail(MIFDTD_EALIGN, "packed psi buffers not 16-byte aligned");
        cp.npml = np_;
        cp.axes = 7;
        cp.bE = d->bE;
        cp.aE = d->aE;
        cp.bH = d->bH;
        cp.aH = d->aH;
        cp.pe = d->psiE;
        cp.pe_out = d->psiE;
        cp.ph = d->psiH;
        cp.sX = (size_t)np_ * ny * nzp;
        cp.sY = (size_t)nx * np_ * nzp;
        cp.sZ = (size_t)nx * ny * np_;
    }
    for (int n = 0; n < d->nsrc; n++) {
        const int *b = d->src_box[n];
        if (d->src_comp[n] < 0 || d->src_comp[n] > 5) return fail(MIFDTD_EINVAL, "source %d component %d", n, d->src_comp[n]);
        if (b[0] < 0 || b[2] < 0 || b[4] < 0 || b[1] >= nx || b[3] >= ny || b[5] >= nzp || b[0] > b[1] || b[2] > b[3] ||
            b[4] > b[5])
            return fail(MIFDTD_EINVAL, "source box %d outside the grid", n);
    }
    SCurl cu{};
    if (d->design_curl) {
        const int *b = d->design_box;  // its cells' i+1, j+1, k+1 neighbours are cells of the grid
        if (b[0] < 0 || b[1] < 0 || b[2] < 0 || b[3] < 1 || b[4] < 1 || b[5] < 1 || b[3] >= nx - b[0] ||
            b[4] >= ny - b[1] || b[5] >= nz - b[2])
            return fail(MIFDTD_EINVAL, "design box outside the grid's inner cells");
        cu = SCurl{b[0], b[1], b[2], b[3], b[4], b[5], d->design_curl};
    }
    const size_t curl_step = 3 * (size_t)cu.di * cu.dj * cu.dk;
    // probes split by half step (E components 0..2 are final after the E pass)
    SProbe pe{}, ph{};
    for (int n = 0; n < d->nprobe; n++) {
        const int *p = d->probe_ijk[n];
        const int c = d->probe_comp[n];
        if (c < 0 || c > 5 || p[0] < 0 || p[0] >= nx || p[1] < 0 || p[1] >= ny || p[2] < 0 || p[2] >= nzp)
            return fail(MIFDTD_EINVAL, "probe %d outside the grid", n);
        SProbe &P = c < 3 ? pe : ph;
        const int m = P.n++;
        P.comp[m] = c;
        P.i[m] = p[0];
        P.j[m] = p[1];
        P.k[m] = p[2];
        P.slot[m] = n;
    }

    const unsigned Q = (unsigned)(nzp / 4);
    const unsigned long long plane_q = (unsigned long long)ny * Q;
    const int S = slab_planes < nx ? slab_planes : nx;
    if (plane_q * (unsigned long long)S + SB >= (1ull << 31)) return fail(MIFDTD_ERANGE, "slab of %d planes too large", S);
    hipStream_t st = to_stream(stream);
    SFields F{};
    for (int c = 0; c < 6; c++) F.e[c] = d->e[c];
    for (int c = 0; c < 3; c++) F.ce[c] = d->ce[c];
    if (tbl) {
        for (int c = 0; c < 3; c++) F.cm[c] = d->ce_mat[c];
        F.lut = d->ce_lut;
    }
    const int ns = (nx + S - 1) / S;
    auto geom = [&](int sl) {
        SGeom g;
        g.nx = nx;
        g.ny = ny;
        g.nzp = nzp;
        g.nz = nz;
        g.i0 = sl * S;
        g.m = yee_order((unsigned)(nx - g.i0 < S ? nx - g.i0 : S), (unsigned)ny, Q, nz, pml ? d->npml : 0, pml ? d->npml : 0);
        return g;
    };
    auto tables = [&](const SProbe &P, int step, bool e_half) {
        SAux A{};
        SSrc &X = A.src;
        for (int n = 0; n < d->nsrc; n++) {
            if ((d->src_comp[n] < 3) != e_half) continue;
            const int *b = d->src_box[n];
            const int m = X.n++;
            X.comp[m] = d->src_comp[n];
            X.i0[m] = b[0];
            X.i1[m] = b[1];
            X.j0[m] = b[2];
            X.j1[m] = b[3];
            X.k0[m] = b[4];
            X.k1[m] = b[5];
            X.sv[m] = d->src_sv[n];
            X.svs[m] = d->src_svs[n];
            X.ow[m] = d->src_overwrite[n];
            X.tval[m] = tvals[(size_t)step * d->nsrc + n];
        }
        A.prb = P;
        A.prb.out = d->nprobe ? probe_series + (size_t)step * d->nprobe : nullptr;
        aux_box(A);
        return A;
    };
    WholeGrid w{};
    w.F = F;
    w.cp = cp;
    w.cem = cem;
    w.st = st;
    for (int n = 0; n < nsteps; n++) {
        const SAux ae = tables(pe, n, true), ah = tables(ph, n, false);
        for (int sl = 0; sl < ns; sl++) {
            w.g = geom(sl);
            if (int rc = whole_e(w, ae, nullptr, nullptr, d->design_curl ? &cu : nullptr)) return rc;
            if (int rc = whole_h(w, ah, nullptr)) return rc;
        }
        cu.out += curl_step;
    }
    return 0;
}

}  // extern "C"
