// Thread -> quad order of the whole-grid passes (slab and batched engines), shared by the
// kernels and a host-side coverage check.
//
// Stripes: blocks are dealt round-robin to the 8 XCDs, each with its own L2.  Stripe x of
// every plane (an eighth of its rows) belongs to the blocks with blockIdx % 8 == x, plane
// after plane, so that the rows j+-1 and the plane i+-1 a quad reads are read again, or
// were read before, by blocks of the same L2.
//
// Groups: the quads of R consecutive rows of a stripe are taken by a whole number of
// 256-thread blocks: first the quads with no cell of a z CPML slab, row after row, then
// those of the z slabs.  A row of 64 to 256 cells is 16 to 64 quads, so with quads in plain
// row order every wave holds some z-slab lanes and issues the z slab's psi loads,
// arithmetic and stores for a few lanes; grouped, they fill waves of their own (at 160
// cells and npml 10: 6 of 40 quads a row, 2 of 10 waves instead of all).  R is the smallest
// group that leaves next to no idle thread.  Quads next to each other in a run are next to
// each other in memory too, so a lane finds its k+4 (k-1) neighbour in the next (previous)
// lane except at a run's end.
#pragma once

#include "common.hpp"

namespace mifdtd {

struct RowQuads {
    unsigned Q;         // quads per row
    unsigned R;         // rows per group
    unsigned bpg;       // blocks per group
    unsigned zf, zb;    // quads [0, zf) and [zb, Q) hold z-slab cells
    unsigned nin, nzq;  // quads per row outside / inside the z slabs
    unsigned m_in, m_z; // ceil(2^31 / nin), ceil(2^31 / nzq): division by multiplication
    unsigned planes;
    unsigned ns;        // stripes: 8, or 1 for planes of few rows
    unsigned jx[9];     // first row of each stripe, and ny
};

struct QuadAt {
    int i, j, q;        // plane, row and quad of the row
    bool active;        // a quad of the grid
    bool next, prev;    // the next / previous thread holds the next / previous quad
};

constexpr unsigned kStripes = 8;       // one per XCD
// Planes of fewer rows are one stripe: E + H pass of a cube with CPML 10, stripes against
// none, 56^3 14.3 / 14.2 us, 64^3 15.1 / 14.3, 80^3 18.9 / 24.3, 96^3 22.5 / 29.2, 112^3
// 28.4 / 33.3.
constexpr unsigned kStripeMinRows = 72;

// Quad of thread t of block b.
__host__ __device__ __forceinline__ QuadAt row_quad(const RowQuads &m, unsigned b, unsigned t)
{
    const unsigned x = b % m.ns, bs = b / m.ns;
    const unsigned jx = m.jx[x], S = m.jx[x + 1] - jx;  // the stripe's rows [jx, jx+S)
    const unsigned nrows = m.planes * S;
    const unsigned grp = bs / m.bpg, part = bs - grp * m.bpg;
    const unsigned row0 = grp * m.R;
    const unsigned rows = row0 >= nrows ? 0u : nrows - row0 < m.R ? nrows - row0 : m.R;
    const unsigned r = part * 256u + t;
    const unsigned n_in = rows * m.nin;
    QuadAt a;
    a.active = r < rows * m.Q;
    const bool in = r < n_in;
    const unsigned y = in ? r : r - n_in;
    const unsigned len = in ? m.nin : m.nzq, mg = in ? m.m_in : m.m_z;
    // y * len < 2^31 (row_quads below), so the product's high word is exactly y / len
    const unsigned rr = m.R == 1 ? 0u : (unsigned)(((unsigned long long)(2u * y) * mg) >> 32);
    const unsigned pos = y - rr * len;
    const unsigned z = pos < m.zf ? pos : pos - m.zf + m.zb;
    a.q = (int)(in ? m.zf + pos : z);
    a.next = pos + 1 < len && (in || pos + 1 != m.zf);
    a.prev = pos > 0 && (in || pos != m.zf);
    unsigned i = row0 / S, j = row0 - i * S + rr;
    while (j >= S) {  // at most R / S steps
        j -= S;
        ++i;
    }
    a.i = (int)i;
    a.j = (int)(jx + j);
    return a;
}

// The stripes' rows: equal shares of the rows' cost, a row of a y slab (psi read and
// written) costing 1.3 rows.  With equal row counts the first and the last XCD, which hold
// the y slabs, end last: 96^3 / 160^3 / 192^3 cells, CPML 10, E + H pass 25.3 / 75.6 / 153.0
// us; with 1.3, 24.3 / 74.2 / 148.5.
inline void stripe_rows(RowQuads &m, unsigned ny, int npml)
{
    const unsigned slab = npml > 0 ? (unsigned)npml : 0u;
    auto cost = [&](unsigned j) { return j < slab || j >= ny - slab ? 13u : 10u; };
    unsigned total = 0;
    for (unsigned j = 0; j < ny; ++j) total += cost(j);
    unsigned x = 0, sum = 0;
    for (unsigned j = 0; j < ny; ++j) {
        while (x < m.ns && (unsigned long long)sum * m.ns >= (unsigned long long)x * total) m.jx[x++] = j;
        sum += cost(j);
    }
    while (x <= 8) m.jx[x++] = ny;
}

// The order for `planes` planes of ny rows of Q quads (nz cells, npml-cell z slabs; npml =
// 0: none).  The E slabs are [0, npml) and [nz-1-npml, nz-1), the H slabs [0, npml) and
// [nz-npml, nz): one order serves both.  front: cells at the front that count as slab cells
// (the adjoint passes reach one cell further).
inline RowQuads row_quads(unsigned planes, unsigned ny, unsigned Q, int nz, int npml, int front = 0)
{
    RowQuads m;
    m.Q = Q;
    m.planes = planes;
    m.ns = ny >= kStripeMinRows ? kStripes : 1;
    stripe_rows(m, ny, npml);
    m.zf = npml > 0 ? (unsigned)(((front > npml ? front : npml) + 3) / 4) : 0u;
    m.zb = npml > 0 ? (unsigned)((nz - 1 - npml) / 4) : Q;
    if (m.zf >= m.zb) {  // every quad may hold a slab cell: one run
        m.zf = 0;
        m.zb = 0;
    }
    m.nin = m.zb - m.zf;
    m.nzq = Q - m.nin;
    // smallest R whose blocks leave at most 1 thread in 64 idle, else the R with the least
    unsigned best = 1;
    double waste = 2.0;
    for (unsigned R = 1; R <= 64 && (R == 1 || R * Q <= 32768u); ++R) {
        const unsigned n = R * Q, pad = (n + 255) / 256 * 256;
        const double w = (double)(pad - n) / pad;
        if (w < waste - 1e-9) {
            waste = w;
            best = R;
        }
        if (w <= 1.0 / 64) break;
    }
    m.R = best;
    m.bpg = (best * Q + 255) / 256;
    m.m_in = m.nin ? (unsigned)(((1ull << 31) + m.nin - 1) / m.nin) : 0u;
    m.m_z = m.nzq ? (unsigned)(((1ull << 31) + m.nzq - 1) / m.nzq) : 0u;
    return m;
}

// Blocks of a pass (a multiple of the stripes; the stripes' own counts differ by a row a plane).
inline unsigned long long row_quads_blocks(const RowQuads &m)
{
    unsigned long long S = 0;
    for (unsigned x = 0; x < m.ns; ++x) S = m.jx[x + 1] - m.jx[x] > S ? m.jx[x + 1] - m.jx[x] : S;
    return (m.planes * S + m.R - 1) / m.R * m.bpg * m.ns;
}

}  // namespace mifdtd
