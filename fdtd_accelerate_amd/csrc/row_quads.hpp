// Thread -> quad order of the whole-grid passes, shared by the
// kernels and a host-side coverage check.
//
// Stripes: blocks are dealt round-robin to the 8 XCDs, each with its own L2.  Stripe x of
// every plane (an eighth of its rows) belongs to the blocks with blockIdx % 8 == x, plane
// after plane, so that the rows j+-1 and the plane i+-1 a quad reads are read again, or
// were read before, by blocks of the same L2.
//
// Groups: the quads of R consecutive rows of a stripe are taken by a whole number of
// 256-thread blocks: first the lines (8 quads) with no cell of a z CPML slab, row after row,
// then those at the rows' ends with the z slabs.  A row of 64 to 256 cells is 16 to 64
// quads, so with quads in plain row order every wave holds some z-slab lanes and issues the
// z slab's psi loads, arithmetic and stores for a few lanes.  Runs cut within a line make
// two waves fetch it.  E + H, CPML 10, 128^3 / 256^3 / 320^3 / 448^3 / 512^3: cut at lines 37.1 /
// 261 / 494 / 1297 / 1872 us, at the slab 38.3 / 278 / 528 / 1358 / 1970, plain row order 38.8 /
// 266 / 510 / 1334 / 1892.  R is the smallest group that leaves next to no idle thread, within
// the caller's limit (yee_order).  Quads next to each other in a run are next to each other in
// memory too, so a lane finds its k+4 (k-1) neighbour in the next (previous) lane except at a
// run's end.
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
    unsigned m_b;       // ceil(2^32 / bpg), 0: divide (grids of more than 2^32 / bpg blocks)
    unsigned m_s[8];    // the same of each stripe's rows per plane
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

// n / d by d's reciprocal r = ceil(2^32 / d) where n * d < 2^32 (then exact), by division
// where r is 0.  Block indices are uniform: a division costs the wave some 20 instructions.
__host__ __device__ __forceinline__ unsigned div_by(unsigned n, unsigned d, unsigned r)
{
    return r ? (unsigned)(((unsigned long long)n * r) >> 32) : n / d;
}
inline unsigned reciprocal(unsigned long long n_max, unsigned d)
{
    if (d < 2 || n_max * d >= (1ull << 32)) return 0u;
    return (unsigned)(((1ull << 32) + d - 1) / d);
}

// Quad of thread t of block b.
__host__ __device__ __forceinline__ QuadAt row_quad(const RowQuads &m, unsigned b, unsigned t)
{
    const unsigned x = m.ns == kStripes ? b & (kStripes - 1) : 0u, bs = m.ns == kStripes ? b / kStripes : b;
    const unsigned jx = m.jx[x], S = m.jx[x + 1] - jx;  // the stripe's rows [jx, jx+S)
    const unsigned nrows = m.planes * S;
    const unsigned grp = div_by(bs, m.bpg, m.m_b), part = bs - grp * m.bpg;
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
    unsigned i = div_by(row0, S, m.m_s[x]), j = row0 - i * S + rr;
    while (j >= S) {  // at most R / S steps
        j -= S;
        ++i;
    }
    a.i = (int)i;
    a.j = (int)(jx + j);
    return a;
}

constexpr unsigned kEqualRows = 512;

// The stripes' rows: equal shares of the rows' cost, a row of a y slab (psi read and
// written) costing 1.3 rows.  With equal row counts the first and the last XCD, which hold
// the y slabs, end last: E + H, CPML 10, equal rows / 1.3, 256^3 271 / 261 us, 300x288x300 427 /
// 402, 448^3 1327 / 1300, 200x480x300 454 / 439.  Planes of kEqualRows rows and more take equal
// stripes: the 4th-order step at 512^3 10.86 ms against 11.10 (256^3 1.47 / 1.44), the Yee passes
// at 512^3 1870 us against 1890; flatter grids would still gain by 1.3 (200x512x300 481 / 469,
// 150x600x256 354 / 352, 150x768x224 412 / 398).
inline void stripe_rows(RowQuads &m, unsigned ny, int npml)
{
    const unsigned slab = npml > 0 ? (unsigned)npml : 0u;
    const unsigned slab_cost = ny >= kEqualRows ? 10u : 13u;
    auto cost = [&](unsigned j) { return j < slab || j >= ny - slab ? slab_cost : 10u; };
    unsigned total = 0;
    for (unsigned j = 0; j < ny; ++j) total += cost(j);
    unsigned x = 0, sum = 0;
    for (unsigned j = 0; j < ny; ++j) {
        while (x < m.ns && (unsigned long long)sum * m.ns >= (unsigned long long)x * total) m.jx[x++] = j;
        sum += cost(j);
    }
    while (x <= 8) m.jx[x++] = ny;
}

// Rows per plane of the largest stripe.
inline unsigned long long stripe_max(const RowQuads &m)
{
    unsigned S = 0;
    for (unsigned x = 0; x < m.ns; ++x) S = m.jx[x + 1] - m.jx[x] > S ? m.jx[x + 1] - m.jx[x] : S;
    return S;
}

// Blocks of a pass (a multiple of the stripes; the stripes' own counts differ by a row a plane).
inline unsigned long long row_quads_blocks(const RowQuads &m)
{
    return (m.planes * stripe_max(m) + m.R - 1) / m.R * m.bpg * m.ns;
}

// The order for `planes` planes of ny rows of Q quads (nz cells, npml-cell z slabs; npml =
// 0: none).  The E slabs are [0, npml) and [nz-1-npml, nz-1), the H slabs [0, npml) and
// [nz-npml, nz): one order serves both.  front: cells at the front that count as slab cells
// (the adjoint passes reach one cell further).  phase: quads from a 128-byte line to each
// row's first quad.  max_rows: the most rows of a group.  npml_y: y slabs of another width
// than the z slabs (a grid with CPML on one of the two axes); -1: the same.
inline RowQuads row_quads(unsigned planes, unsigned ny, unsigned Q, int nz, int npml, int front = 0, unsigned phase = 0,
                          unsigned max_rows = 64, int npml_y = -1)
{
    RowQuads m;
    m.Q = Q;
    m.planes = planes;
    m.ns = ny >= kStripeMinRows ? kStripes : 1;
    stripe_rows(m, ny, npml_y < 0 ? npml : npml_y);
    m.zf = npml > 0 ? (unsigned)(((front > npml ? front : npml) + 3) / 4) : 0u;
    m.zb = npml > 0 ? (unsigned)((nz - 1 - npml) / 4) : Q;
    if (npml > 0) {  // whole 128-byte lines (8 quads) on either side of a run's end
        m.zf = (m.zf + phase + 7) / 8 * 8 - phase;
        m.zb = m.zb + phase < 8 ? 0 : (m.zb + phase) / 8 * 8 - phase;
    }
    if (m.zf >= m.zb) {  // every quad may hold a slab cell: one run
        m.zf = 0;
        m.zb = 0;
    }
    m.nin = m.zb - m.zf;
    m.nzq = Q - m.nin;
    // smallest R whose blocks leave at most 1 thread in 64 idle, else the R with the least
    unsigned best = 1;
    double waste = 2.0;
    for (unsigned R = 1; R <= max_rows && (R == 1 || R * Q <= 32768u); ++R) {
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
    m.m_b = reciprocal(row_quads_blocks(m) + kStripes, m.bpg);
    for (unsigned x = 0; x < 8; ++x) {
        const unsigned S = m.jx[x + 1] - m.jx[x];
        // (the largest stripe's blocks: those past this stripe's rows divide by S too)
        m.m_s[x] = reciprocal(planes * stripe_max(m) + 64 * m.R, S);
    }
    return m;
}

// The order of a Yee E or H pass (npml_y, npml_z: 0 on an axis without CPML).  With CPML a
// group's z-slab runs follow the runs of all its rows: at pitches off the lines a large group
// fetches the lines at the runs' ends twice.
// E + H, CPML 10, groups of up to 64 / 8 / 2 rows: 341x240x258 424 / 379 / 383 us, 333x491x357
// 1053 / 907 / 896, 448^3 1398 / 1298 / 1300, 352^3 673 / 641 / 645, 128^3 36.0 / 36.7 / 38.9,
// 300x300x250 356 / 355 / 365.  The 4th-order stages and the adjoint passes keep 64 (8: 400 x
// 300 x 200 2145 -> 2345 us a step, 160^3 128.9 -> 130.9 ms).
constexpr unsigned kYeeRows = 8;
inline RowQuads yee_order(unsigned planes, unsigned ny, unsigned Q, int nz, int npml_y, int npml_z, unsigned phase = 0)
{
    return row_quads(planes, ny, Q, nz, npml_z, 0, phase, npml_z > 0 ? kYeeRows : 64, npml_y);
}

}  // namespace mifdtd
