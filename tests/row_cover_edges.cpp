// Host-side checks of row_quads.hpp beyond tests/row_cover.cpp: the orders with slab cells
// counted further at the front (the adjoint passes) and with rows off the 128-byte lines (the
// fused engine's placed fields), and the Yee passes' own, take every quad once, with exact neighbour flags and no slab
// cell in a plain run; and blocks past a stripe's rows find their row by an exact division.
// Exit status 0 when all hold.
#include "../fdtd_accelerate_amd/csrc/row_quads.hpp"

#include <cstdio>
#include <vector>

using namespace mifdtd;

static int cover(unsigned planes, unsigned ny, int nz, int nzp, int npml, int front, unsigned phase, int yee_y = -1)
{
    const unsigned Q = (unsigned)nzp / 4;
    const bool yee = yee_y >= 0;
    const RowQuads m = yee ? yee_order(planes, ny, Q, nz, yee_y, npml, phase) : row_quads(planes, ny, Q, nz, npml, front, phase);
    if (yee && m.R > kYeeRows) { std::printf("a group of %u rows: %u x %d, npml %d\n", m.R, ny, nz, npml); return 1; }
    const unsigned nb = (unsigned)row_quads_blocks(m);
    std::vector<int> hits((size_t)planes * ny * Q, 0);
    for (unsigned b = 0; b < nb; ++b)
        for (unsigned t = 0; t < 256; ++t) {
            const QuadAt a = row_quad(m, b, t);
            if (!a.active) continue;
            if (a.i < 0 || (unsigned)a.i >= planes || a.j < 0 || (unsigned)a.j >= ny || a.q < 0 || (unsigned)a.q >= Q) {
                std::printf("out of bounds: block %u thread %u\n", b, t);
                return 1;
            }
            ++hits[((size_t)a.i * ny + a.j) * Q + a.q];
            if (t == 255) continue;
            const QuadAt n = row_quad(m, b, t + 1);
            const bool follows = n.active && n.i == a.i && n.j == a.j && n.q == a.q + 1;
            if ((a.next || (n.active && n.prev)) && !follows) { std::printf("flag: block %u thread %u\n", b, t); return 1; }
            if (follows && a.next != n.prev) { std::printf("flags: block %u thread %u\n", b, t); return 1; }
        }
    for (int h : hits)
        if (h != 1) {
            std::printf("a quad taken %d times: %u x %u x %d (%d), npml %d, front %d, phase %u\n", h, planes, ny, nz, nzp, npml,
                        front, phase);
            return 1;
        }
    for (unsigned q = m.zf; npml && q < m.zf + m.nin; ++q)
        for (int k = 4 * (int)q; k < 4 * (int)q + 4; ++k)
            if (k < npml || k < front || (k >= nz - 1 - npml && k < nz)) { std::printf("slab cell %d in a plain run\n", k); return 1; }
    return 0;
}

// Grids whose stripes differ in rows, with as many planes as the reciprocal of the smaller
// stripe allows: a block past that stripe's rows must not loop over 2^32 / rows steps.
static int idle(unsigned planes, unsigned ny, unsigned Q, int nz, int npml)
{
    const RowQuads m = row_quads(planes, ny, Q, nz, npml);
    const unsigned long long per = row_quads_blocks(m) / kStripes;
    for (unsigned x = 0; x < m.ns; ++x) {
        const unsigned S = m.jx[x + 1] - m.jx[x];
        for (unsigned long long row = (unsigned long long)planes * S; row < per / m.bpg * m.R; row += row % S == S - 1 ? S : S - 1 - row % S)
            if (div_by((unsigned)row, S, m.m_s[x]) != row / S) {
                std::printf("%u x %u, %u quads, npml %d: stripe %u, row %llu / %u\n", planes, ny, Q, npml, x, row, S);
                return 1;
            }
    }
    return 0;
}

// Stripes: equal rows where the y axis has no slabs, whatever the z slabs, and smaller first and
// last ones where it has.
static int stripes(unsigned ny, int npml)
{
    const RowQuads a = yee_order(3, ny, 65, 258, 0, npml), b = yee_order(3, ny, 65, 258, npml, 0);
    for (unsigned x = 0; x < 8; ++x) {
        const unsigned S = a.jx[x + 1] - a.jx[x];
        if (S != ny / 8 && S != (ny + 7) / 8) { std::printf("stripe %u of %u rows: %u\n", x, ny, S); return 1; }
    }
    if (b.jx[1] >= a.jx[1] || ny - b.jx[7] >= ny - a.jx[7]) { std::printf("y slabs of %u rows not weighted\n", ny); return 1; }
    return 0;
}

int main()
{
    const int nzs[][2] = {{26, 32}, {33, 36}, {64, 64}, {75, 76}, {123, 128}, {160, 160}, {258, 260}, {331, 336}, {1043, 1056}};
    const unsigned rows[][2] = {{3, 65}, {5, 71}, {2, 130}, {1, 400}, {9, 12}};
    for (auto &z : nzs)
        for (auto &r : rows)
            for (int p : {1, 4, 8, 10, 12})
                if (z[0] >= 2 * p + 2)
                    for (unsigned phase = 0; phase < 8; ++phase) {
                        if (cover(r[0], r[1], z[0], z[1], p, 0, phase)) return 1;
                        if (cover(r[0], r[1], z[0], z[1], p, 0, phase, phase % 2 ? p : 0)) return 1;
                        if (phase == 0 && cover(r[0], r[1], z[0], z[1], p, p + 1, 0)) return 1;
                    }
    for (unsigned ny : {200u, 240u, 333u, 491u})
        if (stripes(ny, 12)) return 1;
    if (idle(14861237, 144, 1, 4, 1) || idle(1651195, 414, 3, 10, 4) || idle(1651195, 414, 3, 12, 5)) return 1;
    std::printf("row cover edges ok\n");
    return 0;
}
