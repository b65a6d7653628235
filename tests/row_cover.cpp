// Host-side check of the whole-grid passes' thread order (row_quads.hpp, the code the
// kernels use): for row counts, row lengths and CPML widths, the blocks' threads take every
// quad of every row exactly once, a quad at a z slab only in the slab runs, and the next /
// previous flags hold exactly where the neighbouring thread's quad follows / precedes in
// memory.  Exit status 0 when all hold.
#include "../fdtd_accelerate_amd/csrc/row_quads.hpp"

#include <cstdio>
#include <vector>

using namespace mifdtd;

static int check(unsigned planes, unsigned ny, int nz, int nzp, int npml)
{
    const unsigned Q = (unsigned)nzp / 4, nrows = planes * ny;
    const RowQuads m = row_quads(planes, ny, Q, nz, npml);
    const unsigned nb = (unsigned)row_quads_blocks(m);
    std::vector<int> hits((size_t)nrows * Q, 0);
    for (unsigned b = 0; b < nb; ++b) {
        for (unsigned t = 0; t < 256; ++t) {
            const QuadAt a = row_quad(m, b, t);
            if (!a.active) continue;
            if (a.i < 0 || (unsigned)a.i >= planes || a.j < 0 || (unsigned)a.j >= ny || a.q < 0 || (unsigned)a.q >= Q) {
                std::printf("out of bounds: block %u thread %u -> (%d, %d, %d) of (%u, %u, %u)\n", b, t, a.i, a.j, a.q, planes,
                            ny, Q);
                return 1;
            }
            ++hits[((size_t)a.i * ny + a.j) * Q + a.q];
            if (t + 1 < 256) {
                const QuadAt n = row_quad(m, b, t + 1);
                const bool follows = n.active && n.i == a.i && n.j == a.j && n.q == a.q + 1;
                if (a.next && !follows) { std::printf("next: block %u thread %u\n", b, t); return 1; }
                if (n.active && n.prev && !follows) { std::printf("prev: block %u thread %u\n", b, t + 1); return 1; }
                if (follows && a.next != n.prev) { std::printf("flags: block %u thread %u\n", b, t); return 1; }
            }
        }
    }
    for (size_t n = 0; n < hits.size(); ++n)
        if (hits[n] != 1) {
            std::printf("row %zu quad %zu taken %d times (rows %u, nz %d, nzp %d, npml %d)\n", n / Q, n % Q, hits[n], nrows, nz,
                        nzp, npml);
            return 1;
        }
    // the runs outside the slabs hold no cell of an E or H slab
    for (unsigned q = m.zf; q < m.zf + m.nin; ++q)
        for (int k = 4 * (int)q; k < 4 * (int)q + 4; ++k)
            if (npml && (k < npml || (k >= nz - 1 - npml && k < nz))) { std::printf("slab cell %d in a plain run\n", k); return 1; }
    return 0;
}

int main()
{
    const int nzs[][2] = {{4, 4}, {5, 8}, {18, 20}, {26, 32}, {33, 36}, {64, 64}, {65, 80}, {75, 76}, {123, 128}, {160, 160},
                          {193, 208}, {331, 336}, {1000, 1000}, {1024, 1024}, {1043, 1056}, {5000, 5008}};
    const unsigned rows[][2] = {{2, 2}, {1, 7}, {3, 63}, {2, 64}, {3, 65}, {5, 71}, {2, 130}, {1, 400}};
    const int npmls[] = {0, 1, 4, 8, 10, 12, 13};
    for (auto &z : nzs)
        for (auto &r : rows)
            for (int p : npmls)
                if (p == 0 || z[0] >= 2 * p + 2)
                    if (check(r[0], r[1], z[0], z[1], p)) return 1;
    if (check(2, 3, 262140, 262144, 8)) return 1;  // a row of more than 32768 quads
    std::printf("row cover ok\n");
    return 0;
}
