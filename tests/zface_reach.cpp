// Host-side check of the z-face psi loads of the whole-grid passes (zface_at of
// step_quad.hpp, the code the kernels use): with CPML on z alone, every cell of every quad
// that meets a z slab, in a slab or not, loads inside the z faces' part of the packed psi
// buffer, and a cell in a slab loads its own psi.  Exit status 0 when all hold.
#include "../fdtd_accelerate_amd/csrc/step_quad.hpp"

#include <cstdio>

using namespace mifdtd;

template <bool E>
static int check(int nx, int ny, int nz, int nzp, int npml)
{
    SCpml cp{};
    cp.npml = npml;
    cp.axes = 4;
    cp.sX = (size_t)npml * ny * nzp;
    cp.sY = (size_t)nx * npml * nzp;
    cp.sZ = (size_t)nx * ny * npml;
    const size_t first = cp.off(4, 0), end = first + 4 * cp.sZ;
    const int back = E ? nz - 1 - npml : nz - npml;
    for (int i = 0; i < nx; ++i)
        for (int j = 0; j < ny; ++j)
            for (int k0 = 0; k0 < nzp; k0 += 4) {
                if (!(k0 < npml || (k0 + 3 >= back && k0 < nz - (E ? 1 : 0)))) continue;  // the passes' test
                for (int l = 0; l < 4; ++l) {
                    size_t o;
                    const int k = k0 + l, t = zface_at<E>(cp, i, j, k0, l, ny, nz, o);
                    const bool front = k < npml && (E || k > 0), rear = k >= back && k < nz - (E ? 1 : 0);
                    if ((t > 0) != (front || rear) || o < first || o + cp.sZ >= end) {
                        std::printf("%s cell (%d, %d, %d) of nz %d, npml %d: entry %d, offset %zu outside [%zu, %zu)\n",
                                    E ? "E" : "H", i, j, k, nz, npml, t, o, first, end);
                        return 1;
                    }
                    const size_t row = ((size_t)i * ny + j) * npml;
                    if (t > 0 && o != cp.off(front ? 4 : 5, 0) + row + (front ? k : k - back)) {
                        std::printf("%s cell (%d, %d, %d): offset %zu\n", E ? "E" : "H", i, j, k, o);
                        return 1;
                    }
                }
            }
    return 0;
}

int main()
{
    for (int npml = 1; npml <= 13; ++npml)
        for (int nz = 2 * npml + 2; nz < 2 * npml + 40; ++nz)
            for (int pitch = (nz + 3) / 4 * 4; pitch <= nz + 12; pitch += 4)
                if (check<true>(3, 4, nz, pitch, npml) || check<false>(3, 4, nz, pitch, npml)) return 1;
    std::printf("zface reach ok\n");
    return 0;
}
