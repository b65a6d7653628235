// Launches of the whole-grid passes (slab.hip) for the engines that step in place: one
// thread per quad in the order of row_quads.hpp, each half step with its CPML, sources,
// probes and, where given, a Drude box and TFSF patches.
#pragma once

#include "step_quad.hpp"

namespace mifdtd {

struct WholeGrid {
    SGeom g;        // with its thread order
    SFields F;
    SCpml cp;       // npml 0: none
    int cem;        // CeMode: constant, arrays or table
    bool lds_table; // the table staged in LDS (E passes without CPML)
    hipStream_t st;
};

// No sources and probes.
inline SAux no_aux()
{
    SAux a{};
    aux_box(a);
    return a;
}

// E pass, then H pass, each in place; dr / tf / cu: null where the step has none (cu goes
// without the others); ch: the three CH arrays, null for the constant 0.5 (which a step with tf
// has).
int whole_e(const WholeGrid &w, const SAux &a, const SDrude *dr, const STfsf *tf, const SCurl *cu = nullptr);
int whole_h(const WholeGrid &w, const SAux &a, const STfsf *tf, const float *const *ch = nullptr);

// yee_order of the whole grid of Q units of 16 bytes per row; the last one a thread asked for
// is kept.
RowQuads grid_order(int nx, int ny, int Q, int nz, int npml_y, int npml_z);

}  // namespace mifdtd
