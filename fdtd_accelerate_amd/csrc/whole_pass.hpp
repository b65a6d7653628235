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
    hipStream_t st;
};

// E pass, then H pass, each in place; dr / tf: null where the step has none.
int whole_e(const WholeGrid &w, const SAux &a, const SDrude *dr, const STfsf *tf);
int whole_h(const WholeGrid &w, const SAux &a, const STfsf *tf);

}  // namespace mifdtd
