// Launch interface of the XPBD per-colour projection kernels (oe_xpbd.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "oe_device.hpp"
#include "oe_elementwise.hpp"

namespace oe {

// Material ids as seen by device code (same values as oe::Material).
constexpr int NeoHooke_id = 2;
constexpr int Stable_NeoHooke_id = 3;

struct XpbdArgs {
    PSView ps;
    FemView fem;
    MaterialView mt;
    const int* eids;   // colour-major element list
    int first;         // first element of the colour
    int count;         // elements in the colour
    float dt;
    // linear tetrahedra: node ids and records (3 float4: JX_inv, V) of the
    // elements in the order of eids
    const int4* p1_nodes;
    const float4* p1_rec;
    const int* topo;   // the V2 form's node ids, S per element in the order of eids
};

// A whole run of substeps of a small linear-tetrahedron scene in one launch of
// one workgroup (k_xpbd_p1_resident).
constexpr int kXpbdResidentVertices = 2304;   // 28 bytes of LDS each, 63 KB
struct XpbdResidentArgs {
    PSView ps;
    MaterialView mt;
    const int4* nodes;        // as XpbdArgs::p1_nodes / p1_rec
    const float4* rec;
    const int* color_begin;   // n_colors + 1
    int n_colors;
    int substeps;
    VertexConstraints c;
    float dt;
    float global_damping;
    float g[3];
};
void launch_xpbd_p1_resident(const XpbdResidentArgs& a, hipStream_t s);

// v0_form selects the sqrt-constraint formulation with the fixed-vertex mask
// (reference kernel_XPBD_V0); otherwise the energy formulation of V1/V2.
bool launch_xpbd(int S, int Q, bool v0_form, const XpbdArgs& a, hipStream_t s);

}  // namespace oe
