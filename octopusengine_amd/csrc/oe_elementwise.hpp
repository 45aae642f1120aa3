// Launchers of the per-vertex integrator and constraint kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "oe_device.hpp"

namespace oe {

// Rigid target of the fixed vertices: target = offset + com + R (x0 - com).
struct FixTransform {
    float com[3];
    float offset[3];
    float R[9];   // column-major
};

// The constraints of an integrator that act on each vertex by itself: a
// fixation (per-vertex flag, null = none) and a box limit after it.
struct VertexConstraints {
    const unsigned char* fixed = nullptr;
    FixTransform t{};
    int has_box = 0;
    float lo[3] = {0.f, 0.f, 0.f}, hi[3] = {0.f, 0.f, 0.f};
    bool any() const { return fixed || has_box; }
};

void launch_vbd_predict(const PSView& ps, float4* y, float4* prev_it_p, float dt, const float g[3], hipStream_t s);
// What follows a VBD sweep, in one pass over the vertices and in this order:
// the constraints; the Chebyshev step (prev1 / prev2 set, iteration it); the
// velocity; the next substep's predictor.
struct VbdTailArgs {
    PSView ps;
    float4* y;
    float4* prev1;   // Chebyshev history, null = off
    float4* prev2;
    VertexConstraints c;
    int it;
    float omega;
    int velocity;
    int predict;
    float dt;
    float g[3];
};
void launch_vbd_tail(const VbdTailArgs& a, hipStream_t s);
void launch_semi_implicit(const PSView& ps, float dt, const float g[3], hipStream_t s);
// What follows the XPBD projections: constraints, velocity with the global
// damping, and (next) the semi-implicit step of the next substep.
void launch_pbd_tail(const PSView& ps, const VertexConstraints& c, float dt, float global_damping, bool next,
                     const float g[3], hipStream_t s);
void launch_fix(const PSView& ps, const int* ids, int n, const FixTransform& t, hipStream_t s);
void launch_box(const PSView& ps, const float pmin[3], const float pmax[3], hipStream_t s);
// Explicit integrator: each vertex's internal force from the element partials
// (explicit_partial(damping != 0) floats per (element, local node), owners
// order; nbo: incidence count and first partial of every vertex) and the
// damping term.  With gravity set, the semi-implicit update
// (launch_semi_implicit) of the vertex and the constraints follow in the same
// thread.
void launch_explicit_vertex(const PSView& ps, const int2* nbo, const float* partial, int count, float damping,
                            const float* gravity, const VertexConstraints& c, float dt, hipStream_t s);
void launch_copy_colour(const PSView& ps, const int* slot_vid, int first, int count, const float4* p_new,
                        hipStream_t s);
// Read-back: out[0 .. 3 count) = packed xyz of records first .. first + count
// (see Engine::read3); out is pinned host memory, 16-byte aligned.
void launch_pack3(const float4* rec, const float4* rest, float unit, int first, int count, float* out, hipStream_t s);

struct SceneDev;
// All vertices of one scene, covered by blocks [block_begin, next segment's
// block_begin) of a launch (block_begin is launch-local).
struct VSeg {
    int scene;
    int count;
    int block_begin;
};
struct BatchVArgs {
    const SceneDev* scenes;
    const VSeg* segs;   // one launch covers segs[0 .. nsegs)
    int nsegs;
    float dt;
    int iteration;
};
void launch_batch_predict(const BatchVArgs& b, int nblocks, hipStream_t s);
void launch_batch_fix_box(const BatchVArgs& b, int nblocks, hipStream_t s);
void launch_batch_velocity(const BatchVArgs& b, int nblocks, hipStream_t s);

}  // namespace oe
