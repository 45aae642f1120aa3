// Device code of what a pass does to one vertex by itself: the fixation and
// the box limit (on plain and on compensated records) and the XPBD velocity.
//   XPBD velocity + damping   src/GPU/PBD/GPU_PBD.cu:8-18
//   fixed vertices            src/GPU/GPU_Constraint.cu:8-19
//   box limit                 src/GPU/GPU_Constraint.cu:70-81
#pragma once

#include "oe_device.hpp"
#include "oe_elementwise.hpp"

namespace oe {

// v += (g + f w) dt ; p += v dt, with its roundings written out (several
// kernels hold it).
__device__ __forceinline__ void semi_implicit(float4& p, float4& v, const float4& f, float w, float dt, float gx,
                                              float gy, float gz) {
    v.x = fmaf(fmaf(f.x, w, gx), dt, v.x);
    v.y = fmaf(fmaf(f.y, w, gy), dt, v.y);
    v.z = fmaf(fmaf(f.z, w, gz), dt, v.z);
    p.x = fmaf(v.x, dt, p.x);
    p.y = fmaf(v.y, dt, p.y);
    p.z = fmaf(v.z, dt, p.z);
}

// v = (p - last_p) / dt, damped
__device__ __forceinline__ void pbd_velocity_of(float4 p, float4 lp, float w, float dt, float global_damping,
                                                float v[3]) {
    float vx = (p.x - lp.x) / dt, vy = (p.y - lp.y) / dt, vz = (p.z - lp.z) / dt;
    const float nv = sqrtf(fmaf(vz, vz, fmaf(vy, vy, vx * vx)));
    if (nv > 1e-7f) {
        const float coef = global_damping * dt * w;
        const float damp = -nv * (coef > 1.f ? 1.f : coef);
        const float inv = 1.f / nv;
        vx = fmaf(vx * inv, damp, vx);
        vy = fmaf(vy * inv, damp, vy);
        vz = fmaf(vz * inv, damp, vz);
    }
    v[0] = vx;
    v[1] = vy;
    v[2] = vz;
}

// target = offset + com + R (X - com), X = init_p (rest position);  p = target,
// v = f = 0, mask = 0.  p holds the displacement x - X, so the stored value is
// offset + (R d - d) with d = X - com (exactly offset when R = I), with no
// low-order part (w = 0).
__device__ __forceinline__ float4 fix_displacement(float4 X, const float com[3], const float off[3], const float R[9]) {
    const float dx = X.x - com[0], dy = X.y - com[1], dz = X.z - com[2];
    // R is column-major; R d = col0 dx + col1 dy + col2 dz
    const float rx = R[0] * dx + R[3] * dy + R[6] * dz;
    const float ry = R[1] * dx + R[4] * dy + R[7] * dz;
    const float rz = R[2] * dx + R[5] * dy + R[8] * dz;
    return make_float4(off[0] + (rx - dx), off[1] + (ry - dy), off[2] + (rz - dz), 0.f);
}

// clamp the absolute position X + u into [pmin, pmax]; u is rewritten only
// when a component is clamped, and the return value says whether one was
__device__ __forceinline__ bool box_clamp(float4& u, float4 X, const float pmin[3], const float pmax[3]) {
    const float x = X.x + u.x, y = X.y + u.y, z = X.z + u.z;
    const bool cx = x < pmin[0] || x > pmax[0], cy = y < pmin[1] || y > pmax[1], cz = z < pmin[2] || z > pmax[2];
    if (cx) u.x = fminf(fmaxf(x, pmin[0]), pmax[0]) - X.x;
    if (cy) u.y = fminf(fmaxf(y, pmin[1]), pmax[1]) - X.y;
    if (cz) u.z = fminf(fmaxf(z, pmin[2]), pmax[2]) - X.z;
    return cx || cy || cz;
}

// The compensated form: the absolute position X + (hi + lo) in FP64 against the
// box; a clamped component becomes bound - X (packed again).  True when a
// component is clamped.
__device__ __forceinline__ bool box_clamp_comp(float4& h, float unit, float inv, float4 X, const float pmin[3],
                                               const float pmax[3]) {
    // the low-order part (|lo| <= half an ulp of hi) can only matter within a
    // relative 1e-4 of a bound: elsewhere the float sum decides alone
    const float xf[3] = {X.x + h.x, X.y + h.y, X.z + h.z};
    bool near = false;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        near = near || xf[k] < pmin[k] + 1e-4f * (1.f + fabsf(pmin[k])) ||
               xf[k] > pmax[k] - 1e-4f * (1.f + fabsf(pmax[k]));
    if (!near) return false;
    dvec3 U = dunpack(h, unit);
    const double x = X.x + U.x, y = X.y + U.y, z = X.z + U.z;
    const bool cx = x < pmin[0] || x > pmax[0], cy = y < pmin[1] || y > pmax[1], cz = z < pmin[2] || z > pmax[2];
    if (!(cx || cy || cz)) return false;
    if (cx) U.x = fmin(fmax(x, static_cast<double>(pmin[0])), static_cast<double>(pmax[0])) - X.x;
    if (cy) U.y = fmin(fmax(y, static_cast<double>(pmin[1])), static_cast<double>(pmax[1])) - X.y;
    if (cz) U.z = fmin(fmax(z, static_cast<double>(pmin[2])), static_cast<double>(pmax[2])) - X.z;
    h = dpack(U, inv);
    return true;
}

// Fixation then box limit of one vertex whose record is u: a fixed vertex
// (flag set) is snapped and masked, every other vertex with mask 1 is clamped -
// the same result as k_fix then k_box, since the box skips masked vertices.
// True when u changed; v, f and mask of a fixed vertex are stored here.
__device__ __forceinline__ bool constrain(const PSView& ps, int i, float4& u, bool is_fixed, int mask, float4 X,
                                          const float com[3], const float off[3], const float R[9], int has_box,
                                          const float lo[3], const float hi[3]) {
    if (is_fixed) {
        u = fix_displacement(X, com, off, R);
        gstore(ps.v, i, make_float4(0.f, 0.f, 0.f, 0.f));
        gstore(ps.f, i, make_float4(0.f, 0.f, 0.f, 0.f));
        gstore(ps.mask, i, 0);
        return true;
    }
    if (!has_box || mask == 0) return false;
    return ps.comp ? box_clamp_comp(u, ps.lo_unit, ps.lo_inv, X, lo, hi) : box_clamp(u, X, lo, hi);
}

// The same for one scene's constraints; the flag, the mask and the rest
// position are loaded together (waiting on one another they cost three
// round trips).
__device__ __forceinline__ bool constrain(const PSView& ps, int i, float4& u, const VertexConstraints& c) {
    if (!c.fixed && !c.has_box) return false;
    const bool is_fixed = c.fixed && gload(c.fixed, i) != 0;
    const int mask = gload(static_cast<const int*>(ps.mask), i);
    const float4 X = gload(static_cast<const float4*>(ps.init_p), i);
    return constrain(ps, i, u, is_fixed, mask, X, c.t.com, c.t.offset, c.t.R, c.has_box, c.lo, c.hi);
}

}  // namespace oe
