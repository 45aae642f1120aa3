// Per-vertex kernels of the integrators and constraints.  Each is one pass
// over SoA particle state with coalesced 16-byte accesses; they are launch- or
// HBM-bound and carry no reuse.  Positions are stored as displacements from
// the rest position (init_p); the integrators are linear in the positions and
// read them unchanged, the constraints convert to absolute positions.
//   VBD predictor             src/GPU/VBD/GPU_VBD.cu:6-18
//   VBD velocity              src/GPU/VBD/GPU_VBD.cu:20-25
//   Chebyshev acceleration    src/GPU/VBD/GPU_VBD.cu:27-35
//   semi-implicit Euler       src/GPU/GPU_Integrator.cu:27-34
//   XPBD velocity + damping   src/GPU/PBD/GPU_PBD.cu:8-18
//   fixed vertices            src/GPU/GPU_Constraint.cu:8-19
//   box limit                 src/GPU/GPU_Constraint.cu:70-81
//   Jacobi colour copy        src/GPU/VBD/GPU_VBD_FEM.cu:402-413
#include "oe_elementwise.hpp"
#include "oe_gather.hpp"
#include "oe_kernels.hpp"
#include "oe_vertex.hpp"

namespace oe {

namespace {

constexpr int kBlock = 256;
inline int grid_for(long long n) { return static_cast<int>((n + kBlock - 1) / kBlock); }

__device__ __forceinline__ float4 f4(float x, float y, float z, float w) { return make_float4(x, y, z, w); }

// y = p + ((p - last_p) / dt + (g + f w) dt) dt ; last_p = p ; p = y, on the
// compensated state in FP64.
__device__ __forceinline__ void vbd_predict_from(const PSView& ps, float4* y, int i, float4 p, float4 last_p, float4 f,
                                                 float w, float dt, float gx, float gy, float gz, float4* prev_it_p) {
    const dvec3 P = dunpack(p, ps.lo_unit), LP = dunpack(last_p, ps.lo_unit);
    if (prev_it_p) prev_it_p[i] = p;
    const double ddt = dt;
    const double ax = gx + static_cast<double>(f.x) * w, ay = gy + static_cast<double>(f.y) * w,
                 az = gz + static_cast<double>(f.z) * w;
    const float4 Y = dpack(dvec3{P.x + ((P.x - LP.x) / ddt + ax * ddt) * ddt, P.y + ((P.y - LP.y) / ddt + ay * ddt) * ddt,
                                 P.z + ((P.z - LP.z) / ddt + az * ddt) * ddt},
                           ps.lo_inv);
    y[i] = Y;
    ps.last_p[i] = p;
    ps.p[i] = Y;
}

// the same from the stored state; f = 0 after it
__device__ __forceinline__ void vbd_predict_one(const PSView& ps, float4* y, int i, float dt, float gx, float gy,
                                                float gz, float4* prev_it_p) {
    const float4 p = ps.p[i], f = ps.f[i];
    const float w = ps.w[i];
    vbd_predict_from(ps, y, i, p, ps.last_p[i], f, w, dt, gx, gy, gz, prev_it_p);
    ps.f[i] = f4(0.f, 0.f, 0.f, 0.f);
}

__global__ __launch_bounds__(kBlock) void k_vbd_predict(PSView ps, float4* y, float4* prev_it_p, float dt, float gx,
                                                        float gy, float gz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ps.n) return;
    vbd_predict_one(ps, y, i, dt, gx, gy, gz, prev_it_p);
}

// v = (p - last_p) / dt
__device__ __forceinline__ void vbd_velocity_from(const PSView& ps, int i, float4 p, float4 last_p, float dt) {
    const dvec3 P = dunpack(p, ps.lo_unit), LP = dunpack(last_p, ps.lo_unit);
    const double ddt = dt;
    ps.v[i] = f4(static_cast<float>((P.x - LP.x) / ddt), static_cast<float>((P.y - LP.y) / ddt),
                 static_cast<float>((P.z - LP.z) / ddt), 0.f);
}

// last_p = p ; v += (g + f w) dt ; p += v dt ; f = 0
__global__ __launch_bounds__(kBlock) void k_semi_implicit(PSView ps, float dt, float gx, float gy, float gz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ps.n) return;
    float4 p = ps.p[i];
    float4 v = ps.v[i];
    const float4 f = ps.f[i];
    const float w = ps.w[i];
    ps.last_p[i] = p;
    semi_implicit(p, v, f, w, dt, gx, gy, gz);
    ps.v[i] = v;
    ps.p[i] = p;
    ps.f[i] = f4(0.f, 0.f, 0.f, 0.f);
}

__global__ __launch_bounds__(kBlock) void k_fix(PSView ps, const int* ids, int n, FixTransform t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int id = ids[i];
    ps.p[id] = fix_displacement(ps.init_p[id], t.com, t.offset, t.R);
    ps.v[id] = f4(0.f, 0.f, 0.f, 0.f);
    ps.f[id] = f4(0.f, 0.f, 0.f, 0.f);
    ps.mask[id] = 0;
}

// One pass over the vertices after a VBD sweep (see VbdTailArgs).  Each of its
// parts needs only the vertex's own records; as passes of their own they were
// 2-3 us of launch each (two of six launches of an iteration of the P1
// 64x16x16 beam with Chebyshev).  The predictor finds f = 0: the one that
// opened the step cleared it, and only a fixation writes it since (zero).
__global__ __launch_bounds__(kBlock) void k_vbd_tail(VbdTailArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const PSView& ps = a.ps;
    if (i >= ps.n) return;
    float4 p = gload(static_cast<const float4*>(ps.p), i);
    float4 last = f4(0.f, 0.f, 0.f, 0.f), h1 = last, h2 = last;
    if (a.velocity || a.predict) last = gload(static_cast<const float4*>(ps.last_p), i);
    if (a.prev1) {
        h1 = gload(static_cast<const float4*>(a.prev1), i);
        h2 = gload(static_cast<const float4*>(a.prev2), i);
    }
    bool moved = constrain(ps, i, p, a.c);
    if (a.prev1) {
        // p = prev2 + omega (p - prev2) from the third iteration on; prev2 = prev1, prev1 = p
        if (a.it >= 2) {
            const dvec3 P = dunpack(p, ps.lo_unit), Q = dunpack(h2, ps.lo_unit);
            const double om = a.omega;
            p = dpack(dvec3{Q.x + om * (P.x - Q.x), Q.y + om * (P.y - Q.y), Q.z + om * (P.z - Q.z)}, ps.lo_inv);
            moved = true;
        }
        gstore(a.prev2, i, h1);
        gstore(a.prev1, i, p);
    }
    if (a.velocity) vbd_velocity_from(ps, i, p, last, a.dt);
    if (a.predict)
        vbd_predict_from(ps, a.y, i, p, last, f4(0.f, 0.f, 0.f, 0.f), 0.f, a.dt, a.g[0], a.g[1], a.g[2], a.prev1);
    else if (moved)
        gstore(ps.p, i, p);
}

// One pass over the vertices after the XPBD projections: constraints, velocity
// and the next substep's k_semi_implicit (f = 0 since the last one; the
// velocity in between is not stored).  Three passes of 2-3 us of launch each
// before, of 12 in a substep of the 27-node 32x8x8 beam.
__global__ __launch_bounds__(kBlock) void k_pbd_tail(PSView ps, VertexConstraints c, float dt, float global_damping,
                                                     int next, float gx, float gy, float gz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ps.n) return;
    float4 p = gload(static_cast<const float4*>(ps.p), i);
    const float4 lp = gload(static_cast<const float4*>(ps.last_p), i);
    const float w = gload(ps.w, i);
    const bool moved = constrain(ps, i, p, c);
    float v[3];
    pbd_velocity_of(p, lp, w, dt, global_damping, v);
    if (!next) {
        if (moved) gstore(ps.p, i, p);
        gstore(ps.v, i, f4(v[0], v[1], v[2], 0.f));
        return;
    }
    gstore(ps.last_p, i, p);
    float4 vel = f4(v[0], v[1], v[2], 0.f);
    semi_implicit(p, vel, f4(0.f, 0.f, 0.f, 0.f), 0.f, dt, gx, gy, gz);
    gstore(ps.p, i, p);
}

__global__ __launch_bounds__(kBlock) void k_box(PSView ps, float3 pmin, float3 pmax) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ps.n) return;
    if (ps.mask[i] == 0) return;
    const float lo[3] = {pmin.x, pmin.y, pmin.z}, hi[3] = {pmax.x, pmax.y, pmax.z};
    float4 u = ps.p[i];
    const float4 X = ps.init_p[i];
    if (ps.comp ? box_clamp_comp(u, ps.lo_unit, ps.lo_inv, X, lo, hi) : box_clamp(u, X, lo, hi))
        ps.p[i] = u;   // written only when clamped
}

__global__ __launch_bounds__(kBlock) void k_copy_colour(PSView ps, const int* slot_vid, int first, int count,
                                                        const float4* p_new) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const int vid = slot_vid[first + i];
    if (ps.mask[vid] == 0) return;
    ps.p[vid] = p_new[vid];
}

// Internal force of each vertex from the element partials of k_explicit_elem
// (3 floats per (element, local node), with damping 9, in owners order, so a
// vertex's partials are contiguous): they are added in owners order, then the
// damping term of the reference's force pass, f = sum(-V P g) - k H v
// (src/GPU/Explicit/GPU_FEM_Explicit.cu:45-62), overwrites ps.f.  Eight
// incidences are loaded at a time, and the vertex's own records before them, so
// that the chain is {range, records} -> partials.  With damping three lanes take
// a vertex's nine sums, three neighbouring floats each, and one of them finishes:
// 36 floats a round in one lane took 7.7 us, nine lanes of one float 6.5, this
// 5.5 us on the damped 20-node 32x8x8 beam.  With integrate set (a semi-implicit
// integrator whose only dynamic is this force pass) the thread then runs
// k_semi_implicit's update of its vertex and the constraints; those passes are
// skipped (2.9 us each).  Undamped 27-node 32x8x8 beam: 3.3 us, 3.8 us when the
// undamped partials had nine floats too.
constexpr int kExplicitVertices = 64;   // per block
template <bool DAMP>
__global__ __launch_bounds__(kExplicitVertices * (DAMP ? 3 : 1)) void k_explicit_vertex(
    PSView ps, const int2* nbo, const float* partial, int count, float damping, int integrate, float dt, float gx,
    float gy, float gz, VertexConstraints c) {
    constexpr int NP = explicit_partial(DAMP), LANES = NP / 3, NV = kExplicitVertices, N = 8;
    const int t = threadIdx.x;
    const int2 range = gload(nbo, min(static_cast<int>(blockIdx.x) * NV + t / LANES, count - 1));
    const int vid = blockIdx.x * NV + t;
    const bool mine = t < NV && vid < count;
    float4 p = f4(0.f, 0.f, 0.f, 0.f), v = p, X = p;
    float w = 0.f;
    bool is_fixed = false;
    int mask = 0;
    if (mine) {
        p = gload(static_cast<const float4*>(ps.p), vid);
        v = gload(static_cast<const float4*>(ps.v), vid);
        w = gload(ps.w, vid);
        is_fixed = c.fixed && gload(c.fixed, vid) != 0;
        if (c.has_box) mask = gload(static_cast<const int*>(ps.mask), vid);
        if (c.fixed || c.has_box) X = gload(static_cast<const float4*>(ps.init_p), vid);
    }
    const float* __restrict__ src = partial + static_cast<size_t>(range.y) * NP + t % LANES * 3;
    float part[3] = {0.f, 0.f, 0.f};
    for (int j = 0; j < range.x; j += N) {
        float x[3 * N];
#pragma unroll
        for (int k = 0; k < 3 * N; ++k) x[k] = gload(src, NP * min(j + k / 3, range.x - 1) + k % 3);
#pragma unroll
        for (int k = 0; k < 3 * N; ++k) part[k % 3] += j + k / 3 < range.x ? x[k] : 0.f;
    }
    float a[NP];
    if constexpr (DAMP) {
        __shared__ float sums[NV * NP];
#pragma unroll
        for (int i = 0; i < 3; ++i) sums[3 * t + i] = part[i];
        __syncthreads();
        if (!mine) return;
#pragma unroll
        for (int i = 0; i < NP; ++i) a[i] = sums[NP * t + i];
    } else {
        if (!mine) return;
#pragma unroll
        for (int i = 0; i < NP; ++i) a[i] = part[i];
    }
    float4 f = f4(a[0], a[1], a[2], 0.f);
    if constexpr (DAMP) {
        f.x -= damping * (a[3] * v.x + a[4] * v.y + a[5] * v.z);
        f.y -= damping * (a[4] * v.x + a[6] * v.y + a[7] * v.z);
        f.z -= damping * (a[5] * v.x + a[7] * v.y + a[8] * v.z);
    }
    if (!integrate) {
        ps.f[vid] = f;
        return;
    }
    gstore(ps.last_p, vid, p);
    semi_implicit(p, v, f, w, dt, gx, gy, gz);
    if (!is_fixed) {   // constrain() stores v and f of a fixed vertex
        gstore(ps.v, vid, v);
        gstore(ps.f, vid, f4(0.f, 0.f, 0.f, 0.f));
    }
    constrain(ps, vid, p, is_fixed, mask, X, c.t.com, c.t.offset, c.t.R, c.has_box, c.lo, c.hi);
    gstore(ps.p, vid, p);
}

// Packed xyz of a run of records for the host.  The output is pinned host
// memory, so the pass is bound by the link: a block transposes its 256 records
// through LDS and writes whole 16-byte words (three 4-byte stores per vertex,
// 12 bytes apart, would send each link packet a third full).  The sum
// rest + u is formed in double and rounded once, as the state is stored.
__global__ __launch_bounds__(kBlock) void k_pack3(const float4* rec, const float4* rest, float unit, int first,
                                                  int count, float* out) {
    __shared__ float4 words[kBlock * 3 / 4];
    float* const flat = reinterpret_cast<float*>(words);
    const int b0 = blockIdx.x * kBlock, t = threadIdx.x;
    if (b0 + t < count) {
        const size_t i = static_cast<size_t>(first) + b0 + t;
        float4 u = gload(rec, i);
        if (rest) {
            const float4 X = gload(rest, i);
            if (unit == 0.f) u.w = 0.f;
            const dvec3 d = dunpack(u, unit);
            u.x = static_cast<float>(X.x + d.x);
            u.y = static_cast<float>(X.y + d.y);
            u.z = static_cast<float>(X.z + d.z);
        }
        flat[3 * t] = u.x;
        flat[3 * t + 1] = u.y;
        flat[3 * t + 2] = u.z;
    }
    __syncthreads();
    const int n_float = 3 * min(kBlock, count - b0);
    const size_t o = static_cast<size_t>(b0) * 3;   // a multiple of 768 floats
    if (4 * t + 4 <= n_float)
        reinterpret_cast<float4*>(out + o)[t] = words[t];
    else
        for (int k = 4 * t; k < n_float; ++k) out[o + k] = flat[k];
}

// ------------------------------------------------------------ batched forms
// One launch covers every vertex of every scene of a batch; each block belongs
// to one scene (VSeg), whose description is read with scalar loads.
__device__ __forceinline__ const SceneDev& vseg_scene(const BatchVArgs& b, int& i, int& ok) {
    const int blk = static_cast<int>(blockIdx.x);
    const VSeg seg = find_seg(b.segs, 0, b.nsegs, blk);
    i = (blk - seg.block_begin) * kBlock + threadIdx.x;
    ok = i < seg.count;
    return b.scenes[seg.scene];
}

__global__ __launch_bounds__(kBlock) void k_batch_predict(BatchVArgs b) {
    int i, ok;
    const SceneDev& sd = vseg_scene(b, i, ok);
    if (!ok) return;
    const PSView ps = sd.ps;
    vbd_predict_one(ps, sd.y, i, b.dt, sd.g[0], sd.g[1], sd.g[2], nullptr);
}

// fixation then box limit, fused: a fixed vertex is snapped and masked, every
// other vertex (mask 1) is clamped - the same result as the two kernels in
// sequence, since the box skips masked vertices.
__global__ __launch_bounds__(kBlock) void k_batch_fix_box(BatchVArgs b) {
    int i, ok;
    const SceneDev& sd = vseg_scene(b, i, ok);
    if (!ok || b.iteration >= sd.iterations) return;
    const PSView ps = sd.ps;
    const unsigned char* fixed = sd.fixed;
    // every load at once (global address space): the flag, the mask, the
    // displacement and the rest position
    const bool is_fixed = fixed != nullptr && gload(fixed, i) != 0;
    const int mask = gload(static_cast<const int*>(ps.mask), i);
    float4 u = gload(static_cast<const float4*>(ps.p), i);
    const float4 X = gload(static_cast<const float4*>(ps.init_p), i);
    if (constrain(ps, i, u, is_fixed, mask, X, sd.fix_com, sd.fix_offset, sd.fix_R, sd.has_box, sd.box_min, sd.box_max))
        gstore(ps.p, i, u);   // written only when it changed
}

__global__ __launch_bounds__(kBlock) void k_batch_velocity(BatchVArgs b) {
    int i, ok;
    const SceneDev& sd = vseg_scene(b, i, ok);
    if (!ok) return;
    const PSView ps = sd.ps;
    vbd_velocity_from(ps, i, gload(static_cast<const float4*>(ps.p), i), gload(static_cast<const float4*>(ps.last_p), i),
                      b.dt);
}

}  // namespace

void launch_batch_predict(const BatchVArgs& b, int nblocks, hipStream_t s) {
    if (nblocks > 0) hipLaunchKernelGGL(k_batch_predict, dim3(nblocks), dim3(kBlock), 0, s, b);
}
void launch_batch_fix_box(const BatchVArgs& b, int nblocks, hipStream_t s) {
    if (nblocks > 0) hipLaunchKernelGGL(k_batch_fix_box, dim3(nblocks), dim3(kBlock), 0, s, b);
}
void launch_batch_velocity(const BatchVArgs& b, int nblocks, hipStream_t s) {
    if (nblocks > 0) hipLaunchKernelGGL(k_batch_velocity, dim3(nblocks), dim3(kBlock), 0, s, b);
}

void launch_pack3(const float4* rec, const float4* rest, float unit, int first, int count, float* out, hipStream_t s) {
    if (count > 0)
        hipLaunchKernelGGL(k_pack3, dim3(grid_for(count)), dim3(kBlock), 0, s, rec, rest, unit, first, count, out);
}

void launch_vbd_predict(const PSView& ps, float4* y, float4* prev_it_p, float dt, const float g[3], hipStream_t s) {
    if (ps.n <= 0) return;
    hipLaunchKernelGGL(k_vbd_predict, dim3(grid_for(ps.n)), dim3(kBlock), 0, s, ps, y, prev_it_p, dt, g[0], g[1], g[2]);
}

void launch_vbd_tail(const VbdTailArgs& a, hipStream_t s) {
    if (a.ps.n <= 0) return;
    hipLaunchKernelGGL(k_vbd_tail, dim3(grid_for(a.ps.n)), dim3(kBlock), 0, s, a);
}

void launch_semi_implicit(const PSView& ps, float dt, const float g[3], hipStream_t s) {
    if (ps.n <= 0) return;
    hipLaunchKernelGGL(k_semi_implicit, dim3(grid_for(ps.n)), dim3(kBlock), 0, s, ps, dt, g[0], g[1], g[2]);
}

void launch_pbd_tail(const PSView& ps, const VertexConstraints& c, float dt, float global_damping, bool next,
                     const float g[3], hipStream_t s) {
    if (ps.n <= 0) return;
    hipLaunchKernelGGL(k_pbd_tail, dim3(grid_for(ps.n)), dim3(kBlock), 0, s, ps, c, dt, global_damping, next ? 1 : 0,
                       g[0], g[1], g[2]);
}

void launch_fix(const PSView& ps, const int* ids, int n, const FixTransform& t, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fix, dim3(grid_for(n)), dim3(kBlock), 0, s, ps, ids, n, t);
}

void launch_box(const PSView& ps, const float pmin[3], const float pmax[3], hipStream_t s) {
    if (ps.n <= 0) return;
    hipLaunchKernelGGL(k_box, dim3(grid_for(ps.n)), dim3(kBlock), 0, s, ps, make_float3(pmin[0], pmin[1], pmin[2]),
                       make_float3(pmax[0], pmax[1], pmax[2]));
}

void launch_explicit_vertex(const PSView& ps, const int2* nbo, const float* partial, int count, float damping,
                            const float* gravity, const VertexConstraints& c, float dt, hipStream_t s) {
    if (count <= 0) return;
    const float g0 = gravity ? gravity[0] : 0.f, g1 = gravity ? gravity[1] : 0.f, g2 = gravity ? gravity[2] : 0.f;
    const dim3 grid((count + kExplicitVertices - 1) / kExplicitVertices);
    const dim3 block(kExplicitVertices * (damping != 0.f ? 3 : 1));
    if (damping != 0.f)
        hipLaunchKernelGGL((k_explicit_vertex<true>), grid, block, 0, s, ps, nbo, partial, count, damping,
                           gravity ? 1 : 0, dt, g0, g1, g2, c);
    else
        hipLaunchKernelGGL((k_explicit_vertex<false>), grid, block, 0, s, ps, nbo, partial, count, damping,
                           gravity ? 1 : 0, dt, g0, g1, g2, c);
}

void launch_copy_colour(const PSView& ps, const int* slot_vid, int first, int count, const float4* p_new,
                        hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_copy_colour, dim3(grid_for(count)), dim3(kBlock), 0, s, ps, slot_vid, first, count, p_new);
}

}  // namespace oe
