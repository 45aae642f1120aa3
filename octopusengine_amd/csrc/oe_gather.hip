// Per-vertex gather over incident (element, quadrature point) pairs: the hot
// kernel of VBD (one launch per colour, reference kernel_vbd_solve_v3/v4,
// src/GPU/VBD/GPU_VBD_FEM.cu:234-400) and of the explicit integrator's internal
// force pass (reference kernel_fem_eval_force,
// src/GPU/Explicit/GPU_FEM_Explicit.cu:5-64).
//
// Work decomposition (CDNA4, wave64): a group of L consecutive lanes owns one
// vertex.  The vertex's incident elements are split into work items of QL
// quadrature points; lane t handles items t, t+L, ...  A work item loads the S
// node positions of its element once (one 16-byte load each) and reuses them
// for its QL quadrature points.  Each lane accumulates the force and the
// 3x3 Hessian block in registers; the group then reduces with cross-lane
// shuffles (no LDS, no barrier) and its first lane solves the 3x3 system in
// double precision.  L and QL are tile parameters chosen per element type.
//
// Cached form (CACHED = true, one quadrature point per work item): the
// displacement gradient Ju(e, q) = sum_k u_k (x) dN_k(q) is read from a
// per-(element, quadrature point) array instead of being rebuilt from the S
// node positions (S loads and 9 S FMAs per point), and after the solve the
// group adds du (x) dN_r(q) to the records of the vertex's elements.  The
// array is rebuilt from the positions at the start of every iteration
// (k_ju_refresh), after the predictor, constraints and any other position
// change.  Within one colour each element has at most one vertex being
// solved, so each record has a single reader-writer per launch.
//
// This file is compiled once per element type (OE_GATHER_S / OE_GATHER_Q set
// on the command line) so that the template instances build in parallel.
#include <cmath>
#include <stdexcept>

#include "oe_gather.hpp"
#include "oe_host.hpp"
#include "oe_kernels.hpp"

namespace oe {

// Work items of a lane whose gradient records stay in registers between the
// gather and the update in the cached form: enough for vertices with up to 4
// incident elements (ceil(4 Q / L), at most 2); further items are re-read.
template <int Q, int L>
constexpr int kept_items() {
    return (4 * Q + L - 1) / L < 2 ? (4 * Q + L - 1) / L : 2;
}

// (e, q, local node) of work item t of a vertex whose owner records start at own
__device__ __forceinline__ void work_item(const int* __restrict__ own, int t, int QC, int& eid, int& qc, int& r) {
    const int j = t / QC;
    qc = t - j * QC;
    const int pk = gload(own, j);
    eid = pk >> 5;
    r = pk & 31;
}

// dN_r at one point, from the shape-derivative table in device memory
__device__ __forceinline__ void load_dnr(const float* dn, int at, float dnr[3]) {
    dnr[0] = gload(dn, at);
    dnr[1] = gload(dn, at + 1);
    dnr[2] = gload(dn, at + 2);
}

// column-major: Ju[c*3 + k] += du[k] dN_r[c]
__device__ __forceinline__ void rank1_update(float* g, const float Ju[9], const float du[3],
                                             const float* __restrict__ dn) {
    const float d0 = dn[0], d1 = dn[1], d2 = dn[2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        g[k] = fmaf(du[k], d0, Ju[k]);
        g[3 + k] = fmaf(du[k], d1, Ju[3 + k]);
        g[6 + k] = fmaf(du[k], d2, Ju[6 + k]);
    }
}

// Gather + local solve of one vertex slot by a group of L lanes.
template <int S, int Q, int L, int QL, bool CACHED>
__device__ __forceinline__ void gather_body(const GatherArgs& a, int grp, int lane) {
    static_assert(!CACHED || QL == 1, "cached gradients take one quadrature point per work item");
    constexpr int QC = Q / QL;
    constexpr int KEEP = CACHED ? kept_items<Q, L>() : 1;
    if (grp >= a.count) return;                 // whole group leaves together
    const int slot = a.first_slot + grp;
    const int vid = gload(a.own.slot_vid, slot);
    if (a.mode != GATHER_EXPLICIT_FORCE && gload(a.ps.mask, vid) == 0) return;
    const int2 nbo = gload(a.own.slot_nbo, slot);
    const int nwork = nbo.x * QC;
    const int* __restrict__ own = a.own.own + nbo.y;
    Acc9 acc;
    acc_zero(acc);
    const float4* __restrict__ P = a.ps.p;
    float keep[KEEP][9];
    if constexpr (CACHED) {
#pragma unroll
        for (int it = 0; it < KEEP; ++it) {
            const int t = lane + it * L;
            if (t < nwork) {
                int eid, q, r;
                work_item(own, t, Q, eid, q, r);
                const size_t g = (static_cast<size_t>(eid) * Q + q) * 9;
                float JXi[9], V;
#pragma unroll
                for (int i = 0; i < 9; ++i) keep[it][i] = gload(a.ju, g + i);
                load_element_record(a.fem, eid, q, JXi, V);
                float dnr[3];
                load_dnr(a.fem.dN, (q * S + r) * 3, dnr);
                nh_contrib(keep[it], JXi, V, dnr, a.mt, acc);
            }
        }
        for (int t = lane + KEEP * L; t < nwork; t += L) {
            int eid, q, r;
            work_item(own, t, Q, eid, q, r);
            const size_t g = (static_cast<size_t>(eid) * Q + q) * 9;
            float Ju[9], JXi[9], V;
#pragma unroll
            for (int i = 0; i < 9; ++i) Ju[i] = gload(a.ju, g + i);
            load_element_record(a.fem, eid, q, JXi, V);
            float dnr[3];
            load_dnr(a.fem.dN, (q * S + r) * 3, dnr);
            nh_contrib(Ju, JXi, V, dnr, a.mt, acc);
        }
    } else {
        for (int t = lane; t < nwork; t += L) {
            int eid, qc, r;
            work_item(own, t, QC, eid, qc, r);
            const size_t tp = static_cast<size_t>(eid) * S;
            float4 h[S];
#pragma unroll
            for (int k = 0; k < S; ++k) h[k] = gload(static_cast<const float4*>(P), gload(a.fem.topo, tp + k));
            float xs[S][3];
#pragma unroll
            for (int k = 0; k < S; ++k) rel_node(h[k], h[0], a.ps.lo_unit, xs[k]);
#pragma unroll
            for (int qq = 0; qq < QL; ++qq) {
                const int q = qc * QL + qq;
                const float* __restrict__ dn = a.fem.dN + q * S * 3;
                float Ju[9], JXi[9], V;
                load_element_record(a.fem, eid, q, JXi, V);
                jx_from_nodes<S>(xs, dn, Ju);
                float dnr[3];
                load_dnr(dn, 3 * r, dnr);
                nh_contrib(Ju, JXi, V, dnr, a.mt, acc);
            }
        }
    }
    group_sum<L>(acc);
    if (a.mode == GATHER_EXPLICIT_FORCE) {
        if (lane != 0) return;
        // f = sum(-V P g) - k H v  (damping uses the vertex's own block)
        float4 f = make_float4(acc.v[0], acc.v[1], acc.v[2], 0.f);
        if (a.damping != 0.f) {
            const float4 v = a.ps.v[vid];
            f.x -= a.damping * (acc.v[3] * v.x + acc.v[4] * v.y + acc.v[5] * v.z);
            f.y -= a.damping * (acc.v[4] * v.x + acc.v[6] * v.y + acc.v[7] * v.z);
            f.z -= a.damping * (acc.v[5] * v.x + acc.v[7] * v.y + acc.v[8] * v.z);
        }
        a.ps.f[vid] = f;
        return;
    }
    if (a.mode == GATHER_VBD_RESIDUAL) {
        if (lane == 0) {
            const float u = a.ps.lo_unit;
            const float4 rv = vbd_residual(acc, dunpack(gload(static_cast<const float4*>(P), vid), u),
                                           dunpack(gload(static_cast<const float4*>(a.ps.last_p), vid), u),
                                           dunpack(gload(a.y, vid), u), a.ps.m[vid], a.damping, a.dt);
            if (a.out3) {
                a.out3[3 * static_cast<size_t>(vid)] = rv.x;
                a.out3[3 * static_cast<size_t>(vid) + 1] = rv.y;
                a.out3[3 * static_cast<size_t>(vid) + 2] = rv.z;
            } else {
                a.p_new[vid] = rv;
            }
        }
        return;
    }
    float du[3] = {0.f, 0.f, 0.f};
    if (lane == 0) {
        const float4 pv = gload(static_cast<const float4*>(P), vid);
        const float un = a.ps.lo_unit;
        const dvec3 p = dunpack(pv, un);
        double dx[3];
        vbd_local_solve(acc, p, dunpack(gload(static_cast<const float4*>(a.ps.last_p), vid), un),
                        dunpack(gload(a.y, vid), un), gload(a.ps.m, vid), a.damping, a.dt, dx);
        const float4 out = dpack(dvec3{p.x + dx[0], p.y + dx[1], p.z + dx[2]}, a.ps.lo_inv);
        gstore(a.mode == GATHER_VBD_JACOBI ? a.p_new : a.ps.p, vid, out);
        // the move of the full value (the cached gradients are built from
        // hi + lo); zero when the solve left the vertex where it was
        du[0] = static_cast<float>(dx[0]);
        du[1] = static_cast<float>(dx[1]);
        du[2] = static_cast<float>(dx[2]);
    }
    if constexpr (CACHED) {
        // broadcast the move from the group's first lane, then update the
        // gradients of every (element, quadrature point) the group read
#pragma unroll
        for (int k = 0; k < 3; ++k) du[k] = __shfl(du[k], 0, L);
        if (du[0] == 0.f && du[1] == 0.f && du[2] == 0.f) return;
#pragma unroll
        for (int it = 0; it < KEEP; ++it) {
            const int t = lane + it * L;
            if (t < nwork) {
                int eid, q, r;
                work_item(own, t, Q, eid, q, r);
                rank1_update(a.ju + (static_cast<size_t>(eid) * Q + q) * 9, keep[it], du, a.fem.dN + (q * S + r) * 3);
            }
        }
        for (int t = lane + KEEP * L; t < nwork; t += L) {
            int eid, q, r;
            work_item(own, t, Q, eid, q, r);
            float* g = a.ju + (static_cast<size_t>(eid) * Q + q) * 9;
            float Ju[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) Ju[i] = g[i];
            rank1_update(g, Ju, du, a.fem.dN + (q * S + r) * 3);
        }
    }
}

// One quadrature point per work item keeps the live state small; ask for at
// least 4 waves per SIMD there so that the scheduler does not trade occupancy
// for early issue of all S node loads.
template <int QL>
constexpr int gather_min_waves() { return QL == 1 ? 4 : 1; }

template <int S, int Q, int L, int QL, bool CACHED>
__global__ __launch_bounds__(256, gather_min_waves<QL>()) void k_vertex_gather(GatherArgs a) {
    const int gt = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    gather_body<S, Q, L, QL, CACHED>(a, gt / L, gt & (L - 1));
}

// Batched form: one launch covers one colour of many scenes.  Every block
// belongs to one (scene, colour) segment, so the scene's description is read
// once per block with scalar loads.
template <int S, int Q, int L, int QL, bool CACHED>
__global__ __launch_bounds__(256, gather_min_waves<QL>()) void k_batch_gather(BatchGatherArgs b) {
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const BatchSeg seg = find_seg(b.segs, b.seg_first, b.seg_count, blk);
    const SceneDev& sd = b.scenes[seg.scene];
    if (b.iteration >= sd.iterations) return;
    GatherArgs a;
    a.ps = sd.ps;
    a.fem = sd.fem;
    a.own = sd.own;
    a.mt = sd.mt;
    a.y = sd.y;
    a.p_new = nullptr;
    a.ju = sd.ju;
    a.damping = sd.damping;
    a.dt = b.dt;
    a.first_slot = seg.first;
    a.count = seg.count;
    a.mode = GATHER_VBD_INPLACE;
    a.out3 = nullptr;
    const int local = (blk - seg.block_begin) * 256 + threadIdx.x;
    gather_body<S, Q, L, QL, CACHED>(a, local / L, local & (L - 1));
}

// Refresh of the cached gradients, Ju(e, q) = sum_k u_k (x) dN_k(q): a block
// takes REFRESH_EPB(Q) = 256 / Q consecutive elements, stages their S node
// displacements in LDS once (one 16-byte load per node instead of one per
// (node, quadrature point)), then thread (element, q) builds its record; the
// records of one element are contiguous, so the stores are coalesced.
template <int Q>
constexpr int refresh_epb() { return 256 / Q; }

template <int S, int Q>
__device__ __forceinline__ void ju_refresh_block(const float4* __restrict__ P, float unit, const FemView& f, float* ju,
                                                 int e0, int ne) {
    constexpr int EPB = refresh_epb<Q>();
    __shared__ float4 sx[EPB * S];
    for (int t = threadIdx.x; t < ne * S; t += blockDim.x) sx[t] = P[f.topo[static_cast<size_t>(e0) * S + t]];
    __syncthreads();
    const int le = threadIdx.x / Q;
    const int q = threadIdx.x - le * Q;
    if (le >= ne) return;
    float xs[S][3];
    const float4 ref = sx[le * S];
#pragma unroll
    for (int k = 0; k < S; ++k) rel_node(sx[le * S + k], ref, unit, xs[k]);
    float Ju[9];
    jx_from_nodes<S>(xs, f.dN + q * S * 3, Ju);
    float* g = ju + (static_cast<size_t>(e0 + le) * Q + q) * 9;
#pragma unroll
    for (int i = 0; i < 9; ++i) g[i] = Ju[i];
}

template <int S, int Q>
__global__ __launch_bounds__(256) void k_ju_refresh(PSView ps, FemView f, float* ju) {
    constexpr int EPB = refresh_epb<Q>();
    const int e0 = xcd_block(blockIdx.x, gridDim.x) * EPB;
    const int ne = min(EPB, f.E - e0);
    ju_refresh_block<S, Q>(ps.p, ps.lo_unit, f, ju, e0, ne);
}

// Batched form: VSeg.count is the scene's element count, each block takes
// REFRESH_EPB elements of one scene.
template <int S, int Q>
__global__ __launch_bounds__(256) void k_batch_ju_refresh(BatchRefreshArgs b) {
    constexpr int EPB = refresh_epb<Q>();
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const VSeg seg = find_seg(b.segs, b.seg_first, b.seg_count, blk);
    const SceneDev& sd = b.scenes[seg.scene];
    if (b.iteration >= sd.iterations) return;      // uniform over the block
    const int e0 = (blk - seg.block_begin) * EPB;
    const int ne = min(EPB, seg.count - e0);
    ju_refresh_block<S, Q>(sd.ps.p, sd.ps.lo_unit, sd.fem, sd.ju, e0, ne);
}

#if OE_GATHER_S != 27   // 27-node hexahedra have their own task kernels
// Element tasks (see FusedTaskArgs).  Fixed vertices' incidences are not skipped:
// their solves are.
//
// Point tasks: the task form with an incidence's points spread over LQ lanes
// (LQ PPL >= Q), for linear tetrahedra (1 lane), 8-node hexahedra (8), 20-node
// tetrahedra (4 lanes, 3 points each) and, in launches too small to fill the
// chip, quadratic tetrahedra (4).  A pass of a single scene lasts as long as one
// wave's chain of loads and instructions (about 2 ns each): the gather runs
// ceil(incidences Q / L) work items per lane in turn, each loading and unpacking
// all S nodes; here a lane loads S / LQ nodes, passes them to its group through
// LDS, and runs one point.  Against the gather (the former default): a frame of
// 4 steps of the 64x16x16 beam Q1 4.35 -> 2.72 ms, P1 1.24 -> 1.18 ms (2.53 and
// 0.94 with the slots' sums spread over the block, sum_slots); 16 P3
// beams of 32x8x8 in a batch 22.6 -> 8.2 ms a step.  Against a thread per
// incidence: a step of the quadratic 16x4x4 beam 721 -> 627 us.
// A block takes a vertex block's incidences kFusedThreads / LQ at a time (more
// than one round only for vertices of very many elements).
template <int S>
constexpr int point_lanes() { return S == 4 ? 1 : S == 8 ? 8 : 4; }

template <int S, int Q>
struct PointLDS {
    static constexpr int LQ = point_lanes<S>(), G = kFusedThreads / LQ;
    // node values per group; the odd row stride spreads the groups over the banks
    float4 xs[LQ > 1 ? G : 1][LQ > 1 ? (S | 1) : 1];
    float part[kFusedIncPerBlock][9];
    int2 range[kFusedMaxSlots];         // per slot: first partial, partials
    float dn[LQ > 1 ? Q * S * 3 : 1];   // (k Q + q) 3 + c: neighbouring lanes read neighbouring words
};

// lane 0 of each group of LQ lanes, in every lane of the group
template <int LQ>
__device__ __forceinline__ float group_first(float x) {
    const int v = __float_as_int(x);
    if constexpr (LQ == 4) return __int_as_float(__builtin_amdgcn_update_dpp(0, v, 0x00, 0xF, 0xF, false));
    if constexpr (LQ == 8) {
        // row_newbcast 0 and 8: lanes 0 and 8 of each 16-lane row
        const int a = __builtin_amdgcn_update_dpp(0, v, 0x150, 0xF, 0xF, false);
        const int b = __builtin_amdgcn_update_dpp(0, v, 0x158, 0xF, 0xF, false);
        return __int_as_float((threadIdx.x & 8) ? b : a);
    }
    return x;
}

template <int S, int Q>
__device__ __forceinline__ void point_block(const PSView& ps, const FemView& f, const OwnersView& own,
                                            const MaterialView& mt, const float4* y, float damping, float dt,
                                            const int4 blk, PointLDS<S, Q>& sh) {
    constexpr int LQ = PointLDS<S, Q>::LQ, G = PointLDS<S, Q>::G;
    constexpr int PPL = (Q + LQ - 1) / LQ, NPL = (S + LQ - 1) / LQ;
    const int first_slot = blk.x, n_slots = blk.y, first_own = blk.z, n_inc = blk.w;
    const int t0 = threadIdx.x, g = t0 / LQ, sub = t0 % LQ;
    // loads in the order of the chain owners entry -> node ids -> positions; the
    // slot's state rides along (see slot_state_level1)
    int pk = gload(own.own, first_own + min(g, n_inc - 1));
    SlotState st{};
    slot_state_level1(own, first_slot + min(t0, n_slots - 1), st);
    constexpr int kStage = LQ > 1 ? (Q * S * 3 + kFusedThreads - 1) / kFusedThreads : 1;
    float stage[kStage];
    if constexpr (LQ > 1) {
#pragma unroll
        for (int j = 0; j < kStage; ++j) {
            const int i = min(t0 + kFusedThreads * j, Q * S * 3 - 1);
            const int k = i / (3 * Q), q = i / 3 % Q, c = i % 3;
            stage[j] = gload(f.dN, (q * S + k) * 3 + c);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    int nid[NPL];
#pragma unroll
    for (int j = 0; j < NPL; ++j) nid[j] = gload(f.topo, static_cast<size_t>(pk >> 5) * S + min(sub + LQ * j, S - 1));
    slot_state_level2(ps, y, st);
    const bool busy = __builtin_amdgcn_readfirstlane(g) < n_inc;   // the wave has an incidence in the first round
    if constexpr (LQ > 1) {
#pragma unroll
        for (int j = 0; j < kStage; ++j) sh.dn[min(t0 + kFusedThreads * j, Q * S * 3 - 1)] = stage[j];
    }
    for (int base = 0; base < n_inc; base += G) {
        const bool has = base + g < n_inc;
        if (base > 0) {
            pk = gload(own.own, first_own + min(base + g, n_inc - 1));
#pragma unroll
            for (int j = 0; j < NPL; ++j)
                nid[j] = gload(f.topo, static_cast<size_t>(pk >> 5) * S + min(sub + LQ * j, S - 1));
        }
        const int eid = pk >> 5, r = pk & 31;
        float xs[LQ > 1 ? 1 : S][3];
        float JXi[9], detB = 0.f, V = 0.f, dnr[3];
        if (busy) {
            float4 h[NPL];
#pragma unroll
            for (int j = 0; j < NPL; ++j) h[j] = gload(static_cast<const float4*>(ps.p), nid[j]);
            if (f.affine) {
#pragma unroll
                for (int i = 0; i < 9; ++i) JXi[i] = gload(f.jxv, static_cast<size_t>(eid) * 10 + i);
                detB = gload(f.jxv, static_cast<size_t>(eid) * 10 + 9);
                V = detB * gload(f.wq, min(sub, Q - 1));
            } else {
                load_element_record(f, eid, min(sub, Q - 1), JXi, V);
            }
            if constexpr (LQ == 1) load_dnr(f.dN, 3 * r, dnr);
            float4 ref = h[0];   // node 0 is lane 0's first
            ref.x = group_first<LQ>(ref.x);
            ref.y = group_first<LQ>(ref.y);
            ref.z = group_first<LQ>(ref.z);
            if constexpr (LQ == 1) {
#pragma unroll
                for (int k = 0; k < S; ++k) rel_node(h[k], ref, ps.lo_unit, xs[k]);
            } else {
                if (base > 0) wave_lds_sync();   // the group has read the last round's values
#pragma unroll
                for (int j = 0; j < NPL; ++j) {
                    float d[3];
                    rel_node(h[j], ref, ps.lo_unit, d);
                    sh.xs[g][min(sub + LQ * j, S - 1)] = make_float4(d[0], d[1], d[2], 0.f);
                }
                if (base > 0) wave_lds_sync();
            }
        }
        if constexpr (LQ > 1)
            if (base == 0) __syncthreads();   // the shape derivatives are every wave's
        if (!busy) continue;
        Acc9 acc;
        acc_zero(acc);
        if constexpr (LQ == 1) {
            // dN of a linear tetrahedron is (-1,-1,-1) and the unit vectors
            float Ju[9];
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int k = 0; k < 3; ++k) Ju[3 * c + k] = xs[c + 1][k] - xs[0][k];
            nh_contrib(Ju, JXi, V, dnr, mt, acc);
        } else {
#pragma unroll 1
            for (int i = 0; i < PPL; ++i) {
                const int q = min(sub + LQ * i, Q - 1);
                if (i > 0) {
                    if (f.affine) V = detB * gload(f.wq, q);
                    else load_element_record(f, eid, q, JXi, V);
                }
                const float Vq = sub + LQ * i < Q ? V : 0.f;
                float Ju[9];
#pragma unroll
                for (int k = 0; k < 9; ++k) Ju[k] = 0.f;
                const float* dn = &sh.dn[q * 3];
#pragma unroll
                for (int k = 0; k < S; ++k) {
                    const float4 x = sh.xs[g][k];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const float d = dn[k * Q * 3 + c];
                        Ju[3 * c] = fmaf(x.x, d, Ju[3 * c]);
                        Ju[3 * c + 1] = fmaf(x.y, d, Ju[3 * c + 1]);
                        Ju[3 * c + 2] = fmaf(x.z, d, Ju[3 * c + 2]);
                    }
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) dnr[c] = dn[r * Q * 3 + c];
                nh_contrib(Ju, JXi, Vq, dnr, mt, acc);
            }
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) acc.v[i] = lanes_sum<LQ>(acc.v[i]);
        if (has && sub == 0) {
#pragma unroll
            for (int i = 0; i < 9; ++i) sh.part[base + g][i] = acc.v[i];
        }
    }
    if (t0 < n_slots) {
        slot_state_settle(st);
        sh.range[t0] = make_int2(st.first_inc - first_own, st.n_inc);
    }
    __syncthreads();
    sum_slots<kFusedThreads>(sh.part, sh.range, n_slots);
    __syncthreads();
    if (t0 < n_slots && st.free != 0) solve_slot_from_sum(ps, st, sh.part[st.first_inc - first_own], damping, dt);
}

template <int S, int Q>
__global__ __launch_bounds__(kFusedThreads) void k_point_tasks(const int4* blocks, int first, int count,
                                                               FusedTaskArgs a) {
    __shared__ PointLDS<S, Q> sh;
    const int4 blk = gload(blocks, first + xcd_block(blockIdx.x, count));
    point_block<S, Q>(a.ps, a.fem, a.own, a.mt, a.y, a.damping, a.dt, blk, sh);
}

template <int S, int Q>
__global__ __launch_bounds__(kFusedThreads) void k_batch_point_tasks(BatchFusedArgs b) {
    __shared__ PointLDS<S, Q> sh;
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const BatchSeg seg = find_seg(b.segs, b.seg_first, b.seg_count, bid);
    const SceneDev& sd = b.scenes[seg.scene];
    if (b.iteration >= sd.iterations) return;
    // the scene's views, read before the first store
    const PSView ps = sd.ps;
    const FemView fem = sd.fem;
    const OwnersView own = sd.own;
    const MaterialView mt = sd.mt;
    const float4* y = sd.y;
    const float damping = sd.damping;
    const int4 blk = gload(S == 10 ? sd.fblocks_split : sd.fblocks, seg.first + (bid - seg.block_begin));
    point_block<S, Q>(ps, fem, own, mt, y, damping, b.dt, blk, sh);
}

#if OE_GATHER_S == 10   // one thread per incidence: quadratic tetrahedra in larger launches
// Quadratic tetrahedra.  With M_ii the corner and M_ij the edge values, u =
// sum_i l_i (2 l_i - 1) M_ii + 4 sum_{i<j} l_i l_j M_ij in the barycentric
// coordinates l, so the derivative along xi_c (l_c against l_0) is
//   D_c = 4 sum_j l_j (M_cj - M_0j) - (M_cc - M_00).
// The 4-point rule's points have three coordinates a and one b, the b at
// corner q* = 1, 2, 3, 0, so with E_cj = M_cj - M_0j
//   D_c(q) = 4a sum_j E_cj - E_cc - E_c0 + 4(b - a) E_c,q*
// - 9 multiply-adds per point on a base shared by the four, against 90 per
// point for the sum over the nodes (a third of the table is zero), and no
// table reads in the point loop.
struct P2Factors {
    float a4, k4;   // 4a, 4(b - a)
};
constexpr int kP2Edge[4][4] = {{0, 4, 6, 7}, {4, 1, 5, 8}, {6, 5, 2, 9}, {7, 8, 9, 3}};   // node of M_ij
constexpr int kP2Corner[4] = {1, 2, 3, 0};                                              // q* of point q
struct P2Gradients {
    float E[3][4][3];   // E_cj, c = 1..3
    float base[9];      // column-major, column c - 1
    __device__ __forceinline__ void init(const float (&x)[10][3], const P2Factors& f) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                float sum = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    E[c][j][k] = x[kP2Edge[c + 1][j]][k] - x[kP2Edge[0][j]][k];
                    sum = j == 0 ? E[c][j][k] : sum + E[c][j][k];
                }
                base[3 * c + k] = fmaf(f.a4, sum, -(E[c][c + 1][k] + E[c][0][k]));
            }
    }
    __device__ __forceinline__ void at(int corner, const P2Factors& f, float Jx[9]) const {
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) Jx[3 * c + k] = fmaf(f.k4, E[c][corner][k], base[3 * c + k]);
    }
};
// In the throughput form the shape-derivative table is copied to LDS, one copy
// per wave, at the start of a block: a lane's dN_r at each point is then an LDS
// read, not a device-memory load that the point loop waits on (batch: 84.9
// against 89.1 us per colour pass).  The latency form keeps the loads: it issues
// the vertex state's loads first, and vector-memory loads complete in order, so
// the copy's LDS write would wait for them (single scene: 1.22 against 1.19 ms
// per step).
template <int S, int Q, bool DNL>
constexpr int dn_lds_size() { return DNL ? S * Q * 3 : 1; }

// Partial (force, Hessian) of local node r of element eid over its Q points.
// dnw: the wave's LDS copy of the shape-derivative table (DNL only).
template <int S, int Q, bool DNL>
__device__ __forceinline__ void elem_partial(const FemView& f, const MaterialView& mt, const P2Factors& shape,
                                             int eid, int r, const float (&xs)[S][3], const float* dnw, Acc9& acc) {
    acc_zero(acc);
    // affine: one record per element, JX_inv and |det B|, V_q = |det B| w_q
    float JXi[9], detB = 0.f;
    if (f.affine) {
#pragma unroll
        for (int i = 0; i < 9; ++i) JXi[i] = gload(f.jxv, static_cast<size_t>(eid) * 10 + i);
        detB = gload(f.jxv, static_cast<size_t>(eid) * 10 + 9);
    }
    // dN_r at the four points: issued here with the record's loads when it
    // comes from memory (in the point loop each would be waited for)
    float dnr[Q][3];
    if constexpr (!DNL) {
#pragma unroll
        for (int q = 0; q < Q; ++q) load_dnr(f.dN, (q * S + r) * 3, dnr[q]);
    }
    float Ju[9], V = detB * gload(f.wq, 0);   // the rule's four weights are equal (shape_arg)
    P2Gradients g;
    g.init(xs, shape);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        g.at(kP2Corner[q], shape, Ju);
        if constexpr (DNL) {
#pragma unroll
            for (int c = 0; c < 3; ++c) dnr[q][c] = dnw[(q * S + r) * 3 + c];
        }
        if (!f.affine) load_element_record(f, eid, q, JXi, V);
        nh_contrib(Ju, JXi, V, dnr[q], mt, acc);
        acc_settle(acc);   // or the four points' sums are formed together at the end (138 VGPRs, 3 waves)
    }
}

// Phase 1 of a fused block: the partials of the block's incidences into LDS.
// Thread t takes the incidences t, t + kFusedThreads, ... of the vertex block.
template <int S, int Q, bool DNL>
__device__ __forceinline__ void fused_phase1(const PSView& ps, const FemView& f, const OwnersView& own,
                                             const MaterialView& mt, const P2Factors& shape, const int4 blk,
                                             float (*part)[9], float* dnw) {
    const int first_own = blk.z, n_inc = blk.w;
    const int t0 = threadIdx.x;
    // the table copy's loads go first and its LDS writes after the first
    // owners load is issued, so waiting for them overlaps that load; every
    // lane of the wave writes its share before any lane leaves
    constexpr int kDnPerLane = DNL ? (S * Q * 3 + 63) / 64 : 0;
    float dn_stage[kDnPerLane > 0 ? kDnPerLane : 1];
    const int lane = t0 & 63;
    if constexpr (kDnPerLane > 0) {
#pragma unroll
        for (int j = 0; j < kDnPerLane; ++j)
            if (lane + 64 * j < S * Q * 3) dn_stage[j] = gload(f.dN, lane + 64 * j);
    }
    const int pk0 = t0 < n_inc ? gload(own.own, first_own + t0) : 0;
    if constexpr (kDnPerLane > 0) {
#pragma unroll
        for (int j = 0; j < kDnPerLane; ++j)
            if (lane + 64 * j < S * Q * 3) dnw[lane + 64 * j] = dn_stage[j];
        // a wave's LDS operations complete in order; keep the compiler from
        // moving the table reads above the writes
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_wave_barrier();
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
    }
    if (t0 >= n_inc) return;
#pragma unroll 1
    for (int t = t0; t < n_inc; t += kFusedThreads) {
        const int pk = t == t0 ? pk0 : gload(own.own, first_own + t);
        float4 h[S];
#pragma unroll
        for (int k = 0; k < S; ++k)
            h[k] = gload(static_cast<const float4*>(ps.p), gload(f.topo, static_cast<size_t>(pk >> 5) * S + k));
        float xs[S][3];
#pragma unroll
        for (int k = 0; k < S; ++k) rel_node(h[k], h[0], ps.lo_unit, xs[k]);
        const int eid = pk >> 5, r = pk & 31;
        Acc9 acc;
        elem_partial<S, Q, DNL>(f, mt, shape, eid, r, xs, dnw, acc);
#pragma unroll
        for (int i = 0; i < 9; ++i) part[t][i] = acc.v[i];
    }
}

// The latency form's phase 1: one incidence per thread, and the slot state's
// loads issued by after_owner / after_topo right after the owners-entry and
// node-id loads, so that no wait of the element chain covers them.  A wave past
// the block's incidences returns at once (it holds no slot either).  The rest
// is straight-line: a lane past the incidences works on the last one and
// stores nothing (every vertex block has an incidence), so that no wait has to
// cover the loads of another path, which would make the compiler wait for
// every load in flight, the slot state's included.  (The throughput form keeps
// the loop above: this form's prologue cost it 2%, 86.7 against 84.5 us per P2
// batch pass on one GPU.)
template <int S, int Q, class AfterOwner, class AfterTopo>
__device__ __forceinline__ void fused_phase1_lat(const PSView& ps, const FemView& f, const OwnersView& own,
                                                 const MaterialView& mt, const P2Factors& shape, const int4 blk,
                                                 float (*part)[9], AfterOwner&& after_owner, AfterTopo&& after_topo) {
    static_assert(kFusedRuns == 1, "one incidence per thread");
    const int first_own = blk.z, n_inc = blk.w;
    const int t0 = threadIdx.x;
    if (__builtin_amdgcn_readfirstlane(t0 & ~63) >= n_inc) return;
    const bool has = t0 < n_inc;
    const int pk = gload(own.own, first_own + (has ? t0 : n_inc - 1));
    after_owner();
    __builtin_amdgcn_sched_barrier(0);
    int nid[S];
#pragma unroll
    for (int k = 0; k < S; ++k) nid[k] = gload(f.topo, static_cast<size_t>(pk >> 5) * S + k);
    after_topo();
    float4 h[S];
#pragma unroll
    for (int k = 0; k < S; ++k) h[k] = gload(static_cast<const float4*>(ps.p), nid[k]);
    float xs[S][3];
#pragma unroll
    for (int k = 0; k < S; ++k) rel_node(h[k], h[0], ps.lo_unit, xs[k]);
    const int eid = pk >> 5, r = pk & 31;
    Acc9 acc;
    elem_partial<S, Q, false>(f, mt, shape, eid, r, xs, nullptr, acc);
    if (has) {
#pragma unroll
        for (int i = 0; i < 9; ++i) part[t0][i] = acc.v[i];
    }
}

template <int S, int Q, bool LAT>
__device__ __forceinline__ void fused_block(const PSView& ps, const FemView& f, const OwnersView& own,
                                            const MaterialView& mt, const P2Factors& shape, const float4* y,
                                            float damping, float dt, const int4 blk, float (*part)[9], float* dnw) {
    const int first_slot = blk.x, n_slots = blk.y, first_own = blk.z;
    const int t0 = threadIdx.x;
    if constexpr (LAT) {
        // the slot state rides along the element chain (a thread past the
        // block's slots loads the last one and does not use it; every vertex
        // block has a slot)
        SlotState st{};
        const int ts = first_slot + min(t0, n_slots - 1);
        fused_phase1_lat<S, Q>(ps, f, own, mt, shape, blk, part, [&] { slot_state_level1(own, ts, st); },
                               [&] { slot_state_level2(ps, y, st); });
        __syncthreads();
        if (t0 < n_slots) {
            slot_state_settle(st);
            if (st.free != 0) solve_slot_from_lds(ps, st, part, first_own, damping, dt);
        }
    } else {
        // the slots' vertex ids and owners ranges, loaded now rather than after
        // the barrier (one dependent load less in phase 2; a thread past the
        // slots loads the last one)
        const int ts = first_slot + min(t0, n_slots - 1);
        const int slot_vid = gload(own.slot_vid, ts);
        const int2 slot_nbo = gload(own.slot_nbo, ts);
        fused_phase1<S, Q, !LAT>(ps, f, own, mt, shape, blk, part, dnw);
        __syncthreads();
        // phase 2: one thread per slot, partials in the owners order, local solve
        if (t0 >= n_slots) return;
        solve_slot_at(ps, slot_vid, slot_nbo, y, damping, dt, part, first_own);
    }
}

template <int S, int Q, bool LAT>
__global__ __launch_bounds__(kFusedThreads) void k_fused_tasks(const int4* blocks, int first, int count,
                                                               FusedTaskArgs a, P2Factors g) {
    __shared__ float part[LAT ? kFusedIncPerBlockLat : kFusedIncPerBlock][9];
    __shared__ float dn_lds[kFusedThreads / 64][dn_lds_size<S, Q, !LAT>()];
    const int4 blk = gload(blocks, first + xcd_block(blockIdx.x, count));
    fused_block<S, Q, LAT>(a.ps, a.fem, a.own, a.mt, g, a.y, a.damping, a.dt, blk, part,
                              dn_lds[threadIdx.x >> 6]);
}

template <int S, int Q, bool LAT>
__global__ __launch_bounds__(kFusedThreads) void k_batch_fused_tasks(BatchFusedArgs b, P2Factors g) {
    __shared__ float part[LAT ? kFusedIncPerBlockLat : kFusedIncPerBlock][9];
    __shared__ float dn_lds[kFusedThreads / 64][dn_lds_size<S, Q, !LAT>()];
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const BatchSeg seg = find_seg(b.segs, b.seg_first, b.seg_count, bid);
    const SceneDev& sd = b.scenes[seg.scene];
    if (b.iteration >= sd.iterations) return;
    // the scene's views, read before the first store
    const PSView ps = sd.ps;
    const FemView fem = sd.fem;
    const OwnersView own = sd.own;
    const MaterialView mt = sd.mt;
    const float4* y = sd.y;
    const float damping = sd.damping;
    const int4 blk = gload(LAT ? sd.fblocks_lat : sd.fblocks, seg.first + (bid - seg.block_begin));
    fused_block<S, Q, LAT>(ps, fem, own, mt, g, y, damping, b.dt, blk, part, dn_lds[threadIdx.x >> 6]);
}

#endif   // OE_GATHER_S == 10
#endif

namespace {

template <int S, int Q, int L, int QL, bool CACHED>
void launch_one(const GatherArgs& a, hipStream_t s) {
    if (a.count <= 0) return;
    const long long threads = static_cast<long long>(a.count) * L;
    const int block = 256;
    const int grid = static_cast<int>((threads + block - 1) / block);
    hipLaunchKernelGGL((k_vertex_gather<S, Q, L, QL, CACHED>), dim3(grid), dim3(block), 0, s, a);
}

template <int S, int Q, int L, int QL, bool CACHED>
void launch_batch_one(const BatchGatherArgs& b, int nblocks, hipStream_t s) {
    if (nblocks <= 0) return;
    hipLaunchKernelGGL((k_batch_gather<S, Q, L, QL, CACHED>), dim3(nblocks), dim3(256), 0, s, b);
}

template <int S, int Q, int QL, bool CACHED>
bool launch_batch_L(int L, const BatchGatherArgs& b, int nblocks, hipStream_t s) {
    switch (L) {
        case 4: launch_batch_one<S, Q, 4, QL, CACHED>(b, nblocks, s); return true;
        case 8: launch_batch_one<S, Q, 8, QL, CACHED>(b, nblocks, s); return true;
        case 16: launch_batch_one<S, Q, 16, QL, CACHED>(b, nblocks, s); return true;
        case 32: launch_batch_one<S, Q, 32, QL, CACHED>(b, nblocks, s); return true;
        case 64: launch_batch_one<S, Q, 64, QL, CACHED>(b, nblocks, s); return true;
        default: return false;
    }
}

template <int S, int Q, int QL, bool CACHED>
bool launch_L(int L, const GatherArgs& a, hipStream_t s) {
    switch (L) {
        case 4: launch_one<S, Q, 4, QL, CACHED>(a, s); return true;
        case 8: launch_one<S, Q, 8, QL, CACHED>(a, s); return true;
        case 16: launch_one<S, Q, 16, QL, CACHED>(a, s); return true;
        case 32: launch_one<S, Q, 32, QL, CACHED>(a, s); return true;
        case 64: launch_one<S, Q, 64, QL, CACHED>(a, s); return true;
        default: return false;
    }
}

// Element-centric internal forces of the explicit integrator.  The reference
// computes them per vertex (kernel_fem_eval_force,
// src/GPU/Explicit/GPU_FEM_Explicit.cu:5-64), so a vertex rebuilds F at every
// point of each incident element: S times over per (element, point).  Here a
// block takes NE elements in three stages, each dealt evenly over its threads
// (as many elements as make the points, or the nodes, fill whole waves):
//   nodes:  thread (e, k) puts node k's displacement relative to node 0 in LDS;
//   points: thread (e, q) forms Ju = sum_k x_k (x) dN_k(q), F, cof F and
//           s = lambda (J - alpha) once, and from them (M = JX_inv^T, so that
//           g = M dN_r)
//             Pm = V (mu F + s C) M    force  -V (mu F g + s C g) = -Pm dN_r
//           and with damping
//             G  = V mu M^T M          V mu |g|^2 = dN_r^T G dN_r
//             K  = C M                 C g = K dN_r
//           and V lambda, in LDS;
//   nodes:  thread (e, r) adds node r's terms over the points: the force, and
//           with damping the Hessian block V mu |g|^2 I + V lambda (C g)(C g)^T
//           of the reference's -k H v.  They go to the owners position of
//           (e, r), so that each vertex's partials are contiguous.
// k_explicit_vertex then adds each vertex's partials in owners order.  Explicit
// substeps carry every rounding of the force on (high modes are undamped), so
// each sum keeps its order.  With one element per 32 or 64 lanes (11 of 32 in
// the point stage of a 20-node element), scalar LDS reads and the Hessian also
// where nothing reads it, the pass took 11.1 us on the 27-node 32x8x8 beam and
// 18.5 us on the damped 20-node one; now 7.1 us and 13.3 us.
// Damped it is bound by the 47 VALU instructions per (node, point),
// 6.8 us on that beam, undamped by the three stages' latencies.
constexpr int kExplicitThreads = 256;
template <int S, int Q>
constexpr int explicit_elements() { return S == 4 ? 64 : S == 8 ? 32 : S == 10 ? 25 : S == 20 ? 11 : 9; }

template <int S, int Q, bool DAMP>
__global__ __launch_bounds__(kExplicitThreads) void k_explicit_elem(ExplicitElemArgs a) {
    constexpr int T = kExplicitThreads, NE = explicit_elements<S, Q>();
    static_assert(NE * S <= T && NE * Q <= T, "one round per stage");
    constexpr int R = (Q * 3) | 1;              // row of dn: node k's 3 Q values; odd, so nodes spread over the banks
    constexpr int W = DAMP ? 7 : 3;             // float4 per point: Pm (9), then K (9), G (6), V lambda
    __shared__ float dn[S * R];
    __shared__ float4 xs[NE][S | 1];
    __shared__ float4 pt[NE * Q][W];
    const int t = threadIdx.x;
    const int E = a.fem.E, e0 = blockIdx.x * NE;
    // the thread's node (threads past the last work on it and store nothing)
    const int nt = min(t, NE * S - 1), ne = nt / S, r = nt % S;
    const int ec = min(e0 + ne, E - 1);
    const size_t inc = static_cast<size_t>(ec) * S + r;
    const int node = gload(a.fem.topo, inc);
    const int at = gload(a.inc_at, inc);
    // the thread's point
    const int qt = min(t, NE * Q - 1), qe = qt / Q, q = qt % Q;
    float JXi[9], V;
    load_element_record(a.fem, min(e0 + qe, E - 1), q, JXi, V);
    constexpr int kStage = (S * Q * 3 + T - 1) / T;
    float stage[kStage];
#pragma unroll
    for (int j = 0; j < kStage; ++j) stage[j] = gload(a.fem.dN, min(t + T * j, S * Q * 3 - 1));
    const float4 u = gload(static_cast<const float4*>(a.ps.p), node);
#pragma unroll
    for (int j = 0; j < kStage; ++j) {
        const int i = min(t + T * j, S * Q * 3 - 1);   // (q S + k) 3 + c
        dn[i / 3 % S * R + i / (3 * S) * 3 + i % 3] = stage[j];
    }
    if (t < NE * S) xs[ne][r] = u;
    __syncthreads();
    if (t < NE * Q) {
        float Ju[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) Ju[i] = 0.f;
        const float4 ref = xs[qe][0];
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const float4 h = xs[qe][k];
            const float x[3] = {h.x - ref.x, h.y - ref.y, h.z - ref.z};   // an explicit state has no low-order parts
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float d = dn[k * R + q * 3 + c];
                Ju[3 * c] = fmaf(x[0], d, Ju[3 * c]);
                Ju[3 * c + 1] = fmaf(x[1], d, Ju[3 * c + 1]);
                Ju[3 * c + 2] = fmaf(x[2], d, Ju[3 * c + 2]);
            }
        }
        float F[9], C[9], P[9];
        deformation_gradient(Ju, JXi, F);
        cofactor(F, C);
        const float J = det_fixup(dot3_plain(F[0], C[0], F[1], C[1], F[2], C[2]), F);
        const float sl = a.mt.lambda * (J - a.mt.alpha);
#pragma unroll
        for (int i = 0; i < 9; ++i) P[i] = fmaf(a.mt.mu, F[i], sl * C[i]);
        // X(row, col) = X[col * 3 + row]; M(c, l) = JX_inv[c * 3 + l]
        float w[4 * W];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int l = 0; l < 3; ++l) {
                w[i * 3 + l] = V * fmaf(P[6 + i], JXi[6 + l], fmaf(P[3 + i], JXi[3 + l], P[i] * JXi[l]));
                if constexpr (DAMP)
                    w[9 + i * 3 + l] = fmaf(C[6 + i], JXi[6 + l], fmaf(C[3 + i], JXi[3 + l], C[i] * JXi[l]));
            }
        if constexpr (DAMP) {
            const float vm = V * a.mt.mu;
            constexpr int gl[6] = {0, 0, 0, 1, 1, 2}, gm[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
            for (int i = 0; i < 6; ++i)
                w[18 + i] = vm * dot3_plain(JXi[gl[i]], JXi[gm[i]], JXi[3 + gl[i]], JXi[3 + gm[i]], JXi[6 + gl[i]],
                                            JXi[6 + gm[i]]);
            w[24] = V * a.mt.lambda;
            w[25] = w[26] = w[27] = 0.f;
        } else {
            w[9] = w[10] = w[11] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < W; ++i) pt[qt][i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    }
    __syncthreads();
    if (t >= NE * S || e0 + ne >= E) return;
    // force, and with damping the Hessian block xx xy xz yy yz zz; a 27-node
    // hexahedron's points in two partial sums
    constexpr int NP = explicit_partial(DAMP);
    constexpr int QH = Q >= 16 ? (Q + 1) / 2 : Q;
    float acc[NP], lo[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) acc[i] = lo[i] = 0.f;
#pragma unroll 3
    for (int p = 0; p < Q; ++p) {
        if (QH < Q && p == QH) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                lo[i] = acc[i];
                acc[i] = 0.f;
            }
        }
        const float d0 = dn[r * R + p * 3], d1 = dn[r * R + p * 3 + 1], d2 = dn[r * R + p * 3 + 2];
        float w[4 * W];
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const float4 x = pt[ne * Q + p][i];
            w[4 * i] = x.x;
            w[4 * i + 1] = x.y;
            w[4 * i + 2] = x.z;
            w[4 * i + 3] = x.w;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) acc[i] -= dot3_plain(w[3 * i], d0, w[3 * i + 1], d1, w[3 * i + 2], d2);
        if constexpr (DAMP) {
            float c[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) c[i] = w[9 + i * 3] * d0 + w[9 + i * 3 + 1] * d1 + w[9 + i * 3 + 2] * d2;
            const float gd = w[18] * d0 * d0 + w[21] * d1 * d1 + w[23] * d2 * d2 +
                             2.f * (w[19] * d0 * d1 + w[20] * d0 * d2 + w[22] * d1 * d2);
            const float vl = w[24];
            acc[3] += gd + vl * c[0] * c[0];
            acc[4] += vl * c[1] * c[0];
            acc[5] += vl * c[2] * c[0];
            acc[6] += gd + vl * c[1] * c[1];
            acc[7] += vl * c[2] * c[1];
            acc[8] += gd + vl * c[2] * c[2];
        }
    }
    float* out = a.partial + static_cast<size_t>(at) * NP;
#pragma unroll
    for (int i = 0; i < NP; ++i) out[i] = QH < Q ? lo[i] + acc[i] : acc[i];
}

}  // namespace

#if defined(OE_GATHER_S) && defined(OE_GATHER_Q)
// OE_FN(launch_gather_) -> launch_gather_<S>_<Q>
#define OE_CAT3(p, s, q) p##s##_##q
#define OE_NAME(p, s, q) OE_CAT3(p, s, q)
#define OE_FN(p) OE_NAME(p, OE_GATHER_S, OE_GATHER_Q)

// Quadrature points per lane that divide Q: 1, Q, and for Q = 4 / 27 the
// intermediate divisors.  The cached form takes QL = 1 only.
bool OE_FN(launch_gather_)(int L, int QL, const GatherArgs& a, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q;
    if (a.ju) return QL == 1 && a.mode == GATHER_VBD_INPLACE && launch_L<S, Q, 1, true>(L, a, s);
    if (QL == 1) return launch_L<S, Q, 1, false>(L, a, s);
    if (QL == Q) return launch_L<S, Q, Q, false>(L, a, s);
#if OE_GATHER_Q == 4
    if (QL == 2) return launch_L<S, Q, 2, false>(L, a, s);
#endif
#if OE_GATHER_Q == 27
    if (QL == 3) return launch_L<S, Q, 3, false>(L, a, s);
    if (QL == 9) return launch_L<S, Q, 9, false>(L, a, s);
#endif
    return false;
}

bool OE_FN(launch_batch_gather_)(int L, int QL, bool cached, const BatchGatherArgs& b, int nblocks, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q;
    if (cached) return QL == 1 && launch_batch_L<S, Q, 1, true>(L, b, nblocks, s);
    if (QL == 1) return launch_batch_L<S, Q, 1, false>(L, b, nblocks, s);
    if (QL == Q) return launch_batch_L<S, Q, Q, false>(L, b, nblocks, s);
#if OE_GATHER_Q == 4
    if (QL == 2) return launch_batch_L<S, Q, 2, false>(L, b, nblocks, s);
#endif
#if OE_GATHER_Q == 27
    if (QL == 3) return launch_batch_L<S, Q, 3, false>(L, b, nblocks, s);
    if (QL == 9) return launch_batch_L<S, Q, 9, false>(L, b, nblocks, s);
#endif
    return false;
}

void OE_FN(launch_ju_refresh_)(const PSView& ps, const FemView& f, float* ju, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q;
    constexpr int EPB = refresh_epb<Q>();
    if (f.E <= 0) return;
    hipLaunchKernelGGL((k_ju_refresh<S, Q>), dim3((f.E + EPB - 1) / EPB), dim3(256), 0, s, ps, f, ju);
}

int OE_FN(refresh_elements_per_block_)() { return refresh_epb<OE_GATHER_Q>(); }

#if OE_GATHER_S == 10
namespace {
// The P2 factors from the element's quadrature points, checked against its
// shape-derivative table (to float rounding: the reference's points are floats
// whose coordinates add to 1 within an ulp).
const P2Factors& shape_arg() {
    static const P2Factors g = [] {
        P2Factors t{};
        const ShapeTable& st = shape_table(Tetra10);
        const double b = st.qpoints[0], a = (1.0 - b) / 3.0;
        for (int q = 0; q < 4; ++q)
            for (int c = 1; c < 4; ++c) {
                double want[10] = {};
                for (int j = 0; j < 4; ++j) {
                    const double l = j == kP2Corner[q] ? b : a;
                    want[kP2Edge[c][j]] += 4.0 * l;
                    want[kP2Edge[0][j]] -= 4.0 * l;
                }
                want[c] -= 1.0;
                want[0] += 1.0;
                for (int k = 0; k < 10; ++k)
                    if (st.weights[q] != st.weights[0] || std::fabs(want[k] - st.dN[(q * 10 + k) * 3 + c - 1]) > 5e-7)
                        throw std::logic_error("the P2 table does not have the 4-point rule's form");
            }
        t.a4 = static_cast<float>(4.0 * a);
        t.k4 = static_cast<float>(4.0 * (b - a));
        return t;
    }();
    return g;
}
}  // namespace

#endif

#if OE_GATHER_S != 27
void OE_FN(launch_fused_tasks_)(const FusedTaskArgs& a, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q;
    if (a.count <= 0) return;
#if OE_GATHER_S == 10
    if (a.form == TASKS_THROUGHPUT) {
        hipLaunchKernelGGL((k_fused_tasks<S, Q, false>), dim3(a.count), dim3(kFusedThreads), 0, s, a.blocks,
                           a.first_block, a.count, a, shape_arg());
        return;
    }
    if (a.form == TASKS_LATENCY) {
        hipLaunchKernelGGL((k_fused_tasks<S, Q, true>), dim3(a.count), dim3(kFusedThreads), 0, s, a.blocks,
                           a.first_block, a.count, a, shape_arg());
        return;
    }
#endif
    hipLaunchKernelGGL((k_point_tasks<S, Q>), dim3(a.count), dim3(kFusedThreads), 0, s, a.blocks, a.first_block, a.count,
                       a);
}

void OE_FN(launch_batch_fused_tasks_)(const BatchFusedArgs& b, int nblocks, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q;
    if (nblocks <= 0) return;
#if OE_GATHER_S == 10
    if (b.form == TASKS_THROUGHPUT) {
        hipLaunchKernelGGL((k_batch_fused_tasks<S, Q, false>), dim3(nblocks), dim3(kFusedThreads), 0, s, b,
                           shape_arg());
        return;
    }
    if (b.form == TASKS_LATENCY) {
        hipLaunchKernelGGL((k_batch_fused_tasks<S, Q, true>), dim3(nblocks), dim3(kFusedThreads), 0, s, b,
                           shape_arg());
        return;
    }
#endif
    hipLaunchKernelGGL((k_batch_point_tasks<S, Q>), dim3(nblocks), dim3(kFusedThreads), 0, s, b);
}
#endif

void OE_FN(launch_explicit_elem_)(const ExplicitElemArgs& a, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q, NE = explicit_elements<S, Q>();
    if (a.fem.E <= 0) return;
    const dim3 grid((a.fem.E + NE - 1) / NE), block(kExplicitThreads);
    if (a.damped)
        hipLaunchKernelGGL((k_explicit_elem<S, Q, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((k_explicit_elem<S, Q, false>), grid, block, 0, s, a);
}

void OE_FN(launch_batch_ju_refresh_)(const BatchRefreshArgs& b, int nblocks, hipStream_t s) {
    constexpr int S = OE_GATHER_S, Q = OE_GATHER_Q;
    if (nblocks <= 0) return;
    hipLaunchKernelGGL((k_batch_ju_refresh<S, Q>), dim3(nblocks), dim3(256), 0, s, b);
}
#endif

}  // namespace oe
