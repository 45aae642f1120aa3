// XPBD per-colour element projection.  Elements of one colour share no vertex,
// so every element of a colour is projected concurrently and writes its own
// nodes only.  Each element carries two constraints (lambda term, then mu
// term), solved one after the other with the positions updated in between.
//
// Two formulations, as in the reference:
//  * "V0" (src/GPU/PBD/GPU_PBD_FEM.cu:13-93): C = sqrt|E|, grad C = grad E/(2C),
//    dl = -C / (sum w |grad C|^2 + 1/(k dt^2)), fixed vertices are not moved.
//    Used for P1 and when the XPBD version is requested.  One thread per element.
//  * "V2" (src/GPU/PBD/GPU_PBD_FEM.cu:206-263, and V1 :141-204 which has the
//    same arithmetic): beta = -2E / (sum w |grad E|^2 + 4E/(k dt^2)), zero when
//    E < 1e-12, every node moved.  One group of lanes per element (V2Plan);
//    the node positions and per-quadrature stresses are staged in LDS.
// Energies per material: src/GPU/PBD/GPU_PBD_FEM_Materials.cu:31-66,97-118.
#include "oe_kernels.hpp"
#include "oe_vertex.hpp"
#include "oe_xpbd.hpp"

namespace oe {

namespace {

// energy e and dE/dF for constraint m of the XPBD energy split.  The
// NeoHooke split uses alpha = 1 + mu/lambda (PBD_ContinuousMaterial.h:61-65,
// GPU_PBD_FEM_Materials.cu:105-107), unlike the GPU VBD NeoHooke stress.
__device__ __forceinline__ void xpbd_material(int material, int m, float alpha, const float F[9], float P[9],
                                              float& e) {
    float C[9];
    cofactor(F, C);
    const float J = det_from_cof(F, C);
    if (material == Stable_NeoHooke_id) {
        if (m == 0) {
            const float d = J - 1.f;
            e = d * d;
#pragma unroll
            for (int i = 0; i < 9; ++i) P[i] = 2.f * d * C[i];
        } else {
            float n2 = 0.f;
#pragma unroll
            for (int i = 0; i < 9; ++i) n2 = fmaf(F[i], F[i], n2);
            e = fmaf(-2.f, J - 1.f, n2 - 3.f);
#pragma unroll
            for (int i = 0; i < 9; ++i) P[i] = 2.f * F[i] - 2.f * C[i];
        }
    } else {  // NeoHooke: (J - alpha)^2 and |F|^2 - 3
        if (m == 0) {
            const float d = J - alpha;
            e = d * d;
#pragma unroll
            for (int i = 0; i < 9; ++i) P[i] = 2.f * d * C[i];
        } else {
            float n2 = 0.f;
#pragma unroll
            for (int i = 0; i < 9; ++i) n2 = fmaf(F[i], F[i], n2);
            e = n2 - 3.f;
#pragma unroll
            for (int i = 0; i < 9; ++i) P[i] = 2.f * F[i];
        }
    }
}

// Ps = P * JX_inv^T * V (column-major): Ps(r,c) = V sum_l P(r,l) JX_inv(c,l)
__device__ __forceinline__ void scale_stress(const float P[9], const float JXi[9], float V, float Ps[9]) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 3; ++r)
            Ps[c * 3 + r] = dot3(P[r], JXi[c], P[3 + r], JXi[3 + c], P[6 + r], JXi[6 + c]) * V;
}

template <int S, int Q>
__global__ __launch_bounds__(256) void k_xpbd_v0(XpbdArgs a) {
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= a.count) return;
    const int eid = a.eids[a.first + tid];
    const int* __restrict__ tp = a.fem.topo + static_cast<size_t>(eid) * S;
    for (int m = 0; m < 2; ++m) {
        float xs[S][3];
        float grad[S][3];
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const float4 x = a.ps.p[tp[k]];
            xs[k][0] = x.x; xs[k][1] = x.y; xs[k][2] = x.z;
            grad[k][0] = grad[k][1] = grad[k][2] = 0.f;
        }
        float C = 0.f;
        for (int q = 0; q < Q; ++q) {
            const float* dn = a.fem.dN + q * S * 3;
            float Jx[9], JXi[9], F[9], P[9], Ps[9], e, V;
            load_element_record(a.fem, eid, q, JXi, V);
            jx_from_nodes<S>(xs, dn, Jx);
            deformation_gradient(Jx, JXi, F);
            xpbd_material(a.mt.material, m, 1.f + a.mt.mu / a.mt.lambda, F, P, e);
            scale_stress(P, JXi, V, Ps);
            C += e * V;
#pragma unroll
            for (int k = 0; k < S; ++k)
#pragma unroll
                for (int r = 0; r < 3; ++r)
                    grad[k][r] += Ps[r] * dn[3 * k] + Ps[3 + r] * dn[3 * k + 1] + Ps[6 + r] * dn[3 * k + 2];
        }
        C = fabsf(C);
        C = sqrtf(C);
        const float Cinv = C < 1e-12f ? 0.f : 1.f / (2.f * C);
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < S; ++k) {
            grad[k][0] *= Cinv; grad[k][1] *= Cinv; grad[k][2] *= Cinv;
            sum += (grad[k][0] * grad[k][0] + grad[k][1] * grad[k][1] + grad[k][2] * grad[k][2]) * a.ps.w[tp[k]];
        }
        const float stiff = (m == 0) ? a.mt.lambda : a.mt.mu;
        const float alpha = 1.f / (stiff * a.dt * a.dt);
        const float dl = -C / (sum + alpha);
#pragma unroll
        for (int k = 0; k < S; ++k) {
            const int vid = tp[k];
            if (a.ps.mask[vid] == 0) continue;
            const float wv = a.ps.w[vid];
            float4 x = a.ps.p[vid];
            x.x += dl * wv * grad[k][0];
            x.y += dl * wv * grad[k][1];
            x.z += dl * wv * grad[k][2];
            a.ps.p[vid] = x;
        }
    }
}

// One linear tetrahedron, both constraints: x the nodes' values, w their
// inverse masses, free whether a node may move.  dN is (-1,-1,-1) and the unit
// vectors, so Jx holds edge differences and the gradient of node k > 0 is
// column k - 1 of the scaled stress: the sums of the general form with its zero
// terms left out, the same bits.
struct P1Element {
    float JXi[9], V;
};
__device__ __forceinline__ P1Element p1_element(float4 r0, float4 r1, float4 r2) {
    return P1Element{{r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x}, r2.y};
}
__device__ __forceinline__ void p1_project(const MaterialView& mt, float dt, const P1Element& el, const float (&w)[4],
                                           const bool (&free)[4], float (&x)[4][3]) {
    const float alpha_nh = 1.f + mt.mu / mt.lambda;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        float Jx[9], F[9], P[9], Ps[9], e;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int r = 0; r < 3; ++r) Jx[3 * c + r] = x[c + 1][r] - x[0][r];
        deformation_gradient(Jx, el.JXi, F);
        xpbd_material(mt.material, m, alpha_nh, F, P, e);
        scale_stress(P, el.JXi, el.V, Ps);
        const float C = sqrtf(fabsf(e * el.V));
        const float Cinv = C < 1e-12f ? 0.f : 1.f / (2.f * C);
        float grad[4][3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            grad[0][r] = (-Ps[r] - Ps[3 + r] - Ps[6 + r]) * Cinv;
            grad[1][r] = Ps[r] * Cinv;
            grad[2][r] = Ps[3 + r] * Cinv;
            grad[3][r] = Ps[6 + r] * Cinv;
        }
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            sum = fmaf(dot3(grad[k][0], grad[k][0], grad[k][1], grad[k][1], grad[k][2], grad[k][2]), w[k], sum);
        const float stiff = (m == 0) ? mt.lambda : mt.mu;
        const float alpha = 1.f / (stiff * dt * dt);
        const float dl = -C / (sum + alpha);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float s = dl * w[k];
#pragma unroll
            for (int r = 0; r < 3; ++r) x[k][r] = free[k] ? fmaf(s, grad[k][r], x[k][r]) : x[k][r];
        }
    }
}

// One thread per linear tetrahedron of a colour; the element's four nodes are
// read once and written once for its two constraints.  Bound by the launch and
// the chain nodes -> positions -> ~450 instructions; reading the nodes again
// for the second constraint, after an element id and an index load, it took
// 5.9 us per colour; with the first arguments preloaded 3.2 us.
__global__ __launch_bounds__(64) void k_xpbd_p1(const int4* nodes, int first, int count, XpbdArgs a) {
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t >= count) return;
    const size_t i = static_cast<size_t>(first) + t;
    const int4 n4 = gload(nodes, i);
    const float4 r0 = gload(a.p1_rec, 3 * i), r1 = gload(a.p1_rec, 3 * i + 1), r2 = gload(a.p1_rec, 3 * i + 2);
    const int n[4] = {n4.x, n4.y, n4.z, n4.w};
    float4 u[4];
    float w[4], x[4][3];
    bool free[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        u[k] = gload(static_cast<const float4*>(a.ps.p), n[k]);
        w[k] = gload(a.ps.w, n[k]);
        free[k] = gload(static_cast<const int*>(a.ps.mask), n[k]) != 0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        x[k][0] = u[k].x;
        x[k][1] = u[k].y;
        x[k][2] = u[k].z;
    }
    p1_project(a.mt, a.dt, p1_element(r0, r1, r2), w, free, x);
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (free[k]) gstore(a.ps.p, n[k], make_float4(x[k][0], x[k][1], x[k][2], u[k].w));
}

// The workgroup's LDS operations ordered for all of its waves.  Unlike
// __syncthreads it names LDS alone, so loads in flight stay in flight.
__device__ __forceinline__ void block_lds_sync() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A run of substeps of a small linear-tetrahedron scene in one workgroup.  A
// colour of such a scene is a wave or a few of work (59 elements on the
// 16x4x4 beam), and a substep has ~28 of them: as launches the frame is the
// launches.  Here the positions stay in LDS (xyz and the inverse mass, its sign
// bit set on masked vertices: the zero of an infinite mass has one too), a colour
// boundary is a workgroup barrier, and the next colour's element is loaded while
// the current one computes.  One compute unit does all the work, so the form is
// for scenes whose positions fit LDS (kXpbdResidentVertices), where a colour is
// at most ~6 waves.  The arithmetic is that of k_xpbd_p1 and the vertex passes, in
// their order.
constexpr int kXpbdResidentThreads = 512;
__device__ __forceinline__ bool unmasked(float w) { return __float_as_int(w) >= 0; }
__global__ __launch_bounds__(kXpbdResidentThreads) void k_xpbd_p1_resident(XpbdResidentArgs a) {
    constexpr int T = kXpbdResidentThreads;
    __shared__ float4 pos[kXpbdResidentVertices];
    __shared__ float last[kXpbdResidentVertices * 3];
    const int tid = threadIdx.x, n = a.ps.n;
    // load, then the first semi-implicit step (k_semi_implicit)
    for (int i = tid; i < n; i += T) {
        float4 p = gload(static_cast<const float4*>(a.ps.p), i), v = gload(static_cast<const float4*>(a.ps.v), i);
        const float4 f = gload(static_cast<const float4*>(a.ps.f), i);
        const float w = gload(a.ps.w, i);
        const int mask = gload(static_cast<const int*>(a.ps.mask), i);
        last[3 * i] = p.x;
        last[3 * i + 1] = p.y;
        last[3 * i + 2] = p.z;
        semi_implicit(p, v, f, w, a.dt, a.g[0], a.g[1], a.g[2]);
        pos[i] = make_float4(p.x, p.y, p.z, mask != 0 ? w : -w);
        gstore(a.ps.f, i, make_float4(0.f, 0.f, 0.f, 0.f));
    }
    // the thread's element of the next colour to come, loaded ahead
    int4 nn = make_int4(0, 0, 0, 0);
    float4 r0 = make_float4(0.f, 0.f, 0.f, 0.f), r1 = r0, r2 = r0;
    auto fetch = [&](int i) {
        nn = gload(a.nodes, i);
        r0 = gload(a.rec, 3 * i);
        r1 = gload(a.rec, 3 * i + 1);
        r2 = gload(a.rec, 3 * i + 2);
    };
    if (tid < a.color_begin[1]) fetch(tid);
    for (int sub = 0; sub < a.substeps; ++sub) {
        int begin = 0, end = a.color_begin[1];
        for (int c = 0; c < a.n_colors; ++c) {
            block_lds_sync();
            const int nc = c + 1 < a.n_colors ? c + 1 : 0;   // after the last colour, the first of the next substep
            const int nb = a.color_begin[nc], ne = a.color_begin[nc + 1];
            for (int i = begin + tid; i < end; i += T) {
                if (i >= begin + T) fetch(i);
                const int nd[4] = {nn.x, nn.y, nn.z, nn.w};
                const P1Element el = p1_element(r0, r1, r2);
                if (i + T >= end && nb + tid < ne) fetch(nb + tid);
                float w[4], x[4][3], ws[4];
                bool free[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float4 u = pos[nd[k]];
                    x[k][0] = u.x;
                    x[k][1] = u.y;
                    x[k][2] = u.z;
                    ws[k] = u.w;
                    w[k] = fabsf(u.w);
                    free[k] = unmasked(u.w);
                }
                p1_project(a.mt, a.dt, el, w, free, x);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (free[k]) pos[nd[k]] = make_float4(x[k][0], x[k][1], x[k][2], ws[k]);
            }
            if (begin + tid >= end && nb + tid < ne) fetch(nb + tid);   // a thread without work in this colour
            begin = nb;
            end = ne;
        }
        block_lds_sync();
        // k_pbd_tail
        const bool next = sub + 1 < a.substeps;
        for (int i = tid; i < n; i += T) {
            const float4 q = pos[i];
            const float4 lp = make_float4(last[3 * i], last[3 * i + 1], last[3 * i + 2], 0.f);
            float4 p = make_float4(q.x, q.y, q.z, 0.f);
            const float w = fabsf(q.w);
            float ws = q.w;
            if (a.c.fixed || a.c.has_box) {
                const bool is_fixed = a.c.fixed && gload(a.c.fixed, i) != 0;
                const float4 X = gload(static_cast<const float4*>(a.ps.init_p), i);
                constrain(a.ps, i, p, is_fixed, unmasked(q.w) ? 1 : 0, X, a.c.t.com, a.c.t.offset, a.c.t.R, a.c.has_box,
                          a.c.lo, a.c.hi);
                if (is_fixed) ws = -w;
            }
            float v[3];
            pbd_velocity_of(p, lp, w, a.dt, a.global_damping, v);
            if (!next) {
                gstore(a.ps.p, i, make_float4(p.x, p.y, p.z, 0.f));
                gstore(a.ps.last_p, i, lp);
                gstore(a.ps.v, i, make_float4(v[0], v[1], v[2], 0.f));
                continue;
            }
            last[3 * i] = p.x;
            last[3 * i + 1] = p.y;
            last[3 * i + 2] = p.z;
            float4 vel = make_float4(v[0], v[1], v[2], 0.f);
            semi_implicit(p, vel, make_float4(0.f, 0.f, 0.f, 0.f), 0.f, a.dt, a.g[0], a.g[1], a.g[2]);
            pos[i] = make_float4(p.x, p.y, p.z, ws);
        }
    }
}

// Lanes of one element in the V2 projection.  The point stage gives a
// quadrature point WP lanes' worth of room, PP times over: part p sums its KP
// nodes of every point's Jx.  The node stage gives the nodes WN lanes, PN
// times over: part p sums its QN points of every node's gradient.  A colour
// holds a few hundred elements, far too few to fill the chip, so a pass lasts
// as long as one wave's chain of instructions: the sums are split over as many
// lanes as an element can use, and LDS is read 16 bytes at a time.
// NARROW (8-node hexahedra, 8 lanes): colours that fill the chip by themselves.
template <int S, int Q, bool NARROW = false>
struct V2Lanes;
template <> struct V2Lanes<8, 8, true> { static constexpr int WP = 8, PP = 1, WN = 8, PN = 1; };
template <> struct V2Lanes<8, 8> { static constexpr int WP = 8, PP = 4, WN = 8, PN = 4; };
template <> struct V2Lanes<10, 4> { static constexpr int WP = 4, PP = 4, WN = 16, PN = 1; };
template <> struct V2Lanes<20, 11> { static constexpr int WP = 16, PP = 4, WN = 32, PN = 2; };
template <> struct V2Lanes<27, 27> { static constexpr int WP = 32, PP = 2, WN = 32, PN = 2; };

template <int S, int Q, bool NARROW = false>
struct V2Plan {
    using L = V2Lanes<S, Q, NARROW>;
    static constexpr int WP = L::WP, WN = L::WN, LPE = L::WP * L::PP;
    static_assert(LPE == L::WN * L::PN && LPE <= 64 && Q <= WP && S <= WN, "lanes of one element");
    static constexpr int KP = (S + L::PP - 1) / L::PP;   // nodes a part sums (point stage)
    static constexpr int QN = (Q + L::PN - 1) / L::PN;   // points a part sums (node stage)
    int q, k;            // the lane's point and node (clamped)
    bool point, node;    // whether it has one
    int kp[KP];          // the nodes of the lane's part (clamped, weight 0 past the last)
    float dp[KP][3];     // their dN at point q
    int qn[QN];          // the points of the lane's part
    float dn[QN][3];     // dN of node k there
    __device__ __forceinline__ void place(int lane) {
        const int sp = lane % WP, sn = lane % WN;
        point = sp < Q;
        node = sn < S;
        q = point ? sp : Q - 1;
        k = node ? sn : S - 1;
    }
    __device__ __forceinline__ void init(const float* dN, int lane) {
#pragma unroll
        for (int j = 0; j < KP; ++j) {
            const int n = lane / WP * KP + j;
            const bool in = n < S;
            kp[j] = in ? n : S - 1;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float d = gload(dN, (q * S + kp[j]) * 3 + c);
                dp[j][c] = in ? d : 0.f;
            }
        }
#pragma unroll
        for (int j = 0; j < QN; ++j) {
            const int n = lane / WN * QN + j;
            const bool in = n < Q;
            qn[j] = in ? n : Q - 1;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float d = gload(dN, (qn[j] * S + k) * 3 + c);
                dn[j][c] = in ? d : 0.f;
            }
        }
    }
};

// Both constraints of the element whose node values are x[0 .. S) in LDS (xyz;
// w the inverse mass), moved in place.  sP: Q rows of 3 float4 of scratch of
// the lane group.  Every lane of the wave must call it.
template <class P_>
__device__ __forceinline__ void v2_project(const MaterialView& mt, float dt, const P_& pl, const float JXi[9], float V,
                                           float4* x, float4* sP) {
    const float alpha_nh = 1.f + mt.mu / mt.lambda;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        float Jx[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) Jx[i] = 0.f;
#pragma unroll
        for (int j = 0; j < P_::KP; ++j) {
            const float4 u = x[pl.kp[j]];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                Jx[3 * c] = fmaf(u.x, pl.dp[j][c], Jx[3 * c]);
                Jx[3 * c + 1] = fmaf(u.y, pl.dp[j][c], Jx[3 * c + 1]);
                Jx[3 * c + 2] = fmaf(u.z, pl.dp[j][c], Jx[3 * c + 2]);
            }
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) Jx[i] = parts_sum<P_::WP, P_::LPE>(Jx[i]);
        float F[9], P[9], Ps[9], e;
        deformation_gradient(Jx, JXi, F);
        xpbd_material(mt.material, m, alpha_nh, F, P, e);
        scale_stress(P, JXi, V, Ps);
        if (pl.point) {   // the parts hold the same values
            sP[3 * pl.q] = make_float4(Ps[0], Ps[1], Ps[2], Ps[3]);
            sP[3 * pl.q + 1] = make_float4(Ps[4], Ps[5], Ps[6], Ps[7]);
            sP[3 * pl.q + 2] = make_float4(Ps[8], 0.f, 0.f, 0.f);
        }
        const float C = lanes_sum<P_::WP>(pl.point ? e * V : 0.f);
        wave_lds_sync();
        float g0 = 0.f, g1 = 0.f, g2 = 0.f;
#pragma unroll
        for (int j = 0; j < P_::QN; ++j) {
            const float4 a = sP[3 * pl.qn[j]], b = sP[3 * pl.qn[j] + 1];
            const float c = sP[3 * pl.qn[j] + 2].x;
            g0 += a.x * pl.dn[j][0] + a.w * pl.dn[j][1] + b.z * pl.dn[j][2];
            g1 += a.y * pl.dn[j][0] + b.x * pl.dn[j][1] + b.w * pl.dn[j][2];
            g2 += a.z * pl.dn[j][0] + b.y * pl.dn[j][1] + c * pl.dn[j][2];
        }
        g0 = parts_sum<P_::WN, P_::LPE>(g0);
        g1 = parts_sum<P_::WN, P_::LPE>(g1);
        g2 = parts_sum<P_::WN, P_::LPE>(g2);
        const float4 u = x[pl.k];
        const float sn = pl.node ? (g0 * g0 + g1 * g1 + g2 * g2) * u.w : 0.f;
        const float ssum = lanes_sum<P_::WN>(sn);
        const float stiff = (m == 0) ? mt.lambda : mt.mu;
        const float alpha = 4.f * C / (stiff * dt * dt);
        const float beta = C < 1e-12f ? 0.f : -2.f * C / (ssum + alpha);
        wave_lds_sync();   // every lane has read x
        if (pl.node) {
            const float s = beta * u.w;
            x[pl.k] = make_float4(u.x + s * g0, u.y + s * g1, u.z + s * g2, u.w);
        }
        wave_lds_sync();
    }
}

// One group of LPE lanes per element, one-wave blocks (an element's lanes
// never span waves, so no workgroup barrier is needed and the blocks spread
// over the chip).  Bound by one wave's chain: launch 1.6 us, three dependent
// loads, then about 950 instructions (27 nodes).  A frame of 50 substeps of the
// 32 x 8 x 8 beams: 27-node hexahedra 4.84 -> 2.76 ms (227 elements per
// colour), 20-node tetrahedra 10.16 -> 7.25 ms (424 per colour), against
// 256-thread blocks with workgroup barriers, rolled sums and 4-byte LDS reads.
// The arguments the chain starts with come first and are preloaded into scalar
// registers; the node ids lie in colour order, so they do not wait for the
// element id, and the positions are issued before the dN table (P2 64x16x16,
// 3,300 elements per colour: 161 -> 147 us a substep).
template <int S, int Q, bool NARROW>
__global__ __launch_bounds__(64) void k_xpbd_v2(const int* topo, int first, int count, XpbdArgs a) {
    using P_ = V2Plan<S, Q, NARROW>;
    constexpr int EPB = 64 / P_::LPE;
    __shared__ float4 sx[EPB][S];
    __shared__ float4 sP[EPB][Q * 3];
    const int le = threadIdx.x / P_::LPE, lane = threadIdx.x % P_::LPE;
    const int ei = blockIdx.x * EPB + le;
    const bool valid = ei < count;
    // a group past the colour's end works on its last element and stores nothing
    const int at = first + (valid ? ei : count - 1);
    P_ pl;
    pl.place(lane);
    const int vid = gload(topo, static_cast<size_t>(at) * S + pl.k);
    const int eid = gload(a.eids, at);
    __builtin_amdgcn_sched_barrier(0);
    float4 u = gload(static_cast<const float4*>(a.ps.p), vid);
    const float w = gload(a.ps.w, vid);
    float JXi[9], V;
    load_element_record(a.fem, eid, pl.q, JXi, V);
    __builtin_amdgcn_sched_barrier(0);
    pl.init(a.fem.dN, lane);
    const float keep = u.w;
    u.w = w;
    if (lane < S) sx[le][lane] = u;
    wave_lds_sync();
    v2_project(a.mt, a.dt, pl, JXi, V, sx[le], sP[le]);
    if (valid && lane < S) {
        const float4 r = sx[le][lane];
        gstore(a.ps.p, vid, make_float4(r.x, r.y, r.z, keep));
    }
}

template <int S, int Q>
void launch_v0(const XpbdArgs& a, hipStream_t s) {
    const int grid = (a.count + 255) / 256;
    hipLaunchKernelGGL((k_xpbd_v0<S, Q>), dim3(grid), dim3(256), 0, s, a);
}

template <int S, int Q, bool NARROW = false>
void launch_v2(const XpbdArgs& a, hipStream_t s) {
    constexpr int EPB = 64 / V2Plan<S, Q, NARROW>::LPE;
    hipLaunchKernelGGL((k_xpbd_v2<S, Q, NARROW>), dim3((a.count + EPB - 1) / EPB), dim3(64), 0, s, a.topo, a.first,
                       a.count, a);
}

}  // namespace

void launch_xpbd_p1_resident(const XpbdResidentArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_xpbd_p1_resident, dim3(1), dim3(kXpbdResidentThreads), 0, s, a);
}

bool launch_xpbd(int S, int Q, bool v0_form, const XpbdArgs& a, hipStream_t s) {
    if (a.count <= 0) return true;
    if (v0_form) {
        if (S == 4 && Q == 1) {
            hipLaunchKernelGGL(k_xpbd_p1, dim3((a.count + 63) / 64), dim3(64), 0, s, a.p1_nodes, a.first, a.count, a);
            return true;
        }
        if (S == 8 && Q == 8) { launch_v0<8, 8>(a, s); return true; }
        if (S == 10 && Q == 4) { launch_v0<10, 4>(a, s); return true; }
        if (S == 20 && Q == 11) { launch_v0<20, 11>(a, s); return true; }
        if (S == 27 && Q == 27) { launch_v0<27, 27>(a, s); return true; }
        return false;
    }
    if (S == 8 && Q == 8) {
        // 32 lanes per element up to one wave per SIMD (2,048 elements), 8 past
        // that.  A substep (the ten colours and the vertex pass) with 32 and with
        // 8 lanes: largest colour 2,047 elements (64x16x16 beam) 45.2 and 45.7 us,
        // 2,303 (72x16x16) 49.3 and 46.7, 4,095 51.9 and 47.7, 8,191 68.4 and 52.2
        if (a.count <= 2048) launch_v2<8, 8>(a, s);
        else launch_v2<8, 8, true>(a, s);
        return true;
    }
    if (S == 10 && Q == 4) { launch_v2<10, 4>(a, s); return true; }
    if (S == 20 && Q == 11) { launch_v2<20, 11>(a, s); return true; }
    if (S == 27 && Q == 27) { launch_v2<27, 27>(a, s); return true; }
    return false;
}

}  // namespace oe
