#include "oe_batch.hpp"

#include "oe_q2.hpp"

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <stdexcept>

namespace oe {

namespace {
constexpr int kBlock = 256;
GPU_Box_Limit* find_box(const Scene& s) {
    GPU_Box_Limit* box = nullptr;
    for (const auto& c : s.integrator->_constraints) {
        if (auto* b = dynamic_cast<GPU_Box_Limit*>(c.get())) {
            if (box) throw std::invalid_argument("batched scenes support one box limit");
            box = b;
        }
    }
    return box;
}
}  // namespace

std::map<int, GatherTile> default_tiles() {
    std::map<int, GatherTile> t;
    for (Element e : {Tetra, Hexa, Tetra10, Tetra20, Hexa27}) t[e] = default_tile(e);
    return t;
}

bool needs_gather(const Scene& s) {
    return s.mesh.element != Tetra10 && s.mesh.element != Hexa27 && !s.vbd_fem->fits_tasks();
}

// A batch's launches are a server's (default_tile) or much longer, and run
// beside one another.
//  * Q2 blocks of 28 incidences from kLongBlocks of them per colour pass on (2 a
//    SIMD): a block's rounds then overlap other blocks'.  Below, 14 (two rounds
//    in place of four): 24 beams of 32x8x8 (1,650 blocks of 28) step in 7.7 ms
//    (8.9 with 28), 32 of them in 9.1 (9.5), 32 mixed beams (2,600) in 14.4 (12.6).
//  * Q2 passes of fewer than 1024 blocks of 14 take the latency form (a scene and
//    a server 512): 4 beams of 32x8x8 (546 blocks) step in 3.6 ms (5.3), 6 in 5.4
//    (5.6), 8 (1,090) in 5.5 either way, 12 in 6.6 (8.0 in the latency form).
//  * P2 passes of fewer than 256 blocks take the latency or split form (512): 16
//    beams of 16x4x4 (88 blocks) step in 1.41 ms (1.47 in the throughput form),
//    64 of them (350) in 1.80 (1.75).
std::map<int, GatherTile> batch_tiles(const std::vector<Scene*>& scenes) {
    constexpr double kLongBlocks = 2048;
    std::map<int, GatherTile> t = default_tiles();
    double per_pass = 0.0;
    for (const Scene* s : scenes) {
        if (needs_gather(*s)) t[s->mesh.element].mode = PASS_GATHER;
        if (s->mesh.element == Hexa27)
            per_pass += 27.0 * s->fem->E / std::max(1, s->vbd_fem->nb_colors());
    }
    if (per_pass >= kLongBlocks * kQ2PencilIncPerBlock) t[Hexa27].inc = kQ2PencilIncPerBlock;
    else t[Hexa27].lat_blocks = 1024;
    t[Tetra10].lat_blocks = 256;
    return t;
}

void check_batchable(const Scene& s) {
    if (!s.vbd_fem) throw std::invalid_argument("batched stepping needs VBD scenes");
    if (s.vbd_fem->version == Better_Coloration)
        throw std::invalid_argument("batched stepping needs a proper colouring (not Better_Coloration)");
    if (s.cfg.rho > 0.f) throw std::invalid_argument("batched stepping does not run the Chebyshev acceleration");
    if (s.vbd_fem->shuffle) throw std::invalid_argument("batched stepping uses the ascending colour order");
    for (const auto& c : s.integrator->_constraints)
        if (!dynamic_cast<GPU_Fix_Constraint*>(c.get()) && !dynamic_cast<GPU_Box_Limit*>(c.get()))
            throw std::invalid_argument("unsupported constraint in a batched scene");
    (void)find_box(s);
}

std::vector<unsigned char> fixed_flags(const Scene& s) {
    std::vector<unsigned char> f(s.ps->n, 0);
    if (s.fix)
        for (int id : s.fix->ids) f[id] = 1;
    return f;
}

namespace {
GatherTile tile_of(const std::map<int, GatherTile>& tiles, Element el) {
    const auto it = tiles.find(el);
    return it != tiles.end() ? it->second : default_tile(el);
}
}  // namespace

SceneDev make_scene_dev(Scene& s, const unsigned char* fixed, const std::map<int, GatherTile>& tiles) {
    check_batchable(s);
    SceneDev d{};
    const GatherTile t = tile_of(tiles, s.mesh.element);
    if (t.mode == PASS_TASKS && s.mesh.element == Hexa27 && !s.vbd_fem->has_q2_basis)
        throw std::invalid_argument("no tensor factors for this 27-node hexahedron");
    d.ju = t.mode == PASS_CACHE ? s.vbd_fem->ensure_ju() : nullptr;
    d.fblocks = d.fblocks_lat = d.fblocks_split = nullptr;
    if (t.mode == PASS_TASKS) {
        d.fblocks = s.vbd_fem->throughput_tables(t.inc).blocks.get();
        const TaskTables* lt = s.vbd_fem->latency_tables();
        d.fblocks_lat = lt ? lt->blocks.get() : nullptr;
        const TaskTables* sp = s.vbd_fem->split_form();
        d.fblocks_split = sp ? sp->blocks.get() : nullptr;
    }
    d.ps = s.ps->get_parameters();
    d.fem = s.fem->fem_view();
    d.own = OwnersView{s.vbd_fem->d_slot_vid.get(), s.vbd_fem->d_slot_nbo.get(), s.vbd_fem->d_own.get()};
    d.mt = s.fem->mt;
    auto* vbd = dynamic_cast<GPU_VBD*>(s.integrator.get());
    if (!vbd) throw std::logic_error("VBD scene without a GPU_VBD integrator");
    d.y = vbd->y.get();
    d.damping = s.vbd_fem->damping;
    d.iterations = vbd->iteration;
    for (int k = 0; k < 3; ++k) d.g[k] = vbd->gravity[k];
    d.fixed = s.fix ? fixed : nullptr;
    if (s.fix) {
        std::memcpy(d.fix_com, s.fix->t.com, sizeof(d.fix_com));
        std::memcpy(d.fix_offset, s.fix->t.offset, sizeof(d.fix_offset));
        std::memcpy(d.fix_R, s.fix->t.R, sizeof(d.fix_R));
    }
    if (GPU_Box_Limit* box = find_box(s)) {
        d.has_box = 1;
        for (int k = 0; k < 3; ++k) {
            d.box_min[k] = box->pmin[k];
            d.box_max[k] = box->pmax[k];
        }
    }
    return d;
}

void Schedule::clear() {
    segs.clear();
    glaunches.clear();
    vsegs.clear();
    vblocks = 0;
    jlaunches.clear();
    jsegs.clear();
    max_iterations = 0;
    vertex_updates_per_substep = 0;
    algorithmic_bytes_per_substep = 0.0;
    algorithmic_bytes_by_element.clear();
    vertex_updates_by_element.clear();
}

void Schedule::build(const std::vector<Scene*>& scenes, const std::vector<int>& table_index,
                     const std::map<int, GatherTile>& tiles, const Schedule* whole) {
    clear();
    int max_colors = 0;
    for (Scene* s : scenes) {
        max_colors = std::max(max_colors, s->vbd_fem->nb_colors());
        max_iterations = std::max(max_iterations, s->cfg.iterations);
        vertex_updates_per_substep += static_cast<int64_t>(s->ps->n) * s->cfg.iterations;
        const int S = s->fem->S, Q = s->fem->Q;
        const double bytes =
            (static_cast<double>(s->fem->E) * S * (40.0 * Q + 16.0 * S + 8.0) + 56.0 * s->ps->n) * s->cfg.iterations;
        algorithmic_bytes_per_substep += bytes;
        algorithmic_bytes_by_element[s->mesh.element] += bytes;
        vertex_updates_by_element[s->mesh.element] += static_cast<int64_t>(s->ps->n) * s->cfg.iterations;
    }
    static const Element order[] = {Tetra, Tetra10, Tetra20, Hexa, Hexa27};
    for (int c = 0; c < max_colors; ++c) {
        for (Element el : order) {
            GLaunch gl{};
            gl.color = c;
            gl.element = el;
            gl.seg_first = static_cast<int>(segs.size());
            // Task passes take the latency form when every scene of the launch has
            // its vertex blocks and the throughput form would give fewer than the
            // tile's latency_blocks (2 per CU).
            const GatherTile et = tile_of(tiles, el);
            if (whole) {
                for (const GLaunch& w : whole->glaunches)
                    if (w.color == c && w.element == el) gl.form = w.form;
            } else if (et.mode == PASS_TASKS) {
                bool all = true;
                int64_t through_blocks = 0, incidences = 0;
                for (Scene* s : scenes) {
                    if (s->mesh.element != el || c >= s->vbd_fem->nb_colors()) continue;
                    if (!s->vbd_fem->latency_tables()) all = false;
                    through_blocks += s->vbd_fem->throughput_tables(et.inc).color_blocks(c);
                    incidences += s->vbd_fem->owners.color_incidences[c];
                }
                if (all && through_blocks < et.lat_blocks)
                    gl.form = el == Tetra10 && incidences <= kSplitIncidences ? TASKS_SPLIT : TASKS_LATENCY;
            }
            bool any = false;
            for (size_t i = 0; i < scenes.size(); ++i) {
                Scene* s = scenes[i];
                if (s->mesh.element != el || c >= s->vbd_fem->nb_colors()) continue;
                const GatherTile t = tile_of(tiles, el);
                const int first = s->vbd_fem->owners.color_begin[c];
                const int count = s->vbd_fem->owners.color_begin[c + 1] - first;
                if (count <= 0) continue;
                if (!any) {
                    gl.S = s->fem->S;
                    gl.Q = s->fem->Q;
                    gl.L = t.L;
                    gl.QL = t.QL;
                    gl.mode = t.mode;
                    gl.inc = t.inc;
                    any = true;
                    if (gl.mode == PASS_TASKS) q2_basis = s->vbd_fem->q2_basis;
                }
                if (gl.mode == PASS_TASKS) {
                    // fused tasks: one block per vertex block of the colour
                    const TaskTables* tt = gl.form == TASKS_SPLIT     ? s->vbd_fem->split_form()
                                           : gl.form == TASKS_LATENCY ? s->vbd_fem->latency_tables()
                                                                      : &s->vbd_fem->throughput_tables(t.inc);
                    if (!tt) throw std::logic_error("vertex blocks not prepared");
                    const int nfb = tt->color_blocks(c);
                    segs.push_back(BatchSeg{table_index[i], tt->color_begin[c], nfb, gl.nblocks});
                    gl.nblocks += nfb;
                } else {
                    // gather: L lanes per slot
                    const int nb = static_cast<int>((static_cast<int64_t>(count) * gl.L + kBlock - 1) / kBlock);
                    segs.push_back(BatchSeg{table_index[i], first, count, gl.nblocks});
                    gl.nblocks += nb;
                }
                gl.slots += count;
                gl.incidences += s->vbd_fem->owners.color_incidences[c];
            }
            gl.seg_count = static_cast<int>(segs.size()) - gl.seg_first;
            if (any) glaunches.push_back(gl);
        }
    }
    for (size_t i = 0; i < scenes.size(); ++i) {
        const int n = scenes[i]->ps->n;
        vsegs.push_back(VSeg{table_index[i], n, vblocks});
        vblocks += (n + kBlock - 1) / kBlock;
    }
    for (Element el : order) {
        if (tile_of(tiles, el).mode != PASS_CACHE) continue;
        JLaunch jl{};
        jl.seg_first = static_cast<int>(jsegs.size());
        bool any = false;
        for (size_t i = 0; i < scenes.size(); ++i) {
            Scene* s = scenes[i];
            if (s->mesh.element != el) continue;
            const int E = s->fem->E;
            if (E <= 0) continue;
            if (static_cast<int64_t>(E) * s->fem->Q > INT32_MAX)
                throw std::invalid_argument("scene too large for the gradient cache");
            jl.S = s->fem->S;
            jl.Q = s->fem->Q;
            any = true;
            const int epb = refresh_elements_per_block(jl.S, jl.Q);
            if (epb <= 0) throw std::invalid_argument("unsupported element");
            jsegs.push_back(VSeg{table_index[i], E, jl.nblocks});
            jl.nblocks += (E + epb - 1) / epb;
        }
        jl.seg_count = static_cast<int>(jsegs.size()) - jl.seg_first;
        if (any) jlaunches.push_back(jl);
    }
}

namespace {
template <typename T>
void upload_grow(Engine* eng, DBuf<T>& buf, const std::vector<T>& h, hipStream_t s) {
    if (buf.size() < h.size() || !buf.get()) buf.allocate(&eng->pool, std::max<size_t>(h.size() + h.size() / 2, 16));
    if (!h.empty()) OE_HIP(hipMemcpyAsync(buf.get(), h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s));
}
}  // namespace

void DeviceSchedule::upload(Engine* eng, const Schedule& s, hipStream_t stream, bool sync) {
    upload_grow(eng, segs, s.segs, stream);
    upload_grow(eng, vsegs, s.vsegs, stream);
    upload_grow(eng, jsegs, s.jsegs, stream);
    if (sync) OE_HIP(hipStreamSynchronize(stream));
}

void GatherTimer::before(hipStream_t s, int tag) {
    if (!enabled) return;
    while (pool.size() < used + 2) {
        hipEvent_t ev;
        OE_HIP(hipEventCreate(&ev));
        pool.push_back(ev);
    }
    tags.resize(used / 2 + 1);
    tags[used / 2] = tag;
    OE_HIP(hipEventRecord(pool[used], s));
}

void GatherTimer::after(hipStream_t s) {
    if (!enabled) return;
    OE_HIP(hipEventRecord(pool[used + 1], s));
    used += 2;
}

void GatherTimer::collect(hipStream_t s) {
    if (used == 0) return;
    OE_HIP(hipStreamSynchronize(s));
    for (size_t i = 0; i + 1 < used; i += 2) {
        float t = 0.f;
        OE_HIP(hipEventElapsedTime(&t, pool[i], pool[i + 1]));
        ms += t;
        launches++;
        tag_ms[tags[i / 2]] += t;
        tag_launches[tags[i / 2]]++;
    }
    used = 0;
}

GatherTimer::~GatherTimer() {
    for (hipEvent_t e : pool) (void)hipEventDestroy(e);
}

namespace {
// One schedule's launches on its stream.
struct Chain {
    const Schedule& sch;
    hipStream_t stream;
    GatherTimer* timer;
    BatchVArgs v;
    BatchGatherArgs g;
    BatchRefreshArgs r;
    BatchQ2FusedArgs tk;
    BatchFusedArgs ft;

    Chain(const Schedule& s, const DeviceSchedule& dev, const SceneDev* d_scenes, float h, hipStream_t st,
          GatherTimer* t)
        : sch(s), stream(st), timer(t), v{d_scenes, dev.vsegs.get(), static_cast<int>(s.vsegs.size()), h, 0},
          g{d_scenes, dev.segs.get(), 0, 0, 0, h}, r{d_scenes, dev.jsegs.get(), 0, 0, 0},
          tk{d_scenes, dev.segs.get(), 0, 0, 0, h, s.q2_basis, 0}, ft{d_scenes, dev.segs.get(), 0, 0, 0, h, 0} {}

    void predict() { launch_batch_predict(v, sch.vblocks, stream); }
    void velocity() { launch_batch_velocity(v, sch.vblocks, stream); }
    void refresh(int it) {
        g.iteration = r.iteration = tk.iteration = ft.iteration = v.iteration = it;
        for (const Schedule::JLaunch& jl : sch.jlaunches) {
            r.seg_first = jl.seg_first;
            r.seg_count = jl.seg_count;
            if (!launch_batch_ju_refresh(jl.S, jl.Q, r, jl.nblocks, stream))
                throw std::invalid_argument("unsupported element in batch");
        }
    }
    void pass(const Schedule::GLaunch& gl) {
        g.seg_first = tk.seg_first = ft.seg_first = gl.seg_first;
        g.seg_count = tk.seg_count = ft.seg_count = gl.seg_count;
        if (timer) timer->before(stream, gl.element);
        if (gl.mode == PASS_TASKS && gl.element == Hexa27) {
            tk.latency = gl.form == TASKS_LATENCY ? 1 : 0;
            if (gl.form == TASKS_THROUGHPUT && q2_pencil(gl.inc))
                launch_batch_q2_pencil(tk, gl.nblocks, stream);
            else
                launch_batch_q2_fused(tk, gl.nblocks, stream);
        } else if (gl.mode == PASS_TASKS) {
            ft.form = gl.form;
            if (!launch_batch_fused_tasks(gl.S, gl.Q, ft, gl.nblocks, stream))
                throw std::invalid_argument("unsupported element in batch");
        } else if (!launch_batch_gather(gl.S, gl.Q, gl.L, gl.QL, gl.mode == PASS_CACHE, g, gl.nblocks, stream)) {
            throw std::invalid_argument("unsupported gather tile in batch");
        }
        if (timer) timer->after(stream);
    }
    void constraints() { launch_batch_fix_box(v, sch.vblocks, stream); }
};

// The chains' launches dealt out in turn, so that none waits for the host.
void run_chains(std::vector<Chain>& chains, int substeps) {
    int iterations = 0;
    for (const Chain& c : chains) iterations = std::max(iterations, c.sch.max_iterations);
    for (int sub = 0; sub < substeps; ++sub) {
        for (Chain& c : chains) c.predict();
        for (int it = 0; it < iterations; ++it) {
            auto runs = [&](const Chain& c) { return it < c.sch.max_iterations; };
            size_t passes = 0;
            for (Chain& c : chains)
                if (runs(c)) {
                    c.refresh(it);
                    passes = std::max(passes, c.sch.glaunches.size());
                }
            for (size_t i = 0; i < passes; ++i)
                for (Chain& c : chains)
                    if (runs(c) && i < c.sch.glaunches.size()) c.pass(c.sch.glaunches[i]);
            for (Chain& c : chains)
                if (runs(c)) c.constraints();
        }
        for (Chain& c : chains) c.velocity();
    }
}
}  // namespace

void launch_schedule(const Schedule& sch, const DeviceSchedule& dev, const SceneDev* d_scenes, float dt, int substeps,
                     hipStream_t stream, GatherTimer* timer) {
    if (sch.vsegs.empty()) return;
    std::vector<Chain> chains;
    chains.emplace_back(sch, dev, d_scenes, dt / static_cast<float>(substeps), stream, timer);
    run_chains(chains, substeps);
}

namespace {
// The scenes of a batch by chain: 27-node hexahedra apart from the other
// element types, and up to 3 chains of about equal work, the class with more
// work per chain split first.  A chain's passes wait for one another with the
// chip partly idle (a pass's last blocks, its launch, blocks that all wait on
// the same loads); other chains' blocks run there.  Mixed beams of 8-64 x 4-16 x
// 4-16 cells, 4 / 8 / 16 / 32 / 64 / 128 scenes, ms per 4 substeps: on one stream
// 21.8 / 23.5 / 26.1 / 34.6 / 53.5 / 87.6; with the Q2 passes on a second stream
// joined in every iteration 18.2 / 19.4 / 20.9 / 30.2 / 45.9 / 75.1; now 17.0 /
// 18.1 / 19.2 / 25.0 / 39.4 / 70.9.
// A fourth chain, on as many hardware queues as the runtime has by default, was
// slower again (16 scenes 25.2, 32 scenes 31.7, 64 scenes 47.0).
// A chain keeps at least kChainPoints (incidence, quadrature point) pairs per
// colour pass (about 15,000 Q2 incidences, or 100,000 P2): below, the passes are
// launch-bound and more of them only cost the host.
constexpr int kMaxChains = 1 + Engine::kSideStreams;
// And no chain may hold over kChainBalance times its share, or the others wait
// for it at the end of the step.
constexpr double kChainPoints = 4e5, kChainBalance = 1.15;
std::vector<std::vector<int>> group_scenes(const std::vector<Scene*>& scenes) {
    std::vector<int> member[2];   // Hexa27, the others
    double total[2] = {0.0, 0.0}, pass[2] = {0.0, 0.0};
    auto work = [&](int i) { return static_cast<double>(scenes[i]->fem->E) * scenes[i]->fem->S * scenes[i]->fem->Q; };
    for (int i = 0; i < static_cast<int>(scenes.size()); ++i) {
        const int k = scenes[i]->mesh.element == Hexa27 ? 0 : 1;
        member[k].push_back(i);
        total[k] += work(i);
        pass[k] += work(i) / std::max(1, scenes[i]->vbd_fem->nb_colors());
    }
    // member[k] in n groups: largest scene first, each to the group with the least work so far
    for (std::vector<int>& m : member)
        std::stable_sort(m.begin(), m.end(), [&](int a, int b) { return work(a) > work(b); });
    auto dealt = [&](int k, int n) {
        std::vector<std::vector<int>> g(n);
        std::vector<double> load(n, 0.0);
        for (int i : member[k]) {
            const size_t j = std::min_element(load.begin(), load.end()) - load.begin();
            g[j].push_back(i);
            load[j] += work(i);
        }
        if (*std::max_element(load.begin(), load.end()) * n > kChainBalance * total[k]) g.clear();
        return g;
    };
    std::vector<std::vector<int>> groups[2];
    for (int k = 0; k < 2; ++k)
        if (!member[k].empty()) groups[k] = dealt(k, 1);
    while (groups[0].size() + groups[1].size() < kMaxChains) {
        std::vector<std::vector<int>> next;
        int best = -1;
        for (int k = 0; k < 2; ++k) {
            const int n = static_cast<int>(groups[k].size()) + 1;
            if (n == 1 || pass[k] < kChainPoints * n) continue;
            if (best >= 0 && total[k] / (n - 1) <= total[best] / groups[best].size()) continue;
            std::vector<std::vector<int>> g = dealt(k, n);
            if (g.empty()) continue;
            next = std::move(g);
            best = k;
        }
        if (best < 0) break;
        groups[best] = std::move(next);
    }
    std::vector<std::vector<int>> out;
    for (auto& g : groups) out.insert(out.end(), g.begin(), g.end());
    for (std::vector<int>& g : out) std::sort(g.begin(), g.end());
    return out;
}
}  // namespace

Batch::Batch(Engine* e, std::vector<Scene*> sc) : eng(e), scenes(std::move(sc)) {
    if (scenes.empty()) throw std::invalid_argument("empty batch");
    for (size_t i = 0; i < scenes.size(); ++i) {
        Scene* s = scenes[i];
        if (!s) throw std::invalid_argument("null scene in batch");
        if (s->eng != eng) throw std::invalid_argument("scene belongs to another engine");
        // two segments of one launch would update the same vertices
        if (std::find(scenes.begin(), scenes.begin() + static_cast<long>(i), s) != scenes.begin() + static_cast<long>(i))
            throw std::invalid_argument("a scene appears twice in the batch");
        if (s->server) throw std::logic_error("the scene is held by a server");
        check_batchable(*s);
    }
    tiles = batch_tiles(scenes);
    flags.reserve(scenes.size());
    for (Scene* s : scenes) flags.emplace_back(&eng->pool, fixed_flags(*s));
    d_scenes.allocate(&eng->pool, scenes.size());
    rebuild();
    for (Scene* s : scenes) s->batches.push_back(this);
}

Batch::~Batch() {
    drop_graph();
    if (fork) (void)hipEventDestroy(fork);
    for (Scene* s : scenes) {
        if (!s) continue;
        auto& v = s->batches;
        v.erase(std::remove(v.begin(), v.end(), this), v.end());
    }
}

void Batch::scene_destroyed(Scene* s) {
    for (Scene*& p : scenes)
        if (p == s) p = nullptr;
    broken = true;
    drop_graph();
}

void Batch::rebuild() {
    drop_graph();
    std::vector<SceneDev> host;
    for (size_t i = 0; i < scenes.size(); ++i) host.push_back(make_scene_dev(*scenes[i], flags[i].get(), tiles));
    d_scenes.upload(host, eng->stream);
    std::vector<int> idx(scenes.size());
    for (size_t i = 0; i < idx.size(); ++i) idx[i] = static_cast<int>(i);
    sched.build(scenes, idx, tiles);
    dsched.upload(eng, sched, eng->stream, true);
    const std::vector<std::vector<int>> parts = group_scenes(scenes);
    if (groups.size() != parts.size()) groups = std::vector<Group>(parts.size());
    for (size_t i = 0; i < parts.size(); ++i) {
        std::vector<Scene*> sc;
        for (int k : parts[i]) sc.push_back(scenes[k]);
        groups[i].sched.build(sc, parts[i], tiles, &sched);
        groups[i].dev.upload(eng, groups[i].sched, eng->stream, true);
        groups[i].stream = i > 0 ? eng->side_stream(static_cast<int>(i) - 1) : eng->stream;
        if (i > 0 && !groups[i].join) OE_HIP(hipEventCreateWithFlags(&groups[i].join, hipEventDisableTiming));
    }
    if (!fork) OE_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
}

void Batch::launch(float dt, int substeps) {
    if (streams != 2 || timer.enabled || groups.size() < 2) {
        launch_schedule(sched, dsched, d_scenes.get(), dt, substeps, eng->stream, timer.enabled ? &timer : nullptr);
        return;
    }
    const float h = dt / static_cast<float>(substeps);
    std::vector<Chain> chains;
    OE_HIP(hipEventRecord(fork, eng->stream));
    for (Group& g : groups) {
        if (g.join) OE_HIP(hipStreamWaitEvent(g.stream, fork, 0));
        chains.emplace_back(g.sched, g.dev, d_scenes.get(), h, g.stream, nullptr);
    }
    auto join = [&] {
        for (Group& g : groups)
            if (g.join) {
                OE_HIP(hipEventRecord(g.join, g.stream));
                OE_HIP(hipStreamWaitEvent(eng->stream, g.join, 0));
            }
    };
    try {
        run_chains(chains, substeps);
    } catch (...) {
        join();   // what was launched stays ordered before the engine's later work
        throw;
    }
    join();
}

void Batch::set_tile(Element e, GatherTile t) {
    if (broken) throw std::logic_error("a scene of this batch was destroyed");
    tiles[e] = t;
    rebuild();
}

void Batch::set_graph(bool on) {
    if (!on) drop_graph();
    use_graph = on;
}

void Batch::set_streams(int n) {
    if (n != streams) drop_graph();   // a captured graph holds the old launch structure
    streams = n;
}

void Batch::drop_graph() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    graph_exec = nullptr;
    graph = nullptr;
}

void Batch::step(float dt, int substeps) {
    if (broken) throw std::logic_error("a scene of this batch was destroyed");
    if (!(dt > 0.f) || substeps <= 0) throw std::invalid_argument("step needs dt > 0 and substeps > 0");
    if (!use_graph || timer.enabled) {
        launch(dt, substeps);
    } else {
        if (!graph_exec || graph_dt != dt || graph_sub != substeps) {
            drop_graph();
            OE_HIP(hipStreamBeginCapture(eng->stream, hipStreamCaptureModeThreadLocal));
            try {
                launch(dt, substeps);
            } catch (...) {
                hipGraph_t g = nullptr;
                (void)hipStreamEndCapture(eng->stream, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            OE_HIP(hipStreamEndCapture(eng->stream, &graph));
            OE_HIP(hipGraphInstantiate(&graph_exec, graph, nullptr, nullptr, 0));
            graph_dt = dt;
            graph_sub = substeps;
        }
        OE_HIP(hipGraphLaunch(graph_exec, eng->stream));
    }
    OE_LAUNCH_CHECK();
    for (Scene* s : scenes) s->steps_done++;
}

}  // namespace oe
