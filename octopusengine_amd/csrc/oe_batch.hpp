// Batched VBD stepping of many independent scenes on one GPU.
//
// The reference steps each scene (entity) on its own, one launch per colour
// (src/GPU/VBD/GPU_VBD_FEM.cu:712-756, driven scene after scene by
// src/Core/Engine.cpp:15-21).  Here a launch covers colour c of every scene
// that has a colour c: scenes are independent, so colour c of scene A and
// colour c of scene B can be solved concurrently, and a launch carries enough
// vertices to fill the chip.  Per step the launch sequence is
//   predictor (all vertices of all scenes)
//   for each iteration:  refresh of the cached displacement gradients (per
//                          element type whose tile caches them)
//                        for each global colour c, for each element type:
//                          gather + local solve of colour c
//                        fixation + box limit (all vertices, one fused kernel)
//   velocity update
// Each scene still sees the reference's order: ascending colours, constraints
// after every sweep.  A batch deals its scenes into up to three groups, each with
// this sequence on a stream of its own (group_scenes in oe_batch.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <vector>

#include "oe_gather.hpp"
#include "oe_scene.hpp"

namespace oe {

// Launch plan for a set of scenes.  Scene indices refer to a SceneDev table.
// Every launch covers a contiguous run of segments whose block_begin values
// are launch-local; kernels find their segment by binary search, so the plan
// is O(segments), not O(blocks), to build and upload.
struct Schedule {
    struct GLaunch {
        int color, element, S, Q, L, QL;
        int mode;                         // PassMode
        int form;                         // of a task pass: TaskForm (27-node hexahedra: throughput or latency)
        int inc = 0;                      // task pass: the tile's incidences per throughput-form block
        int seg_first, seg_count, nblocks;   // gather: slot ranges; tasks: vertex-block ranges
        int64_t slots;   // vertex slots covered (all scenes)
        int64_t incidences;
    };
    // refresh of cached gradients: one launch per element type, over jsegs
    struct JLaunch {
        int S, Q;
        int seg_first, seg_count, nblocks;
    };
    std::vector<BatchSeg> segs;
    std::vector<GLaunch> glaunches;   // ascending colour, then element type
    std::vector<VSeg> vsegs;          // every vertex of every scene, one launch
    int vblocks = 0;
    std::vector<JLaunch> jlaunches;
    std::vector<VSeg> jsegs;          // count = the scene's elements
    q2::Basis1D q2_basis{};
    int max_iterations = 0;
    int64_t vertex_updates_per_substep = 0;
    double algorithmic_bytes_per_substep = 0.0;   // gather kernels, all iterations
    std::map<int, double> algorithmic_bytes_by_element;    // the same per element type
    std::map<int, int64_t> vertex_updates_by_element;

    void clear();
    // scenes[i] is placed at SceneDev table index table_index[i]; task passes
    // too small to fill the GPU take the latency form, or those of a part of a
    // schedule the forms of the whole
    void build(const std::vector<Scene*>& scenes, const std::vector<int>& table_index,
               const std::map<int, GatherTile>& tiles, const Schedule* whole = nullptr);
};

// Device copies of a schedule's tables (grown on demand, reused across uploads).
struct DeviceSchedule {
    DBuf<BatchSeg> segs;
    DBuf<VSeg> vsegs;
    DBuf<VSeg> jsegs;
    void upload(Engine* eng, const Schedule& s, hipStream_t stream, bool sync);
};

// Validates that a scene can be stepped in a batch and describes it for the
// batched kernels.  `fixed` is the scene's per-vertex fixation flag array; the
// scene's gradient cache is allocated when its element type's tile uses it.
SceneDev make_scene_dev(Scene& s, const unsigned char* fixed, const std::map<int, GatherTile>& tiles);
std::vector<unsigned char> fixed_flags(const Scene& s);
void check_batchable(const Scene& s);

// HIP events around colour-pass launches; durations are summed in total and
// per tag (the launch's element type).
struct GatherTimer {
    bool enabled = false;
    std::vector<hipEvent_t> pool;
    std::vector<int> tags;   // one per event pair
    size_t used = 0;
    double ms = 0.0;
    int64_t launches = 0;
    std::map<int, double> tag_ms;
    std::map<int, int64_t> tag_launches;
    void before(hipStream_t s, int tag = 0);
    void after(hipStream_t s);
    void collect(hipStream_t s);
    ~GatherTimer();
};

// Enqueue `substeps` substeps of dt/substeps for every scene of the schedule.
void launch_schedule(const Schedule& sch, const DeviceSchedule& dev, const SceneDev* d_scenes, float dt, int substeps,
                     hipStream_t stream, GatherTimer* timer);

// The tile of every element type: a scene's (default_tile), which a server's
// ticks start with, and what a batch of these scenes starts with.
std::map<int, GatherTile> default_tiles();
std::map<int, GatherTile> batch_tiles(const std::vector<Scene*>& scenes);
// Whether default layouts that are to hold s take its element type to the
// gather: a vertex of more elements than a task block holds, of the types that
// fall back (linear tetrahedra, 8-node hexahedra, 20-node tetrahedra) as the
// scene by itself does.  The other two are refused with such a vertex.
bool needs_gather(const Scene& s);

// A batch registers itself with its scenes (Scene::batches).  A scene may be
// in several batches but appear once per batch, and a scene held by a server
// cannot join one.  Destroying a scene first detaches it: the batch then
// refuses to step (std::logic_error).
struct Batch {
    Batch(Engine* eng, std::vector<Scene*> scenes);
    ~Batch();
    void step(float dt, int substeps);
    void set_graph(bool on);
    void set_streams(int n);   // 1, or 2: the groups side by side
    void set_tile(Element e, GatherTile t);
    void rebuild();
    void scene_destroyed(Scene* s);

    Engine* eng;
    std::vector<Scene*> scenes;
    std::vector<DBuf<unsigned char>> flags;
    DBuf<SceneDev> d_scenes;   // rewritten by rebuild()
    std::map<int, GatherTile> tiles;
    Schedule sched;
    DeviceSchedule dsched;
    GatherTimer timer;

private:
    // Scenes whose steps run on one stream (group 0: the engine's, group i: its
    // side stream i - 1).  Groups share nothing, so a step forks and joins once.
    struct Group {
        Schedule sched;
        DeviceSchedule dev;
        hipStream_t stream = nullptr;
        hipEvent_t join = nullptr;
        Group() = default;
        Group(const Group&) = delete;
        ~Group() {
            if (join) (void)hipEventDestroy(join);
        }
    };
    std::vector<Group> groups;
    hipEvent_t fork = nullptr;
    void launch(float dt, int substeps);
    bool broken = false;   // a scene of the batch was destroyed
    bool use_graph = false;
    int streams = 2;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    float graph_dt = 0.f;
    int graph_sub = 0;
    void drop_graph();
};

}  // namespace oe
