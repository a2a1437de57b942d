// batch.cpp -- the batched form: many independent scenes resident in device
// memory, advanced by persistent SCENE-engine launches (one per size class),
// replayed as a captured hipGraph, with an autotuner over the launch shape.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/bendy2d.h"
#include "batch.h"
#include "engine.h"
#include "kernels.h"
#include "scene_pack.h"

using namespace bd;

namespace bd {

static int fail(int code, const std::string &msg) {
    set_last_error(msg);
    return code;
}

BatchCore::~BatchCore() { release(); }

void BatchCore::release() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    graph_exec = nullptr;
    if (stream) (void)hipStreamSynchronize(stream);
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    if (ev_join) (void)hipEventDestroy(ev_join);
    if (ev_join2) (void)hipEventDestroy(ev_join2);
    if (side) (void)hipStreamDestroy(side);
    if (side2) (void)hipStreamDestroy(side2);
    if (stream && own_stream) (void)hipStreamDestroy(stream);
    ev0 = ev1 = ev_fork = ev_join = ev_join2 = nullptr;
    side = side2 = nullptr;
    stream = nullptr;
}

int BatchCore::init_device(std::string &err) {
    if (stream) return BD_OK;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) { err = "no HIP device visible"; return BD_ERR_NODEVICE; }
    BD_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    own_stream = true;
    BD_HIP(hipStreamCreateWithFlags(&side, hipStreamNonBlocking));
    BD_HIP(hipStreamCreateWithFlags(&side2, hipStreamNonBlocking));
    BD_HIP(hipEventCreate(&ev0));
    BD_HIP(hipEventCreate(&ev1));
    BD_HIP(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming));
    BD_HIP(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming));
    BD_HIP(hipEventCreateWithFlags(&ev_join2, hipEventDisableTiming));
    hipDeviceProp_t prop;
    BD_HIP(hipGetDeviceProperties(&prop, 0));
    num_cu = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    return scene_kernels_init(err);
}

void BatchCore::invalidate_graph() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    graph_exec = nullptr;
}

// Split active scenes into the size classes, each ordered largest first (the
// work queue hands the longest scenes out first).
void BatchCore::build_order(const std::vector<uint32_t> &active) {
    std::vector<uint32_t> tiny, small, large;
    for (uint32_t i : active) {
        const uint32_t n = descs[i].N;
        (n <= cfg.split_tiny ? tiny : n <= cfg.split_points ? small : large).push_back(i);
    }
    auto by_cost = [&](uint32_t a, uint32_t b) {
        uint64_t ca = (uint64_t)descs[a].N + descs[a].L, cb = (uint64_t)descs[b].N + descs[b].L;
        return ca != cb ? ca > cb : a < b;
    };
    std::sort(tiny.begin(), tiny.end(), by_cost);
    std::sort(small.begin(), small.end(), by_cost);
    std::sort(large.begin(), large.end(), by_cost);
    order.clear();
    order.insert(order.end(), tiny.begin(), tiny.end());
    order.insert(order.end(), small.begin(), small.end());
    order.insert(order.end(), large.begin(), large.end());
    n_tiny = (uint32_t)tiny.size();
    n_small = (uint32_t)small.size();
    n_large = (uint32_t)large.size();
    order_dirty = true;
    invalidate_graph();
    choose_shapes();
}

// The classes' workgroups and LDS.  The configured ones suit a full device: few
// lanes to a small scene, so that many scenes share a CU.  While every scene of
// the launch can have lanes of its own, the launch takes as long as its slowest
// scene, and the classes run on what their largest scene would run on alone:
// about two bodies to a lane, everything in LDS.  The line is where all
// scenes' own workgroups and LDS are resident at once (3 wavefronts to a SIMD
// at the kernels' register counts, 144 KiB of LDS to a CU): 48 flying bodies of
// up to 40 x 40 (12,000 lanes) ran 375 us an update on 64 and 128 lanes and run
// 116 on 256 and 1,024; 640 bodies of up to 128 x 128 (400,000 lanes) stay as
// configured.
void BatchCore::choose_shapes() {
    tiny = Shape{cfg.wg_tiny, cfg.lds_tiny};
    small = Shape{cfg.wg_small, cfg.lds_small};
    large = Shape{cfg.wg_large, cfg.lds_large};
    if (!adapt) return;
    Shape own[3];
    const uint32_t count[3] = {n_tiny, n_small, n_large};
    uint64_t lanes = 0, lds = 0;
    for (size_t k = 0; k < order.size(); k++) {
        const int c = k < n_tiny ? 0 : k < n_tiny + n_small ? 1 : 2;
        uint32_t wg, bytes;
        scene_launch_shape(descs[order[k]], wg, bytes);
        own[c].wg = std::max(own[c].wg, wg);
        own[c].lds = std::max(own[c].lds, bytes);
    }
    for (int c = 0; c < 3; c++) {
        lanes += (uint64_t)count[c] * own[c].wg;
        lds += (uint64_t)count[c] * own[c].lds;
    }
    if (lanes > (uint64_t)num_cu * 768u || lds > (uint64_t)num_cu * scene_max_lds()) return;
    tiny = Shape{std::max(tiny.wg, own[0].wg), std::max(tiny.lds, own[0].lds)};
    small = Shape{std::max(small.wg, own[1].wg), std::max(small.lds, own[1].lds)};
    large = Shape{std::max(large.wg, own[2].wg), std::max(large.lds, own[2].lds)};
}

void BatchCore::order_by(const std::vector<uint64_t> &cost) {
    auto by = [&](uint32_t a, uint32_t b) {
        if (cost[a] != cost[b]) return cost[a] > cost[b];
        uint64_t ca = (uint64_t)descs[a].N + descs[a].L, cb = (uint64_t)descs[b].N + descs[b].L;
        return ca != cb ? ca > cb : a < b;
    };
    auto cls = order.begin();
    for (uint32_t n : {n_tiny, n_small, n_large}) {
        std::sort(cls, cls + n, by);
        cls += n;
    }
    order_dirty = true;
}

int BatchCore::upload_tables(std::string &err) {
    size_t nd = std::max<size_t>(descs.size(), 1);
    if (d_desc_cap < nd) {
        d_desc.release(); d_order.release();
        BD_HIP(d_desc.alloc(nd * sizeof(SceneDesc)));
        BD_HIP(d_order.alloc(nd * sizeof(uint32_t)));
        d_desc_cap = nd;
        invalidate_graph();
    }
    if (!d_queue.p) BD_HIP(d_queue.alloc(64));
    if (descs_dirty && !descs.empty()) {
        BD_HIP(hipMemcpyAsync(d_desc.p, descs.data(), descs.size() * sizeof(SceneDesc), hipMemcpyHostToDevice, stream));
        descs_dirty = false;
    }
    if (order_dirty && !order.empty()) {
        BD_HIP(hipMemcpyAsync(d_order.p, order.data(), order.size() * sizeof(uint32_t), hipMemcpyHostToDevice, stream));
        order_dirty = false;
    }
    // pageable sources: make sure the copies are done before vectors change
    BD_HIP(hipStreamSynchronize(stream));
    return BD_OK;
}

// One launch of every size class: reset the queues (a kernel, never a
// memset node), then the persistent kernels, one per class, on their own
// streams.
int BatchCore::enqueue_launch(uint32_t steps, std::string &err) {
    launch_fill_u32((uint32_t *)d_queue.p, 3, 0u, stream);
    int vs = variant_for_wg((int)small.wg), vl = variant_for_wg((int)large.wg);
    int vt = n_tiny ? variant_for_wg((int)tiny.wg) : 0;
    if (vs < 0 || vl < 0 || vt < 0) { err = "no kernel variant for the configured workgroup size"; return BD_ERR_ARG; }
    const SceneDesc *dd = (const SceneDesc *)d_desc.p;
    const uint32_t *od = (const uint32_t *)d_order.p;
    uint32_t *q = (uint32_t *)d_queue.p;
    BD_HIP(hipEventRecord(ev_fork, stream));
    BD_HIP(hipStreamWaitEvent(side, ev_fork, 0));
    if (n_tiny) BD_HIP(hipStreamWaitEvent(side2, ev_fork, 0));
    auto launch = [&](int v, const Shape &shape, hipStream_t st, uint32_t first, uint32_t n, uint32_t *queue) {
        const uint32_t blocks = std::min<uint32_t>(n, (uint32_t)(num_cu * scene_blocks_per_cu(v, shape.lds)));
        return launch_scene_variant(v, std::max<uint32_t>(blocks, 1), shape.lds, st, dd, states_dev(), od + first, n,
                                    queue, steps, err);
    };
    // the largest first: a large scene takes nearly all of a CU's LDS, and finds no
    // place on one that holds smaller scenes already
    int rc = BD_OK;
    if (n_large) rc = launch(vl, large, side, n_tiny + n_small, n_large, q + 1);
    if (!rc && n_small) rc = launch(vs, small, stream, n_tiny, n_small, q);
    if (!rc && n_tiny) rc = launch(vt, tiny, side2, 0, n_tiny, q + 2);
    if (rc) return rc;
    if (n_tiny) BD_HIP(hipEventRecord(ev_join2, side2));
    BD_HIP(hipEventRecord(ev_join, side));
    BD_HIP(hipStreamWaitEvent(stream, ev_join, 0));
    if (n_tiny) BD_HIP(hipStreamWaitEvent(stream, ev_join2, 0));
    return BD_OK;
}

// Run `launches` launches of `steps` updates each; replays a captured graph
// when configured.
int BatchCore::run(uint32_t launches, uint32_t steps, std::string &err, bool open_timing, bool close_timing) {
    if (!launches) return BD_OK;
    int rc = upload_tables(err);
    if (rc) return rc;
    if (open_timing) {
        BD_HIP(hipEventRecord(ev0, stream));
        last_launches = 0;
    }
    if (cfg.use_graph) {
        if (!graph_exec || graph_steps != steps) {
            invalidate_graph();
            hipGraph_t g;
            BD_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
            rc = enqueue_launch(steps, err);
            hipGraph_t gg = nullptr;
            hipError_t e = hipStreamEndCapture(stream, &gg);
            if (rc) { if (gg) (void)hipGraphDestroy(gg); return rc; }
            if (e != hipSuccess) { err = std::string("graph capture: ") + hipGetErrorString(e); return BD_ERR_DEVICE; }
            g = gg;
            e = hipGraphInstantiate(&graph_exec, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            if (e != hipSuccess) { graph_exec = nullptr; err = std::string("graph instantiate: ") + hipGetErrorString(e); return BD_ERR_DEVICE; }
            graph_steps = steps;
        }
        for (uint32_t l = 0; l < launches; l++) BD_HIP(hipGraphLaunch(graph_exec, stream));
    } else {
        for (uint32_t l = 0; l < launches; l++) {
            rc = enqueue_launch(steps, err);
            if (rc) return rc;
        }
    }
    last_launches += launches * (1 + (n_tiny ? 1 : 0) + (n_small ? 1 : 0) + (n_large ? 1 : 0));
    if (close_timing) {
        BD_HIP(hipEventRecord(ev1, stream));
        timing_pending = true;
    }
    return BD_OK;
}

int BatchCore::finish_timing(std::string &err) {
    if (!timing_pending) return BD_OK;
    BD_HIP(hipEventSynchronize(ev1));
    BD_HIP(hipEventElapsedTime(&last_ms, ev0, ev1));
    timing_pending = false;
    return BD_OK;
}

}  // namespace bd

// ---------------------------------------------------------------------------
// bd_batch
// ---------------------------------------------------------------------------

struct bd_batch {
    BatchCore core;
    std::vector<SceneImage> images;   // host images until the first upload
    std::vector<uint32_t> sub_steps;  // per scene
    std::vector<StepParams> params;   // per scene (dt filled per update)
    std::vector<uint8_t> acc_pending;
    std::vector<uint64_t> chunk_off;  // byte offset of each scene's chunk
    std::vector<uint64_t> updates_run;
    DevBuf<uint8_t> arena;
    DevBuf<SceneState> states;
    PinnedBuf staging;  // bd_batch_read_scene
    uint64_t arena_bytes = 0;
    uint64_t total_points = 0;
    bool uploaded = false;
    float last_dt = NAN;
};

static SceneState *batch_states(bd_batch *b) { return b->states.p; }

static int batch_upload(bd_batch *b, std::string &err) {
    if (b->uploaded) return BD_OK;
    int rc = b->core.init_device(err);
    if (rc) return rc;
    size_t n = b->images.size();
    b->chunk_off.resize(n);
    uint64_t off = 0;
    for (size_t i = 0; i < n; i++) {
        b->chunk_off[i] = off;
        off += (b->images[i].total_bytes + 255) & ~uint64_t(255);
    }
    b->arena_bytes = std::max<uint64_t>(off, 256);
    BD_HIP(b->arena.alloc(b->arena_bytes));
    BD_HIP(b->states.alloc(std::max<size_t>(n, 1)));
    std::vector<SceneState> st(n);
    b->core.descs.resize(n);
    for (size_t i = 0; i < n; i++) {
        const SceneImage &img = b->images[i];
        if (img.init_bytes)
            BD_HIP(hipMemcpyAsync(b->arena.p + b->chunk_off[i], img.bytes.data(), img.init_bytes, hipMemcpyHostToDevice,
                                  b->core.stream));
        SceneDesc d = img.desc;
        d.base = (uint64_t)(uintptr_t)(b->arena.p + b->chunk_off[i]);
        d.steps = 0xffffffffu;
        d.state_slot = (uint32_t)i;
        b->core.descs[i] = d;
        std::memset(&st[i], 0, sizeof(SceneState));
        st[i].skin = img.skin0;
    }
    if (n) BD_HIP(hipMemcpyAsync(b->states.p, st.data(), n * sizeof(SceneState), hipMemcpyHostToDevice, b->core.stream));
    BD_HIP(hipStreamSynchronize(b->core.stream));
    b->core.states_ptr = b->states.p;
    for (auto &img : b->images) { std::vector<uint8_t>().swap(img.bytes); }
    std::vector<uint32_t> all(n);
    std::iota(all.begin(), all.end(), 0u);
    b->core.build_order(all);
    b->core.descs_dirty = true;
    b->uploaded = true;
    return BD_OK;
}

extern "C" {

bd_batch *bd_batch_new(void) {
    try {
        bd_batch *b = new bd_batch();
        b->core.cfg = bd_batch_config{128, 1024, 2048, 32 * 1024, 144 * 1024, 1, 1, 400, 64, 8 * 1024};
        b->core.adapt = true;
        return b;
    } catch (...) {
        set_last_error("allocation failed");
        return nullptr;
    }
}

void bd_batch_free(bd_batch *b) {
    if (!b) return;
    b->core.release();
    delete b;
}

int64_t bd_batch_add_scene(bd_batch *b, const bd_solver *scene) {
    if (!b || !scene) return BD_ERR_ARG;
    if (b->uploaded) return fail(BD_ERR_STATE, "scenes must be added before the first bd_batch_update");
    std::string err;
    HostScene h;
    int rc = solver_export(scene, h, err);
    if (rc) return fail(rc, err);
    Plan p;
    rc = build_plan(h, p, err);
    if (rc) return fail(rc, err);
    if (p.N > 16384) return fail(BD_ERR_CAPACITY, "batch scenes hold at most 16384 bodies");
    SceneImage img;
    rc = build_scene_image(h, p, img, err);
    if (rc) return fail(rc, err);
    b->images.push_back(std::move(img));
    b->params.push_back(make_params(h, 0.0f, false));
    b->acc_pending.push_back(b->images.back().acc_pending ? 1 : 0);
    b->updates_run.push_back(0);
    b->total_points += p.N;
    return (int64_t)b->images.size() - 1;
}

uint64_t bd_batch_len(const bd_batch *b) { return b ? b->images.size() : 0; }
uint64_t bd_batch_total_points(const bd_batch *b) { return b ? b->total_points : 0; }

// Each class's queue hands out the longest scenes first: by bodies plus
// links until every scene has run, then by the device time each scene took
// since the previous ranking (its phase timers), which also counts what that
// estimate misses (circle sweeps, list rebuilds, dependency depth).  Sets
// *contact when the scenes ran more than 64 pair rounds each on average
// since then: their costs then change as they settle, and a long update call
// ranks them again every kRerankLaunches launches.
constexpr uint32_t kRerankLaunches = 4;
static int order_by_measured_time(bd_batch *b, std::string &err, bool *contact) {
    BatchCore &c = b->core;
    const size_t n = b->images.size();
    *contact = false;
    if (!n || c.order.size() != n) return BD_OK;
    std::vector<SceneState> st(n);
    BD_HIP(hipMemcpyAsync(st.data(), b->states.p, n * sizeof(SceneState), hipMemcpyDeviceToHost, c.stream));
    BD_HIP(hipStreamSynchronize(c.stream));
    if (c.order_ticks.size() != n) c.order_ticks.assign(n, 0);
    if (c.order_rounds.size() != n) c.order_rounds.assign(n, 0u);
    std::vector<uint64_t> cost(n);
    uint64_t rounds = 0;
    for (size_t i = 0; i < n; i++) {
        const uint64_t t = st[i].t_links + st[i].t_build + st[i].t_sweep + st[i].t_bodies;
        if (t <= c.order_ticks[i]) return BD_OK;
        cost[i] = t - c.order_ticks[i];
        rounds += st[i].rounds - c.order_rounds[i];
    }
    for (size_t i = 0; i < n; i++) {
        c.order_ticks[i] += cost[i];
        c.order_rounds[i] = st[i].rounds;
    }
    *contact = rounds > 64ull * n;
    c.order_by(cost);
    return BD_OK;
}

int32_t bd_batch_update(bd_batch *b, float dt, uint32_t steps) {
    if (!b) return BD_ERR_ARG;
    std::string err;
    int rc = batch_upload(b, err);
    if (rc) return fail(rc, err);
    if (!steps || b->images.empty()) return BD_OK;
    BatchCore &c = b->core;
    bool contact = false;
    rc = order_by_measured_time(b, err, &contact);
    if (rc) return fail(rc, err);
    // descriptors depend on dt and on the pending initial acc
    bool any_acc = false;
    for (uint8_t a : b->acc_pending) any_acc |= a != 0;
    if (!(dt == b->last_dt) || any_acc) {
        for (size_t i = 0; i < b->images.size(); i++) {
            StepParams sp = b->params[i];
            float mult = 1.0f / (float)sp.sub_steps;  // src/solver.rs:107-108
            sp.delta = dt * mult;
            set_scene_params(c.descs[i], sp, 0xffffffffu, b->acc_pending[i] != 0);
        }
        c.descs_dirty = true;
        b->last_dt = dt;
    }
    uint32_t spl = std::max<uint32_t>(c.cfg.steps_per_launch, 1);
    const uint32_t full = (steps - (any_acc ? 1u : 0u)) / spl, rem = (steps - (any_acc ? 1u : 0u)) % spl;
    if (any_acc) {
        // the first launch consumes the initial acc; the rest use plain descs
        rc = c.run(1, 1, err, true, !full && !rem);
        if (rc) return fail(rc, err);
        for (size_t i = 0; i < b->images.size(); i++) {
            c.descs[i].flags &= ~kFlagAcc;
            b->acc_pending[i] = 0;
        }
        c.descs_dirty = true;
        steps -= 1;
    }
    for (uint32_t done = 0; done < full;) {
        // in contact, a long call ranks the scenes again between chunks
        const uint32_t chunk = contact ? std::min(full - done, kRerankLaunches) : full - done;
        rc = c.run(chunk, spl, err, !any_acc && done == 0, !rem && done + chunk == full);
        if (rc) return fail(rc, err);
        done += chunk;
        if (contact && done < full) {
            rc = order_by_measured_time(b, err, &contact);
            if (rc) return fail(rc, err);
        }
    }
    if (rem) { rc = c.run(1, rem, err, !any_acc && !full, true); if (rc) return fail(rc, err); }
    for (auto &u : b->updates_run) u += steps + (any_acc ? 1 : 0);
    return BD_OK;
}

int32_t bd_batch_sync(bd_batch *b) {
    if (!b) return BD_ERR_ARG;
    if (!b->core.stream) return BD_OK;
    std::string err;
    if (hipStreamSynchronize(b->core.stream) != hipSuccess) return fail(BD_ERR_DEVICE, "hipStreamSynchronize");
    int rc = b->core.finish_timing(err);
    return rc ? fail(rc, err) : BD_OK;
}

int32_t bd_batch_read_scene(bd_batch *b, int64_t id, bd_solver *out) {
    if (!b || !out || id < 0 || (uint64_t)id >= b->images.size()) return BD_ERR_ARG;
    std::string err;
    if (!b->uploaded) {
        int rc = batch_upload(b, err);
        if (rc) return fail(rc, err);
    }
    const SceneDesc &d = b->core.descs[id];
    SceneState st;
    const uint64_t bytes = scene_read_bytes(d, b->images[id].init_bytes);
    // through page-locked memory, without what the device never changes: 640
    // scenes of up to 128 x 128 circles 27 -> 13 ms
    const size_t at = (bytes + 255) & ~(size_t)255;
    if (b->staging.alloc(at + sizeof(st)) != hipSuccess) return fail(BD_ERR_NOMEM, "scene readback buffer");
    if ((bytes && hipMemcpyAsync(b->staging.p, b->arena.p + b->chunk_off[id], bytes, hipMemcpyDeviceToHost,
                                 b->core.stream) != hipSuccess) ||
        hipMemcpyAsync(b->staging.p + at, b->states.p + id, sizeof(st), hipMemcpyDeviceToHost, b->core.stream) !=
            hipSuccess ||
        hipStreamSynchronize(b->core.stream) != hipSuccess)
        return fail(BD_ERR_DEVICE, "scene readback failed");
    std::memcpy(&st, b->staging.p + at, sizeof(st));
    int rc = import_scene_chunk(out, d, b->staging.p, b->updates_run[id], err);
    if (rc) return fail(rc, err);
    if (st.err) return fail(BD_ERR_COLLISION, "circle pair schedule failed for this scene");
    return BD_OK;
}

// Sets the configuration; adapt: whether the classes may take wider shapes than it
// says (see choose_shapes).
static int apply_config(bd_batch *b, const bd_batch_config *cfg, bool adapt) {
    if (variant_for_wg((int)cfg->wg_small) < 0 || variant_for_wg((int)cfg->wg_large) < 0 ||
        (cfg->split_tiny && variant_for_wg((int)cfg->wg_tiny) < 0))
        return fail(BD_ERR_ARG, "workgroup sizes must be 64, 128, 256, 512 or 1024");
    if (cfg->wg_large * 16ull < 16384 && cfg->split_points < 16384) {
        // any size is accepted: larger scenes simply loop over their points
    }
    bool reorder = cfg->split_points != b->core.cfg.split_points || cfg->split_tiny != b->core.cfg.split_tiny;
    b->core.cfg = *cfg;
    if (b->core.cfg.lds_small > scene_max_lds()) b->core.cfg.lds_small = (uint32_t)scene_max_lds();
    if (b->core.cfg.lds_large > scene_max_lds()) b->core.cfg.lds_large = (uint32_t)scene_max_lds();
    if (b->core.cfg.lds_tiny > scene_max_lds()) b->core.cfg.lds_tiny = (uint32_t)scene_max_lds();
    if (b->core.cfg.steps_per_launch < 1) b->core.cfg.steps_per_launch = 1;
    b->core.invalidate_graph();
    b->core.adapt = adapt;
    b->core.choose_shapes();
    if (reorder && b->uploaded) {
        std::vector<uint32_t> all(b->images.size());
        std::iota(all.begin(), all.end(), 0u);
        b->core.build_order(all);
    }
    return BD_OK;
}

int32_t bd_batch_set_config(bd_batch *b, const bd_batch_config *cfg) {
    if (!b || !cfg) return BD_ERR_ARG;
    // the classes run as asked once their shape has been asked for
    auto shapes = [](const bd_batch_config &c) {
        return std::make_tuple(c.wg_small, c.wg_large, c.split_points, c.lds_small, c.lds_large, c.split_tiny,
                               c.wg_tiny, c.lds_tiny);
    };
    return apply_config(b, cfg, b->core.adapt && shapes(*cfg) == shapes(b->core.cfg));
}

int32_t bd_batch_get_shapes(const bd_batch *b, uint32_t *wg, uint32_t *lds) {
    if (!b || !wg || !lds) return BD_ERR_ARG;
    const BatchCore::Shape *const s[3] = {&b->core.tiny, &b->core.small, &b->core.large};
    for (int c = 0; c < 3; c++) { wg[c] = s[c]->wg; lds[c] = s[c]->lds; }
    return BD_OK;
}

int32_t bd_batch_get_config(const bd_batch *b, bd_batch_config *cfg) {
    if (!b || !cfg) return BD_ERR_ARG;
    *cfg = b->core.cfg;
    return BD_OK;
}

int32_t bd_batch_last_timing(const bd_batch *b, float *ms, uint32_t *launches) {
    if (!b) return BD_ERR_ARG;
    std::string err;
    int rc = const_cast<bd_batch *>(b)->core.finish_timing(err);
    if (rc) return fail(rc, err);
    if (ms) *ms = b->core.last_ms;
    if (launches) *launches = b->core.last_launches;
    return BD_OK;
}

int32_t bd_batch_cc_stats(bd_batch *b, uint64_t *rounds, uint64_t *redos, uint64_t *rebuilds, uint64_t *err_scenes) {
    if (!b) return BD_ERR_ARG;
    size_t n = b->images.size();
    std::vector<SceneState> st(n);
    if (b->uploaded && n) {
        if (hipMemcpy(st.data(), b->states.p, n * sizeof(SceneState), hipMemcpyDeviceToHost) != hipSuccess)
            return fail(BD_ERR_DEVICE, "state readback failed");
    }
    uint64_t r = 0, d = 0, u = 0, e = 0;
    for (const SceneState &s : st) { r += s.rounds; d += s.redos; u += s.rebuilds; e += s.err ? 1 : 0; }
    if (rounds) *rounds = r;
    if (redos) *redos = d;
    if (rebuilds) *rebuilds = u;
    if (err_scenes) *err_scenes = e;
    return BD_OK;
}

int32_t bd_batch_cc_fallbacks(bd_batch *b, uint64_t *fallbacks, uint64_t *scenes) {
    if (!b) return BD_ERR_ARG;
    size_t n = b->images.size();
    std::vector<SceneState> st(n);
    if (b->uploaded && n) {
        if (hipMemcpy(st.data(), b->states.p, n * sizeof(SceneState), hipMemcpyDeviceToHost) != hipSuccess)
            return fail(BD_ERR_DEVICE, "state readback failed");
    }
    uint64_t f = 0, k = 0;
    for (const SceneState &x : st) { f += x.fallbacks; k += x.fallbacks ? 1 : 0; }
    if (fallbacks) *fallbacks = f;
    if (scenes) *scenes = k;
    return BD_OK;
}

int32_t bd_batch_scene_status(bd_batch *b, int64_t id, float *skin, uint32_t *err, uint32_t *rounds,
                              uint32_t *redos, uint32_t *rebuilds, uint32_t *pairs) {
    if (!b || id < 0 || (uint64_t)id >= b->images.size()) return BD_ERR_ARG;
    SceneState st{};
    if (b->uploaded) {
        if (hipMemcpy(&st, b->states.p + id, sizeof(st), hipMemcpyDeviceToHost) != hipSuccess)
            return fail(BD_ERR_DEVICE, "state readback failed");
    }
    if (skin) *skin = st.skin;
    if (err) *err = st.err;
    if (rounds) *rounds = st.rounds;
    if (redos) *redos = st.redos;
    if (rebuilds) *rebuilds = st.rebuilds;
    if (pairs) *pairs = st.pairs;
    return BD_OK;
}

// Period of the device wall clock that the kernels' phase timers read.
static double wall_tick_seconds() {
    int dev = 0, khz = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
        khz = 100000;
    return 1.0 / (1000.0 * (double)khz);
}

int32_t bd_batch_scene_times(bd_batch *b, int64_t id, double *links, double *build, double *sweep, double *bodies) {
    if (!b || id < 0 || (uint64_t)id >= b->images.size()) return BD_ERR_ARG;
    SceneState st{};
    if (b->uploaded && hipMemcpy(&st, b->states.p + id, sizeof(st), hipMemcpyDeviceToHost) != hipSuccess)
        return fail(BD_ERR_DEVICE, "state readback failed");
    const double tick = wall_tick_seconds();
    if (links) *links = st.t_links * tick;
    if (build) *build = st.t_build * tick;
    if (sweep) *sweep = st.t_sweep * tick;
    if (bodies) *bodies = st.t_bodies * tick;
    return BD_OK;
}

int32_t bd_batch_scene_lists(bd_batch *b, int64_t id, uint32_t *n_out, uint32_t *n_far, uint32_t *max_list,
                             float *s_cell, float *smax, double *t_count, double *t_lists, double *t_sort,
                             uint32_t *kept, uint32_t *unchecked, uint32_t *fallbacks) {
    if (!b || id < 0 || (uint64_t)id >= b->images.size()) return BD_ERR_ARG;
    SceneState st{};
    if (b->uploaded && hipMemcpy(&st, b->states.p + id, sizeof(st), hipMemcpyDeviceToHost) != hipSuccess)
        return fail(BD_ERR_DEVICE, "state readback failed");
    const double tick = wall_tick_seconds();
    if (n_out) *n_out = st.n_out;
    if (n_far) *n_far = st.n_far;
    if (max_list) *max_list = st.max_list;
    if (s_cell) *s_cell = st.s_cell;
    if (smax) *smax = st.smax;
    if (t_count) *t_count = st.t_count * tick;
    if (t_lists) *t_lists = st.t_lists * tick;
    if (t_sort) *t_sort = st.t_sort * tick;
    if (kept) *kept = st.kept;
    if (unchecked) *unchecked = st.unchecked;
    if (fallbacks) *fallbacks = st.fallbacks;
    return BD_OK;
}

int32_t bd_batch_autotune(bd_batch *b, float dt, uint32_t steps) {
    if (!b) return BD_ERR_ARG;
    std::string err;
    int rc = batch_upload(b, err);
    if (rc) return fail(rc, err);
    if (b->images.empty()) return 0;
    BatchCore &c = b->core;
    // snapshot the whole arena and scene states; restored after tuning
    DevBuf<uint8_t> snap;
    DevBuf<SceneState> snap_st;
    size_t n = b->images.size();
    if (snap.alloc(b->arena_bytes) != hipSuccess || snap_st.alloc(n) != hipSuccess)
        return fail(BD_ERR_NOMEM, "no device memory for the autotune snapshot");
    if (hipMemcpyAsync(snap.p, b->arena.p, b->arena_bytes, hipMemcpyDeviceToDevice, c.stream) != hipSuccess ||
        hipMemcpyAsync(snap_st.p, b->states.p, n * sizeof(SceneState), hipMemcpyDeviceToDevice, c.stream) != hipSuccess)
        return fail(BD_ERR_DEVICE, "snapshot copy failed");
    auto restore = [&]() {
        (void)hipMemcpyAsync(b->arena.p, snap.p, b->arena_bytes, hipMemcpyDeviceToDevice, c.stream);
        (void)hipMemcpyAsync(b->states.p, snap_st.p, n * sizeof(SceneState), hipMemcpyDeviceToDevice, c.stream);
    };
    std::vector<uint8_t> acc_save = b->acc_pending;
    std::vector<uint64_t> upd_save = b->updates_run;
    bd_batch_config best = c.cfg;
    bool best_adapt = c.adapt;
    float best_ms = INFINITY;
    int tried = 0;
    auto trial = [&](const bd_batch_config &cf, bool adapt) -> float {
        if (apply_config(b, &cf, adapt)) return INFINITY;
        restore();
        b->acc_pending = acc_save;
        float total = 0.0f;
        for (int rep = 0; rep < 2; rep++) {
            // the same updates untimed first: the scenes' first candidate lists
            // are built once and would otherwise dominate a short trial (same
            // launch shape, so a captured graph is reused)
            if (bd_batch_update(b, dt, steps) != BD_OK) return INFINITY;
            if (bd_batch_update(b, dt, steps) != BD_OK) return INFINITY;
            float ms = 0.0f;
            if (bd_batch_sync(b) != BD_OK) return INFINITY;
            ms = c.last_ms;
            if (rep == 1) total = ms;  // second run: graph built, caches warm
            restore();
            b->acc_pending = acc_save;
        }
        tried++;
        return total;
    };
    const uint32_t wgs[] = {64, 128, 256, 512, 1024};
    const uint32_t splits[] = {512, 1024, 2048, 4096, 8192};
    // what an untuned batch runs on, where that is wider than its configuration
    if (c.adapt && c.widened()) {
        bd_batch_config cf = best;
        cf.steps_per_launch = 1;
        best_ms = trial(cf, true);
        if (best_ms < INFINITY) best = cf;
    }
    // 1) workgroup sizes and the class split
    for (uint32_t split : splits)
        for (uint32_t ws : wgs)
            for (uint32_t wl : wgs) {
                if (wl < ws || ws > 256 || wl < 256) continue;
                bd_batch_config cf = best;
                cf.split_points = split; cf.wg_small = ws; cf.wg_large = wl;
                cf.steps_per_launch = 1;
                float ms = trial(cf, false);
                // a larger class split has to win by more than 1 %: it puts more
                // mid-size scenes on the small workgroups, which fall behind once
                // the scenes come into dense contact
                const float margin = cf.split_points > best.split_points ? 0.99f : 1.0f;
                if (ms < best_ms * margin) { best_ms = ms; best = cf; best_adapt = false; }
            }
    // the class of the smallest scenes keeps its configured shape (by default
    // 400 bodies, 64 lanes, 8 KiB): two-update trials do not rank it the way
    // long runs do (measured: 8.8 % faster over 100 updates with it)
    // 2) LDS budget (residency) per class
    const uint32_t lds_opts[] = {16 * 1024, 32 * 1024, 64 * 1024, 144 * 1024};
    for (uint32_t ls : lds_opts)
        for (uint32_t ll : lds_opts) {
            if (ll < 64 * 1024) continue;
            bd_batch_config cf = best;
            cf.lds_small = ls; cf.lds_large = ll;
            float ms = trial(cf, false);
            if (ms < best_ms) { best_ms = ms; best = cf; best_adapt = false; }
        }
    // 3) updates per launch
    for (uint32_t spl : {1u, 2u, 4u, 8u}) {
        if (spl > steps) break;
        bd_batch_config cf = best;
        cf.steps_per_launch = spl;
        float ms = trial(cf, best_adapt);
        if (ms < best_ms * 0.98f) { best_ms = ms; best = cf; }
    }
    apply_config(b, &best, best_adapt);
    restore();
    b->acc_pending = acc_save;
    b->updates_run = upd_save;
    (void)hipStreamSynchronize(c.stream);
    b->last_dt = NAN;
    return tried;
}

}  // extern "C"
