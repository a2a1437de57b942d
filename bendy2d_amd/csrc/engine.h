// engine.h -- interface between the C ABI layer and the device engines.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/bendy2d.h"
#include "scene.h"

namespace bd {

// Per-solver counters, mirrored into bd_stats.
struct Stats {
    uint64_t updates = 0, substeps = 0, launches = 0;
    uint64_t cc_rounds = 0, cc_redos = 0, cc_pairs = 0;
    float cc_margin = 0.0f;
    uint32_t tile_passes = 0;
};

// Per-update scalar parameters, computed on the host exactly as the
// reference does (src/solver.rs:107-108, src/particle.rs:52-54).
struct StepParams {
    float delta;            // dt * (1.0f / sub_steps)
    uint32_t sub_steps, link_iters;
    float gx, gy;           // raw gravity
    float gex, gey;         // 0.0f + gravity: the acc every body holds after apply_gravity
    float lox, loy, hix, hiy;  // bounds.pos and bounds.pos + bounds.size
    bool first_acc;         // initial circle / polygon-point acc still pending
};

StepParams make_params(const HostScene &s, float dt, bool acc_pending);

// An engine's state as up to four arrays of 8-byte words in device memory, which
// follow each other in a copy.  With an index, word i of the copy is src[index[i]].
struct StateParts {
    struct Part {
        const void *src;
        const uint32_t *index;
        uint32_t words;
    } part[4] = {};
    int n = 0;
    void add(const void *src, size_t words, const uint32_t *index = nullptr) {
        if (words) part[n++] = Part{src, index, (uint32_t)words};
    }
};

// Queues the copy of the parts into dst, in device or page-locked host memory.
hipError_t gather_state(const StateParts &parts, void *dst, hipStream_t stream);

struct PinnedPool;

class Engine {
public:
    virtual ~Engine() {}
    // Copy the host scene into device buffers following the plan.
    virtual int upload(const HostScene &s, const Plan &p, std::string &err) = 0;
    // Run one update (all substeps).
    virtual int update(const StepParams &sp, Stats &st, std::string &err) = 0;
    // Copy positions back into the host scene (and static polygon centres):
    // the state gathered into page-locked memory, one launch and one wait (a
    // copy per array into pageable memory cost about 12 us each, and a large
    // scene the page faults of a fresh buffer).
    int download(HostScene &s, PinnedPool &pool, std::string &err);
    // What a download reads, as state_count() float2: pos[N], prev[N], then
    // the engine's extra words (polygon centres, the circle-pair state);
    // state_parts describes where it lies (see gather_state), unpack fills the
    // host scene from a host copy of it.
    virtual size_t state_count() const = 0;
    virtual StateParts state_parts() = 0;
    virtual int unpack(const float2 *src, HostScene &s, std::string &err) = 0;
    virtual hipStream_t stream() const = 0;
    virtual int sync(std::string &err) = 0;
    virtual int kind() const = 0;
};

Engine *make_global_engine(hipStream_t stream);
Engine *make_scene_engine(hipStream_t stream);
Engine *make_tiled_engine(hipStream_t stream, uint32_t tile_points, uint32_t wg);

// A download writes the device's bodies into the host scene by index; the
// host scene must still have the shape the engine was uploaded with.
inline bool host_shape_matches(const HostScene &s, uint64_t Np, uint64_t Nc, uint64_t Ng, std::string &err) {
    if (s.p_pos.size() == Np && s.c_pos.size() == Nc && s.g_pos.size() == Ng) return true;
    err = "host scene changed shape since the device copy was made";
    return false;
}

// True when the SCENE engine (one workgroup, LDS-resident) can run this plan.
bool scene_engine_fits(const HostScene &s, const Plan &p);
bool tiled_engine_fits(const HostScene &s, const Plan &p);

// Thread-local detailed error message used by bd_last_error().
void set_last_error(const std::string &msg);

}  // namespace bd
struct bd_solver;
namespace bd {
int solver_export(const bd_solver *s, HostScene &out, std::string &err);
int solver_import_state(bd_solver *s, const HostScene &src, uint64_t updates, std::string &err);
// The same from pos[N] and prev[N] (particles, then circles) of a scene without
// polygons, in one pass over them.
int solver_import_bodies(bd_solver *s, uint64_t np, uint64_t nc, const void *pos, const void *prev, uint64_t updates,
                         std::string &err);
const HostScene &solver_host(const bd_solver *s);

#define BD_HIP(call)                                                                   \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess) {                                                        \
            err = std::string(#call) + ": " + hipGetErrorString(e_);                   \
            return BD_ERR_DEVICE;                                                      \
        }                                                                              \
    } while (0)

// Page-locked host memory for copies from the device, grown to the largest asked.
struct PinnedBuf {
    uint8_t *p = nullptr;
    size_t n = 0;
    PinnedBuf() {}
    PinnedBuf(const PinnedBuf &) = delete;
    PinnedBuf &operator=(const PinnedBuf &) = delete;
    PinnedBuf(PinnedBuf &&o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    PinnedBuf &operator=(PinnedBuf &&o) noexcept {
        std::swap(p, o.p);
        std::swap(n, o.n);
        return *this;
    }
    ~PinnedBuf() {
        if (p) (void)hipHostFree(p);
    }
    hipError_t alloc(size_t bytes) {
        if (bytes <= n) return hipSuccess;
        if (p) (void)hipHostFree(p);
        p = nullptr; n = 0;
        hipError_t e = hipHostMalloc((void **)&p, bytes, hipHostMallocPortable);
        if (e == hipSuccess) n = bytes; else p = nullptr;
        return e;
    }
};

// Page-locked buffers that downloads borrow: allocating one takes longer than the
// download of a small scene.  At most kKept buffers of together kKeptBytes wait
// here for the next download; all solvers of the process share them, and they are
// freed with the last solver.  A state of more than kKeptBytes gets none: page-locking
// a buffer that is not kept takes longer than a copy into pageable memory (6 and 12
// million bodies: 40 and 78 ms a download, 27 and 54 pageable).  The first download
// pays for its buffer (a million bodies 6.8 ms, then 0.9; pageable 1.7 each time).
struct PinnedPool {
    static constexpr int kKept = 4;
    static constexpr size_t kKeptBytes = 64u << 20, kLeast = 64u << 10;
    // a buffer of at least `bytes` (p null when there is no memory, or not so much is kept)
    PinnedBuf take(size_t bytes);
    void give(PinnedBuf &&b);
    static std::shared_ptr<PinnedPool> shared();

private:
    std::mutex m_;
    PinnedBuf kept_[kKept];
};

// Device buffer with RAII release.
template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    DevBuf() {}
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf(DevBuf &&o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    DevBuf &operator=(DevBuf &&o) noexcept {
        if (this != &o) { release(); p = o.p; n = o.n; o.p = nullptr; o.n = 0; }
        return *this;
    }
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr; n = 0;
    }
    hipError_t alloc(size_t count) {
        if (count <= n && p) return hipSuccess;
        release();
        if (count == 0) return hipSuccess;
        hipError_t e = hipMalloc((void **)&p, count * sizeof(T));
        if (e == hipSuccess) n = count; else p = nullptr;
        return e;
    }
};

}  // namespace bd
