// Internal state behind an xt_dev handle.
#pragma once
#include <hip/hip_runtime.h>

#include <deque>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "device/xt_kernels.h"

#define XT_TRACE_STAMPS 256

struct DevScene {
    SceneView view;
    std::vector<void *> allocs;
    uint64_t bytes = 0;
    uint64_t kd_bytes = 0;            // of the kd nodes, references and leaf copies (in `allocs`)
    uint32_t n_kd_nodes = 0, n_kd_refs = 0;
    uint32_t bvh_depth = 0;           // levels of the wide BVH (view.bvh), 0 without one
    xt_kd_build_stats kd_stats{};     // of the last device build (zero for a host-built tree)
    bool pt_supported = true;
    bool materials_supported = true;
    bool missing_material = false;
};

struct WaveQueue {
    float4 *r0 = nullptr, *r1 = nullptr;
    uint32_t *path = nullptr;
};

#define XT_MAX_LANES 16
#define XT_LANE_STREAMS 4  // streams the groups of a served pass spread over

struct WaveBuffers {
    size_t cap = 0;
    WaveQueue q[2];
    float4 *hit = nullptr;
    uint32_t *retest = nullptr;
    uint4 *recheck = nullptr;
    float4 *ps0 = nullptr, *ps1 = nullptr, *rad = nullptr;
    uint32_t *flags = nullptr;
    Counters *cnt = nullptr;  // XT_MAX_LANES counter blocks
    double *ray64 = nullptr;
    float4 *chan = nullptr;  // 3 per slot: sampled material colours (k_channels)
    std::vector<void *> allocs;
    uint64_t bytes = 0;
};

struct AccumBuffers {
    size_t npix = 0;
    float4 *accf = nullptr;
    double2 *acc64 = nullptr;
    float4 *out = nullptr;
    std::vector<void *> allocs;
    uint64_t bytes = 0;
};

// What kernels report to the host without a copy: fine-grained pinned memory.
struct HostReports {
    uint64_t stamp[2 * XT_TRACE_STAMPS];  // wall clock at a timed trace launch's start and end
    uint32_t count[XT_MAX_LANES];         // queue counts of the early-stop check
    JobTotals totals[XT_MAX_LANES];
};

struct ServeState;  // continuous-batching server (xt_serve.hip)

struct xt_dev {
    int device = 0;
    int n_cu = 256;
    hipStream_t stream = nullptr;
    hipStream_t lane_stream[XT_LANE_STREAMS] = {};  // default priority, like `stream`
    hipEvent_t lane_ev[XT_LANE_STREAMS] = {}, fork_ev = nullptr;
    uint64_t budget = 0, used = 0;
    std::map<uint32_t, DevScene> scenes;
    uint32_t next_scene = 1;
    WaveBuffers wave;
    AccumBuffers accum;
    Counters *host_counters = nullptr;  // pinned, XT_MAX_LANES blocks
    HostReports *reports = nullptr;     // pinned, written by kernels (xt_ensure_reports)
    double clock_khz = 100000.0;        // of the stamps
    uint64_t *host_words = nullptr;     // pinned, 8 KiB: read-backs of an index build
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int trace_launches = 0;  // trace launches with a stamp in this call
    ServeState *serve = nullptr;
    xt_tuning tuning{12, 256, 64u << 20, 0, 1, 1, 1, 1, 2};
    void *scratch = nullptr;  // this device's address of xt_trace_device_static's scratch array
    std::string err;
};

// Blocks for a grid-stride launch over n items, at least 1, at most cap.
static inline unsigned grid_for(size_t n, unsigned block, unsigned cap) {
    size_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned)g;
}

int xt_dev_ensure_wave(xt_dev *d, size_t cap, bool need64, bool need_chan = false);
int xt_dev_ensure_accum(xt_dev *d, size_t npix);
void xt_dev_free_wave(xt_dev *d);
void xt_dev_free_accum(xt_dev *d);
// A sub-queue of the wavefront buffers: slots [off, off + cap) of the ray
// queues, the hit and the re-test arrays, counted by its own counter block.
// A one-job render uses one lane over the whole buffers; the server gives
// each (scene, integrator, accel) group of a pass a lane of its own.
struct WaveLane {
    size_t off = 0, cap = 0;
    Counters *cnt = nullptr;
};
int xt_launch_trace(xt_dev *d, const DevScene &ds, int accel, int qi, const WaveLane &lane, const double *ray64,
                    uint32_t *flags, bool time_it, hipStream_t st, uint32_t *post = nullptr);
int xt_ensure_reports(xt_dev *d);
// Milliseconds between two stamps.
inline double xt_stamp_ms(const xt_dev *d, uint64_t a, uint64_t b) {
    return b > a ? (double)(b - a) / d->clock_khz : 0.0;
}
// The buffers one trace launch reads and writes.
struct TraceBufs {
    Queue q;
    const uint32_t *count = nullptr;  // rays in q
    float4 *hit = nullptr;
    uint32_t *retest = nullptr;
    uint4 *recheck = nullptr;
    Counters *cnt = nullptr;
    size_t cap = 0;  // queue capacity (sizes the grids)
    uint32_t par = 0;          // parity of the round (Counters)
    uint32_t *post = nullptr;  // pinned: where the trace posts its ray count
};
int xt_launch_trace_bufs(xt_dev *d, const DevScene &ds, int accel, const TraceBufs &B, const double *ray64,
                         uint32_t *flags, bool time_it, hipStream_t st);
class XtScratch;

// Builds the kd-tree of a resident scene on the device (xt_kdbuild.hip) and
// replaces the scene's kd arrays with it, with `leaf_copies` the copies of the
// leaves' primitives among them. When that fails, the scene keeps its old ones.
int xt_kd_build_into(xt_dev *d, DevScene &ds, const xt_build_params *p, bool leaf_copies, XtScratch &mem);
// Builds the scene's wide BVH, unless its FP32 walk stays on the kd-tree
// (view.bvh is null then). xt_bvhbuild.hip
int xt_bvh_build_into(xt_dev *d, DevScene &ds, XtScratch &mem);
// Copies the kd leaves' primitives into leaf order for a scene that is walked
// on its kd-tree (xt_kdbuild.hip).
int xt_kd_leaf_copies(xt_dev *d, DevScene &ds);
void xt_serve_shutdown(xt_dev *d);
bool xt_serve_uses_scene(const xt_dev *d, uint32_t scene_id);
void xt_serve_forget_scene(xt_dev *d, uint32_t scene_id);
