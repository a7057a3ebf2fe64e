#include "fake_hip.hpp"

#include <algorithm>
#include <functional>
#include <iterator>
#include <map>
#include <mutex>
#include <set>
#include <vector>

#include "mcdp_grad.hpp"
#include "mcdp_internal.hpp"
#include "mcdp_kernels.hpp"
#include "mcdp_stats.hpp"

using Work = std::function<void()>;
struct ihipStream_t {
    bool capturing = false, broken = false;
    hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
    ihipStream_t *origin = nullptr;  // captured through an event of this stream
    std::vector<Work> work;
};
struct ihipEvent_t {
    ihipStream_t *stream = nullptr;
};
struct ihipGraph {
    std::vector<Work> work;
};
struct hipGraphExec {
    std::vector<Work> work;
};

namespace fake {
size_t memory = (size_t)64 << 30, used = 0;
int dead_accesses = 0, launches = 0, graph_launches = 0, allocations = 0;
}  // namespace fake

namespace {
std::recursive_mutex mu;
std::map<uintptr_t, size_t> ranges;
uintptr_t next_address = (uintptr_t)1 << 44;
std::set<ihipStream_t *> capturing;
thread_local hipStreamCaptureMode thread_mode = hipStreamCaptureModeGlobal;

// Whether a call that a capture forbids is refused; the captures end in error.
bool refused() {
    std::lock_guard<std::recursive_mutex> lock(mu);
    if (thread_mode == hipStreamCaptureModeRelaxed) return false;
    bool any = false;
    for (ihipStream_t *s : capturing)
        if (s->mode != hipStreamCaptureModeRelaxed) any = s->broken = true;
    return any;
}

void touch(const void *p) {
    if (!p) return;
    std::lock_guard<std::recursive_mutex> lock(mu);
    const auto a = (uintptr_t)p;
    auto it = ranges.upper_bound(a);
    const bool live = it != ranges.begin() && a < std::prev(it)->first + std::prev(it)->second;
    if (!live) ++fake::dead_accesses;
}

hipError_t enqueue(hipStream_t s, Work w) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    if (s && s->capturing) {
        (s->origin ? s->origin : s)->work.push_back(std::move(w));
        return hipSuccess;
    }
    w();
    return hipSuccess;
}

hipError_t kernel(hipStream_t s, std::vector<const void *> arrays) {
    return enqueue(s, [arrays] {
        ++fake::launches;
        for (const void *p : arrays) touch(p);
    });
}

bool on_device(const void *p) { return (uintptr_t)p >= (uintptr_t)1 << 44 && (uintptr_t)p < next_address; }
}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "fake error"; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) { return *p = hipDeviceProp_tR0600{}, hipSuccess; }
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    *total = fake::memory;
    *free_bytes = fake::memory - fake::used;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    *p = nullptr;
    if (refused()) return hipErrorStreamCaptureUnsupported;
    if (fake::used + n > fake::memory) return hipErrorOutOfMemory;
    fake::used += n;
    ++fake::allocations;
    ranges[next_address] = n;
    *p = (void *)next_address;
    next_address += (n + 4095) / 4096 * 4096 + 4096;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    std::lock_guard<std::recursive_mutex> lock(mu);
    if (refused()) return hipErrorStreamCaptureUnsupported;
    auto it = ranges.find((uintptr_t)p);
    if (it == ranges.end()) return ++fake::dead_accesses, hipErrorInvalidValue;
    fake::used -= it->second;
    ranges.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (refused()) return hipErrorStreamCaptureUnsupported;
    return *p = malloc(n), *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipDeviceSynchronize() { return refused() ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t, hipMemcpyKind, hipStream_t s) {
    return enqueue(s, [dst, src] {
        if (on_device(dst)) touch(dst);
        if (on_device(src)) touch(src);
    });
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind kind) {
    return refused() ? hipErrorStreamCaptureUnsupported : hipMemcpyAsync(dst, src, n, kind, nullptr);
}
hipError_t hipMemcpy2DAsync(void *dst, size_t, const void *src, size_t, size_t w, size_t, hipMemcpyKind kind,
                            hipStream_t s) {
    return hipMemcpyAsync(dst, src, w, kind, s);
}
hipError_t hipMemcpy2D(void *dst, size_t, const void *src, size_t, size_t w, size_t, hipMemcpyKind kind) {
    return hipMemcpy(dst, src, w, kind);
}
hipError_t hipMemset(void *dst, int, size_t) {
    if (refused()) return hipErrorStreamCaptureUnsupported;
    touch(dst);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = new ihipStream_t, hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamDestroy(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    capturing.erase(s);
    delete s;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (s && s->capturing) return s->broken = true, hipErrorStreamCaptureUnsupported;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = new ihipEvent_t, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return e->stream = s, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return refused() ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    ihipStream_t *from = e->stream;
    if (from && from->capturing && !s->capturing) {  // the event's capture takes in this stream
        s->capturing = true;
        s->origin = from->origin ? from->origin : from;
    }
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *mode) {
    std::swap(*mode, thread_mode);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    *st = !s || !s->capturing ? hipStreamCaptureStatusNone
          : s->broken         ? hipStreamCaptureStatusInvalidated
                              : hipStreamCaptureStatusActive;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode mode) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    s->capturing = true;
    s->broken = false;
    s->mode = mode;
    s->work.clear();
    capturing.insert(s);
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    capturing.erase(s);
    s->capturing = false;
    *g = nullptr;
    if (s->broken) return hipErrorStreamCaptureInvalidated;
    *g = new ihipGraph{s->work};
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    return *e = new hipGraphExec{g->work}, hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete g, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return delete e, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    ++fake::graph_launches;
    for (const Work &w : e->work) w();
    return hipSuccess;
}
}  // extern "C"

// ---- the kernels' launchers --------------------------------------------------

namespace mcdp {
static std::vector<const void *> arrays(const WalkParams &p) {
    return {p.recs, p.seeds, p.dur_in, p.realized, p.durations, p.cause, p.cause_pos};
}
hipError_t launch_walk(const WalkParams &p, WalkVariant, int, size_t, hipStream_t s) { return kernel(s, arrays(p)); }
// As the kernels' registers allow: six waves a SIMD of one sample per lane, four of two.
hipError_t walk_occupancy(WalkVariant v, int waves, size_t lds, int *blocks) {
    *blocks = std::min((v.spl == 1 ? 6 : 4) / ((waves + 3) / 4), (int)((size_t)160 * 1024 / std::max<size_t>(lds, 1)));
    return hipSuccess;
}
hipError_t launch_walk_wide(const WalkParams &p, bool, int32_t, int32_t, int32_t, hipStream_t s) {
    return kernel(s, arrays(p));
}
hipError_t launch_walk_wide_orphans(const WalkParams &p, int32_t, hipStream_t s) { return kernel(s, arrays(p)); }
hipError_t launch_draws(const DrawParams &p, int, hipStream_t s) { return kernel(s, {p.recs, p.seeds, p.durations}); }
hipError_t launch_levels(const LevelParams &p, bool, int, int, int, hipStream_t s) {
    return kernel(s, {p.quad, p.dur, p.realized, p.cause, p.cause_pos});
}
hipError_t launch_copy(double *d, const double *x, int64_t, hipStream_t s) { return kernel(s, {d, x}); }
hipError_t launch_math_debug(int, int64_t, const double *, double *, hipStream_t) { return hipSuccess; }
hipError_t launch_philox_debug(int, int64_t, const uint32_t *, const uint32_t *, uint32_t *, hipStream_t) {
    return hipSuccess;
}
hipError_t launch_event_quantiles(const double *x, int32_t, int32_t, int32_t, const QuantileArgs &, double *out,
                                  double *mean, hipStream_t s) {
    return kernel(s, {x, out, mean});
}
hipError_t launch_event_mean(const double *x, int32_t, int32_t, int32_t, double *mean, hipStream_t s) {
    return kernel(s, {x, mean});
}
hipError_t launch_cause_counts(const int32_t *c, int32_t, int32_t, int32_t, const int32_t *off, const int32_t *,
                               const int32_t *, const int32_t *, int64_t *counts, int32_t, hipStream_t s) {
    return kernel(s, {c, off, counts});
}
hipError_t launch_cause_pos_counts(const uint8_t *c, int32_t, int32_t, int32_t, const int32_t *off, const int32_t *,
                                   int64_t *counts, int32_t, hipStream_t s) {
    return kernel(s, {c, off, counts});
}
}  // namespace mcdp
