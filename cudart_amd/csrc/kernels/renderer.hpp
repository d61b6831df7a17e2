// prt_renderer: one image on one device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../host/scene.hpp"
#include "kernel_api.hpp"

namespace prt {
struct WavefrontState;
}

struct prt_renderer {
    prt_scene* scene = nullptr;
    prt_camera cam{};
    uint32_t w = 0, h = 0, spp = 0;
    prt_render_config cfg{};
    prt::SceneArgs sc{};
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float4* accum = nullptr;               // w*h running sums
    unsigned long long* counters = nullptr;
    uint32_t* tickets = nullptr;   // kTicketSets x kTicketWords, behind the counters
    uint32_t ticket_sets_used = 0;
    uint8_t* gamma_lut = nullptr;
    int* spill = nullptr;
    uint64_t spill_columns = 0;  // one per thread of a launch (ensure_spill)
    uint32_t tiles_x = 0, tiles = 0;  // 8x8 pixel tiles
    uint32_t compute_units = 0;
    uint32_t samples_done = 0;
    uint64_t samples_total = 0;
    double last_ms = 0.0;
    double kernel_ms[3] = {0, 0, 0};  // profile_kernels: extend, shade, shadow of the last wavefront render
    uint32_t kernel_launches[3] = {0, 0, 0};
    prt::WavefrontState* wf = nullptr;
    // keep_samples: radiance of pixel-sample (p, s) at samples[p * spp + s], s < spp, and
    // (where it fits) its path's vertex at bounce b at
    // vertices[(b * w * h + p) * spp + s]. Valid for the adjoint while every sample since the last reset was rendered with
    // the scene's current materials (samples_version).
    float4* samples = nullptr;
    uint32_t* vertices = nullptr;
    uint32_t vertex_users = 0;              // VertexUse
    prt_renderer* next_keeper = nullptr;    // of the renderers that keep vertices
    bool samples_ok = false;
    // Device memory of the calls that hand results out, kept until the renderer goes: at most
    // 12 bytes per pixel (scratch_for).
    void* out = nullptr;
    size_t out_bytes = 0;
    uint64_t samples_version = 0;
};

namespace prt {
int hip_fail(hipError_t e, const char* what);
// Copies and fills ordered on the caller's stream and waited for. The library never
// uses the legacy (null) stream: HIP fails a legacy-stream operation issued while
// another thread captures a stream into a graph, and ends that capture, so renderers
// driven from several host threads at once would break each other's launches.
inline hipError_t copy_wait(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}
inline hipError_t fill_wait(void* dst, int value, size_t bytes, hipStream_t s) {
    hipError_t e = hipMemsetAsync(dst, value, bytes, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}
// buffers.hip.
// hipMalloc; if there is no room, after idle memory has been given back, and then the vertices kept
// by renderers that no call is using.
hipError_t device_alloc(void** p, size_t bytes);
// Kept vertices save an adjoint its forward pass, and it can do without: a renderer that has them
// offers them (until it withdraws), and a call that reads or writes r->vertices holds a VertexUse
// meanwhile. Every such call waits for its launches.
void offer_vertices(prt_renderer* r);
void withdraw_vertices(prt_renderer* r);
class VertexUse {
public:
    explicit VertexUse(prt_renderer* r);
    ~VertexUse();
    VertexUse(const VertexUse&) = delete;
    VertexUse& operator=(const VertexUse&) = delete;

private:
    prt_renderer* r_;
};
// Device memory to the caller's host buffers, ordered on `stream` and waited for.
struct CopyOut {
    void* dst;
    const void* src;
    size_t bytes;
};
hipError_t copy_out(const CopyOut* c, size_t n, int device, hipStream_t stream);
// Device memory of one call (scratch_for makes it large enough). take_scratch gives an idle block of
// the device, if possible of at least `bytes`, or an empty one; give_scratch takes it back, once no
// launch uses it any more, and keeps or frees it.
struct Scratch {
    int device = -1;
    void* mem = nullptr;
    size_t bytes = 0;
};
Scratch take_scratch(int device, size_t bytes);
void give_scratch(Scratch& s);
// While a scene is on a device, idle memory is kept for the next call.
void scene_uploaded();
void scene_released();
bool scenes_on_devices();
void release_idle_queues();  // wavefront.hip
// At least `bytes` of scratch memory p (of `have` bytes), grown as needed; its contents are lost.
int scratch_for(void*& p, size_t& have, size_t bytes);
// Uploads the scene to `device` on first use (copies ordered on `stream`).
int device_scene(prt_scene* s, int device, SceneArgs& out, hipStream_t stream);
CamArgs cam_args(const prt_camera& c);
int set_device(int device);
// Entries the deepest walk of the scene's BVH can hold: a node visit pushes at most its
// three farther children, once per level 0..max_depth. (At most kStackMax.) What does not
// fit a kernel's LDS stack goes to a spill area of that many rows, a column per thread; with
// kStackMax rows it took 235 MB for the wavefront's resident threads, 0.8 GB for a 1080p
// megakernel.
inline uint32_t stack_entries(const prt_scene* s) { return 3 * (s->bvh.max_depth + 1); }
// At least `columns` columns of the renderer's spill area, where its scene needs one. Every launch
// that uses the area calls this first, with its own threads.
int ensure_spill(prt_renderer* r, uint64_t columns);
int render_wavefront(prt_renderer* r, uint32_t n);  // wavefront.hip
// Samples 0..spp-1 of the renderer's view into `accum` (zeroed), each sample's radiance
// into `samples` ([pixel * spp + sample]) and, unless null, its path's vertices into
// `vertices` ([(bounce * pixels + pixel) * spp + sample]), without touching the renderer's
// own accumulation or counters.
int wavefront_samples(prt_renderer* r, uint32_t spp, float4* accum, float4* samples,
                      uint32_t* vertices);  // wavefront.hip
MegaArgs megakernel_args(prt_renderer* r, float4* accum, float4* samples, uint32_t* vertices, uint32_t cap);  // device.hip
int megakernel_samples(prt_renderer* r, MegaArgs& a, uint32_t first, uint32_t n, uint32_t spp_per_launch, bool count);
// Whether path vertices of spp samples of this view can be kept (index and depth limits).
inline bool vertices_fit(uint32_t w, uint32_t h, uint32_t spp, uint32_t max_depth) {
    return max_depth <= 16 && uint64_t(w) * h <= (1u << 24) && uint64_t(w) * h * spp < (uint64_t(1) << 32);
}
void release_wavefront(prt_renderer* r);            // wavefront.hip
}  // namespace prt
