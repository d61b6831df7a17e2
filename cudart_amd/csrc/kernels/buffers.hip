// Memory that calls share or leave for the next one, and copies to the caller's buffers.
//
// Idle memory is bounded (two staging blocks, and per device one set of queues of at most a
// sixteenth of its memory and a quarter of what is free beside it, and as much in blocks of
// scratch memory), is taken by one call at a time, and is given back when no scene is on a
// device any more or when an allocation of the library finds no room.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <utility>

#include "renderer.hpp"

namespace prt {

namespace {

// A pinned staging block: the device fills one segment while the host empties another.
// Copies to pageable memory went through HIP's own staging one megabyte at a time, the
// device waiting for the host and the host for the device, and the memory is mostly fresh, a
// page fault every 4 KB. Mean radiance to a new array, 640 x 480 (3.7 MB): 0.33 -> 0.22 ms,
// 1271 x 713: 0.83 -> 0.58, 3840 x 2160: 10.9 -> 7.5. (Emptying segments with 4 threads took
// 0.18, 0.46 and 6.2, but first hits at 1271 x 713, 0.87 ms, then took 0.74 to 1.2: the page
// faults of one process take turns.)
constexpr size_t kSegment = size_t(1) << 20;
constexpr int kSegments = 4;
constexpr int kMaxIdleStages = 2;

struct Stage {
    int device = -1;
    char* mem = nullptr;
    hipEvent_t done[kSegments] = {};
};

// Scratch blocks are few: a call takes one, so several are only left by several threads.
constexpr int kMaxIdleScratch = 4;
constexpr size_t kSmallScratch = size_t(64) << 20;  // kept without asking for the device's memory

std::mutex g_mutex;
Stage g_idle[kMaxIdleStages];  // device < 0: none
Scratch g_idle_scratch[kMaxIdleScratch];  // mem == nullptr: none
prt_renderer* g_keepers = nullptr;        // renderers that keep vertices
std::atomic<int> g_scenes{0};

void free_stage(Stage& s) {
    for (hipEvent_t e : s.done)
        if (e) (void)hipEventDestroy(e);
    if (s.mem) (void)hipHostFree(s.mem);
    s = Stage();
}

bool take_stage(int device, Stage& s) {
    {
        std::lock_guard<std::mutex> g(g_mutex);
        for (Stage& o : g_idle)
            if (o.device == device) {
                s = o;
                o = Stage();
                return true;
            }
    }
    s.device = device;
    bool ok = hipHostMalloc(reinterpret_cast<void**>(&s.mem), kSegment * kSegments, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t& e : s.done) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        free_stage(s);
    }
    return ok;
}

void give_stage(Stage& s) {
    {
        std::lock_guard<std::mutex> g(g_mutex);
        for (Stage& o : g_idle)
            if (g_scenes.load() > 0 && o.device < 0) {
                o = s;
                return;
            }
    }
    free_stage(s);
}

void release_idle() {
    Stage all[kMaxIdleStages];
    Scratch scratch[kMaxIdleScratch];
    {
        std::lock_guard<std::mutex> g(g_mutex);
        for (int k = 0; k < kMaxIdleStages; ++k) std::swap(all[k], g_idle[k]);
        for (int k = 0; k < kMaxIdleScratch; ++k) std::swap(scratch[k], g_idle_scratch[k]);
    }
    for (Stage& s : all) free_stage(s);
    for (Scratch& s : scratch)
        if (s.mem) (void)hipFree(s.mem);
    release_idle_queues();
}

// The vertices of `device`'s renderers that no call is using.
void release_vertices(int device) {
    std::lock_guard<std::mutex> g(g_mutex);
    for (prt_renderer* r = g_keepers; r; r = r->next_keeper) {
        if (!r->vertices || r->vertex_users != 0 || r->cfg.device != device) continue;
        (void)hipFree(r->vertices);
        r->vertices = nullptr;
    }
}

}  // namespace

void offer_vertices(prt_renderer* r) {
    std::lock_guard<std::mutex> g(g_mutex);
    r->next_keeper = g_keepers;
    g_keepers = r;
}
void withdraw_vertices(prt_renderer* r) {
    std::lock_guard<std::mutex> g(g_mutex);
    for (prt_renderer** p = &g_keepers; *p; p = &(*p)->next_keeper)
        if (*p == r) {
            *p = r->next_keeper;
            return;
        }
}
VertexUse::VertexUse(prt_renderer* r) : r_(r) {
    std::lock_guard<std::mutex> g(g_mutex);
    ++r->vertex_users;
}
VertexUse::~VertexUse() {
    std::lock_guard<std::mutex> g(g_mutex);
    --r_->vertex_users;
}

void scene_uploaded() { ++g_scenes; }
void scene_released() {
    if (--g_scenes == 0) release_idle();
}
bool scenes_on_devices() { return g_scenes.load() > 0; }

hipError_t device_alloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        release_idle();
        e = hipMalloc(p, bytes);
    }
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        int device = -1;
        (void)hipGetDevice(&device);
        release_vertices(device);
        e = hipMalloc(p, bytes);
    }
    return e;
}

Scratch take_scratch(int device, size_t bytes) {
    std::lock_guard<std::mutex> g(g_mutex);
    Scratch* best = nullptr;  // the smallest that is large enough, else the largest
    for (Scratch& o : g_idle_scratch) {
        if (!o.mem || o.device != device) continue;
        if (!best || (best->bytes < bytes ? o.bytes > best->bytes : o.bytes >= bytes && o.bytes < best->bytes)) best = &o;
    }
    Scratch s;
    if (best) std::swap(s, *best);
    s.device = device;
    return s;
}

void give_scratch(Scratch& s) {
    if (!s.mem) return;
    size_t free_b = 0, total_b = 0;
    if (s.bytes > kSmallScratch && hipMemGetInfo(&free_b, &total_b) != hipSuccess) free_b = total_b = 0;
    {
        std::lock_guard<std::mutex> g(g_mutex);
        Scratch* slot = nullptr;
        size_t idle = s.bytes;
        for (Scratch& o : g_idle_scratch) {
            if (!o.mem) slot = &o;
            else if (o.device == s.device) idle += o.bytes;
        }
        if (slot && g_scenes.load() > 0 && (s.bytes <= kSmallScratch || may_stay_idle(idle, free_b, total_b))) {
            *slot = s;
            s = Scratch();
            return;
        }
    }
    (void)hipFree(s.mem);
    s = Scratch();
}

hipError_t copy_out(const CopyOut* c, size_t n, int device, hipStream_t stream) {
    size_t bytes = 0;
    for (size_t k = 0; k < n; ++k) bytes += c[k].bytes;
    Stage st;
    // Below 1 MB the fixed costs of segments and events are more than they save (786 KB of mean
    // radiance: 72 us staged, 62 plain; 1.2 MB of 8-bit image: 90 and 112).
    if (bytes < kSegment || !take_stage(device, st)) {
        for (size_t k = 0; k < n; ++k) {
            const hipError_t e = hipMemcpyAsync(c[k].dst, c[k].src, c[k].bytes, hipMemcpyDeviceToHost, stream);
            if (e != hipSuccess) return e;
        }
        return hipStreamSynchronize(stream);
    }
    // Small results in two segments, so that emptying the first overlaps sending the second.
    const size_t segment = std::min(kSegment, (bytes / 2 + 4095) / 4096 * 4096);
    // A segment is one device copy: a run of source bytes, over as many destinations as
    // follow one another in the source.
    struct Part {
        size_t k, at, bytes;  // starts at byte `at` of c[k]
    };
    Part part[kSegments] = {};
    size_t k = 0, at = 0;             // the next byte to send
    uint32_t sent = 0, received = 0;  // segments
    auto src_of = [&](size_t i) { return static_cast<const char*>(c[i].src); };
    hipError_t e = hipSuccess;
    while (e == hipSuccess) {
        while (k < n && at == c[k].bytes) {
            ++k;
            at = 0;
        }
        if (k < n && sent - received < uint32_t(kSegments)) {
            const int s = int(sent++ % kSegments);
            const char* from = src_of(k) + at;
            Part& p = part[s] = Part{k, at, 0};
            while (k < n && p.bytes < segment && src_of(k) + at == from + p.bytes) {
                const size_t len = std::min(segment - p.bytes, c[k].bytes - at);
                p.bytes += len;
                at += len;
                if (at < c[k].bytes) break;
                ++k;
                at = 0;
            }
            e = hipMemcpyAsync(st.mem + size_t(s) * kSegment, from, p.bytes, hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(st.done[s], stream);
        } else if (received < sent) {
            const int s = int(received++ % kSegments);
            e = hipEventSynchronize(st.done[s]);
            Part p = part[s];
            for (const char* from = st.mem + size_t(s) * kSegment; e == hipSuccess && p.bytes > 0; ++p.k, p.at = 0) {
                const size_t len = std::min(p.bytes, c[p.k].bytes - p.at);
                std::memcpy(static_cast<char*>(c[p.k].dst) + p.at, from, len);
                from += len;
                p.bytes -= len;
            }
        } else {
            break;
        }
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // no copy into the block is left in flight
    give_stage(st);
    return e;
}

}  // namespace prt
