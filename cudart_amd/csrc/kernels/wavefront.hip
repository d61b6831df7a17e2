// Persistent wavefront path tracer with batching over views and scenes.
//
// Work is cut into chunks of at most `queue_slots` pixel-samples. A chunk is a
// list of tiles (job, pixel range, sample range); slots are numbered tile by tile.
// One chunk runs as a captured HIP graph:
//
//   setup -> generate -> [extend -> shade -> shadow] x max_depth -> resolve
//
//   generate camera rays (origin, direction) of the chunk's pixel-samples, queued
//            in groups of 64 that share a pixel (or a small pixel block)
//   extend   closest hit of every ray in the current queue (traversal only, low
//            register pressure, persistent waves fetching 64 rays at a time; the
//            first iteration's camera rays are traced 64 at a time as packets where there
//            are enough of them)
//   shade    shade_vertex() of every hit; survivors are compacted into the next
//            queue and shadow rays into the shadow queue (wave ballots + one atomic
//            per workgroup and queue); what a vertex adds goes to the path's result slot
//   shadow   occlusion test of every shadow ray; adds mask * direct to the result
//   resolve  adds the result slots of each pixel to its running sum in sample order
//
// All paths of a chunk are at bounce `it` during iteration `it`, and the vertex
// arithmetic is the megakernel's (path.hpp), so every image is bit-identical to
// the megakernel's for the same seed, view and depth. The graph is replayed once
// per chunk; kernels find their chunk through a device-side index, and every
// counter is cleared by a kernel (no memset nodes in the graph).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../host/common.hpp"
#include "path.hpp"
#include "renderer.hpp"

namespace prt {

constexpr int kMaxIter = 64;
// Same-address atomics serialise (about 11 ns each on MI355X), so work beyond each
// wave's first batch is handed out by kSpread counters, one kBatch-item batch per
// atomic, and appends to a queue are aggregated per workgroup.
// Fetch counters per (kernel, iteration), items per fetch atomic (launch_shape.hpp), and shade
// workgroup size. With every counter on its own line, 1080p x 128 spp measured
// within noise of 64 / 512 for batch 128 and 1024-thread shade workgroups;
// 256-thread shade workgroups were 2-4 % slower.
#ifndef PRT_SHADE_BLOCK
#define PRT_SHADE_BLOCK 512
#endif
constexpr int kShadeBlock = PRT_SHADE_BLOCK;
// Waves of wf_shade per compute unit in its grid (its occupancy limit, 4 waves per SIMD).
#ifndef PRT_SHADE_GRID_WAVES
#define PRT_SHADE_GRID_WAVES 16
#endif
constexpr int kShadeGridWaves = PRT_SHADE_GRID_WAVES;
// Bytes of queues and path state per slot: 2 queues x 48, hit record 4, shadow 48 + 4, result 16.
constexpr size_t kSlotBytes = 2 * 48 + 4 + 48 + 4 + 16;
// Counter words per 128-byte cache line. Each queue counter and each fetch counter
// has a line of its own: atomics on one line serialize in its L2 channel, and the
// appends of wf_shade and the batch fetches of the traversal kernels would otherwise
// share a few lines.
#ifndef PRT_CTR_LINE
#define PRT_CTR_LINE 32
#endif
constexpr uint32_t kCtrLine = PRT_CTR_LINE;
enum WfCounter : uint32_t {
    kChunk = 0,                // number of the chunk being rendered, from 1
    kStats = kCtrLine,         // kCntNum 64-bit counters (two words each) of a batch
    kQueue = 4 * kCtrLine,     // rays of each iteration's queues: extension at kQueue + 2 * it lines, shadow after it
    kFetch = kQueue + 2 * (kMaxIter + 1) * kCtrLine,  // fetch counters: 2 * kMaxIter groups of kSpread,
                               // counter c of group g at kFetch + (g * kSpread + c) * kCtrLine
    kNumCounters = kFetch + 2 * kMaxIter * kSpread * kCtrLine,
};
static_assert(kStats + 2 * kCntNum <= kQueue, "the statistics lie below the queue counters");
constexpr uint32_t ext_count(uint32_t it) { return kQueue + 2 * it * kCtrLine; }
constexpr uint32_t shadow_count(uint32_t it) { return kQueue + (2 * it + 1) * kCtrLine; }
// First fetch counter of an iteration's extension or shadow rays.
constexpr uint32_t ext_fetch(uint32_t it) { return kFetch + 2 * it * kSpread * kCtrLine; }
constexpr uint32_t shadow_fetch(uint32_t it) { return kFetch + (2 * it + 1) * kSpread * kCtrLine; }

struct WfJob {
    SceneArgs sc;
    CamArgs cam;
    PathArgs path;
    uint32_t width, height;
    float4* accum;
    float4* samples;       // nullptr, or each sample's radiance at [pixel * samples_cap + sample]
    uint32_t samples_cap;  // samples stored per pixel
};

struct WfTile {
    uint32_t job, p0, p1, s0, s1;
    uint32_t slot0;  // first slot of the tile in its chunk
    uint32_t pix0;   // first resolve thread of the tile in its chunk
    uint32_t pad;
};

struct WfChunk {
    uint32_t tile0, ntiles, paths, pixels;
};

// Queue entry (structure of arrays, one float4 each, coalesced by queue index):
//   A  origin.xyz, pixel | job << 24
//   B  direction.xyz, sample index
//   C  throughput.xyz, slot | (previous bsdf specular or refractive) << 31
// Shadow entry: E origin.xyz, distance to the light sample | F direction.xyz, light id |
//   non-finite throughput channels << 28 | G contribution.xyz, slot; and the job.
// A path's slot is its position in the chunk's first queue; result[slot] is its colour so
// far, touched only by the vertices that change it (first vertex, emission, sky, a visible
// light sample). Queue order and slots keep neighbouring paths together, so those accesses
// coalesce. (Carrying the colour in the queue entries, and the light sample's position,
// normal, coordinates and throughput in the shadow entries, took 64 bytes each, and
// wf_shade, whose first launch runs at the memory's rate, wrote them.)
constexpr uint32_t kSlotMask = 0x7FFFFFFFu;   // a queue of 2^31 slots would not fit the memory
constexpr uint32_t kLightIdMask = 0x0FFFFFFFu;  // triangle ids are below 2^28
struct WfArgs {
    const WfJob* jobs;
    const WfTile* tiles;
    const WfChunk* chunks;
    uint32_t* ctr;
    unsigned long long* stats;  // kCntNum counters that the rays are added to
    float4* qa[2];
    float4* qb[2];
    float4* qc[2];
    uint32_t* hits;  // record of the closest hit (0xFFFFFFFF = miss)
    float4* se;
    float4* sf;
    float4* sg;
    uint32_t* sj;    // the shadow entry's job or, with `vertices`, its pixel-sample
    float4* result;  // per slot colour
    // One job only: nullptr, or every path's vertices, pixel-sample (p, s) at bounce b at
    // vertices[b * vertex_stride + p * vertex_cap + s], s < vertex_cap.
    uint32_t* vertices;
    size_t vertex_stride;
    uint32_t vertex_cap;
    int* spill;
    uint32_t spill_stride;
    uint32_t max_depth;
    uint32_t one_scene;  // every job traverses the same scene
    uint32_t group_lg;  // log2 of the forced camera-path block side, or kNone: choose per section
};

// What a captured launch sequence was made for.
struct LaunchKey {
    WfArgs args;
    uint32_t max_depth;
    int pblocks, gblocks, sblocks;
    bool packets, count;
};

struct WavefrontState {
    uint32_t capacity = 0;       // slots
    size_t spill_ints = 0;
    void* mem = nullptr;  // the queues
    int* spill = nullptr;
    uint32_t* ctr = nullptr;
    WfArgs args{};
    // jobs, tiles and chunks of the plan, one after another
    char* d_plan = nullptr;
    size_t cap_plan = 0;
    std::vector<char> h_plan;
    // The launch sequence of a chunk. Its kernels take their arguments by value, and what
    // those point to are this state's buffers, so it stays good while the key does:
    // capturing and instantiating it again on every call took about 0.1 ms.
    hipGraphExec_t exec = nullptr;
    LaunchKey key;
    hipEvent_t e0 = nullptr, e1 = nullptr;
};

namespace dev {

constexpr uint32_t kNone = 0xFFFFFFFFu;

// Hands out 64-item batches of [0, n) to the waves of a launch. Wave w's first batch
// is batch w, with no atomic; the batches from `waves` on belong to kSpread counters
// in turn, and a wave draws from counter (wave % kSpread): issue() sends the atomic
// for its next batch before the current batch is processed, so the round trip
// overlaps the traversal. When its counter is exhausted the wave tries kSteal others (every
// counter is some wave's own, trace_waves, so none is left out):
// neighbouring batches belong to different counters, so these run out at about the same
// time and there is little to take over. A queue of at most `waves` batches costs no
// atomic. resolve() returns the batch's first item or kNone. All of it but the atomic in
// flight is wave-uniform and stays in scalar registers.
// What bounds small queues is this ending: with every wave asking all other counters one
// after the other, each launch ended in 63 dependent loads, about 45 us (256 x 256 x 16 samples
// of a 36-triangle box, depth 5: the traversal launches 632 -> 400 us per frame);
// one vector load of all 64 counters per wave still read each of their lines once
// per wave, and cost a 0.9 ms packet launch 70 us.
struct WaveFetch {
    uint32_t* ctr;
    uint32_t k, nb, waves;
    __device__ __forceinline__ uint32_t issue() const {
        uint32_t idx = kNone;
        if (nb > waves && (threadIdx.x & 63) == 0) idx = atomicAdd(ctr + k * kCtrLine, 1u);
        return idx;
    }
    __device__ __forceinline__ uint32_t resolve(uint32_t raw) {
        if (nb <= waves) return kNone;
        uint32_t idx = uniform_u32(raw);
        for (uint32_t tries = 0; idx >= fetch_limit(nb, waves, k); ++tries) {
            if (tries == kSteal) return kNone;
            k = next_counter(k);
            idx = kNone;
            if ((threadIdx.x & 63) == 0) idx = atomicAdd(ctr + k * kCtrLine, 1u);
            idx = uniform_u32(idx);
        }
        return fetch_batch(waves, k, idx) * kBatch;
    }
    // The wave's first batch (counted from the last wave if `reversed`); sets up the fetch
    // of the others.
    __device__ __forceinline__ uint32_t start(uint32_t* counters, uint32_t n, bool reversed = false) {
        const uint32_t wave = uniform_u32(blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64);
        ctr = counters;
        k = wave % kSpread;
        nb = (n + kBatch - 1) / kBatch;
        waves = gridDim.x * (blockDim.x / 64);
        const uint32_t first = reversed ? waves - 1u - wave : wave;
        return first < nb ? first * kBatch : kNone;
    }
};
// Hands single items of [0, n) to individual lanes: the wave holds one 64-item
// batch of a WaveFetch at a time (one atomic per 64 items, the next one already
// in flight) and gives its items to whichever lanes ask, so a lane whose ray has
// finished takes a new one while the others keep traversing. Every issued atomic
// is resolved before more() turns false. Calls must be wave-uniform.
struct LaneFeeder {
    WaveFetch fetch;
    uint32_t n, base, used, pending;
    __device__ __forceinline__ void start(uint32_t* ctr, uint32_t count, bool reversed = false) {
        n = count;
        base = fetch.start(ctr, count, reversed);
        used = 0;
        pending = base != kNone ? fetch.issue() : kNone;
    }
    __device__ __forceinline__ bool more() const { return base != kNone; }
    // Lanes with `want` get the next item, or kNone once every item is handed out.
    __device__ __forceinline__ uint32_t take(bool want) {
        const uint32_t lane = threadIdx.x & 63;
        const unsigned long long below = (1ull << lane) - 1ull;
        uint32_t item = kNone;
        unsigned long long m = __ballot(want);
        while (m != 0ull && base != kNone) {
            const uint32_t size = min(kBatch, n - base);
            const uint32_t avail = size - used;
            const uint32_t rank = uint32_t(__popcll(m & below));
            if (((m >> lane) & 1ull) && rank < avail) item = base + used + rank;
            used += min(uint32_t(__popcll(m)), avail);
            if (used == size) {
                base = fetch.resolve(pending);
                used = 0;
                pending = base != kNone ? fetch.issue() : kNone;
            }
            m = __ballot(want && item == kNone);
        }
        return item;
    }
};

// Idle lanes of a wave that trigger a refill (the rest keep traversing meanwhile).
// kRefill <= 64, so a wave with no active lane always refills or, with no work
// left, leaves the loop. The finished rays' writes and the new rays' set-up run at
// that point with these lanes only; on 1080p x 128 spp over 1M triangles, 32 took
// 125.7 ms per frame, 16 129.0, 40 128.3 and 48 139.5.
#ifndef PRT_REFILL_LANES
#define PRT_REFILL_LANES 32
#endif
constexpr uint32_t kRefill = PRT_REFILL_LANES;
static_assert(kRefill >= 1 && kRefill <= 64, "refill threshold out of range");

__device__ __forceinline__ uint32_t idle_lanes(bool active) { return uint32_t(__popcll(__ballot(!active))); }

// A pointer that every lane of the wave holds, moved to scalar registers. Read from
// the job table with vector loads (the compiler cannot prove that memory read-only),
// the scene's node and triangle bases would otherwise take four VGPRs and a 64-bit
// add per fetch; from SGPRs the fetches use the scalar base + vector offset form.
template <class T>
__device__ __forceinline__ const T* wave_uniform(const T* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))));
    return reinterpret_cast<const T*>((uint64_t(hi) << 32) | lo);
}

// The first job's scene, by scalar loads.
__device__ __forceinline__ SceneArgs uniform_scene(const WfJob* jobs) {
    const SceneArgs& j = jobs->sc;
    SceneArgs s;
    s.nodes = sload(&j.nodes, 0);
    s.tris = sload(&j.tris, 0);
    s.shade = sload(&j.shade, 0);
    s.mats = sload(&j.mats, 0);
    s.lights = sload(&j.lights, 0);
    s.texels = sload(&j.texels, 0);
    s.texinfo = sload(&j.texinfo, 0);
    s.lin = sload(&j.lin, 0);
    s.lights_area = sload(&j.lights_area, 0);
    s.inv_lights_area = sload(&j.inv_lights_area, 0);
    s.num_lights = sload(&j.num_lights, 0);
    s.num_records = sload(&j.num_records, 0);
    return s;
}

// Phase thresholds of wf_trace's extension and shadow rays (node_phase_for). On 1080p x 128
// spp over 1M triangles, 24 measured best for both (extension 109 -> 92 ms, shadow
// 54 -> 43 ms per frame against no phases; 8 and 32 to 48 were slower).
#ifndef PRT_EXTEND_PHASE_MIN
#define PRT_EXTEND_PHASE_MIN 24
#endif
#ifndef PRT_SHADOW_PHASE_MIN
#define PRT_SHADOW_PHASE_MIN 24
#endif
static_assert(PRT_EXTEND_PHASE_MIN >= 0 && PRT_EXTEND_PHASE_MIN <= 64, "phase threshold out of range");
static_assert(PRT_SHADOW_PHASE_MIN >= 0 && PRT_SHADOW_PHASE_MIN <= 64, "phase threshold out of range");

// Waves per SIMD of the traversal kernels: 8 with the scene bases and the feeder in SGPRs.
// wf_trace then has 4 VGPRs too few and spills on rarely taken paths (7 waves, no spill:
// 66.9 instead of 66.4 ms on 1080p x 128 spp over 1M triangles). Rays of several scenes hold
// their bases in VGPRs too; at 8 waves that spills 8 in the loop (5.25 instead of 4.23 ms on
// 12 views of several scenes), so there wf_trace keeps 7.
#ifndef PRT_PACKET_WAVES
#define PRT_PACKET_WAVES __attribute__((amdgpu_waves_per_eu(8)))
#endif
// Adds the wave's counts to the counter slots; ANYHIT also books nodes and
// triangles as the shadow (any-hit) kernel's share.
template <bool ANYHIT>
__device__ __forceinline__ void flush_stats(unsigned long long* out, const Counts& c) {
    unsigned long long v[6] = {c.primary, c.extension, c.shadow, c.nodes, c.tris, c.hits};
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        unsigned long long x = v[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if ((threadIdx.x & 63) == 0 && x) {
            atomicAdd(out + k, x);
            if (ANYHIT && k == kCntNodes) atomicAdd(out + kCntAnyNodes, x);
            if (ANYHIT && k == kCntTris) atomicAdd(out + kCntAnyTris, x);
        }
    }
}

__device__ __forceinline__ uint32_t find_tile(const WfTile* t, uint32_t first, uint32_t n, uint32_t key, bool by_pix) {
    uint32_t lo = first, hi = first + n - 1;
    while (lo < hi) {
        uint32_t mid = (lo + hi + 1) / 2;
        uint32_t v = by_pix ? t[mid].pix0 : t[mid].slot0;
        if (v <= key) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Goes on to the next chunk: its path count, empty queues and fetch counters for the
// iterations it will run, a thread each (one workgroup clearing all of them took 9 us).
__global__ __launch_bounds__(256) void wf_setup(WfArgs a) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < 2 * a.max_depth * kSpread) a.ctr[kFetch + k * kCtrLine] = 0;
    if (k >= 1 && k <= 2 * a.max_depth) a.ctr[kQueue + k * kCtrLine] = 0;
    if (k != 0) return;
    const uint32_t c = a.ctr[kChunk];
    a.ctr[kChunk] = c + 1;
    a.ctr[ext_count(0)] = a.chunks[c].paths;
}
// The chunk that wf_setup has gone on to.
__device__ __forceinline__ WfChunk current_chunk(const WfArgs& a) {
    return a.chunks[__builtin_amdgcn_readfirstlane(a.ctr[kChunk]) - 1];
}

// Path order within a tile. The tile's samples are cut into sections of m consecutive
// samples: as many full ones as there are (m = 64, or all of fewer), then the rest. Within a
// section the pixels come in order of position q, each with its m samples one after
// another, so 64 consecutive paths (one wave's batch) are the m samples of about 64 / m
// pixels. q runs through bands of g rows, column by column, with g near sqrt(64 / m):
// those pixels are a block, whatever the image's size and sample count. At 128 spp a wave
// traces 64 samples of one pixel: nearly the same primary ray in every lane, then shadow
// and extension rays from nearly the same point. On 1080p x 128 spp over 1M triangles,
// one pixel x 64 samples took 147.3 ms per frame, 4 x 4 x 4 148.1, 8 x 8 x 1 148.6 and row
// order 151.7. (Blocks only where they divided the image and the sample count left every
// other size in row order: packets of 64 pixels of a row; 12 views of odd
// sizes, 8 to 64 spp: 2.43 -> 1.31 ms in the packet launch; 3840 x 2160 x 6 spp, which took
// 8 x 8 x 1: 4.0 -> 2.55.)
// A tile that does not cover whole rows is taken as one row. A path's result slot is its
// position in this order; wf_resolve adds every pixel's samples in sample order.
struct PathOrder {
    uint32_t width, rows;  // of the tile (a tile of part of a row: its pixels, 1)
    uint32_t pixels;
    uint32_t m, full, rest;  // samples of a full section, full sections, samples of the last one (or 0)
    uint32_t g;              // band height of the full sections
};
__device__ __forceinline__ uint32_t band_rows(uint32_t m) { return m >= 32u ? 1u : m >= 7u ? 2u : m >= 2u ? 4u : 8u; }
// force_lg (not kNone) asks for bands of g = 2^force_lg rows and sections of 64 / g^2 samples.
__device__ __forceinline__ PathOrder path_order(const WfTile& t, uint32_t width, uint32_t force_lg) {
    PathOrder o;
    o.pixels = t.p1 - t.p0;
    const bool whole = t.p0 % width == 0u && o.pixels % width == 0u;
    o.width = whole ? width : o.pixels;
    o.rows = whole ? o.pixels / width : 1u;
    const uint32_t ns = t.s1 - t.s0;
    const bool force = force_lg <= 3u;
    o.m = min(force ? 64u >> (2u * force_lg) : 64u, ns);
    o.g = force ? 1u << force_lg : band_rows(o.m);
    o.full = ns / o.m;
    o.rest = ns - o.full * o.m;
    return o;
}
// Pixel offset from the tile's first pixel of position q, in band `band` of bands of g rows
// (a power of two), and back.
__device__ __forceinline__ uint32_t position_to_pixel(const PathOrder& o, uint32_t g, uint32_t band, uint32_t q) {
    if (g == 1u) return q;
    const uint32_t in = q - band * (o.width * g), h = min(g, o.rows - band * g);
    const uint32_t x = h == g ? in >> (31 - __builtin_clz(g)) : in / h;
    return (band * g + (in - x * h)) * o.width + x;
}
__device__ __forceinline__ uint32_t position_to_pixel(const PathOrder& o, uint32_t g, uint32_t q) {
    return position_to_pixel(o, g, g == 1u ? 0u : q / (o.width * g), q);
}
__device__ __forceinline__ uint32_t pixel_to_position(const PathOrder& o, uint32_t g, uint32_t pixel) {
    if (g == 1u) return pixel;
    const uint32_t y = pixel / o.width, x = pixel - y * o.width;
    const uint32_t band = y / g, h = min(g, o.rows - band * g);
    return band * g * o.width + x * h + (y - band * g);
}

// n / d for inv = 1.0 / d, any 32-bit n and d >= 1: (n + 1/2) / d is at least 1 / (2d) from a
// whole number, and the roundings of inv and of the product move it by less than 2^-20 / d.
__device__ __forceinline__ uint32_t quotient(uint32_t n, double inv) { return uint32_t((double(n) + 0.5) * inv); }

// The camera rays of the chunk's paths, one thread each, striding over the slots. Bound by
// VALU issue: of about 400 instructions a path 200 were the divisions that find its tile's
// order, pixel and sample. A thread now keeps its tile, the tile's order and the reciprocals
// of its divisors until its slot leaves the tile, which hundreds of its slots share.
// (2.70 -> 2.02 ms on 1080p x 128 spp, 0.55 -> 0.37 at 4K x 6 spp; 32 bytes a path are
// written, 4.2 TB/s.)
__global__ __launch_bounds__(256) void wf_generate(WfArgs a) {
    const WfChunk ch = current_chunk(a);
    WfTile t;
    PathOrder o;
    uint32_t paths = 0, g_rest = 1, width = 1;  // `paths` slots from t.slot0 on are the tile's
    double by_section = 0, by_m = 0, by_rest = 0, by_band = 0, by_band_rest = 0, by_width = 0;
    t.slot0 = 0;
    for (uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x; slot < ch.paths; slot += gridDim.x * blockDim.x) {
        if (slot - t.slot0 >= paths) {
            t = a.tiles[find_tile(a.tiles, ch.tile0, ch.ntiles, slot, false)];
            width = a.jobs[t.job].width;
            o = path_order(t, width, a.group_lg);
            paths = o.pixels * (t.s1 - t.s0);
            g_rest = band_rows(o.rest);
            by_section = 1.0 / double(o.pixels * o.m);
            by_m = 1.0 / double(o.m);
            by_rest = 1.0 / double(max(o.rest, 1u));
            by_band = 1.0 / double(o.width * o.g);
            by_band_rest = 1.0 / double(o.width * g_rest);
            by_width = 1.0 / double(width);
        }
        const WfJob& j = a.jobs[t.job];
        const uint32_t r = slot - t.slot0;
        const uint32_t sec = quotient(r, by_section), in = r - sec * (o.pixels * o.m);
        const bool last = sec == o.full;
        const uint32_t q = quotient(in, last ? by_rest : by_m);
        const uint32_t g = last ? g_rest : o.g;
        const uint32_t band = g == 1u ? 0u : quotient(q, last ? by_band_rest : by_band);
        const uint32_t pixel = t.p0 + position_to_pixel(o, g, band, q);
        const uint32_t sample = t.s0 + sec * o.m + (in - q * (last ? o.rest : o.m));
        const uint32_t row = quotient(pixel, by_width);
        Rng rng{j.path.seed, j.path.view, pixel, sample};
        V3 ro, rd;
        camera_ray(j.cam, int(pixel - row * width), int(row), rng.block(0), ro, rd);
        // C of a new path (throughput 1, no previous vertex, its slot) and its colour are
        // made by wf_shade(0): the slot is the queue position.
        a.qa[0][slot] = make_float4(ro.x, ro.y, ro.z, __uint_as_float(pixel | (t.job << 24)));
        a.qb[0][slot] = make_float4(rd.x, rd.y, rd.z, __uint_as_float(sample));
    }
}

// Closest hit of every ray in the queue of iteration `it`. ONE_SCENE: every job of the
// batch traverses the same scene, so the node and triangle arrays are wave-uniform
// (scalar registers).
template <bool COUNT, bool ONE_SCENE>
__device__ __forceinline__ void extend_rays(const WfArgs& a, uint32_t it, StackT<kStackLdsQueue>& st) {
    const uint32_t q = it & 1u;
    const uint32_t n = uniform_u32(a.ctr[ext_count(it)]);
    Counts cnt = {0, 0, 0, 0, 0, 0};
    LaneFeeder feed;
    feed.start(&a.ctr[ext_fetch(it)], n, true);
    bool active = false;
    // A lane whose ray has finished keeps its hit record in a register until the next
    // refill point, where every such lane writes it at once.
    bool finished = false;
    uint32_t i = 0;
    TravRay ray;
    ray.leaf = kNoChild;
    HitRec h;
    const float4* nodes = ONE_SCENE ? wave_uniform(a.jobs[0].sc.nodes) : nullptr;
    const float4* tris = ONE_SCENE ? wave_uniform(a.jobs[0].sc.tris) : nullptr;
    while (true) {
        const uint32_t idle = idle_lanes(active);
        if (idle >= kRefill) {
            if (finished) {
                a.hits[i] = h.rec;
                finished = false;
            }
            if (!feed.more()) {
                if (idle == 64) break;
            } else if (const uint32_t got = feed.take(!active); got != kNone) {
                i = got;
                const float4 o = a.qa[q][i], d = a.qb[q][i];
                if (!ONE_SCENE) {
                    const SceneArgs& sc = a.jobs[__float_as_uint(o.w) >> 24].sc;
                    nodes = sc.nodes;
                    tris = sc.tris;
                }
                if (COUNT) {
                    if (it == 0) cnt.primary++; else cnt.extension++;
                }
                h.t = kFltMax;
                h.id = 0;
                h.rec = 0xFFFFFFFFu;
                h.mat = 0;
                h.u = h.v = 0.f;
                st.sp = 0;
                active = trav_begin(ray, v3(o), v3(d));
                if (!active) a.hits[i] = 0xFFFFFFFFu;  // zero direction: no triangle can be hit
            }
        }
        // One node phase or leaf phase per step; a refill is considered every step.
        const bool node_phase = node_phase_for<PRT_EXTEND_PHASE_MIN>(active && trav_wants_nodes(ray), active);
        if (active) {
            if (trav_step<false, COUNT, true>(node_phase, nodes, tris, ray, kEps, h, st, cnt) != kTravRunning) {
                active = false;
                finished = true;
            }
        }
    }
    if (COUNT) flush_stats<false>(a.stats, cnt);
}

// Occlusion test of every shadow ray of iteration `it`; a visible light sample's
// contribution is added to the path's colour. A finished ray's update waits for the next
// refill point too; it is read back from the entry there, so that a lane holds only the
// entry's index meanwhile (with the light geometry set up here and throughput, light and
// destination held per lane, this took 72 VGPRs and 7 waves per SIMD).
template <bool COUNT, bool ONE_SCENE>
__device__ __forceinline__ void shadow_rays(const WfArgs& a, uint32_t it, StackT<kStackLdsQueue>& st) {
    const uint32_t n = uniform_u32(a.ctr[shadow_count(it)]);
    Counts cnt = {0, 0, 0, 0, 0, 0};
    LaneFeeder feed;
    feed.start(&a.ctr[shadow_fetch(it)], n);
    bool active = false;
    TravRay ray;
    ray.leaf = kNoChild;
    HitRec occ;
    const float4* nodes = ONE_SCENE ? wave_uniform(a.jobs[0].sc.nodes) : nullptr;
    const float4* tris = ONE_SCENE ? wave_uniform(a.jobs[0].sc.tris) : nullptr;
    uint32_t i = 0;
    bool finished = false, lit = false;
    while (true) {
        const uint32_t idle = idle_lanes(active);
        if (idle >= kRefill) {
            if (finished) {
                const uint32_t odd = __float_as_uint(a.sf[i].w) >> 28;
                if (lit || odd != 0u) {
                    const float4 g = a.sg[i];
                    float4* dst = a.result + __float_as_uint(g.w);
                    const float4 c = *dst;
                    const float nan = __builtin_nanf("");
                    const V3 add = lit ? v3(g) : v3(odd & 1u ? nan : 0.f, odd & 2u ? nan : 0.f, odd & 4u ? nan : 0.f);
                    const V3 s = v3(c) + add;
                    *dst = make_float4(s.x, s.y, s.z, 0.f);
                    if (lit && a.vertices) {
                        const uint32_t path = a.sj[i];
                        if (path != kNone) atomicOr(a.vertices + it * a.vertex_stride + path, kVertexLit);
                    }
                }
                finished = false;
            }
            if (!feed.more()) {
                if (idle == 64) break;
            } else if (const uint32_t got = feed.take(!active); got != kNone) {
                i = got;
                const float4 e = a.se[i], f = a.sf[i];
                if (!ONE_SCENE) {
                    const SceneArgs& sc = a.jobs[a.sj[i]].sc;
                    nodes = sc.nodes;
                    tris = sc.tris;
                }
                occ.t = e.w;
                occ.id = __float_as_uint(f.w) & kLightIdMask;
                occ.rec = 0;
                occ.mat = 0;
                occ.u = occ.v = 0.f;
                st.sp = 0;
                active = trav_begin(ray, v3(e), v3(f));  // true: wf_shade queues only rays that can hit
            }
        }
        const bool node_phase = node_phase_for<PRT_SHADOW_PHASE_MIN>(active && trav_wants_nodes(ray), active);
        if (active) {
            const int r = trav_step<true, COUNT, true>(node_phase, nodes, tris, ray, kEps, occ, st, cnt);
            if (r != kTravRunning) {
                active = false;
                finished = true;
                lit = r == kTravDone;
            }
        }
    }
    if (COUNT) flush_stats<true>(a.stats, cnt);
}

// The shadow rays of iteration it - 1 and the extension rays of iteration `it`, both made
// by wf_shade(it - 1) and independent of each other, in one launch: a wave that finds no
// more shadow rays goes on to extension rays, so the end of the one, where a few long rays
// are left, is filled by the other, and in small queues (fewer batches than waves) the
// first waves take the shadow rays while the last take the extension rays. (1280 x 720 x
// 16 samples, 1M triangles, depth 8: 6.96 -> 6.13 ms per frame for the two together; 1080p x
// 128: 73.9 -> 73.1; a 256 x 256 x 16 box: 376 -> 325 us.)
enum : uint32_t { kTraceShadow = 1, kTraceExtend = 2 };
template <bool COUNT, bool ONE_SCENE>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(ONE_SCENE ? 8 : 7)))
void wf_trace(WfArgs a, uint32_t it, uint32_t parts) {
    __shared__ int s_stack[kStackLdsQueue * kBlock];
    StackT<kStackLdsQueue> st;
    st.bind(s_stack, a.spill + size_t(blockIdx.x) * kBlock, a.spill_stride);
    if (parts & kTraceShadow) shadow_rays<COUNT, ONE_SCENE>(a, it - 1, st);
    if (parts & kTraceExtend) extend_rays<COUNT, ONE_SCENE>(a, it, st);
}

// Runs f(lanes, job) once per distinct job among the wave's `live` lanes, with
// `lanes` true for the lanes of that job and the job index wave-uniform: a packet
// traversal needs one scene per pass. With ONE_SCENE there is one pass.
template <bool ONE_SCENE, class F>
__device__ __forceinline__ void per_scene_pass(bool live, uint32_t job, F&& f) {
    if (ONE_SCENE) {
        f(live, 0u);
        return;
    }
    bool todo = live;
    unsigned long long m = __ballot(todo);
    while (m != 0ull) {
        const uint32_t jl = uint32_t(__builtin_amdgcn_readlane(int(job), __builtin_ctzll(m)));
        const bool mine = todo && job == jl;
        f(mine, jl);
        todo = todo && !mine;
        m = __ballot(todo);
    }
}

// The first iteration's extension rays, whose queue holds the camera rays in 64-ray
// batches of 64 samples of a pixel or pixel block (wf_generate): nearly the same
// ray in every lane. Each wave takes one batch at a time and traces it as a packet
// (packet_traverse). On the 1080p 128-spp frame over 1M triangles this launch took
// 15.8 ms with per-lane traversal and 9.9 ms as packets. (Packets measured 5x
// slower for the first iteration's occlusion rays, whose batches fan out over the
// lights, and later iterations' rays leave diffuse bounces in all directions.)
static_assert(kBatch == 64 && kBlock == 64, "a packet is one fetch batch traced by one wave");
template <bool COUNT, bool ONE_SCENE>
__global__ __launch_bounds__(kBlock) PRT_PACKET_WAVES void wf_extend_packet(WfArgs a) {
    __shared__ int s_pk[kPacketStack];
    const uint32_t n = uniform_u32(a.ctr[ext_count(0)]);
    Counts cnt = {0, 0, 0, 0, 0, 0};
    const uint32_t lane = threadIdx.x & 63u;
    WaveFetch fetch;
    uint32_t base = fetch.start(&a.ctr[ext_fetch(0)], n);
    uint32_t pending = base != kNone ? fetch.issue() : kNone;
    while (base != kNone) {
        const uint32_t i = base + lane;
        const bool valid = i < n;
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f), d = o;
        if (valid) {
            o = a.qa[0][i];
            d = a.qb[0][i];
        }
        if (COUNT && valid) cnt.primary++;
        TravRay ray;
        const bool began = trav_begin(ray, v3(o), v3(d));  // false for the zero ray of an empty lane
        const bool live = valid && began;
        HitRec h;
        h.t = kFltMax;
        h.id = 0;
        h.rec = 0xFFFFFFFFu;
        h.mat = 0;
        h.u = h.v = 0.f;
        per_scene_pass<ONE_SCENE>(live, __float_as_uint(o.w) >> 24, [&](bool mine, uint32_t job) {
            const float4* nodes = wave_uniform(a.jobs[job].sc.nodes);
            const float4* tris = wave_uniform(a.jobs[job].sc.tris);
            bool occ;
            packet_traverse<false, COUNT>(nodes, tris, mine, ray, kEps, h, (lds_int*)s_pk, cnt, occ);
        });
        if (valid) {
            a.hits[i] = h.rec;
        }
        base = fetch.resolve(pending);
        pending = base != kNone ? fetch.issue() : kNone;
    }
    if (COUNT) flush_stats<false>(a.stats, cnt);
}

// Appends to two queues for a whole workgroup with one atomic per queue: lanes
// with more / nee get consecutive positions. Returns (next-queue, shadow) positions.
// (Grouping a workgroup's shadow rays by the light they aim at, so that 64-ray
// batches mostly share a light, measured 2% slower per frame on the 1M-triangle
// scene with its two lights 10 units apart: the queue order of shade, pixel by
// pixel, is the better one for the L2.)
// Every wave of the workgroup waits here for the atomics' round trip, so what comes before and
// after it is kept short: 8 lanes per queue add up the waves' counts, both atomics go out in
// one instruction, and the LDS slots alternate (`turn`), so that two barriers a turn are
// enough. 1080p x 128 spp over 1M triangles: wf_shade 25.4 ms with one thread adding up and
// three barriers, 24.7 so; 256 x 256 x 16 over 36 155 and 151 us. (The counters themselves are
// not what bounds it: with eight counters and queue segments, one per XCD, 24.7 too.)
constexpr uint32_t kShadeWaves = kShadeBlock / 64;
static_assert(kShadeWaves <= 32 && (kShadeWaves & (kShadeWaves - 1)) == 0, "a wave holds both queues' counts");
__device__ __forceinline__ uint2 block_append(bool more, bool nee, uint32_t* ctr_next, uint32_t* ctr_shadow,
                                              uint32_t turn) {
    __shared__ uint32_t s_off[2][2 * kShadeWaves];
    uint32_t* off = s_off[turn & 1u];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const unsigned long long m0 = __ballot(more), m1 = __ballot(nee);
    if (lane == 0) {
        off[wave] = uint32_t(__popcll(m0));
        off[kShadeWaves + wave] = uint32_t(__popcll(m1));
    }
    __syncthreads();
    if (wave == 0 && lane < 2 * kShadeWaves) {
        const uint32_t count = off[lane], w = lane & (kShadeWaves - 1u);
        uint32_t sum = count;  // of the queue's waves up to this one
#pragma unroll
        for (uint32_t d = 1; d < kShadeWaves; d <<= 1) {
            const uint32_t below = __shfl_up(sum, d, kShadeWaves);
            if (w >= d) sum += below;
        }
        uint32_t base = 0;
        if (w == kShadeWaves - 1u && sum != 0u) base = atomicAdd(lane < kShadeWaves ? ctr_next : ctr_shadow, sum);
        off[lane] = __shfl(base, kShadeWaves - 1, kShadeWaves) + sum - count;
    }
    __syncthreads();
    const unsigned long long lt = (1ull << lane) - 1ull;
    return make_uint2(off[wave] + uint32_t(__popcll(m0 & lt)), off[kShadeWaves + wave] + uint32_t(__popcll(m1 & lt)));
}

// Channels of a throughput that are not finite, as bits: mask * 0 is then NaN, not 0.
__device__ __forceinline__ uint32_t nonfinite(V3 m) {
    return (fabsf(m.x) <= kFltMax ? 0u : 1u) | (fabsf(m.y) <= kFltMax ? 0u : 2u) | (fabsf(m.z) <= kFltMax ? 0u : 4u);
}

// Shades every hit of the queue, sets up the shadow rays of the light samples and
// compacts the survivors. The colour the vertex adds starts at 0 (0 + x = x exactly) and
// is added to the path's result; a visible light sample's part is added by wf_trace.
//
// A path's loads are a chain (its entry and hit, the triangle, the material, the light), and
// 16 waves per compute unit hide little of it, so the chain is kept short. With ONE_SCENE the
// scene's arrays come from scalar registers: read through the job they took vector loads of
// the descriptor before every other load (the compiler reads memory that the kernel may have
// written, and the queues might be that, by vector loads), 23.05 -> 21.15 ms on 1080p x 128
// spp over 1M triangles. The triangle's loads go out before the Philox blocks (-> 20.25),
// the light's index, the light's records and its material before they are known to be needed
// (24.8 -> 23.3 with hit_details without branches), all as global instead of flat loads
// (-> 23.05). The launches now move 4.6 TB/s, the rate of a copy. 512-thread workgroups, 128
// VGPRs: 5 or 6 waves per SIMD spilled and took 2 % and 12 % longer, 256- and 128-thread
// workgroups at 5 and 6 waves 4 % and 25 %.
template <bool COUNT, bool ONE_SCENE>
__global__ __launch_bounds__(kShadeBlock) __attribute__((amdgpu_waves_per_eu(4)))
void wf_shade(WfArgs a, uint32_t it) {
    const SceneArgs shared = uniform_scene(a.jobs);
    const uint32_t q = it & 1u;
    const uint32_t n = uniform_u32(a.ctr[ext_count(it)]);
    Counts cnt = {0, 0, 0, 0, 0, 0};
    // Static, workgroup-uniform partition of the queue (shading cost varies little).
    uint32_t turn = 0;
    for (uint32_t base = blockIdx.x * kShadeBlock; base < n; base += gridDim.x * kShadeBlock) {
        const uint32_t i = base + threadIdx.x;
        const bool valid = i < n;
        bool more = false, want_nee = false;
        PathState ps;
        NeeSample ns;
        ShadowReq sr;
        float4 A = make_float4(0.f, 0.f, 0.f, 0.f), B = A;
        float4 Cc = make_float4(1.f, 1.f, 1.f, __uint_as_float(i));  // a new path's
        uint32_t rec = 0xFFFFFFFFu;
        if (valid) {
            A = a.qa[q][i];
            B = a.qb[q][i];
            if (it != 0) Cc = a.qc[q][i];
            rec = a.hits[i];
        }
        const uint32_t pj = __float_as_uint(A.w);
        const uint32_t slot = __float_as_uint(Cc.w) & kSlotMask;
        const uint32_t sample = __float_as_uint(B.w);
        const bool keep = a.vertices != nullptr && sample < a.vertex_cap;
        const uint32_t path = keep ? (pj & 0xFFFFFFu) * a.vertex_cap + sample : kNone;
        if (keep && valid) a.vertices[it * a.vertex_stride + path] = rec == 0xFFFFFFFFu ? kVertexMiss : rec;
        ps.ro = v3(A);
        ps.rd = v3(B);
        ps.mask = v3(Cc);
        ps.color = v3(0.f, 0.f, 0.f);
        ps.prev = __float_as_uint(Cc.w) >> 31 ? 1 /*SPECULAR*/ : 0;
        ps.b = it;
        ps.input = it == 0 ? v3(0.f, 0.f, 0.f) : ps.rd;  // at b >= 1 the stale input is the ray direction
        if (valid && rec == 0xFFFFFFFFu) {
            path_miss(ps);
        } else if (valid) {
            const WfJob& j = a.jobs[pj >> 24];
            const SceneArgs& sc = ONE_SCENE ? shared : j.sc;
            const PathArgs path_args = j.path;
            HitRec h;
            h.rec = rec;
            h.id = 0;
            // With several scenes the normals' loads go out first as well (2.67 -> 2.49 ms on 12
            // views); with one, 20.2 ms become 20.8 on 1080p x 128 spp.
            float4 normals[3] = {};
            if (!ONE_SCENE)
                for (uint32_t k = 0; k < 3; ++k) normals[k] = gload(sc.shade, size_t(rec) * 4 + k);
            __builtin_amdgcn_sched_barrier(0);
            hit_details(sc.tris, ps.ro, ps.rd, h);
            Rng rng{path_args.seed, path_args.view, pj & 0xFFFFFFu, sample};
            more = shade_vertex<COUNT, true>(sc, path_args, rng, ps, h, &want_nee, ns, cnt, nullptr,
                                             ONE_SCENE ? nullptr : normals);
            if (want_nee && !(nee_prepare<COUNT>(sc, ns, sr, cnt) && can_hit(sr.sd))) {
                want_nee = false;  // the light sample cannot be seen: add mask * 0
                ps.color = add_direct(ps.color, ns.mask, sr.direct, false);
            }
        }
        if (valid) {
            if (it == 0) {
                a.result[slot] = make_float4(ps.color.x, ps.color.y, ps.color.z, 0.f);
            } else if (ps.color.x != 0.f || ps.color.y != 0.f || ps.color.z != 0.f) {  // (NaN too)
                const V3 c = v3(a.result[slot]) + ps.color;
                a.result[slot] = make_float4(c.x, c.y, c.z, 0.f);
            }
        }
        const uint2 pos = block_append(more, want_nee, &a.ctr[ext_count(it + 1)], &a.ctr[shadow_count(it)], turn++);
        if (more) {
            const uint32_t special = ps.prev == 1 /*SPECULAR*/ || ps.prev == 4 /*REFRACTIVE*/ ? ~kSlotMask : 0u;
            a.qa[q ^ 1u][pos.x] = make_float4(ps.ro.x, ps.ro.y, ps.ro.z, A.w);
            a.qb[q ^ 1u][pos.x] = make_float4(ps.rd.x, ps.rd.y, ps.rd.z, B.w);
            a.qc[q ^ 1u][pos.x] = make_float4(ps.mask.x, ps.mask.y, ps.mask.z, __uint_as_float(slot | special));
        }
        if (want_nee) {
            const V3 c = ns.mask * sr.direct;
            const uint32_t id = sr.lid | nonfinite(ns.mask) << 28;
            a.se[pos.y] = make_float4(sr.so.x, sr.so.y, sr.so.z, sr.tL);
            a.sf[pos.y] = make_float4(sr.sd.x, sr.sd.y, sr.sd.z, __uint_as_float(id));
            a.sg[pos.y] = make_float4(c.x, c.y, c.z, __uint_as_float(slot));
            if (a.vertices) a.sj[pos.y] = path;
            else if (!a.one_scene) a.sj[pos.y] = pj >> 24;
        }
    }
    if (COUNT) {
        flush_stats<false>(a.stats, cnt);
        // Each shadow ray's own light triangle counts among the any-hit triangles.
        unsigned long long x = cnt.shadow;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if ((threadIdx.x & 63) == 0 && x) atomicAdd(a.stats + kCntAnyTris, x);
    }
}

// Adds each pixel's results to its running sum in sample order. A thread per pixel, in the
// order of the full sections, so a wave reads one run of memory; a lane's samples of a
// section lie one after another, and eight are read at once, the 128 bytes of a line.
__global__ __launch_bounds__(256) void wf_resolve(WfArgs a) {
    const WfChunk ch = current_chunk(a);
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < ch.pixels; k += gridDim.x * blockDim.x) {
        const WfTile t = a.tiles[find_tile(a.tiles, ch.tile0, ch.ntiles, k, true)];
        const WfJob& jb = a.jobs[t.job];
        const PathOrder o = path_order(t, jb.width, a.group_lg);
        const uint32_t q = k - t.pix0, off = position_to_pixel(o, o.g, q), p = t.p0 + off;
        float4* acc = jb.accum + p;
        const float4 s = *acc;
        V3 sum = v3(s.x, s.y, s.z);
        uint32_t smp = t.s0;
        auto add = [&](float4 r) {
            sum = sum + v3(r);
            if (jb.samples && smp < jb.samples_cap) jb.samples[size_t(p) * jb.samples_cap + smp] = make_float4(r.x, r.y, r.z, 0.f);
            ++smp;
        };
        for (uint32_t sec = 0; sec <= o.full; ++sec) {
            const bool last = sec == o.full;
            const uint32_t m = last ? o.rest : o.m;
            if (m == 0u) break;
            const uint32_t at = last ? pixel_to_position(o, band_rows(m), off) : q;
            const float4* r = a.result + t.slot0 + sec * (o.pixels * o.m) + at * m;
            uint32_t j = 0;
            for (; j + 8u <= m; j += 8u) {
                float4 v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = r[j + e];
#pragma unroll
                for (int e = 0; e < 8; ++e) add(v[e]);
            }
            for (; j < m; ++j) add(r[j]);
        }
        *acc = make_float4(sum.x, sum.y, sum.z, 0.f);
    }
}

}  // namespace dev

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
namespace {

#define WF_TRY(expr)                                        \
    do {                                                    \
        hipError_t e_ = (expr);                             \
        if (e_ != hipSuccess) return hip_fail(e_, #expr);   \
    } while (0)

struct PlanJob {
    uint32_t pixels;
    uint32_t s_begin, s_end;
};

// Tiles of at most `cap` slots, packed in order into chunks of at most `cap` slots.
void make_plan(const std::vector<PlanJob>& jobs, uint32_t cap, std::vector<WfTile>& tiles,
               std::vector<WfChunk>& chunks) {
    tiles.clear();
    chunks.clear();
    std::vector<WfTile> raw;
    for (uint32_t j = 0; j < jobs.size(); ++j) {
        const PlanJob& pj = jobs[j];
        if (pj.s_end <= pj.s_begin || pj.pixels == 0) continue;
        if (pj.pixels >= cap) {
            for (uint32_t s = pj.s_begin; s < pj.s_end; ++s)
                for (uint32_t p0 = 0; p0 < pj.pixels; p0 += cap)
                    raw.push_back(WfTile{j, p0, std::min(pj.pixels, p0 + cap), s, s + 1, 0, 0, 0});
        } else {
            const uint32_t k = cap / pj.pixels;
            for (uint32_t s = pj.s_begin; s < pj.s_end; s += k)
                raw.push_back(WfTile{j, 0, pj.pixels, s, std::min(pj.s_end, s + k), 0, 0, 0});
        }
    }
    WfChunk cur{0, 0, 0, 0};
    for (WfTile t : raw) {
        const uint32_t n = (t.p1 - t.p0) * (t.s1 - t.s0);
        // A pixel may appear in only one tile of a chunk: resolve adds each tile's
        // samples with one thread per pixel.
        bool overlap = false;
        for (uint32_t k = cur.tile0; k < tiles.size() && !overlap; ++k)
            overlap = tiles[k].job == t.job && tiles[k].p0 < t.p1 && t.p0 < tiles[k].p1;
        if (cur.ntiles && (cur.paths + n > cap || overlap)) {
            chunks.push_back(cur);
            cur = WfChunk{uint32_t(tiles.size()), 0, 0, 0};
        }
        t.slot0 = cur.paths;
        t.pix0 = cur.pixels;
        tiles.push_back(t);
        cur.ntiles++;
        cur.paths += n;
        cur.pixels += t.p1 - t.p0;
    }
    if (cur.ntiles) chunks.push_back(cur);
}

// Resident workgroups of a kernel on the whole device, and the device's compute units.
int persistent_blocks(const void* kernel, uint32_t blocks_per_cu, int device, int* compute_units) {
    if (hipDeviceGetAttribute(compute_units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        *compute_units = 128;
    int occ = 0;
    if (!blocks_per_cu && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, kBlock, 0) != hipSuccess || occ <= 0))
        occ = 8;
    const uint32_t per = blocks_per_cu ? blocks_per_cu : uint32_t(occ);
    return int(std::max<uint32_t>(1, per * uint32_t(*compute_units)));
}

// Queues of at least `capacity` slots and a spill area of at least `spill_ints`. Each grows by
// itself: calls of few paths over a deep scene and of many over a shallow one leave each other's.
int ensure_state(WavefrontState& w, uint32_t capacity, size_t spill_ints, hipStream_t stream) {
    WfArgs& a = w.args;
    if (!w.ctr) {
        WF_TRY(device_alloc(reinterpret_cast<void**>(&w.ctr), kNumCounters * sizeof(uint32_t)));
        a.ctr = w.ctr;
        WF_TRY(fill_wait(w.ctr, 0, kNumCounters * sizeof(uint32_t), stream));
    }
    if (w.spill_ints < spill_ints) {
        if (w.spill) (void)hipFree(w.spill);
        a.spill = w.spill = nullptr;
        w.spill_ints = 0;
        WF_TRY(device_alloc(reinterpret_cast<void**>(&w.spill), spill_ints * sizeof(int)));
        a.spill = w.spill;
        w.spill_ints = spill_ints;
    }
    if (w.capacity < capacity) {
        if (w.mem) (void)hipFree(w.mem);
        w.mem = nullptr;
        w.capacity = 0;
        const size_t C = capacity;
        WF_TRY(device_alloc(&w.mem, kSlotBytes * C));
        w.capacity = capacity;
        char* p = static_cast<char*>(w.mem);
        auto take = [&](size_t bytes) {
            void* r = p;
            p += bytes;
            return r;
        };
        for (int k = 0; k < 2; ++k) {
            a.qa[k] = static_cast<float4*>(take(16 * C));
            a.qb[k] = static_cast<float4*>(take(16 * C));
            a.qc[k] = static_cast<float4*>(take(16 * C));
        }
        a.se = static_cast<float4*>(take(16 * C));
        a.sf = static_cast<float4*>(take(16 * C));
        a.sg = static_cast<float4*>(take(16 * C));
        a.result = static_cast<float4*>(take(16 * C));
        a.hits = static_cast<uint32_t*>(take(4 * C));
        a.sj = static_cast<uint32_t*>(take(4 * C));
    }
    return PRT_OK;
}

void free_state(WavefrontState& w) {
    void* ptrs[] = {w.mem, w.spill, w.ctr, w.d_plan};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    if (w.exec) (void)hipGraphExecDestroy(w.exec);
    if (w.e0) (void)hipEventDestroy(w.e0);
    if (w.e1) (void)hipEventDestroy(w.e1);
    w = WavefrontState();
}

struct RunStats {
    unsigned long long c[kCntNum];
    double ms;
    double kernel_ms[3];  // profile: extend, shade, shadow
    uint32_t launches[3];
};

// Whether a chunk's camera rays are traced as packets. A packet visits what any of its rays
// would, one dependent step after another, so a launch lasts at least one packet: 0.012 ms
// over 36 triangles, 0.1 over 20,000, 0.3 over 1M, 0.65 over 2.8M, about the triangles'
// square root (their number across an image); from there on it is faster per ray. Per-lane
// rays take 0.09 ms and 0.065 ns each. Measured, packets against rays, in us: 1M triangles,
// 640 x 480 x 1 329 / 148, 1920 x 1080 x 2 340 / 370, x 16 1058 / 1833; 20,000 triangles,
// 125 x 93 x 8 179 / 53, 640 x 480 x 4 82 / 93; 2.8M triangles, 1280 x 720 x 6 720 / 576,
// 640 x 480 x 64 1405 / 1678; 36 triangles, 64 x 64 x 1 12 / 15.
bool use_packets(uint32_t paths, uint32_t triangles) { return double(paths) >= 4096.0 * std::sqrt(double(triangles)); }

// Launches one chunk's kernels on `stream`: setup, generate, the camera rays' extension
// (as packets or per lane), then per iteration shade and one launch that traces its shadow rays
// and the next iteration's extension rays, then resolve. With `ev` (4 per iteration) those
// two are launched one after the other, and each extend / shade / shadow part is bracketed
// by events.
template <bool COUNT, bool ONE_SCENE>
void launch_chunk(const WfArgs& a, hipStream_t stream, uint32_t max_depth, int pblocks, int gblocks, int sblocks,
                  bool packets, hipEvent_t* ev) {
    auto mark = [&](uint32_t k) {
        if (ev) (void)hipEventRecord(ev[k], stream);
    };
    auto trace = [&](uint32_t it, uint32_t parts) {
        hipLaunchKernelGGL((dev::wf_trace<COUNT, ONE_SCENE>), dim3(pblocks), dim3(kBlock), 0, stream, a, it, parts);
    };
    hipLaunchKernelGGL(dev::wf_setup, dim3((2 * max_depth * kSpread + 255) / 256), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(dev::wf_generate, dim3(gblocks), dim3(256), 0, stream, a);
    for (uint32_t it = 0; it < max_depth; ++it) {
        mark(4 * it);
        if (it == 0 && packets)
            hipLaunchKernelGGL((dev::wf_extend_packet<COUNT, ONE_SCENE>), dim3(pblocks), dim3(kBlock), 0, stream, a);
        else if (it == 0 || ev)
            trace(it, dev::kTraceExtend);
        mark(4 * it + 1);
        hipLaunchKernelGGL((dev::wf_shade<COUNT, ONE_SCENE>), dim3(sblocks), dim3(kShadeBlock), 0, stream, a, it);
        mark(4 * it + 2);
        // The last iteration leaves no extension rays.
        trace(it + 1, ev || it + 1 == max_depth ? dev::kTraceShadow : dev::kTraceShadow | dev::kTraceExtend);
        mark(4 * it + 3);
    }
    hipLaunchKernelGGL(dev::wf_resolve, dim3(gblocks), dim3(256), 0, stream, a);
}

void launch_chunk_any(bool count, bool one_scene, const WfArgs& a, hipStream_t stream, uint32_t max_depth,
                      int pblocks, int gblocks, int sblocks, bool packets, hipEvent_t* ev) {
    auto go = count ? one_scene ? launch_chunk<true, true> : launch_chunk<true, false>
                    : one_scene ? launch_chunk<false, true> : launch_chunk<false, false>;
    go(a, stream, max_depth, pblocks, gblocks, sblocks, packets, ev);
}

// The captured launch sequence for `k`: the state's own when it was made for the same.
int chunk_graph(WavefrontState& w, hipStream_t stream, const LaunchKey& k) {
    if (w.exec && std::memcmp(&w.key, &k, sizeof k) == 0) return PRT_OK;
    if (w.exec) (void)hipGraphExecDestroy(w.exec);
    w.exec = nullptr;
    hipGraph_t graph = nullptr;
    WF_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    launch_chunk_any(k.count, k.args.one_scene != 0, k.args, stream, k.max_depth, k.pblocks, k.gblocks, k.sblocks,
                     k.packets, nullptr);
    hipError_t e = hipStreamEndCapture(stream, &graph);
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    e = hipGraphInstantiate(&w.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
        w.exec = nullptr;
        return hip_fail(e, "hipGraphInstantiate");
    }
    std::memcpy(&w.key, &k, sizeof k);
    return PRT_OK;
}

// Profile mode: every chunk launched directly, each extend / shade / shadow launch
// timed with events; per-kernel device time summed into rs.
int run_profiled(const WfArgs& a, hipStream_t stream, size_t nchunks, uint32_t max_depth, int pblocks, int gblocks,
                 int sblocks, bool packets, bool count, bool one_scene, RunStats* rs) {
    std::vector<hipEvent_t> ev(4 * max_depth, nullptr);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = PRT_OK;
    double total = 0.0;
    double kms[3] = {0, 0, 0};
    hipError_t e = hipSuccess;
    for (auto& x : ev)
        if (e == hipSuccess) e = hipEventCreate(&x);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    for (size_t c = 0; c < nchunks && e == hipSuccess; ++c) {
        e = hipEventRecord(e0, stream);
        if (e != hipSuccess) break;
        launch_chunk_any(count, one_scene, a, stream, max_depth, pblocks, gblocks, sblocks, packets, ev.data());
        e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(e1, stream);
        if (e == hipSuccess) e = hipEventSynchronize(e1);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
        total += ms;
        for (uint32_t it = 0; it < max_depth && e == hipSuccess; ++it)
            for (int k = 0; k < 3 && e == hipSuccess; ++k) {
                e = hipEventElapsedTime(&ms, ev[4 * it + k], ev[4 * it + k + 1]);
                kms[k] += ms;
            }
    }
    if (e != hipSuccess) rc = hip_fail(e, "profiled wavefront launch");
    for (auto& x : ev)
        if (x) (void)hipEventDestroy(x);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (rc == PRT_OK && rs) {
        rs->ms = total;
        for (int k = 0; k < 3; ++k) {
            rs->kernel_ms[k] = kms[k];
            rs->launches[k] = uint32_t(nchunks * max_depth);
        }
    }
    return rc;
}

// Renders every job of the plan on `stream`. Returns PRT_OK or an error.
// entries: traversal stack entries that the scenes need (stack_entries).
// group_side: camera-path block side g for wf_generate (1, 2, 4, 8; 0 = choose per section).
// stats: device counters that the rays are added to (else rs->c receives them).
int run_wavefront(WavefrontState& w, int device, hipStream_t stream, uint32_t entries, const std::vector<WfJob>& jobs,
                  const std::vector<PlanJob>& pjobs, uint32_t max_depth, uint32_t capacity, uint32_t blocks_per_cu,
                  uint32_t group_side, bool count, RunStats* rs, bool profile = false, uint32_t* vertices = nullptr,
                  uint32_t vertex_cap = 0, unsigned long long* stats = nullptr) {
    if (max_depth == 0 || max_depth > uint32_t(kMaxIter)) return fail(PRT_ERR_INVALID_ARG, "max_depth out of range");
    uint32_t group_lg = dev::kNone;
    if (group_side != 0) {
        if (group_side != 1 && group_side != 2 && group_side != 4 && group_side != 8)
            return fail(PRT_ERR_INVALID_ARG, "wavefront group side must be 0, 1, 2, 4 or 8");
        group_lg = group_side == 1 ? 0u : group_side == 2 ? 1u : group_side == 4 ? 2u : 3u;
    }
    // Queue entries pack pixel | job << 24.
    if (jobs.size() > 256) return fail(PRT_ERR_LIMIT, "more than 256 jobs in one batch");
    for (const PlanJob& pj : pjobs)
        if (pj.pixels > (1u << 24)) return fail(PRT_ERR_LIMIT, "a view with more than 2^24 pixels");
    std::vector<WfTile> tiles;
    std::vector<WfChunk> chunks;
    make_plan(pjobs, capacity, tiles, chunks);
    if (chunks.empty()) return PRT_OK;
    uint32_t need = 0;
    for (auto& c : chunks) need = std::max(need, c.paths);
    bool one_scene = true;
    for (const WfJob& j : jobs)
        one_scene = one_scene && j.sc.nodes == jobs[0].sc.nodes && j.sc.tris == jobs[0].sc.tris;
    const void* ktrace = count ? (one_scene ? reinterpret_cast<const void*>(dev::wf_trace<true, true>)
                                          : reinterpret_cast<const void*>(dev::wf_trace<true, false>))
                             : (one_scene ? reinterpret_cast<const void*>(dev::wf_trace<false, true>)
                                          : reinterpret_cast<const void*>(dev::wf_trace<false, false>));
    int cus = 0;
    const int resident = persistent_blocks(ktrace, blocks_per_cu, device, &cus);
    const int pblocks = int(trace_waves(uint32_t(resident), (need + kBatch - 1) / kBatch));
    const size_t rows = entries > uint32_t(kStackLdsQueue) ? entries - kStackLdsQueue : 0;
    int rc = ensure_state(w, need, rows * size_t(pblocks) * kBlock, stream);
    if (rc != PRT_OK) return rc;
    // The plan in one upload. (Every part is a multiple of 16 bytes.)
    const size_t at_tiles = jobs.size() * sizeof(WfJob), at_chunks = at_tiles + tiles.size() * sizeof(WfTile);
    const size_t plan_bytes = at_chunks + chunks.size() * sizeof(WfChunk);
    static_assert(sizeof(WfJob) % 8 == 0 && sizeof(WfTile) % 16 == 0 && sizeof(WfChunk) % 16 == 0, "plan alignment");
    w.h_plan.resize(plan_bytes);
    std::memcpy(w.h_plan.data(), jobs.data(), at_tiles);
    std::memcpy(w.h_plan.data() + at_tiles, tiles.data(), at_chunks - at_tiles);
    std::memcpy(w.h_plan.data() + at_chunks, chunks.data(), plan_bytes - at_chunks);
    if (w.cap_plan < plan_bytes) {
        if (w.d_plan) (void)hipFree(w.d_plan);
        w.d_plan = nullptr;
        w.cap_plan = 0;
        WF_TRY(device_alloc(reinterpret_cast<void**>(&w.d_plan), std::max<size_t>(plan_bytes, 4096)));
        w.cap_plan = std::max<size_t>(plan_bytes, 4096);
    }
    WF_TRY(hipMemcpyAsync(w.d_plan, w.h_plan.data(), plan_bytes, hipMemcpyHostToDevice, stream));
    WF_TRY(hipMemsetAsync(w.ctr, 0, kQueue * sizeof(uint32_t), stream));  // wf_setup clears the rest
    WfArgs a = w.args;
    a.jobs = reinterpret_cast<const WfJob*>(w.d_plan);
    a.tiles = reinterpret_cast<const WfTile*>(w.d_plan + at_tiles);
    a.chunks = reinterpret_cast<const WfChunk*>(w.d_plan + at_chunks);
    a.stats = stats ? stats : reinterpret_cast<unsigned long long*>(w.ctr + kStats);
    a.max_depth = max_depth;
    a.group_lg = group_lg;
    a.one_scene = one_scene ? 1u : 0u;
    a.spill_stride = uint32_t(pblocks) * kBlock;
    a.vertices = vertices;
    a.vertex_cap = vertex_cap;
    a.vertex_stride = size_t(pjobs[0].pixels) * vertex_cap;

    const int gblocks = cus * 8;
    const int sblocks = cus * kShadeGridWaves * 64 / kShadeBlock;

    uint32_t triangles = 0;
    for (const WfJob& j : jobs) triangles = std::max(triangles, j.sc.num_records);
    const bool packets = use_packets(need, triangles);

    // The counters of a run that adds them to its own (a batch); a run that counts nothing
    // leaves them 0.
    auto read_stats = [&]() -> int {
        std::memset(rs->c, 0, sizeof rs->c);
        if (count && !stats) WF_TRY(copy_wait(rs->c, a.stats, sizeof rs->c, hipMemcpyDeviceToHost, stream));
        return PRT_OK;
    };
    if (profile) {
        rc = run_profiled(a, stream, chunks.size(), max_depth, pblocks, gblocks, sblocks, packets, count, one_scene,
                          rs);
        return rc == PRT_OK && rs ? read_stats() : rc;
    }
    LaunchKey key;
    std::memset(&key, 0, sizeof key);  // padding too: keys are compared as bytes
    std::memcpy(&key.args, &a, sizeof a);
    key.max_depth = max_depth;
    key.pblocks = pblocks;
    key.gblocks = gblocks;
    key.sblocks = sblocks;
    key.packets = packets;
    key.count = count;
    rc = chunk_graph(w, stream, key);
    if (rc != PRT_OK) return rc;
    if (!w.e0) WF_TRY(hipEventCreate(&w.e0));
    if (!w.e1) WF_TRY(hipEventCreate(&w.e1));
    hipError_t e = hipEventRecord(w.e0, stream);
    for (size_t c = 0; c < chunks.size() && e == hipSuccess; ++c) e = hipGraphLaunch(w.exec, stream);
    if (e == hipSuccess) e = hipEventRecord(w.e1, stream);
    if (e == hipSuccess) e = hipEventSynchronize(w.e1);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, w.e0, w.e1);
    if (e != hipSuccess) return hip_fail(e, "wavefront launch");
    if (rs) {
        rs->ms = ms;
        for (int k = 0; k < 3; ++k) {
            rs->kernel_ms[k] = 0.0;
            rs->launches[k] = 0;
        }
        return read_stats();
    }
    return PRT_OK;
}

// The most path slots worth holding: a quarter of the device's free memory (an
// MI355X's 288 GB holds a whole 1080p x 128-spp frame, 265M paths, in one chunk),
// at most 2^28. Fewer, larger chunks leave fewer nearly empty late iterations. What the
// state already holds counts as free.
uint64_t max_slots(const WavefrontState& w) {
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) free_b = size_t(8) << 30;
    return std::max<uint64_t>(1u << 20, std::min<uint64_t>(1ull << 28, (free_b + kSlotBytes * w.capacity) / 4 / kSlotBytes));
}

uint32_t default_capacity(const WavefrontState& w, uint64_t total_paths) {
    if (w.mem && w.capacity >= total_paths && total_paths > 0) return uint32_t(total_paths);
    return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(max_slots(w), total_paths)));
}

// What a call without a renderer needs: queues, its views' accumulators and images, a
// stream. One call uses it at a time, and waits for its stream before it gives it back.
struct CallSpace {
    int device = -1;
    WavefrontState w;
    void* accum = nullptr;
    size_t accum_bytes = 0;
    void* rgb = nullptr;
    size_t rgb_bytes = 0;
    hipStream_t stream = nullptr;
    size_t bytes() const {
        return kSlotBytes * w.capacity + w.spill_ints * sizeof(int) + w.cap_plan + accum_bytes + rgb_bytes;
    }
};

void free_space(CallSpace* c) {
    int prev = 0;
    (void)hipGetDevice(&prev);
    (void)hipSetDevice(c->device);
    free_state(c->w);
    if (c->accum) (void)hipFree(c->accum);
    if (c->rgb) (void)hipFree(c->rgb);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    (void)hipSetDevice(prev);
    delete c;
}

std::mutex g_space_mutex;
constexpr int kSpaceDevices = 64;
CallSpace* g_idle_space[kSpaceDevices] = {};  // one per device (none kept beyond these)

// Takes the device's idle space or makes a new one; the destructor gives it back, or frees
// it when it holds too much to stay (may_stay_idle), another one is there, or the call has
// failed. (Allocating and freeing the queues on every call: 12 views, 42M paths,
// 7 GB took 278 ms a call, of which 10 ms were kernels; once a process has used as much
// memory as the device has, the driver clears every page that it hands out again.)
class CallSpaceLease {
public:
    int take(int device) {
        {
            std::lock_guard<std::mutex> g(g_space_mutex);
            if (device < kSpaceDevices) std::swap(c_, g_idle_space[device]);
        }
        if (c_) return PRT_OK;
        c_ = new CallSpace;
        c_->device = device;
        WF_TRY(hipStreamCreateWithFlags(&c_->stream, hipStreamNonBlocking));
        return PRT_OK;
    }
    void done() { ok_ = true; }
    CallSpace* operator->() const { return c_; }
    ~CallSpaceLease() {
        if (!c_) return;
        size_t free_b = 0, total_b = 0;
        if (ok_ && scenes_on_devices() && hipMemGetInfo(&free_b, &total_b) == hipSuccess &&
            may_stay_idle(c_->bytes(), free_b, total_b)) {
            std::lock_guard<std::mutex> g(g_space_mutex);
            if (c_->device < kSpaceDevices && !g_idle_space[c_->device]) {
                g_idle_space[c_->device] = c_;
                return;
            }
        }
        if (c_->stream) (void)hipStreamSynchronize(c_->stream);
        free_space(c_);
    }

private:
    CallSpace* c_ = nullptr;
    bool ok_ = false;
};

}  // namespace

void release_idle_queues() {
    CallSpace* all[kSpaceDevices] = {};
    {
        std::lock_guard<std::mutex> g(g_space_mutex);
        for (int k = 0; k < kSpaceDevices; ++k) std::swap(all[k], g_idle_space[k]);
    }
    for (CallSpace* c : all)
        if (c) free_space(c);
}

int render_wavefront(prt_renderer* r, uint32_t n) {
    PRT_TRY_BEGIN
    if (!r->wf) r->wf = new WavefrontState();
    WfJob j;
    j.sc = r->sc;
    j.cam = cam_args(r->cam);
    j.path = PathArgs{r->cfg.seed, r->cfg.view_id, r->cfg.max_depth, r->cfg.rr_start};
    j.width = r->w;
    j.height = r->h;
    j.accum = r->accum;
    j.samples = r->samples;
    j.samples_cap = r->samples ? r->spp : 0;
    std::vector<WfJob> jobs = {j};
    std::vector<PlanJob> pj = {PlanJob{r->w * r->h, r->samples_done, r->samples_done + n}};
    const uint64_t total = uint64_t(r->w) * r->h * n;
    const uint32_t cap = r->cfg.wavefront_queue ? r->cfg.wavefront_queue : default_capacity(*r->wf, total);
    RunStats rs;
    int rc = run_wavefront(*r->wf, r->cfg.device, r->stream, stack_entries(r->scene), jobs, pj, r->cfg.max_depth, cap,
                           r->cfg.wavefront_blocks_per_cu, r->cfg.wavefront_group, r->cfg.count_rays != 0, &rs,
                           r->cfg.profile_kernels != 0, r->vertices, r->spp, r->counters);
    if (rc != PRT_OK) return rc;
    r->last_ms = rs.ms;
    for (int k = 0; k < 3; ++k) {
        r->kernel_ms[k] = rs.kernel_ms[k];
        r->kernel_launches[k] = rs.launches[k];
    }
    r->samples_done += n;
    r->samples_total += total;
    return PRT_OK;
    PRT_TRY_END
}

int wavefront_samples(prt_renderer* r, uint32_t spp, float4* accum, float4* samples, uint32_t* vertices) {
    PRT_TRY_BEGIN
    // A megakernel renderer does not keep the queues of a one-off forward pass.
    CallSpaceLease space;
    WavefrontState* w = r->wf;
    if (!w && r->cfg.integrator == PRT_INTEGRATOR_WAVEFRONT) w = r->wf = new WavefrontState();
    if (!w) {
        const int rc = space.take(r->cfg.device);
        if (rc != PRT_OK) return rc;
        w = &space->w;
    }
    WfJob j;
    j.sc = r->sc;
    j.cam = cam_args(r->cam);
    j.path = PathArgs{r->cfg.seed, r->cfg.view_id, r->cfg.max_depth, r->cfg.rr_start};
    j.width = r->w;
    j.height = r->h;
    j.accum = accum;
    j.samples = samples;
    j.samples_cap = spp;
    std::vector<WfJob> jobs = {j};
    std::vector<PlanJob> pj = {PlanJob{r->w * r->h, 0, spp}};
    const uint64_t total = uint64_t(r->w) * r->h * spp;
    const uint32_t cap = r->cfg.wavefront_queue ? r->cfg.wavefront_queue : default_capacity(*w, total);
    RunStats rs;
    // On the renderer's stream, and waited for: the queues are idle when the call returns.
    const int rc = run_wavefront(*w, r->cfg.device, r->stream, stack_entries(r->scene), jobs, pj, r->cfg.max_depth, cap,
                                 r->cfg.wavefront_blocks_per_cu, r->cfg.wavefront_group, false, &rs, false, vertices,
                                 spp);
    if (rc == PRT_OK) space.done();
    else (void)hipStreamSynchronize(r->stream);
    return rc;
    PRT_TRY_END
}

void release_wavefront(prt_renderer* r) {
    if (!r->wf) return;
    free_state(*r->wf);
    delete r->wf;
    r->wf = nullptr;
}

namespace {

// Device memory for a batch's images (CallSpace::rgb) at most.
constexpr size_t kImageBytes = size_t(256) << 20;

struct BatchCtx {
    std::vector<WfJob> jobs;
    std::vector<PlanJob> pjobs;
    std::vector<size_t> pixel0;  // each view's first pixel in the accumulators
    size_t pixels = 0;
    uint32_t max_depth = 0;
    uint32_t entries = 0;  // traversal stack entries that the scenes need
    uint64_t total = 0;
};

// Checks the jobs, uploads their scenes and clears accumulators for all of them.
int batch_prepare(prt_job* jobs, uint32_t n, const prt_render_config& c, BatchCtx& b, CallSpace& space) {
    hipStream_t stream = space.stream;
    if (!jobs || n == 0) return fail(PRT_ERR_INVALID_ARG, "no jobs");
    b.max_depth = c.max_depth;
    for (uint32_t i = 0; i < n; ++i) {
        const prt_job& jb = jobs[i];
        if (!jb.scene) return fail(PRT_ERR_INVALID_ARG, "job without a scene");
        if (jb.scene->lights.empty()) return fail(PRT_ERR_NO_EMITTERS, "job scene has no emitters");
        if (jb.camera.xpixels <= 0 || jb.camera.ypixels <= 0) return fail(PRT_ERR_INVALID_ARG, "job camera size");
        if (jb.spp == 0) return fail(PRT_ERR_INVALID_ARG, "job with zero samples per pixel");
        if (uint64_t(jb.camera.xpixels) * uint64_t(jb.camera.ypixels) > (1u << 24))
            return fail(PRT_ERR_LIMIT, "a view with more than 2^24 pixels");
        WfJob w;
        int rc = device_scene(jb.scene, c.device, w.sc, stream);
        if (rc != PRT_OK) return rc;
        b.entries = std::max(b.entries, stack_entries(jb.scene));
        w.cam = cam_args(jb.camera);
        w.path = PathArgs{c.seed, jb.view_id, c.max_depth, c.rr_start};
        w.width = uint32_t(jb.camera.xpixels);
        w.height = uint32_t(jb.camera.ypixels);
        const size_t px = size_t(w.width) * w.height;
        w.accum = nullptr;
        b.pixel0.push_back(b.pixels);
        b.pixels += px;
        w.samples = nullptr;
        w.samples_cap = 0;
        b.jobs.push_back(w);
        b.pjobs.push_back(PlanJob{uint32_t(px), 0, jb.spp});
        b.total += uint64_t(px) * jb.spp;
    }
    const int rc = scratch_for(space.accum, space.accum_bytes, b.pixels * sizeof(float4));
    if (rc != PRT_OK) return rc;
    for (uint32_t i = 0; i < n; ++i) b.jobs[i].accum = static_cast<float4*>(space.accum) + b.pixel0[i];
    WF_TRY(hipMemsetAsync(space.accum, 0, b.pixels * sizeof(float4), stream));
    return PRT_OK;
}

}  // namespace

}  // namespace prt

using namespace prt;

extern "C" int prt_render_batch(prt_job* jobs, uint32_t n, const prt_render_config* cfg, const prt_tune* tune,
                                prt_stats* stats) {
    clear_error();
    if (tune && tune->block_size != 0 && tune->block_size != uint32_t(kBlock))
        return fail(PRT_ERR_INVALID_ARG, "prt_tune.block_size: the traversal kernels are built for 64 threads");
    prt_render_config c;
    if (cfg) c = *cfg;
    else prt_render_config_default(&c);
    int rc = set_device(c.device);
    if (rc != PRT_OK) return rc;
    PRT_TRY_BEGIN
    BatchCtx b;
    CallSpaceLease space;
    rc = space.take(c.device);
    if (rc == PRT_OK) rc = batch_prepare(jobs, n, c, b, *space.operator->());
    if (rc != PRT_OK) return rc;
    hipStream_t s = space->stream;
    const uint32_t cap = tune && tune->queue_slots ? tune->queue_slots : default_capacity(space->w, b.total);
    RunStats rs;
    rc = run_wavefront(space->w, c.device, s, b.entries, b.jobs, b.pjobs, c.max_depth, cap, tune ? tune->blocks_per_cu : 0,
                       tune ? tune->group_side : c.wavefront_group, c.count_rays != 0, &rs);
    // The images' means, then their copies in one run, as many as fit kImageBytes (an image always
    // does) at a time: the accumulators of a large batch leave little room.
    static_assert((size_t(1) << 24) * 3 * sizeof(float) <= kImageBytes, "the largest view's image");
    size_t images = 0, at = 0;
    for (uint32_t i = 0; i < n; ++i)
        if (jobs[i].out_rgb) images += size_t(b.jobs[i].width) * b.jobs[i].height * 3 * sizeof(float);
    if (rc == PRT_OK && images) rc = scratch_for(space->rgb, space->rgb_bytes, std::min(images, kImageBytes));
    std::vector<CopyOut> out;
    hipError_t e = hipSuccess;
    for (uint32_t i = 0; i < n && rc == PRT_OK && e == hipSuccess; ++i) {
        if (!jobs[i].out_rgb) continue;
        const size_t px = size_t(b.jobs[i].width) * b.jobs[i].height, bytes = px * 3 * sizeof(float);
        if (at + bytes > space->rgb_bytes) {
            e = copy_out(out.data(), out.size(), c.device, s);
            out.clear();
            at = 0;
        }
        float* rgb = reinterpret_cast<float*>(static_cast<char*>(space->rgb) + at);
        if (e == hipSuccess) e = launch_mean(b.jobs[i].accum, uint32_t(px), jobs[i].spp, rgb, s);
        out.push_back(CopyOut{jobs[i].out_rgb, rgb, bytes});
        at += bytes;
    }
    if (rc == PRT_OK && e == hipSuccess) e = copy_out(out.data(), out.size(), c.device, s);
    if (e != hipSuccess) rc = hip_fail(e, "batch readback");
    if (rc == PRT_OK && stats) {
        stats->primary_rays = rs.c[kCntPrimary];
        stats->extension_rays = rs.c[kCntExtension];
        stats->shadow_rays = rs.c[kCntShadow];
        stats->nodes_visited = rs.c[kCntNodes];
        stats->tris_tested = rs.c[kCntTris];
        stats->hits = rs.c[kCntHits];
        stats->samples = b.total;
        stats->last_render_ms = rs.ms;
    }
    if (rc == PRT_OK) space.done();
    return rc;
    PRT_TRY_END
}

extern "C" int prt_autotune(prt_job* jobs, uint32_t n, const prt_render_config* cfg, prt_tune* best,
                            double* best_ms) {
    clear_error();
    if (!best) return fail(PRT_ERR_INVALID_ARG, "null argument");
    prt_render_config c;
    if (cfg) c = *cfg;
    else prt_render_config_default(&c);
    c.count_rays = 0;
    int rc = set_device(c.device);
    if (rc != PRT_OK) return rc;
    PRT_TRY_BEGIN
    // Trial workload: every job at its own samples per pixel and width, but with only
    // kTrialRows rows (the camera's vertical field kept, so the rows spread over the
    // whole view): the camera-path grouping, whose candidates depend on the sample
    // count and the row count, then behaves as in the full run, at a small fraction
    // of its paths.
    constexpr int32_t kTrialRows = 8;
    std::vector<prt_job> trial(jobs, jobs + n);
    uint64_t paths = 0;
    for (auto& t : trial) {
        t.camera.ypixels = std::min<int32_t>(t.camera.ypixels, kTrialRows);
        t.out_rgb = nullptr;
        paths += uint64_t(t.camera.xpixels) * t.camera.ypixels * t.spp;
    }
    BatchCtx b;
    CallSpaceLease space;
    rc = space.take(c.device);
    if (rc == PRT_OK) rc = batch_prepare(trial.data(), n, c, b, *space.operator->());
    if (rc != PRT_OK) return rc;
    hipStream_t s = space->stream;
    WavefrontState& w = space->w;
    uint64_t full = 0;
    for (uint32_t i = 0; i < n; ++i) full += uint64_t(jobs[i].camera.xpixels) * jobs[i].camera.ypixels * jobs[i].spp;
    double bms = 1e30;
    prt_tune bt{};
    // Every candidate is timed (best of two) on the trial cut into as many chunks as
    // the full run at that chunk size would take. Occupancy candidates stay near full
    // occupancy: wf_trace fits 32 one-wave workgroups per CU (8 per SIMD), 28 with several
    // scenes. Chunk counts: the fewest that fit the path slots (larger chunks were faster
    // at every size measured on one view, since every chunk ends in nearly empty
    // iterations), and twice and four times as many.
    const uint64_t limit = max_slots(w);
    const uint32_t full_cap = uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(full, limit)));
    // The trial's path slots for a full-run chunk size: the trial is cut into as many
    // chunks as the full run would take, so its queues drain like the full run's.
    auto trial_cap_for = [&](uint32_t cap) {
        const uint64_t chunks = (full + cap - 1) / cap;
        return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(paths, (paths + chunks - 1) / chunks)));
    };
    auto time_trial = [&](const prt_tune& t) -> double {
        double best_t = 1e30;
        for (int rep = 0; rep < 2 && rc == PRT_OK; ++rep) {  // best of two
            RunStats rs;
            rc = run_wavefront(w, c.device, s, b.entries, b.jobs, b.pjobs, c.max_depth, trial_cap_for(t.queue_slots),
                               t.blocks_per_cu, t.group_side, false, &rs);
            best_t = std::min(best_t, rs.ms);
        }
        return best_t;
    };
    // A candidate replaces the best so far only when it is at least 2% faster on the
    // trial: smaller differences are within the trial's run-to-run spread and need
    // not carry over to the full run.
    auto consider = [&](const prt_tune& t) {
        const double ms = time_trial(t);
        if (rc == PRT_OK && (bms >= 1e30 || ms < 0.98 * bms)) {
            bms = ms;
            bt = t;
        }
    };
    // Coordinate search from the defaults (fewest chunks, groups chosen per section):
    // occupancy, then the camera-path grouping, then the chunk count.
    bt = prt_tune{full_cap, 0, kBlock, 0};
    consider(bt);
    for (uint32_t bpc : {20u, 24u, 28u}) {
        prt_tune t = bt;
        t.blocks_per_cu = bpc;
        if (rc == PRT_OK) consider(t);
    }
    const prt_tune occ = bt;
    for (uint32_t g : {1u, 2u, 4u, 8u}) {
        prt_tune t = occ;
        t.group_side = g;
        if (rc == PRT_OK) consider(t);
    }
    const prt_tune grp = bt;
    for (uint32_t div : {2u, 4u}) {
        prt_tune t = grp;
        t.queue_slots = std::max<uint32_t>(1u << 16, full_cap / div);
        if (t.queue_slots < full_cap && rc == PRT_OK) consider(t);
    }
    if (rc != PRT_OK) return rc;
    space.done();
    *best = bt;
    if (best_ms) *best_ms = bms;
    return PRT_OK;
    PRT_TRY_END
}

