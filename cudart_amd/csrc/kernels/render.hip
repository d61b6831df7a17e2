// Megakernel path tracer, primary-hit kernel and output kernels for gfx950.
//
// A wave64 workgroup renders blocks of pixels, one after another. With `nspp` samples per
// pixel in the launch, the lanes that share a pixel take a sample each, and one of them adds
// the results to the running sum in sample order, the order
// SequentialRenderer::renderOneSamplePerPixel (src/renderer/sequential_renderer.cu:91-116)
// and renderKernel (src/renderer/parallel_renderer.cu:318-342) accumulate in.
#include "path.hpp"

#include <type_traits>

namespace prt {
namespace dev {

template <bool COUNT>
__device__ __forceinline__ void flush_counts(unsigned long long* out, const Counts& c) {
    // Wave-level sums, one atomic per wave and slot.
    unsigned long long v[6] = {c.primary, c.extension, c.shadow, c.nodes, c.tris, c.hits};
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        unsigned long long x = v[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if ((threadIdx.x & 63) == 0 && x) atomicAdd(out + k, x);
    }
}

constexpr uint32_t kNoBlock = 0xFFFFFFFFu;

// The blocks of pixels, handed out to the workgroups of a launch. XCD x has a band of
// consecutive blocks (its L2 then sees one part of the image), workgroup w starts with block
// w / 8 of band w % 8, and the rest of a band is handed out by its ticket; a workgroup whose
// band is done helps with the next. Where lanes share pixels the grid is the resident
// workgroups, not the blocks, so that the traversal stacks' spill area has one entry per
// resident thread: a workgroup per 8x8 block takes 0.8 GB at 1080p, and per one-pixel block
// it would take 64 times that. For 8x8 blocks a workgroup each it stays: with one sample
// per pixel a launch lasts as long as its slowest block, and the tickets made 640 x 480 x 1
// over 36 triangles 184 -> 200 us.
struct BlockQueue {
    uint32_t* tickets;
    uint32_t blocks, per, x;
    // Blocks of band b beyond the workgroups' first ones.
    __device__ __forceinline__ uint32_t rest(uint32_t b) const {
        const uint32_t all = b * per < blocks ? min(per, blocks - b * per) : 0u, first = gridDim.x >> 3;
        return all > first ? all - first : 0u;
    }
    __device__ __forceinline__ uint32_t start(uint32_t* t, uint32_t n) {
        tickets = t;
        blocks = n;
        per = (n + 7u) / 8u;
        x = blockIdx.x & 7u;
        const uint32_t first = blockIdx.x >> 3;
        return first < per && x * per + first < n ? x * per + first : kNoBlock;
    }
    __device__ __forceinline__ uint32_t next() {
        if (blocks <= gridDim.x) return kNoBlock;
        const uint32_t lane = threadIdx.x;
        unsigned long long left = 1ull << x;
        while (true) {
            if (rest(x) != 0u && left != 0ull) {
                uint32_t idx = 0u;
                if (lane == 0) idx = atomicAdd(tickets + x * kTicketLine, 1u);
                idx = uniform_u32(idx);
                if (idx < rest(x)) return x * per + (gridDim.x >> 3) + idx;
            }
            // The band is done: one load shows the tickets of all.
            uint32_t seen = 0u;
            if (lane < 8u)
                seen = __hip_atomic_load(tickets + lane * kTicketLine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            left = __ballot(lane < 8u && seen < rest(lane));
            if (left == 0ull) return kNoBlock;
            do x = (x + 1u) & 7u;
            while (((left >> x) & 1ull) == 0ull);
        }
    }
};

// What bounds it is the slowest lane: at every bounce a wave waits for its longest ray, and a
// launch for its longest wave. With a launch per sample and a pixel per lane, 961 x 541 x 8
// over 1M triangles took 13.0 ms. Lanes that share a pixel start from nearly the same ray and
// meet the same surfaces, and a launch of 8 samples has 8 times the waves: 5.8 ms; 125 x 93 x 8
// over 97,292 triangles (192 waves before) 5.3 -> 0.82. Held at 5 and 6 waves per SIMD it
// spills 30 / 47 registers: 5.9 / 6.0 ms.
//
// SHARED: lanes share pixels (lanes_lg != 0). Such a wave's lanes trace nearly the same
// camera ray and reach their leaves together, so a leaf phase begins when fewer than 4 lanes
// want nodes (961 x 541 x 8 over 1M triangles 4.92 -> 4.77 ms, 512 x 512 x 16 over 100k
// 8.20 -> 7.86, 125 x 93 x 8 0.69 -> 0.63; thresholds 2 and 6 are 1 % behind). A wave of 64
// pixels waits for the last lane (4: 640 x 480 x 1 186 -> 206 us, 1280 x 720 x 1 522 -> 560).
// It also fetches nodes a step ahead and keeps only the record of its best hit (4.76 -> 4.52,
// 7.86 -> 7.59 and, 1280 x 720 x 64 over 1M triangles, 59.0 -> 56.1 ms); with 64 pixels, where
// the leaf phases wait for every lane, fetching ahead takes 186 -> 191 us at 640 x 480 x 1.
//
// KEEP: a.vertices is given (an instantiation of its own: the 15 instead of 11 registers spilled
// make the others 1 % slower).
template <bool COUNT, bool SHARED, bool KEEP>
__global__ __launch_bounds__(kBlock, 4) void megakernel(MegaArgs a) {
    __shared__ int s_stack[kStackLds * kBlock];
    __shared__ float s_rgb[3][kBlock];
    const uint32_t lanes_lg = SHARED ? a.lanes_lg : 0u;
    const uint32_t lane = threadIdx.x, share = 1u << lanes_lg, sub = lane & (share - 1u), px = lane >> lanes_lg;
    const uint32_t wlg = block_width_lg(lanes_lg), hlg = block_height_lg(lanes_lg);
    Stack st;
    st.bind(s_stack, a.spill + size_t(blockIdx.x) * kBlock, a.spill_stride);
    Counts cnt = {0, 0, 0, 0, 0, 0};
    BlockQueue queue;
    for (uint32_t block = queue.start(a.tickets, a.tiles); block != kNoBlock; block = queue.next()) {
        const uint32_t x = ((block % a.tiles_x) << wlg) + (px & ((1u << wlg) - 1u));
        const uint32_t y = ((block / a.tiles_x) << hlg) + (px >> wlg);
        const bool inside = x < a.width && y < a.height;
        const size_t idx = size_t(y) * a.width + x;
        V3 sum = v3(0.f, 0.f, 0.f);
        if (inside && sub == 0u) sum = v3(a.accum[idx]);
        for (uint32_t k = 0; k < a.nspp; k += share) {
            const uint32_t sample = a.s0 + k + sub;
            V3 L = v3(0.f, 0.f, 0.f);
            if (inside) {
                const size_t path = idx * a.samples_cap + sample;
                const bool keep = a.samples && sample < a.samples_cap;
                L = sample_path<COUNT, SHARED, KEEP>(a.sc, a.cam, a.path, int(x), int(y), sample,
                                               KEEP && keep ? a.vertices + path : nullptr,
                                               size_t(a.width) * a.height * a.samples_cap, st, cnt);
                if (keep) a.samples[path] = make_float4(L.x, L.y, L.z, 0.f);
            }
            if (share == 1u) {
                sum = sum + L;
                continue;
            }
            s_rgb[0][lane] = L.x;
            s_rgb[1][lane] = L.y;
            s_rgb[2][lane] = L.z;
            __syncthreads();
            if (sub == 0u)
                for (uint32_t j = lane; j < lane + share; ++j) sum = sum + v3(s_rgb[0][j], s_rgb[1][j], s_rgb[2][j]);
            __syncthreads();
        }
        if (inside && sub == 0u) a.accum[idx] = make_float4(sum.x, sum.y, sum.z, 0.f);
    }
    if (COUNT) flush_counts<COUNT>(a.counters, cnt);
}

// An 8x8 tile per workgroup. What bounds it is the waves in flight: a tile lasts as long as its
// longest ray, a dependent load per step. With 32 stack entries in LDS per lane 5 waves fitted a
// SIMD; with 16, and only the hit's record held through the traversal, 8 do. The lanes' rays are
// alike and reach leaves together, so a leaf phase with fewer than 16 lanes wanting nodes pays
// (the megakernel's lanes, at different bounces of different rays, wait best for the last).
// 1271 x 713 over 1M triangles: 232 -> 207 -> 161 us (a threshold of 8: 155, 24: 165); 1920 x
// 1080 over 2.8M 559 -> 437 -> 362; 3840 x 2160 over 1M 981 -> 790 -> 652.
__global__ __launch_bounds__(kBlock) void first_hit_kernel(FirstHitArgs a) {
    __shared__ int s_stack[kStackLdsQueue * kBlock];
    const uint32_t tile = xcd_tile(blockIdx.x, a.tiles);
    if (tile >= a.tiles) return;
    const int lane = int(threadIdx.x);
    const int x = int(tile % a.tiles_x) * 8 + (lane & 7);
    const int y = int(tile / a.tiles_x) * 8 + (lane >> 3);
    if (x >= int(a.width) || y >= int(a.height)) return;
    StackT<kStackLdsQueue> st;
    st.bind(s_stack, a.spill + size_t(blockIdx.x) * kBlock, a.spill_stride);
    Rng rng{a.path.seed, a.path.view, uint32_t(y) * uint32_t(a.cam.xpixels) + uint32_t(x), a.sample};
    V3 ro, rd;
    camera_ray(a.cam, x, y, rng.block(0), ro, rd);
    HitRec h;
    h.t = kFltMax;
    h.id = 0;
    h.rec = 0;
    Counts cnt;
    const bool hit = traverse<false, false, true, 16>(a.sc, ro, rd, kEps, h, st, cnt);
    const size_t idx = size_t(y) * a.width + size_t(x);
    if (a.tri) a.tri[idx] = hit ? int32_t(h.id) : -1;
    if (a.mat) a.mat[idx] = hit ? int32_t(__float_as_uint(gload(a.sc.tris, size_t(h.rec) * 3 + 1).w)) : -1;
    if (a.t) a.t[idx] = hit ? h.t : kFltMax;
}

// float3ToUchar4 then gammaCorrectPixel (renderer.h:149-156, renderer.cu:495-504)
// of accum / samples; negative and NaN map to 0.
__global__ void tonemap_kernel(const float4* accum, uint32_t n, uint32_t samples, const uint8_t* lut, uchar4* out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 a = accum[i];
    float s = float(samples);
    float c[3] = {a.x / s, a.y / s, a.z / s};
    uint8_t b[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float v = c[k];
        uint8_t q = 0;
        if (v > 0.0f) q = uint8_t((v > 1.0f ? 1.0f : v) * 255.f);
        b[k] = lut[q];
    }
    out[i] = make_uchar4(b[0], b[1], b[2], 255);
}

__global__ void mean_kernel(const float4* accum, uint32_t n, uint32_t samples, float* out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 a = accum[i];
    float s = float(samples);
    out[size_t(i) * 3] = a.x / s;
    out[size_t(i) * 3 + 1] = a.y / s;
    out[size_t(i) * 3 + 2] = a.z / s;
}

}  // namespace dev

hipError_t launch_megakernel(const MegaArgs& a, uint32_t grid, bool count, hipStream_t s) {
    auto pick = [&](auto keep) {
        constexpr bool kKeep = decltype(keep)::value;
        return a.lanes_lg != 0 ? count ? dev::megakernel<true, true, kKeep> : dev::megakernel<false, true, kKeep>
                               : count ? dev::megakernel<true, false, kKeep> : dev::megakernel<false, false, kKeep>;
    };
    auto kernel = a.vertices ? pick(std::true_type{}) : pick(std::false_type{});
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_first_hit(const FirstHitArgs& a, hipStream_t s) {
    const uint32_t grid = ((a.tiles + 7) / 8) * 8;
    hipLaunchKernelGGL(dev::first_hit_kernel, dim3(grid), dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_tonemap(const float4* accum, uint32_t n, float, uint32_t samples, const uint8_t* lut, uint8_t* out,
                          hipStream_t s) {
    hipLaunchKernelGGL(dev::tonemap_kernel, dim3((n + 255) / 256), dim3(256), 0, s, accum, n, samples, lut,
                       reinterpret_cast<uchar4*>(out));
    return hipGetLastError();
}

hipError_t launch_mean(const float4* accum, uint32_t n, uint32_t samples, float* out, hipStream_t s) {
    hipLaunchKernelGGL(dev::mean_kernel, dim3((n + 255) / 256), dim3(256), 0, s, accum, n, samples, out);
    return hipGetLastError();
}

}  // namespace prt
