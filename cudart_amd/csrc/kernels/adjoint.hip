// Path-replay backpropagation (Vicini, Speierer, Jakob: "Path Replay
// Backpropagation: Differentiating Light Paths using Constant Memory and Linear
// Time", SIGGRAPH 2021) for the reference's estimator.
//
// Given dLoss/dI for every pixel (I = mean of `spp` samples), each sample's
// radiance L has adjoint delta = dLoss/dI / spp. For each pixel-sample the kernel
// takes L and the path's vertices from a forward pass that kept them (adjoint_stored), or
// traces the path once (the megakernel's arithmetic) to get them (adjoint_traced), then
// replays the path with the same Philox slots, tracing no ray, keeping the radiance still to
// be collected, rem = L - (what the path collected so far). Parameters:
//   kd_m (RGB)  a diffuse vertex multiplies everything collected after it by
//               kd_c, so it contributes delta_c * rem_c / kd_c (rem taken after
//               that vertex's emission, before its next-event estimate);
//   e_m         MTL Ka = e_m (1,1,1), ka = 3 e_m A_L: emission terms contribute
//               delta . mask * 3 A_L / A_L and next-event terms delta . mask * 3 A_L wf.
// Russian roulette (p = max(mask) after the vertex's weight) is differentiated
// as well: where p >= 1 the path always survives and mask /= p is a
// deterministic rescale; where p < 1 the survival probability depends on the
// albedos, and the boundary (score) term of that decision is weighted by the
// loss change it causes, which for a loss with curvature hess includes
// -(hess / 2) |R / spp|^2 (R = radiance collected after the decision). With
// both, the result is an unbiased estimate of the derivative of the expected
// loss, the quantity a central difference of renders with common random
// numbers estimates. Textured albedos get no kd gradient.
// Gradients accumulate in fp64: LDS per workgroup, then a fixed-order reduction.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "../host/common.hpp"
#include "path.hpp"
#include "renderer.hpp"

namespace prt {

struct AdjArgs {
    SceneArgs sc;
    CamArgs cam;
    PathArgs path;
    uint32_t width, height, spp;
    uint32_t tiles_x, tiles;
    uint32_t parts;       // workgroups per tile, each replaying a 1/parts range of its pixel-samples
    const float* grad;    // W*H*3 dLoss / dI
    const float4* samples;  // nullptr, or each sample's radiance from the forward pass [p * sample_cap + s]
    const uint32_t* vertices;  // nullptr, or its path's vertices [(b * W * H + p) * sample_cap + s]
    uint32_t sample_cap;
    double norm;          // 1 / spp: dI / dL of one sample
    double half_hess;     // (d2 Loss / dI2) / (2 spp^2): loss curvature per sample radiance
    uint32_t num_params;  // 4 * materials: kd (M*3) then emission (M)
    uint32_t num_materials;
    double* partial;      // grid x num_params (grid: tiles x parts rounded up to 8)
    uint32_t stack_rows;  // entries of a traversal stack
};

namespace dev {

struct D3 {
    double x, y, z;
};
__device__ __forceinline__ D3 d3(V3 v) { return D3{double(v.x), double(v.y), double(v.z)}; }
__device__ __forceinline__ double ddot(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ D3 dsub(D3 a, D3 b) { return D3{a.x - b.x, a.y - b.y, a.z - b.z}; }

// Tie-aware weight of each channel in d log max(mask): 1 for a unique maximum,
// 1/2 for each of two or three equal maxima (the mean of the one-sided
// derivatives of max, which is what a central difference measures).
__device__ __forceinline__ D3 rr_weight(uint32_t ties) {
    const double w = __popc(ties) == 1 ? 1.0 : 0.5;
    return D3{(ties & 1u) ? w : 0.0, (ties & 2u) ? w : 0.0, (ties & 4u) ? w : 0.0};
}

// Materials of the path's untextured diffuse vertices, 8 bits each (at most 16).
struct VertexList {
    uint64_t lo = 0, hi = 0;
    uint32_t n = 0;
    __device__ __forceinline__ void push(uint32_t m) {
        if (n < 8) lo |= uint64_t(m) << (8 * n);
        else hi |= uint64_t(m) << (8 * (n - 8));
        ++n;
    }
    __device__ __forceinline__ uint32_t at(uint32_t i) const {
        return uint32_t(((i < 8 ? lo : hi) >> (8 * (i & 7))) & 0xffu);
    }
};

// The replay state of one pixel-sample. L is its radiance.
struct Replay {
    PathState ps;
    Rng rng;
    D3 rem, delta;
    V3 L;
    VertexList vl;
    uint32_t prev_ties;  // channels at the maximum at the previous roulette step (0: none)
};

__device__ __forceinline__ void replay_begin(const AdjArgs& a, int x, int y, uint32_t sample, D3 delta, V3 L,
                                             Replay& r) {
    r.rem = d3(L);
    r.delta = delta;
    r.L = L;
    r.vl = VertexList();
    r.prev_ties = 0;
    r.rng = Rng{a.path.seed, a.path.view, uint32_t(y) * uint32_t(a.cam.xpixels) + uint32_t(x), sample};
    V3 ro, rd;
    camera_ray(a.cam, x, y, r.rng.block(0), ro, rd);
    path_init(r.ps, ro, rd);
}

// Russian roulette: everything collected after survived step j, R_j = L - C_j, carries 1/p_j,
// and with S_k[c] = sum over diffuse vertices v <= k of d log kd_{m_v,c}:
// d log p_j = w_j . S_j - w_{j-1} . S_{j-1}. The step adds -kappa_j d log p_j, with
// kappa_j = delta . R_j where p_j >= 1 (the path always survives; mask /= p_j is a
// deterministic rescale), and where p_j < 1 kappa_j = (hess / 2) |R_j / spp|^2: the score term
// of the survival probability times the loss change of that decision, delta . R_j -
// (hess / 2) |R_j / spp|^2, less the derivative of 1/p_j.
// So it adds kappa_j (w_{j-1} - w_j) for every diffuse vertex before the step and
// -kappa_j w_j for the step's own. The first is the same for all of them, so with P the
// running sum of kappa (w_{j-1} - w_j), a vertex adds
// -kappa_j w_j - P at its own step and P's last value when the path has ended: two adds per
// vertex and channel instead of one per vertex, step and channel.
// The vertex `word` of the path. Returns true when the path goes on.
__device__ __forceinline__ bool stored_vertex(const AdjArgs& a, Replay& r, uint32_t word, D3& P, double* g,
                                              Counts& cnt) {
    const SceneArgs& sc = a.sc;
    const uint32_t M = a.num_materials;
    const double gain = 3.0 * double(sc.lights_area);  // d ka / d e
    PathState& ps = r.ps;
    HitRec h;
    h.rec = word & kVertexMiss;
    h.id = 0;
    hit_details(sc.tris, ps.ro, ps.rd, h);
    const float4 mkd = sc.mats[size_t(h.mat) * 4], mka = sc.mats[size_t(h.mat) * 4 + 1];
    if (ps.b == 0 || ps.prev == 1 || ps.prev == 4) {
        const V3 e = ps.mask * v3(mka) * sc.inv_lights_area;
        atomicAdd(&g[3 * M + h.mat], ddot(r.delta, d3(ps.mask)) * gain * double(sc.inv_lights_area));
        r.rem = dsub(r.rem, d3(e));
    }
    const uint32_t b = ps.b;
    bool want_nee;
    NeeSample ns;
    RrInfo rr;
    const bool more = shade_vertex<false, false>(sc, a.path, r.rng, ps, h, &want_nee, ns, cnt, &rr);
    const bool diffuse = ps.prev == 0 /*DIFFUSE*/ && __float_as_int(mka.w) < 0;
    D3 own{r.delta.x * r.rem.x, r.delta.y * r.rem.y, r.delta.z * r.rem.z};
    if (want_nee) {
        ShadowReq sr;
        sr.direct = v3(0.f, 0.f, 0.f);
        const bool reach = nee_prepare<false>(sc, ns, sr, cnt);
        const bool visible = reach && ((word & kVertexLit) != 0u || !can_hit(sr.sd));
        if (visible) {
            r.rem = dsub(r.rem, d3(ns.mask * sr.direct));
            atomicAdd(&g[3 * M + sr.lmat], ddot(r.delta, d3(ns.mask)) * gain * double(sr.wf));
        }
        ps.color = add_direct(ps.color, ns.mask, sr.direct, visible);
    }
    const bool survived = rr.p >= 0.f && ps.b == b + 1;
    if (survived) {
        const D3 R = dsub(d3(r.L), d3(ps.color));
        const double kappa = rr.p >= 1.f ? ddot(r.delta, R) : a.half_hess * ddot(R, R);
        const D3 w = rr_weight(rr.ties), wp = rr_weight(r.prev_ties);
        if (wp.x != w.x) P.x += kappa * (wp.x - w.x);
        if (wp.y != w.y) P.y += kappa * (wp.y - w.y);
        if (wp.z != w.z) P.z += kappa * (wp.z - w.z);
        own.x -= (w.x != 0.0 ? kappa * w.x : 0.0) + P.x;
        own.y -= (w.y != 0.0 ? kappa * w.y : 0.0) + P.y;
        own.z -= (w.z != 0.0 ? kappa * w.z : 0.0) + P.z;
        r.prev_ties = rr.ties;
    }
    if (diffuse) {
        if (mkd.x != 0.f) atomicAdd(&g[3 * h.mat], own.x / double(mkd.x));
        if (mkd.y != 0.f) atomicAdd(&g[3 * h.mat + 1], own.y / double(mkd.y));
        if (mkd.z != 0.f) atomicAdd(&g[3 * h.mat + 2], own.z / double(mkd.z));
        // A vertex whose roulette step ended the path has no part in P.
        if (survived || rr.p < 0.f) r.vl.push(h.mat);
    }
    return more;
}

// A traversal stack with all its entries in LDS: AdjArgs::stack_rows rows of kBlock ints.
struct LdsStack {
    lds_int* lds;
    int sp;
    __device__ __forceinline__ void push(int v) { lds[sp++ * kBlock + threadIdx.x] = v; }
    __device__ __forceinline__ int pop() { return lds[--sp * kBlock + threadIdx.x]; }
};

// A workgroup's share of the pixel-samples: their terms into its LDS sums, then into its
// partials. Each closest hit's record and each light sample's visibility are known before a
// path is replayed, kept by a forward pass or (TRACE) found by tracing the path just before.
// The terms and the order in which they are added are the same either way, so the sums are
// too, bit for bit.
template <bool TRACE>
__device__ __forceinline__ void replay_unit(const AdjArgs& a, double* sums, uint32_t* words, LdsStack& st) {
    const uint32_t lane = threadIdx.x;
    for (uint32_t k = lane; k < a.num_params; k += kBlock) sums[k] = 0.0;
    __syncthreads();
    const uint32_t units = a.tiles * a.parts;
    const uint32_t unit = xcd_tile(blockIdx.x, units);
    if (unit < units) {
        const uint32_t tile = unit / a.parts, part = unit - tile * a.parts;
        const uint32_t tx = (tile % a.tiles_x) * 8, ty = (tile / a.tiles_x) * 8;
        const uint32_t cols = min(8u, a.width - tx), rows = min(8u, a.height - ty);
        const uint64_t items = uint64_t(cols) * rows * a.spp;
        const uint32_t i0 = uint32_t(items * part / a.parts), i1 = uint32_t(items * (part + 1) / a.parts);
        const size_t stride = TRACE ? kBlock : size_t(a.width) * a.height * a.sample_cap;
        Counts cnt = {0, 0, 0, 0, 0, 0};
        for (uint32_t j = i0 + lane; j < i1; j += kBlock) {
            const uint32_t p = j / a.spp, s = j - p * a.spp;
            const int x = int(tx + p % cols), y = int(ty + p / cols);
            const size_t pix = size_t(y) * a.width + size_t(x), path = pix * a.sample_cap + s;
            const uint32_t* at = TRACE ? words + lane : a.vertices + path;
            const V3 L = TRACE ? sample_path<false, true, true>(a.sc, a.cam, a.path, x, y, s, words + lane, stride,
                                                                st, cnt)
                               : v3(a.samples[path]);
            const D3 delta{a.norm * double(a.grad[pix * 3]), a.norm * double(a.grad[pix * 3 + 1]),
                           a.norm * double(a.grad[pix * 3 + 2])};
            Replay r;
            replay_begin(a, x, y, s, delta, L, r);
            D3 P{0.0, 0.0, 0.0};
            for (bool more = true; more; at += stride) {
                const uint32_t word = *at;
                more = word != kVertexMiss && stored_vertex(a, r, word, P, sums, cnt);  // the sky carries no parameter
            }
            if (P.x != 0.0 || P.y != 0.0 || P.z != 0.0)
                for (uint32_t i = 0; i < r.vl.n; ++i) {
                    const uint32_t m = r.vl.at(i);
                    const float4 kd = a.sc.mats[size_t(m) * 4];
                    if (kd.x != 0.f) atomicAdd(&sums[3 * m], P.x / double(kd.x));
                    if (kd.y != 0.f) atomicAdd(&sums[3 * m + 1], P.y / double(kd.y));
                    if (kd.z != 0.f) atomicAdd(&sums[3 * m + 2], P.z / double(kd.z));
                }
        }
    }
    __syncthreads();
    double* out = a.partial + size_t(blockIdx.x) * a.num_params;
    for (uint32_t k = lane; k < a.num_params; k += kBlock) out[k] = sums[k];
}

// The replay from kept vertices: no ray is traced.
//
// A lane replays one path, 64 consecutive samples of a pixel to a wave, with the bounces in
// step (the vertices, [bounce][pixel][sample], are read coalesced). A replay that traced the
// rays itself waited for node fetches for 0.43 of its waves' time, had 0.39 of its lanes active
// and took 167 VGPRs; on 512^2 x 64 samples of the 100k-triangle scene it took 35.6 ms, this
// 3.01, and the forward pass pays for the vertices with 4 bytes written per vertex (within its
// run-to-run spread). What is left is the vertices' arithmetic (127 VGPRs, 4 waves per SIMD;
// held at 5: 3.31 ms). The fp64 sums in LDS are not what bounds it: 4 or 8 copies of them, a
// lane adding to copy lane % 8, so that lanes meeting one material do not take turns, measured
// the same.
__global__ __launch_bounds__(kBlock) void adjoint_stored(AdjArgs a) {
    extern __shared__ double s_sums[];  // num_params
    LdsStack st{nullptr, 0};
    replay_unit<false>(a, s_sums, nullptr, st);
}

// The replay where no vertices are kept: each wave traces its 64 paths as the megakernel
// does, leaves their vertices in LDS (max_depth x 64 words) and replays them from there.
// It allocates nothing and uses no scratch or spill memory: the traversal stacks, as deep as
// the scene needs, are in LDS as well (9 KB for the 100k-triangle scene; 12 waves per compute
// unit, what the registers allow, fit up to about 44 entries).
__global__ __launch_bounds__(kBlock) void adjoint_traced(AdjArgs a) {
    extern __shared__ double s_sums[];  // num_params, then the words and the stacks
    uint32_t* words = reinterpret_cast<uint32_t*>(s_sums + a.num_params);
    LdsStack st{(lds_int*)(words + a.path.max_depth * kBlock), 0};
    replay_unit<true>(a, s_sums, words, st);
}

// Sums the per-workgroup partials of parameter blockIdx.x in a fixed order: thread t
// adds partials t, t + 256, t + 512, ... in turn, then the 256 sums are added in a
// fixed pairwise tree. The result depends only on the partials, not on scheduling.
constexpr uint32_t kReduceBlock = 256;
__global__ __launch_bounds__(kReduceBlock) void adjoint_reduce(const double* partial, uint32_t blocks,
                                                              uint32_t num_params, double* out) {
    __shared__ double s[kReduceBlock];
    const uint32_t k = blockIdx.x;
    double v = 0.0;
    for (uint32_t b = threadIdx.x; b < blocks; b += kReduceBlock) v += partial[size_t(b) * num_params + k];
    s[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t w = kReduceBlock / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = s[0];
}

}  // namespace dev

// Scratch of prt_adjoint_grad_static, the entry point that allocates nothing: the
// per-workgroup partial gradients (grid x P doubles), then the P reduced
// gradients. 16 MiB on every device the library runs that entry point on, held
// until the process ends. In host code `scratch` names a host-side stand-in, not
// device memory: host code uses only the address hipGetSymbolAddress returns.
constexpr size_t kStaticScratchDoubles = size_t(1) << 21;
static __device__ __align__(256) double scratch[kStaticScratchDoubles];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mutex;
double* g_scratch_ptr[kMaxScratchDevices] = {};

// The device address of `scratch` on `device` (the current device), looked up once
// per device on that device's first call.
int static_scratch(int device, double** out) {
    if (device < 0 || device >= kMaxScratchDevices) return fail(PRT_ERR_LIMIT, "device ordinal above 63");
    std::lock_guard<std::mutex> g(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!ptr) return fail(PRT_ERR_HIP, "hipGetSymbolAddress(scratch) returned a null address");
        g_scratch_ptr[device] = static_cast<double*>(ptr);
    }
    *out = g_scratch_ptr[device];
    return PRT_OK;
}
}  // namespace

namespace {
#define ADJ_TRY(expr)                                           \
    do {                                                        \
        hipError_t e_ = (expr);                                 \
        if (e_ != hipSuccess) {                                 \
            rc = hip_fail(e_, #expr);                           \
            goto done;                                          \
        }                                                       \
    } while (0)
// PRT_ADJOINT_PRIMAL_IN_REPLAY=1: without kept vertices, trace each sample's
// path inside the replay kernel even where the per-sample buffers would fit (tests).
#define HIP_CHECK(expr)                                    \
    do {                                                   \
        hipError_t e_ = (expr);                            \
        if (e_ != hipSuccess) return hip_fail(e_, #expr);  \
    } while (0)
bool primal_in_replay() {
    const char* v = std::getenv("PRT_ADJOINT_PRIMAL_IN_REPLAY");
    return v && v[0] == '1';
}

// Workgroups per 8x8 tile of the replay. One workgroup per tile left most of the GPU
// idle for the second half of the kernel: 512^2 x 64 samples of the 100k-triangle
// scene is 4,096 tiles against 3,072 resident waves (3 per SIMD), and the tiles'
// path costs differ, so the kernel ran 2.5 times as long as a tile's replay
// (6.4 of 12 wave slots per compute unit occupied on average). Splitting each tile's
// pixel-samples into `parts` ranges gives about 8 workgroups per resident wave slot.
// The partials (ceil8(tiles x parts) x 4 x materials doubles) must also fit the
// allocation-free entry point's scratch, so both entry points pick the same split and
// give the same sums. Nothing that a call may change takes part: the same call gives the
// same bits whatever came before it.
uint32_t adjoint_parts(const prt_renderer* r, uint32_t spp) {
    constexpr uint64_t kTargetUnits = 8ull * 3 * 4 * 256;  // 8 x (3 waves x 4 SIMDs x 256 CUs)
    const uint64_t tiles = std::max<uint32_t>(1, r->tiles);
    const uint64_t P = 4ull * r->scene->num_materials;
    uint64_t parts = std::max<uint64_t>(1, (kTargetUnits + tiles - 1) / tiles);
    parts = std::min<uint64_t>(parts, std::max<uint32_t>(1, spp));
    while (parts > 1 && ((tiles * parts + 7) / 8) * 8 * P + P > kStaticScratchDoubles) --parts;
    return uint32_t(parts);
}

// The replay's arguments for the renderer's view: seed, view, depth and the scene
// as the renderer holds them; grad = W*H*3 dLoss/dI on the device.
AdjArgs adjoint_args(const prt_renderer* r, const float* grad, float hess, uint32_t spp, double* partial) {
    AdjArgs a;
    a.sc = r->sc;
    a.cam = cam_args(r->cam);
    a.path = PathArgs{r->cfg.seed, r->cfg.view_id, r->cfg.max_depth, r->cfg.rr_start};
    a.width = r->w;
    a.height = r->h;
    a.spp = spp;
    a.tiles_x = r->tiles_x;
    a.tiles = r->tiles;
    a.parts = adjoint_parts(r, spp);
    a.grad = grad;
    // The forward pass's per-sample radiance, when it was kept for exactly these
    // samples with the scene's current materials (same seed, view and depth: the
    // renderer's configuration).
    a.samples = r->samples && r->samples_ok && r->samples_done >= spp && spp <= r->spp &&
                        r->samples_version == r->scene->mats_version
                    ? r->samples
                    : nullptr;
    a.vertices = a.samples ? r->vertices : nullptr;
    a.sample_cap = r->spp;
    a.norm = 1.0 / double(spp);
    a.half_hess = double(hess) / (2.0 * double(spp) * double(spp));
    a.num_params = 4 * r->scene->num_materials;
    a.num_materials = r->scene->num_materials;
    a.partial = partial;
    a.stack_rows = stack_entries(r->scene);
    return a;
}

// The replay over `grid` workgroups.
hipError_t launch_adjoint(const AdjArgs& a, uint32_t grid, hipStream_t s) {
    const size_t sums = a.num_params * sizeof(double);
    // At most 4 + 4 + 32 KB.
    const size_t rows = a.path.max_depth + a.stack_rows;
    if (a.vertices)
        hipLaunchKernelGGL(dev::adjoint_stored, dim3(grid), dim3(kBlock), sums, s, a);
    else
        hipLaunchKernelGGL(dev::adjoint_traced, dim3(grid), dim3(kBlock), sums + rows * kBlock * sizeof(int), s, a);
    return hipGetLastError();
}
}  // namespace

}  // namespace prt

using namespace prt;

extern "C" int prt_adjoint_grad(prt_renderer* r, const float* grad_rgb, float hess, uint32_t spp, float* d_albedo,
                                float* d_emission) {
    clear_error();
    if (!r || !grad_rgb || !d_albedo || !d_emission || spp == 0 || !(hess >= 0.f))
        return fail(PRT_ERR_INVALID_ARG, "bad argument");
    if (r->cfg.max_depth > 16) return fail(PRT_ERR_LIMIT, "the adjoint supports max_depth <= 16");
    const VertexUse use(r);
    int rc = set_device(r->cfg.device);
    if (rc != PRT_OK) return rc;
    rc = device_scene(r->scene, r->cfg.device, r->sc, r->stream);
    if (rc != PRT_OK) return rc;
    const size_t px = size_t(r->w) * r->h;
    const uint32_t M = r->scene->num_materials;
    const uint32_t P = 4 * M;
    const uint32_t grid = ((r->tiles * adjoint_parts(r, spp) + 7) / 8) * 8;
    // One block: gradient image, partials, results, and what a forward pass of this call keeps.
    auto part = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
    const size_t b_grad = part(px * 3 * sizeof(float)), b_part = part(size_t(grid) * P * sizeof(double));
    const size_t b_out = part(P * sizeof(double)), b_acc = part(px * sizeof(float4));
    const size_t b_samp = part(px * spp * sizeof(float4)), b_vert = part(px * spp * r->cfg.max_depth * sizeof(uint32_t));
    std::vector<double> g;
    try {
        g.resize(P);
    } catch (const std::bad_alloc&) {
        return fail(PRT_ERR_OUT_OF_MEMORY, "host allocation failed");
    }
    struct Lease {
        Scratch s;
        ~Lease() { give_scratch(s); }
    } scratch{take_scratch(r->cfg.device, b_grad + b_part + b_out + b_acc + b_samp + b_vert)};
    float ms = 0.f;
    AdjArgs a = adjoint_args(r, nullptr, hess, spp, nullptr);
    // Without kept vertices, a forward pass first writes each sample's radiance and
    // path vertices to buffers of this call (when they fit in a quarter of the free memory),
    // and the replay traces no ray. Otherwise each lane traces its sample's path before
    // replaying it. Radiance and vertices are the same either way, and so are the gradients.
    bool forward = false;
    if (!a.vertices && !primal_in_replay()) {
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) {
            free_b += scratch.s.bytes;
            forward = vertices_fit(r->w, r->h, spp, r->cfg.max_depth) && b_acc + b_samp + b_vert <= free_b / 4;
            if (!forward && !a.samples && px > (size_t(1) << 24) && b_acc + b_samp <= free_b / 4)
                return fail(PRT_ERR_LIMIT, "a view with more than 2^24 pixels");
        }
    }
    const size_t bytes = b_grad + b_part + b_out + (forward ? b_acc + b_samp + b_vert : 0);
    rc = scratch_for(scratch.s.mem, scratch.s.bytes, bytes);
    if (rc != PRT_OK) return rc;
    char* at = static_cast<char*>(scratch.s.mem);
    float* d_grad = reinterpret_cast<float*>(at);
    double* d_part = reinterpret_cast<double*>(at += b_grad);
    double* d_out = reinterpret_cast<double*>(at += b_part);
    float4* d_acc = reinterpret_cast<float4*>(at += b_out);
    float4* d_samp = reinterpret_cast<float4*>(at += b_acc);
    uint32_t* d_vert = reinterpret_cast<uint32_t*>(at += b_samp);
    a.grad = d_grad;
    a.partial = d_part;
    ADJ_TRY(hipMemcpyAsync(d_grad, grad_rgb, px * 3 * sizeof(float), hipMemcpyHostToDevice, r->stream));
    ADJ_TRY(hipEventRecord(r->ev0, r->stream));
    if (forward) {
        ADJ_TRY(hipMemsetAsync(d_acc, 0, px * sizeof(float4), r->stream));
        // Small passes by the megakernel, whose one launch is over before the wavefront's many are:
        // 125 x 93 x 8 over 100k triangles 0.63 against 0.98 ms, 256 x 256 x 4 0.87 / 1.19, 640 x 480 x 4
        // over 36 triangles (1.2M paths) 0.48 / 0.53; 961 x 541 x 8 over 1M triangles 4.5 / 3.3.
        if (px * spp <= (size_t(1) << 20)) {
            MegaArgs m = megakernel_args(r, d_acc, d_samp, d_vert, spp);
            rc = megakernel_samples(r, m, 0, spp, 0, false);
        } else {
            rc = wavefront_samples(r, spp, d_acc, d_samp, d_vert);
        }
        if (rc != PRT_OK) goto done;
        a.samples = d_samp;
        a.vertices = d_vert;
        a.sample_cap = spp;
    }
    ADJ_TRY(launch_adjoint(a, grid, r->stream));
    hipLaunchKernelGGL(dev::adjoint_reduce, dim3(P), dim3(dev::kReduceBlock), 0, r->stream, d_part, grid, P, d_out);
    ADJ_TRY(hipGetLastError());
    ADJ_TRY(hipEventRecord(r->ev1, r->stream));
    ADJ_TRY(copy_wait(g.data(), d_out, P * sizeof(double), hipMemcpyDeviceToHost, r->stream));
    ADJ_TRY(hipEventElapsedTime(&ms, r->ev0, r->ev1));
    for (uint32_t k = 0; k < 3 * M; ++k) d_albedo[k] = float(g[k]);
    for (uint32_t k = 0; k < M; ++k) d_emission[k] = float(g[3 * M + k]);
    r->last_ms = ms;
done:
    if (rc != PRT_OK) (void)hipStreamSynchronize(r->stream);  // nothing in flight uses the block
    return rc;
}

extern "C" int prt_adjoint_grad_static(prt_renderer* r, const float* grad_rgb_device, float hess, uint32_t spp,
                                       float* d_albedo, float* d_emission) {
    clear_error();
    if (!r || !grad_rgb_device || !d_albedo || !d_emission || spp == 0 || !(hess >= 0.f))
        return fail(PRT_ERR_INVALID_ARG, "bad argument");
    if (r->cfg.max_depth > 16) return fail(PRT_ERR_LIMIT, "the adjoint supports max_depth <= 16");
    const VertexUse use(r);
    int rc = set_device(r->cfg.device);
    if (rc != PRT_OK) return rc;
    {
        hipPointerAttribute_t at;
        hipError_t e = hipPointerGetAttributes(&at, grad_rgb_device);
        if (e != hipSuccess) (void)hipGetLastError();
        if (e != hipSuccess || at.type != hipMemoryTypeDevice || at.device != r->cfg.device)
            return fail(PRT_ERR_INVALID_ARG, "grad_rgb_device is not device memory of the renderer's device");
    }
    // The renderer's creation uploaded the scene to this device: this refreshes at
    // most the material table in place (a copy, no allocation).
    rc = device_scene(r->scene, r->cfg.device, r->sc, r->stream);
    if (rc != PRT_OK) return rc;
    const uint32_t M = r->scene->num_materials;
    const uint32_t P = 4 * M;
    const uint32_t grid = ((r->tiles * adjoint_parts(r, spp) + 7) / 8) * 8;
    if (size_t(grid) * P + P > kStaticScratchDoubles)
        return fail(PRT_ERR_LIMIT, "image too large for the static scratch: (8x8 tiles rounded up to 8) x 4 x "
                                   "materials + 4 x materials must be at most 2^21 doubles");
    double* base = nullptr;
    rc = static_scratch(r->cfg.device, &base);
    if (rc != PRT_OK) return rc;
    // Every workgroup writes all P of its partials and the reduction writes all P
    // results, so nothing in the scratch needs clearing between calls.
    AdjArgs a = adjoint_args(r, grad_rgb_device, hess, spp, base);
    double* d_out = base + size_t(grid) * P;
    double g[4 * PRT_MAX_MATERIALS];
    float ms = 0.f;
    HIP_CHECK(hipEventRecord(r->ev0, r->stream));
    HIP_CHECK(launch_adjoint(a, grid, r->stream));
    hipLaunchKernelGGL(dev::adjoint_reduce, dim3(P), dim3(dev::kReduceBlock), 0, r->stream,
                       static_cast<const double*>(base), grid, P, d_out);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipEventRecord(r->ev1, r->stream));
    HIP_CHECK(copy_wait(g, d_out, P * sizeof(double), hipMemcpyDeviceToHost, r->stream));
    HIP_CHECK(hipEventElapsedTime(&ms, r->ev0, r->ev1));
    for (uint32_t k = 0; k < 3 * M; ++k) d_albedo[k] = float(g[k]);
    for (uint32_t k = 0; k < M; ++k) d_emission[k] = float(g[3 * M + k]);
    r->last_ms = ms;
    return PRT_OK;
}

extern "C" int prt_adjoint(prt_renderer* r, const float* target_rgb, const float* image_rgb, uint32_t spp,
                           float* d_albedo, float* d_emission, float* loss) {
    clear_error();
    if (!r || !target_rgb || !d_albedo || !d_emission || spp == 0) return fail(PRT_ERR_INVALID_ARG, "bad argument");
    const size_t n = size_t(r->w) * r->h * 3;
    std::vector<float> img(n), grad(n);
    int rc = PRT_OK;
    if (image_rgb) {
        std::memcpy(img.data(), image_rgb, n * sizeof(float));
    } else {
        // Forward pass at the same seed: the renderer's accumulation is replaced.
        rc = prt_renderer_reset(r);
        if (rc == PRT_OK) rc = prt_render_spp(r, spp);
        if (rc == PRT_OK) rc = prt_get_radiance(r, img.data());
        if (rc != PRT_OK) return rc;
    }
    // d/dI of sum (I - T)^2 / n
    double l = 0.0;
    for (size_t k = 0; k < n; ++k) {
        const double d = double(img[k]) - double(target_rgb[k]);
        l += d * d;
        grad[k] = float(2.0 * d / double(n));
    }
    if (loss) *loss = float(l / double(n));
    return prt_adjoint_grad(r, grad.data(), float(2.0 / double(n)), spp, d_albedo, d_emission);
}
