// Plain-data interface between the host library and the HIP kernels.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

#include "launch_shape.hpp"

namespace prt {

constexpr int kStackLds = 32;    // traversal stack entries per lane in LDS (megakernel)
#ifndef PRT_QUEUE_STACK_LDS
#define PRT_QUEUE_STACK_LDS 16
#endif
constexpr int kStackLdsQueue = PRT_QUEUE_STACK_LDS;  // LDS entries of the queue-based traversal kernels
constexpr int kStackMax = 128;   // total entries (those of the deepest scene; the rest in the global spill area)

// Device view of a built scene. Layouts:
//   nodes   4 x float4 per four-wide node (64 B, quantized child boxes)
//   tris    3 x float4 per record: {v1.xyz, id}{e1.xyz, material}{e2.xyz, 0} (48 B)
//   shade   4 x float4 per record: normals, uvs, area (64 B)
//   mats    4 x float4 per material: {kd, bsdf}{ka*3*A_L, tex}{ks, ns}{ni, dcoef, 0, 0}
struct SceneArgs {
    const float4* nodes;
    const float4* tris;
    const float4* shade;
    const float4* mats;
    const uint32_t* lights;   // record index of each emissive triangle, by original id
    const uint8_t* texels;    // RGBA8, all textures back to back
    const uint4* texinfo;     // per texture: first texel, width, height, 0
    const float* lin;         // 256-entry RGBA8 -> linear table
    float lights_area;
    float inv_lights_area;    // 1.f / lights_area, as samplePixel computes it
    uint32_t num_lights;
    uint32_t num_records;
};

struct CamArgs {
    float eye[3], dir[3], up[3], right[3];
    float fov, aspect, aperture_width, focus_distance;
    int32_t xpixels, ypixels;
};

struct PathArgs {
    uint32_t seed, view;
    uint32_t max_depth, rr_start;
};

// A path vertex as a forward pass keeps it: the record of the closest hit, whether the
// vertex's light sample was visible, or kVertexMiss. Records are below 2^28 - 1.
constexpr uint32_t kVertexLit = 0x80000000u;
constexpr uint32_t kVertexMiss = 0x0FFFFFFFu;

// Counter slots (unsigned long long each).
enum CounterSlot {
    kCntPrimary = 0,
    kCntExtension,
    kCntShadow,
    kCntNodes,
    kCntTris,
    kCntHits,
    kCntSamples,
    kCntAnyNodes,  // wavefront shadow kernel's share of kCntNodes
    kCntAnyTris,   // and of kCntTris
    kCntNum
};

struct MegaArgs {
    SceneArgs sc;
    CamArgs cam;
    PathArgs path;
    uint32_t width, height;
    uint32_t s0, nspp;
    uint32_t lanes_lg;        // log2 of the lanes that share a pixel, each a sample of its own; nspp is a multiple of them
    uint32_t tiles_x, tiles;  // pixel blocks of a wave
    uint32_t* tickets;        // one per XCD, kTicketLine words apart: blocks of its band handed out beyond the first
    float4* accum;            // width*height, .xyz = running sum
    float4* samples;          // nullptr, or each sample's radiance at [pixel * samples_cap + sample]
    uint32_t* vertices;       // nullptr, or with `samples`: its path's vertices, [(b * width * height + pixel) * samples_cap + sample]
    uint32_t samples_cap;     // samples stored per pixel
    unsigned long long* counters;  // kCntNum or nullptr
    int* spill;               // a row of spill_stride ints per stack entry beyond the LDS ones
    uint32_t spill_stride;
};

struct FirstHitArgs {
    SceneArgs sc;
    CamArgs cam;
    PathArgs path;
    uint32_t width, height, sample;
    uint32_t tiles_x, tiles;
    int32_t* tri;
    int32_t* mat;
    float* t;
    int* spill;
    uint32_t spill_stride;
};

// Launchers (render.hip). Return hipError_t.
hipError_t launch_megakernel(const MegaArgs& a, uint32_t grid, bool count, hipStream_t s);
hipError_t launch_first_hit(const FirstHitArgs& a, hipStream_t s);
hipError_t launch_tonemap(const float4* accum, uint32_t n, float inv_unused, uint32_t samples, const uint8_t* gamma_lut,
                          uint8_t* out, hipStream_t s);
hipError_t launch_mean(const float4* accum, uint32_t n, uint32_t samples, float* out_rgb, hipStream_t s);

constexpr uint32_t kTicketLine = 32;             // words between tickets: a cache line each
constexpr uint32_t kTicketSets = 32;             // launches between two clearings
constexpr uint32_t kTicketWords = 8 * kTicketLine;  // of one launch

}  // namespace prt
