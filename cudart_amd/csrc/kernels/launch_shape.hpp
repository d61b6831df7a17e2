// Sizes of launches and of what they share: rules on numbers alone, the same on the host and in
// the kernels (constexpr functions are compiled for both), and checked on the CPU.
#pragma once

#include <cstdint>

namespace prt {

constexpr int kBlock = 64;  // one wave64 per workgroup: an 8x8 pixel tile

// Pixel block of a wave in which 2^lg lanes share a pixel: 8x8, 8x4, 4x4, 4x2, 2x2, 2x1, 1x1.
constexpr uint32_t block_width_lg(uint32_t lg) { return (7u - lg) / 2u; }
constexpr uint32_t block_height_lg(uint32_t lg) { return 6u - lg - block_width_lg(lg); }

// Workgroup order: consecutive workgroups land on different XCDs (round robin),
// so tile k is given to workgroup (k % per) * 8 + k / per, making each XCD's L2
// see a contiguous band of tiles.
constexpr uint32_t xcd_tile(uint32_t wg, uint32_t tiles) {
    const uint32_t per = (tiles + 7) / 8;
    return wg % 8 * per + wg / 8;
}

// A launch of the megakernel.
struct MegaShape {
    uint32_t samples;         // of every pixel
    uint32_t lanes_lg;        // log2 of the lanes that share a pixel
    uint32_t tiles_x, tiles;  // pixel blocks of a wave
    uint32_t grid;            // workgroups
};

// The next launch when `left` samples per pixel are to be rendered: spp_per_launch of them
// (0: the largest power of two, up to a wave's lanes). Where lanes share pixels the grid is at
// most the `resident` workgroups, else a workgroup per 8x8 block.
constexpr MegaShape mega_shape(uint32_t w, uint32_t h, uint32_t left, uint32_t spp_per_launch, uint32_t resident) {
    MegaShape s{1, 0, 0, 0, 0};
    if (spp_per_launch) s.samples = spp_per_launch < left ? spp_per_launch : left;
    else
        while (s.samples < 64 && 2 * s.samples <= left) s.samples *= 2;
    while (s.lanes_lg < 6 && s.samples % (2u << s.lanes_lg) == 0) ++s.lanes_lg;
    const uint32_t wlg = block_width_lg(s.lanes_lg), hlg = block_height_lg(s.lanes_lg);
    s.tiles_x = (w + (1u << wlg) - 1) >> wlg;
    s.tiles = s.tiles_x * ((h + (1u << hlg) - 1) >> hlg);
    s.grid = (s.tiles + 7) / 8 * 8;
    if (s.lanes_lg != 0 && s.grid > resident) s.grid = resident;
    return s;
}

// Threads of a first-hit launch, a workgroup per 8x8 block, and of the largest launch that renders
// `n` samples per pixel with the megakernel: the columns that they need in a spill area.
constexpr uint64_t first_hit_columns(uint32_t w, uint32_t h) {
    return (uint64_t((w + 7) / 8) * ((h + 7) / 8) + 7) / 8 * 8 * kBlock;
}
constexpr uint64_t mega_columns(uint32_t w, uint32_t h, uint32_t n, uint32_t spp_per_launch, uint32_t resident) {
    const uint32_t whole = spp_per_launch ? spp_per_launch : 64;  // samples of all launches but the last ones
    uint64_t most = 0;
    for (uint32_t left = n < whole ? n : whole + n % whole; left != 0;) {
        const MegaShape s = mega_shape(w, h, left, spp_per_launch, resident);
        most = s.grid > most ? s.grid : most;
        left -= s.samples;
    }
    return most * kBlock;
}

// How a launch's waves share the 64-item batches of a queue (WaveFetch): wave w's first batch is
// batch w, the batches from `waves` on belong to kSpread counters in turn, and a wave draws from
// counter w % kSpread, then from kSteal others, 21 apart.
#ifndef PRT_FETCH_BATCH
#define PRT_FETCH_BATCH 64
#endif
constexpr uint32_t kSpread = 64;
constexpr uint32_t kSteal = 2;  // other counters a wave tries when its own is exhausted
constexpr uint32_t kBatch = PRT_FETCH_BATCH;  // items per fetch atomic
// Batches of counter c, and the batch that its idx-th draw gives.
constexpr uint32_t fetch_limit(uint32_t batches, uint32_t waves, uint32_t c) {
    return batches > waves + c ? (batches - waves - c + kSpread - 1) / kSpread : 0u;
}
constexpr uint32_t fetch_batch(uint32_t waves, uint32_t c, uint32_t idx) { return waves + idx * kSpread + c; }
constexpr uint32_t next_counter(uint32_t c) { return (c + 21u) % kSpread; }
// Waves of a launch over `batches`: the resident ones, no more than there are batches, and at
// least one for every counter: one that is no wave's own might not be among those tried, and its
// rays would not be traced. (20 waves leave out batches of 41 to 62, more waves of none.)
constexpr uint32_t trace_waves(uint32_t resident, uint32_t batches) {
    const uint32_t waves = resident < kSpread ? kSpread : resident;
    return batches < waves ? batches : waves;
}

// Whether `bytes` of idle memory of a device may stay for the next call: at most a sixteenth of the
// device's, and at most a quarter of what is free beside it. Other allocators of the process
// cannot take it back, so where they have left little, none is kept.
constexpr bool may_stay_idle(uint64_t bytes, uint64_t free_bytes, uint64_t device_bytes) {
    return bytes <= device_bytes / 16 && bytes <= free_bytes / 4;
}

// Makes an area of `have` units one of at least `need`. The old one goes only when the new one is
// there: a failure leaves it, and the launches that it was large enough for, as they were.
template <class T, class Make, class Release>
bool grow(T*& area, uint64_t& have, uint64_t need, Make make, Release release) {
    if (area && have >= need) return true;
    T* larger = make(need);
    if (!larger) return false;
    if (area) release(area);
    area = larger;
    have = need;
    return true;
}

}  // namespace prt
