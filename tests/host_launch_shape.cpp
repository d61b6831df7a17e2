// Rules of launch_shape.hpp over the sizes that the entry points accept.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <vector>

#include "launch_shape.hpp"

using namespace prt;

#define CHECK(c, ...)                                  \
    do {                                               \
        if (!(c)) {                                    \
            std::printf("%s: ", #c);                   \
            std::printf(__VA_ARGS__);                  \
            std::printf("\n");                         \
            std::exit(1);                              \
        }                                              \
    } while (0)

// Every launch of a call finds a spill column for each of its threads, and its blocks cover the
// image.
static void spill_fits_every_launch() {
    const uint32_t sides[] = {1, 2, 3, 7, 8, 9, 15, 33, 64, 100, 517, 1080, 1920, 4096, 9001, 65536};
    for (uint32_t resident : {16u, 512u, 4096u})
        for (uint32_t w : sides)
            for (uint32_t h : sides) {
                if (uint64_t(w) * h >= (uint64_t(1) << 32)) continue;
                const uint64_t blocks = uint64_t((w + 7) / 8) * ((h + 7) / 8);
                CHECK(first_hit_columns(w, h) >= blocks * kBlock, "%u x %u", w, h);
                for (uint32_t per : {0u, 1u, 2u, 3u, 6u, 8u, 48u, 64u, 96u, 1000u})
                    for (uint32_t n : {1u, 2u, 3u, 5u, 8u, 13u, 64u, 65u, 127u, 129u, 300u}) {
                        const uint64_t columns = mega_columns(w, h, n, per, resident);
                        uint32_t left = n;
                        while (left != 0) {
                            const MegaShape s = mega_shape(w, h, left, per, resident);
                            CHECK(s.samples >= 1 && s.samples <= left, "%u of %u", s.samples, left);
                            CHECK(s.samples % (1u << s.lanes_lg) == 0, "%u samples, %u", s.samples, s.lanes_lg);
                            CHECK(uint64_t(s.grid) * kBlock <= columns, "%u x %u, %u of %u, %u per", w, h, left, n, per);
                            CHECK(s.grid % 8 == 0 && s.grid > 0, "%u", s.grid);
                            const uint64_t bw = 1u << block_width_lg(s.lanes_lg), bh = 1u << block_height_lg(s.lanes_lg);
                            CHECK((bw * bh) << s.lanes_lg == 64, "%u", s.lanes_lg);
                            CHECK(s.tiles_x * bw >= w && uint64_t(s.tiles / s.tiles_x) * bh >= h, "%u x %u", w, h);
                            left -= s.samples;
                        }
                    }
            }
    // A call of very many samples ends quickly.
    CHECK(mega_columns(640, 480, 0xFFFFFFFFu, 0, 4096) == 640 * 480 / 64 * 64u, "%u", 0u);
}

// A failed growth leaves the area and frees nothing.
static void failed_growth_leaves_the_area() {
    int small[8] = {}, large[64] = {};
    int* area = nullptr;
    uint64_t have = 0;
    int freed = 0;
    auto none = [](uint64_t) { return static_cast<int*>(nullptr); };
    auto release = [&](int*) { ++freed; };
    CHECK(!grow(area, have, 8, none, release) && !area && have == 0 && freed == 0, "%d", freed);
    CHECK(grow(area, have, 8, [&](uint64_t) { return small; }, release) && area == small && have == 8, "%d", freed);
    CHECK(!grow(area, have, 64, none, release) && area == small && have == 8 && freed == 0, "%d", freed);
    CHECK(grow(area, have, 3, none, release) && area == small && have == 8 && freed == 0, "%d", freed);
    CHECK(grow(area, have, 64, [&](uint64_t) { return large; }, release) && area == large && have == 64 && freed == 1,
          "%d", freed);
}

// Batches that the waves of a launch hand out, each at most once; every wave in turn draws until
// it finds nothing.
static uint32_t handed_out(uint32_t batches, uint32_t waves) {
    std::vector<uint32_t> counter(kSpread, 0), given(batches, 0);
    for (uint32_t w = 0; w < waves; ++w) {
        if (w >= batches) continue;
        ++given[w];
        if (batches <= waves) continue;
        uint32_t k = w % kSpread;
        while (true) {
            uint32_t idx = counter[k]++, tries = 0;
            for (; idx >= fetch_limit(batches, waves, k) && tries < kSteal; ++tries) {
                k = next_counter(k);
                idx = counter[k]++;
            }
            if (idx >= fetch_limit(batches, waves, k)) break;
            const uint32_t b = fetch_batch(waves, k, idx);
            CHECK(b < batches, "batch %u of %u", b, batches);
            ++given[b];
        }
    }
    uint32_t n = 0;
    for (uint32_t g : given) {
        CHECK(g <= 1, "a batch given %u times", g);
        n += g;
    }
    return n;
}

static void every_batch_is_handed_out() {
    for (uint32_t resident : {1u, 7u, 16u, 20u, 32u, 63u, 64u, 65u, 100u, 8192u})
        for (uint32_t batches : {1u, 2u, 19u, 20u, 21u, 63u, 64u, 65u, 129u, 1000u, 20000u}) {
            const uint32_t waves = trace_waves(resident, batches);
            CHECK(waves >= 1 && waves <= batches, "%u waves, %u batches", waves, batches);
            CHECK(handed_out(batches, waves) == batches, "%u waves, %u batches", waves, batches);
        }
    // What trace_waves is for: fewer waves than counters may leave batches.
    CHECK(handed_out(50, 20) < 50, "%u", handed_out(50, 20));
}

static void idle_memory_is_bounded() {
    const uint64_t GB = 1ull << 30, device = 288 * GB;
    CHECK(may_stay_idle(7 * GB, 270 * GB, device) && may_stay_idle(18 * GB, 72 * GB, device), "%d", 0);
    CHECK(!may_stay_idle(19 * GB, 270 * GB, device), "%d", 0);
    CHECK(!may_stay_idle(7 * GB, 27 * GB, device) && !may_stay_idle(1, 0, device) && !may_stay_idle(1, 0, 0), "%d", 0);
}

int main() {
    idle_memory_is_bounded();
    every_batch_is_handed_out();
    spill_fits_every_launch();
    failed_growth_leaves_the_area();
    std::puts("ok");
    return 0;
}
