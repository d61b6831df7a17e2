// Rules of launch_shape.hpp over the sizes that the entry points accept.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

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

int main() {
    spill_fits_every_launch();
    failed_growth_leaves_the_area();
    std::puts("ok");
    return 0;
}
