// Arrays put one after the other, an alignment of 256 apart, travel in one copy;
// an array between two that are put, however small, keeps its bytes.
#include "fake_hip.h"

#include <random>

#include "host_stage.h"

using namespace aw;

int main()
{
    std::vector<char> dev(size_t(3) << 20, 7), src(size_t(3) << 20);
    std::mt19937 rng(3);
    for (char &c : src) c = (char)(rng() | 1);
    hipStream_t st;
    hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
    const auto put = [&](const std::vector<std::pair<size_t, size_t>> &at) {
        std::fill(dev.begin(), dev.end(), 7);
        const StageUse use;
        REQUIRE(use.s);
        {
            Uploader up(*use.s, st);
            for (auto [off, n] : at) REQUIRE(up.put(&dev[off], &src[off], n) == 0);
            REQUIRE(up.flush() == 0);
        }
        for (auto [off, n] : at) REQUIRE(memcmp(&dev[off], &src[off], n) == 0);
    };
    // the skipped array takes one alignment, or two, or three
    for (size_t skip : {256, 512, 768}) {
        put({{0, 256}, {256 + skip, 40}});
        for (size_t x = 256; x < 256 + skip; x++) REQUIRE(dev[x] == 7);
    }
    // random plans: every other array is skipped or not
    for (int trial = 0; trial < 200; trial++) {
        std::vector<std::pair<size_t, size_t>> at, kept;
        size_t off = 0;
        while (off < dev.size() - 70000) {
            const size_t n = 1 + rng() % (rng() % 8 ? 600 : 60000);
            (rng() % 3 ? at : kept).push_back({off, n});
            off = (off + n + 255) & ~size_t(255);
        }
        put(at);
        for (auto [o, n] : kept)
            for (size_t x = o; x < o + n; x++) REQUIRE(dev[x] == 7);
    }
    fake::copies = 0;
    put({{0, 100}, {256, 1}, {512, 3000}, {3584, 8}});
    REQUIRE(fake::copies == 1);
    // pieces of the staging memory
    fake::copies = 0;
    put({{0, dev.size() - 5}});
    REQUIRE(fake::copies == 2);
    printf("ok\n");
}
