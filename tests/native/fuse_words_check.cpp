// The numbering of one-launch passes (csrc/fuse_words.h) across the point where the 32-bit numbers turn: launches of
// random sizes publish their words as the kernels do; no launch may find a word of an earlier one under its number.
#include <cstdio>
#include <random>
#include <vector>

#include "../../blitzen_amd/csrc/fuse_words.h"

int main()
{
    constexpr uint32_t kWords = 640;
    std::mt19937 rng(1);
    struct Word {
        uint32_t number = 0;
        uint64_t written = 0;  // the launch, counted in 64 bits
    };
    std::vector<Word> words(kWords);
    uint32_t last = 0xffffffffu - 5000u;
    for (uint64_t k = 1; k <= 20000; ++k) {
        const uint32_t launch = bz::fuse_next(last);
        const uint32_t n_tiles = k % 3000 < 2990 ? 1u + rng() % 3u : 1u + rng() % kWords;  // large ones are rare
        if (launch == 0u) return std::puts("number zero"), 1;
        for (uint32_t t = 0; t < kWords; ++t) {
            if (words[t].number == launch) return std::printf("stale word %u\n", t), 1;
            if (words[t].number != 0u && k - words[t].written > 2u * kWords) return std::printf("old word %u\n", t), 1;
        }
        for (uint32_t t = 0; t < n_tiles; ++t) words[t] = Word{ launch, k };
        const uint32_t aged = bz::fuse_aged(launch, kWords);
        if (aged >= n_tiles) words[aged] = Word{};
        last = launch;
    }
    std::puts("ok");
    return 0;
}
