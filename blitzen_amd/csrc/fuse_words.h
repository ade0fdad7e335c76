// fuse_words.h — how the launches of one-launch passes are numbered (plain C++, host and device).
//
// A tile's published word counts when it carries the launch's number. Numbers are 32 bits, so a word must not be left
// standing until its number comes round again: a stream that culls every 10 us is there after twelve hours.
#pragma once
#include <cstdint>

namespace bz {

// The launch after number `last`. Zero is no launch's number: the words start as zero, and are set back to it.
constexpr uint32_t fuse_next(uint32_t last) { return last == 0xffffffffu ? 1u : last + 1u; }

// Each launch sets one word back to zero, this one, unless it is a word of its own `n_tiles` (which it has written): so
// every word has been written or cleared within the last `words` launches, or once more `words` where the numbers turn.
constexpr uint32_t fuse_aged(uint32_t launch, uint32_t words) { return launch % words; }

}  // namespace bz
