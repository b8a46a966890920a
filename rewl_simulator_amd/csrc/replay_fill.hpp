// Host side of the replay streams: every walker's ring filled up to `cap` words
// past its cursor.  No HIP, so that a host compiler can test it.
#pragma once
#include <algorithm>
#include <cstdint>

namespace rewl {

// Words drawn into host memory between two waits, at most.  A wait per segment
// costs more than the draws of a small lattice; a buffer for all segments is as
// large as the rings (over 4 GB for 2048 walkers at L = 64) and, written for
// the first time, slower than the draws.  2 MB stay in cache: creation and first
// fill of 512 walkers at L = 64 take 188 ms (one buffer for all 376, a wait per
// segment 193) and 10 MB of host memory (1024 more), of 1024 walkers at L = 12
// 25 ms (48, 33).
constexpr uint64_t kReplayStage = 1u << 18;

// Words that the rings lack.
inline uint64_t replay_lack(int walkers, const uint64_t* cursor, const uint64_t* filled, uint64_t cap) {
    uint64_t words = 0;
    for (int g = 0; g < walkers; ++g) words += cursor[g] + cap - std::min(cursor[g] + cap, filled[g]);
    return words;
}

// draw(g): the next word of walker g's stream.  copy(g, pos, words, n): starts
// a copy of n words to position pos of g's ring; wait(): until the copies
// started are done with their words; both false on failure.  filled[g]: words
// put into g's ring so far.  stage: room for `room` words, the caller's until
// the last copies are done.
template <class Draw, class Copy, class Wait>
bool replay_fill(int walkers, const uint64_t* cursor, uint64_t* filled, uint64_t cap, uint64_t* stage, uint64_t room,
                 Draw draw, Copy copy, Wait wait) {
    uint64_t used = 0;
    for (int g = 0; g < walkers; ++g) {
        const uint64_t target = cursor[g] + cap;
        uint64_t& f = filled[g];
        while (f < target) {
            if (used == room) {
                if (!wait()) return false;
                used = 0;
            }
            const uint64_t pos = f & (cap - 1);
            const uint64_t n = std::min({target - f, cap - pos, room - used});
            uint64_t* const w = stage + used;
            for (uint64_t k = 0; k < n; ++k) w[k] = draw(g);
            if (!copy(g, pos, w, n)) return false;
            used += n;
            f += n;
        }
    }
    return true;
}

}  // namespace rewl
