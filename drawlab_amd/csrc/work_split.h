// How the waves of a persistent traversal share its work slots.  Plain
// arithmetic, so that a host test can check that every slot is dealt once.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define DL_SPLIT_FN __host__ __device__ __forceinline__
#else
#define DL_SPLIT_FN inline
#endif

namespace dl {

// Groups of blocks that claim from a counter of their own, at most.
constexpr uint32_t kWorkGroups = 64;
// From this many slots per wave on, some are claimed rather than given out.
constexpr uint32_t kClaimShare = 16;

DL_SPLIT_FN uint32_t split_min(uint32_t a, uint32_t b) { return a < b ? a : b; }
DL_SPLIT_FN uint32_t wave_share(uint32_t n, uint32_t waves) { return (n + waves - 1) / waves; }

struct WorkSplit {
    uint32_t n;       // slots in all
    uint32_t first;   // this wave's first slots: [first, first + count)
    uint32_t count;
    uint32_t base;    // slots from here on are claimed
    uint32_t unit;    // slots of a chunk
    uint32_t group;   // this block's group
    uint32_t groups;  // at most one per block: each has a block that claims its chunks
};

// wave / waves: the wave's index among those that start with slots of their
// own, and their number; a wave beyond them only claims.
DL_SPLIT_FN WorkSplit split_work(uint32_t n, uint32_t wave, uint32_t waves, uint32_t block, uint32_t blocks) {
    // (n is at most 2^31 and a grid has at most 2^13 waves)
    const uint32_t share = wave_share(n, waves);
    // Few slots: a few lanes of every wave rather than all lanes of some, as
    // a wave takes as long as the slowest of its lanes.  From kClaimShare per
    // wave on half of them, at most 64, are given out at once, the rest in
    // chunks of a quarter of a wave's share, 8 to 64 slots, so the waves end
    // together (1M shadow rays took 4 to 5 % longer with a sixteenth).
    const uint32_t per = share < kClaimShare ? share : split_min(64u, share / 2u);
    WorkSplit w;
    w.groups = split_min(kWorkGroups, blocks);
    w.group = block % w.groups;
    w.n = n;
    w.base = split_min(n, per * waves);
    w.first = split_min(split_min(wave, waves) * per, w.base);
    w.count = wave < waves ? split_min(per, w.base - w.first) : 0u;
    w.unit = share >= 256u ? 64u : share >= 128u ? 32u : share >= 64u ? 16u : 8u;
    return w;
}

// First slot of the chunk that the group's claim number `claim` names (at or
// beyond n: none is left).
DL_SPLIT_FN uint32_t chunk_start(const WorkSplit& w, uint32_t claim) {
    return w.base + (claim * w.groups + w.group) * w.unit;
}

}  // namespace dl
