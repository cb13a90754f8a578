// Plays a traversal launch of `blocks` blocks of `per_block` waves over n work
// slots: counts how often every slot is started, by the waves' own slots and
// by the chunks each block group claims until none is left.  Of the waves only
// the first `own` start with slots of their own.
#include "../../drawlab_amd/csrc/work_split.h"

#include <vector>

extern "C" int work_split_check(uint32_t n, uint32_t blocks, uint32_t per_block, uint32_t own) {
    std::vector<uint8_t> seen(n, 0);
    auto take = [&](uint32_t first, uint32_t count) {
        for (uint32_t k = 0; k < count; k++) {
            if (first + k >= n || ++seen[first + k] > 1) return false;
        }
        return true;
    };
    std::vector<uint32_t> claims(dl::kWorkGroups, 0);
    std::vector<uint8_t> done(dl::kWorkGroups, 0);
    for (uint32_t b = 0; b < blocks; b++) {
        for (uint32_t k = 0; k < per_block; k++) {
            const uint32_t wave = b * per_block + k;
            const dl::WorkSplit w = dl::split_work(n, wave, own, b, blocks);
            if (w.group >= dl::kWorkGroups || w.count > 64 || w.unit > 64) return 1;
            if (!take(w.first, w.count)) return 2;
        }
        const dl::WorkSplit w = dl::split_work(n, 0, own, b, blocks);
        while (w.base < n && !done[w.group]) {
            const uint32_t at = dl::chunk_start(w, claims[w.group]++);
            if (at >= n)
                done[w.group] = 1;
            else if (!take(at, dl::split_min(w.unit, n - at)))
                return 3;
        }
    }
    for (uint32_t i = 0; i < n; i++)
        if (!seen[i]) return 4;
    return 0;
}
