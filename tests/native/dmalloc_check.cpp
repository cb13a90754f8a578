// The context's tracked allocation over a device of `capacity` bytes played by
// the host: hipMalloc and hipFree are replaced below.
#include "../../drawlab_amd/csrc/hip/backend.h"

#include <cstdlib>

static size_t g_capacity, g_used, g_trims;
static std::unordered_map<void*, size_t> g_blocks;

extern "C" hipError_t hipMalloc(void** p, size_t bytes) {
    if (g_used + bytes > g_capacity) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    g_blocks[*p] = bytes;
    g_used += bytes;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
    g_used -= g_blocks.at(p);
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

namespace dl {
void trim_build(Ctx* c, bool all) {
    if (!all) return;
    g_trims++;
    for (DevBuf* b : {&c->build_scratch, &c->build_nodes}) {
        if (b->p) (void)dfree(c, b->p);
        *b = DevBuf{};
    }
}
}  // namespace dl

// A context holding 600 + 200 bytes of a build's buffers on a 1000-byte
// device asks for `bytes`, during a build or not; returns 1 if it gets them,
// plus 2 if the buffers are still there, plus 4 if the accounting is off.
extern "C" int dmalloc_check(size_t bytes, int building) {
    g_capacity = 1000;
    g_used = g_trims = 0;
    g_blocks.clear();
    dl::Ctx c;
    c.build_scratch.bytes = 600;
    c.build_nodes.bytes = 200;
    if (dl::dmalloc(&c, &c.build_scratch.p, 600) != hipSuccess) return -1;
    if (dl::dmalloc(&c, &c.build_nodes.p, 200) != hipSuccess) return -1;
    c.building = building != 0;
    void* p = nullptr;
    const bool got = dl::dmalloc(&c, &p, bytes) == hipSuccess;
    const bool kept = c.build_scratch.p && c.build_nodes.p;
    const bool counted = c.dev_bytes == g_used && c.dev_bytes == (got ? bytes : 0) + (kept ? 800 : 0);
    return (got ? 1 : 0) + (kept ? 2 : 0) + (counted ? 0 : 4);
}
