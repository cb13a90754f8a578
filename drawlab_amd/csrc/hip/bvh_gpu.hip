// Device BVH builder (DL_BUILD_GPU): a linear BVH (Karras, "Maximizing
// parallelism in the construction of BVHs, octrees and k-d trees", HPG 2012)
// emitted directly in the child-pair layout of bvh_layout.h.
//
//   1. primitive boxes and the centroid bounds (block reduction + atomics,
//      spread over kSlots cache lines)
//   2. 64-bit keys: 30-bit Morton code of the centroid << 32 | primitive id
//      (unique, so the tree and the traversal order are deterministic)
//   3. radix sort of the keys (hipCUB)
//   4. hierarchy: every internal node finds its key range and split in
//      parallel; children covering <= kMaxLeafSize primitives become leaves
//   5. bottom-up boxes with per-node arrival counters
//   6. node emission (padded child boxes) and triangle pre-gather
//
// Each level of a Karras tree strictly lengthens the common key prefix, so
// over 64-bit keys no internal node is deeper than 64: the traversal stack
// (kMaxBinaryDepth) always suffices.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>

#include "../host/bvh_build.h"
#include "backend.h"
#include "dl_math.h"

namespace dl {

namespace {

constexpr int kB = 256;

__device__ __forceinline__ uint32_t ordered(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float unordered(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// Reductions of a build over its blocks: kSlots lines of kSlotWords words, a
// block using line blockIdx % kSlots: [0..2] ordered min of the centroids,
// [3..5] ordered max, [6] largest depth, [7] leaves.  Atomics on one line pass
// at some 55 per us: with a single line k_prim_boxes took 154 us for 2,097,152
// triangles (now 31), k_ploc_offsets 297 (232) and k_ploc_emit 167 (120).
constexpr int kSlots = 64, kSlotWords = 32;
static_assert(kSlots == 64, "one slot per lane");
__device__ __forceinline__ uint32_t* slot(uint32_t* red) { return red + (blockIdx.x & (kSlots - 1)) * kSlotWords; }

// The centroid bounds from the slots, in every lane of the wave.
__device__ __forceinline__ void scene_bounds(const uint32_t* __restrict__ red, float* lo, float* ext) {
    const uint32_t* b = red + (threadIdx.x & 63) * kSlotWords;
    for (int a = 0; a < 3; a++) {
        uint32_t mn = b[a], mx = b[3 + a];
        for (int off = 32; off > 0; off >>= 1) {
            mn = min(mn, (uint32_t)__shfl_xor((int)mn, off));
            mx = max(mx, (uint32_t)__shfl_xor((int)mx, off));
        }
        lo[a] = unordered(mn);
        ext[a] = unordered(mx) - lo[a];
    }
}

__global__ __launch_bounds__(kB) void k_prim_boxes(const float* __restrict__ pos, const uint32_t* __restrict__ idx,
                                                   uint32_t n, float4* __restrict__ blo, float4* __restrict__ bhi,
                                                   uint32_t* __restrict__ red) {
    __shared__ uint32_t smin[3][kB], smax[3][kB];
    uint32_t lmin[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, lmax[3] = {0, 0, 0};
    for (uint32_t i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) {
        float lo[3], hi[3];
        for (int a = 0; a < 3; a++) {
            const float x = pos[3 * idx[3 * i] + a], y = pos[3 * idx[3 * i + 1] + a], z = pos[3 * idx[3 * i + 2] + a];
            lo[a] = fminf(x, fminf(y, z));
            hi[a] = fmaxf(x, fmaxf(y, z));
            const uint32_t c = ordered(0.5f * (lo[a] + hi[a]));
            lmin[a] = min(lmin[a], c);
            lmax[a] = max(lmax[a], c);
        }
        blo[i] = make_float4(lo[0], lo[1], lo[2], 0.f);
        bhi[i] = make_float4(hi[0], hi[1], hi[2], 0.f);
    }
    for (int a = 0; a < 3; a++) {
        smin[a][threadIdx.x] = lmin[a];
        smax[a][threadIdx.x] = lmax[a];
    }
    __syncthreads();
    for (int s = kB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 3; a++) {
                smin[a][threadIdx.x] = min(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
                smax[a][threadIdx.x] = max(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int a = 0; a < 3; a++) {
            atomicMin(&slot(red)[a], smin[a][0]);
            atomicMax(&slot(red)[3 + a], smax[a][0]);
        }
}

__device__ __forceinline__ uint32_t expand_bits(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__global__ __launch_bounds__(kB) void k_keys(const float4* __restrict__ blo, const float4* __restrict__ bhi, uint32_t n,
                                             const uint32_t* __restrict__ red, unsigned long long* __restrict__ keys) {
    float lo[3], ext[3];
    scene_bounds(red, lo, ext);
    for (uint32_t i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) {
        const float4 l = blo[i], h = bhi[i];
        const float c[3] = {0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z)};
        uint32_t q[3];
        for (int a = 0; a < 3; a++) {
            const float t = ext[a] > 0.f ? (c[a] - lo[a]) / ext[a] : 0.5f;
            q[a] = (uint32_t)fminf(fmaxf(t * 1024.0f, 0.0f), 1023.0f);
        }
        const uint32_t m = (expand_bits(q[0]) << 2) | (expand_bits(q[1]) << 1) | expand_bits(q[2]);
        keys[i] = ((unsigned long long)m << 32) | (unsigned long long)i;
    }
}

// 21-bit integer -> 63-bit word with two zero bits after every bit (the
// interleave of a 3-D Morton code), by shift-and-mask halving steps.
__device__ __forceinline__ unsigned long long spread3(uint32_t a) {
    unsigned long long x = a & 0x1fffffull;
    x = (x | (x << 32)) & 0x001f00000000ffffull;
    x = (x | (x << 16)) & 0x001f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

// 63-bit Morton codes (21 bits per axis) of the centroids, with the
// primitive ids as sort values (PLOC: finer than the 30-bit keys, so
// dense meshes keep a spatial order inside a cell of the coarse grid).
__global__ __launch_bounds__(kB) void k_keys63(const float4* __restrict__ blo, const float4* __restrict__ bhi,
                                               uint32_t n, const uint32_t* __restrict__ red,
                                               unsigned long long* __restrict__ keys, uint32_t* __restrict__ ids) {
    float lo[3], ext[3];
    scene_bounds(red, lo, ext);
    for (uint32_t i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) {
        const float4 l = blo[i], h = bhi[i];
        const float c[3] = {0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z)};
        uint32_t q[3];
        for (int a = 0; a < 3; a++) {
            const float t = ext[a] > 0.f ? (c[a] - lo[a]) / ext[a] : 0.5f;
            q[a] = (uint32_t)fminf(fmaxf(t * 2097152.0f, 0.0f), 2097151.0f);
        }
        keys[i] = (spread3(q[0]) << 2) | (spread3(q[1]) << 1) | spread3(q[2]);
        ids[i] = i;
    }
}

__device__ __forceinline__ int delta(const unsigned long long* __restrict__ k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    return __clzll(k[i] ^ k[j]);
}

// Internal node i: range [first, last], split gamma (left child ends at gamma).
__global__ __launch_bounds__(kB) void k_hierarchy(const unsigned long long* __restrict__ keys, int n,
                                                  int2* __restrict__ range, int* __restrict__ split,
                                                  int* __restrict__ parent_int, int* __restrict__ parent_leaf) {
    for (int i = blockIdx.x * kB + threadIdx.x; i < n - 1; i += gridDim.x * kB) {
        const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
        const int dmin = delta(keys, n, i, i - d);
        int lmax = 2;
        while (delta(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
        int l = 0;
        for (int t = lmax / 2; t >= 1; t /= 2)
            if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
        const int j = i + l * d;
        const int dnode = delta(keys, n, i, j);
        int s = 0;
        int t = l;
        do {
            t = (t + 1) / 2;
            if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
        } while (t > 1);
        const int gamma = i + s * d + min(d, 0);
        const int first = min(i, j), last = max(i, j);
        range[i] = make_int2(first, last);
        split[i] = gamma;
        if (first == gamma)
            parent_leaf[gamma] = i;
        else
            parent_int[gamma] = i;
        if (last == gamma + 1)
            parent_leaf[gamma + 1] = i;
        else
            parent_int[gamma + 1] = i;
    }
}

// ilo/ihi are written by other lanes of the same kernel (k_boxes): plain
// pointers, no __restrict__, so loads stay ordered after the acquire fence.
__device__ __forceinline__ void child_box(int first, int last, int node_or_leaf, bool leaf, const float4* blo,
                                          const float4* bhi, const uint32_t* sorted, const float4* ilo,
                                          const float4* ihi, float4& lo, float4& hi) {
    (void)first;
    (void)last;
    if (leaf) {
        const uint32_t p = sorted[node_or_leaf];
        lo = blo[p];
        hi = bhi[p];
    } else {
        lo = ilo[node_or_leaf];
        hi = ihi[node_or_leaf];
    }
}

__global__ __launch_bounds__(kB) void k_boxes(int n, const int2* __restrict__ range, const int* __restrict__ split,
                                              const int* __restrict__ parent_int, const int* __restrict__ parent_leaf,
                                              const uint32_t* __restrict__ sorted, const float4* __restrict__ blo,
                                              const float4* __restrict__ bhi, float4* ilo, float4* ihi,
                                              int* __restrict__ arrive) {
    for (int k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB) {
        int node = parent_leaf[k];
        // A well-formed tree reaches the root within 64 levels; the bound
        // only guarantees termination.
        for (int level = 0; level < 2 * kMaxBinaryDepth; ++level) {
            __threadfence();
            if (atomicAdd(&arrive[node], 1) == 0) break;
            __threadfence();
            const int2 r = range[node];
            const int g = split[node];
            float4 a0, a1, b0, b1;
            child_box(r.x, g, g, r.x == g, blo, bhi, sorted, ilo, ihi, a0, a1);
            child_box(g + 1, r.y, g + 1, r.y == g + 1, blo, bhi, sorted, ilo, ihi, b0, b1);
            ilo[node] = make_float4(fminf(a0.x, b0.x), fminf(a0.y, b0.y), fminf(a0.z, b0.z), 0.f);
            ihi[node] = make_float4(fmaxf(a1.x, b1.x), fmaxf(a1.y, b1.y), fmaxf(a1.z, b1.z), 0.f);
            if (node == 0) break;
            node = parent_int[node];
        }
    }
}

// Number of internal ancestors of every leaf (an upper bound on the
// traversal depth of the collapsed tree).
__global__ __launch_bounds__(kB) void k_depth(int n, const int* __restrict__ parent_int,
                                              const int* __restrict__ parent_leaf, uint32_t* __restrict__ red) {
    uint32_t dmax = 0;
    for (int k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB) {
        int node = parent_leaf[k];
        uint32_t d = 1;
        while (node != 0 && d < 2 * kMaxBinaryDepth) {
            node = parent_int[node];
            ++d;
        }
        dmax = max(dmax, d);
    }
    atomicMax(&slot(red)[6], dmax);
}

__device__ __forceinline__ void pad(const float4& lo, const float4& hi, float* plo, float* phi) {
    float m = fmaxf(fmaxf(fmaxf(fabsf(lo.x), fabsf(hi.x)), fmaxf(fabsf(lo.y), fabsf(hi.y))),
                    fmaxf(fabsf(lo.z), fabsf(hi.z)));
    const float p = fmaxf(m, 1.17549435e-38f) * (1.0f / 65536.0f);
    plo[0] = lo.x - p;
    plo[1] = lo.y - p;
    plo[2] = lo.z - p;
    phi[0] = hi.x + p;
    phi[1] = hi.y + p;
    phi[2] = hi.z + p;
}

__global__ __launch_bounds__(kB) void k_emit(int n, const int2* __restrict__ range, const int* __restrict__ split,
                                             const uint32_t* __restrict__ sorted, const float4* __restrict__ blo,
                                             const float4* __restrict__ bhi, const float4* __restrict__ ilo,
                                             const float4* __restrict__ ihi, float4* __restrict__ nodes,
                                             uint32_t* __restrict__ red) {
    uint32_t nl = 0;
    for (int i = blockIdx.x * kB + threadIdx.x; i < n - 1; i += gridDim.x * kB) {
        const int2 r = range[i];
        const int g = split[i];
        const int cf[2] = {r.x, g + 1}, cl[2] = {g, r.y};
        float lo[2][3], hi[2][3];
        int ref[2], cnt[2];
        for (int c = 0; c < 2; c++) {
            const int size = cl[c] - cf[c] + 1;
            const int id = c == 0 ? g : g + 1;
            float4 a, b;
            child_box(cf[c], cl[c], id, size == 1, blo, bhi, sorted, ilo, ihi, a, b);
            pad(a, b, lo[c], hi[c]);
            if (size <= kMaxLeafSize) {
                ref[c] = ~cf[c];
                cnt[c] = size;
                nl++;
            } else {
                ref[c] = id;
                cnt[c] = 0;
            }
        }
        float4* np = nodes + 4 * (size_t)i;
        np[0] = make_float4(lo[0][0], hi[0][0], lo[1][0], hi[1][0]);
        np[1] = make_float4(lo[0][1], hi[0][1], lo[1][1], hi[1][1]);
        np[2] = make_float4(lo[0][2], hi[0][2], lo[1][2], hi[1][2]);
        reinterpret_cast<int4*>(np)[3] = make_int4(ref[0], ref[1], cnt[0], cnt[1]);
    }
    if (nl) atomicAdd(&slot(red)[7], nl);
}

__global__ __launch_bounds__(kB) void k_gather(int n, const uint32_t* __restrict__ sorted, const float* __restrict__ pos,
                                               const uint32_t* __restrict__ idx, float4* __restrict__ tris) {
    for (int k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB) {
        const uint32_t p = sorted[k];
        const uint32_t i0 = idx[3 * p], i1 = idx[3 * p + 1], i2 = idx[3 * p + 2];
        const float p0x = pos[3 * i0], p0y = pos[3 * i0 + 1], p0z = pos[3 * i0 + 2];
        const float e1x = pos[3 * i1] - p0x, e1y = pos[3 * i1 + 1] - p0y, e1z = pos[3 * i1 + 2] - p0z;
        const float e2x = pos[3 * i2] - p0x, e2y = pos[3 * i2 + 1] - p0y, e2z = pos[3 * i2 + 2] - p0z;
        float4* t = tris + 3 * (size_t)k;
        t[0] = make_float4(p0x, p0y, p0z, e1x);
        t[1] = make_float4(e1y, e1z, e2x, e2y);
        t[2] = make_float4(e2z, __uint_as_float(p), 0.f, 0.f);
    }
}

__global__ __launch_bounds__(kB) void k_low_ids(const unsigned long long* __restrict__ keys, int n,
                                                uint32_t* __restrict__ sorted) {
    for (int k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB)
        sorted[k] = (uint32_t)(keys[k] & 0xffffffffull);
}

__global__ void k_fill_int(int* p, int v, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_init_slots(uint32_t* red) {
    uint32_t* b = red + threadIdx.x * kSlotWords;
    for (int a = 0; a < 3; a++) {
        b[a] = 0xffffffffu;
        b[3 + a] = 0u;
    }
    b[6] = b[7] = 0u;
}

// Depth and leaves of a build from its slots (synchronises the stream).
dl_status read_slots(Ctx* c, const uint32_t* red, uint32_t* depth, uint32_t* leaves) {
    uint32_t h[kSlots * kSlotWords];
    DL_HIP_CHECK(c, hipMemcpyAsync(h, red, sizeof(h), hipMemcpyDeviceToHost, c->stream));
    DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    *depth = *leaves = 0;
    for (int k = 0; k < kSlots; k++) {
        *depth = std::max(*depth, h[k * kSlotWords + 6]);
        *leaves += h[k * kSlotWords + 7];
    }
    return DL_OK;
}

// Scratch arrays of a build: want() names them, alloc() lays them out in the
// context's kept build scratch.  (A hipMalloc and hipFree per array, 27 of
// each, cost more than a build's kernels: 18 ms of a build of 2,097,152
// triangles and a query were 5 ms of kernels.  With one allocation, given back
// after every build, it takes 3.7 ms; kept for the next one, see
// kBuildKeepBytes, 2.9.  A process's first build also loads the kernels: 12 ms.)
struct Scratch {
    Ctx* c;
    size_t bytes = 0;
    std::vector<std::pair<void**, size_t>> parts;
    template <typename T>
    void want(T** p, size_t count) {
        parts.emplace_back((void**)p, bytes);
        bytes += (std::max<size_t>(1, count) * sizeof(T) + 255) & ~(size_t)255;
    }
    dl_status alloc() {
        const dl_status e = grow(c, c->build_scratch, bytes);
        if (e != DL_OK) return e;
        for (auto& p : parts) *p.first = (char*)c->build_scratch.p + p.second;
        return DL_OK;
    }
    ~Scratch() {
        if (c->stream) (void)hipStreamSynchronize(c->stream);
    }
};

#define DL_TRY(expr)                \
    do {                            \
        dl_status s_ = (expr);      \
        if (s_ != DL_OK) return s_; \
    } while (0)

}  // namespace

// Kept by a context between builds at most: the scratch and binary nodes of
// 3.5 million triangles.  They serve the builds of the scenes that replace each
// other on the context, and are given back when a scene is put aside
// (dl_hip_scene_keep), with dl_hip_trim and with the context.
constexpr size_t kBuildKeepBytes = 1ull << 30;

void trim_build(Ctx* c, bool all) {
    if (!all && c->build_scratch.bytes + c->build_nodes.bytes <= kBuildKeepBytes) return;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (DevBuf* b : {&c->build_scratch, &c->build_nodes}) {
        if (b->p) (void)dfree(c, b->p);
        *b = DevBuf{};
    }
    c->num_binary = 0;
}

dl_status grow(Ctx* c, DevBuf& b, size_t bytes) {
    if (b.bytes >= bytes) return DL_OK;
    if (b.p) (void)dfree(c, b.p);
    b = DevBuf{};
    const hipError_t e = dmalloc(c, &b.p, bytes);
    if (e != hipSuccess) {
        b.p = nullptr;
        return hip_fail(c, e, "hipMalloc");
    }
    b.bytes = bytes;
    return DL_OK;
}

dl_status resize_exact(Ctx* c, float4** p, size_t bytes) {
    const auto it = c->dev_allocs.find(*p);
    if (*p && it != c->dev_allocs.end() && it->second == bytes) return DL_OK;
    if (*p) (void)dfree(c, *p);
    *p = nullptr;
    void* q = nullptr;
    const hipError_t e = dmalloc(c, &q, bytes);
    if (e != hipSuccess) return hip_fail(c, e, "hipMalloc");
    *p = (float4*)q;
    return DL_OK;
}

dl_status upload_host_bvh(Ctx* c, const HostBvh& bvh) {
    DL_TRY(grow(c, c->build_nodes, bvh.nodes.size() * sizeof(BvhNodeH)));
    DL_TRY(resize_exact(c, &c->ds.tris, std::max<size_t>(1, bvh.tris.size()) * sizeof(BvhTriH)));
    DL_HIP_CHECK(c, hipMemcpy(c->build_nodes.p, bvh.nodes.data(), bvh.nodes.size() * sizeof(BvhNodeH),
                              hipMemcpyHostToDevice));
    if (!bvh.tris.empty())
        DL_HIP_CHECK(c, hipMemcpy(c->ds.tris, bvh.tris.data(), bvh.tris.size() * sizeof(BvhTriH),
                                  hipMemcpyHostToDevice));
    c->num_binary = (uint32_t)bvh.nodes.size();
    return DL_OK;
}

// Scenes of at most kMaxLeafSize triangles: the host builder makes the
// single node.
static dl_status build_small(Ctx* c, dl_accel_stats* stats) {
    HostBvh bvh;
    build_bvh_host(c->tri_verts.data(), c->nprims, bvh);
    DL_TRY(upload_host_bvh(c, bvh));
    stats->num_nodes = (uint32_t)bvh.nodes.size();
    stats->num_leaves = bvh.num_leaves;
    stats->max_depth = bvh.max_depth;
    return DL_OK;
}

dl_status build_bvh_lbvh(Ctx* c, dl_accel_stats* stats) {
    const int n = (int)c->nprims;
    if (n <= kMaxLeafSize) return build_small(c, stats);
    Scratch sc{c};
    float4 *blo, *bhi, *ilo, *ihi;
    unsigned long long *keys, *keys_sorted;
    uint32_t *red, *sorted;
    int2* range;
    int *split, *parent_int, *parent_leaf, *arrive;
    sc.want(&blo, n);
    sc.want(&bhi, n);
    sc.want(&ilo, n);
    sc.want(&ihi, n);
    sc.want(&keys, n);
    sc.want(&keys_sorted, n);
    sc.want(&red, kSlots * kSlotWords);
    sc.want(&sorted, n);
    sc.want(&range, n);
    sc.want(&split, n);
    sc.want(&parent_int, n);
    sc.want(&parent_leaf, n);
    sc.want(&arrive, n);
    keys = keys_sorted = nullptr;
    size_t temp_bytes = 0;
    DL_HIP_CHECK(c, hipcub::DeviceRadixSort::SortKeys(nullptr, temp_bytes, keys, keys_sorted, n, 0, 64, c->stream));
    char* temp = nullptr;
    sc.want(&temp, temp_bytes);
    DL_TRY(sc.alloc());
    DL_TRY(grow(c, c->build_nodes, (size_t)(n - 1) * kNodeBytes));
    DL_TRY(resize_exact(c, &c->ds.tris, (size_t)n * kTriBytes));
    float4 *const pn = (float4*)c->build_nodes.p, *const pt = c->ds.tris;

    const int grid = std::max(1, c->num_cus) * 8;
    DL_HIP_CHECK(c, hipEventRecord(c->ev0, c->stream));
    k_init_slots<<<1, kSlots, 0, c->stream>>>(red);
    k_fill_int<<<grid, kB, 0, c->stream>>>(arrive, 0, (size_t)n);
    k_prim_boxes<<<grid, kB, 0, c->stream>>>(c->ds.pos, c->ds.idx, (uint32_t)n, blo, bhi, red);
    k_keys<<<grid, kB, 0, c->stream>>>(blo, bhi, (uint32_t)n, red, keys);
    DL_HIP_CHECK(c, hipcub::DeviceRadixSort::SortKeys(temp, temp_bytes, keys, keys_sorted, n, 0, 64, c->stream));
    k_low_ids<<<grid, kB, 0, c->stream>>>(keys_sorted, n, sorted);
    k_hierarchy<<<grid, kB, 0, c->stream>>>(keys_sorted, n, range, split, parent_int, parent_leaf);
    k_boxes<<<grid, kB, 0, c->stream>>>(n, range, split, parent_int, parent_leaf, sorted, blo, bhi, ilo, ihi, arrive);
    k_depth<<<grid, kB, 0, c->stream>>>(n, parent_int, parent_leaf, red);
    k_emit<<<grid, kB, 0, c->stream>>>(n, range, split, sorted, blo, bhi, ilo, ihi, pn, red);
    k_gather<<<grid, kB, 0, c->stream>>>(n, sorted, c->ds.pos, c->ds.idx, pt);
    DL_HIP_CHECK(c, hipGetLastError());
    DL_HIP_CHECK(c, hipEventRecord(c->ev1, c->stream));
    DL_HIP_CHECK(c, hipEventSynchronize(c->ev1));
    float ms = 0.f;
    DL_HIP_CHECK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    DL_TRY(read_slots(c, red, &stats->max_depth, &stats->num_leaves));
    stats->num_nodes = c->num_binary = (uint32_t)(n - 1);
    stats->build_ms = ms;
    if (stats->max_depth > (uint32_t)kMaxBinaryDepth) {
        c->bvh_too_deep = true;
        return set_error(c, DL_ERR_STATE, "LBVH deeper than the traversal stack");
    }
    return DL_OK;
}


// ===========================================================================
// PLOC (Meister and Bittner, "Parallel locally-ordered clustering for
// bounding volume hierarchy construction", TVCG 2018): starting from the
// Morton-ordered primitives, every cluster finds its nearest neighbour
// (smallest merged surface area) within kPlocRadius positions, mutual
// nearest neighbours merge, and the survivors are compacted in order, until
// one cluster remains.  Each merge also computes the node's SAH cost
// bottom-up (traversal kSahNode per node, kSahTri per triangle test):
// a subtree of at most kMaxLeafSize primitives becomes one leaf when that
// is cheaper than keeping it as internal nodes.  The triangles are laid out
// in depth-first leaf order, so every leaf's triangles are contiguous.
// ===========================================================================
namespace {

constexpr int kPlocRadius = 24;
// a visit of the 4-wide node that the binary node becomes costs about a
// triangle test, the traversal testing a leaf's triangles two at a time
// (measured on the 2M-triangle workload: 1.0 beats 0.35, 0.5, 0.7, 1.5 and
// 2.0 by 1-3%, with 8.48 node visits and 3.16 triangle tests per ray
// against 8.87 and 2.59 at 0.5)
constexpr float kSahNode = 1.0f, kSahTri = 1.0f;

__device__ __forceinline__ float half_area(const float4& lo, const float4& hi) {
    const float dx = hi.x - lo.x, dy = hi.y - lo.y, dz = hi.z - lo.z;
    return dx * dy + dy * dz + dz * dx;
}

// A step of the clustering reads how many clusters there are and where the
// next node goes from device memory and leaves the next step's values there,
// so that steps follow each other without the host.
struct PlocState {
    int count;  // clusters
    int top;    // index of the next internal node (they are handed out downwards)
};
// A step is three kernels: the neighbour search, the counts of merges and of
// absorbed partners per chunk of consecutive clusters (at most kPlocChunks),
// and the merge, which adds up the counts before its chunk and writes merged
// and unmerged clusters straight to their compacted places.  (As flags, two
// library scans, merge and compaction with the counts read back in between, a
// step was eleven launches and a wait; 72 of them at 2,097,152 triangles.)
// Once at most kPlocTail clusters are left, one block does the remaining steps
// (half of all, 196 us) in its LDS.  Bound by the latency of the many short
// kernels: 40 steps of 28 us on average at 2,097,152 triangles; the whole build
// took 17.8 ms and takes 3.0.
constexpr int kPlocChunks = 2048;
constexpr int kPlocTail = 2048, kPlocTailThreads = 1024;
constexpr int kPlocBatch = 8;  // steps launched between two reads of the count
__device__ __forceinline__ int ploc_chunk(int n) { return max(kB, (n + kPlocChunks * kB - 1) / (kPlocChunks * kB) * kB); }

struct PlocNodes {
    int2* child;
    float4 *lo, *hi;
    int *count, *ecount, *parent_int, *parent_leaf, *leaf;
    float* cost;
};

// Cluster references: r >= 0 internal node, r < 0 leaf of sorted position ~r.
__global__ __launch_bounds__(kB) void k_ploc_init(int n, const uint32_t* __restrict__ sorted,
                                                  const float4* __restrict__ blo, const float4* __restrict__ bhi,
                                                  int* __restrict__ cref, float4* __restrict__ clo,
                                                  float4* __restrict__ chi, PlocState* __restrict__ st) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *st = PlocState{n, n - 2};
    for (int k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB) {
        const uint32_t p = sorted[k];
        cref[k] = ~k;
        clo[k] = blo[p];
        chi[k] = bhi[p];
    }
}

// Nearest neighbour of cluster at (tile position) i among positions j0..j1 of
// the tile: smallest merged area, the lowest position on ties, the previous
// cluster when no area is finite.
__device__ __forceinline__ int ploc_nearest(const float4* s_lo, const float2* s_hi, int i, int j0, int j1, int other) {
    const float4 a = s_lo[i];
    const float2 b = s_hi[i];
    float best = INFINITY;
    int bj = other;
    for (int j = j0; j <= j1; ++j) {
        const float4 c = s_lo[j];
        const float2 d = s_hi[j];
        const float dx = fmaxf(a.w, c.w) - fminf(a.x, c.x), dy = fmaxf(b.x, d.x) - fminf(a.y, c.y),
                    dz = fmaxf(b.y, d.y) - fminf(a.z, c.z);
        const float ar = dx * dy + dy * dz + dz * dx;
        if (j != i && ar < best) {  // j increases, so ties keep the lowest position
            best = ar;
            bj = j;
        }
    }
    return bj;
}

// A block's 256 clusters and the kPlocRadius on each side are staged in LDS:
// read from the caches, the 48 candidates' boxes cost 96 16-byte reads a
// thread (1.10 ms per build of 2,097,152 triangles; now 0.58 ms).
__global__ __launch_bounds__(kB) void k_ploc_nn(const PlocState* __restrict__ st, const float4* __restrict__ clo,
                                                const float4* __restrict__ chi, int* __restrict__ nn) {
    __shared__ float4 s_lo[kB + 2 * kPlocRadius];  // lo, hi.x
    __shared__ float2 s_hi[kB + 2 * kPlocRadius];  // hi.y, hi.z
    const int n = st->count;
    for (int t0 = blockIdx.x * kB; t0 < n; t0 += gridDim.x * kB) {
        const int first = max(0, t0 - kPlocRadius), last = min(n, t0 + kB + kPlocRadius) - 1;
        for (int k = first + threadIdx.x; k <= last; k += kB) {
            const float4 l = clo[k], h = chi[k];
            s_lo[k - first] = make_float4(l.x, l.y, l.z, h.x);
            s_hi[k - first] = make_float2(h.y, h.z);
        }
        __syncthreads();
        const int i = t0 + threadIdx.x;
        if (i < n) {
            const int j0 = max(0, i - kPlocRadius), j1 = min(n - 1, i + kPlocRadius);
            nn[i] = first + ploc_nearest(s_lo, s_hi, i - first, j0 - first, j1 - first,
                                         (i > 0 ? i - 1 : i + 1) - first);
        }
        __syncthreads();
    }
}

// Merges that start at cluster i (low half: a mutual pair, i < partner) and
// whether i is absorbed by a merge (high half).
__device__ __forceinline__ uint32_t ploc_flags(int i, const int* nn) {
    const int j = nn[i];
    const bool mutual = nn[j] == i;
    return (mutual && i < j ? 1u : 0u) | (mutual && i > j ? 0x10000u : 0u);
}

// Exclusive sum over the block's threads (halves apart, each at most 2^16 - 1)
// and its total; s_wave: one word per wave.
template <int WAVES>
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* s_wave, uint32_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = v;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)inc, off);
        if (lane >= off) inc += o;
    }
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (int w = 0; w < WAVES; w++) {
        if (w < wave) before += s_wave[w];
        total += s_wave[w];
    }
    __syncthreads();
    return before + inc - v;
}

__global__ __launch_bounds__(kB) void k_ploc_count(const PlocState* __restrict__ st, const int* __restrict__ nn,
                                                   int2* __restrict__ sums) {
    __shared__ int s_part[kB / 64][2];
    const int n = st->count, chunk = ploc_chunk(n);
    if (n < 2 || (long long)blockIdx.x * chunk >= n) return;
    const int c0 = blockIdx.x * chunk, c1 = min(n, c0 + chunk);
    int m = 0, r = 0;
    for (int i = c0 + threadIdx.x; i < c1; i += kB) {
        const uint32_t f = ploc_flags(i, nn);
        m += f & 0xffff;
        r += f >> 16;
    }
    for (int off = 32; off > 0; off >>= 1) {
        m += __shfl_xor(m, off);
        r += __shfl_xor(r, off);
    }
    if ((threadIdx.x & 63) == 0) {
        s_part[threadIdx.x >> 6][0] = m;
        s_part[threadIdx.x >> 6][1] = r;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        m = r = 0;
        for (int w = 0; w < kB / 64; w++) {
            m += s_part[w][0];
            r += s_part[w][1];
        }
        sums[blockIdx.x] = make_int2(m, r);
    }
}

// Node of the merge of clusters (ra, a) and (rb, b); returns its box.
__device__ __forceinline__ void ploc_node(const PlocNodes& t, int node, int ra, int rb, const float4& a0,
                                          const float4& a1, const float4& b0, const float4& b1, float4& lo,
                                          float4& hi) {
    lo = make_float4(fminf(a0.x, b0.x), fminf(a0.y, b0.y), fminf(a0.z, b0.z), 0.f);
    hi = make_float4(fmaxf(a1.x, b1.x), fmaxf(a1.y, b1.y), fmaxf(a1.z, b1.z), 0.f);
    t.child[node] = make_int2(ra, rb);
    t.lo[node] = lo;
    t.hi[node] = hi;
    const int cnt = (ra < 0 ? 1 : t.count[ra]) + (rb < 0 ? 1 : t.count[rb]);
    t.count[node] = cnt;
    // SAH: internal cost from the children's (already final) costs;
    // a small enough subtree becomes one leaf when that is not dearer
    const float area = half_area(lo, hi);
    const float ca = ra < 0 ? kSahTri : t.cost[ra], cb = rb < 0 ? kSahTri : t.cost[rb];
    const float cint = area > 0.0f ? kSahNode + (half_area(a0, a1) * ca + half_area(b0, b1) * cb) / area
                                   : kSahNode + ca + cb;
    const bool leaf = cnt <= kMaxLeafSize && (float)cnt * kSahTri <= cint;
    t.cost[node] = leaf ? (float)cnt * kSahTri : cint;
    t.leaf[node] = leaf ? 1 : 0;
    // nodes emitted in this subtree (none below a leaf)
    t.ecount[node] = leaf ? 0 : 1 + (ra < 0 ? 0 : t.ecount[ra]) + (rb < 0 ? 0 : t.ecount[rb]);
    if (ra < 0) t.parent_leaf[~ra] = node; else t.parent_int[ra] = node;
    if (rb < 0) t.parent_leaf[~rb] = node; else t.parent_int[rb] = node;
}

__global__ __launch_bounds__(kB) void k_ploc_merge(const PlocState* __restrict__ st, PlocState* __restrict__ next,
                                                   const int* __restrict__ nn, const int2* __restrict__ sums,
                                                   const int* __restrict__ cref, const float4* __restrict__ clo,
                                                   const float4* __restrict__ chi, int* __restrict__ oref,
                                                   float4* __restrict__ olo, float4* __restrict__ ohi, PlocNodes t) {
    __shared__ int s_before[kB / 64][2];
    __shared__ uint32_t s_wave[kB / 64];
    const int n = st->count, top = st->top, chunk = ploc_chunk(n);
    if (n < 2) {
        // done: the cluster's data is not read again
        if (blockIdx.x == 0 && threadIdx.x == 0) *next = PlocState{n, top};
        return;
    }
    if ((long long)blockIdx.x * chunk >= n) return;
    int m = 0, r = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += kB) {
        const int2 v = sums[k];
        m += v.x;
        r += v.y;
    }
    for (int off = 32; off > 0; off >>= 1) {
        m += __shfl_xor(m, off);
        r += __shfl_xor(r, off);
    }
    if ((threadIdx.x & 63) == 0) {
        s_before[threadIdx.x >> 6][0] = m;
        s_before[threadIdx.x >> 6][1] = r;
    }
    __syncthreads();
    m = r = 0;
    for (int w = 0; w < kB / 64; w++) {
        m += s_before[w][0];
        r += s_before[w][1];
    }
    const int c0 = blockIdx.x * chunk, c1 = min(n, c0 + chunk);
    for (int b = c0; b < c1; b += kB) {
        const int i = b + threadIdx.x;
        const uint32_t f = i < c1 ? ploc_flags(i, nn) : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive<kB / 64>(f, s_wave, total);
        if (i < c1 && !(f >> 16)) {
            const int d = i - (r + (int)(ex >> 16));
            int ref = cref[i];
            float4 lo = clo[i], hi = chi[i];
            if (f & 0xffff) {
                const int j = nn[i], node = top - (m + (int)(ex & 0xffff));
                float4 nlo, nhi;
                ploc_node(t, node, ref, cref[j], lo, hi, clo[j], chi[j], nlo, nhi);
                ref = node;
                lo = nlo;
                hi = nhi;
            }
            oref[d] = ref;
            olo[d] = lo;
            ohi[d] = hi;
        }
        m += (int)(total & 0xffff);
        r += (int)(total >> 16);
    }
    if (c1 == n && threadIdx.x == 0) *next = PlocState{n - r, top - m};
}

// The last steps, in one block: at most kPlocTail clusters.
__global__ __launch_bounds__(kPlocTailThreads) void k_ploc_tail(PlocState* st, const int* __restrict__ cref,
                                                                const float4* __restrict__ clo,
                                                                const float4* __restrict__ chi, PlocNodes t) {
    constexpr int kPer = kPlocTail / kPlocTailThreads;
    __shared__ float4 s_lo[kPlocTail];
    __shared__ float2 s_hi[kPlocTail];
    __shared__ int s_ref[kPlocTail], s_nn[kPlocTail];
    __shared__ uint32_t s_wave[kPlocTailThreads / 64];
    int n = st->count, top = st->top;
    if (n > kPlocTail) return;
    for (int k = threadIdx.x; k < n; k += kPlocTailThreads) {
        const float4 l = clo[k], h = chi[k];
        s_lo[k] = make_float4(l.x, l.y, l.z, h.x);
        s_hi[k] = make_float2(h.y, h.z);
        s_ref[k] = cref[k];
    }
    __syncthreads();
    while (n > 1) {
        for (int i = threadIdx.x; i < n; i += kPlocTailThreads)
            s_nn[i] = ploc_nearest(s_lo, s_hi, i, max(0, i - kPlocRadius), min(n - 1, i + kPlocRadius),
                                   i > 0 ? i - 1 : i + 1);
        __syncthreads();
        int m = 0, r = 0, d[kPer], ref[kPer];
        float4 lo[kPer], hi[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = k * kPlocTailThreads + threadIdx.x;
            const uint32_t f = i < n ? ploc_flags(i, s_nn) : 0u;
            uint32_t total;
            const uint32_t ex = block_exclusive<kPlocTailThreads / 64>(f, s_wave, total);
            d[k] = -1;
            if (i < n && !(f >> 16)) {
                d[k] = i - (r + (int)(ex >> 16));
                ref[k] = s_ref[i];
                const float4 a = s_lo[i];
                const float2 b = s_hi[i];
                lo[k] = make_float4(a.x, a.y, a.z, 0.f);
                hi[k] = make_float4(a.w, b.x, b.y, 0.f);
                if (f & 0xffff) {
                    const int j = s_nn[i], node = top - (m + (int)(ex & 0xffff));
                    const float4 e = s_lo[j];
                    const float2 g = s_hi[j];
                    float4 nlo, nhi;
                    ploc_node(t, node, ref[k], s_ref[j], lo[k], hi[k], make_float4(e.x, e.y, e.z, 0.f),
                              make_float4(e.w, g.x, g.y, 0.f), nlo, nhi);
                    ref[k] = node;
                    lo[k] = nlo;
                    hi[k] = nhi;
                }
            }
            m += (int)(total & 0xffff);
            r += (int)(total >> 16);
        }
        __syncthreads();  // the nodes of this step and the old clusters have been read and written
#pragma unroll
        for (int k = 0; k < kPer; k++)
            if (d[k] >= 0) {
                s_ref[d[k]] = ref[k];
                s_lo[d[k]] = make_float4(lo[k].x, lo[k].y, lo[k].z, hi[k].x);
                s_hi[d[k]] = make_float2(hi[k].y, hi[k].z);
            }
        n -= r;
        top -= m;
        __syncthreads();
        if (m == 0) break;  // (cannot happen; the host reports it)
    }
    if (threadIdx.x == 0) *st = PlocState{n, top};
}

// Depth-first position of every leaf (element k < n, sorted position k) and
// of every internal node (element n + i): the number of primitives to its
// left, summed over the ancestors it descends from as a right child.
// Also the depth-first pre-order rank of every surviving internal node among
// the surviving nodes (its ancestors, plus the surviving nodes of every left
// sibling subtree), which becomes its index in the emitted node array.
__global__ __launch_bounds__(kB) void k_ploc_offsets(int n, const int2* __restrict__ child,
                                                     const int* __restrict__ ncount, const int* __restrict__ ecount,
                                                     const int* __restrict__ parent_int,
                                                     const int* __restrict__ parent_leaf, int* __restrict__ leaf_pos,
                                                     int* __restrict__ node_pos, int* __restrict__ node_rank,
                                                     uint32_t* __restrict__ red) {
    uint32_t dmax = 0;
    for (int e = blockIdx.x * kB + threadIdx.x; e < 2 * n - 1; e += gridDim.x * kB) {
        int ref, node;
        if (e < n) {
            ref = ~e;
            node = parent_leaf[e];
        } else {
            ref = e - n;
            if (ref == 0) {
                node_pos[0] = 0;
                node_rank[0] = 0;
                continue;
            }
            node = parent_int[ref];
        }
        int off = 0, rank = 0;
        uint32_t d = 1;
        for (;;) {
            const int2 ch = child[node];
            if (ch.y == ref && ch.x >= 0) rank += ecount[ch.x];
            if (ch.y == ref) off += ch.x < 0 ? 1 : ncount[ch.x];
            rank += 1;  // the ancestor itself precedes its subtree
            if (node == 0 || d >= 4 * kMaxBinaryDepth) break;
            ref = node;
            node = parent_int[node];
            ++d;
        }
        if (e < n) {
            leaf_pos[e] = off;
            dmax = max(dmax, d);
        } else {
            node_pos[e - n] = off;
            node_rank[e - n] = rank;
        }
    }
    atomicMax(&slot(red)[6], dmax);
}

// Node i lies inside a leaf: it or an ancestor was made a leaf (only
// subtrees of at most kMaxLeafSize primitives can be, so the walk is short).
__device__ __forceinline__ bool in_leaf(int i, const int* __restrict__ ncount, const int* __restrict__ nleaf,
                                        const int* __restrict__ parent_int) {
    for (;;) {
        if (nleaf[i]) return true;
        if (i == 0) return false;
        i = parent_int[i];
        if (ncount[i] > kMaxLeafSize) return false;
    }
}

__global__ __launch_bounds__(kB) void k_ploc_emit(int n, const int2* __restrict__ child,
                                                  const float4* __restrict__ nlo, const float4* __restrict__ nhi,
                                                  const int* __restrict__ ncount, const int* __restrict__ nleaf,
                                                  const int* __restrict__ parent_int, const int* __restrict__ leaf_pos,
                                                  const int* __restrict__ node_pos, const int* __restrict__ node_rank,
                                                  const uint32_t* __restrict__ sorted, const float4* __restrict__ blo,
                                                  const float4* __restrict__ bhi, float4* __restrict__ nodes,
                                                  uint32_t* __restrict__ red) {
    uint32_t nl = 0;
    for (int i = blockIdx.x * kB + threadIdx.x; i < n - 1; i += gridDim.x * kB) {
        if (in_leaf(i, ncount, nleaf, parent_int)) continue;  // part of a leaf of an ancestor
        const int2 ch = child[i];
        const int refs[2] = {ch.x, ch.y};
        float lo[2][3], hi[2][3];
        int ref[2], cnt[2];
        for (int c = 0; c < 2; c++) {
            const int r = refs[c];
            float4 a, b;
            int count, pos;
            bool leaf;
            if (r < 0) {
                const uint32_t p = sorted[~r];
                a = blo[p];
                b = bhi[p];
                count = 1;
                pos = leaf_pos[~r];
                leaf = true;
            } else {
                a = nlo[r];
                b = nhi[r];
                count = ncount[r];
                pos = node_pos[r];
                leaf = nleaf[r] != 0;
            }
            pad(a, b, lo[c], hi[c]);
            if (leaf) {
                ref[c] = ~pos;
                cnt[c] = count;
                nl++;
            } else {
                ref[c] = node_rank[r];
                cnt[c] = 0;
            }
        }
        float4* np = nodes + 4 * (size_t)node_rank[i];
        np[0] = make_float4(lo[0][0], hi[0][0], lo[1][0], hi[1][0]);
        np[1] = make_float4(lo[0][1], hi[0][1], lo[1][1], hi[1][1]);
        np[2] = make_float4(lo[0][2], hi[0][2], lo[1][2], hi[1][2]);
        reinterpret_cast<int4*>(np)[3] = make_int4(ref[0], ref[1], cnt[0], cnt[1]);
    }
    if (nl) atomicAdd(&slot(red)[7], nl);
}

// Triangle of sorted position k goes to its depth-first position.
__global__ __launch_bounds__(kB) void k_ploc_gather(int n, const uint32_t* __restrict__ sorted,
                                                    const int* __restrict__ leaf_pos, const float* __restrict__ pos,
                                                    const uint32_t* __restrict__ idx, float4* __restrict__ tris) {
    for (int k = blockIdx.x * kB + threadIdx.x; k < n; k += gridDim.x * kB) {
        const uint32_t p = sorted[k];
        const uint32_t i0 = idx[3 * p], i1 = idx[3 * p + 1], i2 = idx[3 * p + 2];
        const float p0x = pos[3 * i0], p0y = pos[3 * i0 + 1], p0z = pos[3 * i0 + 2];
        const float e1x = pos[3 * i1] - p0x, e1y = pos[3 * i1 + 1] - p0y, e1z = pos[3 * i1 + 2] - p0z;
        const float e2x = pos[3 * i2] - p0x, e2y = pos[3 * i2 + 1] - p0y, e2z = pos[3 * i2 + 2] - p0z;
        float4* t = tris + 3 * (size_t)leaf_pos[k];
        t[0] = make_float4(p0x, p0y, p0z, e1x);
        t[1] = make_float4(e1y, e1z, e2x, e2y);
        t[2] = make_float4(e2z, __uint_as_float(p), 0.f, 0.f);
    }
}

}  // namespace

dl_status build_bvh_ploc(Ctx* c, dl_accel_stats* stats) {
    const int n = (int)c->nprims;
    if (n <= kMaxLeafSize) return build_small(c, stats);
    Scratch sc{c};
    float4 *blo, *bhi, *clo[2], *chi[2];
    unsigned long long *keys = nullptr, *keys_sorted = nullptr;
    uint32_t *red, *sorted = nullptr, *ids = nullptr;
    int *cref[2], *nn, *leaf_pos, *node_pos, *node_rank;
    int2* sums;
    PlocNodes t;
    PlocState* st;
    sc.want(&blo, n);
    sc.want(&bhi, n);
    for (int b = 0; b < 2; b++) {
        sc.want(&clo[b], n);
        sc.want(&chi[b], n);
        sc.want(&cref[b], n);
    }
    sc.want(&t.child, n);
    sc.want(&t.lo, n);
    sc.want(&t.hi, n);
    sc.want(&t.count, n);
    sc.want(&t.ecount, n);
    sc.want(&t.parent_int, n);
    sc.want(&t.parent_leaf, n);
    sc.want(&t.leaf, n);
    sc.want(&t.cost, n);
    sc.want(&keys, n);
    sc.want(&keys_sorted, n);
    sc.want(&ids, n);
    sc.want(&sorted, n);
    sc.want(&nn, n);
    sc.want(&sums, kPlocChunks);
    sc.want(&leaf_pos, n);
    sc.want(&node_pos, n);
    sc.want(&node_rank, n);
    sc.want(&red, kSlots * kSlotWords);
    sc.want(&st, 2);
    size_t sort_bytes = 0;
    DL_HIP_CHECK(c, hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, keys, keys_sorted, ids, sorted, n, 0, 63,
                                                       c->stream));
    char* temp = nullptr;
    sc.want(&temp, sort_bytes);
    DL_TRY(sc.alloc());
    DL_TRY(grow(c, c->build_nodes, (size_t)(n - 1) * kNodeBytes));
    DL_TRY(resize_exact(c, &c->ds.tris, (size_t)n * kTriBytes));
    float4 *const pn = (float4*)c->build_nodes.p, *const pt = c->ds.tris;

    const int grid = std::max(1, c->num_cus) * 8;
    DL_HIP_CHECK(c, hipEventRecord(c->ev0, c->stream));
    k_init_slots<<<1, kSlots, 0, c->stream>>>(red);
    k_prim_boxes<<<grid, kB, 0, c->stream>>>(c->ds.pos, c->ds.idx, (uint32_t)n, blo, bhi, red);
    k_keys63<<<grid, kB, 0, c->stream>>>(blo, bhi, (uint32_t)n, red, keys, ids);
    // stable: equal codes keep increasing primitive ids
    DL_HIP_CHECK(c, hipcub::DeviceRadixSort::SortPairs(temp, sort_bytes, keys, keys_sorted, ids, sorted, n, 0, 63,
                                                       c->stream));
    k_ploc_init<<<grid, kB, 0, c->stream>>>(n, sorted, blo, bhi, cref[0], clo[0], chi[0], st);
    PlocState now{n, n - 2};
    int cur = 0;
    while (now.count > kPlocTail) {
        // (the count only falls, so grids for the last one read are enough)
        const int blocks = (now.count + kB - 1) / kB;
        for (int k = 0; k < kPlocBatch; k++, cur ^= 1) {
            k_ploc_nn<<<std::min(blocks, grid), kB, 0, c->stream>>>(st + cur, clo[cur], chi[cur], nn);
            k_ploc_count<<<std::min(blocks, kPlocChunks), kB, 0, c->stream>>>(st + cur, nn, sums);
            k_ploc_merge<<<std::min(blocks, kPlocChunks), kB, 0, c->stream>>>(
                st + cur, st + (cur ^ 1), nn, sums, cref[cur], clo[cur], chi[cur], cref[cur ^ 1], clo[cur ^ 1],
                chi[cur ^ 1], t);
        }
        const int before = now.count;
        DL_HIP_CHECK(c, hipMemcpyAsync(&now, st + cur, sizeof(now), hipMemcpyDeviceToHost, c->stream));
        DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
        DL_HIP_CHECK(c, hipGetLastError());
        if (now.count < 1 || now.count >= before || now.top != now.count - 2)
            return set_error(c, DL_ERR_STATE, "PLOC merge step inconsistent");
    }
    k_ploc_tail<<<1, kPlocTailThreads, 0, c->stream>>>(st + cur, cref[cur], clo[cur], chi[cur], t);
    DL_HIP_CHECK(c, hipMemcpyAsync(&now, st + cur, sizeof(now), hipMemcpyDeviceToHost, c->stream));
    DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    DL_HIP_CHECK(c, hipGetLastError());
    if (now.count != 1 || now.top != -1) return set_error(c, DL_ERR_STATE, "PLOC node count mismatch");
    k_ploc_offsets<<<grid, kB, 0, c->stream>>>(n, t.child, t.count, t.ecount, t.parent_int, t.parent_leaf, leaf_pos,
                                               node_pos, node_rank, red);
    k_ploc_emit<<<grid, kB, 0, c->stream>>>(n, t.child, t.lo, t.hi, t.count, t.leaf, t.parent_int, leaf_pos, node_pos,
                                            node_rank, sorted, blo, bhi, pn, red);
    k_ploc_gather<<<grid, kB, 0, c->stream>>>(n, sorted, leaf_pos, c->ds.pos, c->ds.idx, pt);
    DL_HIP_CHECK(c, hipGetLastError());
    DL_HIP_CHECK(c, hipEventRecord(c->ev1, c->stream));
    int emitted = 0;
    DL_HIP_CHECK(c, hipMemcpyAsync(&emitted, t.ecount, sizeof(int), hipMemcpyDeviceToHost, c->stream));  // root = node 0
    DL_TRY(read_slots(c, red, &stats->max_depth, &stats->num_leaves));
    float ms = 0.f;
    DL_HIP_CHECK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    stats->num_nodes = c->num_binary = (uint32_t)emitted;
    stats->build_ms = ms;
    if (stats->max_depth > (uint32_t)kMaxBinaryDepth) {
        c->bvh_too_deep = true;
        return set_error(c, DL_ERR_STATE, "PLOC tree deeper than the traversal stack");
    }
    return DL_OK;
}

// ===========================================================================
// Collapse of a binary BVH (any builder) into 4-wide nodes: every 4-wide
// node takes a binary node's two children and opens the internal child of
// largest surface area (lowest slot on ties) until it has four children or
// only leaves.  Top-down, one level per step: the frontier holds binary
// nodes that become 4-wide nodes; their internal children get consecutive
// indices (prefix sum), so the 4-wide nodes are in breadth-first order and
// frontier entry i of a level is node start + i.  A level is two kernels (the
// internal children per chunk of the frontier; the nodes, quantised and
// written in place, and the next frontier) which take the level's size from
// device memory, so that levels follow each other without the host.  (With
// library scans, a read of the count per level and 128-byte nodes quantised by
// a pass of their own, the 14 levels of 2,097,152 triangles were 70 launches
// and 14 waits.)
// ===========================================================================
namespace {

struct Cand {
    float lo[3], hi[3];
    int ref, cnt;
};

__device__ __forceinline__ void bin_child(const float4* __restrict__ bn, int b, int k, Cand& c) {
    const float4* np = bn + 4 * (size_t)b;
    const float4 r0 = np[0], r1 = np[1], r2 = np[2];
    const int4 r3 = reinterpret_cast<const int4*>(np)[3];
    c.lo[0] = k ? r0.z : r0.x;
    c.hi[0] = k ? r0.w : r0.y;
    c.lo[1] = k ? r1.z : r1.x;
    c.hi[1] = k ? r1.w : r1.y;
    c.lo[2] = k ? r2.z : r2.x;
    c.hi[2] = k ? r2.w : r2.y;
    c.ref = k ? r3.y : r3.x;
    c.cnt = k ? r3.w : r3.z;
}

__device__ __forceinline__ float cand_area(const Cand& c) {
    const float dx = c.hi[0] - c.lo[0], dy = c.hi[1] - c.lo[1], dz = c.hi[2] - c.lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// Children of the 4-wide node made from binary node b; returns how many.
__device__ __forceinline__ int gather4(const float4* __restrict__ bn, int b, Cand (&c)[4]) {
    bin_child(bn, b, 0, c[0]);
    bin_child(bn, b, 1, c[1]);
    int m = 2;
    // (constant indices only: a dynamic one puts the children in scratch memory)
#pragma unroll
    for (int step = 2; step < 4; ++step) {
        int best = -1, r = 0;
        float ba = -1.0f;
#pragma unroll
        for (int k = 0; k < step; ++k)
            if (c[k].ref >= 0) {
                const float a = cand_area(c[k]);
                if (a > ba) {
                    ba = a;
                    best = k;
                    r = c[k].ref;
                }
            }
        if (m < step || best < 0) continue;
        bin_child(bn, r, 1, c[step]);
        Cand first;
        bin_child(bn, r, 0, first);
#pragma unroll
        for (int k = 0; k < step; ++k)
            if (k == best) c[k] = first;
        ++m;
    }
    return m;
}

// Quantises a 4-wide node with float child boxes (q: lo.x, hi.x, lo.y, hi.y,
// lo.z, hi.z of children 0..3) into the 64-byte traversal layout.  Per axis
// the origin is the least lo of the used children and the step the smallest
// power of two whose 255 steps span them; qlo / qhi are rounded outward and
// then checked with the traversal's own decode (origin + q * step in
// binary32), stepping down / up until the decoded box contains the float box
// (a wider step when 255 steps do not reach), so quantisation never shrinks a
// box.
__device__ float q_decode(float o, uint32_t q, float s) { return o + (float)q * s; }

__device__ __forceinline__ void quantize4(const float (&b)[6][4], const int (&refs)[4], const int (&cnts)[4],
                                          float4* __restrict__ dst) {
    bool used[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) used[j] = !(refs[j] == ~0 && cnts[j] == 0);
    float origin[3];
    uint32_t ebits[3], qlo[3] = {0, 0, 0}, qhi[3] = {0, 0, 0};
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        float o = INFINITY, m = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (used[j]) {
                o = fminf(o, b[2 * ax][j]);
                m = fmaxf(m, b[2 * ax + 1][j]);
            }
        if (!(o <= m)) o = m = 0.0f;
        origin[ax] = o;
        // smallest exponent whose 255 steps cover m - o
        const double ext = (double)m - (double)o;
        int e = -126;
        if (ext > 0.0) {
            int ex;
            (void)frexp(ext / 255.0, &ex);  // ext / 255 < 2^ex
            e = max(-126, ex);
        }
        uint32_t lo4 = 0, hi4 = 0;
        for (;; ++e) {
            const float s = __uint_as_float((uint32_t)(e + 127) << 23);
            bool fits = true;
            lo4 = hi4 = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t ql = 0, qh = 0;
                if (used[j]) {
                    const float lo = b[2 * ax][j], hi = b[2 * ax + 1][j];
                    double fl = floor(((double)lo - (double)o) / (double)s);
                    double fh = ceil(((double)hi - (double)o) / (double)s);
                    ql = (uint32_t)fmin(fmax(fl, 0.0), 255.0);
                    qh = (uint32_t)fmin(fmax(fh, 0.0), 255.0);
                    while (ql > 0 && q_decode(o, ql, s) > lo) --ql;
                    while (qh < 255 && q_decode(o, qh, s) < hi) ++qh;
                    if (q_decode(o, ql, s) > lo || q_decode(o, qh, s) < hi) fits = false;
                }
                lo4 |= ql << (8 * j);
                hi4 |= qh << (8 * j);
            }
            if (fits || e >= 127) break;
        }
        ebits[ax] = (uint32_t)(e + 127);
        qlo[ax] = lo4;
        qhi[ax] = hi4;
    }
    uint32_t c4 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) c4 |= ((uint32_t)cnts[j] & 0xffu) << (8 * j);
    dst[0] = make_float4(origin[0], origin[1], origin[2], __uint_as_float(ebits[0] | ebits[1] << 8 | ebits[2] << 16));
    reinterpret_cast<uint4*>(dst)[1] = make_uint4(qlo[0], qhi[0], qlo[1], qhi[1]);
    reinterpret_cast<uint4*>(dst)[2] = make_uint4(qlo[2], qhi[2], c4, 0u);
    reinterpret_cast<int4*>(dst)[3] = make_int4(refs[0], refs[1], refs[2], refs[3]);
}

struct C4State {
    int nf, start;  // the level's frontier and its first node
    int levels;     // levels done
    int bad;        // more nodes than the binary tree has
};
constexpr int kC4Batch = 8;  // levels launched between two reads of the state

__global__ void k_c4_init(int* __restrict__ fbin, C4State* __restrict__ st) {
    fbin[0] = 0;
    *st = C4State{1, 0, 0, 0};
}

__global__ __launch_bounds__(kB) void k_c4_count(const C4State* __restrict__ st, const float4* __restrict__ bn,
                                                 const int* __restrict__ fbin, int* __restrict__ sums) {
    __shared__ int s_part[kB / 64];
    const int nf = st->nf, chunk = ploc_chunk(nf);
    if ((long long)blockIdx.x * chunk >= nf) return;
    const int c0 = blockIdx.x * chunk, c1 = min(nf, c0 + chunk);
    int k = 0;
    for (int i = c0 + threadIdx.x; i < c1; i += kB) {
        Cand c[4];
        const int m = gather4(bn, fbin[i], c);
#pragma unroll
        for (int j = 0; j < 4; ++j) k += j < m && c[j].ref >= 0 ? 1 : 0;
    }
    for (int off = 32; off > 0; off >>= 1) k += __shfl_xor(k, off);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        k = 0;
        for (int w = 0; w < kB / 64; w++) k += s_part[w];
        sums[blockIdx.x] = k;
    }
}

__global__ __launch_bounds__(kB) void k_c4_emit(const C4State* __restrict__ st, C4State* __restrict__ next,
                                                const float4* __restrict__ bn, const int* __restrict__ fbin,
                                                const int* __restrict__ sums, int cap, float4* __restrict__ out,
                                                int* __restrict__ nbin) {
    __shared__ int s_before[kB / 64];
    __shared__ uint32_t s_wave[kB / 64];
    const C4State s = *st;
    const int chunk = ploc_chunk(s.nf);
    if (s.nf == 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *next = s;
        return;
    }
    if ((long long)blockIdx.x * chunk >= s.nf) return;
    int before = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += kB) before += sums[k];
    for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off);
    if ((threadIdx.x & 63) == 0) s_before[threadIdx.x >> 6] = before;
    __syncthreads();
    before = 0;
    for (int w = 0; w < kB / 64; w++) before += s_before[w];
    const int base = s.start + s.nf;  // node of the next frontier's first entry
    const int c0 = blockIdx.x * chunk, c1 = min(s.nf, c0 + chunk);
    for (int b = c0; b < c1; b += kB) {
        const int i = b + threadIdx.x;
        Cand c[4];
        int m = 0;
        uint32_t mine = 0;
        if (i < c1) {
            m = gather4(bn, fbin[i], c);
#pragma unroll
            for (int j = 0; j < 4; ++j) mine += j < m && c[j].ref >= 0 ? 1u : 0u;
        }
        uint32_t total;
        int k = before + (int)block_exclusive<kB / 64>(mine, s_wave, total);
        before += (int)total;
        if (i >= c1) continue;
        float q[6][4];
        int ref[4], cnt[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < m) {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    q[2 * a][j] = c[j].lo[a];
                    q[2 * a + 1][j] = c[j].hi[a];
                }
                if (c[j].ref >= 0) {
                    if (base + k < cap) nbin[k] = c[j].ref;
                    ref[j] = base + k;
                    cnt[j] = 0;
                    ++k;
                } else {
                    ref[j] = c[j].ref;
                    cnt[j] = c[j].cnt;
                }
            } else {  // unused slot: an empty leaf
#pragma unroll
                for (int a = 0; a < 6; ++a) q[a][j] = 0.0f;
                ref[j] = ~0;
                cnt[j] = 0;
            }
        }
        quantize4(q, ref, cnt, out + 4 * (size_t)(s.start + i));
    }
    if (c1 == s.nf && threadIdx.x == 0) {
        const bool bad = base + before > cap;
        *next = C4State{bad ? 0 : before, base, s.levels + 1, bad ? 1 : 0};
    }
}

}  // namespace

// The 4-wide nodes of the scene from the binary nodes of its build
// (num_binary, root 0); stats get the 4-wide node count and depth.
dl_status collapse_bvh4(Ctx* c, dl_accel_stats* stats) {
    const int cap = (int)std::max<uint32_t>(1, c->num_binary);
    const float4* const bin = (const float4*)c->build_nodes.p;
    Scratch sc{c};
    int *fbin[2], *sums;
    float4* out;
    C4State* st;
    for (int b = 0; b < 2; b++) sc.want(&fbin[b], cap);
    sc.want(&sums, kPlocChunks);
    sc.want(&out, (size_t)cap * (kNode4Bytes / sizeof(float4)));
    sc.want(&st, 2);
    DL_TRY(sc.alloc());
    const int grid = std::min(kPlocChunks, (cap + kB - 1) / kB);
    k_c4_init<<<1, 1, 0, c->stream>>>(fbin[0], st);
    C4State now{1, 0, 0, 0};
    int cur = 0;
    while (now.nf > 0) {
        for (int k = 0; k < kC4Batch; k++, cur ^= 1) {
            k_c4_count<<<grid, kB, 0, c->stream>>>(st + cur, bin, fbin[cur], sums);
            k_c4_emit<<<grid, kB, 0, c->stream>>>(st + cur, st + (cur ^ 1), bin, fbin[cur], sums, cap, out,
                                                  fbin[cur ^ 1]);
        }
        DL_HIP_CHECK(c, hipMemcpyAsync(&now, st + cur, sizeof(now), hipMemcpyDeviceToHost, c->stream));
        DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
        DL_HIP_CHECK(c, hipGetLastError());
        if (now.bad || now.levels + (now.nf > 0 ? 1 : 0) > kMaxBinaryDepth)
            return set_error(c, DL_ERR_STATE, "4-wide BVH collapse exceeded its bounds");
    }
    const size_t bytes = (size_t)now.start * kNode4Bytes;
    if (resize_exact(c, &c->ds.nodes, bytes) != DL_OK)
        return set_error(c, DL_ERR_OOM, "out of device memory for the 4-wide BVH");
    DL_HIP_CHECK(c, hipMemcpyAsync(c->ds.nodes, out, bytes, hipMemcpyDeviceToDevice, c->stream));
    DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    stats->num_nodes = (uint32_t)now.start;
    stats->max_depth = (uint32_t)now.levels;
    return DL_OK;
}

dl_status build_bvh_gpu(Ctx* c, dl_accel_stats* stats, int method) {
    return method == DL_BUILD_GPU_LBVH ? build_bvh_lbvh(c, stats) : build_bvh_ploc(c, stats);
}

}  // namespace dl
