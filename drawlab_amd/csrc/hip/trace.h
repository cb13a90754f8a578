// BVH traversal for gfx950: one ray per lane, 4-wide nodes (bvh_layout.h:
// one 64-byte node per visit, four slab tests, the nearest hit internal
// child next and the others stacked farthest first), persistent lanes with
// per-lane ray refill,
// per-lane traversal stack staged in LDS with a lane-interleaved layout
// (entry k of lane l at stack[k * blockDim + l]: every wave touches 64
// consecutive dwords whatever the stack depths, so the accesses are
// bank-conflict free).
//
// Closest hit: the binary32 Moller-Trumbore test of the reference
// (src/tracer/mesh/mesh.cpp:180-220), accepting t in [tmin, t_best] and
// keeping the lowest primitive id on equal t, so the result equals the
// brute-force argmin over all triangles bit-for-bit.  Any hit: the first
// accepted triangle (src/tracer/accel/octree.cpp:112-133).
#pragma once
#include "../bvh_layout.h"
#include "../work_split.h"
#include "backend.h"
#include "dl_math.h"

namespace dl {

constexpr int kTraceBlock = kTraceBlockHost;
// Slack on the far slab distance: absorbs the rounding of the slab
// arithmetic and of Moller-Trumbore's t (Ize, "Robust BVH ray traversal", 2013).
constexpr float kFarSlack = 1.0f + 1.0f / 65536.0f;

struct BvhView {
    const float4* __restrict__ nodes;
    const float4* __restrict__ tris;
};

struct TraceCounters {
    uint32_t nodes = 0;
    uint32_t tris = 0;
};

// Lane-private traversal stack: entries [0, kLdsStack) in LDS
// (lane-interleaved), [kLdsStack, kMaxStack) in a global overflow buffer
// (entry k of grid thread g at ovf[k * grid_threads + g], coalesced).
struct LaneStack {
    int* __restrict__ lds;
    int lane, stride;
    int* __restrict__ ovf;
    uint32_t ostride;
    // Pushes a, b, c in this order, each only if its flag is set.  While the
    // three cannot reach the overflow they are stored without a branch (a
    // store whose flag is clear leaves the entry to the next one).  No tree is
    // deeper than kMaxStack, so the last test never fails; it keeps every
    // access in bounds regardless.
    __device__ __forceinline__ void push3(int& sp, int a, bool pa, int b, bool pb, int c, bool pc) {
        if (sp <= kLdsStack - 3) {
            lds[sp * stride + lane] = a;
            sp += pa ? 1 : 0;
            lds[sp * stride + lane] = b;
            sp += pb ? 1 : 0;
            lds[sp * stride + lane] = c;
            sp += pc ? 1 : 0;
        } else {
#pragma unroll 1
            for (int k = 0; k < 3; k++) {
                const int v = k == 0 ? a : k == 1 ? b : c;
                if (!(k == 0 ? pa : k == 1 ? pb : pc)) continue;
                if (sp < kLdsStack)
                    lds[sp * stride + lane] = v;
                else if (sp < kMaxStack)
                    ovf[(size_t)(sp - kLdsStack) * ostride] = v;
                else
                    break;
                ++sp;
            }
        }
    }
    __device__ __forceinline__ int pop(int& sp) {
        --sp;
        return sp < kLdsStack ? lds[sp * stride + lane] : ovf[(size_t)(sp - kLdsStack) * ostride];
    }
};

// Compare-exchange of (key, ref) pairs: smaller key first.
__device__ __forceinline__ void cswap(float& ka, int& ra, float& kb, int& rb) {
    const bool s = kb < ka;
    const float k = s ? kb : ka;
    kb = s ? ka : kb;
    ka = k;
    const int r = s ? rb : ra;
    rb = s ? ra : rb;
    ra = r;
}

// One plane of a child box: its byte of `word` (children 0..3 in bytes 0..3)
// as origin + q * step.  q * step is exact (an 8-bit integer times a power of
// two), so the fused multiply-add rounds once, exactly like the separate
// product and sum the quantiser checked.
__device__ __forceinline__ float qplane(uint32_t word, int sh, float step, float origin) {
    return __builtin_fmaf((float)((word >> sh) & 0xffu), step, origin);
}
// Slab test of the child at bit `sh` of the words of its near and far planes
// (per axis the lo planes are the near ones for a direction whose reciprocal
// is positive, else the hi planes: chosen once per node as whole words, which
// takes 6 selects instead of 24 minima and maxima of plane distances): entry
// distance n, and whether [n, far] meets [tmin, tmax] (far widened by
// kFarSlack).
__device__ __forceinline__ bool slab_q(const uint32_t (&nw)[3], const uint32_t (&fw)[3], int sh, const vec3& step,
                                       const vec3& org, const vec3& o, const vec3& rcp, float tmin, float tmax,
                                       float& n) {
    const float n0 = (qplane(nw[0], sh, step.x, org.x) - o.x) * rcp.x, f0 = (qplane(fw[0], sh, step.x, org.x) - o.x) * rcp.x;
    const float n1 = (qplane(nw[1], sh, step.y, org.y) - o.y) * rcp.y, f1 = (qplane(fw[1], sh, step.y, org.y) - o.y) * rcp.y;
    const float n2 = (qplane(nw[2], sh, step.z, org.z) - o.z) * rcp.z, f2 = (qplane(fw[2], sh, step.z, org.z) - o.z) * rcp.z;
    n = fmaxf(fmaxf(n0, n1), fmaxf(n2, tmin));
    const float f = fminf(fminf(f0, f1), fminf(f2, tmax));
    return n <= f * kFarSlack;
}

// Moller-Trumbore on a pre-gathered triangle; returns false on a miss.
// Branch-free: every quantity is computed and the reference's early-out
// tests (mesh.cpp:195, 204, 213) are combined into the returned predicate,
// which accepts exactly the rays the early-out sequence accepts.  The triangle
// is therefore fetched by three loads issued together.
__device__ __forceinline__ bool mt_test(const float4& a, const float4& b, const float4& c, const vec3& o,
                                        const vec3& d, float& u, float& v, float& t) {
    const vec3 p0 = v3(a.x, a.y, a.z);
    const vec3 e1 = v3(a.w, b.x, b.y);
    const vec3 e2 = v3(b.z, b.w, c.x);
    const vec3 pvec = cross(d, e2);
    const float det = dot(e1, pvec);
    const float inv = 1.0f / det;
    const vec3 tvec = sub(o, p0);
    u = dot(tvec, pvec) * inv;
    const vec3 qvec = cross(tvec, e1);
    v = dot(d, qvec) * inv;
    t = dot(e2, qvec) * inv;
    const bool parallel = det > -1e-8f && det < 1e-8f;
    const bool out_u = u < 0.0f || u > 1.0f;
    const bool out_v = v < 0.0f || u + v > 1.0f;
    return !(parallel | out_u | out_v);
}

// Adds v of every lane of a converged wave to *dst with one atomic (none
// when the sum is 0: the waves of a short launch mostly traced nothing).
__device__ __forceinline__ void wave_add(unsigned long long* dst, uint32_t v) {
    unsigned long long sum = v;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (__lane_id() == 0 && sum != 0) atomicAdd(dst, sum);
}

// Relative VALU cost of the traversal's two step kinds, triangle step :
// node visit (2 : 5 measured best on the 2M-triangle displaced-sphere
// render with one triangle per step, whose instruction count to a node
// visit's is about 130 : 300; with two triangles per step 1 : 2, 3 : 5 and
// 4 : 5 measure within 0.5% of it).
constexpr uint32_t kTriCost = 2, kNodeCost = 5;

// How a persistent grid's waves share n work slots (work_split.h): slots
// [0, base) are spread evenly over them, the others handed out in chunks of
// `unit` slots.  The chunks are dealt in turn to kWorkGroups groups of blocks
// (one per block in a smaller grid), and a wave claims its group's next chunk
// with one atomic on the group's counter (zero at launch).  One counter for
// all waves would serialise: its atomics pass at about 55 per microsecond
// (measured), so the 8192 waves of a full grid claiming once each would
// already take 150 us.  The blocks of a group run on one XCD (block b runs on
// XCD b mod 8), whose L2 holds their counter.
struct TraceWork : WorkSplit {
    uint32_t* counter;  // of this wave's group
};
__device__ __forceinline__ TraceWork trace_work(uint32_t* counters, uint32_t n, uint32_t wave, uint32_t waves) {
    TraceWork w;
    static_cast<WorkSplit&>(w) = split_work(n, wave, waves, blockIdx.x, gridDim.x);
    w.counter = counters + w.group * kWorkStride;
    return w;
}

// This wave's index in the grid and the grid's number of waves.
__device__ __forceinline__ uint32_t grid_wave() {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
}
__device__ __forceinline__ uint32_t grid_waves() { return gridDim.x * (blockDim.x >> 6); }

// One ray in flight: a lane's traversal state and its two kinds of step.
struct RayState {
    vec3 o, d, rcp;
    float tmin, best_t, bu, bv;
    uint32_t best;
    int sp, cur;
    // triangles of the last visited node's hit leaves: triangle j lies at
    // j + lb[c], c the first slot whose running total of triangles exceeds j
    // (totals of slots 0, 0-1 and 0-2 packed in lend, 10 bits each: a leaf
    // holds at most kMaxLeafCount = 255), their number and the next one to
    // test; `last`: no node left to visit once they are tested
    int4 lb;
    uint32_t lend;
    int ltri, lj;
    bool last;

    __device__ __forceinline__ void clear() {
        o = d = rcp = v3(0, 0, 0);
        tmin = best_t = bu = bv = 0.f;
        best = 0xffffffffu;
        sp = cur = 0;
        lb = make_int4(0, 0, 0, 0);
        lend = 0;
        ltri = lj = 0;
        last = false;
    }

    // Starts the ray in o, d, tmin at node `root`.  False for a ray that holds
    // a NaN: it makes every Moller-Trumbore comparison false (no hit), but
    // would pass every slab test, so it is finished at once as a miss.
    __device__ __forceinline__ bool start(float tmax, int root) {
        rcp = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
        best_t = tmax;
        best = 0xffffffffu;
        bu = bv = 0.0f;
        sp = 0;
        cur = root;
        ltri = lj = 0;
        last = false;
        return !(isnan(o.x) || isnan(o.y) || isnan(o.z) || isnan(d.x) || isnan(d.y) || isnan(d.z) || isnan(tmin) ||
                 isnan(tmax));
    }

    // The next one or two triangles of the last visit's hit leaves, in slot
    // order: both fetched before the first is tested, so a pair costs one
    // dependent wait; the second is accepted against the best t the first
    // left, as a sequential loop would.  any: stops at the first accepted
    // triangle, and returns true for it.
    __device__ __forceinline__ bool test_triangles(const BvhView& bvh, bool any) {
        const int e0 = (int)(lend & 0x3ffu), e1 = (int)((lend >> 10) & 0x3ffu), e2 = (int)(lend >> 20);
        const int j = lj;
        const bool two = j + 1 < ltri;
        const int j1 = two ? j + 1 : j;
        int k0 = lb.w, k1 = lb.w;
        k0 = j < e2 ? lb.z : k0;
        k1 = j1 < e2 ? lb.z : k1;
        k0 = j < e1 ? lb.y : k0;
        k1 = j1 < e1 ? lb.y : k1;
        k0 = (j < e0 ? lb.x : k0) + j;
        k1 = (j1 < e0 ? lb.x : k1) + j1;
        const float4* tp0 = bvh.tris + 3 * k0;
        const float4* tp1 = bvh.tris + 3 * k1;
        const float4 ta = tp0[0], tb = tp0[1], tc = tp0[2];
        const float4 sa = tp1[0], sb = tp1[1], sc = tp1[2];
        float u, v, t;
        const bool h0 = mt_test(ta, tb, tc, o, d, u, v, t) && t >= tmin && t <= best_t;
        lj++;
        if (any && h0) return true;
        if (!any && h0) accept(t, u, v, __float_as_uint(tc.y));
        if (two) {
            lj++;
            if (mt_test(sa, sb, sc, o, d, u, v, t) && t >= tmin && t <= best_t) {
                if (any) return true;
                accept(t, u, v, __float_as_uint(sc.y));
            }
        }
        return false;
    }
    __device__ __forceinline__ void accept(float t, float u, float v, uint32_t id) {
        if (t < best_t || id < best) {
            best_t = t;
            best = id;
            bu = u;
            bv = v;
        }
    }

    // Visits node cur: its hit leaves' triangles become the ones to test, the
    // nearest hit internal child (or a stack pop) the next node.
    __device__ __forceinline__ void visit_node(const BvhView& bvh, LaneStack& stk) {
        const float4* np = bvh.nodes + 4 * (size_t)cur;
        const float4 r0 = np[0];
        const uint4 r1 = reinterpret_cast<const uint4*>(np)[1];
        const uint4 r2 = reinterpret_cast<const uint4*>(np)[2];
        const int4 ref = reinterpret_cast<const int4*>(np)[3];
        // child boxes: origin + q * step (q * step exact, one rounding)
        const uint32_t eb = __float_as_uint(r0.w);
        const vec3 step = v3(__uint_as_float((eb & 0xffu) << 23), __uint_as_float(((eb >> 8) & 0xffu) << 23),
                             __uint_as_float(((eb >> 16) & 0xffu) << 23));
        const vec3 org = v3(r0.x, r0.y, r0.z);
        const bool px = rcp.x >= 0.0f, py = rcp.y >= 0.0f, pz = rcp.z >= 0.0f;
        const uint32_t nw[3] = {px ? r1.x : r1.y, py ? r1.z : r1.w, pz ? r2.x : r2.y};
        const uint32_t fw[3] = {px ? r1.y : r1.x, py ? r1.w : r1.z, pz ? r2.y : r2.x};
        float n0, n1, n2, n3;
        const bool h0 = slab_q(nw, fw, 0, step, org, o, rcp, tmin, best_t, n0);
        const bool h1 = slab_q(nw, fw, 8, step, org, o, rcp, tmin, best_t, n1);
        const bool h2 = slab_q(nw, fw, 16, step, org, o, rcp, tmin, best_t, n2);
        const bool h3 = slab_q(nw, fw, 24, step, org, o, rcp, tmin, best_t, n3);
        // triangles of the hit leaf children, tested in the next steps (the
        // closest hit is the minimum over (t, id), so their order does not
        // change it)
        const int c0n = (h0 && ref.x < 0) ? (int)(r2.z & 0xffu) : 0;
        const int c1n = (h1 && ref.y < 0) ? (int)((r2.z >> 8) & 0xffu) : 0;
        const int c2n = (h2 && ref.z < 0) ? (int)((r2.z >> 16) & 0xffu) : 0;
        const int c3n = (h3 && ref.w < 0) ? (int)(r2.z >> 24) : 0;
        const int e1 = c0n + c1n, e2 = e1 + c2n;
        lend = (uint32_t)c0n | ((uint32_t)e1 << 10) | ((uint32_t)e2 << 20);
        lb = make_int4(~ref.x, ~ref.y - c0n, ~ref.z - e1, ~ref.w - e2);
        ltri = e2 + c3n;
        lj = 0;
        // hit internal children: keys = entry distances (+inf: not taken),
        // sorted by a 5-exchange network; the nearest is visited next and the
        // others are stacked farthest first
        float k0 = (h0 && ref.x >= 0) ? n0 : INFINITY, k1 = (h1 && ref.y >= 0) ? n1 : INFINITY;
        float k2 = (h2 && ref.z >= 0) ? n2 : INFINITY, k3 = (h3 && ref.w >= 0) ? n3 : INFINITY;
        int c0 = ref.x, c1 = ref.y, c2 = ref.z, c3 = ref.w;
        cswap(k0, c0, k1, c1);
        cswap(k2, c2, k3, c3);
        cswap(k0, c0, k2, c2);
        cswap(k1, c1, k3, c3);
        cswap(k1, c1, k2, c2);
        if (k0 != INFINITY) {
            stk.push3(sp, c3, k3 != INFINITY, c2, k2 != INFINITY, c1, k1 != INFINITY);
            cur = c0;
        } else if (sp == 0) {
            last = true;
        } else {
            cur = stk.pop(sp);
        }
    }
};

// Which kind of step a wave takes next: the lanes whose next step is a
// triangle test and those whose next step is a node visit would otherwise run
// both branches every iteration under partial masks.  Triangle steps run when
// enough lanes wait for one (a triangle step costs about kTriCost / kNodeCost
// of a node visit); the other lanes hold their step, so every ray still makes
// its own sequence of visits and tests.
__device__ __forceinline__ bool wave_tests_triangles(bool active, bool tri_step) {
    const uint32_t ntri = (uint32_t)__popcll(__ballot(active && tri_step));
    const uint32_t nnode = (uint32_t)__popcll(__ballot(active && !tri_step));
    return ntri != 0 && ntri * kNodeCost >= nnode * kTriCost;
}

// Persistent traversal with per-lane ray refill.  Every lane of a wave stays
// in the loop until the wave has run out of rays; lanes whose rays finished
// start the wave's next rays as soon as enough of them wait, so a wave never
// idles behind its slowest ray.  A wave holds a chunk of up to 64 consecutive
// slots, their entries loaded together (one per lane); while it works on it,
// the claim of the next chunk is already on its way.  (With lane g taking
// rays g, g + G, g + 2G, ... of the queue instead, a launch waited for the
// waves that chance gave the longest rays, CUs idle a quarter of the time,
// and the rays a wave had in flight lay far apart: 4.19M diffuse-bounce rays
// against 2M triangles took 1.36 ms, now 0.81 ms, of which the branch-free
// near / far planes, triangle indices and pushes are the smaller part.)
//
// A step visits one node, or tests the next one or two of the triangles of
// the leaves the lane's last node visit hit.  A node visit decides the next
// node (the nearest hit internal child, or a stack pop) with the best t of
// that moment, then the lane works through that visit's triangles, two per
// step, before it visits the next node -- the sequence of node visits and
// triangle tests of a ray is the one a node-by-node loop makes (and the CPU
// replay follows), but a wave does not wait at every node for its lane with
// the most leaf triangles: a pair of triangle tests costs one step of the
// lane that needs it, one dependent fetch.  Each iteration the wave takes steps
// of one kind: the lanes whose next step is of that kind take it, the
// others hold theirs.
//
// IO provides: kRefillMin, kRefillMinAny (lanes of a wave that start new
// rays together, for closest-hit and any-hit queries: a refill waits on the
// ray's loads, so a wave whose loads take long refills once that many of its
// lanes are idle, or none is busy, rather than at every finished ray),
// entry(slot) (the ray of work slot `slot`), load(e, o, d,
// tmin, tmax), root(e) (the node traversal starts from), store_hit(e, prim,
// t, u, v, nodes, tris) for closest hits and store_occ(e, occluded, nodes,
// tris) for any-hit queries, e being an entry.  With kResolve an any-hit
// query has no occlusion store: for every ray that finished unoccluded the
// lane calls resolve_load(e, a, b) and resolve_store(e, a, b) at the wave's
// next refill, so those loads wait together with the next rays'.
template <bool ANY, bool COUNT, class IO>
__device__ __forceinline__ void traverse_persistent(const BvhView& bvh, const TraceWork& work, LaneStack& stk, IO& io,
                                                    TraceCounters& total) {
    const uint32_t lane = __lane_id();
    const uint32_t n = work.n;
    // the wave's chunk: slots pos .. len - 1 of its entries are still to start
    uint32_t pos = 0, len = work.count;
    uint32_t ent = lane < len ? io.entry(work.first + lane) : 0u;
    bool more = work.base < n;  // slots may be left to claim
    uint32_t claim = 0;
    auto claim_next = [&]() {
        if (lane == 0) claim = atomicAdd(work.counter, 1u);
    };
    if (more) claim_next();
    uint32_t ray = 0;
    bool active = false;
    RayState r;
    r.clear();
    bool pend = false;  // (kResolve) the lane's finished ray is unoccluded and not yet resolved
    TraceCounters cnt;
    for (;;) {
        if (pos == len && more) {
            const uint32_t b = chunk_start(work, (uint32_t)__builtin_amdgcn_readfirstlane((int)claim));
            if (b < n) {
                pos = 0;
                len = min(work.unit, n - b);
                ent = lane < len ? io.entry(b + lane) : 0u;
                claim_next();
            } else {
                more = false;
            }
        }
        const unsigned long long busy = __ballot(active);
        const uint32_t refill_min = ANY ? IO::kRefillMinAny : IO::kRefillMin;
        const uint32_t idle = 64u - (uint32_t)__popcll(busy);
        if (pos < len && idle >= refill_min) {
            const uint32_t at = pos + (uint32_t)__builtin_amdgcn_mbcnt_hi(
                                          ~(uint32_t)(busy >> 32), __builtin_amdgcn_mbcnt_lo(~(uint32_t)busy, 0));
            const uint32_t e = (uint32_t)__shfl((int)ent, (int)(at & 63u));
            if (!active) {
                const uint32_t fin = ray;
                const bool resolve = ANY && IO::kResolve && pend;
                float4 ra, rb;
                if (resolve) {
                    io.resolve_load(fin, ra, rb);
                    pend = false;
                }
                if (at < len) {
                    ray = e;
                    float tmax;
                    io.load(ray, r.o, r.d, r.tmin, tmax);
                    cnt = TraceCounters();
                    active = r.start(tmax, io.root(ray));
                    if (!active) {
                        if (ANY && IO::kResolve)
                            pend = true;
                        else if (ANY)
                            io.store_occ(ray, false, 0, 0);
                        else
                            io.store_hit(ray, r.best, r.best_t, 0.0f, 0.0f, 0, 0);
                    }
                }
                if (resolve) io.resolve_store(fin, ra, rb);
            }
            pos = min(len, pos + idle);
        } else if (idle == 64u && pos == len && !more) {
            break;
        }
        const bool tri_step = r.lj < r.ltri;
        const bool tri_mode = wave_tests_triangles(active, tri_step);
        if (!active || tri_step != tri_mode) continue;

        bool hit_any = false;
        if (tri_mode) {
            const int j = r.lj;
            hit_any = r.test_triangles(bvh, ANY);
            if (COUNT) cnt.tris += (uint32_t)(r.lj - j);
        } else {
            if (COUNT) cnt.nodes++;
            r.visit_node(bvh, stk);
        }
        const bool done = hit_any || (r.last && r.lj == r.ltri);
        if (done) {
            if (ANY && IO::kResolve)
                pend = !hit_any;
            else if (ANY)
                io.store_occ(ray, hit_any, cnt.nodes, cnt.tris);
            else
                io.store_hit(ray, r.best, r.best_t, r.bu, r.bv, cnt.nodes, cnt.tris);  // a miss keeps t = tmax
            if (COUNT) {
                total.nodes += cnt.nodes;
                total.tris += cnt.tris;
            }
            active = false;
        }
    }
    if (ANY && IO::kResolve && pend) {
        float4 ra, rb;
        io.resolve_load(ray, ra, rb);
        io.resolve_store(ray, ra, rb);
    }
}

}  // namespace dl
