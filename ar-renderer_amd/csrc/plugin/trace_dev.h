// Device traversal of the 8-wide quantised BVH (gfx950, wave64).
//
// One ray per lane. A lane's traversal stack lives in LDS, interleaved by lane so that the 64
// lanes of a wave touch 64 consecutive banks; entries beyond the LDS part spill to a per-thread
// HBM slab (sized by the host from the tree depth: at most 7 entries per level are pending).
// Children that a ray's slab test hits are ordered near-to-far with an 8-key sorting network
// (key = distance bits | slot), the nearest is taken next and the rest are pushed far-to-near.
//
// What bounds it: VALU issue. With a node or a whole leaf per iteration (every lane in whichever it
// was at) the kernel issued VALU instructions in 87 % of the cycles of every SIMD at 41 % of the
// lanes (configuration 2 at 1920x1080). A step is therefore one node or one record, for the kind
// that more of the wave's lanes wait for (trace_step), so that both kinds run with most lanes; and
// the node step is short: no child count (empty slots have inverted boxes), one byte per child
// instead of a reference, stack entries written without branches. Finished lanes hand in their hits
// and take new rays together (trace_queue). Measured on 3 M bounce rays of configurations 2 / 4 / 5:
// 1.45 / 1.30 / 1.46 ms before, 0.70 / 0.50 / 0.66 ms now, at half the VALU instructions.
//
// The triangle test is the reference's Moller-Trumbore in float (src/geometry/shape.cpp:202-222)
// operation for operation; the file is compiled without FMA contraction so that the hit
// distances, and therefore the closest-hit primitive ids, are bit-identical to the CPU's.
#pragma once

#include <hip/hip_runtime.h>

#include "wbvh.h"

namespace pgpu {

// Tuning knobs (compile-time): LDS stack entries per lane and the idle-lane threshold of the
// per-lane ray fetch.
#ifndef PG_STACK_LDS
#define PG_STACK_LDS 16
#endif
#ifndef PG_REFILL
#define PG_REFILL 16
#endif
#ifndef PG_SPREAD_WAVES
#define PG_SPREAD_WAVES 2048
#endif
#ifndef PG_FEED_PARTS
#define PG_FEED_PARTS 4
#endif
#ifndef PG_DEALT_NUM
#define PG_DEALT_NUM 3
#define PG_DEALT_DEN 4
#endif
#ifndef PG_LEAF_NUM
#define PG_LEAF_NUM 1
#define PG_LEAF_DEN 2
#endif
constexpr int kTraceBlock = 256;
constexpr int kStackLds = PG_STACK_LDS;  // LDS entries per lane

struct DRay {
    float ox, oy, oz, dx, dy, dz;
};

// Reference Moller-Trumbore, no contraction. Returns true and updates t/b1/b2 on a closer hit.
__device__ __forceinline__ bool dev_hit_triangle(const DRay &r, float p0x, float p0y, float p0z, float e1x, float e1y,
                                                 float e1z, float e2x, float e2y, float e2z, float tMax, float *tOut,
                                                 float *uOut, float *vOut) {
    // pvec = cross(d, e2)
    float px = r.dy * e2z - r.dz * e2y;
    float py = r.dz * e2x - r.dx * e2z;
    float pz = r.dx * e2y - r.dy * e2x;
    float det = e1x * px + e1y * py + e1z * pz;
    if (det == 0.f || !__builtin_isfinite(det)) return false;
    float inv = 1.f / det;
    float tx = r.ox - p0x, ty = r.oy - p0y, tz = r.oz - p0z;
    float u = (tx * px + ty * py + tz * pz) * inv;
    if (u < 0.f || u > 1.f) return false;
    // qvec = cross(tvec, e1)
    float qx = ty * e1z - tz * e1y;
    float qy = tz * e1x - tx * e1z;
    float qz = tx * e1y - ty * e1x;
    float v = (r.dx * qx + r.dy * qy + r.dz * qz) * inv;
    if (v < 0.f || u + v > 1.f) return false;
    float t = (e2x * qx + e2y * qy + e2z * qz) * inv;
    if (t <= 0.f || t >= tMax) return false;
    *tOut = t;
    *uOut = u;
    *vOut = v;
    return true;
}

// Robust quadratic in double precision (src/geometry/shape.cpp:42-61).
__device__ __forceinline__ bool dev_hit_sphere(const DRay &r, float cx, float cy, float cz, float rad, float tMax,
                                               float *tOut) {
    double ox = r.ox - cx, oy = r.oy - cy, oz = r.oz - cz;
    double dx = r.dx, dy = r.dy, dz = r.dz;
    double a = dx * dx + dy * dy + dz * dz;
    double b = ox * dx + oy * dy + oz * dz;
    double c = ox * ox + oy * oy + oz * oz - double(rad) * rad;
    double k = b / a;
    double lx = ox - k * dx, ly = oy - k * dy, lz = oz - k * dz;
    double disc = double(rad) * rad - (lx * lx + ly * ly + lz * lz);
    if (disc < 0) return false;
    double q = -b - __builtin_copysign(__builtin_sqrt(a * disc), b);
    double t0 = c / q, t1 = q / a;
    if (t0 > t1) {
        double s = t0;
        t0 = t1;
        t1 = s;
    }
    double t = t0;
    if (t <= 0) t = t1;
    if (t <= 0 || t >= tMax) return false;
    *tOut = float(t);
    return true;
}

__device__ __forceinline__ void cswap(uint32_t &a, uint32_t &b) {
    uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
}

// Optimal 19-comparator network for 8 keys.
__device__ __forceinline__ void sort8(uint32_t k[8]) {
    cswap(k[0], k[2]); cswap(k[1], k[3]); cswap(k[4], k[6]); cswap(k[5], k[7]);
    cswap(k[0], k[4]); cswap(k[1], k[5]); cswap(k[2], k[6]); cswap(k[3], k[7]);
    cswap(k[0], k[1]); cswap(k[2], k[3]); cswap(k[4], k[5]); cswap(k[6], k[7]);
    cswap(k[2], k[4]); cswap(k[3], k[5]);
    cswap(k[1], k[4]); cswap(k[3], k[6]);
    cswap(k[1], k[2]); cswap(k[3], k[4]); cswap(k[5], k[6]);
}

struct TraceCtx {
    const WNode *nodes;
    const TriRec *recs;
    uint32_t *spill;       // per-thread spill slab: entry k at spill[k * spillStride + tid]
    int spillStride;       // number of threads sharing the slab layout
    int spillCap;          // entries available per thread in the slab
    int *errorFlag;        // set to 1 if a traversal stack would overflow its slab
};

// Counters for the algorithmic-traffic figures (nodes fetched, leaf records tested), by query kind.
struct TraceStats {
    uint32_t nodes = 0, recs = 0, anyNodes = 0, anyRecs = 0;
};

// Traversal state of one ray: the inverse direction, what it stands at (an inner node, a leaf
// record, or kIdle: complete), the stack depth and the best hit so far (prim -1: none; its distance
// is tMax). The stack itself lives in LDS (+ the HBM spill slab).
constexpr uint32_t kIdle = 0xffffffffu;
constexpr int kSpStep = 4 * kTraceBlock;
struct TravState {
    float ix, iy, iz;
    float tMax;
    uint32_t cur;
    int sp;  // byte offset of the stack's next free entry in the block's LDS area (entry k of a lane: kSpStep k + 4 lane)
    int prim;
    float b1, b2;
    bool any;  // any-hit query: complete at the first hit
    __device__ bool at_node() const { return int(cur) >= 0; }
    __device__ bool at_leaf() const { return int(cur) < -1; }
    __device__ bool found() const { return prim >= 0; }
};

// Inverse direction for the ordered slab test: |1/d| clamped to 2^64, so that the per-node
// products with the node scale (a power of two at most 2^60) and the origin offset stay finite
// and an axis the ray is parallel to yields signed, very large but never infinite distances.
__device__ __forceinline__ float slab_inv(float d) {
    float r = 1.f / d;
    return __builtin_copysignf(fminf(fabsf(r), 0x1p64f), d);
}

// The end of an unlimited ray. A plane distance that overflows is +inf: past this end, also once it is
// widened (kSlabWiden), so a box at such a distance is not entered.
constexpr float kTraceFar = 0x1.ffffp127f;

// A ray whose origin is not finite, or whose range is empty or NaN, hits nothing and is complete at
// once: the slab test's minima and maxima drop a NaN, so it would enter every node.
__device__ __forceinline__ void trace_begin(TravState &t, const DRay &r, float tMax, bool any) {
    t.ix = slab_inv(r.dx);
    t.iy = slab_inv(r.dy);
    t.iz = slab_inv(r.dz);
    t.tMax = fminf(tMax, kTraceFar);
    const bool valid = __builtin_isfinite(r.ox) && __builtin_isfinite(r.oy) && __builtin_isfinite(r.oz) && tMax > 0.f;
    t.cur = valid ? 0 : kIdle;  // the root node
    t.sp = 4 * int(threadIdx.x);
    t.any = any;
    t.prim = -1;
    t.b1 = t.b2 = 0.f;
}

__device__ __forceinline__ uint32_t *lds_at(uint32_t *lds, int sp) {
    return reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(lds) + sp);
}
__device__ __forceinline__ uint32_t *spill_at(const TraceCtx &c, int sp, int tid) {
    return c.spill + size_t(sp / kSpStep - kStackLds) * c.spillStride + tid;
}

// The next reference of the stack, kIdle when it is empty.
__device__ __forceinline__ void trace_pop(const TraceCtx &c, TravState &t, uint32_t *lds, int tid) {
    const int sp = t.sp - kSpStep;
    t.sp = sp;
    t.cur = kIdle;
    if (sp >= 0) {
        if (sp < kStackLds * kSpStep) t.cur = *lds_at(lds, sp);
        else t.cur = *spill_at(c, sp, tid);
    }
}

// Conservative widening of the slab test (the reference's, bvh.cpp:137-156, on both ends), applied
// to the far end alone, the lesser of the exit distance and the best hit: (1 + 6 eps) / (1 - 6 eps),
// rounded up. The best hit's distance needs it as the exit does: a flat box's entry distance and its
// triangle's hit distance are rounded separately. (To the distance, not to the planes' coefficients: a
// flat box's entry and exit are then the same FMA and stay equal.)
constexpr float kSlabWiden = 1.f + 1.6e-6f;

// One wide node: slab-tests its children, pushes the hit ones far to near and continues with the
// nearest (or pops). `lds` is the block's stack area (kStackLds * kTraceBlock entries), `tid` the
// global thread index for the spill slab. For lanes at an inner node.
template <bool kStats>
__device__ __forceinline__ void trace_node(const TraceCtx &c, const DRay &r, TravState &t, uint32_t *lds, int tid,
                                           TraceStats *st) {
    const uint4 *np = reinterpret_cast<const uint4 *>(c.nodes + t.cur);
    const uint4 h0 = np[0], h1 = np[1], q0 = np[2], q1 = np[3], q2 = np[4];
    uint32_t nodeBase = h1.x, leafBase = h1.y, metaLo = h1.z, metaHi = h1.w;
    // (keeps the second load whole and up here: its words are used after the sort, and a load moved
    // down there would stall the wave once more)
    asm volatile("" : "+v"(nodeBase), "+v"(leafBase), "+v"(metaLo), "+v"(metaHi));
    if (kStats) ++(t.any ? st->anyNodes : st->nodes);
    // scale / d per axis: exact (power-of-two scales); clamped so that q * a stays finite
    const float sx = __uint_as_float((h0.w & 0xffu) << 23), sy = __uint_as_float((h0.w & 0xff00u) << 15),
                sz = __uint_as_float((h0.w & 0xff0000u) << 7);
    const float ax = __builtin_amdgcn_fmed3f(sx * t.ix, -0x1p118f, 0x1p118f);
    const float ay = __builtin_amdgcn_fmed3f(sy * t.iy, -0x1p118f, 0x1p118f);
    const float az = __builtin_amdgcn_fmed3f(sz * t.iz, -0x1p118f, 0x1p118f);
    const float cx = (__uint_as_float(h0.x) - r.ox) * t.ix, cy = (__uint_as_float(h0.y) - r.oy) * t.iy,
                cz = (__uint_as_float(h0.z) - r.oz) * t.iz;
    // Ordered slab test: the direction's signs pick each axis's entry (near) and exit (far) planes
    // once per node, and a plane distance is one FMA, q (scale / d) + (origin - o) / d. The quantised
    // child boxes are rounded outwards by a grid step, far more than these roundings.
    const bool px = t.ix >= 0.f, py = t.iy >= 0.f, pz = t.iz >= 0.f;
    const uint32_t nx[2] = {px ? q0.x : q1.z, px ? q0.y : q1.w}, fx[2] = {px ? q1.z : q0.x, px ? q1.w : q0.y};
    const uint32_t ny[2] = {py ? q0.z : q2.x, py ? q0.w : q2.y}, fy[2] = {py ? q2.x : q0.z, py ? q2.y : q0.w};
    const uint32_t nz[2] = {pz ? q1.x : q2.z, pz ? q1.y : q2.w}, fz[2] = {pz ? q2.z : q1.x, pz ? q2.w : q1.y};
    uint32_t key[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int w = i >> 2, sh = (i & 3) * 8;
        const float tn = fmaxf(fmaxf(fmaxf(__builtin_fmaf(float((nx[w] >> sh) & 0xff), ax, cx),
                                           __builtin_fmaf(float((ny[w] >> sh) & 0xff), ay, cy)),
                                     __builtin_fmaf(float((nz[w] >> sh) & 0xff), az, cz)), 0.f);
        const float tf = fminf(fminf(fminf(__builtin_fmaf(float((fx[w] >> sh) & 0xff), ax, cx),
                                           __builtin_fmaf(float((fy[w] >> sh) & 0xff), ay, cy)),
                                     __builtin_fmaf(float((fz[w] >> sh) & 0xff), az, cz)), t.tMax) * kSlabWiden;
        key[i] = tn <= tf ? ((__float_as_uint(tn) & ~7u) | uint32_t(i)) : 0xffffffffu;
    }
    sort8(key);
    if (key[0] == 0xffffffffu) {
        trace_pop(c, t, lds, tid);
        return;
    }
    // A child's reference from its slot (key & 7): its meta byte by one byte permute, plus the base
    // of its kind.
    const uint32_t leafMore = leafBase - nodeBase;
    auto child = [=](uint32_t k) {
        const uint32_t m = __builtin_amdgcn_perm(metaHi, metaLo, (k & 7u) | 0x0c0c0c00u);
        return nodeBase + m + (m & 0x80u ? leafMore : 0u);
    };
    if (__ballot(t.sp >= (kStackLds - 6) * kSpStep) == 0) {
        // Seven more entries fit every lane's LDS part: written without branches, an empty key's entry
        // below the stack pointer, where the next overwrites it. Few waves have a lane with five hits.
        auto push = [&](uint32_t k) {
            *lds_at(lds, t.sp) = child(k);
            t.sp += k != 0xffffffffu ? kSpStep : 0;
        };
        if (__ballot(key[4] != 0xffffffffu)) {
            push(key[7]);
            push(key[6]);
            push(key[5]);
            push(key[4]);
        }
        push(key[3]);
        push(key[2]);
        push(key[1]);
    } else {
#pragma unroll
        for (int i = 7; i >= 1; --i) {
            if (key[i] != 0xffffffffu) {
                const uint32_t ref = child(key[i]);
                if (t.sp < kStackLds * kSpStep) {
                    *lds_at(lds, t.sp) = ref;
                } else if (t.sp / kSpStep - kStackLds < c.spillCap) {
                    *spill_at(c, t.sp, tid) = ref;
                } else {
                    *c.errorFlag = 1;
                    t.sp -= kSpStep;  // keep the stack in bounds; the error flag reports the lost subtree
                }
                t.sp += kSpStep;
            }
        }
    }
    t.cur = child(key[0]);
}

// One leaf record: tests it, then goes on to the leaf's next record or pops. For lanes at a leaf.
template <bool kStats>
__device__ __forceinline__ void trace_leaf(const TraceCtx &c, const DRay &r, TravState &t, uint32_t *lds, int tid,
                                           TraceStats *st) {
    const float4 *rp = reinterpret_cast<const float4 *>(c.recs + (t.cur & ~kLeafBit));
    const float4 a = rp[0], b = rp[1], d = rp[2];
    if (kStats) ++(t.any ? st->anyRecs : st->recs);
    const uint32_t prim = __float_as_uint(d.y);
    float th, u = 0.f, v = 0.f;
    bool h;
    if (prim & kSphereBit) h = dev_hit_sphere(r, a.x, a.y, a.z, a.w, t.tMax, &th);
    else h = dev_hit_triangle(r, a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, d.x, t.tMax, &th, &u, &v);
    if (h) {
        t.tMax = th;
        t.prim = int(prim & kPrimMask);
        t.b1 = u;
        t.b2 = v;
    }
    if (h && t.any) t.cur = kIdle;
    else if (prim & kLastBit) trace_pop(c, t, lds, tid);
    else ++t.cur;
}

// One step of a wave whose lanes stand at nodes, at records or idle: nodes when at least
// PG_LEAF_DEN / PG_LEAF_NUM times as many lanes wait at nodes as at records, else records (a record
// costs about a third of a node's instructions). 3 M bounce rays of configuration 2: 0.77 ms at a
// ratio of 1, 0.71 at 2, 0.70 at 3.
template <bool kStats>
__device__ __forceinline__ void trace_step(const TraceCtx &c, const DRay &r, TravState &t, uint32_t *lds, int tid,
                                           TraceStats *st) {
    const int nodes = __popcll(__ballot(t.at_node())), leaves = __popcll(__ballot(t.at_leaf()));
    if (nodes * PG_LEAF_NUM >= leaves * PG_LEAF_DEN) {
        if (t.at_node()) trace_node<kStats>(c, r, t, lds, tid, st);
    } else {
        if (t.at_leaf()) trace_leaf<kStats>(c, r, t, lds, tid, st);
    }
}

// Rays of a persistent traversal: items [0, n) dealt to the lanes of a launch's waves in runs of
// consecutive items; a wave's idle lanes take the next items of its run once at least kRefill of
// them are idle. A launch with no more items than it has lanes gives each wave one run (of a size
// that makes at least kSpreadWaves runs), so a short queue spreads over the chip instead of filling
// a few waves. Otherwise runs are tiles of 64: a block is dealt every gridDim-th group of as many
// tiles as it has waves, which its waves take in turn from a counter in LDS, and the last tiles go to
// whoever asks, from counters in device memory (undealt tile u belongs to part u % kFeedParts; a
// block drains one part, then the next). The deal keeps a block's waves on neighbouring
// tiles (they share the L1; single tiles, 2048 apart, were a seventh slower) and the blocks about
// abreast, so the rays in flight stay a narrow, coherent part of the queue.
// Atomics on one cache line of device memory complete one after the other, about every 8 ns, and
// each is a round trip that stalls its wave: with every take from one counter they set the time of a
// launch (4 M rays at 16, 24 and 40 lanes a take: 1.9, 1.3 and 0.9 ms), and even one failed take per
// wave at the end is 60 us. So few tiles are undealt, they have kFeedParts counters in lines of their
// own, and a block remembers in LDS which are drained.
constexpr int kRefill = PG_REFILL;
constexpr int kSpreadWaves = PG_SPREAD_WAVES;
constexpr int kFeedParts = PG_FEED_PARTS, kFeedStride = 32;  // device counters (they start at zero), ints between them
constexpr int kFeedInts = kFeedParts * kFeedStride;
constexpr int kBlockWaves = kTraceBlock / 64;
struct FeedLds {
    int taken;  // tiles of the block's deal that its waves have taken
    int gone;   // parts of the undealt tiles found drained
};
struct RayFeed {
    int n;
    int tiles, dealt;  // tiles; dealt tiles of each block (a multiple of its waves)
    int next, end;      // what is left of the wave's run
    bool done;          // no run left to take
};  // wave-uniform
// Called by the whole block.
__device__ __forceinline__ RayFeed feed_begin(int n, FeedLds *fl) {
    if (threadIdx.x == 0) fl->taken = fl->gone = 0;
    __syncthreads();
    RayFeed f;
    f.n = n;
    const int waves = int(gridDim.x) * kBlockWaves;
    const int fair = (n + waves - 1) / waves, spread = (n + kSpreadWaves - 1) / kSpreadWaves;
    f.next = f.end = f.tiles = f.dealt = 0;
    f.done = fair <= 64;
    if (f.done) {
        const int wave = int(blockIdx.x) * kBlockWaves + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
        const int per = max(fair, min(64, spread));
        f.next = min(n, wave * per);
        f.end = min(n, f.next + per);
    } else {
        f.tiles = (n + 63) >> 6;
        f.dealt = f.tiles / waves * PG_DEALT_NUM / PG_DEALT_DEN * kBlockWaves;
    }
    return f;
}
// The wave's next run into f.next, f.end.
__device__ __forceinline__ void feed_run(RayFeed &f, int *counter, FeedLds *fl) {
    const int lane = __lane_id();
    int tile = f.tiles, k = 0;
    if (lane == 0) k = atomicAdd(&fl->taken, 1);
    k = __builtin_amdgcn_readfirstlane(k);
    if (k < f.dealt) {
        tile = (k / kBlockWaves * int(gridDim.x) + int(blockIdx.x)) * kBlockWaves + k % kBlockWaves;
    } else {
        int gone = __builtin_amdgcn_readfirstlane(*static_cast<volatile int *>(&fl->gone));
        for (; gone < kFeedParts; ++gone) {
            const int part = (int(blockIdx.x) + gone) % kFeedParts;
            int got = 0;
            if (lane == 0) got = atomicAdd(&counter[part * kFeedStride], 1);
            tile = f.dealt * int(gridDim.x) + __builtin_amdgcn_readfirstlane(got) * kFeedParts + part;
            if (tile < f.tiles) break;
            if (lane == 0) *static_cast<volatile int *>(&fl->gone) = gone + 1;
        }
    }
    f.done = tile >= f.tiles;
    f.next = f.done ? f.n : tile * 64;
    f.end = min(f.n, f.next + 64);
}
// Gives idle lanes their next item (-1: none). Called by the whole wave with some lane idle.
__device__ __forceinline__ int feed_take(RayFeed &f, int *counter, FeedLds *fl, bool idle) {
    if (f.next == f.end && !f.done) feed_run(f, counter, fl);
    const unsigned long long mask = __ballot(idle);
    const int i = f.next + __popcll(mask & ((1ull << __lane_id()) - 1ull));
    const int item = idle && i < f.end ? i : -1;
    f.next = min(f.end, f.next + __popcll(mask));
    return item;
}

// The loop of a persistent traversal, run by whole blocks. begin(i, r, t) loads item i's ray into r
// and starts t; end(i, r, t) takes a finished query's result and may start the item's next query,
// returning true. Finished lanes call end when the wave next takes rays, so that neither interrupts
// the others' steps. Every step completes a node or a record of at least one lane. A node is visited at
// most once by a query (references lead down the tree only) and adds at most eight references, of which
// one from a slot without a child, which only extreme distances enter (see wbvh.h), is to a record; so a
// query takes a bounded number of steps and the loop ends.
template <bool kStats, class Begin, class End>
__device__ __forceinline__ void trace_queue(const TraceCtx &c, int n, int *counter, uint32_t *lds, int tid, TraceStats *st,
                                            Begin begin, End end) {
    __shared__ FeedLds fl;
    RayFeed f = feed_begin(n, &fl);
    int item = -1;
    DRay r{};
    TravState t{};
    t.cur = kIdle;
    while (true) {
        const int idles = __popcll(__ballot(t.cur == kIdle));
        const bool drained = f.done && f.next == f.end;
        if (idles >= (drained ? 64 : kRefill)) {
            if (t.cur == kIdle && item >= 0 && !end(item, r, t)) item = -1;
            const bool idle = item < 0;
            if (drained) {
                if (__ballot(!idle) == 0) break;
            } else {
                const int next = feed_take(f, counter, &fl, idle);
                if (next >= 0) {
                    item = next;
                    begin(next, r, t);
                }
            }
            continue;
        }
        trace_step<kStats>(c, r, t, lds, tid, st);
    }
}

}  // namespace pgpu
