// tracer.hip -- wavefront Monte-Carlo acoustic tracer (gfx950).
//
// One render replaces Scene::Render (src/Scene.cpp:111-318) for every band of
// ear_render_desc.band_mask at once; each band is its own reference context
// (SceneContext, src/SceneContext.h:26-54) with its own Philox streams.  The
// reference's per-ray loop over num_bounces (src/Scene.cpp:143-281) becomes a
// loop over wavefront iterations, each a chain of kernels over a compacted
// queue of live rays:
//   k_generate  emission, k = 0 (SoundRay, src/SoundFile.cpp:215-228; mesh
//               sources also connect to the recorders at k = 0)
//   k_extend    closest hit, BVH traversal (Mesh::RayIntersection)
//   k_shade     Scene::Bounce + Material::Bounce + energy bookkeeping + the
//               NEE weight of src/Scene.cpp:197-261; emits shadow requests and
//               the next ray (Sample_Hemi) into the next queue
//   k_shadow    any hit on the segment to the recorder (Mesh::LineIntersection)
//               and, when visible, Recorder::Record as a fixed-point ramp splat
//   k_finalize  exact prefix sums of the second-difference histograms,
//               1/N, direct sound (src/Scene.cpp:286-316), gain^2
// Histograms are 128-bit two's-complement fixed point (2^-80 units).  A ramp of
// width w and slope S (MonoRecorder::Record, src/MonoRecorder.cpp:83-97) is
// stored as three second-difference points (+wS at s, -(w+1)S at s+1, +S at
// s+w+1); integer sums are order independent, so results are bitwise
// deterministic whatever the launch shape.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "ear_internal.hpp"

namespace ear {
namespace {

constexpr int kBlock = 256;
constexpr uint32_t kMaxBounces = 0xFFFFu;  // the bounce number's field in a queue entry (bits 8..23)
constexpr int kLdsMin = 16;  // smallest LDS part of the traversal stack; the overflow area covers the rest
constexpr int kShadeBlock = 256;  // k_shade: its block-wide appends take one counter atomic per block step
// no-allocation render: traversal grids of at most this many waves per CU
// (their overflow stacks come out of the fixed region), and the fewest rays
// in flight it accepts
constexpr uint32_t kNoallocWaves = 16;
constexpr size_t kNoallocMinRays = 4096;
constexpr double kBinMetres = 343.0 / 44100.0;       // a histogram bin as a distance

enum StatIdx {
    ST_SEGMENTS = 0,
    ST_SHADOW = 1,
    ST_CONTRIB = 2,
    ST_NV_CL = 3,
    ST_NT_CL = 4,
    ST_NV_SH = 5,
    ST_NT_SH = 6,
    ST_RAYS = 7,
    ST_TAIL_SEG = 8,  // segments and shadow rays traced by k_tail (not by the
    ST_TAIL_SH = 9,   // wavefront kernels whose launch times are measured)
    ST_DROPPED = 10,  // ramps cut at the end of the histogram
    ST_BINS = 11,     // the largest ramp end among them (a maximum, not a sum)
    ST_SH_CONTRIB = 12,  // connections recorded by the shadow kernels (not k_tail)
    ST_SH_RAMPS = 13,    // and the ramps they made (one per channel)
    ST_N = 14
};

struct Queue {
    float4* o;  // {ox, oy, oz, I}
    float4* d;  // {dx, dy, dz, L}
    uint4* m;   // {ray id, draw counter, band | k << 8, -}
};

struct ShadowQ {
    float4* p;  // {px, py, pz, c}
    float4* m;  // {L, rec | band << 8, -, -}
};

struct Traversal {
    const BvhNode* __restrict__ nodes;    // 2-wide tree
    const Bvh4Node* __restrict__ nodes4;  // 4-wide tree (null when the scene is 2-wide)
    const float4* __restrict__ tris;
    uint32_t n_tris;
    int* gstack;        // overflow stack [(kStackDepth - LDS)][gthreads]
    uint32_t gthreads;  // persistent threads sharing gstack
};

// Lane refilling for the persistent traversal kernels: once at least `refill`
// lanes of a wave are idle, the wave hands them queue entries from its claimed
// run, claiming a new run with one atomic on `counter` (zero at launch) when
// its run is used up: `chunk` entries, or (chunk = 0) one per idle lane.
struct Fetch {
    uint32_t* counter;  // n_seg counters, one per 128-byte line (stride kSegStride)
    uint32_t refill;
    uint32_t chunk;
    uint32_t n_seg;
};
constexpr uint32_t kSegStride = 32;  // uint32 words per counter line
constexpr uint32_t kMaxSeg = 64;
// a batch of 32 rooms: 174 ms at 16 segments, 177 at 64, 177 at 8; the
// 200k-triangle hall: 375, 377, 374
constexpr uint32_t kSegDefault = 16;

// ---------------------------------------------------------------------------
// wave helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Appends the lanes with pred set; returns each such lane's slot.  All lanes
// of the wave must call it.
__device__ __forceinline__ uint32_t wave_append(uint32_t* counter, bool pred) {
    uint64_t mask = __ballot(pred);
    uint32_t base = 0;
    if (mask) {
        int leader = __ffsll((unsigned long long)mask) - 1;
        if ((int)lane_id() == leader) base = atomicAdd(counter, (uint32_t)__popcll(mask));
        base = __shfl(base, leader);
    }
    uint64_t below = mask & ((1ull << lane_id()) - 1ull);
    return base + (uint32_t)__popcll(below);
}

// Two appends of a block with one atomic: a wave's `a` entries to the counter
// in the low word and `b` to the one in the high word of `counter` (neither
// overflows: a queue holds fewer than 2^32).  Adds to one address take about
// 12.5 ns each whoever makes them, so with one per block step and queue the
// appends were k_shade's whole time.  Every thread of the block calls it with
// its wave's counts; `sc`: scratch of BLOCK / 64 words that consecutive calls
// must not share.  Returns the wave's first slots {a, b}.
template <int BLOCK>
__device__ __forceinline__ uint2 block_append2(unsigned long long* counter, uint32_t a, uint32_t b,
                                               unsigned long long* sc) {
    const uint32_t wave = threadIdx.x >> 6;
    if (lane_id() == 0) sc[wave] = (unsigned long long)a | ((unsigned long long)b << 32);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0;
        for (uint32_t w = 0; w < BLOCK / 64; ++w) tot += sc[w];
        unsigned long long base = tot ? atomicAdd(counter, tot) : 0ull;
        for (uint32_t w = 0; w < BLOCK / 64; ++w) {
            const unsigned long long c = sc[w];
            sc[w] = base;
            base += c;
        }
    }
    __syncthreads();
    const unsigned long long mine = sc[wave];
    return make_uint2((uint32_t)mine, (uint32_t)(mine >> 32));
}

// Orders one wave's LDS accesses (lanes read what other lanes of the same
// wave wrote; the LDS executes a wave's instructions in order).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sample_Hemi's rejection loops (src/Distributions.h:48-70) for the lanes of
// one wave together.  A lane's candidates are its consecutive triples of
// uniforms, so which one it accepts and how many draws it uses do not depend
// on which lane computes its Philox blocks.  In each round the wave's lanes
// compute blocks for the A lanes still sampling (64 / A blocks for each),
// and every sampling lane scans its own words in order with sample_hemi's
// tests and arithmetic: same vector, same draw count.  A wave then runs
// until its sampling lanes' candidates are used up together, instead of one
// block per candidate until its slowest lane accepts.  All lanes of the wave
// call it; `need` marks those that sample: around normal n if `hemi`
// (sample_hemi), else the whole sphere (sample_sphere).
//
// A candidate f of squared length l is in the hemisphere if dot(n, f / |f|) is
// not negative.  Almost always dot(n, f) tells: the two differ by at most
// 4.2e-7 |n| |f| in rounding (four and three roundings of 2^-24 each on terms
// whose sum of sizes is at most |n| |f|), so past 1e-6 its sign is the
// quotient's.  The root and three divisions are then left for the accepted
// candidate, after the rounds.
__device__ __forceinline__ bool upper(V3 n, V3 f, float l) {
    const float a = dot(n, f);
    if (a < -1e-6f) return false;
    if (fabsf(a) > 1e-6f) return true;
    const float s = sqrtf(l);
    return !(dot(n, V3{f.x / s, f.y / s, f.z / s}) < 0.0f);
}
struct HemiLds {
    uint4 own[64];   // the rank-th sampling lane's ray, ctx, inst and first block to compute
    uint2 key[64];   // its Philox key
    uint4 blk[128];  // per sampling lane (m + 1 each): its current block, then its m new blocks
};
__device__ __forceinline__ V3 sample_hemi_wave(bool need, bool hemi, Rng& rng, V3 n, HemiLds& S) {
    const uint32_t lane = lane_id();
    V3 v{0.0f, 0.0f, 0.0f};  // the accepted candidate and its squared length
    float vl = 1.0f;
    uint64_t act = __ballot(need);
    while (act) {
        const uint32_t A = (uint32_t)__popcll(act);
        const uint32_t m = 64u / A;  // A * (m + 1) <= 64 + A block slots
        const bool mine = (act >> lane) & 1ull;
        const uint32_t rank = (uint32_t)__popcll(act & ((1ull << lane) - 1ull));
        uint32_t ph = 0;
        if (mine) {
            ph = rng.draw & 3u;
            S.own[rank] = make_uint4(rng.ray, rng.ctx, rng.inst, (rng.draw >> 2) + (ph ? 1u : 0u));
            S.key[rank] = make_uint2(rng.k0, rng.k1);
            S.blk[rank * (m + 1)] = make_uint4(rng.buf[0], rng.buf[1], rng.buf[2], rng.buf[3]);
        }
        wave_sync();
        const uint32_t a = lane / m, o = lane - a * m;
        if (a < A) {
            const uint4 w = S.own[a];
            const uint2 k = S.key[a];
            uint32_t c[4] = {w.w + o, w.x, w.y, w.z};
            philox4x32_10(c, k.x, k.y);
            S.blk[a * (m + 1) + 1 + o] = make_uint4(c[0], c[1], c[2], c[3]);
        }
        wave_sync();
        bool left = false;
        if (mine) {
            // word `off` of this lane's run; the first unused one is its draw
            const uint32_t* words = (const uint32_t*)&S.blk[rank * (m + 1)];
            const uint32_t off0 = ph ? ph : 4u, end = 4u * (m + 1u);
            uint32_t off = off0;
            left = true;
            while (off + 3u <= end) {
                const float f1 = Rng::to_unit(words[off]) * 2.0f - 1.0f;
                const float f2 = Rng::to_unit(words[off + 1u]) * 2.0f - 1.0f;
                const float f3 = Rng::to_unit(words[off + 2u]) * 2.0f - 1.0f;
                off += 3u;
                const float l = f1 * f1 + f2 * f2 + f3 * f3;
                if (l < 0.001f || l > 1.0f) continue;
                if (hemi && !upper(n, V3{f1, f2, f3}, l)) continue;
                v = V3{f1, f2, f3};
                vl = l;
                left = false;
                break;
            }
            rng.draw += off - off0;
            if (off & 3u) {
                const uint4 b = S.blk[rank * (m + 1) + (off >> 2)];
                rng.buf[0] = b.x;
                rng.buf[1] = b.y;
                rng.buf[2] = b.z;
                rng.buf[3] = b.w;
            }
        }
        wave_sync();  // this round's reads before the next round's writes
        act = __ballot(left);
    }
    const float s = sqrtf(vl);
    return V3{v.x / s, v.y / s, v.z / s};
}

// Statistics counters: [kStatCopies][ST_N], a block adding into copy
// blockIdx % kStatCopies (the host sums the copies), so that the one atomic
// per wave at the end of every launch does not pile up on one address.
constexpr uint32_t kStatCopies = 64;
__device__ __forceinline__ void stat_add(unsigned long long* stats, int idx, uint64_t v) {
    // reduce within the wave, one atomic per wave
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    if (lane_id() == 0 && v) atomicAdd(stats + (size_t)(blockIdx.x % kStatCopies) * ST_N + idx, (unsigned long long)v);
}

// Ramps that run past the last bin of the histogram.  The reference grows its
// buffer on such a write (FloatBuffer::operator[], src/Recorder.cpp:52-59);
// here the late bins are not recorded, and each such ramp is counted with the
// bin count that would have kept it whole, so that a caller can size the
// histogram and render again.
struct Drops {
    uint32_t n = 0, end = 0;
    __device__ __forceinline__ void add(uint32_t e) {
        if (e) {
            ++n;
            end = max(end, e);
        }
    }
};
// All lanes of the wave must call it.
__device__ __forceinline__ void stat_drops(unsigned long long* stats, const Drops& d) {
    stat_add(stats, ST_DROPPED, d.n);
    uint32_t e = d.end;
    for (int off = 32; off > 0; off >>= 1) e = max(e, (uint32_t)__shfl_down(e, off));
    if (lane_id() == 0 && e)
        atomicMax(stats + (size_t)(blockIdx.x % kStatCopies) * ST_N + ST_BINS, (unsigned long long)e);
}

// Queue entries handed to the lanes of a wave (see Fetch).  The queue [0, n)
// is cut into f.n_seg segments with a counter each, so that claims of many
// waves do not serialise on one address: a wave claims from its current
// segment and moves on to the next one when that is used up; after f.n_seg
// used-up segments in a row everything has been taken.  A queue no longer
// than the grid's lanes needs no claim: each wave has its own 64 entries (the
// blocks' first waves before the second ones, so that a short queue spreads
// over all CUs) and the waves past its end leave at once; trying the
// segments in turn to learn that nothing is left took such launches longer
// than their walks (400 bounces of 0.5M rays in a room, 64 segments: 22 ms,
// 8 ms without).  The state is the same in the whole wave and kept in scalar
// registers, and no claim divides (with a segment's bounds formed per lane
// and claim in 64 bits a refill cost about 300 instructions).
struct Claim {
    uint32_t n, next, end, seg, seg_len, n_seg, want, fails;
    // own: entries a wave has of a short queue (64, or fewer to spread it out)
    __device__ __forceinline__ Claim(uint32_t n_, uint32_t gtid, uint32_t threads, const Fetch& f, uint32_t own = 64u) {
        n = (uint32_t)__builtin_amdgcn_readfirstlane((int)n_);
        n_seg = f.n_seg;
        seg = (uint32_t)__builtin_amdgcn_readfirstlane((int)((gtid >> 6) % n_seg));
        seg_len = n / n_seg + (n % n_seg ? 1u : 0u);
        next = end = fails = 0;
        // entries per atomic: what one refill needs, or while the queue is
        // long (256 for every wave) enough for several refills
        // (a chunk so large that the waves' last, failing claims wrap a counter
        // would hand its segment out again: at most n + chunk (waves + n_seg))
        want = f.chunk ? min(f.chunk, (0xFFFFFFFFu - n) / (threads / 64u + n_seg))
                       : (n / 256u >= threads / 64u ? 64u : 0u);
        if (n <= threads) {
            const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)((threadIdx.x >> 6) * gridDim.x + blockIdx.x));
            next = min(wave * own, n);
            end = min(next + own, n);
            fails = n_seg;
        }
    }
    __device__ __forceinline__ bool exhausted() const { return fails >= n_seg && next >= end; }
    // the whole wave; idle: the ballot of its idle lanes.  The entry handed to
    // this lane, or ~0u.
    __device__ __forceinline__ uint32_t take(const Fetch& f, uint64_t idle, uint32_t lane) {
        const uint32_t n_idle = (uint32_t)__popcll(idle);
        while (next >= end && fails < n_seg) {
            const uint32_t lo = min(seg * seg_len, n), hi = min(lo + seg_len, n), k = want ? want : n_idle;
            uint32_t old = 0;
            if (lane == 0) old = atomicAdd(f.counter + seg * kSegStride, k);
            old = (uint32_t)__builtin_amdgcn_readfirstlane((int)old);
            if (old < hi - lo) {
                next = lo + old;
                end = min(next + k, hi);
                fails = 0;
            } else {
                ++fails;
                seg = seg + 1 == n_seg ? 0u : seg + 1;
            }
        }
        const uint32_t rank = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
        const uint32_t avail = end - next, base = next;
        next += min(avail, n_idle);
        return (((idle >> lane) & 1ull) && rank < avail) ? base + rank : 0xFFFFFFFFu;
    }
};

// ---------------------------------------------------------------------------
// BVH traversal
// ---------------------------------------------------------------------------
// Loads through a pointer known to address global memory (the scene arrays
// reach the kernels inside structs, where the compiler would otherwise emit
// flat loads that also wait on the LDS counter).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ldg(const float4* p) {
    const f32x4 v = *(const __attribute__((address_space(1))) f32x4*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ int4 ldg(const int4* p) {
    const i32x4 v = *(const __attribute__((address_space(1))) i32x4*)p;
    return make_int4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 ldg(const uint4* p) {
    const i32x4 v = *(const __attribute__((address_space(1))) i32x4*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ float safe_inv(float x) {
    float y = fabsf(x) > 1e-20f ? x : copysignf(1e-20f, x);
    return 1.0f / y;
}

struct SlabRay {
    float ox, oy, oz, ix, iy, iz;
};

// entry/exit of the ray against box {lo, hi}; robust form (lo - o) * inv
__device__ __forceinline__ void slab(const SlabRay& r, float lx, float ly, float lz, float hx, float hy, float hz,
                                     float& tn, float& tf) {
    float ax = (lx - r.ox) * r.ix, bx = (hx - r.ox) * r.ix;
    float ay = (ly - r.oy) * r.iy, by = (hy - r.oy) * r.iy;
    float az = (lz - r.oz) * r.iz, bz = (hz - r.oz) * r.iz;
    tn = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fminf(az, bz));
    tf = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz));
}

// Per-thread traversal stack: the first LDS entries in shared memory
// (column-major over the block so a wave's accesses are conflict free), the
// rest in a global overflow area indexed [entry][persistent thread].  The
// pointers carry their address space: a choice between two generic pointers
// compiles to flat accesses, which go through the global memory's address
// unit even when they hit LDS.
typedef __attribute__((address_space(3))) int LdsInt;
typedef __attribute__((address_space(1))) int GlobalInt;
template <int LDS, int BLOCK>
struct Stack {
    LdsInt* lds;
    GlobalInt* over;
    uint32_t n_over;  // persistent threads sharing the overflow area
    int sp = 0;
    __device__ __forceinline__ Stack(int* lds_, int* gstack, uint32_t gtid, uint32_t gthreads)
        : lds((LdsInt*)lds_), over((GlobalInt*)gstack + gtid), n_over(gthreads) {}
    __device__ __forceinline__ void push(int v) {
        if (__builtin_expect(sp < LDS, 1))
            lds[sp * BLOCK] = v;
        else
            over[(size_t)(uint32_t)(sp - LDS) * n_over] = v;
        ++sp;
    }
    __device__ __forceinline__ int pop() {
        --sp;
        if (__builtin_expect(sp < LDS, 1)) return lds[sp * BLOCK];
        return over[(size_t)(uint32_t)(sp - LDS) * n_over];
    }
};

// Tests the triangles of leaf reference `cref`.  Closest hit (ANY = false):
// t in (0.001, best_t) with the lower original index winning ties, as the
// reference's strict '<' scan does (src/Mesh.cpp:39-45).  Any hit (ANY =
// true): segment parameter t in (1e-5, 1) (src/Mesh.cpp:58-71); best_s = 0 as
// soon as one is found.
template <bool ANY, bool INSTR>
__device__ __forceinline__ void test_leaf(const Traversal& T, int32_t cref, V3 o, V3 d, float& best_t, int& best_s,
                                          uint32_t& best_o, uint32_t& ntri) {
    uint32_t u = (uint32_t)cref;
    uint32_t first = u & 0x00FFFFFFu;
    uint32_t cnt = ((u >> 24) & 0x7Fu) + 1;
    for (uint32_t i = first; i < first + cnt; ++i) {
        float4 t0 = ldg(T.tris + 3 * i), t1 = ldg(T.tris + 3 * i + 1), t2 = ldg(T.tris + 3 * i + 2);
        V3 v0{t0.x, t0.y, t0.z}, e1{t0.w, t1.x, t1.y}, e2{t1.z, t1.w, t2.x};
        float t;
        if (INSTR) ++ntri;
        if (mt_intersect(v0, e1, e2, o, d, t)) {
            if (ANY) {
                if (t > 1e-5f && t < 1.0f) {
                    best_s = 0;
                    return;
                }
            } else {
                uint32_t orig = __float_as_uint(t2.y);
                if (t > 0.001f && (t < best_t || (t == best_t && orig < best_o))) {
                    best_t = t;
                    best_s = (int)i;
                    best_o = orig;
                }
            }
        }
    }
}

// A walk of one ray as a resumable state machine, so that a persistent lane
// can interleave the walks of rays it fetches one after another.  Closest hit
// (ANY = false): best_* hold the nearest hit so far (order independent: ties
// go to the lower original index).  Any hit: best_s = 0 once a blocker is
// found.
//   idle()   no walk (or it has ended)
//   start()  begins one (an empty scene's ends at once)
//   step()   one step of every lane's walk, called by all (active) lanes of
//            the wave; true for a lane whose walk has just ended
//
// 2-wide tree: a step visits one node and tests its leaf children at once.
template <int LDS, int BLOCK, int WIDTH, bool ANY, bool INSTR>
struct Walker {
    static constexpr int kIdle = kEmpty4;
    SlabRay sr;
    V3 o, d;
    float best_t = 0.0f;
    int best_s = -1;
    uint32_t best_o = 0;
    int node = kIdle;  // next internal node to visit, -1: pop one
    Stack<LDS, BLOCK> stk;

    __device__ __forceinline__ Walker(int* lds, int* gstack, uint32_t gtid, uint32_t gthreads)
        : stk(lds, gstack, gtid, gthreads) {}
    __device__ __forceinline__ bool idle() const { return node == kIdle; }
    __device__ __forceinline__ bool found() const { return best_s >= 0; }
    __device__ __forceinline__ void start(const Traversal& T, V3 o_, V3 d_, float t_max) {
        o = o_;
        d = d_;
        sr = SlabRay{o.x, o.y, o.z, safe_inv(d.x), safe_inv(d.y), safe_inv(d.z)};
        best_t = t_max;
        best_s = -1;
        best_o = 0;
        node = T.n_tris != 0 ? 0 : kIdle;
        stk.sp = 0;
    }
    __device__ __forceinline__ bool step(const Traversal& T, uint32_t& nvis, uint32_t& ntri) {
        if (idle()) return false;
        if (node < 0) node = stk.pop();  // not ended: the stack holds a node
        if (INSTR) ++nvis;
        const BvhNode* N = T.nodes + node;
        float4 a = ldg(&N->a), b = ldg(&N->b), c = ldg(&N->c);
        int4 ch = ldg(&N->d);
        float tn0, tf0, tn1, tf1;
        slab(sr, a.x, a.y, a.z, a.w, b.x, b.y, tn0, tf0);
        slab(sr, b.z, b.w, c.x, c.y, c.z, c.w, tn1, tf1);
        float lim = ANY ? 1.0f : best_t;
        bool h0 = tn0 <= tf0 && tf0 >= 0.0f && tn0 <= lim;
        bool h1 = tn1 <= tf1 && tf1 >= 0.0f && tn1 <= lim;
        if (h0 && ch.x < 0) {
            test_leaf<ANY, INSTR>(T, ch.x, o, d, best_t, best_s, best_o, ntri);
            h0 = false;
        }
        if (h1 && ch.y < 0 && !(ANY && found())) {
            test_leaf<ANY, INSTR>(T, ch.y, o, d, best_t, best_s, best_o, ntri);
            h1 = false;
        }
        if (ANY && found()) {
            node = kIdle;
            return true;
        }
        node = -1;
        if (h0 && h1) {
            bool first0 = tn0 <= tn1;
            stk.push(first0 ? ch.y : ch.x);
            node = first0 ? ch.x : ch.y;
        } else if (h0) {
            node = ch.x;
        } else if (h1) {
            node = ch.y;
        }
        if (node >= 0 || stk.sp > 0) return false;
        node = kIdle;
        return true;
    }
};

// 4-wide tree: cur is the node to visit or the leaf to test; a visit sorts
// the node's hit children (inner or leaf) by entry distance, takes the nearest
// and pushes the others farthest first.  What bounds it is the vector unit:
// of its instructions only f32 add, mul and fma, 32-bit logic, shifts and
// adds issue at two per clock and CU (measured 1.7), while min, max, compares,
// conversions and selects issue at one.  So the boxes' planes are folded to
// one multiply-add each, the near and far planes are chosen by the sign of
// the direction for all four children at once instead of by min and max, and
// a wave's step is either a node visit or a triangle test, for the lanes at
// one (whichever more of the wave's walks are at), so that no step runs both
// for a few lanes each.  Hall of 200k triangles, 3 x 10M rays: closest hit
// 176 -> 128 ms and any hit 137 -> 92 ms per render (1.34e11 -> 7.8e10 vector
// instructions).  A lane's 16-byte piece of a node or triangle is an L1 access
// of its own unless another lane reads the same, 63 per closest-hit query, and
// the L1 takes one per clock and CU: that is now the closest-hit kernel's bound
// (1.02 measured).  Popped children are not held against the best hit, and an
// any-hit walk takes children unsorted: 5.66 triangle tests a closest-hit query
// where the walk that held leaves back made 5.31, 9.54 node visits a shadow
// query for 8.90 (2.85 triangle tests for 3.13).
template <int LDS, int BLOCK, bool ANY, bool INSTR>
struct Walker<LDS, BLOCK, 4, ANY, INSTR> {
    static constexpr int kIdle = kEmpty4;  // above every node index
    V3 o, d;
    float ix, iy, iz;  // 1 / d
    float best_t = 0.0f;
    int best_s = -1;
    uint32_t best_o = 0;
    int cur = kIdle;  // >= 0: the node to visit; < 0: the leaf to test
    Stack<LDS, BLOCK> stk;

    __device__ __forceinline__ Walker(int* lds, int* gstack, uint32_t gtid, uint32_t gthreads)
        : stk(lds, gstack, gtid, gthreads) {}
    __device__ __forceinline__ bool idle() const { return cur == kIdle; }
    __device__ __forceinline__ bool found() const { return best_s >= 0; }
    // 1 / x to an ulp: the boxes' padding covers it
    static __device__ __forceinline__ float inv(float x) {
        return __builtin_amdgcn_rcpf(fabsf(x) > 1e-20f ? x : copysignf(1e-20f, x));
    }
    __device__ __forceinline__ void start(const Traversal& T, V3 o_, V3 d_, float t_max) {
        o = o_;
        d = d_;
        ix = inv(d.x);
        iy = inv(d.y);
        iz = inv(d.z);
        best_t = t_max;
        best_s = -1;
        best_o = 0;
        // an origin that is no number on any axis is in no box (the minima and
        // maxima of visit() pass over a NaN, so it would be in all of them)
        const float px = o.x * ix, py = o.y * iy, pz = o.z * iz;
        const bool nowhere = (px != px) & (py != py) & (pz != pz);
        cur = T.n_tris != 0 && !nowhere ? 0 : kIdle;
        stk.sp = 0;
    }

    // a and b swapped if m is all ones
    static __device__ __forceinline__ void swap_if(uint32_t m, uint32_t& a, uint32_t& b) {
        const uint32_t t = (a ^ b) & m;
        a ^= t;
        b ^= t;
    }
    static __device__ __forceinline__ uint32_t sign_mask(float x) { return (uint32_t)((int)__float_as_uint(x) >> 31); }

    // orders two (entry distance, child) pairs
    static __device__ __forceinline__ void order(float& ka, int& va, float& kb, int& vb) {
        const bool sw = kb < ka;
        const float k0 = fminf(ka, kb), k1 = fmaxf(ka, kb);
        const int v0 = sw ? vb : va, v1 = sw ? va : vb;
        ka = k0;
        kb = k1;
        va = v0;
        vb = v1;
    }

    __device__ __forceinline__ bool visit(const Traversal& T) {
        const Bvh4Node* N = (const Bvh4Node*)((const char*)T.nodes4 + ((uint32_t)cur << 6));
        const uint4 og = ldg(&N->org);
        uint4 qa = ldg(&N->qa), qb = ldg(&N->qb);
        const int4 rf = ldg(&N->ref);
        // planes org + q 2^e against the ray, one multiply-add each:
        // (2^e / d) q + (org - o) / d.  The rounding moves a plane by a few
        // 2^-24 of |org - o| (the boxes are padded by 1e-5 of the scene) and a
        // distance by a few 2^-24 of itself, which the widened exit covers;
        // the triangle test decides the hit.
        const float ax = __uint_as_float((og.w << 23) & 0x7F800000u) * ix,
                    ay = __uint_as_float((og.w << 15) & 0x7F800000u) * iy,
                    az = __uint_as_float((og.w << 7) & 0x7F800000u) * iz;
        const float bx = (__uint_as_float(og.x) - o.x) * ix, by = (__uint_as_float(og.y) - o.y) * iy,
                    bz = (__uint_as_float(og.z) - o.z) * iz;
        swap_if(sign_mask(ix), qa.x, qa.y);  // near, far
        swap_if(sign_mask(iy), qa.z, qa.w);
        swap_if(sign_mask(iz), qb.x, qb.y);
        int r[4] = {rf.x, rf.y, rf.z, rf.w};
        float key[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float nx = __builtin_fmaf((float)((qa.x >> (8 * k)) & 0xFFu), ax, bx);
            const float fx = __builtin_fmaf((float)((qa.y >> (8 * k)) & 0xFFu), ax, bx);
            const float ny = __builtin_fmaf((float)((qa.z >> (8 * k)) & 0xFFu), ay, by);
            const float fy = __builtin_fmaf((float)((qa.w >> (8 * k)) & 0xFFu), ay, by);
            const float nz = __builtin_fmaf((float)((qb.x >> (8 * k)) & 0xFFu), az, bz);
            const float fz = __builtin_fmaf((float)((qb.y >> (8 * k)) & 0xFFu), az, bz);
            const float tn = fmaxf(fmaxf(fmaxf(nx, ny), nz), 0.0f);
            const float tf = fminf(fminf(fminf(fx, fy), fz) * 1.000001f, ANY ? 1.0f : best_t);
            key[k] = (tn <= tf) & (r[k] != kEmpty4) ? tn : INFINITY;
        }
        if (!ANY) {
            // nearest first
            order(key[0], r[0], key[1], r[1]);
            order(key[2], r[2], key[3], r[3]);
            order(key[0], r[0], key[2], r[2]);
            order(key[1], r[1], key[3], r[3]);
            order(key[1], r[1], key[2], r[2]);
            if (key[3] != INFINITY) stk.push(r[3]);
            if (key[2] != INFINITY) stk.push(r[2]);
            if (key[1] != INFINITY) stk.push(r[1]);
            cur = key[0] != INFINITY ? r[0] : kIdle;
        } else {
            // any order: the last hit child is taken, the others pushed
            cur = key[0] != INFINITY ? r[0] : kIdle;
#pragma unroll
            for (int k = 1; k < 4; ++k) {
                if (key[k] == INFINITY) continue;
                if (cur != kIdle) stk.push(cur);
                cur = r[k];
            }
        }
        return cur == kIdle;
    }

    // the leaf's next two triangles (leaves hold two by default), their six
    // loads in flight together
    __device__ __forceinline__ bool test(const Traversal& T, uint32_t& ntri) {
        const uint32_t i = (uint32_t)cur & 0x00FFFFFFu;
        const int more = (int)(((uint32_t)cur >> 24) & 0x7Fu);  // triangles after the first
        const float4* tp = (const float4*)((const char*)T.tris + i * 48u);
        const float4* tq = tp + (more ? 3 : 0);
        const float4 t0 = ldg(tp), t1 = ldg(tp + 1), t2 = ldg(tp + 2);
        const float4 u0 = ldg(tq), u1 = ldg(tq + 1), u2 = ldg(tq + 2);
        if (INSTR) ntri += more ? 2u : 1u;
        accept(i, V3{t0.x, t0.y, t0.z}, V3{t0.w, t1.x, t1.y}, V3{t1.z, t1.w, t2.x}, __float_as_uint(t2.y));
        // (a leaf of one: the same triangle again, which changes nothing)
        accept(i + (more ? 1u : 0u), V3{u0.x, u0.y, u0.z}, V3{u0.w, u1.x, u1.y}, V3{u1.z, u1.w, u2.x},
               __float_as_uint(u2.y));
        cur = more > 1 ? cur - (2 << 24) + 2 : kIdle;
        if (ANY && found()) {
            cur = kIdle;
            stk.sp = 0;
        }
        return cur == kIdle;
    }
    // mt_intersect's steps without branches: a wave of walks that rarely agree
    // runs every one anyway
    __device__ __forceinline__ void accept(uint32_t i, V3 v0, V3 e1, V3 e2, uint32_t orig) {
        const V3 pvec = cross(d, e2);
        const float det = dot(e1, pvec);
        const float inv_det = 1.0f / det;
        const V3 tvec = sub(o, v0);
        const float u = dot(tvec, pvec) * inv_det;
        const V3 qvec = cross(tvec, e1);
        const float v = dot(d, qvec) * inv_det;
        const float t = dot(e2, qvec) * inv_det;
        bool in = !((det > -0.00001f) & (det < 0.00001f)) & !(u < 0.0f) & !(u > 1.0f) & !(v < 0.0f) & !(u + v > 1.0f);
        if (ANY) {
            in &= (t > 1e-5f) & (t < 1.0f);
            best_s = in ? 0 : best_s;
        } else {
            in &= (t > 0.001f) & ((t < best_t) | ((t == best_t) & (orig < best_o)));
            best_t = in ? t : best_t;
            best_s = in ? (int)i : best_s;
            best_o = in ? orig : best_o;
        }
    }

    __device__ __forceinline__ bool step(const Traversal& T, uint32_t& nvis, uint32_t& ntri) {
        const uint64_t ml = __ballot(cur < 0), mn = __ballot((uint32_t)cur < (uint32_t)kIdle);
        bool pops = false;
        if (__popcll(ml) >= __popcll(mn)) {
            if (cur < 0) pops = test(T, ntri);
        } else if ((uint32_t)cur < (uint32_t)kIdle) {
            if (INSTR) ++nvis;
            pops = visit(T);
        }
        if (!pops) return false;
        if (stk.sp == 0) return true;
        cur = stk.pop();
        return false;
    }
};

// Returns true on a hit; best_* hold the closest hit (ANY = false).
template <int LDS, int BLOCK, int WIDTH, bool ANY, bool INSTR>
__device__ bool traverse(const Traversal& T, V3 o, V3 d, float& best_t, int& best_s, uint32_t& best_o, int* lds,
                         uint32_t gtid, uint32_t& nvis, uint32_t& ntri) {
    Walker<LDS, BLOCK, WIDTH, ANY, INSTR> w(lds, T.gstack, gtid, T.gthreads);
    w.start(T, o, d, best_t);
    while (!w.idle()) w.step(T, nvis, ntri);
    best_t = w.best_t;
    best_s = w.best_s;
    best_o = w.best_o;
    return w.found();
}

// ---------------------------------------------------------------------------
// histogram splat
// ---------------------------------------------------------------------------
// (global atomics: the accumulators' pointer comes out of a struct, and as a
// generic one it would make flat atomics, which also wait for the LDS)
typedef __attribute__((address_space(1))) unsigned long long GlobalU64;
__device__ __forceinline__ unsigned long long add_global(unsigned long long* p, unsigned long long v) {
    return __hip_atomic_fetch_add((GlobalU64*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void acc128(unsigned long long* cell, I128 q) {
    unsigned long long lo = q.lo;
    unsigned long long old = add_global(cell, lo);
    unsigned long long carry = (old + lo) < old ? 1ull : 0ull;
    unsigned long long hi = (unsigned long long)q.hi + carry;
    if (hi) add_global(cell + 1, hi);
}

// Ramp of values (w - i) * A / w at bins s + i, i in [0, w), bins < 0 and
// >= nb dropped, added to the second-difference row h: +w*S at s, -(w+1)*S
// at s+1, +S at s+w+1.  Each point is added as a magnitude to the row's "+"
// or "-" part, so no add is negative and the high word is touched only on a
// carry (one atomic per point instead of two for negative values).  Returns
// the ramp's end (one past its last bin) if bins at or past nb were cut, else
// 0 (a start before bin 0 is the reference's own skip, src/StereoRecorder.cpp:92-95).
// The span of such a ramp: start s clipped to 0 (width ww = w + s then) and
// *cut as splat_ramp returns it; false when no point lands in [0, nb).
__device__ __forceinline__ bool ramp_span(uint32_t nb, int& s, int w, int& ww, uint32_t& cut) {
    cut = 0;
    if (w <= 0) return false;
    ww = w;
    if (s < 0) {
        ww = w + s;
        s = 0;
        if (ww <= 0) return false;
    }
    const uint32_t end = (uint32_t)s + (uint32_t)ww;
    cut = end > nb ? end : 0u;
    return (uint32_t)s < nb;
}

// The three points of a ramp of slope S = A / w (its original width) from
// bin s0 (already clipped, ww bins), as magnitudes: part `hp` of the row gets
// ww * Sq at s0 and Sq at s0 + ww + 1, part `hm` (ww + 1) * Sq at s0 + 1.
struct RampPoints {
    I128 sq, aq, p1;
    bool neg;  // S < 0: the "+" and "-" parts swap
};
__device__ __forceinline__ RampPoints ramp_points(float A, int w, int ww) {
    RampPoints r;
    const double S = (double)A / (double)w;
    r.neg = S < 0.0;
    r.sq = fixed_from_double(r.neg ? -S : S);
    r.aq = i128_mul_small(r.sq, (uint32_t)ww);
    r.p1 = i128_add(r.aq, r.sq);
    return r;
}

// The one point of a ramp (see OnePoint): its slope, in two's complement
__device__ __forceinline__ I128 ramp_slope(float A, int w) {
    const double S = (double)A / (double)w;
    const I128 q = fixed_from_double(S < 0.0 ? -S : S);
    return S < 0.0 ? i128_neg(q) : q;
}

// The points of a clipped ramp (s0 < nb) added to row h with global atomics.
__device__ __forceinline__ void splat_span(unsigned long long* h, uint32_t nb, uint32_t one, uint32_t s0, int ww, int w,
                                           float A) {
    if (one) {
        acc128(h + 2 * (size_t)(s0 + ((uint32_t)w & 1u) * nb), ramp_slope(A, w));
        return;
    }
    const RampPoints q = ramp_points(A, w, ww);
    unsigned long long* hp = q.neg ? h + 2 * (size_t)nb : h;  // gets +w*S and +S
    unsigned long long* hm = q.neg ? h : h + 2 * (size_t)nb;  // gets (w+1)*S
    acc128(hp + 2 * (size_t)s0, q.aq);
    if (s0 + 1 < nb) acc128(hm + 2 * (size_t)(s0 + 1), q.p1);
    if (s0 + (uint32_t)ww + 1 < nb) acc128(hp + 2 * (size_t)(s0 + ww + 1), q.sq);
}

__device__ uint32_t splat_ramp(unsigned long long* h, uint32_t nb, uint32_t one, int s, int w, float A) {
    int ww;
    uint32_t cut;
    if (!ramp_span(nb, s, w, ww, cut)) return cut;
    splat_span(h, nb, one, (uint32_t)s, ww, w, A);
    return cut;
}

// ---------------------------------------------------------------------------
// time-tiled splat (EAR_SPLAT_TILED)
// ---------------------------------------------------------------------------
// The shadow kernel does not add a visible connection's ramps to the
// histogram itself: it writes one record per ramp, slot-indexed (the shadow
// request's index times the records per request), keyed by (histogram row,
// time tile of kTile bins).  Per bounce iteration a counting sort groups the
// records by key (k_tile_count, k_tile_scan, k_tile_scatter), and
// k_tile_splat cuts the sorted records into chunks of kTileChunk, one
// workgroup each: for every key among its records it adds the points of
// each ramp into a 128-bit accumulator tile in LDS (64-bit LDS atomics with an
// explicit carry), then adds that tile to the row in HBM, one global 128-bit
// add per touched bin.  The rays of one bounce iteration have travelled
// similar distances, so an iteration's records crowd into a few tiles; fixed
// chunks spread a crowded tile over many workgroups.  The sums are the same
// integers in another order, so the histograms are bitwise those of the
// direct splat.
constexpr uint32_t kTile = 256;             // bins per tile
constexpr uint32_t kTileChunk = 4096;       // sorted records per k_tile_splat workgroup
constexpr uint32_t kHalo = 64;              // bins past its tile that a ramp starting in it may reach
constexpr int kTileMaxW = (int)kHalo - 2;   // wider ramps are added directly
constexpr uint32_t kNoKey = 0xFFFFFFFFu;    // an empty record slot
constexpr uint32_t kLdsKeys = 8192;         // keys counted in LDS (more: global atomics)
constexpr uint32_t kTileDirect = 32;        // keys with at most this many ramps skip the LDS tile
constexpr int kTileBlock = 256;

// where the shadow kernels put their records (key == nullptr: direct splat)
struct TileOut {
    uint32_t* key;    // [request * stride + r]: tile key or kNoKey
    uint2* pay;       // {A bits, offset in tile | ww << 16 | w << 24}
    uint32_t stride;  // records per request: the most channels of one recorder
};

// Row layout of the accumulators.  Without the |c| histogram one signed row
// per channel.  With it, contributions are split by sign: row 0 takes the
// ramps of c >= 0, row 1 the ramps of |c| for c < 0, so each contribution
// updates one row; the finalize step turns them into signed = P - N and
// |.| = P + N (exact: quantisation is odd-symmetric, the sums are integers).
//
// OnePoint: a ramp's width is the ceiling of the root of its distance, and its
// bin is that distance over the speed of sound, moved by at most the head's
// half delay: the distances that fall on one bin span less than a metre, and
// their widths are one of two consecutive numbers.  So a row's two parts hold
// the slopes of the ramps of even and of odd width that start at each bin, one
// 128-bit add per ramp instead of three (a negative slope as its two's
// complement), and k_finish, which knows from the bin which two widths they
// are, sums the ramps into the bins they cover: the same integers.  Per pass
// (adds skipped altogether in a copy): 32 rooms 36 of 198 ms, the 1M-ray box 6
// of 40, a room with an emitting mesh 10 of 54 went to the three adds.
// Without it (a head of nearly half a metre, or bins too late for binary32
// distances: make_params) the parts are the "+" and "-" of second differences.
struct Hist {
    unsigned long long* cells;  // [band slot][channel][kind][part][bin] x {lo, hi}
    uint32_t n_bins, n_ch, kinds, one;
    uint32_t key_base, n_tiles;  // the time-tiled splat's keys of this render
    __device__ uint32_t row_index(int band, int ch, int kind) const {
        return ((uint32_t)band * n_ch + (uint32_t)ch) * kinds + (uint32_t)kind;
    }
    // the row's first part; its second follows at + 2 * n_bins
    __device__ unsigned long long* row(int band, int ch, int kind) const {
        return cells + 4 * (size_t)n_bins * row_index(band, ch, kind);
    }
};

// Records of one connection for the time-tiled splat: they go to
// out.key / out.pay [base, base + out.stride); `used` so far.
struct TileSink {
    TileOut out;
    uint32_t base, used;
    // the slots this connection left empty
    __device__ void close() {
        for (uint32_t r = used; r < out.stride; ++r) out.key[base + r] = kNoKey;
    }
};

// One ramp into row (band, ch, kind): splat directly, or as a record when a
// sink is given (ramps wider than the tile halo are still splatted).
__device__ __forceinline__ void put_ramp(const Hist& H, int band, int ch, int kind, int s, int w, float A, Drops& dr,
                                         TileSink& sink, bool tiled) {
    if (!tiled) {
        dr.add(splat_ramp(H.row(band, ch, kind), H.n_bins, H.one, s, w, A));
        return;
    }
    int ww;
    uint32_t cut;
    const bool any = ramp_span(H.n_bins, s, w, ww, cut);
    dr.add(cut);
    if (!any) return;
    if (w > kTileMaxW) {
        splat_span(H.row(band, ch, kind), H.n_bins, H.one, (uint32_t)s, ww, w, A);
        return;
    }
    const uint32_t i = sink.base + sink.used++;
    sink.out.key[i] = H.key_base + H.row_index(band, ch, kind) * H.n_tiles + (uint32_t)s / kTile;
    sink.out.pay[i] = make_uint2(__float_as_uint(A), ((uint32_t)s % kTile) | ((uint32_t)ww << 16) | ((uint32_t)w << 24));
}

// Recorder::Record: MonoRecorder (src/MonoRecorder.cpp:83-97) or
// StereoRecorder (src/StereoRecorder.cpp:97-130).
// MonoRecorder::Record (src/MonoRecorder.cpp:83-97) into channel ch
__device__ __forceinline__ void record_channel(const Hist& H, int band, int ch, float a, float t, float dist,
                                               Drops& dr, TileSink& sink, bool tiled) {
    const bool split = H.kinds > 1;
    const uint32_t kind = split && a < 0.0f ? 1u : 0u;
    int s = (int)((double)t * 44100.0);
    float width = sqrtf(dist);
    float ampl = 2.0f * a / width;
    int w = (int)ceilf(width);
    put_ramp(H, band, ch, (int)kind, s, w, split ? fabsf(ampl) : ampl, dr, sink, tiled);
}
__device__ void record_channel(const Hist& H, int band, int ch, float a, float t, float dist, Drops& dr) {
    TileSink none{};
    record_channel(H, band, ch, a, t, dist, dr, none, false);
}

// Returns the number of ramps (channels) of the connection.
__device__ __forceinline__ uint32_t record(const Hist& H, int band, const RecParams& R, V3 dir, float a, float t,
                                           float dist, Drops& dr, TileSink& sink, bool tiled) {
    const bool split = H.kinds > 1;
    const uint32_t kind = split && a < 0.0f ? 1u : 0u;
    if (R.kind == EAR_REC_MONO) {
        record_channel(H, band, R.channel, a, t, dist, dr, sink, tiled);
        return 1;
    } else {
        float dt = dot(dir, V3{R.rx, R.ry, R.rz});
        float td = R.head_size / 343.0f;
        int s_right = (int)((double)(t - dt * td) * 44100.0);
        int s_left = (int)((double)(t + dt * td) * 44100.0);
        float width = sqrtf(dist);
        float ampl = 2.0f * a / width;
        float al = ampl, ar = ampl;
        float factor = powf_ear_l2(R.head_abs[band], R.l2_head_abs[band], fabsf(dt) * R.head_size);
        if (dt < 0.0f)
            ar *= factor * factor;
        else
            al *= factor * factor;
        int w = (int)ceilf(width);
        put_ramp(H, band, R.channel, (int)kind, s_left, w, split ? fabsf(al) : al, dr, sink, tiled);
        put_ramp(H, band, R.channel + 1, (int)kind, s_right, w, split ? fabsf(ar) : ar, dr, sink, tiled);
        return 2;
    }
}
__device__ uint32_t record(const Hist& H, int band, const RecParams& R, V3 dir, float a, float t, float dist,
                           Drops& dr) {
    TileSink none{};
    return record(H, band, R, dir, a, t, dist, dr, none, false);
}

// Receiver spheres (EAR_EST_SPHERE): the segment o + s u, s in [0, seg),
// deposits into every sphere it crosses I0 air^s0 (s1 - s0) / (4/3 pi r^3)
// at distance L0 + s0, [s0, s1) being the chord clipped to the segment (the
// track-length form of counting crossings).  j = reflections before the
// segment: sign (-1)^j, and dry on a point source's first segment.  Returns
// the number of deposits.
__device__ uint32_t sphere_deposits(const Hist& H, const RenderParams& P, int band, V3 o, V3 u, float seg, float I0,
                                    float L0, uint32_t j, Drops& dr) {
    uint32_t n = 0;
    for (uint32_t r = 0; r < P.n_rec; ++r) {
        const RecParams& R = P.rec[r];
        const int nc = R.kind == EAR_REC_STEREO ? 2 : 1;
        for (int e = 0; e < nc; ++e) {
            const V3 oc = sub(o, V3{R.cen[e][0], R.cen[e][1], R.cen[e][2]});
            const float b = dot(oc, u);
            const float disc = b * b - (dot(oc, oc) - R.r2);
            if (!(disc > 0.0f)) continue;
            const float q = sqrtf(disc);
            const float s0 = fmaxf(-b - q, 0.0f), s1 = fminf(-b + q, seg);
            if (!(s1 > s0)) continue;
            float c = I0;
            c *= powf_ear_l2(P.air[band], P.l2_air[band], s0);
            c *= s1 - s0;
            c *= R.inv_vol;
            if (j == 0 && P.src_kind == EAR_SRC_POINT) c *= P.dry;
            if (!is_normal(c)) continue;
            if (j & 1u) c *= -1.0f;
            const float dist = L0 + s0;
            record_channel(H, band, R.channel + e, c, dist / 343.0f, dist, dr);
            ++n;
        }
    }
    return n;
}

// ---------------------------------------------------------------------------
// per-instance device table
// ---------------------------------------------------------------------------
struct MeshSrc {
    const float* v;     // [n][9]
    const float* area;  // [n]
    const float* nrm;   // [n][3]
};

// direct sound per (band, channel) (src/Scene.cpp:299-311): {visible, s, w, A}
struct DirectRamp {
    int32_t visible, s, w;
    float a;
};

// One render instance: a (scene, render description) pair of a batch.  A
// plain render is a batch of one.
struct InstDev {
    RenderParams P;
    const BvhNode* nodes;
    const Bvh4Node* nodes4;
    const float4* tris;
    const float4* nm;
    const float4* mat_band;
    uint32_t n_tris;
    uint32_t key_base;  // time-tiled splat: first tile key of this render
    uint32_t n_tiles;   // and tiles per histogram row
    uint32_t pad0;
    MeshSrc M;
    unsigned long long* hist;  // [3][n_ch][kinds][bins] x 2
    DirectRamp* direct;        // [3][n_ch]
    double* value;             // [3][n_ch][kinds][bins] or null
    int32_t* log_hits;         // [3][trace_rays][trace_segs] or null
    uint32_t* log_nseg;        // [3][trace_rays]
    double inv_n, gain2;
};

// a run of rays of one (instance, band) context inside a chunk
struct GenSeg {
    uint32_t inst, band, ray0, count;
};

__device__ __forceinline__ Traversal make_trav(const InstDev& I, int* gstack, uint32_t gthreads) {
    return Traversal{I.nodes, I.nodes4, I.tris, I.n_tris, gstack, gthreads};
}
__device__ __forceinline__ Hist make_hist(const InstDev& I) {
    return Hist{I.hist, I.P.n_bins, I.P.n_channels, I.P.hist_kinds, I.P.one_point, I.key_base, I.n_tiles};
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// Emission, k = 0 (AbstractSoundFile::SoundRay, src/SoundFile.cpp:215-228).
// Thread gid of the chunk maps to (instance, band, ray) through the segment
// table (exclusive prefix `seg_off`, binary search).
template <bool BATCH>
__global__ void __launch_bounds__(kBlock) k_generate(const InstDev* __restrict__ inst, const GenSeg* __restrict__ segs,
                                                      const uint32_t* __restrict__ seg_off, uint32_t n_segs,
                                                      uint32_t total, const uint32_t* __restrict__ plan,
                                                      uint32_t max_rec, uint32_t any_mesh, uint32_t dense, Queue q,
                                                      uint32_t* __restrict__ n_q, ShadowQ sq,
                                                      uint32_t* __restrict__ n_sq, unsigned long long* __restrict__ stats) {
    // rays [first, first + total) of the segment table; a plan written on the
    // device (k_plan) overrides the host's range.  dense: every ray is live, so
    // ray i of the range has slot plan[2] + i and k_plan counts them (an
    // append's atomic per wave, 12.5 ns each on one address, was this kernel's
    // whole time: 5.7 ms of a 30M-ray render, 1.3 ms without)
    uint32_t first = 0;
    if (plan) {
        first = plan[0];
        total = plan[1];
    }
    __shared__ HemiLds hl[kBlock / 64];
    uint32_t n_done = 0;
    for (uint32_t base = blockIdx.x * kBlock; base < total; base += gridDim.x * kBlock) {
        uint32_t gid = first + base + threadIdx.x;
        const uint32_t end = first + total;
        bool valid = gid < end;
        bool live = false;
        float4 ro{}, rd{};
        uint4 rm{};
        int band = 0;
        uint32_t id = 0;
        Rng rng;
        V3 o{0, 0, 0}, sn{0, 0, 0};
        bool mesh_src = false;
        uint32_t n_rec = 0;
        if (valid) {
            uint32_t lo = 0, hi = n_segs - 1;
            while (lo < hi) {  // last segment with seg_off <= gid
                uint32_t mid = (lo + hi + 1) >> 1;
                if (seg_off[mid] <= gid)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            const GenSeg g = segs[lo];
            id = BATCH ? g.inst : 0;
            const InstDev& I = inst[id];
            const RenderParams& P = I.P;
            band = (int)g.band;
            uint32_t ray = g.ray0 + (gid - seg_off[lo]);
            rng.init(P.seed, ray, P.ctx_word[band], P.instance, 0);
            mesh_src = P.src_kind == EAR_SRC_MESH;
            n_rec = P.n_rec;
            if (mesh_src) {
                float x = rng.next() * P.src_total_area;
                uint32_t pick = P.src_n_tris - 1;
                for (uint32_t i = 0; i < P.src_n_tris; ++i) {
                    x -= I.M.area[i];
                    if (x < 0.0f) {
                        pick = i;
                        break;
                    }
                }
                const float* v = I.M.v + 9 * (size_t)pick;
                float r1 = rng.next();
                float r2 = rng.next();
                float sr1 = sqrtf(r1);
                float ca = 1.0f - sr1, cb = sr1 * (1.0f - r2), cc = sr1 * r2;
                o = V3{ca * v[0] + cb * v[3] + cc * v[6], ca * v[1] + cb * v[4] + cc * v[7],
                       ca * v[2] + cb * v[5] + cc * v[8]};
                sn = V3{I.M.nrm[3 * pick], I.M.nrm[3 * pick + 1], I.M.nrm[3 * pick + 2]};
            } else {
                o = V3{P.src_pos[0], P.src_pos[1], P.src_pos[2]};
            }
            live = !((double)1.0f < P.cutoff) && P.max_bounces > 0;
        }
        // a mesh source's hemisphere, a point source's sphere
        const V3 d = sample_hemi_wave(valid, mesh_src, rng, sn, hl[threadIdx.x >> 6]);
        if (valid) {
            ro = make_float4(o.x, o.y, o.z, 1.0f);
            rd = make_float4(d.x, d.y, d.z, 0.0f);
            rm = make_uint4(rng.ray, rng.draw, (uint32_t)band, id);
        }
        // mesh sources connect to every recorder at k = 0 (src/Scene.cpp:185)
        if (any_mesh) {
            for (uint32_t r = 0; r < max_rec; ++r) {
                bool emit = false;
                float c = 0.0f;
                if (valid && mesh_src && r < n_rec && inst[id].P.estimator == EAR_EST_NEE) {
                    const RecParams& R = inst[id].P.rec[r];
                    V3 dv = sub(V3{R.px, R.py, R.pz}, o);
                    float l = length(dv);
                    c = 1.0f;
                    c *= powf_ear_l2(inst[id].P.air[band], inst[id].P.l2_air[band], l);
                    c *= 2.0f / (4.0f * kPi * l * l);
                    emit = is_normal(c);
                }
                uint32_t slot = wave_append(n_sq, emit);
                if (emit) {
                    sq.p[slot] = make_float4(o.x, o.y, o.z, c);
                    sq.m[slot] = make_float4(0.0f, __uint_as_float(r | ((uint32_t)band << 8)), __uint_as_float(id),
                                             0.0f);
                }
            }
        }
        const uint32_t slot = dense ? plan[2] + base + threadIdx.x : wave_append(n_q, live);
        if (live) {
            q.o[slot] = ro;
            q.d[slot] = rd;
            q.m[slot] = rm;
        }
        n_done += valid ? 1u : 0u;
    }
    stat_add(stats, ST_RAYS, n_done);
}

template <int BLOCK, int LDS, int WIDTH, bool INSTR, bool BATCH>
__global__ void __launch_bounds__(BLOCK) k_extend(const InstDev* __restrict__ inst, int* gstack, uint32_t gthreads,
                                                   Queue q, const uint32_t* __restrict__ n_q, int2* __restrict__ hits,
                                                   unsigned long long* __restrict__ stats, Fetch /*fetch*/) {
    __shared__ int lds[LDS * BLOCK];
    uint32_t n = *n_q;
    uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    uint32_t nvis = 0, ntri = 0;
    for (uint32_t base = blockIdx.x * BLOCK; base < n; base += gridDim.x * BLOCK) {
        uint32_t i = base + threadIdx.x;
        if (i < n) {
            float4 o = q.o[i], d = q.d[i];
            uint32_t id = BATCH ? q.m[i].w : 0;
            Traversal T = make_trav(inst[id], gstack, gthreads);
            float bt = 1000000.0f;
            int bs = -1;
            uint32_t bo = 0;
            traverse<LDS, BLOCK, WIDTH, false, INSTR>(T, V3{o.x, o.y, o.z}, V3{d.x, d.y, d.z}, bt, bs, bo,
                                                      lds + threadIdx.x, gtid, nvis, ntri);
            hits[i] = make_int2(__float_as_int(bt), bs);
        }
    }
    if (INSTR) {
        stat_add(stats, ST_NV_CL, nvis);
        stat_add(stats, ST_NT_CL, ntri);
    }
}

// Scene::Bounce + Material::Bounce + the energy bookkeeping and NEE weight of
// Scene::Render (src/Scene.cpp:49-82, 151-277, src/Material.cpp:76-83).
// Six waves per SIMD: the register cap that costs no spills (2% faster than
// the five the compiler picks by itself).
// The surface interaction of a segment from ro/rd that hit triangle h.y at
// t = h.x (src/Scene.cpp:143-175): hit point, the normal facing the ray
// (negated for REFRACT), Material::Bounce's uniform (its Philox stream
// starts here), air over the segment and the material's retention.
__device__ __forceinline__ void surface_hit(const InstDev& In, const RenderParams& P, int band, float4 ro, float4 rd,
                                            uint4 rm, int2 h, Rng& rng, V3& p, V3& nrm, V3& prev, V3& d, float& I,
                                            float& L, float& spec, float& seg, int& bt, bool& alive) {
    float t = __int_as_float(h.x);
    V3 o{ro.x, ro.y, ro.z};
    d = V3{rd.x, rd.y, rd.z};
    p = V3{o.x + d.x * t, o.y + d.y * t, o.z + d.z * t};
    float4 nmv = ldg(In.nm + h.y);
    V3 N{nmv.x, nmv.y, nmv.z};
    nrm = dot(N, d) > 0.0f ? V3{N.x * -1.0f, N.y * -1.0f, N.z * -1.0f} : N;
    uint32_t mat = __float_as_uint(nmv.w);
    float4 mb = ldg(In.mat_band + 3 * mat + band);  // {fl2 | -1, spec, retention, -}
    rng.init(P.seed, rm.x, P.ctx_word[band], P.instance, rm.y);
    bt = kReflect;
    if (mb.x >= 0.0f) bt = (rng.next() <= mb.x) ? kReflect : kRefract;
    spec = mb.y;
    if (bt == kRefract) nrm = neg(nrm);
    float l = length(sub(p, o));
    I = ro.w;
    I *= powf_ear_l2(P.air[band], P.l2_air[band], l);
    L = rd.w + l;
    I *= mb.z;
    alive = is_normal(I);
    prev = normalized(d);
    seg = l;
}

// The next-event weight of the connection from hit point p to recorder R
// (src/Scene.cpp:185-268): false if it faces away or is not FP_NORMAL;
// c carries the sign of the k-th reflection.
__device__ __forceinline__ bool nee_weight(const RenderParams& P, const RecParams& R, int band, V3 p, V3 nrm, V3 prev,
                                           int bt, float spec, float I, uint32_t k, float& c) {
    V3 dv = sub(V3{R.px, R.py, R.pz}, p);
    V3 lsdir = normalized(dv);
    float dt = dot(lsdir, nrm);
    if (!(dt > 0.0f)) return false;
    // factor = spec * 1001 * sf^1000 + (1 - spec) * diff; with spec == 0 the
    // lobe term is exactly +0 (sf^1000 is finite), so its binary64 pow is
    // skipped without changing a bit
    float diff, sf;
    if (bt == kReflect) {
        V3 rv = reflect(prev, nrm);
        diff = -dot(nrm, prev);
        sf = fmaxf(0.0f, dot(rv, lsdir));
    } else {
        diff = dot(nrm, prev);
        sf = fmaxf(0.0f, dot(prev, lsdir));
    }
    const float lobe = spec != 0.0f ? spec * kExpInt * powf_ear(sf, kExp) : 0.0f;
    const float factor = lobe + (1.0f - spec) * diff;
    c = I;
    c *= factor;
    float l = length(dv);
    c *= powf_ear_l2(P.air[band], P.l2_air[band], l);
    c *= 2.0f / (4.0f * kPi * l * l);
    if (!is_normal(c)) return false;
    if (k & 1u) c *= -1.0f;
    return true;
}

template <bool BATCH>
__global__ void __launch_bounds__(kShadeBlock, 6) k_shade(const InstDev* __restrict__ inst, Queue qin,
                                                   const uint32_t* __restrict__ n_in, const int2* __restrict__ hits,
                                                   Queue qout, ShadowQ sq, unsigned long long* __restrict__ n_out,
                                                   uint32_t max_rec, unsigned long long* __restrict__ stats) {
    __shared__ unsigned long long sc[2][kShadeBlock / 64];  // scratch of the block-wide appends, alternated
    __shared__ HemiLds hl[kShadeBlock / 64];
    uint32_t n = *n_in;
    uint32_t n_done = 0, n_sph = 0;
    Drops drops;
    for (uint32_t base = blockIdx.x * kShadeBlock; base < n; base += gridDim.x * kShadeBlock) {
        uint32_t i = base + threadIdx.x;
        bool valid = i < n;
        bool alive = false;  // hit and intensity normal: NEE runs
        bool cont = false;   // continues to the next segment
        uint4 rm{};
        V3 p{0, 0, 0}, nrm{0, 0, 0}, prev{0, 0, 0}, d{0, 0, 0};
        float I = 0.0f, L = 0.0f, spec = 0.0f;
        int bt = kReflect;
        int band = 0;
        uint32_t k = 0, id = 0, n_rec = 0;
        float seg = __int_as_float(0x7f800000);  // segment length; +inf for a miss
        bool nee = true;
        Rng rng;
        if (valid) {
            float4 ro = qin.o[i];
            float4 rd = qin.d[i];
            rm = qin.m[i];
            id = BATCH ? rm.w : 0;
            const InstDev& In = inst[id];
            const RenderParams& P = In.P;
            n_rec = P.n_rec;
            band = (int)(rm.z & 0xFFu);
            k = ((rm.z >> 8) & 0xFFFFu) + 1;  // this segment's bounce number
            int2 h = hits[i];
            if (In.log_hits && rm.x < P.trace_rays) {
                if (k - 1 < P.trace_segs)
                    In.log_hits[((size_t)band * P.trace_rays + rm.x) * P.trace_segs + (k - 1)] =
                        h.y >= 0 ? (int32_t)__float_as_uint(ldg(In.tris + 3 * h.y + 2).y) : -1;
                In.log_nseg[(size_t)band * P.trace_rays + rm.x] = k;
            }
            if (h.y >= 0) surface_hit(In, P, band, ro, rd, rm, h, rng, p, nrm, prev, d, I, L, spec, seg, bt, alive);
            if (P.estimator == EAR_EST_SPHERE) {
                // hit or miss, the segment crosses the receiver spheres
                n_sph += sphere_deposits(make_hist(In), P, band, V3{ro.x, ro.y, ro.z},
                                         normalized(V3{rd.x, rd.y, rd.z}), seg, ro.w, rd.w, k - 1, drops);
                nee = false;
            }
        }
        // NEE to every recorder (src/Scene.cpp:185-268).  The slots of the
        // connections and of the continuing rays come from one append, so the
        // connections are counted before they are stored; the first two
        // recorders' weights are kept for that, the others' computed again
        // (the 200k hall of 3 x 3M rays with 8 recorders: 290 ms, 548 with an
        // append and one weight per recorder).
        auto weight = [&](uint32_t r, float& c) -> bool {
            if (!(alive && nee && r < n_rec)) return false;
            const RenderParams& P = inst[id].P;
            return nee_weight(P, P.rec[r], band, p, nrm, prev, bt, spec, I, k, c);
        };
        if (alive) cont = !((double)I < inst[id].P.cutoff) && k < inst[id].P.max_bounces;
        float c0 = 0.0f, c1 = 0.0f;
        const bool e0 = max_rec > 0 && weight(0, c0), e1 = max_rec > 1 && weight(1, c1);
        uint32_t n_con = (uint32_t)(__popcll(__ballot(e0)) + __popcll(__ballot(e1)));
        for (uint32_t r = 2; r < max_rec; ++r) {
            float c = 0.0f;
            n_con += (uint32_t)__popcll(__ballot(weight(r, c)));
        }
        const uint64_t mcont = __ballot(cont);
        const uint64_t below = (1ull << lane_id()) - 1ull;
        const uint2 first = block_append2<kShadeBlock>(n_out, (uint32_t)__popcll(mcont), n_con,
                                                       sc[(base / (gridDim.x * kShadeBlock)) & 1u]);
        uint32_t next = first.y;
        for (uint32_t r = 0; r < max_rec; ++r) {
            float c = r == 0 ? c0 : c1;
            const bool emit = r == 0 ? e0 : r == 1 ? e1 : weight(r, c);
            const uint64_t m = __ballot(emit);
            if (emit) {
                const uint32_t slot = next + (uint32_t)__popcll(m & below);
                sq.p[slot] = make_float4(p.x, p.y, p.z, c);
                sq.m[slot] = make_float4(L, __uint_as_float(r | ((uint32_t)band << 8)), __uint_as_float(id), 0.0f);
            }
            next += (uint32_t)__popcll(m);
        }
        const V3 hv = sample_hemi_wave(cont, true, rng, nrm, hl[threadIdx.x >> 6]);
        if (cont) {
            // REFRACT: the negated normal and the incoming direction; REFLECT:
            // the mirror direction about the ray-facing normal (src/Scene.cpp:65-74)
            V3 rdir = bt == kRefract ? d : reflect(d, nrm);
            V3 v = blend_spec(hv, rdir, spec);
            const uint32_t slot = first.x + (uint32_t)__popcll(mcont & below);
            qout.o[slot] = make_float4(p.x, p.y, p.z, I);
            qout.d[slot] = make_float4(v.x, v.y, v.z, L);
            qout.m[slot] = make_uint4(rm.x, rng.draw, (uint32_t)band | (k << 8), id);
        }
        n_done += valid ? 1u : 0u;
    }
    stat_add(stats, ST_SEGMENTS, n_done);
    stat_add(stats, ST_CONTRIB, n_sph);
    stat_drops(stats, drops);
}

// The tail of the bounce loop: once every ray has been emitted and few are
// left, each lane carries its rays through all their remaining segments in
// one launch (closest hit as k_extend, the surface interaction and
// next-event weights as k_shade, visibility and splat as k_shadow, the next
// direction as k_shade), instead of one launch of each kernel per segment,
// whose time is then set by the latency of a few walks.  The same device
// functions in the same order: every path, and so every histogram sum, is
// the wavefront loop's.  A path ends by a miss, a non-normal intensity, the
// cut-off or max_bounces, so every lane's loop ends.  Not used with hit
// logging or counter instrumentation.
//
// A wave's lanes go through one segment of their paths together: walk, shade,
// connect, sample.  A lane whose path has ended takes the next ray before the
// next segment (with the lanes of a wave on one ray each until the longest
// path ended, and each lane drawing its own hemisphere candidates, the
// 12-triangle box of 1M rays took 21.7 ms here against 14.5).  A queue
// shorter than the grid is spread over all its waves, down to kTailMin rays
// each: a segment then waits for the longest of fewer walks, and the chip has
// the waves to spare.
constexpr uint32_t kTailMin = 8;
template <int BLOCK, int LDS, int WIDTH, bool BATCH>
__global__ void __launch_bounds__(BLOCK, 4) k_tail(const InstDev* __restrict__ inst, int* gstack, uint32_t gthreads,
                                                Queue q, const uint32_t* __restrict__ n_q, uint32_t max_rec,
                                                Fetch fetch, unsigned long long* __restrict__ stats) {
    __shared__ int lds[LDS * BLOCK];
    __shared__ HemiLds hl[BLOCK / 64];
    const uint32_t n = *n_q;
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t waves = gridDim.x * (BLOCK / 64);
    uint32_t n_seg = 0, nsh = 0, ncon = 0, nvis = 0, ntri = 0;
    Drops drops;
    Claim claim(n, gtid, gridDim.x * BLOCK, fetch, min(64u, max(kTailMin, n / waves + (n % waves ? 1u : 0u))));
    bool live = false;
    float4 ro{}, rd{};
    uint4 rm{};
    uint32_t id = 0;
    for (;;) {
        const uint64_t idle = __ballot(!live);
        if (idle && !claim.exhausted()) {
            const uint32_t mine = claim.take(fetch, idle, lane);
            if (mine != 0xFFFFFFFFu) {
                ro = q.o[mine];
                rd = q.d[mine];
                rm = q.m[mine];
                id = BATCH ? rm.w : 0u;
                live = true;
            }
        }
        if (__ballot(live) == 0) break;
        const InstDev& In = inst[id];
        const RenderParams& P = In.P;
        const Traversal T = make_trav(In, gstack, gthreads);
        const int band = (int)(rm.z & 0xFFu);
        const uint32_t k = ((rm.z >> 8) & 0xFFFFu) + 1;  // this segment's bounce number
        int2 h = make_int2(0, -1);
        {
            Walker<LDS, BLOCK, WIDTH, false, false> w(lds + threadIdx.x, gstack, gtid, gthreads);
            if (live) w.start(T, V3{ro.x, ro.y, ro.z}, V3{rd.x, rd.y, rd.z}, 1000000.0f);
            while (__ballot(!w.idle())) w.step(T, nvis, ntri);
            h = make_int2(__float_as_int(w.best_t), w.best_s);
        }
        n_seg += live ? 1u : 0u;
        Rng rng;
        V3 p{0, 0, 0}, nrm{0, 0, 0}, prev{0, 0, 0}, d{0, 0, 0};
        float I = 0.0f, L = 0.0f, spec = 0.0f;
        float seg = __int_as_float(0x7f800000);  // segment length; +inf for a miss
        int bt = kReflect;
        bool alive = false;
        // no hit ends the path (src/Scene.cpp:166)
        if (live && h.y >= 0) surface_hit(In, P, band, ro, rd, rm, h, rng, p, nrm, prev, d, I, L, spec, seg, bt, alive);
        const bool nee = P.estimator == EAR_EST_NEE;
        if (live && !nee)
            ncon += sphere_deposits(make_hist(In), P, band, V3{ro.x, ro.y, ro.z}, normalized(V3{rd.x, rd.y, rd.z}), seg,
                                    ro.w, rd.w, k - 1, drops);
        for (uint32_t r = 0; r < max_rec; ++r) {
            float c = 0.0f;
            const RecParams& R = P.rec[r];
            const bool emit = alive && nee && r < P.n_rec && nee_weight(P, R, band, p, nrm, prev, bt, spec, I, k, c);
            // Scene::Connect: the segment from the hit point to the recorder
            const V3 dv = sub(V3{R.px, R.py, R.pz}, p);
            Walker<LDS, BLOCK, WIDTH, true, false> w(lds + threadIdx.x, gstack, gtid, gthreads);
            if (emit) w.start(T, p, dv, 0.0f);
            while (__ballot(!w.idle())) w.step(T, nvis, ntri);
            nsh += emit ? 1u : 0u;
            if (emit && !w.found()) {
                const float l = length(dv);
                record(make_hist(In), band, R, normalized(dv), c, (L + l) / 343.0f, L + l, drops);
                ++ncon;
            }
        }
        live = alive && !((double)I < P.cutoff) && k < P.max_bounces;
        const V3 hv = sample_hemi_wave(live, true, rng, nrm, hl[threadIdx.x >> 6]);
        if (live) {
            // REFRACT: the negated normal and the incoming direction; REFLECT:
            // the mirror direction about the ray-facing normal (src/Scene.cpp:65-74)
            const V3 rdir = bt == kRefract ? d : reflect(d, nrm);
            const V3 v = blend_spec(hv, rdir, spec);
            ro = make_float4(p.x, p.y, p.z, I);
            rd = make_float4(v.x, v.y, v.z, L);
            rm = make_uint4(rm.x, rng.draw, (uint32_t)band | (k << 8), id);
        }
    }
    stat_add(stats, ST_SEGMENTS, n_seg);
    stat_add(stats, ST_SHADOW, nsh);
    stat_add(stats, ST_CONTRIB, ncon);
    stat_add(stats, ST_TAIL_SEG, n_seg);
    stat_add(stats, ST_TAIL_SH, nsh);
    stat_drops(stats, drops);
}

// Scene::Connect + Mesh::LineIntersection (src/Scene.cpp:84-96,
// src/Mesh.cpp:58-71), then Recorder::Record for visible connections.
template <int BLOCK, int LDS, int WIDTH, bool INSTR, bool BATCH, bool TILED>
__global__ void __launch_bounds__(BLOCK) k_shadow(const InstDev* __restrict__ inst, int* gstack, uint32_t gthreads,
                                                   ShadowQ sq, const uint32_t* __restrict__ n_sq,
                                                   unsigned long long* __restrict__ stats, Fetch /*fetch*/,
                                                   TileOut to) {
    __shared__ int lds[LDS * BLOCK];
    uint32_t n = *n_sq;
    uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    uint32_t nvis = 0, ntri = 0, ncon = 0, nsh = 0, nramp = 0;
    Drops drops;
    for (uint32_t base = blockIdx.x * BLOCK; base < n; base += gridDim.x * BLOCK) {
        uint32_t i = base + threadIdx.x;
        if (i < n) {
            float4 pc = sq.p[i], m = sq.m[i];
            uint32_t packed = __float_as_uint(m.y);
            int r = (int)(packed & 0xFFu), band = (int)((packed >> 8) & 0xFFu);
            uint32_t id = BATCH ? __float_as_uint(m.z) : 0;
            const InstDev& In = inst[id];
            const RecParams& R = In.P.rec[r];
            V3 p{pc.x, pc.y, pc.z};
            V3 dv = sub(V3{R.px, R.py, R.pz}, p);
            float bt = 0.0f;
            int bs = -1;
            uint32_t bo = 0;
            ++nsh;
            Traversal T = make_trav(In, gstack, gthreads);
            bool occ = traverse<LDS, BLOCK, WIDTH, true, INSTR>(T, p, dv, bt, bs, bo, lds + threadIdx.x, gtid, nvis,
                                                                ntri);
            TileSink sink{to, i * to.stride, 0};
            if (!occ) {
                float l = length(dv);
                V3 lsdir = normalized(dv);
                float L = m.x;
                nramp += record(make_hist(In), band, R, lsdir, pc.w, (L + l) / 343.0f, L + l, drops, sink, TILED);
                ++ncon;
            }
            if (TILED) sink.close();
        }
    }
    stat_add(stats, ST_SHADOW, nsh);
    stat_add(stats, ST_CONTRIB, ncon);
    stat_add(stats, ST_SH_CONTRIB, ncon);
    stat_add(stats, ST_SH_RAMPS, nramp);
    stat_drops(stats, drops);
    if (INSTR) {
        stat_add(stats, ST_NV_SH, nvis);
        stat_add(stats, ST_NT_SH, ntri);
    }
}

// Persistent variants of k_extend / k_shadow: a lane whose walk has ended
// takes the next queue entry, so a wave keeps its lanes busy instead of
// waiting for its slowest ray (Aila & Laine, "Understanding the Efficiency of
// Ray Traversal on GPUs", HPG 2009).  A wave hands out entries when at least
// fetch.refill of its lanes are idle, from a run of fetch.chunk entries it
// claims with one atomic.  Each lane keeps its own traversal stack across the
// rays it takes.

template <int BLOCK, int LDS, int WIDTH, bool INSTR, bool BATCH>
__global__ void __launch_bounds__(BLOCK) k_extend_f(const InstDev* __restrict__ inst, int* gstack, uint32_t gthreads,
                                                     Queue q, const uint32_t* __restrict__ n_q,
                                                     int2* __restrict__ hits, unsigned long long* __restrict__ stats,
                                                     Fetch fetch) {
    __shared__ int lds[LDS * BLOCK];
    const uint32_t n = *n_q;
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t lane = lane_id();
    uint32_t nvis = 0, ntri = 0;
    Walker<LDS, BLOCK, WIDTH, false, INSTR> w(lds + threadIdx.x, gstack, gtid, gthreads);
    Traversal T = make_trav(inst[0], gstack, gthreads);
    Claim claim(n, gtid, gridDim.x * blockDim.x, fetch);
    uint32_t refill = fetch.refill;  // idle lanes that trigger a refill
    // A finished hit is stored with the wave's others at its next refill, so
    // that the 8-byte records of a claimed run reach their cache lines in a
    // few bursts instead of one lane at a time.
    uint32_t slot = 0xFFFFFFFFu;  // this lane's queue entry
    for (;;) {
        const uint64_t idle = __ballot(w.idle());
        if ((uint32_t)__popcll(idle) >= refill) {
            const uint32_t mine = claim.take(fetch, idle, lane);
            if (w.idle()) {
                if (slot != 0xFFFFFFFFu) hits[slot] = make_int2(__float_as_int(w.best_t), w.best_s);
                slot = mine;
                if (slot != 0xFFFFFFFFu) {
                    const float4 o = q.o[slot], d = q.d[slot];
                    if (BATCH) T = make_trav(inst[q.m[slot].w], gstack, gthreads);
                    w.start(T, V3{o.x, o.y, o.z}, V3{d.x, d.y, d.z}, 1000000.0f);
                }
            }
            // the loop is left by the whole wave at once, with no walk and no
            // hit left; with nothing left to take the next look is at the end
            if (__ballot(slot != 0xFFFFFFFFu) == 0) break;
            if (claim.exhausted()) refill = 64u;
        }
        w.step(T, nvis, ntri);
    }
    if (INSTR) {
        stat_add(stats, ST_NV_CL, nvis);
        stat_add(stats, ST_NT_CL, ntri);
    }
}

template <int BLOCK, int LDS, int WIDTH, bool INSTR, bool BATCH, bool TILED>
__global__ void __launch_bounds__(BLOCK, 6) k_shadow_f(const InstDev* __restrict__ inst, int* gstack, uint32_t gthreads,
                                                     ShadowQ sq, const uint32_t* __restrict__ n_sq,
                                                     unsigned long long* __restrict__ stats, Fetch fetch,
                                                     TileOut to) {
    __shared__ int lds[LDS * BLOCK];
    // per wave: request slots of visible connections awaiting their records
    // (a lane adds at most one per pass of the loop below and each pass
    // starts by recording 64 once 64 wait, so at most 127 ever wait)
    __shared__ uint32_t visq[BLOCK / 64][192];
    const uint32_t n = *n_sq;
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t lane = lane_id();
    uint32_t nvis = 0, ntri = 0, ncon = 0, nsh = 0, nramp = 0;
    Drops drops;
    Walker<LDS, BLOCK, WIDTH, true, INSTR> w(lds + threadIdx.x, gstack, gtid, gthreads);
    Traversal T = make_trav(inst[0], gstack, gthreads);
    // A lane is walking (active) or free.  A walk that ends visible leaves
    // its request slot in the wave's list and the lane takes new work at the
    // next refill; once 64 slots wait, every lane of the wave records one
    // (the splat then runs with the whole wave instead of the few lanes that
    // happened to finish together).  The rest are recorded at the end.
    uint32_t* vq = visq[threadIdx.x >> 6];
    uint32_t nq = 0;  // slots in vq, the same in every lane
    auto push = [&](bool v, uint32_t s) {  // the whole wave
        const uint64_t b = __ballot(v);
        if (v) vq[nq + (uint32_t)__popcll(b & ((1ull << lane) - 1ull))] = s;
        nq += (uint32_t)__popcll(b);
    };
    auto drain = [&](uint32_t take) {  // the whole wave: records the last `take` (<= 64) slots
        wave_sync();
        const bool mine = lane < take;
        const uint32_t rs = mine ? vq[nq - take + lane] : 0u;
        wave_sync();
        nq -= take;
        if (mine) {
            const float4 pc = sq.p[rs], m = sq.m[rs];
            const uint32_t packed = __float_as_uint(m.y);
            const int r = (int)(packed & 0xFFu), band = (int)((packed >> 8) & 0xFFu);
            const uint32_t id = BATCH ? __float_as_uint(m.z) : 0;
            const InstDev& In = inst[id];
            const RecParams& R = In.P.rec[r];
            const V3 dv = sub(V3{R.px, R.py, R.pz}, V3{pc.x, pc.y, pc.z});
            const float l = length(dv);
            TileSink sink{to, rs * to.stride, 0};
            nramp += record(make_hist(In), band, R, normalized(dv), pc.w, (m.x + l) / 343.0f, m.x + l, drops, sink,
                            TILED);
            if (TILED) sink.close();
            ++ncon;
        }
    };
    Claim claim(n, gtid, gridDim.x * blockDim.x, fetch);
    uint32_t refill = fetch.refill;  // idle lanes that trigger a refill
    uint32_t slot = 0;
    for (;;) {
        if (nq >= 64) drain(64);
        const uint64_t idle = __ballot(w.idle());
        if ((uint32_t)__popcll(idle) >= refill) {
            const uint32_t mine = claim.take(fetch, idle, lane);
            if (mine != 0xFFFFFFFFu) {
                slot = mine;
                ++nsh;
                const float4 pc = sq.p[mine], m = sq.m[mine];
                const uint32_t packed = __float_as_uint(m.y);
                const uint32_t id = BATCH ? __float_as_uint(m.z) : 0;
                if (BATCH) T = make_trav(inst[id], gstack, gthreads);
                const RecParams& R = inst[id].P.rec[packed & 0xFFu];
                const V3 p{pc.x, pc.y, pc.z};
                w.start(T, p, sub(V3{R.px, R.py, R.pz}, p), 0.0f);
            }
            push(mine != 0xFFFFFFFFu && w.idle(), slot);  // empty scene: visible
            // the loop is left by the whole wave at once, after the waiting
            // records; with nothing left to take the next look is at the end
            if (idle == ~0ull && __ballot(mine != 0xFFFFFFFFu) == 0) {
                while (nq > 0) drain(nq < 64u ? nq : 64u);
                break;
            }
            if (claim.exhausted()) refill = 64u;
        }
        const bool ended = w.step(T, nvis, ntri);
        if (TILED && ended && w.found()) TileSink{to, slot * to.stride, 0}.close();  // occluded: no records
        push(ended && !w.found(), slot);
    }
    stat_add(stats, ST_SHADOW, nsh);
    stat_add(stats, ST_CONTRIB, ncon);
    stat_add(stats, ST_SH_CONTRIB, ncon);
    stat_add(stats, ST_SH_RAMPS, nramp);
    stat_drops(stats, drops);
    if (INSTR) {
        stat_add(stats, ST_NV_SH, nvis);
        stat_add(stats, ST_NT_SH, ntri);
    }
}

// ---------------------------------------------------------------------------
// time-tiled splat: counting sort of the records by key, then one workgroup
// per key accumulating its tile in LDS
// ---------------------------------------------------------------------------
// Record slots are read kTileBatch per thread at a time (all loads issued
// before the first is used): one wave step then waits for one memory round
// trip instead of kTileBatch.  Slot i of step t of workgroup b is
// (t gridDim + b) kTileBlock kTileBatch + j kTileBlock + threadIdx, j < kTileBatch.
constexpr uint32_t kTileBatch = 16;

// cnt[key] += records of that key among the n_sq * stride slots.  Blocks
// count their share in LDS when the keys fit, then add each non-zero count
// to HBM once.  k_tile_scatter must run with the same grid (it recounts the
// same records per block).
__global__ void __launch_bounds__(kTileBlock) k_tile_count(const uint32_t* __restrict__ keys,
                                                           const uint32_t* __restrict__ n_sq, uint32_t stride,
                                                           uint32_t* __restrict__ cnt, uint32_t K) {
    __shared__ uint32_t h[kLdsKeys];
    const size_t n = (size_t)*n_sq * stride;
    const bool in_lds = K <= kLdsKeys;
    if (in_lds) {
        for (uint32_t j = threadIdx.x; j < K; j += kTileBlock) h[j] = 0;
        __syncthreads();
    }
    constexpr size_t kStep = (size_t)kTileBlock * kTileBatch;
    for (size_t base = (size_t)blockIdx.x * kStep; base < n; base += (size_t)gridDim.x * kStep) {
        uint32_t k[kTileBatch];
#pragma unroll
        for (uint32_t j = 0; j < kTileBatch; ++j) {
            const size_t i = base + j * kTileBlock + threadIdx.x;
            k[j] = i < n ? keys[i] : kNoKey;
        }
#pragma unroll
        for (uint32_t j = 0; j < kTileBatch; ++j) {
            if (k[j] == kNoKey) continue;
            if (in_lds)
                atomicAdd(&h[k[j]], 1u);
            else
                atomicAdd(&cnt[k[j]], 1u);
        }
    }
    if (in_lds) {
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < K; j += kTileBlock)
            if (h[j]) atomicAdd(&cnt[j], h[j]);
    }
}

// Keys with more than kTileDirect records (crowded) get a range of the
// sorted array: off[k] = cur[k] = the sum of the crowded counts before k,
// off[K] = their total; a key with fewer has an empty range and cur[k] =
// kSparse (k_tile_scatter adds its ramps to HBM directly).  cnt is cleared
// for the next iteration; first[c] = the key holding sorted record
// c kTileChunk (for the chunks that start inside the total).  One block of
// 1024 threads.
constexpr uint32_t kSparse = 0xFFFFFFFFu;
__global__ void __launch_bounds__(1024) k_tile_scan(uint32_t* __restrict__ cnt, uint32_t* __restrict__ off,
                                                    uint32_t* __restrict__ cur, uint32_t K,
                                                    uint32_t* __restrict__ first) {
    __shared__ uint32_t wsum[16];
    __shared__ uint32_t carry;
    const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint32_t base = 0; base < K; base += 1024) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t c = i < K ? cnt[i] : 0u;
        const uint32_t v = c > kTileDirect ? c : 0u;
        if (i < K) cnt[i] = 0;
        // inclusive scan within the wave
        uint32_t x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o);
            if ((int)lane >= o) x += y;
        }
        if (lane == 63) wsum[wave] = x;
        __syncthreads();
        if (wave == 0) {
            uint32_t t = lane < 16 ? wsum[lane] : 0u;
            for (int o = 1; o < 16; o <<= 1) {
                const uint32_t y = __shfl_up(t, o);
                if ((int)lane >= o) t += y;
            }
            if (lane < 16) wsum[lane] = t;  // inclusive over waves
        }
        __syncthreads();
        const uint32_t excl = carry + (wave ? wsum[wave - 1] : 0u) + x - v;
        if (i < K) {
            off[i] = excl;
            cur[i] = v ? excl : kSparse;
            // the chunks whose first record is one of this key's [excl, excl + v)
            for (uint32_t c = (excl + kTileChunk - 1) / kTileChunk; c * kTileChunk < excl + v; ++c) first[c] = i;
        }
        __syncthreads();
        if (threadIdx.x == 0) carry += wsum[15];
        __syncthreads();
    }
    if (threadIdx.x == 0) off[K] = carry;
}

// The row and first bin of tile key k: its render is the last item with
// kbase <= k (kbase ascending, kbase[n_items] = K).
struct TileRow {
    unsigned long long* row;
    uint32_t nb, t0, one;
};
__device__ __forceinline__ TileRow tile_row(const InstDev* __restrict__ inst, const uint32_t* __restrict__ kbase,
                                            uint32_t n_items, uint32_t k) {
    uint32_t lo = 0, hi = n_items;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (kbase[mid] <= k)
            lo = mid;
        else
            hi = mid;
    }
    const InstDev& In = inst[lo];
    const uint32_t rel = k - kbase[lo];
    const uint32_t nb = In.P.n_bins;
    return TileRow{In.hist + 4 * (size_t)nb * (rel / In.n_tiles), nb, (rel % In.n_tiles) * kTile, In.P.one_point};
}

// A record's ramp added to HBM directly.
__device__ __forceinline__ void splat_record(const TileRow& r, uint2 p) {
    splat_span(r.row, r.nb, r.one, r.t0 + (p.y & 0xFFFFu), (int)((p.y >> 16) & 0xFFu), (int)(p.y >> 24), __uint_as_float(p.x));
}

// Records of crowded keys to out[] grouped by key: a block recounts its share
// (the records k_tile_count gave it), takes a range per key from cur with one
// atomic each, then places its records there (LDS atomics give the ranks; the
// order within a key does not matter to integer sums).  Records of sparse
// keys (cur[k] = kSparse) are added to HBM here.
__global__ void __launch_bounds__(kTileBlock) k_tile_scatter(const InstDev* __restrict__ inst,
                                                             const uint32_t* __restrict__ kbase, uint32_t n_items,
                                                             const uint32_t* __restrict__ keys,
                                                             const uint2* __restrict__ pay,
                                                             const uint32_t* __restrict__ n_sq, uint32_t stride,
                                                             uint32_t* __restrict__ cur, uint32_t K,
                                                             uint2* __restrict__ out) {
    __shared__ uint32_t h[kLdsKeys];
    const size_t n = (size_t)*n_sq * stride;
    constexpr size_t kStep = (size_t)kTileBlock * kTileBatch;
    const size_t step = (size_t)gridDim.x * kStep;
    const bool in_lds = K <= kLdsKeys;
    if (in_lds) {
        for (uint32_t j = threadIdx.x; j < K; j += kTileBlock) h[j] = 0;
        __syncthreads();
        for (size_t base = (size_t)blockIdx.x * kStep; base < n; base += step) {
            uint32_t k[kTileBatch];
#pragma unroll
            for (uint32_t j = 0; j < kTileBatch; ++j) {
                const size_t i = base + j * kTileBlock + threadIdx.x;
                k[j] = i < n ? keys[i] : kNoKey;
            }
#pragma unroll
            for (uint32_t j = 0; j < kTileBatch; ++j)
                if (k[j] != kNoKey) atomicAdd(&h[k[j]], 1u);
        }
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < K; j += kTileBlock) {
            if (!h[j]) continue;
            const uint32_t c = cur[j];
            h[j] = c == kSparse ? kSparse : atomicAdd(&cur[j], h[j]);
        }
        __syncthreads();
    }
    for (size_t base = (size_t)blockIdx.x * kStep; base < n; base += step) {
        uint32_t k[kTileBatch];
        uint2 v[kTileBatch];
#pragma unroll
        for (uint32_t j = 0; j < kTileBatch; ++j) {
            const size_t i = base + j * kTileBlock + threadIdx.x;
            k[j] = i < n ? keys[i] : kNoKey;
        }
#pragma unroll
        for (uint32_t j = 0; j < kTileBatch; ++j) {
            const size_t i = base + j * kTileBlock + threadIdx.x;
            if (k[j] != kNoKey) v[j] = pay[i];
        }
#pragma unroll
        for (uint32_t j = 0; j < kTileBatch; ++j) {
            if (k[j] == kNoKey) continue;
            const uint32_t c = in_lds ? h[k[j]] : cur[k[j]];
            if (c == kSparse)
                splat_record(tile_row(inst, kbase, n_items, k[j]), v[j]);
            else
                out[in_lds ? atomicAdd(&h[k[j]], 1u) : atomicAdd(&cur[k[j]], 1u)] = v[j];
        }
    }
}

// 128-bit add into the LDS tile (lo at 2 i, hi at 2 i + 1)
__device__ __forceinline__ void lds_acc128(unsigned long long* tile, uint32_t i, I128 q) {
    const unsigned long long lo = q.lo;
    const unsigned long long old = atomicAdd(&tile[2 * i], lo);
    const unsigned long long hi = (unsigned long long)q.hi + ((old + lo) < old ? 1ull : 0ull);
    if (hi) atomicAdd(&tile[2 * i + 1], hi);
}

// The key whose records include sorted position p (off[0] <= p < off[K]):
// the last k with off[k] <= p.
__device__ __forceinline__ uint32_t key_at(const uint32_t* __restrict__ off, uint32_t K, uint32_t p) {
    uint32_t lo = 0, hi = K;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= p)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Workgroup b takes the sorted records [b kTileChunk, (b + 1) kTileChunk) (all
// of crowded keys) and walks the keys among them: the ramps of one (render,
// row, tile) are added into an LDS copy of the tile's bins
// [t0, t0 + kTile + kHalo) of both parts, which is then added to the row in
// HBM (bins < n_bins); a key with at most kTileDirect records in the chunk
// goes straight to HBM.  kbase: the first key of each render of the batch,
// ascending, kbase[n_items] = K.
__global__ void __launch_bounds__(kTileBlock) k_tile_splat(const InstDev* __restrict__ inst,
                                                           const uint32_t* __restrict__ kbase, uint32_t n_items,
                                                           const uint32_t* __restrict__ off, uint32_t K,
                                                           const uint32_t* __restrict__ first,
                                                           const uint2* __restrict__ pay) {
    constexpr uint32_t kSpan = kTile + kHalo;
    constexpr uint32_t kPer = kTileChunk / kTileBlock;  // records per thread and key, at most
    constexpr uint32_t kSplatBatch = 8;
    __shared__ unsigned long long acc[2 * kSpan * 2];  // [part][bin] x {lo, hi}
    const uint32_t total = off[K];
    const uint32_t c0 = blockIdx.x * kTileChunk;
    if (c0 >= total) return;
    const uint32_t c1 = min(c0 + kTileChunk, total);
    for (uint32_t b = c0; b < c1;) {
        const uint32_t k = b == c0 ? first[blockIdx.x] : key_at(off, K, b);
        const uint32_t e = min(off[k + 1], c1);
        const TileRow tr = tile_row(inst, kbase, n_items, k);
        unsigned long long* row = tr.row;
        const uint32_t nb = tr.nb, t0 = tr.t0;
        if (e - b <= kTileDirect) {
            // the chunk's share of the key is small: straight to HBM
            for (uint32_t i = b + threadIdx.x; i < e; i += kTileBlock) splat_record(tr, pay[i]);
        } else {
            for (uint32_t j = threadIdx.x; j < 4 * kSpan; j += kTileBlock) acc[j] = 0;
            __syncthreads();
            // this thread's records of the key, kSplatBatch loads at a time
            for (uint32_t jb = 0; jb < kPer && b + jb * kTileBlock < e; jb += kSplatBatch) {
                uint2 pv[kSplatBatch];
#pragma unroll
                for (uint32_t j = 0; j < kSplatBatch; ++j) {
                    const uint32_t i = b + (jb + j) * kTileBlock + threadIdx.x;
                    if (i < e) pv[j] = pay[i];
                }
#pragma unroll
                for (uint32_t j = 0; j < kSplatBatch; ++j) {
                    if (b + (jb + j) * kTileBlock + threadIdx.x >= e) break;
                    const uint2 p = pv[j];
                    const uint32_t o = p.y & 0xFFFFu;
                    const int ww = (int)((p.y >> 16) & 0xFFu), w = (int)(p.y >> 24);
                    if (tr.one) {
                        lds_acc128(acc + ((uint32_t)w & 1u) * 2 * kSpan, o, ramp_slope(__uint_as_float(p.x), w));
                        continue;
                    }
                    const RampPoints q = ramp_points(__uint_as_float(p.x), w, ww);
                    unsigned long long* tp = acc + (q.neg ? 2 * kSpan : 0u);  // gets +w*S and +S
                    unsigned long long* tm = acc + (q.neg ? 0u : 2 * kSpan);  // gets (w+1)*S
                    lds_acc128(tp, o, q.aq);
                    if (t0 + o + 1 < nb) lds_acc128(tm, o + 1, q.p1);
                    if (t0 + o + (uint32_t)ww + 1 < nb) lds_acc128(tp, o + (uint32_t)ww + 1, q.sq);
                }
            }
            __syncthreads();
            for (uint32_t j = threadIdx.x; j < 2 * kSpan; j += kTileBlock) {
                const uint32_t part = j >= kSpan ? 1u : 0u, loc = j - part * kSpan;
                const unsigned long long vlo = acc[2 * j], vhi = acc[2 * j + 1];
                if ((vlo | vhi) && t0 + loc < nb)
                    acc128(row + 2 * (size_t)nb * part + 2 * (size_t)(t0 + loc), I128{vlo, (int64_t)vhi});
            }
            __syncthreads();  // the tile is cleared again for the next key
        }
        b = e;
    }
}

// p[0, n) = v, grid-stride (clears device memory without a memset node)
__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_reset2(uint32_t* a, uint32_t* b) {
    if (threadIdx.x == 0) {
        *a = 0;
        *b = 0;
    }
}

// Ray regeneration: tops the current queue up to `cap` with the next rays of
// the segment table.  plan = {first ray, count, first free slot} for
// k_generate; the cursor counts the rays taken so far.  dense: the rays are
// counted into the queue here (k_generate appends them otherwise).
__global__ void k_plan(uint32_t* cursor, uint32_t total, uint32_t cap, uint32_t dense, uint32_t* n_q, uint32_t* plan) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        const uint32_t taken = *cursor, live = *n_q;
        const uint32_t room = cap > live ? cap - live : 0u;
        const uint32_t take = min(room, total - taken);
        plan[0] = taken;
        plan[1] = take;
        plan[2] = live;
        *cursor = taken + take;
        if (dense) *n_q = live + take;
    }
}

// End of a bounce-loop iteration: zeroes the counters c[i] for the bits i of
// mask and the n_seg refill counters (a kernel, not memset nodes, so a
// captured loop replays it correctly)
__global__ void k_reset_iter(uint32_t* c, uint32_t mask, uint32_t* seg, uint32_t n_seg) {
    if (threadIdx.x < 32 && ((mask >> threadIdx.x) & 1u)) c[threadIdx.x] = 0;
    for (uint32_t i = threadIdx.x; i < n_seg; i += blockDim.x) seg[i * kSegStride] = 0;
}

// Direct sound (src/Scene.cpp:299-311): one block per instance, one thread
// per (band, recorder).
template <int WIDTH>
__global__ void k_direct(const InstDev* __restrict__ inst, int* gstack, uint32_t gthreads,
                         unsigned long long* __restrict__ stats) {
    __shared__ int lds[kLdsMin * kBlock];
    const InstDev& In = inst[blockIdx.x];
    const RenderParams& P = In.P;
    uint32_t t = threadIdx.x;
    if (t >= 3 * P.n_rec) return;
    int band = (int)(t / P.n_rec);
    if (!((P.band_mask >> band) & 1u)) return;
    const RecParams& R = P.rec[t % P.n_rec];
    DirectRamp* o = In.direct + (size_t)band * P.n_channels + R.channel;
    int nch = R.kind == EAR_REC_STEREO ? 2 : 1;
    for (int c = 0; c < nch; ++c) o[c] = DirectRamp{0, 0, 0, 0.0f};
    if (P.src_kind != EAR_SRC_POINT || P.estimator != EAR_EST_NEE) return;
    V3 rp{R.px, R.py, R.pz}, sp{P.src_pos[0], P.src_pos[1], P.src_pos[2]};
    float bt = 0.0f;
    int bs = -1;
    uint32_t bo = 0, nv = 0, nt = 0;
    Traversal T = make_trav(In, gstack, gthreads);
    if (traverse<kLdsMin, kBlock, WIDTH, true, false>(T, rp, sub(sp, rp), bt, bs, bo, lds + threadIdx.x,
                                                      blockIdx.x * kBlock + t, nv, nt))
        return;
    V3 dist = sub(rp, sp);
    float len = length(dist);
    V3 dir = normalized(dist);
    float a = 1.0f / (4.0f * kPi * len * len) * powf_ear_l2(P.air[band], P.l2_air[band], len) * P.dry;
    float tt = len / 343.0f;
    float width = sqrtf(len);
    float ampl = 2.0f * a / width;
    int w = (int)ceilf(width);
    // a direct ramp cut at the end of the histogram counts as a dropped ramp
    auto cut = [&](int s) {
        const int64_t e = (int64_t)s + (int64_t)w;  // one past the ramp's last bin
        if (e > (int64_t)P.n_bins) {
            atomicAdd(stats + ST_DROPPED, 1ull);
            atomicMax(stats + ST_BINS, (unsigned long long)e);
        }
    };
    if (R.kind == EAR_REC_MONO) {
        o[0] = DirectRamp{1, (int)((double)tt * 44100.0), w, ampl};
        cut(o[0].s);
    } else {
        float dt = dot(dir, V3{R.rx, R.ry, R.rz});
        float td = R.head_size / 343.0f;
        float al = ampl, ar = ampl;
        float factor = powf_ear_l2(R.head_abs[band], R.l2_head_abs[band], fabsf(dt) * R.head_size);
        if (dt < 0.0f)
            ar *= factor * factor;
        else
            al *= factor * factor;
        o[0] = DirectRamp{1, (int)((double)(tt + dt * td) * 44100.0), w, al};
        o[1] = DirectRamp{1, (int)((double)(tt - dt * td) * 44100.0), w, ar};
        cut(o[0].s);
        cut(o[1].s);
    }
}

// Two inclusive prefix sums over a second-difference row (128-bit, exact),
// then value = (raw 2^-80 * inv_n + direct ramp) * gain2.  One block per row;
// row r of the table is {instance, band, channel, kind}.
constexpr int kFinBlock = 1024;
__global__ void __launch_bounds__(kFinBlock) k_finalize(const InstDev* __restrict__ inst, const uint4* __restrict__ rows) {
    __shared__ uint64_t slo[kFinBlock];
    __shared__ int64_t shi[kFinBlock];
    const uint4 rw = rows[blockIdx.x];
    const InstDev& In = inst[rw.x];
    const RenderParams& P = In.P;
    const int band = (int)rw.y;
    const uint32_t ch = rw.z, kind = rw.w, nb = P.n_bins, n_ch = P.n_channels, kinds = P.hist_kinds;
    size_t roff = (((size_t)band * n_ch + ch) * kinds + kind) * 2 * nb;
    unsigned long long* c = In.hist + 2 * roff;      // "+" part, receives the sums
    unsigned long long* cm = c + 2 * (size_t)nb;     // "-" part
    uint32_t per = (nb + kFinBlock - 1) / kFinBlock;
    uint32_t b = threadIdx.x * per, e = min(nb, b + per);
    // pass 0 sums (+) - (-), the second differences; pass 1 their prefix sums
    auto elem = [&](int pass, uint32_t j) {
        I128 v{c[2 * j], (int64_t)c[2 * j + 1]};
        if (pass == 0) v = i128_add(v, i128_neg(I128{cm[2 * j], (int64_t)cm[2 * j + 1]}));
        return v;
    };
    for (int pass = 0; pass < 2; ++pass) {
        I128 sum{0, 0};
        for (uint32_t j = b; j < e; ++j) sum = i128_add(sum, elem(pass, j));
        slo[threadIdx.x] = sum.lo;
        shi[threadIdx.x] = sum.hi;
        __syncthreads();
        for (int off = 1; off < kFinBlock; off <<= 1) {
            I128 v{0, 0};
            if ((int)threadIdx.x >= off) v = I128{slo[threadIdx.x - off], shi[threadIdx.x - off]};
            __syncthreads();
            I128 cur = i128_add(I128{slo[threadIdx.x], shi[threadIdx.x]}, v);
            slo[threadIdx.x] = cur.lo;
            shi[threadIdx.x] = cur.hi;
            __syncthreads();
        }
        I128 run = i128_add(I128{slo[threadIdx.x], shi[threadIdx.x]}, i128_neg(sum));
        for (uint32_t j = b; j < e; ++j) {
            run = i128_add(run, elem(pass, j));
            c[2 * j] = run.lo;
            c[2 * j + 1] = (unsigned long long)run.hi;
        }
        __syncthreads();
    }
}

// The finished track of one bin from its signed (and |.|) sums: 2^-80, 1/N, the
// direct sound (src/Scene.cpp:299-311) and gain^2 (src/Scene.cpp:313-316).
__device__ __forceinline__ void finished_values(const InstDev& In, int band, uint32_t ch, uint32_t j, const I128 v[2]) {
    if (!In.value) return;
    const uint32_t nb = In.P.n_bins, n_ch = In.P.n_channels, kinds = In.P.hist_kinds;
    const size_t r0 = (((size_t)band * n_ch + ch) * kinds) * nb;  // value rows
    const DirectRamp dr = In.direct[(size_t)band * n_ch + ch];
    const double S = dr.visible ? (double)dr.a / (double)dr.w : 0.0;
    for (uint32_t kind = 0; kind < kinds; ++kind) {
        double x = (double)v[kind].hi * 18446744073709551616.0 + (double)v[kind].lo;
        x = x * 0x1p-80;  // 2^-EAR_FRAC_BITS
        x = x * In.inv_n;
        if (dr.visible && (int)j >= dr.s && (int)j < dr.s + dr.w) {
            const double dv = (double)(dr.w - ((int)j - dr.s)) * S;
            x += kind == 1 ? fabs(dv) : dv;
        }
        In.value[r0 + (size_t)kind * nb + j] = x * In.gain2;
    }
}

// Per (instance, band, channel) and bin: the sign-split rows (if any) become
// the signed and |.| sums, then the finished track.
__global__ void __launch_bounds__(256) k_values(const InstDev* __restrict__ inst, const uint4* __restrict__ rows) {
    const uint4 rw = rows[blockIdx.y];
    const InstDev& In = inst[rw.x];
    const RenderParams& P = In.P;
    const int band = (int)rw.y;
    const uint32_t ch = rw.z, nb = P.n_bins, n_ch = P.n_channels, kinds = P.hist_kinds;
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if (j >= nb) return;
    const size_t r0 = (((size_t)band * n_ch + ch) * kinds) * nb;  // value rows
    unsigned long long* c0 = In.hist + 4 * r0;                      // kind 0 "+" part
    I128 v[2];
    v[0] = I128{c0[2 * j], (int64_t)c0[2 * j + 1]};
    if (kinds > 1) {
        unsigned long long* c1 = c0 + 4 * (size_t)nb;  // kind 1 "+" part
        const I128 pos = v[0], neg = I128{c1[2 * j], (int64_t)c1[2 * j + 1]};
        v[0] = i128_add(pos, i128_neg(neg));
        v[1] = i128_add(pos, neg);
        c0[2 * j] = v[0].lo;
        c0[2 * j + 1] = (unsigned long long)v[0].hi;
        c1[2 * j] = v[1].lo;
        c1[2 * j + 1] = (unsigned long long)v[1].hi;
    }
    finished_values(In, band, ch, j, v);
}

// One-point rows (see OnePoint) finished: per (instance, band, channel) and
// bin, the ramps that cover the bin, ramps of width w that start at s adding
// (w - (bin - s)) times their slopes' sum; then signed and |.| sums and the
// finished track as in k_values.  Each bin looks back over the widths of its
// own distance (33 bins at 3 s), so bins are independent: a grid over all of
// them, where the prefix sums of k_finalize are one block per row (the hall's
// 3 s stereo rows: 1.05 ms with 12 blocks, 0.1 ms here).  The rows must not be
// written meanwhile: raw sums go to `raw` ([row][kind][bin - bin0], or null),
// bins [bin0, bin1) of rows [row0, row0 + gridDim.y) of the table.
__global__ void __launch_bounds__(256) k_finish(const InstDev* __restrict__ inst, const uint4* __restrict__ rows,
                                                uint32_t row0, uint32_t bin0, uint32_t bin1,
                                                unsigned long long* __restrict__ raw,
                                                const uint64_t* __restrict__ raw_off) {
    const uint32_t row = row0 + blockIdx.y;
    const uint4 rw = rows[row];
    const InstDev& In = inst[rw.x];
    const RenderParams& P = In.P;
    const int band = (int)rw.y;
    const uint32_t ch = rw.z, nb = P.n_bins, n_ch = P.n_channels, kinds = P.hist_kinds;
    const uint32_t j = bin0 + blockIdx.x * 256 + threadIdx.x, end = min(bin1, nb);
    if (j >= end) return;
    const size_t r0 = (((size_t)band * n_ch + ch) * kinds) * nb;
    const ulonglong2* c0 = (const ulonglong2*)(In.hist + 4 * r0);  // [kind][parity][bin]
    // the two widths of ramps that start at s are wl and wl + 1: the least
    // distance of a ramp on bin s is s kBinMetres - slack
    const double slack = P.ramp_slack;
    const double d0 = (double)j * kBinMetres - slack;
    int wl = d0 > 1.0 ? (int)ceil(sqrt(d0)) : 1;
    I128 sum[2] = {I128{0, 0}, I128{0, 0}};
    for (uint32_t i = 0; i <= j && (int)i <= wl; ++i) {
        const uint32_t s = j - i;
        const double d = (double)s * kBinMetres - slack;
        while (wl > 1 && d <= (double)((wl - 1) * (wl - 1))) --wl;
        if ((int)i > wl) break;  // (widths fall with s: no earlier ramp reaches this bin)
        const uint32_t pe = (uint32_t)wl & 1u;  // the part of width wl; the other one holds wl + 1
        for (uint32_t k = 0; k < kinds; ++k) {
            const ulonglong2* h = c0 + (size_t)k * 2 * nb;
            const ulonglong2 a = h[(size_t)pe * nb + s], b = h[(size_t)(pe ^ 1u) * nb + s];
            // slopes are signed only where there is one kind
            const auto scaled = [](ulonglong2 v, uint32_t m) {
                const I128 q{v.x, (int64_t)v.y};
                return q.hi < 0 ? i128_neg(i128_mul_small(i128_neg(q), m)) : i128_mul_small(q, m);
            };
            if (a.x | a.y) sum[k] = i128_add(sum[k], scaled(a, (uint32_t)(wl - (int)i)));
            if (b.x | b.y) sum[k] = i128_add(sum[k], scaled(b, (uint32_t)(wl + 1 - (int)i)));
        }
    }
    I128 v[2] = {sum[0], I128{0, 0}};
    if (kinds > 1) {
        v[0] = i128_add(sum[0], i128_neg(sum[1]));
        v[1] = i128_add(sum[0], sum[1]);
    }
    if (raw)
        for (uint32_t k = 0; k < kinds; ++k) {
            ulonglong2* o = (ulonglong2*)raw + raw_off[row] - raw_off[row0] + (size_t)k * (end - bin0) + (j - bin0);
            *o = make_ulonglong2(v[k].lo, (unsigned long long)v[k].hi);
        }
    finished_values(In, band, ch, j, v);
}

// batched queries for tests and host tools
template <int WIDTH, bool ANY>
__global__ void __launch_bounds__(kBlock) k_query(Traversal T, uint32_t n, const float* __restrict__ a,
                                                   const float* __restrict__ b, float* __restrict__ tout,
                                                   int32_t* __restrict__ iout, uint8_t* __restrict__ occ) {
    __shared__ int lds[kLdsMin * kBlock];
    uint32_t gtid = blockIdx.x * kBlock + threadIdx.x;
    uint32_t nv = 0, nt = 0;
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        uint32_t i = base + threadIdx.x;
        if (i >= n) continue;
        V3 o{a[3 * i], a[3 * i + 1], a[3 * i + 2]};
        V3 x{b[3 * i], b[3 * i + 1], b[3 * i + 2]};
        float bt = 1000000.0f;
        int bs = -1;
        uint32_t bo = 0;
        if (ANY) {
            occ[i] = traverse<kLdsMin, kBlock, WIDTH, true, false>(T, o, sub(x, o), bt, bs, bo, lds + threadIdx.x,
                                                                   gtid, nv, nt)
                         ? 1
                         : 0;
        } else {
            bool h = traverse<kLdsMin, kBlock, WIDTH, false, false>(T, o, x, bt, bs, bo, lds + threadIdx.x, gtid, nv,
                                                                    nt);
            tout[i] = h ? bt : 0.0f;
            iout[i] = h ? (int32_t)bo : -1;
        }
    }
}

// Traversal kernels are instantiated for every (block, LDS stack part, tree
// width, instrumentation, batch) combination; the render picks one at run time.
struct TravCfg {
    int block, lds, width;
    bool instr, batch, fetch;
    bool tiled;  // shadow kernels: write the time-tiled splat's records
};

using ExtendFn = void (*)(const InstDev*, int*, uint32_t, Queue, const uint32_t*, int2*, unsigned long long*, Fetch);
using ShadowFn = void (*)(const InstDev*, int*, uint32_t, ShadowQ, const uint32_t*, unsigned long long*, Fetch,
                         TileOut);

template <int B, int L, int W, bool BA>
void pick_t(bool instr, bool fetch, bool tiled, ExtendFn* e, ShadowFn* s) {
    if (fetch) {
        *e = instr ? (ExtendFn)k_extend_f<B, L, W, true, BA> : (ExtendFn)k_extend_f<B, L, W, false, BA>;
        if (tiled)
            *s = instr ? (ShadowFn)k_shadow_f<B, L, W, true, BA, true> : (ShadowFn)k_shadow_f<B, L, W, false, BA, true>;
        else
            *s = instr ? (ShadowFn)k_shadow_f<B, L, W, true, BA, false>
                       : (ShadowFn)k_shadow_f<B, L, W, false, BA, false>;
    } else {
        *e = instr ? (ExtendFn)k_extend<B, L, W, true, BA> : (ExtendFn)k_extend<B, L, W, false, BA>;
        if (tiled)
            *s = instr ? (ShadowFn)k_shadow<B, L, W, true, BA, true> : (ShadowFn)k_shadow<B, L, W, false, BA, true>;
        else
            *s = instr ? (ShadowFn)k_shadow<B, L, W, true, BA, false> : (ShadowFn)k_shadow<B, L, W, false, BA, false>;
    }
}

template <bool BA>
void pick_b(const TravCfg& c, ExtendFn* e, ShadowFn* s) {
    int key = (c.block >= 256 ? 4 : 0) | (c.lds >= 32 ? 2 : 0) | (c.width == 4 ? 1 : 0);
    switch (key) {
        case 0: pick_t<128, 16, 2, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        case 1: pick_t<128, 16, 4, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        case 2: pick_t<128, 32, 2, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        case 3: pick_t<128, 32, 4, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        case 4: pick_t<256, 16, 2, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        case 5: pick_t<256, 16, 4, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        case 6: pick_t<256, 32, 2, BA>(c.instr, c.fetch, c.tiled, e, s); break;
        default: pick_t<256, 32, 4, BA>(c.instr, c.fetch, c.tiled, e, s); break;
    }
}

using TailFn = void (*)(const InstDev*, int*, uint32_t, Queue, const uint32_t*, uint32_t, Fetch, unsigned long long*);

template <int B, int L>
TailFn tail_for(int width, bool batch) {
    if (width == 4) return batch ? (TailFn)k_tail<B, L, 4, true> : (TailFn)k_tail<B, L, 4, false>;
    return batch ? (TailFn)k_tail<B, L, 2, true> : (TailFn)k_tail<B, L, 2, false>;
}

TailFn pick_tail(const TravCfg& c) {
    if (c.block == 128) return c.lds == 32 ? tail_for<128, 32>(c.width, c.batch) : tail_for<128, 16>(c.width, c.batch);
    return c.lds == 32 ? tail_for<256, 32>(c.width, c.batch) : tail_for<256, 16>(c.width, c.batch);
}

void pick_kernels(const TravCfg& c, ExtendFn* e, ShadowFn* s) {
    if (c.batch)
        pick_b<true>(c, e, s);
    else
        pick_b<false>(c, e, s);
}

// Blocks per CU that can be resident for kernel `fn` (0 on error).
int resident_blocks(const void* fn, int block) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, block, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return nb;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

uint32_t persistent_grid(Ctx* c, uint32_t work, uint32_t waves_per_cu, uint32_t block = kBlock) {
    uint32_t blocks_needed = (work + block - 1) / block;
    uint32_t cap = (uint32_t)c->num_cus * std::max<uint32_t>(1, waves_per_cu) / std::max<uint32_t>(1, block / 64);
    return std::max<uint32_t>(1, std::min(blocks_needed, std::max<uint32_t>(1, cap)));
}

uint32_t grid_for(uint32_t work, uint32_t cap_blocks, uint32_t block) {
    uint32_t blocks_needed = (work + block - 1) / block;
    return std::max<uint32_t>(1, std::min(blocks_needed, std::max<uint32_t>(1, cap_blocks)));
}

// Block cap of a kernel that loops over its queue with the grid's stride (so
// every block gets the same share): three rounds of the blocks one CU holds
// at once.  A grid of whole rounds leaves no CU a last partial round to run
// alone (32 waves per CU of a kernel that fits 24 ran its last quarter of
// blocks at a third of the occupancy).  waves_per_cu, when set, overrides.
uint32_t rounds_cap(Ctx* c, const void* fn, uint32_t waves_per_cu, int block) {
    if (waves_per_cu) return (uint32_t)c->num_cus * waves_per_cu / (uint32_t)std::max(1, block / 64);
    return (uint32_t)c->num_cus * (uint32_t)std::max(1, resident_blocks(fn, block)) * 3u;
}

struct EventPair {
    hipEvent_t a = nullptr, b = nullptr;
};

float tri_area_host(const float* v) {
    // Triangle::calcArea (src/Triangle.cpp:26-30): |edge(0) x edge(1)| / 2,
    // edge(i) = v[(i+1)%3] - v[i]
    V3 a = sub(V3{v[3], v[4], v[5]}, V3{v[0], v[1], v[2]});
    V3 b = sub(V3{v[6], v[7], v[8]}, V3{v[3], v[4], v[5]});
    return length(cross(a, b)) / 2.0f;
}

// Validates one render description and fills its RenderParams.
ear_status make_params(Ctx* c, const ear_render_desc* D, RenderParams* P) {
    if (!D) return EAR_ERR_INVALID_ARGUMENT;
    if ((D->band_mask & 7u) == 0 || (D->band_mask & ~7u)) {
        c->last_error = "band_mask must select bands among bits 0..2";
        return EAR_ERR_INVALID_ARGUMENT;
    }
    if (D->hist_bins == 0 || D->n_recorders == 0 || !D->recorders) {
        c->last_error = "hist_bins and recorders are required";
        return EAR_ERR_INVALID_ARGUMENT;
    }
    if (D->n_recorders > (uint32_t)kMaxRecorders) {
        c->last_error = "too many recorders";
        return EAR_ERR_CAPACITY;
    }
    if (D->source.kind != EAR_SRC_POINT && D->source.kind != EAR_SRC_MESH) return EAR_ERR_INVALID_ARGUMENT;
    if (D->source.kind == EAR_SRC_MESH && (!D->source.mesh_v || D->source.mesh_n_tris == 0)) {
        c->last_error = "mesh source without triangles";
        return EAR_ERR_INVALID_ARGUMENT;
    }
    if ((uint64_t)D->hist_bins * 3ull * 2ull * kMaxRecorders > (1ull << 36)) {
        c->last_error = "histogram too long";
        return EAR_ERR_CAPACITY;
    }
    for (int b = 0; b < 3; ++b)
        if (!std::isfinite(D->air[b])) return EAR_ERR_INVALID_ARGUMENT;
    if (D->max_bounces > kMaxBounces) {
        // the bounce number travels in 16 bits of a queue entry; past them it
        // would wrap, and a path in a lossless room would never end
        c->last_error = "max_bounces above 65535";
        return EAR_ERR_CAPACITY;
    }
    if (D->estimator > EAR_EST_SPHERE) {
        c->last_error = "unknown estimator";
        return EAR_ERR_INVALID_ARGUMENT;
    }
    std::memset(P, 0, sizeof(*P));
    P->estimator = D->estimator;
    P->seed = D->seed;
    P->instance = D->instance;
    for (int b = 0; b < 3; ++b) {
        P->ctx_word[b] = (uint32_t)b | ((D->sound & 0xFFu) << 8) | ((uint32_t)(D->keyframe + 1) << 16);
        P->air[b] = D->air[b];
        P->l2_air[b] = pow_base_l2(D->air[b]);
    }
    P->dry = D->dry;
    P->cutoff = D->energy_cutoff;
    P->max_bounces = D->max_bounces;
    P->n_bins = D->hist_bins;
    P->n_rec = D->n_recorders;
    P->n_band_slots = 3;
    P->band_mask = D->band_mask;
    P->hist_kinds = (D->flags & EAR_FLAG_ABS_HIST) ? 2 : 1;
    // one point per ramp: a bin's ramps must have one of two consecutive
    // widths, so the distances of one bin must span less than a metre: its own
    // 343 / 44100 m, the head's delay either way, and the rounding of binary32
    // times (2^-24 of the distance each; 1e-6 of the longest, and 1 mm)
    double head = 0.0;
    if (D->estimator == EAR_EST_NEE)
        for (uint32_t r = 0; r < D->n_recorders; ++r) {
            const ear_recorder& R = D->recorders[r];
            if (R.kind != EAR_REC_STEREO) continue;
            const double e = std::sqrt((double)R.right_ear[0] * R.right_ear[0] + (double)R.right_ear[1] * R.right_ear[1] +
                                       (double)R.right_ear[2] * R.right_ear[2]);
            const double h = std::fabs((double)R.head_size) * e;
            head = h >= head ? h : (h < head ? head : 1e30);  // NaN: not one point
        }
    P->ramp_slack = head + 1e-3 + 1e-6 * kBinMetres * (double)D->hist_bins;
    P->one_point = 2.0 * P->ramp_slack + kBinMetres < 0.98 ? 1u : 0u;
    P->src_kind = D->source.kind;
    for (int k = 0; k < 3; ++k) P->src_pos[k] = D->source.pos[k];
    P->flags = D->flags;
    uint32_t nch = 0;
    for (uint32_t r = 0; r < D->n_recorders; ++r) {
        const ear_recorder& R = D->recorders[r];
        if (R.kind != EAR_REC_MONO && R.kind != EAR_REC_STEREO) return EAR_ERR_INVALID_ARGUMENT;
        RecParams& Q = P->rec[r];
        Q.px = R.pos[0];
        Q.py = R.pos[1];
        Q.pz = R.pos[2];
        Q.rx = R.right_ear[0];
        Q.ry = R.right_ear[1];
        Q.rz = R.right_ear[2];
        Q.head_size = R.head_size;
        for (int b = 0; b < 3; ++b) {
            Q.head_abs[b] = R.head_abs[b];
            Q.l2_head_abs[b] = pow_base_l2(R.head_abs[b]);
        }
        Q.kind = R.kind;
        Q.channel = (int32_t)nch;
        nch += R.kind == EAR_REC_STEREO ? 2 : 1;
        if (D->estimator == EAR_EST_SPHERE) {
            // spheres: mono at pos; stereo head_size / 2 either side along
            // the unit right-ear direction (left channel first)
            const float rad = R.radius;
            const float rn = sqrtf(R.right_ear[0] * R.right_ear[0] + R.right_ear[1] * R.right_ear[1] +
                                   R.right_ear[2] * R.right_ear[2]);
            if (!(rad > 0.0f) || !std::isfinite(rad) || (R.kind == EAR_REC_STEREO && !(rn > 0.0f))) {
                c->last_error = "sphere estimator needs radius > 0 (and a right-ear direction for stereo)";
                return EAR_ERR_INVALID_ARGUMENT;
            }
            Q.r2 = rad * rad;
            Q.inv_vol = 3.0f / (4.0f * kPi * rad * rad * rad);
            for (int k = 0; k < 3; ++k) Q.cen[0][k] = Q.cen[1][k] = R.pos[k];
            if (R.kind == EAR_REC_STEREO) {
                const float h = (0.5f * R.head_size) / rn;
                for (int k = 0; k < 3; ++k) {
                    Q.cen[0][k] = R.pos[k] - R.right_ear[k] * h;
                    Q.cen[1][k] = R.pos[k] + R.right_ear[k] * h;
                }
            }
        }
    }
    P->n_channels = nch;
    bool want_log = (D->flags & EAR_FLAG_TRACE_LOG) && D->trace_rays && D->trace_segs;
    P->trace_rays = want_log ? D->trace_rays : 0;
    P->trace_segs = want_log ? D->trace_segs : 0;
    return EAR_OK;
}

}  // namespace

ear_status run_query_closest(Ctx* c, DeviceScene* s, uint32_t n, const float* o, const float* d, float* t,
                             int32_t* tri) {
    if (n == 0) return EAR_OK;
    if (!o || !d || !t || !tri) return EAR_ERR_INVALID_ARGUMENT;
    DevBuf da(c), db(c), dt(c), di(c), gs(c);
    TRY(da.alloc((size_t)n * 12));
    TRY(db.alloc((size_t)n * 12));
    TRY(dt.alloc((size_t)n * 4));
    TRY(di.alloc((size_t)n * 4));
    uint32_t grid = persistent_grid(c, n, 16);
    uint32_t gthreads = grid * kBlock;
    TRY(gs.alloc((size_t)(kStackDepth - kLdsMin) * gthreads * 4));
    hipStream_t st = c->stream;
    EAR_HIP_TRY(c, hipMemcpyAsync(da.p, o, (size_t)n * 12, hipMemcpyHostToDevice, st));
    EAR_HIP_TRY(c, hipMemcpyAsync(db.p, d, (size_t)n * 12, hipMemcpyHostToDevice, st));
    Traversal T{s->nodes, s->nodes4, s->tris, s->n_tris, gs.as<int>(), gthreads};
    if (s->width == 4)
        k_query<4, false><<<grid, kBlock, 0, st>>>(T, n, da.as<float>(), db.as<float>(), dt.as<float>(),
                                                   di.as<int32_t>(), nullptr);
    else
        k_query<2, false><<<grid, kBlock, 0, st>>>(T, n, da.as<float>(), db.as<float>(), dt.as<float>(),
                                                   di.as<int32_t>(), nullptr);
    EAR_HIP_TRY(c, hipGetLastError());
    EAR_HIP_TRY(c, hipMemcpyAsync(t, dt.p, (size_t)n * 4, hipMemcpyDeviceToHost, st));
    EAR_HIP_TRY(c, hipMemcpyAsync(tri, di.p, (size_t)n * 4, hipMemcpyDeviceToHost, st));
    EAR_HIP_TRY(c, hipStreamSynchronize(st));
    return EAR_OK;
}

ear_status run_query_occluded(Ctx* c, DeviceScene* s, uint32_t n, const float* p, const float* q, uint8_t* occ) {
    if (n == 0) return EAR_OK;
    if (!p || !q || !occ) return EAR_ERR_INVALID_ARGUMENT;
    DevBuf da(c), db(c), dk(c), gs(c);
    TRY(da.alloc((size_t)n * 12));
    TRY(db.alloc((size_t)n * 12));
    TRY(dk.alloc((size_t)n));
    uint32_t grid = persistent_grid(c, n, 16);
    uint32_t gthreads = grid * kBlock;
    TRY(gs.alloc((size_t)(kStackDepth - kLdsMin) * gthreads * 4));
    hipStream_t st = c->stream;
    EAR_HIP_TRY(c, hipMemcpyAsync(da.p, p, (size_t)n * 12, hipMemcpyHostToDevice, st));
    EAR_HIP_TRY(c, hipMemcpyAsync(db.p, q, (size_t)n * 12, hipMemcpyHostToDevice, st));
    Traversal T{s->nodes, s->nodes4, s->tris, s->n_tris, gs.as<int>(), gthreads};
    if (s->width == 4)
        k_query<4, true><<<grid, kBlock, 0, st>>>(T, n, da.as<float>(), db.as<float>(), nullptr, nullptr,
                                                  dk.as<uint8_t>());
    else
        k_query<2, true><<<grid, kBlock, 0, st>>>(T, n, da.as<float>(), db.as<float>(), nullptr, nullptr,
                                                  dk.as<uint8_t>());
    EAR_HIP_TRY(c, hipGetLastError());
    EAR_HIP_TRY(c, hipMemcpyAsync(occ, dk.p, n, hipMemcpyDeviceToHost, st));
    EAR_HIP_TRY(c, hipStreamSynchronize(st));
    return EAR_OK;
}

// A batch of renders in one wavefront: every (instance, band) context's rays
// share the queues; per-instance scene data, parameters and histograms come
// from the device instance table.  A plain render is a batch of one.
ear_status run_batch(Ctx* c, uint32_t n_items, DeviceScene* const* scenes, const ear_render_desc* const* descs,
                     ear_hist* const* outs, ear_stats* st_out, Arena* arena) {
    if (n_items == 0) return EAR_ERR_INVALID_ARGUMENT;
    // no-allocation render: every buffer is carved from the arena, device
    // memory is cleared by a kernel, no events, pinned memory or graphs
    const bool noalloc = arena != nullptr;
    const bool batch = n_items > 1;
    const int width = (int)scenes[0]->width;
    std::vector<InstDev> inst(n_items);
    std::vector<std::vector<float>> src_area(n_items), src_nrm(n_items);
    uint64_t total_rays = 0;
    uint32_t max_bounces = 0;
    bool instr = false, any_log = false;
    size_t hist_cells = 0, value_cells = 0, direct_cells = 0, log_hits = 0, log_nseg = 0;
    std::vector<size_t> hist_off(n_items), value_off(n_items), direct_off(n_items), logh_off(n_items),
        logn_off(n_items);
    bool any_value = false, want_raw1 = false;
    size_t max_recs = 0;
    uint32_t any_mesh = 0;
    // time-tiled splat: keys (render, row, tile) of every render, and the
    // most channels of one recorder (records per shadow request)
    uint64_t n_keys = 0;
    uint32_t tile_stride = 1;
    std::vector<uint32_t> kbase(n_items + 1, 0);
    for (uint32_t i = 0; i < n_items; ++i) {
        if (!scenes[i] || !descs[i]) return EAR_ERR_INVALID_ARGUMENT;
        if ((int)scenes[i]->width != width) {
            c->last_error = "all scenes of a batch must have the same BVH width";
            return EAR_ERR_INVALID_ARGUMENT;
        }
        InstDev& I = inst[i];
        std::memset(&I, 0, sizeof(I));
        TRY(make_params(c, descs[i], &I.P));
        const ear_render_desc* D = descs[i];
        const DeviceScene* s = scenes[i];
        I.nodes = s->nodes;
        I.nodes4 = s->nodes4;
        I.tris = s->tris;
        I.nm = s->nm;
        I.mat_band = s->mat_band;
        I.n_tris = s->n_tris;
        I.inv_n = (double)(1.0f / (float)std::max<uint32_t>(1, D->n_rays));  // Recorder::Multiply(1.0f / amount)
        I.gain2 = (double)(D->source.gain * D->source.gain);                  // Recorder::Multiply(gain * gain)
        if (D->source.kind == EAR_SRC_MESH) {
            any_mesh = 1;
            uint32_t m = D->source.mesh_n_tris;
            src_area[i].resize(m);
            src_nrm[i].resize(3 * (size_t)m);
            float total = 0.0f;
            for (uint32_t k = 0; k < m; ++k) {
                const float* v = D->source.mesh_v + 9 * (size_t)k;
                src_area[i][k] = tri_area_host(v);
                total += src_area[i][k];
                V3 nn = normalized(cross(sub(V3{v[3], v[4], v[5]}, V3{v[0], v[1], v[2]}),
                                         sub(V3{v[6], v[7], v[8]}, V3{v[0], v[1], v[2]})));
                src_nrm[i][3 * k] = nn.x;
                src_nrm[i][3 * k + 1] = nn.y;
                src_nrm[i][3 * k + 2] = nn.z;
            }
            I.P.src_n_tris = m;
            I.P.src_total_area = total;
        }
        // raw sums of one-point rows are staged in the overflow stacks, which the
        // no-allocation render keeps small
        const bool raw1 = outs[i] && (outs[i]->raw || outs[i]->abs_raw);
        if (noalloc && raw1) I.P.one_point = 0;
        want_raw1 = want_raw1 || (raw1 && I.P.one_point);
        I.n_tiles = (I.P.n_bins + kTile - 1) / kTile;
        I.key_base = (uint32_t)std::min<uint64_t>(n_keys, 0xFFFFFFFFull);
        kbase[i] = I.key_base;
        n_keys += (uint64_t)3 * I.P.n_channels * I.P.hist_kinds * I.n_tiles;
        for (uint32_t r = 0; r < D->n_recorders; ++r)
            if (D->recorders[r].kind == EAR_REC_STEREO) tile_stride = 2;
        int nb = 0;
        for (int b = 0; b < 3; ++b) nb += (D->band_mask >> b) & 1u;
        total_rays += (uint64_t)D->n_rays * nb;
        max_bounces = std::max(max_bounces, D->max_bounces);
        instr = instr || (D->flags & EAR_FLAG_INSTRUMENT);
        max_recs = std::max<size_t>(max_recs, D->n_recorders);
        size_t cells = (size_t)3 * I.P.n_channels * I.P.hist_kinds * I.P.n_bins;
        hist_off[i] = hist_cells;
        hist_cells += 2 * cells;  // "+" and "-" parts
        value_off[i] = value_cells;
        if (outs[i] && (outs[i]->value || outs[i]->abs_value)) {
            value_cells += cells;
            any_value = true;
        }
        direct_off[i] = direct_cells;
        direct_cells += (size_t)3 * I.P.n_channels;
        logh_off[i] = log_hits;
        logn_off[i] = log_nseg;
        if (I.P.trace_rays) {
            log_hits += (size_t)3 * I.P.trace_rays * I.P.trace_segs;
            log_nseg += (size_t)3 * I.P.trace_rays;
            any_log = true;
        }
    }

    if (total_rays > 0xFFFFFFFFull) {
        c->last_error = "more than 2^32 - 1 rays in one call";
        return EAR_ERR_CAPACITY;
    }
    const ear_tuning& tu = c->tuning;
    kbase[n_items] = (uint32_t)std::min<uint64_t>(n_keys, 0xFFFFFFFFull);
    const uint32_t K = kbase[n_items];
    uint32_t chunk = tu.ray_chunk ? tu.ray_chunk : (1u << 23);
    uint64_t cap64 = std::min<uint64_t>((uint64_t)chunk * 3, std::max<uint64_t>(1, total_rays));
    uint32_t cap_rays = (uint32_t)cap64;
    // the shadow kernels' splat: records binned by time tile and accumulated
    // in LDS, or direct global atomics (always in the no-allocation render:
    // the records would not fit its region).  By default the tiled splat when
    // the call's keys fit the LDS counters and the queues hold at least 2^22
    // rays (on the 200k hall, 3 x 10M rays: 463.9 against 468.5 ms per
    // render); otherwise the atomics: a batch of many renders has too many
    // keys, and smaller renders do not repay the tile kernels' fixed cost per
    // iteration (the 500k hall at 3 x 781k rays: 9% slower tiled).
    const bool tiled = !noalloc && n_keys < 0x7FFFFFFFull &&
                       (tu.splat == EAR_SPLAT_TILED ||
                        (tu.splat == EAR_SPLAT_DEFAULT && n_keys <= kLdsKeys && cap_rays >= (1u << 22)));
    // walks vary in length; refilling idle lanes keeps waves busy (both
    // kernels by default)
    const bool fetch_e = tu.traversal != EAR_TRAVERSAL_STATIC;
    const bool fetch_s = tu.traversal == EAR_TRAVERSAL_FETCH_ALL || tu.traversal == EAR_TRAVERSAL_DEFAULT;
    const TravCfg cfg_e{tu.block_extend == 128 ? 128 : 256, tu.stack_lds >= 32 ? 32 : 16, width, instr, batch, fetch_e,
                        false};
    const TravCfg cfg_s{tu.block_shadow == 128 ? 128 : 256, tu.stack_lds >= 32 ? 32 : 16, width, instr, batch, fetch_s,
                        tiled};
    ExtendFn fe, fe_unused;
    ShadowFn fs, fs_unused;
    pick_kernels(cfg_e, &fe, &fs_unused);
    pick_kernels(cfg_s, &fe_unused, &fs);
    auto cap_for = [&](const void* fn, int block) -> uint32_t {
        uint32_t cap;
        if (tu.waves_per_cu) {
            cap = (uint32_t)c->num_cus * tu.waves_per_cu / std::max(1, block / 64);
        } else {
            int nb = resident_blocks(fn, block);
            cap = (uint32_t)c->num_cus * (uint32_t)std::max(1, nb);
        }
        // the no-allocation render keeps its overflow stacks small: at most
        // kNoallocWaves waves per CU in the traversal grids
        if (noalloc) cap = std::min<uint32_t>(cap, (uint32_t)c->num_cus * kNoallocWaves / std::max(1, block / 64));
        return std::max<uint32_t>(1, cap);
    };
    const uint32_t cap_e = std::max<uint32_t>(1, cap_for((const void*)fe, cfg_e.block));
    const uint32_t cap_s = std::max<uint32_t>(1, cap_for((const void*)fs, cfg_s.block));

    hipStream_t st = c->stream;
    Arena* ar = arena;
    DevBuf qo[2] = {DevBuf(c, ar), DevBuf(c, ar)}, qd[2] = {DevBuf(c, ar), DevBuf(c, ar)},
           qm[2] = {DevBuf(c, ar), DevBuf(c, ar)};
    DevBuf hits(c, ar), so(c, ar), sm(c, ar), counters(c, ar), stats(c, ar), hist(c, ar), gs(c, ar), direct(c, ar),
        value(c, ar), logh(c, ar), logn(c, ar), dinst(c, ar), dsegs(c, ar), dsegoff(c, ar), drows(c, ar),
        dvrows(c, ar), msrc(c, ar), segc(c, ar), tkey(c, ar), tpay(c, ar), tsort(c, ar), tcnt(c, ar), toff(c, ar),
        tcur(c, ar), tkb(c, ar), tfirst(c, ar), dorows(c, ar), dorawo(c, ar);
    // device memory that must start at a value: hipMemsetAsync, or in the
    // no-allocation render a fill kernel (no memset nodes if a caller
    // captures the stream)
    auto clear = [&](DevBuf& b, uint8_t byte) -> ear_status {
        if (!noalloc) {
            EAR_HIP_TRY(c, hipMemsetAsync(b.p, byte, b.n, st));
            return EAR_OK;
        }
        const size_t words = b.n / 4;  // every cleared buffer is a whole number of words
        const uint32_t w = 0x01010101u * byte;
        k_fill_u32<<<persistent_grid(c, (uint32_t)std::min<size_t>(words, 0xFFFFFFFFu), 8), kBlock, 0, st>>>(
            b.as<uint32_t>(), words, w);
        EAR_HIP_TRY(c, hipGetLastError());
        return EAR_OK;
    };
    // see iteration()
    TRY(counters.alloc(16 * 4));
    // refill counters of the closest-hit and shadow kernels, one per line
    TRY(segc.alloc(2 * kMaxSeg * kSegStride * 4));
    TRY(clear(segc, 0));
    TRY(stats.alloc(ST_N * 8 * kStatCopies));
    TRY(hist.alloc(hist_cells * 16));
    uint32_t gthreads = std::max(cap_e * (uint32_t)cfg_e.block, cap_s * (uint32_t)cfg_s.block);
    gthreads = std::max<uint32_t>(gthreads, n_items * kBlock);
    // overflow stack entries per persistent thread: the full depth, or in the
    // no-allocation render the bound of the scenes' own trees (a 4-wide node
    // visit pushes at most 3 entries, a 2-wide one at most 1, per level)
    size_t gs_entries = kStackDepth - kLdsMin;
    if (noalloc) {
        uint32_t need = 1;
        for (uint32_t i = 0; i < n_items; ++i)
            need = std::max(need, scenes[i]->width == 4 ? 3 * scenes[i]->depth4 + 1 : scenes[i]->max_depth);
        gs_entries = need > (uint32_t)kLdsMin ? need - kLdsMin : 1;
    }
    TRY(gs.alloc(gs_entries * gthreads * 4));
    TRY(direct.alloc(direct_cells * sizeof(DirectRamp)));
    if (any_value) TRY(value.alloc(value_cells * 8));
    if (any_log) {
        TRY(logh.alloc(log_hits * 4));
        TRY(logn.alloc(log_nseg * 4));
        TRY(clear(logh, 0xFE));  // 0xFEFEFEFE read back as -2
        TRY(clear(logn, 0));
    }
    // mesh-source tables, one allocation
    size_t msrc_floats = 0;
    std::vector<size_t> msrc_off(n_items);
    for (uint32_t i = 0; i < n_items; ++i) {
        msrc_off[i] = msrc_floats;
        msrc_floats += 9 * (size_t)inst[i].P.src_n_tris + src_area[i].size() + src_nrm[i].size();
    }
    if (msrc_floats) TRY(msrc.alloc(msrc_floats * 4));
    for (uint32_t i = 0; i < n_items; ++i) {
        InstDev& I = inst[i];
        I.hist = hist.as<unsigned long long>() + 2 * hist_off[i];
        I.direct = direct.as<DirectRamp>() + direct_off[i];
        I.value = (outs[i] && (outs[i]->value || outs[i]->abs_value)) ? value.as<double>() + value_off[i] : nullptr;
        I.log_hits = I.P.trace_rays ? logh.as<int32_t>() + logh_off[i] : nullptr;
        I.log_nseg = I.P.trace_rays ? logn.as<uint32_t>() + logn_off[i] : nullptr;
        if (I.P.src_n_tris) {
            float* base = msrc.as<float>() + msrc_off[i];
            size_t m = I.P.src_n_tris;
            EAR_HIP_TRY(c, hipMemcpyAsync(base, descs[i]->source.mesh_v, m * 36, hipMemcpyHostToDevice, st));
            EAR_HIP_TRY(c, hipMemcpyAsync(base + 9 * m, src_area[i].data(), m * 4, hipMemcpyHostToDevice, st));
            EAR_HIP_TRY(c, hipMemcpyAsync(base + 10 * m, src_nrm[i].data(), m * 12, hipMemcpyHostToDevice, st));
            I.M = MeshSrc{base, base + 9 * m, base + 10 * m};
        }
    }
    TRY(dinst.alloc(sizeof(InstDev) * n_items));
    EAR_HIP_TRY(c, hipMemcpyAsync(dinst.p, inst.data(), sizeof(InstDev) * n_items, hipMemcpyHostToDevice, st));
    TRY(clear(hist, 0));
    TRY(clear(stats, 0));
    TRY(clear(counters, 0));

    // every (instance, band) context as a run of rays, cut into chunks
    std::vector<GenSeg> all;
    for (uint32_t i = 0; i < n_items; ++i)
        for (int b = 0; b < 3; ++b)
            if ((descs[i]->band_mask >> b) & 1u && descs[i]->n_rays) all.push_back(GenSeg{i, (uint32_t)b, 0, descs[i]->n_rays});
    TRY(dsegs.alloc(sizeof(GenSeg) * std::max<size_t>(1, all.size())));
    TRY(dsegoff.alloc(4 * std::max<size_t>(1, all.size())));
    // the histogram rows of the finishing kernels: one per (instance, band,
    // channel, kind) for the prefix sums, one per (instance, band, channel)
    // for the combination step
    // (one-point items: one per (instance, band, channel), and where each row's
    // raw sums begin, in cells)
    std::vector<uint4> rows, vrows, orows;
    std::vector<uint64_t> raw_off(1, 0);
    uint32_t max_nb = 1, max_nb1 = 1;
    for (uint32_t i = 0; i < n_items; ++i)
        for (uint32_t b = 0; b < 3; ++b)
            if ((descs[i]->band_mask >> b) & 1u)
                for (uint32_t ch = 0; ch < inst[i].P.n_channels; ++ch) {
                    if (inst[i].P.one_point) {
                        orows.push_back(make_uint4(i, b, ch, 0));
                        raw_off.push_back(raw_off.back() + (uint64_t)inst[i].P.hist_kinds * inst[i].P.n_bins);
                        max_nb1 = std::max(max_nb1, inst[i].P.n_bins);
                        continue;
                    }
                    for (uint32_t kind = 0; kind < inst[i].P.hist_kinds; ++kind) rows.push_back(make_uint4(i, b, ch, kind));
                    vrows.push_back(make_uint4(i, b, ch, 0));
                    max_nb = std::max(max_nb, inst[i].P.n_bins);
                }
    TRY(drows.alloc(sizeof(uint4) * rows.size()));
    TRY(dvrows.alloc(sizeof(uint4) * vrows.size()));
    TRY(dorows.alloc(sizeof(uint4) * orows.size()));
    TRY(dorawo.alloc(8 * raw_off.size()));

    // the ray queues, their hit records and the shadow queue; a queue's
    // shading emits <= cap * recorders requests, and mesh sources add their
    // k = 0 connections of the rays generated in the same iteration
    const size_t sh_per_ray = std::max<size_t>(1, max_recs) * (any_mesh ? 2 : 1);
    if (noalloc) {
        // as many rays in flight as the rest of the region holds
        const size_t per_ray = 6 * 16 + 8 + sh_per_ray * 32;
        const size_t slack = 9 * kArenaAlign;
        const size_t fit = arena->left() > slack ? (arena->left() - slack) / per_ray : 0;
        if (fit < kNoallocMinRays) {
            c->last_error = "render needs more device memory than the no-allocation scratch region holds (" +
                            std::to_string(arena->size >> 20) + " MiB): histograms, stacks and tables take " +
                            std::to_string(arena->used >> 20) + " MiB";
            return EAR_ERR_CAPACITY;
        }
        cap_rays = (uint32_t)std::min<size_t>(cap_rays, fit / 64 * 64);
    }
    for (int k = 0; k < 2; ++k) {
        TRY(qo[k].alloc((size_t)cap_rays * 16));
        TRY(qd[k].alloc((size_t)cap_rays * 16));
        TRY(qm[k].alloc((size_t)cap_rays * 16));
    }
    TRY(hits.alloc((size_t)cap_rays * 8));
    const size_t cap_sh = (size_t)cap_rays * sh_per_ray;
    TRY(so.alloc(cap_sh * 16));
    TRY(sm.alloc(cap_sh * 16));
    TileOut tile_out{nullptr, nullptr, tile_stride};
    if (tiled) {
        const size_t n_rec = cap_sh * tile_stride;
        TRY(tkey.alloc(n_rec * 4));
        TRY(tpay.alloc(n_rec * 8));
        TRY(tsort.alloc(n_rec * 8));
        TRY(tcnt.alloc((size_t)K * 4));
        TRY(toff.alloc(((size_t)K + 1) * 4));
        TRY(tcur.alloc((size_t)K * 4));
        TRY(tkb.alloc(((size_t)n_items + 1) * 4));
        TRY(tfirst.alloc((n_rec + kTileChunk - 1) / kTileChunk * 4));
        TRY(clear(tcnt, 0));
        EAR_HIP_TRY(c, hipMemcpyAsync(tkb.p, kbase.data(), 4 * kbase.size(), hipMemcpyHostToDevice, st));
        tile_out.key = tkey.as<uint32_t>();
        tile_out.pay = tpay.as<uint2>();
    }

    uint32_t* cnt = counters.as<uint32_t>();
    unsigned long long* stp = stats.as<unsigned long long>();
    const InstDev* di = dinst.as<InstDev>();
    int* gsp = gs.as<int>();

    // the queue counters read by the host: pinned memory, or in the
    // no-allocation render a host array (a synchronous copy)
    uint32_t host_cnt[8] = {};
    uint32_t* pinned = host_cnt;
    if (!noalloc) EAR_HIP_TRY(c, hipHostMalloc((void**)&pinned, 32, hipHostMallocDefault));
    struct PinGuard {
        uint32_t* p;
        ~PinGuard() {
            if (p) hipHostFree(p);
        }
    } pg{noalloc ? nullptr : pinned};

    std::vector<EventPair> ev_ext, ev_sha, ev_shw, ev_spl;
    auto mk = [&](std::vector<EventPair>& v) -> EventPair& {
        v.emplace_back();
        hipEventCreate(&v.back().a);
        hipEventCreate(&v.back().b);
        return v.back();
    };
    hipEvent_t t0 = nullptr, t1 = nullptr;
    if (!noalloc) {
        EAR_HIP_TRY(c, hipEventCreate(&t0));
        EAR_HIP_TRY(c, hipEventCreate(&t1));
        EAR_HIP_TRY(c, hipEventRecord(t0, st));
    }

    // The bounce loop is device driven: every iteration tops the current
    // queue up with new rays (k_plan + k_generate), extends and shades it
    // into the other queue, and connects the shadow requests.  Kernels read
    // their counts from device memory and run on fixed persistent grids, so
    // the host only checks for the end every few iterations, and an
    // iteration block can be captured once as a graph and replayed.
    uint32_t bounces = 0, launches = 0;
    ear_status status = EAR_OK;
    Queue qq[2] = {Queue{qo[0].as<float4>(), qd[0].as<float4>(), qm[0].as<uint4>()},
                   Queue{qo[1].as<float4>(), qd[1].as<float4>(), qm[1].as<uint4>()}};
    ShadowQ SQ{so.as<float4>(), sm.as<float4>()};
    {
        std::vector<uint32_t> off(all.size());
        uint64_t acc = 0;
        for (size_t k = 0; k < all.size(); ++k) {
            off[k] = (uint32_t)acc;
            acc += all[k].count;
        }
        if (!all.empty()) {
            EAR_HIP_TRY(c, hipMemcpyAsync(dsegs.p, all.data(), sizeof(GenSeg) * all.size(), hipMemcpyHostToDevice, st));
            EAR_HIP_TRY(c, hipMemcpyAsync(dsegoff.p, off.data(), 4 * off.size(), hipMemcpyHostToDevice, st));
        }
    }
    const uint32_t n_segs = (uint32_t)std::max<size_t>(1, all.size());
    const uint32_t total32 = (uint32_t)total_rays;
    // every emitted ray has a first segment to trace
    uint32_t dense = 1;
    for (uint32_t i = 0; i < n_items; ++i)
        if (1.0 < inst[i].P.cutoff || inst[i].P.max_bounces == 0) dense = 0;
    const uint32_t g_gen = grid_for(
        cap_rays, rounds_cap(c, batch ? (const void*)k_generate<true> : (const void*)k_generate<false>, tu.waves_per_cu, kBlock),
        kBlock);
    const uint32_t g_shade = grid_for(
        cap_rays,
        rounds_cap(c, batch ? (const void*)k_shade<true> : (const void*)k_shade<false>, tu.waves_per_cu, kShadeBlock),
        kShadeBlock);
    const uint32_t g_ext = grid_for(cap_rays, cap_e, cfg_e.block);
    const uint32_t g_shw = grid_for((uint32_t)std::min<size_t>(cap_sh, 0xFFFFFFFFu), cap_s, cfg_s.block);
    // count and scatter: the same grid, two workgroups per CU (at least 16k
    // record slots each).  Fewer, longer-running workgroups give each key
    // longer runs of the sorted array per workgroup, so fewer cache lines are
    // written in part from several XCDs (on the hall: 36.0 -> 30.3 ms of
    // tile kernels per render against four per CU, 31.5 ms at one)
    const uint32_t g_tile = (uint32_t)std::max<size_t>(
        1, std::min<size_t>((size_t)c->num_cus * 2, cap_sh * tile_stride / (kTileBlock * kTileBatch * 4)));
    // splat: one workgroup per kTileChunk records of the most one launch can write
    const uint32_t g_splat = (uint32_t)std::max<size_t>(1, (cap_sh * tile_stride + kTileChunk - 1) / kTileChunk);
    // eager: the bounce loop launched from the host (always in the
    // no-allocation render); timed: with per-kernel events
    const bool eager = tu.graph_iters == 0 || noalloc;
    const bool timed = eager && !noalloc;
    const uint32_t refill = tu.refill ? tu.refill : 24u;
    const uint32_t fchunk = tu.fetch_chunk;  // 0: one entry per idle lane
    const uint32_t nseg = tu.fetch_segments ? std::min<uint32_t>(tu.fetch_segments, kMaxSeg) : kSegDefault;
    const Fetch fq_e{segc.as<uint32_t>(), refill, fchunk, nseg},
        fq_s{segc.as<uint32_t>() + kMaxSeg * kSegStride, refill, fchunk, nseg};
    // tops queue cur up with new rays
    auto generate = [&](int cur) {
        // [2 q] rays of queue q, [2 q + 1] the shadow requests made with it as
        // the output queue; [4] generation cursor, [6..8] plan
        uint32_t *nq = cnt + 2 * cur, *nsq = cnt + 2 * (1 - cur) + 1;
        k_plan<<<1, 64, 0, st>>>(cnt + 4, total32, cap_rays, dense, nq, cnt + 6);
        if (batch)
            k_generate<true><<<g_gen, kBlock, 0, st>>>(di, dsegs.as<GenSeg>(), dsegoff.as<uint32_t>(), n_segs, 0u,
                                                       cnt + 6, (uint32_t)max_recs, any_mesh, dense, qq[cur], nq, SQ,
                                                       nsq, stp);
        else
            k_generate<false><<<g_gen, kBlock, 0, st>>>(di, dsegs.as<GenSeg>(), dsegoff.as<uint32_t>(), n_segs, 0u,
                                                        cnt + 6, (uint32_t)max_recs, any_mesh, dense, qq[cur], nq, SQ,
                                                        nsq, stp);
    };
    // traces the shadow requests of the iteration that consumes queue cur
    auto connect = [&](int cur) {
        uint32_t* nsq = cnt + 2 * (1 - cur) + 1;
        EventPair* e3 = timed ? &mk(ev_shw) : nullptr;
        if (e3) hipEventRecord(e3->a, st);
        hipLaunchKernelGGL(fs, dim3(g_shw), dim3(cfg_s.block), 0, st, di, gsp, gthreads, SQ, (const uint32_t*)nsq,
                           stp, fq_s, tile_out);
        if (e3) hipEventRecord(e3->b, st);
        if (tiled) {
            // the records of this launch, grouped by key and splatted per tile
            EventPair* e4 = timed ? &mk(ev_spl) : nullptr;
            if (e4) hipEventRecord(e4->a, st);
            k_tile_count<<<g_tile, kTileBlock, 0, st>>>(tkey.as<uint32_t>(), nsq, tile_stride, tcnt.as<uint32_t>(),
                                                        K);
            k_tile_scan<<<1, 1024, 0, st>>>(tcnt.as<uint32_t>(), toff.as<uint32_t>(), tcur.as<uint32_t>(), K,
                                            tfirst.as<uint32_t>());
            k_tile_scatter<<<g_tile, kTileBlock, 0, st>>>(di, tkb.as<uint32_t>(), n_items, tkey.as<uint32_t>(),
                                                          tpay.as<uint2>(), nsq, tile_stride, tcur.as<uint32_t>(),
                                                          K, tsort.as<uint2>());
            k_tile_splat<<<g_splat, kTileBlock, 0, st>>>(di, tkb.as<uint32_t>(), n_items, toff.as<uint32_t>(), K,
                                                         tfirst.as<uint32_t>(), tsort.as<uint2>());
            if (e4) hipEventRecord(e4->b, st);
            launches += 4;
        }
    };
    // one iteration; cur = the queue it consumes
    auto iteration = [&](int cur) {
        uint32_t* nq = cnt + 2 * cur;
        generate(cur);
        EventPair* e1 = timed ? &mk(ev_ext) : nullptr;
        if (e1) hipEventRecord(e1->a, st);
        hipLaunchKernelGGL(fe, dim3(g_ext), dim3(cfg_e.block), 0, st, di, gsp, gthreads, qq[cur], (const uint32_t*)nq,
                           hits.as<int2>(), stp, fq_e);
        if (e1) hipEventRecord(e1->b, st);
        EventPair* e2 = timed ? &mk(ev_sha) : nullptr;
        if (e2) hipEventRecord(e2->a, st);
        unsigned long long* n_out = (unsigned long long*)(cnt + 2 * (1 - cur));
        if (batch)
            k_shade<true><<<g_shade, kShadeBlock, 0, st>>>(di, qq[cur], nq, hits.as<int2>(), qq[1 - cur], SQ, n_out,
                                                           (uint32_t)max_recs, stp);
        else
            k_shade<false><<<g_shade, kShadeBlock, 0, st>>>(di, qq[cur], nq, hits.as<int2>(), qq[1 - cur], SQ, n_out,
                                                            (uint32_t)max_recs, stp);
        if (e2) hipEventRecord(e2->b, st);
        connect(cur);
        // the consumed queue, the shadow queue and the fetch counters
        k_reset_iter<<<1, 64, 0, st>>>(cnt, (1u << (2 * cur)) | (1u << (2 * (1 - cur) + 1)), segc.as<uint32_t>(), 2 * kMaxSeg);
        launches += 6;
        ++bounces;
    };
    // the render has ended once every ray was taken and no queue holds any
    auto finished = [&](int cur, bool* done) -> ear_status {
        EAR_HIP_TRY(c, hipMemcpyAsync(pinned, cnt, 20, hipMemcpyDeviceToHost, st));
        EAR_HIP_TRY(c, hipStreamSynchronize(st));
        *done = pinned[2 * cur] == 0 && pinned[4] == total32;
        return EAR_OK;
    };
    // the tail: every ray emitted and few live ones left (queue cur, of
    // pinned[2 cur] rays, read by finished); one launch traces them to their ends
    // (tail_rays 0: 2^21 live rays, or every ray when no scene has more than
    // 64 triangles: their walks are so short that the queues between the
    // wavefront kernels cost more than a segment's wait for the wave's longest
    // walk.  The 12-triangle box of 1M rays: 22 ms, 41 with the last 2^20 only;
    // 32 rooms at 2^20, 2^21, 2^22, all: 116, 113, 110, 100 ms; the 200k hall
    // 326, 321, 319, 356; 12 keyframes of the 100k hall 72.3, 72.2, 74.0,
    // 86.7: rooms would take more, halls do not, and their trees do not tell
    // them apart; 1: no tail launch.  Renders wholly below it, from the first
    // segment in the tail against the last 2^20 and against no tail: the 200k
    // hall of 3 x 200k rays 14.9, 15.0, 31.5 ms, of 3 x 500k 27.6, 30.3, 41.6,
    // of 3 x 650k 32.6, 34.6, 46.2; a 20k hall 24.3, 27.7, 35.0 and a 500k hall
    // 45.9, 46.0, 63.1 of 3 x 650k; a 50k room 24.0, 36.8, 42.3)
    uint32_t max_tris = 0;
    for (uint32_t i = 0; i < n_items; ++i) max_tris = std::max(max_tris, inst[i].n_tris);
    const uint32_t tail_default = max_tris <= 64 ? 0xFFFFFFFFu : (1u << 21);
    const uint32_t tail_rays = tu.tail_rays == 0 ? tail_default : (tu.tail_rays == 1 ? 0u : tu.tail_rays);
    const bool tail_ok = tail_rays > 0 && !instr && !any_log;
    const TailFn ft = tail_ok ? pick_tail(cfg_e) : nullptr;
    auto tail = [&](int cur, bool* done) -> ear_status {
        if (*done || !ft || pinned[4] != total32 || pinned[2 * cur] > tail_rays) return EAR_OK;
        // (one round of resident blocks: the waves of a second one would start
        // on the last rays when the first ends)
        const uint32_t g_tail = std::min(cap_e, cap_for((const void*)ft, cfg_e.block));
        hipLaunchKernelGGL(ft, dim3(g_tail), dim3(cfg_e.block), 0, st, di, gsp, gthreads, qq[cur],
                           (const uint32_t*)(cnt + 2 * cur), (uint32_t)max_recs, fq_e, stp);
        hipError_t le = hipGetLastError();
        if (le != hipSuccess) return hip_status(c, le, "tail launch");
        launches += 1;
        *done = true;
        return EAR_OK;
    };
    const uint32_t max_iters = max_bounces + 2 + (uint32_t)((total_rays + cap_rays - 1) / cap_rays) * (max_bounces + 1);
    int cur = 0;
    bool done = false;
    if (ft && dense && total32 <= cap_rays && total32 <= tail_rays) {
        // all rays are the tail's from the first segment: emission, the
        // connections that an emitting mesh makes, one launch.  (Of the four
        // bounce iterations before a look at the counts, each with the whole
        // population's first hits on the same few bins, the 1M-ray box spent
        // 4 of its 22 ms and a room with an emitting mesh 5 of 36.)
        generate(0);
        if (any_mesh) connect(0);
        k_reset_iter<<<1, 64, 0, st>>>(cnt, 8u, segc.as<uint32_t>(), 2 * kMaxSeg);
        launches += 4;
        pinned[0] = pinned[4] = total32;
        status = tail(0, &done);
    }
    if (done || status != EAR_OK) {
    } else if (eager) {
        const uint32_t every = 4;
        while (!done && status == EAR_OK) {
            for (uint32_t k = 0; k < every; ++k) {
                iteration(cur);
                cur = 1 - cur;
            }
            hipError_t le = hipGetLastError();
            if (le != hipSuccess) status = hip_status(c, le, "tracer launch");
            if (status == EAR_OK) status = finished(cur, &done);
            if (status == EAR_OK) status = tail(cur, &done);
            if (!done && bounces > max_iters) {
                c->last_error = "bounce loop did not drain";
                status = EAR_ERR_INTERNAL;
            }
        }
    } else {
        const uint32_t per = std::max<uint32_t>(2, (tu.graph_iters + 1) & ~1u);  // even: replays start on queue 0
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        EAR_HIP_TRY(c, hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        for (uint32_t k = 0; k < per; ++k) iteration((int)(k & 1u));
        hipError_t ce = hipStreamEndCapture(st, &graph);
        if (ce == hipSuccess) ce = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (ce != hipSuccess) status = hip_status(c, ce, "bounce-loop graph");
        const uint32_t captured = bounces;
        bounces = 0;
        launches = 0;
        while (!done && status == EAR_OK) {
            hipError_t le = hipGraphLaunch(exec, st);
            bounces += captured;
            launches += 1;
            if (le != hipSuccess) status = hip_status(c, le, "bounce-loop graph launch");
            if (status == EAR_OK) status = finished(0, &done);
            if (status == EAR_OK) status = tail(0, &done);  // an even replay ends on queue 0
            if (!done && bounces > max_iters + per) {
                c->last_error = "bounce loop did not drain";
                status = EAR_ERR_INTERNAL;
            }
        }
        if (exec) hipGraphExecDestroy(exec);
        if (graph) hipGraphDestroy(graph);
    }
    if (status != EAR_OK) return status;
    if (width == 4)
        k_direct<4><<<n_items, kBlock, 0, st>>>(di, gsp, gthreads, stp);
    else
        k_direct<2><<<n_items, kBlock, 0, st>>>(di, gsp, gthreads, stp);
    if (!rows.empty()) {
        EAR_HIP_TRY(c, hipMemcpyAsync(drows.p, rows.data(), sizeof(uint4) * rows.size(), hipMemcpyHostToDevice, st));
        k_finalize<<<(uint32_t)rows.size(), kFinBlock, 0, st>>>(di, drows.as<uint4>());
        EAR_HIP_TRY(c, hipMemcpyAsync(dvrows.p, vrows.data(), sizeof(uint4) * vrows.size(), hipMemcpyHostToDevice, st));
        k_values<<<dim3((max_nb + 255) / 256, (uint32_t)vrows.size()), 256, 0, st>>>(di, dvrows.as<uint4>());
    }
    // One-point rows: finished in one launch.  Raw sums that are wanted go to the
    // overflow stacks, which no walk uses any more, and from there to the caller:
    // all of them in that launch, or if they do not fit in runs of rows (of bins,
    // if a row is longer) finished again after the render's time is taken.  (A
    // buffer of their own made a render of few rays with long rows need more
    // memory than its tracing.)
    const uint32_t n_or = (uint32_t)orows.size();
    unsigned long long* stage = gs.as<unsigned long long>();
    const uint64_t cells = gs.n / 16;
    const bool whole = raw_off[n_or] <= cells;
    auto finish = [&](uint32_t r0, uint32_t n, uint32_t b0, uint32_t b1, unsigned long long* raw) {
        for (uint32_t k = 0; k < n; k += 32768u)  // a grid's second dimension
            k_finish<<<dim3((b1 - b0 + 255) / 256, std::min(n - k, 32768u)), 256, 0, st>>>(
                di, dorows.as<uint4>(), r0 + k, b0, b1, raw ? raw + 2 * (raw_off[r0 + k] - raw_off[r0]) : nullptr,
                dorawo.as<uint64_t>());
    };
    if (n_or) {
        EAR_HIP_TRY(c, hipMemcpyAsync(dorows.p, orows.data(), sizeof(uint4) * orows.size(), hipMemcpyHostToDevice, st));
        EAR_HIP_TRY(c, hipMemcpyAsync(dorawo.p, raw_off.data(), 8 * raw_off.size(), hipMemcpyHostToDevice, st));
        finish(0, n_or, 0, max_nb1, want_raw1 && whole ? stage : nullptr);
    }
    EAR_HIP_TRY(c, hipGetLastError());
    if (t1) EAR_HIP_TRY(c, hipEventRecord(t1, st));
    EAR_HIP_TRY(c, hipStreamSynchronize(st));
    // bins [b0, b1) of row r, staged from cell `from` on, to the caller
    auto copy_raw = [&](uint32_t r, uint32_t b0, uint32_t b1, uint64_t from) -> ear_status {
        const uint4 w = orows[r];
        const RenderParams& P = inst[w.x].P;
        for (uint32_t k = 0; outs[w.x] && k < P.hist_kinds; ++k) {
            int64_t* raw = k == 0 ? outs[w.x]->raw : outs[w.x]->abs_raw;
            if (raw)
                EAR_HIP_TRY(c, hipMemcpyAsync(raw + 2 * (((size_t)w.y * P.n_channels + w.z) * P.n_bins + b0),
                                              stage + 2 * (from + (uint64_t)k * (b1 - b0)), (size_t)(b1 - b0) * 16,
                                              hipMemcpyDeviceToHost, st));
        }
        return EAR_OK;
    };
    for (uint32_t r0 = 0; want_raw1 && r0 < n_or;) {
        const RenderParams& P = inst[orows[r0].x].P;
        uint32_t r1 = r0 + 1;
        if (raw_off[r1] - raw_off[r0] > cells) {
            const uint32_t per = (uint32_t)(cells / P.hist_kinds);
            for (uint32_t b0 = 0; b0 < P.n_bins;) {
                const uint32_t b1 = P.n_bins - b0 > per ? b0 + per : P.n_bins;
                finish(r0, 1, b0, b1, stage);
                EAR_HIP_TRY(c, hipGetLastError());
                TRY(copy_raw(r0, b0, b1, 0));
                b0 = b1;
            }
        } else {
            while (r1 < n_or && raw_off[r1 + 1] - raw_off[r0] <= cells) ++r1;
            if (!whole) finish(r0, r1 - r0, 0, max_nb1, stage);
            EAR_HIP_TRY(c, hipGetLastError());
            for (uint32_t r = r0; r < r1; ++r) TRY(copy_raw(r, 0, inst[orows[r].x].P.n_bins, raw_off[r] - raw_off[r0]));
        }
        r0 = r1;
    }

    // copy out [band slot][channel][bin] rows of every rendered band
    for (uint32_t i = 0; i < n_items; ++i) {
        ear_hist* out = outs[i];
        if (!out) continue;
        const RenderParams& P = inst[i].P;
        const size_t nb = P.n_bins;
        const uint32_t nch = P.n_channels;
        for (int b = 0; b < 3; ++b) {
            if (!((descs[i]->band_mask >> b) & 1u)) continue;
            for (uint32_t ch = 0; ch < nch; ++ch) {
                for (uint32_t kind = 0; kind < P.hist_kinds; ++kind) {
                    size_t roff = (((size_t)b * nch + ch) * P.hist_kinds + kind) * nb;
                    size_t ooff = ((size_t)b * nch + ch) * nb;
                    int64_t* raw = kind == 0 ? out->raw : out->abs_raw;
                    double* val = kind == 0 ? out->value : out->abs_value;
                    if (raw && !P.one_point)
                        EAR_HIP_TRY(c, hipMemcpyAsync(raw + 2 * ooff,
                                                      hist.as<unsigned long long>() + 2 * (hist_off[i] + 2 * roff),
                                                      nb * 16, hipMemcpyDeviceToHost, st));
                    if (val && inst[i].value)
                        EAR_HIP_TRY(c, hipMemcpyAsync(val + ooff, value.as<double>() + value_off[i] + roff, nb * 8,
                                                      hipMemcpyDeviceToHost, st));
                }
            }
        }
        if (P.trace_rays) {
            std::vector<int32_t> lh((size_t)3 * P.trace_rays * P.trace_segs);
            std::vector<uint32_t> ln((size_t)3 * P.trace_rays);
            EAR_HIP_TRY(c, hipMemcpyAsync(lh.data(), logh.as<int32_t>() + logh_off[i], lh.size() * 4,
                                          hipMemcpyDeviceToHost, st));
            EAR_HIP_TRY(c, hipMemcpyAsync(ln.data(), logn.as<uint32_t>() + logn_off[i], ln.size() * 4,
                                          hipMemcpyDeviceToHost, st));
            EAR_HIP_TRY(c, hipStreamSynchronize(st));
            for (int b = 0; b < 3; ++b) {
                if (!((descs[i]->band_mask >> b) & 1u)) continue;
                size_t per = (size_t)P.trace_rays * P.trace_segs;
                if (out->trace_hits) {
                    for (size_t j = 0; j < per; ++j) {
                        int32_t v = lh[(size_t)b * per + j];
                        out->trace_hits[(size_t)b * per + j] = v == (int32_t)0xFEFEFEFE ? -2 : v;
                    }
                }
                if (out->trace_nseg)
                    std::memcpy(out->trace_nseg + (size_t)b * P.trace_rays, ln.data() + (size_t)b * P.trace_rays,
                                (size_t)P.trace_rays * 4);
            }
        }
    }
    EAR_HIP_TRY(c, hipStreamSynchronize(st));

    if (st_out) {
        std::vector<unsigned long long> hc((size_t)ST_N * kStatCopies);
        EAR_HIP_TRY(c, hipMemcpy(hc.data(), stats.p, hc.size() * 8, hipMemcpyDeviceToHost));
        unsigned long long hs[ST_N] = {};
        for (uint32_t k = 0; k < kStatCopies; ++k)
            for (int j = 0; j < ST_N; ++j)
                hs[j] = j == ST_BINS ? std::max(hs[j], hc[(size_t)k * ST_N + j]) : hs[j] + hc[(size_t)k * ST_N + j];
        std::memset(st_out, 0, sizeof(*st_out));
        st_out->segments = hs[ST_SEGMENTS];
        st_out->shadow_rays = hs[ST_SHADOW];
        st_out->contributions = hs[ST_CONTRIB];
        st_out->rays = hs[ST_RAYS];
        st_out->node_visits_closest = hs[ST_NV_CL];
        st_out->tri_tests_closest = hs[ST_NT_CL];
        st_out->node_visits_shadow = hs[ST_NV_SH];
        st_out->tri_tests_shadow = hs[ST_NT_SH];
        st_out->bounces_launched = bounces;
        st_out->launches = launches;
        float ms = 0;
        if (t0 && t1) hipEventElapsedTime(&ms, t0, t1);
        st_out->trace_ms = ms;
        auto sum = [](std::vector<EventPair>& v) {
            double a = 0;
            for (auto& e : v) {
                float m = 0;
                hipEventElapsedTime(&m, e.a, e.b);
                a += m;
            }
            return a;
        };
        st_out->extend_ms = sum(ev_ext);
        st_out->shade_ms = sum(ev_sha);
        st_out->shadow_ms = sum(ev_shw);
        st_out->splat_ms = sum(ev_spl);
        st_out->shadow_contributions = hs[ST_SH_CONTRIB];
        st_out->shadow_ramps = hs[ST_SH_RAMPS];
        st_out->extend_launches = (uint32_t)ev_ext.size();
        st_out->shadow_launches = (uint32_t)ev_shw.size();
        st_out->extend_queries = hs[ST_SEGMENTS] - hs[ST_TAIL_SEG];  // the timed k_extend launches' share
        st_out->shadow_queries = hs[ST_SHADOW] - hs[ST_TAIL_SH];
        st_out->dropped_ramps = hs[ST_DROPPED];
        st_out->bins_needed = (uint32_t)std::min<unsigned long long>(hs[ST_BINS], 0xFFFFFFFFull);
    }
    for (auto* v : {&ev_ext, &ev_sha, &ev_shw, &ev_spl})
        for (auto& e : *v) {
            hipEventDestroy(e.a);
            hipEventDestroy(e.b);
        }
    if (t0) hipEventDestroy(t0);
    if (t1) hipEventDestroy(t1);
    return EAR_OK;
}

ear_status run_render(Ctx* c, DeviceScene* s, const ear_render_desc* d, ear_hist* out, ear_stats* st) {
    DeviceScene* sc[1] = {s};
    const ear_render_desc* dd[1] = {d};
    ear_hist* oo[1] = {out};
    return run_batch(c, 1, sc, dd, oo, st);
}

}  // namespace ear

// ===========================================================================
// Adjoint: gradient of a loss on the histograms with respect to the rendered
// bands' per-material reflection coefficient and specularity.
// ===========================================================================
namespace ear {
namespace {

constexpr int kAdMaxMat = 8;
// The gradient is accumulated into kGradCopies copies, a block adding into
// copy blockIdx % kGradCopies, and the copies are summed at the end: the
// per-wave partials of every launch would otherwise all land on the same
// 2 n_mat addresses, and same-address atomics serialise in the L2.
constexpr uint32_t kGradCopies = 128;

// Tangent state of the rays of a queue, SoA [q][field][slot] with fields
// {o.xyz, d.xyz, dL, dlogI} per specularity parameter q, then
// dlogI_refl[q][slot].
struct Tangents {
    float* t;  // [n_mat][8][cap]
    float* r;  // [n_mat][cap]
    uint32_t cap;
    __device__ float& f(uint32_t q, int field, uint32_t slot) const {
        return t[((size_t)q * 8 + field) * cap + slot];
    }
    __device__ float& refl(uint32_t q, uint32_t slot) const { return r[(size_t)q * cap + slot]; }
};

// The adjoint histograms as prefix sums: row (band, channel) holds bins + 1
// pairs {sum_{b<j} a[b], sum_{b<j} b a[b]}, so that a ramp's weighted sum
// sum_b (w + s - b) a[b] over its bins is four loads at any width.
struct AdjArgs {
    const double2* adj_s;  // [3][n_ch][bins + 1] prefix sums of dL / d raw (signed), or null
    const double2* adj_a;  // [3][n_ch][bins + 1] prefix sums of dL / d raw (|.|), or null
    double* grad;         // [3][2][n_mat]: band, {refl, spec}, material (copy 0)
    uint32_t n_mat;
    uint32_t copy_stride;  // doubles from one gradient copy to the next
    __device__ double* grad_copy() const { return grad + (size_t)(blockIdx.x % kGradCopies) * copy_stride; }
};

__device__ __forceinline__ double wave_sum_d(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    return v;
}

// The end-of-launch gradient partials of a block (single instance, one
// band): per-wave sums, then summed over the block's waves in LDS, one
// atomic per value into the block's gradient copy.
__device__ void block_grad_flush(const AdjArgs& A, int band_acc, const double* g_refl, const double* g_spec,
                                 double* red /* LDS [kBlock / 64][2 * kAdMaxMat] */) {
    int band = __shfl(band_acc, 0);
    for (int l = 1; l < 64 && band < 0; ++l) band = __shfl(band_acc, l);
    const uint32_t nm = A.n_mat;
    const uint32_t wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < kAdMaxMat; ++q) {
        const double sr = wave_sum_d((uint32_t)q < nm ? g_refl[q] : 0.0);
        const double ss = wave_sum_d((uint32_t)q < nm ? g_spec[q] : 0.0);
        if (lane_id() == 0) {
            red[wave * 2 * kAdMaxMat + q] = sr;
            red[wave * 2 * kAdMaxMat + kAdMaxMat + q] = ss;
        }
    }
    // the band of the block: any wave's (one band per launch)
    __shared__ int bband;
    if (threadIdx.x == 0) bband = -1;
    __syncthreads();
    if (lane_id() == 0 && band >= 0) bband = band;
    __syncthreads();
    const int b = bband;
    if (threadIdx.x < 2 * nm && b >= 0) {
        const uint32_t q = threadIdx.x % nm, which = threadIdx.x / nm;  // 0 refl, 1 spec
        double v = 0.0;
        for (uint32_t w = 0; w < blockDim.x / 64; ++w) v += red[w * 2 * kAdMaxMat + which * kAdMaxMat + q];
        if (v != 0.0) atomicAdd(A.grad_copy() + ((size_t)b * 2 + which) * nm + q, v);
    }
}

__global__ void k_sum_grad_copies(double* g, uint32_t n, uint32_t copy_stride) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double v = 0.0;
        for (uint32_t c = 0; c < kGradCopies; ++c) v += g[(size_t)c * copy_stride + i];
        g[i] = v;
    }
}

// sum over the ramp's bins b = s .. s + w - 1 inside [0, nb) of
// a[b] (w - (b - s)) / w * per_c, from the row's prefix sums
__device__ double ramp_adjoint(const double2* pre, uint32_t nb, int s, int w, double per_c) {
    const int lo = s < 0 ? 0 : s;
    const int hi = s + w > (int)nb ? (int)nb : s + w;
    if (lo >= hi) return 0.0;
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    const f64x2 a = *(const __attribute__((address_space(1))) f64x2*)(pre + lo),
                b = *(const __attribute__((address_space(1))) f64x2*)(pre + hi);
    return ((double)(w + s) * (b.x - a.x) - (b.y - a.y)) / (double)w * per_c;
}

// dL/dc of a contribution c at time t, distance dist, direction dir.
__device__ double contribution_adjoint(const RenderParams& P, const AdjArgs& A, int band, const RecParams& R,
                                       V3 dir, float c, float t, float dist) {
    const uint32_t nb = P.n_bins, nch = P.n_channels;
    float width = sqrtf(dist);
    int w = (int)ceilf(width);
    double per_c = 2.0 / (double)width;
    double sgn = c < 0.0f ? -1.0 : 1.0;
    double a = 0.0;
    auto row = [&](const double2* base, int ch) { return base + ((size_t)band * nch + ch) * (nb + 1); };
    if (R.kind == EAR_REC_MONO) {
        int s = (int)((double)t * 44100.0);
        if (A.adj_s) a += ramp_adjoint(row(A.adj_s, R.channel), nb, s, w, per_c);
        if (A.adj_a) a += sgn * ramp_adjoint(row(A.adj_a, R.channel), nb, s, w, per_c);
    } else {
        float dt = dot(dir, V3{R.rx, R.ry, R.rz});
        float td = R.head_size / 343.0f;
        int s_right = (int)((double)(t - dt * td) * 44100.0);
        int s_left = (int)((double)(t + dt * td) * 44100.0);
        float factor = powf_ear_l2(R.head_abs[band], R.l2_head_abs[band], fabsf(dt) * R.head_size);
        double gl = 1.0, gr = 1.0;
        if (dt < 0.0f)
            gr = (double)(factor * factor);
        else
            gl = (double)(factor * factor);
        if (A.adj_s) {
            a += gl * ramp_adjoint(row(A.adj_s, R.channel), nb, s_left, w, per_c);
            a += gr * ramp_adjoint(row(A.adj_s, R.channel + 1), nb, s_right, w, per_c);
        }
        if (A.adj_a) {
            a += sgn * gl * ramp_adjoint(row(A.adj_a, R.channel), nb, s_left, w, per_c);
            a += sgn * gr * ramp_adjoint(row(A.adj_a, R.channel + 1), nb, s_right, w, per_c);
        }
    }
    return a;
}

// The primal of k_shade (same draws, same arithmetic) plus forward-mode
// tangents of every specularity parameter through the reparameterised
// direction v = normalize(h (1 - s) + r s) with h and the hit triangles held
// fixed, and of log I with respect to every reflection coefficient.  Each
// visible connection adds (dL/dc)(dc/dtheta) to the gradient.  Arrival-time
// shifts and visibility changes are not differentiated.
// BATCH: the queue holds the rays of several instances (rm.w), each with
// its own adjoint and gradient (adj[id]); the per-lane gradient partials are
// then reduced per instance at the end of every grid-stride step.
//
// Bound by the latency of its tangents (36 bytes a material and ray each way)
// at the few waves that the registers allow.  So the partial sums are in LDS,
// which lets three waves a SIMD fit, and a material's nine values are fetched
// before any is used: left to itself the compiler, short of registers, waits
// for them one after another.  3 x 1M rays in the shoebox: 142 ms with one
// wave, 117 with two, 100 with the nine loads together, 93 with three waves.
template <int WIDTH, bool BATCH>
__global__ void __launch_bounds__(kBlock, 3) k_shade_ad(const InstDev* __restrict__ inst, int* gstack,
                                                      uint32_t gthreads, Queue qin, const uint32_t* __restrict__ n_in,
                                                      const int2* __restrict__ hits, Tangents tin, Queue qout,
                                                      uint32_t* __restrict__ n_out, Tangents tout, AdjArgs A0,
                                                      const AdjArgs* __restrict__ adj,
                                                      unsigned long long* __restrict__ stats) {
    __shared__ int lds[kLdsMin * kBlock];
    uint32_t n = *n_in;
    uint32_t n_done = 0;
    uint32_t gtid = blockIdx.x * kBlock + threadIdx.x;
    __shared__ double sums[2 * kAdMaxMat * kBlock];
    double *g_refl = sums + threadIdx.x, *g_spec = g_refl + kAdMaxMat * kBlock;
    for (int q = 0; q < kAdMaxMat; ++q) g_refl[q * kBlock] = g_spec[q * kBlock] = 0.0;
    int band_acc = -1;
    uint32_t nvis = 0, ntri = 0;
    uint32_t my_id = 0;
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        uint32_t i = base + threadIdx.x;
        bool cont = false;
        float4 no{}, nd{};
        uint4 nmeta{};
        float dtan[kAdMaxMat][8];
        float drefl[kAdMaxMat];
        uint32_t nm = A0.n_mat;
        if (i < n) {
            float4 ro = qin.o[i];
            float4 rd = qin.d[i];
            uint4 rm = qin.m[i];
            const uint32_t id = BATCH ? rm.w : 0u;
            my_id = id;
            const InstDev& In = inst[id];
            const RenderParams& P = In.P;
            const AdjArgs& A = BATCH ? adj[id] : A0;
            nm = A.n_mat;
            int band = (int)(rm.z & 0xFFu);
            band_acc = band;
            uint32_t k = ((rm.z >> 8) & 0xFFFFu) + 1;
            int2 h = hits[i];
            if (h.y >= 0) {
                float t = __int_as_float(h.x);
                V3 o{ro.x, ro.y, ro.z};
                V3 d{rd.x, rd.y, rd.z};
                V3 p{o.x + d.x * t, o.y + d.y * t, o.z + d.z * t};
                float4 nmv = ldg(In.nm + h.y);
                V3 N{nmv.x, nmv.y, nmv.z};
                V3 nrm = dot(N, d) > 0.0f ? V3{N.x * -1.0f, N.y * -1.0f, N.z * -1.0f} : N;
                uint32_t mat = __float_as_uint(nmv.w);
                float4 mb = ldg(In.mat_band + 3 * mat + band);
                Rng rng;
                rng.init(P.seed, rm.x, P.ctx_word[band], P.instance, rm.y);
                int bt = kReflect;
                if (mb.x >= 0.0f) bt = (rng.next() <= mb.x) ? kReflect : kRefract;
                float spec = mb.y;
                if (bt == kRefract) nrm = neg(nrm);
                V3 dist3 = sub(p, o);
                float l = length(dist3);
                float I = ro.w;
                I *= powf_ear_l2(P.air[band], P.l2_air[band], l);
                float L = rd.w + l;
                I *= mb.z;
                V3 prev = normalized(d);
                const double ln_air = log((double)P.air[band]);
                // tangents at the hit point (plane of the hit triangle)
                const double Nd = (double)N.x * d.x + (double)N.y * d.y + (double)N.z * d.z;
                const double dn = (double)length(d);
                double dprev[kAdMaxMat][3];
                for (uint32_t q = 0; q < nm; ++q) {
                    float tv[9];
#pragma unroll
                    for (int f = 0; f < 8; ++f) tv[f] = tin.f(q, f, i);
                    tv[8] = tin.refl(q, i);
                    // (all nine in registers from here on)
                    asm volatile(""
                                 : "+v"(tv[0]), "+v"(tv[1]), "+v"(tv[2]), "+v"(tv[3]), "+v"(tv[4]), "+v"(tv[5]),
                                   "+v"(tv[6]), "+v"(tv[7]), "+v"(tv[8]));
                    double to[3] = {tv[0], tv[1], tv[2]};
                    double td[3] = {tv[3], tv[4], tv[5]};
                    double dL = tv[6], dlogI = tv[7];
                    double Ndo = N.x * to[0] + N.y * to[1] + N.z * to[2];
                    double Ndd = N.x * td[0] + N.y * td[1] + N.z * td[2];
                    double dtt = -(Ndo + (double)t * Ndd) / Nd;
                    double dp[3] = {to[0] + td[0] * t + (double)d.x * dtt, to[1] + td[1] * t + (double)d.y * dtt,
                                    to[2] + td[2] * t + (double)d.z * dtt};
                    double dl = ((double)dist3.x * (dp[0] - to[0]) + (double)dist3.y * (dp[1] - to[1]) +
                                 (double)dist3.z * (dp[2] - to[2])) /
                                (double)l;
                    dL += dl;
                    dlogI += ln_air * dl;
                    double pd = ((double)d.x * td[0] + (double)d.y * td[1] + (double)d.z * td[2]) / dn;
                    dprev[q][0] = (td[0] - (double)d.x / dn * pd) / dn;
                    dprev[q][1] = (td[1] - (double)d.y / dn * pd) / dn;
                    dprev[q][2] = (td[2] - (double)d.z / dn * pd) / dn;
                    dtan[q][0] = (float)dp[0];
                    dtan[q][1] = (float)dp[1];
                    dtan[q][2] = (float)dp[2];
                    dtan[q][3] = (float)td[0];  // incoming direction tangent, replaced below
                    dtan[q][4] = (float)td[1];
                    dtan[q][5] = (float)td[2];
                    dtan[q][6] = (float)dL;
                    dtan[q][7] = (float)dlogI;
                    drefl[q] = tv[8] + ((uint32_t)q == mat ? 1.0f / mb.z : 0.0f);
                }
                if (is_normal(I)) {
                    for (uint32_t r = 0; r < P.n_rec; ++r) {
                        const RecParams& R = P.rec[r];
                        V3 dv = sub(V3{R.px, R.py, R.pz}, p);
                        V3 lsdir = normalized(dv);
                        float dtd = dot(lsdir, nrm);
                        if (!(dtd > 0.0f)) continue;
                        V3 rv{0, 0, 0};
                        float diff, sf;
                        if (bt == kReflect) {
                            rv = reflect(prev, nrm);
                            diff = -dot(nrm, prev);
                            sf = fmaxf(0.0f, dot(rv, lsdir));
                        } else {
                            diff = dot(nrm, prev);
                            sf = fmaxf(0.0f, dot(prev, lsdir));
                        }
                        float pw = powf_ear(sf, kExp);
                        float factor = spec * kExpInt * pw + (1.0f - spec) * diff;
                        float c = I;
                        c *= factor;
                        float ls = length(dv);
                        float geo_air = powf_ear_l2(P.air[band], P.l2_air[band], ls);
                        float geo_inv = 2.0f / (4.0f * kPi * ls * ls);
                        c *= geo_air;
                        c *= geo_inv;
                        if (!is_normal(c)) continue;
                        if (k & 1u) c *= -1.0f;
                        float bt_ = 0.0f;
                        int bs_ = -1;
                        uint32_t bo_ = 0;
                        Traversal T = make_trav(In, gstack, gthreads);
                        if (traverse<kLdsMin, kBlock, WIDTH, true, false>(T, p, dv, bt_, bs_, bo_, lds + threadIdx.x,
                                                                          gtid, nvis, ntri))
                            continue;
                        double a_c = contribution_adjoint(P, A, band, R, lsdir, c, (L + ls) / 343.0f, L + ls);
                        if (a_c == 0.0) continue;
                        const double cnof = ((k & 1u) ? -1.0 : 1.0) * (double)I * (double)geo_air * (double)geo_inv;
                        const double lobe = (double)kExpInt * (double)pw;
                        for (uint32_t q = 0; q < nm; ++q) {
                            double dvv[3] = {-(double)dtan[q][0], -(double)dtan[q][1], -(double)dtan[q][2]};
                            double dls = (dvv[0] * dv.x + dvv[1] * dv.y + dvv[2] * dv.z) / (double)ls;
                            double ld = lsdir.x * dvv[0] + lsdir.y * dvv[1] + lsdir.z * dvv[2];
                            double dld[3] = {(dvv[0] - lsdir.x * ld) / ls, (dvv[1] - lsdir.y * ld) / ls,
                                             (dvv[2] - lsdir.z * ld) / ls};
                            double pn = dprev[q][0] * nrm.x + dprev[q][1] * nrm.y + dprev[q][2] * nrm.z;
                            double ddiff, dsf = 0.0;
                            if (bt == kReflect) {
                                ddiff = -pn;
                                if (sf > 0.0f) {
                                    double drv[3] = {dprev[q][0] - 2.0 * pn * nrm.x, dprev[q][1] - 2.0 * pn * nrm.y,
                                                     dprev[q][2] - 2.0 * pn * nrm.z};
                                    dsf = drv[0] * lsdir.x + drv[1] * lsdir.y + drv[2] * lsdir.z + dld[0] * rv.x +
                                          dld[1] * rv.y + dld[2] * rv.z;
                                }
                            } else {
                                ddiff = pn;
                                if (sf > 0.0f)
                                    dsf = dprev[q][0] * lsdir.x + dprev[q][1] * lsdir.y + dprev[q][2] * lsdir.z +
                                          dld[0] * prev.x + dld[1] * prev.y + dld[2] * prev.z;
                            }
                            double dlobe = sf > 0.0f ? (double)kExpInt * 1000.0 * pow((double)sf, 999.0) * dsf : 0.0;
                            double dfactor = (double)spec * dlobe + (1.0 - (double)spec) * ddiff;
                            if (q == mat) dfactor += lobe - (double)diff;
                            double dgeo = ln_air * dls - 2.0 * dls / (double)ls;
                            double dc = cnof * dfactor + (double)c * ((double)dtan[q][7] + dgeo);
                            g_spec[q * kBlock] += a_c * dc;
                            g_refl[q * kBlock] += a_c * (double)c * (double)drefl[q];
                        }
                    }
                    cont = !((double)I < P.cutoff) && k < P.max_bounces;
                }
                if (cont) {
                    // hemisphere sample and blend exactly as k_shade does
                    V3 hs = sample_hemi(rng, nrm);
                    V3 rdir = bt == kRefract ? d : reflect(d, nrm);
                    float gg = 1.0f - spec;
                    V3 w{hs.x * gg + rdir.x * spec, hs.y * gg + rdir.y * spec, hs.z * gg + rdir.z * spec};
                    float wl = length(w);
                    V3 v = normalized(w);
                    const bool local = (P.flags & EAR_FLAG_ADJ_LOCAL) != 0;
                    for (uint32_t q = 0; q < nm; ++q) {
                        if (local) {
                            for (int f = 0; f < 8; ++f) dtan[q][f] = 0.0f;
                            continue;
                        }
                        double td[3] = {dtan[q][3], dtan[q][4], dtan[q][5]};
                        double dr[3];
                        if (bt == kRefract) {
                            dr[0] = td[0];
                            dr[1] = td[1];
                            dr[2] = td[2];
                        } else {
                            double tn = td[0] * nrm.x + td[1] * nrm.y + td[2] * nrm.z;
                            dr[0] = td[0] - 2.0 * tn * nrm.x;
                            dr[1] = td[1] - 2.0 * tn * nrm.y;
                            dr[2] = td[2] - 2.0 * tn * nrm.z;
                        }
                        double dw[3] = {dr[0] * spec, dr[1] * spec, dr[2] * spec};
                        if (q == mat) {
                            dw[0] += (double)rdir.x - (double)hs.x;
                            dw[1] += (double)rdir.y - (double)hs.y;
                            dw[2] += (double)rdir.z - (double)hs.z;
                        }
                        double vdw = v.x * dw[0] + v.y * dw[1] + v.z * dw[2];
                        dtan[q][3] = (float)((dw[0] - v.x * vdw) / wl);
                        dtan[q][4] = (float)((dw[1] - v.y * vdw) / wl);
                        dtan[q][5] = (float)((dw[2] - v.z * vdw) / wl);
                    }
                    no = make_float4(p.x, p.y, p.z, I);
                    nd = make_float4(v.x, v.y, v.z, L);
                    nmeta = make_uint4(rm.x, rng.draw, (uint32_t)band | (k << 8), id);
                }
            }
        }
        if (BATCH) {
            // reduce the step's partials per instance present in the wave
            const uint32_t nmx = adj[my_id].n_mat;
            uint64_t todo = __ballot(i < n);
            while (todo) {
                const int leader = __ffsll((unsigned long long)todo) - 1;
                const uint32_t key = __shfl(my_id, leader);
                const int kband = __shfl(band_acc, leader);
                const bool mine = i < n && my_id == key;
                const uint32_t nmk = __shfl(nmx, leader);
                for (uint32_t q = 0; q < nmk; ++q) {
                    const double sr = wave_sum_d(mine ? g_refl[q * kBlock] : 0.0);
                    const double ss = wave_sum_d(mine ? g_spec[q * kBlock] : 0.0);
                    if (lane_id() == 0) {
                        double* gk = adj[key].grad_copy();
                        if (sr != 0.0) atomicAdd(gk + ((size_t)kband * 2 + 0) * nmk + q, sr);
                        if (ss != 0.0) atomicAdd(gk + ((size_t)kband * 2 + 1) * nmk + q, ss);
                    }
                }
                todo &= ~__ballot(mine);
            }
            for (int q = 0; q < kAdMaxMat; ++q) g_refl[q * kBlock] = g_spec[q * kBlock] = 0.0;
        }
        uint32_t slot = wave_append(n_out, cont);
        if (cont) {
            qout.o[slot] = no;
            qout.d[slot] = nd;
            qout.m[slot] = nmeta;
            for (uint32_t q = 0; q < nm; ++q) {
                for (int f = 0; f < 8; ++f) tout.f(q, f, slot) = dtan[q][f];
                tout.refl(q, slot) = drefl[q];
            }
        }
        n_done += i < n ? 1u : 0u;
    }
    stat_add(stats, ST_SEGMENTS, n_done);
    if (BATCH) return;
    __shared__ double red[kBlock / 64][2 * kAdMaxMat];
    double r_refl[kAdMaxMat], r_spec[kAdMaxMat];
#pragma unroll
    for (int q = 0; q < kAdMaxMat; ++q) {
        r_refl[q] = g_refl[q * kBlock];
        r_spec[q] = g_spec[q * kBlock];
    }
    block_grad_flush(A0, band_acc, r_refl, r_spec, &red[0][0]);
}

// a vertex of the score form spawns a continuation with probability
// min(1, kScoreRate F), F its rim flux (the rim term's weight: the least
// variance for a given number of continuations)
constexpr float kScoreRate = 0.05f;
constexpr int kAdjLds = 8;  // k_adj_paths' LDS entries of a traversal stack

__device__ __forceinline__ void add_grad(double* p, double v) {
    if (v != 0.0) __hip_atomic_fetch_add((__attribute__((address_space(1))) double*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The adjoint with EAR_FLAG_ADJ_LOCAL (or EAR_FLAG_ADJ_SCORE) for every ray:
// no direction or position tangents travel between vertices, so a ray
// carries only dlogI/drefl (n_mat floats) and, in the score form, S (n_mat
// floats).  At each visible connection of a hit on material m,
// d c / d spec_m = sign I air^l 2 / (4 pi l^2) (lobe - diffuse) and
// d c / d refl_q = c dlogI/drefl_q; the score form adds c S_q to d c / dspec_q;
// times dL/dc they join the lane's sums, which go to the gradient of their
// instance and band when the lane moves to another or ends.  Same primal and
// draws as k_shade; the sums are indexed at compile time only.
//
// SCORE: after its connections, a vertex whose path goes on adds to S_m
// (m its material) d log p(v)/ds - F for the direction v it drew, and with
// probability q = min(1, kScoreRate F) a continuation leaves the vertex along
// a rim direction (score_rim_dir) with weight -F / q on spec_m, F / q being
// added to S_m.  A continuation replays transport only: no refl tangents, no
// explicit lobe term, no score, no spawns.  The lane follows it to its end at
// once and then takes its main path up again, so it needs no queue.
//
// One launch carries the rays of every band to their ends, as k_tail does (a
// wave's lanes go through one segment together and refill).  A bounce at a
// time through queues, with a request of 16 weights per connection, a pair of
// tangent arrays and the continuations' own queues, launches of some 100 us
// each for a few rays and each band by itself made the 1M-ray box 129 ms and 8
// rooms 117 ms; here 69 and 77.  Bound by the vector units at the occupancy
// that the registers allow: with every array in registers (206 to 225 of
// them, two waves a SIMD) the box took 86, so the path's two arrays, indexed
// by material anyway, and a waiting main path are in LDS, which half the usual
// stack makes room for (168 registers, three waves; four waves spill: 100).
template <int WIDTH, bool BATCH, bool SCORE>
__global__ void __launch_bounds__(kBlock, 3) k_adj_paths(const InstDev* __restrict__ inst, int* gstack,
                                                         uint32_t gthreads, Queue q, const uint32_t* __restrict__ n_q,
                                                         uint32_t max_rec, AdjArgs A0,
                                                         const AdjArgs* __restrict__ adj, Fetch fetch) {
    constexpr int LDS = kAdjLds;
    __shared__ int lds[LDS * kBlock];
    __shared__ HemiLds hl[kBlock / 64];
    __shared__ float4 mo[kBlock], md[kBlock];  // a continuation's main path
    __shared__ uint4 mm[kBlock];
    const uint32_t n = *n_q;
    const uint32_t gtid = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t waves = gridDim.x * (kBlock / 64);
    uint32_t nvis = 0, ntri = 0;
    Claim claim(n, gtid, gridDim.x * kBlock, fetch, min(64u, max(kTailMin, n / waves + (n % waves ? 1u : 0u))));
    double g_refl[kAdMaxMat], g_spec[kAdMaxMat];
    __shared__ float drefl_s[kAdMaxMat * kBlock], sacc_s[kAdMaxMat * kBlock];
    float* drefl = drefl_s + threadIdx.x;
    float* sacc = sacc_s + threadIdx.x;
#pragma unroll
    for (int m = 0; m < kAdMaxMat; ++m) {
        g_refl[m] = g_spec[m] = 0.0;
        drefl[m * kBlock] = sacc[m * kBlock] = 0.0f;
    }
    uint32_t key = 0xFFFFFFFFu;  // instance and band of the sums
    int kband = 0;
    bool live = false, contn = false;  // on a path; on a continuation
    float4 ro{}, rd{};                 // the path's state
    uint4 rm{};
    uint32_t id = 0, cmat = 0, kspawn = 0;  // a continuation's material and vertex
    float wcont = 0.0f;                     // and weight
    for (;;) {
        const uint64_t idle = __ballot(!live);
        if (idle && !claim.exhausted()) {
            const uint32_t mine = claim.take(fetch, idle, lane);
            if (mine != 0xFFFFFFFFu) {
                ro = q.o[mine];
                rd = q.d[mine];
                rm = q.m[mine];
                id = BATCH ? rm.w : 0u;
                const int b = (int)(rm.z & 0xFFu);
                if (key != 0xFFFFFFFFu && (key != id || kband != b)) {
                    const AdjArgs& A = BATCH ? adj[key] : A0;
                    double* gk = A.grad_copy() + (size_t)kband * 2 * A.n_mat;
#pragma unroll
                    for (int m = 0; m < kAdMaxMat; ++m) {
                        if ((uint32_t)m < A.n_mat) {
                            add_grad(gk + m, g_refl[m]);
                            add_grad(gk + A.n_mat + m, g_spec[m]);
                        }
                        g_refl[m] = g_spec[m] = 0.0;
                    }
                }
                key = id;
                kband = b;
#pragma unroll
                for (int m = 0; m < kAdMaxMat; ++m) drefl[m * kBlock] = sacc[m * kBlock] = 0.0f;
                live = true;
                contn = false;
            }
        }
        if (__ballot(live) == 0) break;
        const InstDev& In = inst[id];
        const RenderParams& P = In.P;
        const AdjArgs& A = BATCH ? adj[id] : A0;
        const Traversal T = make_trav(In, gstack, gthreads);
        const int band = (int)(rm.z & 0xFFu);
        const uint32_t k = ((rm.z >> 8) & 0xFFFFu) + 1;
        int2 h = make_int2(0, -1);
        {
            Walker<LDS, kBlock, WIDTH, false, false> w(lds + threadIdx.x, gstack, gtid, gthreads);
            if (live) w.start(T, V3{ro.x, ro.y, ro.z}, V3{rd.x, rd.y, rd.z}, 1000000.0f);
            while (__ballot(!w.idle())) w.step(T, nvis, ntri);
            h = make_int2(__float_as_int(w.best_t), w.best_s);
        }
        Rng rng;
        V3 p{0, 0, 0}, nrm{0, 0, 0};
        float I = 0.0f, L = 0.0f, spec = 0.0f;
        uint32_t mat = 0;
        int bt = kReflect;
        bool alive = false, cont = false;
        if (live && h.y >= 0) {
            const float t = __int_as_float(h.x);
            const V3 o{ro.x, ro.y, ro.z};
            const V3 d{rd.x, rd.y, rd.z};
            p = V3{o.x + d.x * t, o.y + d.y * t, o.z + d.z * t};
            const float4 nmv = ldg(In.nm + h.y);
            const V3 N{nmv.x, nmv.y, nmv.z};
            nrm = dot(N, d) > 0.0f ? V3{N.x * -1.0f, N.y * -1.0f, N.z * -1.0f} : N;
            mat = __float_as_uint(nmv.w);
            const float4 mb = ldg(In.mat_band + 3 * mat + band);
            if (SCORE && contn)
                score_rng_init(rng, P.seed, rm.x, P.ctx_word[band], P.instance, kspawn, rm.y);
            else
                rng.init(P.seed, rm.x, P.ctx_word[band], P.instance, rm.y);
            if (mb.x >= 0.0f) bt = (rng.next() <= mb.x) ? kReflect : kRefract;
            spec = mb.y;
            if (bt == kRefract) nrm = neg(nrm);
            const float l = length(sub(p, o));
            I = ro.w;
            I *= powf_ear_l2(P.air[band], P.l2_air[band], l);
            L = rd.w + l;
            I *= mb.z;
            if (!contn) drefl[mat * kBlock] += 1.0f / mb.z;
            alive = is_normal(I);
            if (alive) cont = !((double)I < P.cutoff) && k < P.max_bounces;
        }
        // connections to every recorder (src/Scene.cpp:185-268), then the
        // segment to it (Scene::Connect, src/Scene.cpp:84-96)
        for (uint32_t r = 0; r < max_rec; ++r) {
            const RecParams& R = P.rec[r];
            const V3 dv = sub(V3{R.px, R.py, R.pz}, p);
            bool emit = false;
            float ds = 0.0f, ac = 0.0f;
            if (alive && r < P.n_rec) {
                const V3 lsdir = normalized(dv);
                const V3 prev = normalized(V3{rd.x, rd.y, rd.z});
                if (dot(lsdir, nrm) > 0.0f) {
                    float diff, sf;
                    if (bt == kReflect) {
                        const V3 rv = reflect(prev, nrm);
                        diff = -dot(nrm, prev);
                        sf = fmaxf(0.0f, dot(rv, lsdir));
                    } else {
                        diff = dot(nrm, prev);
                        sf = fmaxf(0.0f, dot(prev, lsdir));
                    }
                    const float pw = powf_ear(sf, kExp);
                    const float factor = spec * kExpInt * pw + (1.0f - spec) * diff;
                    float c = I;
                    c *= factor;
                    const float ls = length(dv);
                    const float geo_air = powf_ear_l2(P.air[band], P.l2_air[band], ls);
                    const float geo_inv = 2.0f / (4.0f * kPi * ls * ls);
                    c *= geo_air;
                    c *= geo_inv;
                    if (is_normal(c)) {
                        if (k & 1u) c *= -1.0f;
                        const double a_c = contribution_adjoint(P, A, band, R, lsdir, c, (L + ls) / 343.0f, L + ls);
                        if (a_c != 0.0) {
                            const double cnof =
                                ((k & 1u) ? -1.0 : 1.0) * (double)I * (double)geo_air * (double)geo_inv;
                            ds = (float)(a_c * cnof * ((double)kExpInt * (double)pw - (double)diff));
                            ac = (float)(a_c * (double)c);
                            emit = true;
                        }
                    }
                }
            }
            Walker<LDS, kBlock, WIDTH, true, false> w(lds + threadIdx.x, gstack, gtid, gthreads);
            if (emit) w.start(T, p, dv, 0.0f);
            while (__ballot(!w.idle())) w.step(T, nvis, ntri);
            if (emit && !w.found()) {
                if (!contn) {
#pragma unroll
                    for (int m = 0; m < kAdMaxMat; ++m) {
                        g_refl[m] += (double)(ac * drefl[m * kBlock]);
                        g_spec[m] += (double)(ac * sacc[m * kBlock] + ((uint32_t)m == mat ? ds : 0.0f));
                    }
                } else {
                    const double v = (double)(ac * wcont);
#pragma unroll
                    for (int m = 0; m < kAdMaxMat; ++m)
                        if ((uint32_t)m == cmat) g_spec[m] += v;
                }
            }
        }
        const V3 hv = sample_hemi_wave(cont, true, rng, nrm, hl[threadIdx.x >> 6]);
        if (cont) {
            const V3 d{rd.x, rd.y, rd.z};
            const V3 rdir = bt == kRefract ? d : reflect(d, nrm);
            const V3 vdir = blend_spec(hv, rdir, spec);
            const uint4 next = make_uint4(rm.x, rng.draw, (uint32_t)band | (k << 8), id);
            ro = make_float4(p.x, p.y, p.z, I);
            rd = make_float4(vdir.x, vdir.y, vdir.z, L);
            if (SCORE && !contn) {
                // the direction just drawn leaves this vertex: its score, the
                // rim flux and perhaps a continuation (after this vertex's
                // connections, which that direction does not reach)
                const double cdir = (double)vdir.x * (double)rdir.x + (double)vdir.y * (double)rdir.y +
                                    (double)vdir.z * (double)rdir.z;
                const double cr = (double)rdir.x * (double)nrm.x + (double)rdir.y * (double)nrm.y +
                                  (double)rdir.z * (double)nrm.z;
                const double F = score_flux(cr, (double)spec);
                double coef = score_dlogp(cdir, (double)spec) - F;
                Rng rs;
                score_rng_init(rs, P.seed, rm.x, P.ctx_word[band], P.instance, k, 0u);
                const float qk = fminf(1.0f, (float)(F * (double)kScoreRate));
                rm = next;
                if (rs.next() < qk) {
                    const V3 vb = score_rim_dir(rs, nrm, rdir, spec);
                    const double wgt = F / (double)qk;
                    coef += wgt;
                    wcont = (float)(-wgt);
                    cmat = mat;
                    kspawn = k;
                    contn = true;
                    mo[threadIdx.x] = ro;  // the main path waits
                    md[threadIdx.x] = rd;
                    mm[threadIdx.x] = rm;
                    rd = make_float4(vb.x, vb.y, vb.z, L);
                    rm.y = rs.draw;
                }
                sacc[mat * kBlock] += (float)coef;
            } else {
                rm = next;
            }
        } else if (SCORE && contn) {
            ro = mo[threadIdx.x];
            rd = md[threadIdx.x];
            rm = mm[threadIdx.x];
            contn = false;
        } else {
            live = false;
        }
    }
    // what is left, summed over the lanes of the wave that hold the same
    // instance and band
    uint64_t todo = __ballot(key != 0xFFFFFFFFu);
    while (todo) {
        const int leader = __ffsll((unsigned long long)todo) - 1;
        const uint32_t lk = __shfl(key, leader);
        const int lb = __shfl(kband, leader);
        const bool mine = key == lk && kband == lb;
        const AdjArgs& A = BATCH ? adj[lk] : A0;
        double* gk = A.grad_copy() + (size_t)lb * 2 * A.n_mat;
#pragma unroll
        for (int m = 0; m < kAdMaxMat; ++m) {
            if ((uint32_t)m >= A.n_mat) break;
            const double sr = wave_sum_d(mine ? g_refl[m] : 0.0);
            const double ss = wave_sum_d(mine ? g_spec[m] : 0.0);
            if (lane == 0) {
                add_grad(gk + m, sr);
                add_grad(gk + A.n_mat + m, ss);
            }
        }
        todo &= ~__ballot(mine);
    }
}

__global__ void k_zero_f32(float* p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

}  // namespace

// Gradient of sum(adj_value * value) + sum(adj_abs * abs_value) with respect
// to refl and spec of every material, for each band of the mask, for every
// item of a batch.  The bands are replayed one after another (the tangent
// arrays and the per-wave partials belong to one band at a time); within a
// band the rays of all items share the queues, in chunks of the ray chunk.
ear_status run_backward_batch(Ctx* c, uint32_t n_items, DeviceScene* const* scenes,
                              const ear_render_desc* const* descs, const double* const* adj_value,
                              const double* const* adj_abs, double* const* grad_refl, double* const* grad_spec) {
    if (n_items == 0) return EAR_ERR_INVALID_ARGUMENT;
    const bool batch = n_items > 1;
    const int width = (int)scenes[0]->width;
    std::vector<InstDev> inst(n_items);
    uint32_t nm_max = 0, max_rec = 0, max_bounces = 0;
    size_t adj_cells = 0;
    std::vector<size_t> adj_off(n_items);
    for (uint32_t i = 0; i < n_items; ++i) {
        const DeviceScene* s = scenes[i];
        const ear_render_desc* D = descs[i];
        if (!s || !D) return EAR_ERR_INVALID_ARGUMENT;
        if ((int)s->width != width) {
            c->last_error = "all scenes of a batch must have the same BVH width";
            return EAR_ERR_INVALID_ARGUMENT;
        }
        InstDev& I = inst[i];
        std::memset(&I, 0, sizeof(I));
        TRY(make_params(c, D, &I.P));
        if (D->source.kind != EAR_SRC_POINT) {
            c->last_error = "the adjoint supports point sources";
            return EAR_ERR_INVALID_ARGUMENT;
        }
        if (s->n_mat > (uint32_t)kAdMaxMat || s->n_mat == 0) {
            c->last_error = "the adjoint supports 1..8 materials";
            return EAR_ERR_CAPACITY;
        }
        if (!adj_value[i] && !adj_abs[i]) {
            c->last_error = "no adjoint given";
            return EAR_ERR_INVALID_ARGUMENT;
        }
        if ((D->flags & EAR_FLAG_ADJ_SCORE) && (D->flags & EAR_FLAG_ADJ_LOCAL)) {
            c->last_error = "EAR_FLAG_ADJ_SCORE and EAR_FLAG_ADJ_LOCAL exclude each other";
            return EAR_ERR_INVALID_ARGUMENT;
        }
        if (D->flags & EAR_FLAG_ADJ_SCORE) {
            // the blend's direction map is one-to-one only below 1/2
            for (uint32_t m = 0; m < s->n_mat; ++m)
                for (uint32_t b = 0; b < 3; ++b)
                    if (((D->band_mask >> b) & 1u) && !(s->mat_band_host[3 * m + b].y < 0.5f)) {
                        c->last_error = "EAR_FLAG_ADJ_SCORE needs every specularity below 0.5";
                        return EAR_ERR_INVALID_ARGUMENT;
                    }
        }
        I.nodes = s->nodes;
        I.nodes4 = s->nodes4;
        I.tris = s->tris;
        I.nm = s->nm;
        I.mat_band = s->mat_band;
        I.n_tris = s->n_tris;
        nm_max = std::max(nm_max, s->n_mat);
        max_rec = std::max(max_rec, I.P.n_rec);
        max_bounces = std::max(max_bounces, D->max_bounces);
        adj_off[i] = adj_cells;
        adj_cells += (size_t)3 * I.P.n_channels * I.P.n_bins;
    }
    // value = raw * (1/N) * gain^2 (k_finalize), so dL/draw = dL/dvalue * (1/N) * gain^2;
    // each row is then turned into prefix sums (ramp_adjoint)
    std::vector<double> as(adj_cells, 0.0), aa(adj_cells, 0.0);
    bool any_s = false, any_a = false;
    for (uint32_t i = 0; i < n_items; ++i) {
        const ear_render_desc* D = descs[i];
        const double scale = (double)(1.0f / (float)std::max<uint32_t>(1, D->n_rays)) *
                             (double)(D->source.gain * D->source.gain);
        const size_t hn = (size_t)3 * inst[i].P.n_channels * inst[i].P.n_bins;
        if (adj_value[i]) {
            any_s = true;
            for (size_t k = 0; k < hn; ++k) as[adj_off[i] + k] = adj_value[i][k] * scale;
        }
        if (adj_abs[i]) {
            any_a = true;
            for (size_t k = 0; k < hn; ++k) aa[adj_off[i] + k] = adj_abs[i][k] * scale;
        }
    }
    const ear_tuning& tu = c->tuning;
    const uint32_t chunk = tu.ray_chunk ? tu.ray_chunk : (1u << 23);
    uint32_t n_local = 0, n_score = 0;
    for (uint32_t i = 0; i < n_items; ++i) {
        n_local += (inst[i].P.flags & EAR_FLAG_ADJ_LOCAL) ? 1u : 0u;
        n_score += (inst[i].P.flags & EAR_FLAG_ADJ_SCORE) ? 1u : 0u;
    }
    if (n_score != 0 && n_score != n_items) {
        c->last_error = "a batch mixes EAR_FLAG_ADJ_SCORE items with others";
        return EAR_ERR_INVALID_ARGUMENT;
    }
    const bool all_score = n_score == n_items;
    const bool all_local = all_score || n_local == n_items;  // one launch per chunk of rays (k_adj_paths)
    // the queue holds a chunk of the rays of one band, or of all of them
    uint64_t rays_band_max = 0, rays_all = 0;
    for (int b = 0; b < 3; ++b) {
        uint64_t t = 0;
        for (uint32_t i = 0; i < n_items; ++i)
            if ((inst[i].P.band_mask >> b) & 1u) t += descs[i]->n_rays;
        rays_band_max = std::max(rays_band_max, t);
        rays_all += t;
    }
    const uint32_t cap =
        (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(chunk, all_local ? rays_all : rays_band_max));
    hipStream_t st = c->stream;
    DevBuf qo[2] = {DevBuf(c), DevBuf(c)}, qd[2] = {DevBuf(c), DevBuf(c)}, qm[2] = {DevBuf(c), DevBuf(c)};
    DevBuf tt[2] = {DevBuf(c), DevBuf(c)}, tr[2] = {DevBuf(c), DevBuf(c)};
    DevBuf hits(c), counters(c), stats(c), gs(c), dinst(c), dsegs(c), dsegoff(c), dplan(c), dadj_s(c), dadj_a(c),
        dgrad(c), dargs(c), sqp(c), sqm(c);
    for (int k = 0; k < (all_local ? 1 : 2); ++k) {
        TRY(qo[k].alloc((size_t)cap * 16));
        TRY(qd[k].alloc((size_t)cap * 16));
        TRY(qm[k].alloc((size_t)cap * 16));
        if (all_local) continue;
        TRY(tt[k].alloc((size_t)cap * nm_max * 8 * 4));
        TRY(tr[k].alloc((size_t)cap * nm_max * 4));
    }
    TRY(counters.alloc(32));
    TRY(stats.alloc(ST_N * 8 * kStatCopies));
    TRY(sqp.alloc(16));
    TRY(sqm.alloc(16));
    if (!all_local) TRY(hits.alloc((size_t)cap * 8));
    // static closest-hit traversal by default (the replayed bands run one
    // at a time, with fewer rays in flight than the forward's, where the
    // refill bookkeeping does not pay); the refilling one on request
    const bool fetch_e = tu.traversal == EAR_TRAVERSAL_FETCH || tu.traversal == EAR_TRAVERSAL_FETCH_ALL;
    ExtendFn fe;
    ShadowFn fs_unused;
    const TravCfg cfg{256, 16, width, false, batch, fetch_e, false};
    pick_kernels(cfg, &fe, &fs_unused);
    DevBuf segc(c);
    TRY(segc.alloc(kMaxSeg * kSegStride * 4));
    EAR_HIP_TRY(c, hipMemsetAsync(segc.p, 0, segc.n, st));
    const uint32_t nseg = tu.fetch_segments ? std::min<uint32_t>(tu.fetch_segments, kMaxSeg) : kSegDefault;
    const Fetch fq_e{segc.as<uint32_t>(), tu.refill ? tu.refill : 24u, tu.fetch_chunk, nseg};
    const uint32_t waves = tu.waves_per_cu ? tu.waves_per_cu : 32;
    const uint32_t cap_e = (uint32_t)c->num_cus * (uint32_t)std::max(1, resident_blocks((const void*)fe, 256));
    const uint32_t gmax = persistent_grid(c, 0xFFFFFFFFu, waves);
    // every thread of either traversal launch owns one overflow stack
    using PathsFn = void (*)(const InstDev*, int*, uint32_t, Queue, const uint32_t*, uint32_t, AdjArgs, const AdjArgs*, Fetch);
    const PathsFn paths = width == 4 ? (batch ? (all_score ? (PathsFn)k_adj_paths<4, true, true> : (PathsFn)k_adj_paths<4, true, false>)
                                              : (all_score ? (PathsFn)k_adj_paths<4, false, true> : (PathsFn)k_adj_paths<4, false, false>))
                                     : (batch ? (all_score ? (PathsFn)k_adj_paths<2, true, true> : (PathsFn)k_adj_paths<2, true, false>)
                                              : (all_score ? (PathsFn)k_adj_paths<2, false, true> : (PathsFn)k_adj_paths<2, false, false>));
    const uint32_t g_paths = (uint32_t)c->num_cus * (uint32_t)std::max(1, resident_blocks((const void*)paths, kBlock));
    const uint32_t gthreads = all_local ? g_paths * (uint32_t)kBlock : std::max(cap_e * 256u, gmax * (uint32_t)kBlock);
    TRY(gs.alloc((size_t)(kStackDepth - (all_local ? kAdjLds : kLdsMin)) * gthreads * 4));
    TRY(dinst.alloc(sizeof(InstDev) * n_items));
    TRY(dsegs.alloc(sizeof(GenSeg) * 3 * (size_t)n_items));
    TRY(dsegoff.alloc(4 * 3 * (size_t)n_items));
    TRY(dplan.alloc(12));
    const uint32_t grad_n = 3 * 2 * nm_max * n_items;  // one copy
    TRY(dgrad.alloc(sizeof(double) * (size_t)grad_n * kGradCopies));
    TRY(dargs.alloc(sizeof(AdjArgs) * n_items));
    // prefix sums of every row (bins + 1 pairs), accumulated in long double
    std::vector<size_t> pre_off(n_items);
    size_t pre_pairs = 0;
    for (uint32_t i = 0; i < n_items; ++i) {
        pre_off[i] = pre_pairs;
        pre_pairs += (size_t)3 * inst[i].P.n_channels * (inst[i].P.n_bins + 1);
    }
    auto prefix = [&](const std::vector<double>& a) {
        std::vector<double> pre(2 * pre_pairs, 0.0);
        for (uint32_t i = 0; i < n_items; ++i) {
            const uint32_t nb = inst[i].P.n_bins, rows = 3 * inst[i].P.n_channels;
            for (uint32_t r = 0; r < rows; ++r) {
                const double* src = a.data() + adj_off[i] + (size_t)r * nb;
                double* dst = pre.data() + 2 * (pre_off[i] + (size_t)r * (nb + 1));
                long double s1 = 0.0L, s2 = 0.0L;
                for (uint32_t b = 0; b <= nb; ++b) {
                    dst[2 * b] = (double)s1;
                    dst[2 * b + 1] = (double)s2;
                    if (b < nb) {
                        s1 += (long double)src[b];
                        s2 += (long double)b * (long double)src[b];
                    }
                }
            }
        }
        return pre;
    };
    if (any_s) {
        const std::vector<double> pre = prefix(as);
        TRY(dadj_s.alloc(pre.size() * 8));
        EAR_HIP_TRY(c, hipMemcpyAsync(dadj_s.p, pre.data(), pre.size() * 8, hipMemcpyHostToDevice, st));
        EAR_HIP_TRY(c, hipStreamSynchronize(st));  // pre leaves scope
    }
    if (any_a) {
        const std::vector<double> pre = prefix(aa);
        TRY(dadj_a.alloc(pre.size() * 8));
        EAR_HIP_TRY(c, hipMemcpyAsync(dadj_a.p, pre.data(), pre.size() * 8, hipMemcpyHostToDevice, st));
        EAR_HIP_TRY(c, hipStreamSynchronize(st));
    }
    std::vector<AdjArgs> args(n_items);
    for (uint32_t i = 0; i < n_items; ++i)
        args[i] = AdjArgs{adj_value[i] ? dadj_s.as<double2>() + pre_off[i] : nullptr,
                          adj_abs[i] ? dadj_a.as<double2>() + pre_off[i] : nullptr,
                          dgrad.as<double>() + (size_t)i * 3 * 2 * nm_max, scenes[i]->n_mat, grad_n};
    EAR_HIP_TRY(c, hipMemcpyAsync(dargs.p, args.data(), sizeof(AdjArgs) * n_items, hipMemcpyHostToDevice, st));
    EAR_HIP_TRY(c, hipMemcpyAsync(dinst.p, inst.data(), sizeof(InstDev) * n_items, hipMemcpyHostToDevice, st));
    EAR_HIP_TRY(c, hipMemsetAsync(dgrad.p, 0, dgrad.n, st));
    EAR_HIP_TRY(c, hipMemsetAsync(counters.p, 0, counters.n, st));
    EAR_HIP_TRY(c, hipMemsetAsync(stats.p, 0, stats.n, st));
    const InstDev* di = dinst.as<InstDev>();
    uint32_t* cnt = counters.as<uint32_t>();
    unsigned long long* stp = stats.as<unsigned long long>();
    uint32_t pinned[4];
    Queue q[2] = {Queue{qo[0].as<float4>(), qd[0].as<float4>(), qm[0].as<uint4>()},
                  Queue{qo[1].as<float4>(), qd[1].as<float4>(), qm[1].as<uint4>()}};
    Tangents T[2] = {Tangents{tt[0].as<float>(), tr[0].as<float>(), cap},
                     Tangents{tt[1].as<float>(), tr[1].as<float>(), cap}};
    const ShadowQ SQ{sqp.as<float4>(), sqm.as<float4>()};
    const AdjArgs A0 = args[0];
    const AdjArgs* dA = dargs.as<AdjArgs>();
    if (all_local) {
        // every (instance, band) context is a run of rays (as many runs at a
        // time as 32-bit ray numbers reach over); a chunk of rays is emitted
        // and carried to its paths' ends at a time
        uint32_t dense = 1;
        std::vector<GenSeg> todo;
        for (uint32_t i = 0; i < n_items; ++i) {
            if (1.0 < inst[i].P.cutoff || inst[i].P.max_bounces == 0) dense = 0;
            for (uint32_t b = 0; b < 3; ++b)
                if (((inst[i].P.band_mask >> b) & 1u) && descs[i]->n_rays != 0)
                    todo.push_back(GenSeg{i, b, 0, descs[i]->n_rays});
        }
        for (size_t s0 = 0; s0 < todo.size();) {
            std::vector<uint32_t> off;
            uint64_t total = 0;
            size_t s1 = s0;
            for (; s1 < todo.size() && (s1 == s0 || total + todo[s1].count <= 0xFFFFFFFFull); ++s1) {
                off.push_back((uint32_t)total);
                total += todo[s1].count;
            }
            EAR_HIP_TRY(c, hipMemcpyAsync(dsegs.p, todo.data() + s0, sizeof(GenSeg) * (s1 - s0), hipMemcpyHostToDevice, st));
            EAR_HIP_TRY(c, hipMemcpyAsync(dsegoff.p, off.data(), 4 * off.size(), hipMemcpyHostToDevice, st));
            for (uint64_t r0 = 0; r0 < total; r0 += cap) {
                const uint32_t n_chunk = (uint32_t)std::min<uint64_t>(cap, total - r0);
                const uint32_t plan[3] = {(uint32_t)r0, n_chunk, 0u}, n_live = dense ? n_chunk : 0u;
                EAR_HIP_TRY(c, hipMemcpyAsync(dplan.p, plan, 12, hipMemcpyHostToDevice, st));
                EAR_HIP_TRY(c, hipMemcpyAsync(cnt, &n_live, 4, hipMemcpyHostToDevice, st));
                const uint32_t g = persistent_grid(c, n_chunk, waves);
                if (batch)
                    k_generate<true><<<g, kBlock, 0, st>>>(di, dsegs.as<GenSeg>(), dsegoff.as<uint32_t>(),
                                                           (uint32_t)off.size(), n_chunk, dplan.as<uint32_t>(), max_rec,
                                                           0u, dense, q[0], cnt, SQ, cnt + 2, stp);
                else
                    k_generate<false><<<g, kBlock, 0, st>>>(di, dsegs.as<GenSeg>(), dsegoff.as<uint32_t>(),
                                                            (uint32_t)off.size(), n_chunk, dplan.as<uint32_t>(), max_rec,
                                                            0u, dense, q[0], cnt, SQ, cnt + 2, stp);
                hipLaunchKernelGGL(paths, dim3(g_paths), dim3(kBlock), 0, st, di, gs.as<int>(), gthreads, q[0],
                                   (const uint32_t*)cnt, max_rec, A0, dA, fq_e);
                k_reset_iter<<<1, 64, 0, st>>>(cnt, 0u, segc.as<uint32_t>(), nseg);
                EAR_HIP_TRY(c, hipGetLastError());
                EAR_HIP_TRY(c, hipStreamSynchronize(st));  // plan, n_live and off leave scope
            }
            s0 = s1;
        }
    }
    for (uint32_t band = 0; !all_local && band < 3; ++band) {
        // this band's contexts as runs of rays
        std::vector<GenSeg> segs;
        std::vector<uint32_t> off;
        uint32_t total = 0;
        for (uint32_t i = 0; i < n_items; ++i) {
            if (!((inst[i].P.band_mask >> band) & 1u) || descs[i]->n_rays == 0) continue;
            segs.push_back(GenSeg{i, band, 0, descs[i]->n_rays});
            off.push_back(total);
            total += descs[i]->n_rays;
        }
        if (segs.empty()) continue;
        EAR_HIP_TRY(c, hipMemcpyAsync(dsegs.p, segs.data(), sizeof(GenSeg) * segs.size(), hipMemcpyHostToDevice, st));
        EAR_HIP_TRY(c, hipMemcpyAsync(dsegoff.p, off.data(), 4 * off.size(), hipMemcpyHostToDevice, st));
        for (uint32_t r0 = 0; r0 < total; r0 += cap) {
            const uint32_t n_chunk = std::min(cap, total - r0);
            const uint32_t plan[2] = {r0, n_chunk};
            EAR_HIP_TRY(c, hipMemcpyAsync(dplan.p, plan, 8, hipMemcpyHostToDevice, st));
            if (batch)
                k_generate<true><<<persistent_grid(c, n_chunk, waves), kBlock, 0, st>>>(
                    di, dsegs.as<GenSeg>(), dsegoff.as<uint32_t>(), (uint32_t)segs.size(), n_chunk,
                    dplan.as<uint32_t>(), max_rec, 0u, 0u, q[0], cnt + 0, SQ, cnt + 2, stp);
            else
                k_generate<false><<<persistent_grid(c, n_chunk, waves), kBlock, 0, st>>>(
                    di, dsegs.as<GenSeg>(), dsegoff.as<uint32_t>(), (uint32_t)segs.size(), n_chunk,
                    dplan.as<uint32_t>(), max_rec, 0u, 0u, q[0], cnt + 0, SQ, cnt + 2, stp);
            k_zero_f32<<<1024, 256, 0, st>>>(T[0].t, (size_t)cap * nm_max * 8);
            k_zero_f32<<<1024, 256, 0, st>>>(T[0].r, (size_t)cap * nm_max);
            EAR_HIP_TRY(c, hipMemcpyAsync(pinned, cnt, 12, hipMemcpyDeviceToHost, st));
            EAR_HIP_TRY(c, hipStreamSynchronize(st));
            uint32_t n_live = pinned[0];
            int cur = 0;
            // bounces in groups of 4 between looks at the queue count: the
            // kernels read their counts on the device, and a queue never grows
            // within a chunk, so grids sized at a group's start cover it
            uint32_t k = 1;
            while (k <= max_bounces && n_live > 0) {
              const uint32_t group = std::min<uint32_t>(4u, max_bounces - k + 1);
              // k_shade_ad walks inside: its grid stays within the overflow stacks' gmax
              const uint32_t gsd = persistent_grid(c, n_live, waves);
              const uint32_t ge = grid_for(n_live, cap_e, 256);
              for (uint32_t gi = 0; gi < group; ++gi, ++k) {
                {
                    hipLaunchKernelGGL(fe, dim3(ge), dim3(256), 0, st, di, gs.as<int>(), gthreads, q[cur],
                                       (const uint32_t*)(cnt + cur), hits.as<int2>(), stp, fq_e);
                    if (fetch_e) k_reset_iter<<<1, 64, 0, st>>>(cnt, 0u, segc.as<uint32_t>(), nseg);
#define EAR_AD_LAUNCH(W, B)                                                                                      \
    k_shade_ad<W, B><<<gsd, kBlock, 0, st>>>(di, gs.as<int>(), gthreads, q[cur], cnt + cur, hits.as<int2>(), \
                                             T[cur], q[1 - cur], cnt + (1 - cur), T[1 - cur], A0, dA, stp)
                    if (width == 4) {
                        if (batch)
                            EAR_AD_LAUNCH(4, true);
                        else
                            EAR_AD_LAUNCH(4, false);
                    } else {
                        if (batch)
                            EAR_AD_LAUNCH(2, true);
                        else
                            EAR_AD_LAUNCH(2, false);
                    }
#undef EAR_AD_LAUNCH
                    k_reset2<<<1, 64, 0, st>>>(cnt + cur, cnt + 2);
                }
                cur = 1 - cur;
              }
              EAR_HIP_TRY(c, hipMemcpyAsync(pinned, cnt, 12, hipMemcpyDeviceToHost, st));
              EAR_HIP_TRY(c, hipStreamSynchronize(st));
              n_live = pinned[cur];
            }
            k_reset2<<<1, 64, 0, st>>>(cnt + 0, cnt + 1);
            EAR_HIP_TRY(c, hipGetLastError());
        }
    }
    k_sum_grad_copies<<<std::min<uint32_t>((grad_n + 255) / 256, 1024), 256, 0, st>>>(dgrad.as<double>(), grad_n,
                                                                                      grad_n);
    EAR_HIP_TRY(c, hipGetLastError());
    std::vector<double> g(grad_n);
    EAR_HIP_TRY(c, hipMemcpyAsync(g.data(), dgrad.p, g.size() * 8, hipMemcpyDeviceToHost, st));
    EAR_HIP_TRY(c, hipStreamSynchronize(st));
    for (uint32_t i = 0; i < n_items; ++i) {
        const uint32_t nm = scenes[i]->n_mat;
        const double* gi = g.data() + (size_t)i * 3 * 2 * nm_max;
        for (uint32_t b = 0; b < 3; ++b) {
            if (!((inst[i].P.band_mask >> b) & 1u)) continue;
            for (uint32_t m = 0; m < nm; ++m) {
                if (grad_refl[i]) grad_refl[i][(size_t)m * 3 + b] = gi[((size_t)b * 2 + 0) * nm + m];
                if (grad_spec[i]) grad_spec[i][(size_t)m * 3 + b] = gi[((size_t)b * 2 + 1) * nm + m];
            }
        }
    }
    return EAR_OK;
}

ear_status run_backward(Ctx* c, DeviceScene* s, const ear_render_desc* D, const double* adj_value,
                        const double* adj_abs, double* grad_refl, double* grad_spec) {
    return run_backward_batch(c, 1, &s, &D, &adj_value, &adj_abs, &grad_refl, &grad_spec);
}

}  // namespace ear
