// Closest-hit tracing for batched worlds on CDNA4: depth / normal / object-ID images, ray queries, and the
// pose backward pass.
//
// The reference walks each ray alone with a private stack of 128 + 64 entries (src/mesh_dev.h:113-159),
// which on a 64-wide wavefront means 64 diverging walks and stacks spilled to scratch. Here a wavefront
// walks as a packet: it holds 64 rays of one world (an 8x8 pixel tile, or 64 consecutive rays of a
// query), fetches each node once for the whole wave through the scalar cache, and every lane tests the
// node's boxes with its own ray and its own closest distance so far. A child is entered when any lane's
// ray enters its box; the lanes that do not are masked out of it. The walk's stack is wave-uniform and
// lives one entry per lane of a vector register (written and read with writelane/readlane), so nothing
// spills. Each lane still finds exactly its own closest hit: a lane only tests triangles inside boxes its
// ray enters before its current closest distance, and keeps a hit only when strictly closer
// (mesh_dev.h:98), so the result equals the per-ray walk's except where two surfaces meet the ray at the
// same distance.
//
// What bounds these kernels is instruction issue, the scalar side of it first: a SIMD starts a scalar instruction or a
// branch every 4.4 cycles and a vector one every 2.4 (add, multiply, move) to 4 (minimum, compare, select, fused), all
// measured with 8 wavefronts, and the 4096-world 128x128 render issued 3.36 G scalar, 0.83 G branch and 5.66 G vector
// instructions in 8.44 ms: the scalar unit was busy nearly throughout. So the walks are written for few scalar
// instructions a visit: arguments read where they are used and the walk's pointers once, wave-uniform stacks in vector
// registers, masked instructions without a branch around them (NGX_LIKELY), lanes that drop out by their limit rather
// than by a mask, rare cases tested once for the wave. 8.44 -> 6.3 ms there, now at 4.3 G vector, 2.6 G scalar and 0.57 G
// branch instructions; 13.7 -> 12.5 ms for 67 M LiDAR rays.
#include <algorithm>
#include <cstddef>
#include <mutex>
#include <type_traits>
#include "ngx_kernels.h"

// Partial sums of ngx_pose_backward_depth_noalloc, which allocates nothing: NOALLOC_SCRATCH_FLOATS floats
// (32 MiB) that every GPU the library runs on holds until the process ends.
static __device__ __align__(256) float scratch[ngx::NOALLOC_SCRATCH_FLOATS];

namespace ngx {
namespace {

// A condition some lane of the wave almost always meets: the compiler then leaves out the branch it would otherwise put
// before the masked instructions, to skip them when no lane does.
#define NGX_LIKELY(x) __builtin_expect_with_probability((x), 1, 0.9999)
#define NGX_UNLIKELY(x) __builtin_expect_with_probability((x), 0, 0.9999)

struct LaneHit {
    int inst;
    int tri;
    float u, v;
};

// The kernel's arguments, read from their segment again wherever this is called: the empty asm statement keeps the
// compiler from seeing that it is the same address, so it loads a field where the field is used (through the scalar
// cache) rather than once at the start. A traversal kernel has more arguments than scalar registers to hold them across
// its walk, and one held all the same is kept in a lane of a vector register, which costs a vector instruction a read.
template <class T>
using KernelArgs = __attribute__((address_space(4))) const T;
template <class T>
__device__ __forceinline__ KernelArgs<T> &kernel_args() {
    auto *p = (KernelArgs<T> *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *p;
}
// A pointer to global memory, which the compiler cannot tell of one read from the arguments this way.
template <class T>
__device__ __forceinline__ T *in_global(T *p) { return (T *)(__attribute__((address_space(1))) T *)p; }

// The scene of the running kernel, whose arguments begin with a TraceScene.
// What every visit reads is held in registers for the walk.
struct Scene {
    const InstanceRec *inst_;
    const MeshRoot *mesh_roots_;
    const float *tris_;
    __device__ __forceinline__ Scene() {
        const auto &A = kernel_args<TraceScene>();
        inst_ = in_global(A.inst);
        mesh_roots_ = in_global(A.mesh_roots);
        tris_ = in_global(A.tris);
    }
    __device__ __forceinline__ const InstanceRec *inst() const { return inst_; }
    __device__ __forceinline__ const MeshRoot *mesh_roots() const { return mesh_roots_; }
    __device__ __forceinline__ const float *tris() const { return tris_; }
#define NGX_SCENE_POINTER(type, name) \
    __device__ __forceinline__ type *name() const { return in_global(kernel_args<TraceScene>().name); }
#define NGX_SCENE_VALUE(type, name) \
    __device__ __forceinline__ type name() const { return kernel_args<TraceScene>().name; }
    NGX_SCENE_POINTER(const WideNode, tlas_wide)
    NGX_SCENE_POINTER(const int, tlas_parent)
    NGX_SCENE_POINTER(const int, blas_parent)
    NGX_SCENE_POINTER(const int, blas_wide_node)
    NGX_SCENE_POINTER(const int, roots)
    NGX_SCENE_POINTER(const WideNode, blas_wide)
    NGX_SCENE_POINTER(const WideNode, blas_octants)
    NGX_SCENE_VALUE(int, octant_nodes)
    NGX_SCENE_POINTER(const float4, attrs)
    NGX_SCENE_POINTER(const float4, spheres)
    NGX_SCENE_POINTER(const SkipNode, skip)
    NGX_SCENE_POINTER(int, overflow)
    NGX_SCENE_VALUE(int, total)
    NGX_SCENE_VALUE(int, sphere_count)
    NGX_SCENE_VALUE(float, floor_y)
    NGX_SCENE_VALUE(float, floor_hx)
    NGX_SCENE_VALUE(float, floor_zmin)
    NGX_SCENE_VALUE(float, floor_zmax)
    NGX_SCENE_VALUE(int, pair_limit)
    NGX_SCENE_VALUE(int, lane_min_tris)
    NGX_SCENE_VALUE(int, share_cap)
#undef NGX_SCENE_POINTER
#undef NGX_SCENE_VALUE
};
static_assert(offsetof(RenderArgs, s) == 0 && offsetof(RgbArgs, r) == 0 && offsetof(RayArgs, s) == 0 &&
              offsetof(DepthBackwardArgs, s) == 0 && offsetof(RangeBackwardArgs, s) == 0, "every kernel's arguments begin with the scene");

// Traversal counters of one wavefront, wave-uniform. NoStats compiles them away; WaveStats is only used by the
// instrumented kernel built with NGX_TRACE_STATS.
enum StatIndex { ST_TLAS_NODES, ST_TLAS_LANES, ST_INSTANCES, ST_INSTANCE_LANES, ST_INSTANCE_ROOT_LANES, ST_BLAS_NODES,
                 ST_BLAS_LANES, ST_TRIANGLES, ST_TRIANGLE_LANES, ST_POPS, ST_VALID, ST_COUNT };
// The same type also says whether the walk is an occlusion test (kAnyHit): then a ray's limit drops below zero
// at its first hit, so its lane leaves every box after it and the walk ends as soon as every ray is blocked or
// done; whether a ray is blocked is all that is read (mesh_dev.h:208-227 stops at the first hit too).
// kHandoff says whether the hybrid walk may hand thin subtrees to the shared per-lane walk, and kTwoChild which shared
// per-lane walk runs: the one testing both children of a node a step, or the one-box-a-step walk of the skip layout, which
// needs fewer registers and is left for one-pass pictures of full wavefronts.
struct NoStats {
    static constexpr bool kAnyHit = false, kHandoff = true, kTwoChild = true, kOneOrigin = false;
    __device__ __forceinline__ void add(int, int) {}
};
// Camera rays: every ray of the wave starts at the camera, so what an instance makes of the origin is one point for the
// wave, held in scalar registers, and the view's tables may hold the top level about it.
struct ViewOfRays {
    const WideNode *nodes = nullptr;  // the view's copies of the top level (VIEW_OCTANTS times total), where `octants` says
    const float4 *inst = nullptr;     // the view's instances, or null
    int octants = VIEW_NO_OCTANTS;
};
struct CameraRays : ViewOfRays {
    static constexpr bool kAnyHit = false, kHandoff = true, kTwoChild = true, kOneOrigin = true;
    __device__ __forceinline__ void add(int, int) {}
};
struct OneBoxRays {
    static constexpr bool kAnyHit = false, kHandoff = false, kTwoChild = false, kOneOrigin = false;
    __device__ __forceinline__ void add(int, int) {}
};
// Shadow rays: the two-child walk, stopping each ray at its first hit. Whether a ray is blocked does not depend on the order
// in which boxes and triangles are tested.
struct Occlusion {
    static constexpr bool kAnyHit = true, kHandoff = true, kTwoChild = true, kOneOrigin = false;
    __device__ __forceinline__ void add(int, int) {}
};
#ifdef NGX_TRACE_STATS
struct WaveStats : ViewOfRays {
    static constexpr bool kAnyHit = false, kHandoff = true, kTwoChild = true, kOneOrigin = true;
    int c[ST_COUNT];
    __device__ __forceinline__ void add(const int k, const int v) { c[k] += v; }
};
#endif

struct Wide {
    float l_lo[3], l_hi[3], r_lo[3], r_hi[3];
    int left, right, lcount, rcount;
};

__device__ __forceinline__ Wide load_wide(const WideNode *nodes, const int index) {
    const float4 *p = reinterpret_cast<const float4 *>(nodes + index);
    const float4 f0 = sload4(p), f1 = sload4(p + 1), f2 = sload4(p + 2);
    const int4 f3 = sload4i(reinterpret_cast<const int4 *>(p + 3));
    Wide w;
    w.l_lo[0] = f0.x; w.r_lo[0] = f0.y; w.l_hi[0] = f0.z; w.r_hi[0] = f0.w;
    w.l_lo[1] = f1.x; w.r_lo[1] = f1.y; w.l_hi[1] = f1.z; w.r_hi[1] = f1.w;
    w.l_lo[2] = f2.x; w.r_lo[2] = f2.y; w.l_hi[2] = f2.z; w.r_hi[2] = f2.w;
    w.left = f3.x; w.right = f3.y; w.lcount = f3.z; w.rcount = f3.w;
    return w;
}

// ---------------------------------------------------------------- batched triangle tests --
//
// Below an instance the packet thins out: a leaf is typically reached by a handful of the wave's rays, so
// testing its triangles one after the other for the whole wave leaves most lanes idle. Instead a leaf
// reached by m rays adds m x count (ray, triangle) pairs to a table in LDS, and once 64 pairs are queued,
// or the instance is finished, every lane tests one pair. A ray's pairs are numbered in the order the walk
// met its triangles, and the ray keeps the closest hit, the lowest pair number among equal distances, with
// one 64-bit LDS minimum per pair (distance bits above pair number; distances are positive, so their bits
// order as the floats do). That is what testing the triangles one by one with a strict "closer than"
// keeps (mesh_dev.h:98, :186-199). A ray's limit is not lowered until its batch is tested, so a few
// more boxes may be entered; that costs time, not correctness.
// 4,608 bytes a wavefront.
struct PairLds {
    int pair[128];                 // ray lane | triangle << 6; the upper half takes writes that count for nothing
    unsigned long long best[64];   // per ray lane: distance bits << 32 | pair number
    int4 hit[64];                  // per ray lane: instance (-1: none), triangle and barycentrics of its closest hit so far
    // the per-lane bottom-level walk's shared work: subtrees given away (ray lane | node << 6), and a ring of
    // leaves waiting for their triangle tests (first triangle; ray lane | count << 6)
    int share[128];
    int2 leaf[256];
};

// v of the lane whose number is in bits 2 to 7 of four_times_lane.
__device__ __forceinline__ float lane_read(const float v, const int four_times_lane) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(four_times_lane, __float_as_int(v)));
}

// Orders a wavefront's LDS accesses: a wavefront's LDS operations are performed in order, so a
// compiler barrier is all that is needed between one lane's write and another lane's read.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int rank_in(const uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// old with lane `lane`'s value replaced by v (both wave-uniform); clang has no builtin of this instruction's name.
extern "C" __device__ __attribute__((const)) int ngx_write_lane(int v, int lane, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ int write_lane(const int v, const int lane, const int old) { return ngx_write_lane(v, lane, old); }

// A wave-uniform value in a scalar register, whose origin the compiler then does not see: it would otherwise compare counts
// of lanes as 64-bit numbers in vector registers, and keep conditions as lane masks.
__device__ __forceinline__ int as_scalar(int v) {
    v = uniform(v);
    asm("" : "+s"(v));
    return v;
}

// A wave-uniform stack of (node reference, lane mask) in three vector registers, entry k in lane k: a push or a pop is
// three instructions and waits for nothing.
struct WaveStack {
    int ref, lo, hi;
    int sp, deepest;
    __device__ __forceinline__ WaveStack() : ref(0), lo(0), hi(0), sp(0), deepest(0) {}
    // Depth bounds keep sp below WALK_STACK (a top-level tree has fewer than 64 levels below a world's root, and the
    // host refuses bottom-level trees deeper than 60). A tree that breaks them anyway loses an entry, and the walk
    // reports it at its end through the scene's overflow flag, which the host turns into an error.
    __device__ __forceinline__ void push(const int r, const uint64_t m) {
        const int at = min(sp, WALK_STACK - 1);
        ref = write_lane(r, at, ref);
        lo = write_lane((int)(uint32_t)m, at, lo);
        hi = write_lane((int)(uint32_t)(m >> 32), at, hi);
        deepest = max(deepest, ++sp);
        sp = min(sp, WALK_STACK);
    }
    // The same where m may be empty, which pushes nothing: the entry is written and not counted. The caller keeps `deepest`.
    __device__ __forceinline__ void push_some(const int r, const uint64_t m) {
        const int at = sp & 63;
        ref = write_lane(r, at, ref);
        lo = write_lane((int)(uint32_t)m, at, lo);
        hi = write_lane((int)(uint32_t)(m >> 32), at, hi);
        sp += as_scalar(min(popc64(m), 1));
    }
    __device__ __forceinline__ void pop(int &r, uint64_t &m) {
        --sp;
        r = __builtin_amdgcn_readlane(ref, sp);
        m = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, sp) << 32) | (uint32_t)__builtin_amdgcn_readlane(lo, sp);
    }
    __device__ __forceinline__ void report() const {
        if (NGX_UNLIKELY(deepest >= WALK_STACK) && lane_id() == 0) *Scene().overflow() = 1;
    }
};
static_assert(WALK_STACK <= 64, "an entry a lane");
static_assert(sizeof(PairLds) == 4608, "as BACKWARD_FEW_BODIES counts it");

// Tests the queued pairs of instance inst, whose mesh-space ray is (lo, ld) in each ray's lane.
template <class Stats>
__device__ __forceinline__ void flush_pairs(const Scene S, PairLds *L, int &pairs, const int inst, const float3 lo,
                                            const float3 ld, float &tmax, Stats &stats) {
    if (pairs == 0) return;
    stats.add(ST_TRIANGLES, 1);
    stats.add(ST_TRIANGLE_LANES, pairs);
    const int lane = lane_id();
    L->best[lane] = ((unsigned long long)__float_as_uint(tmax) << 32) | 0xffffffffull;
    wave_lds_order();
    const int e = L->pair[lane];
    const int r = e & 63, src = e << 2;
    float3 po = lo;
    if (!Stats::kOneOrigin) po = mk3(lane_read(lo.x, src), lane_read(lo.y, src), lane_read(lo.z, src));
    const float3 pd = mk3(lane_read(ld.x, src), lane_read(ld.y, src), lane_read(ld.z, src));
    const float pt = lane_read(tmax, src);
    float3 v0 = mk3(unknown_f(), unknown_f(), unknown_f()), e1 = mk3(unknown_f(), unknown_f(), unknown_f()),
           e2 = mk3(unknown_f(), unknown_f(), unknown_f());
    const bool act = lane < pairs;
    pairs = 0;
    if (NGX_LIKELY(act)) load_tri(S.tris(), (uint32_t)e >> 6, v0, e1, e2);
    float t, bu, bv;
    const bool found = triangle_hit(v0, e1, e2, po, pd, pt, t, bu, bv, act);
    if (ballot(found) == 0) return;
    const unsigned long long mine = ((unsigned long long)__float_as_uint(t) << 32) | (unsigned)lane;
    if (NGX_LIKELY(found)) atomicMin(&L->best[r], mine);
    wave_lds_order();
    // the pair that won writes its ray's hit; it is kept in LDS, not registers, until the walk is over
    if (NGX_LIKELY(found && L->best[r] == mine))
        L->hit[r] = make_int4(inst, (int)((uint32_t)e >> 6), __float_as_int(bu), __float_as_int(bv));
    const unsigned long long b = L->best[lane];
    tmax = !Stats::kAnyHit ? __uint_as_float((unsigned)(b >> 32)) : (unsigned)b != 0xffffffffu ? -1.0f : tmax;
    wave_lds_order();
}

// Queues the triangles first .. first+count-1 for the rays in mask, testing the queue first whenever it
// would overflow.
template <class Stats>
__device__ __forceinline__ void add_leaf(const Scene S, PairLds *L, int &pairs, const int first, const int count,
                                         const uint64_t mask, const int inst, const float3 lo, const float3 ld, float &tmax,
                                         LaneHit &h, Stats &stats) {
    const int m = popc64(mask);
    const int lane = lane_id();
    const bool in = in_mask(mask);
    const int rank = rank_in(mask);
    const int fit = 64 / m;
    for (int done = 0; done < count;) {
        const int c = min(count - done, fit);
        if (pairs + m * c > S.pair_limit()) flush_pairs(S, L, pairs, inst, lo, ld, tmax, stats);
        if (in) {
            const int base = pairs + rank * c;
            for (int k = 0; k < c; ++k) L->pair[base + k] = lane | ((first + done + k) << 6);
        }
        pairs += m * c;
        done += c;
    }
}


// The bottom level of one instance walked lane by lane, for meshes whose triangles are small next to a
// wavefront's tile: there each ray of the packet needs its own leaves, so a shared walk visits the union of
// 64 paths. A lane walks one ray through one subtree of the octant-ordered skip layout (a box test per step;
// a hit descends to the first child for the ray's octant, a miss or a leaf goes to the node's escape for the
// octant), so it keeps no stack. The work is shared: a lane whose remaining range is a whole subtree (its
// node's escape is the range's end) gives the far child's subtree to a shared stack in LDS, while there is
// room, and keeps the near one; idle lanes take the newest given subtrees, with their rays' mesh-space data
// read from the rays' own lanes. So the few rays that enter an instance keep the whole wave busy. Leaves are
// queued, and their triangles are tested in batches of up to 64 (ray, triangle) pairs once 64 leaves or 64
// pairs wait, and at the end; after each batch every walking lane re-reads its ray's closest distance. Every
// node a ray enters is walked by exactly one lane, so each ray's closest hit is its own. (OneBoxRays walk so;
// the others use the two-child walk further below, which shares its work the same way.)
constexpr int SHARE_CAP = SHARE_STACK, LEAF_RING = 256;
// Queued leaves that trigger a batch of triangle tests (at most 64 pairs a batch; fewer leaves wait for more).
#ifndef NGX_LEAF_BATCH
#define NGX_LEAF_BATCH 64
#endif
// In the hybrid walk, a bottom-level subtree entered by at most this many of the packet's rays is walked by the
// shared per-lane walk instead of the packet (0: never).
#ifndef NGX_HANDOFF_LANES
#define NGX_HANDOFF_LANES 16
#endif

template <bool FORCE, class Stats>
__device__ __forceinline__ void test_queued_leaves(const Scene S, PairLds *L, int &head, int &count, const int g,
                                                   const float3 lo, const float3 ld, float &tmax, Stats &stats) {
    const int lane = lane_id();
    while (count > 0) {
        wave_lds_order();
        const int2 leaf = L->leaf[(head + lane) & (LEAF_RING - 1)];  // what is past the queued ones is masked out
        const int rc = lane < count ? leaf.y : 0, first = leaf.x;
        const int c = rc >> 6;
        const int incl = wave_prefix_sum(c);
        const uint64_t take = ballot(lane < count && incl <= 64);
        if (NGX_UNLIKELY(take == 0)) {
            // a leaf of more than 64 triangles (the tree's leaves hold 4, unless a mesh has many coincident
            // triangles): its next 64, the rest stays queued
            const int ray0 = __builtin_amdgcn_readlane(rc, 0) & 63, first0 = __builtin_amdgcn_readlane(first, 0);
            const int c0 = __builtin_amdgcn_readlane(c, 0);
            wave_lds_order();
            L->pair[lane] = ray0 | ((first0 + lane) << 6);
            if (lane == 0) L->leaf[head] = make_int2(first0 + 64, ray0 | ((c0 - 64) << 6));
            int pairs = 64;
            flush_pairs(S, L, pairs, g, lo, ld, tmax, stats);
            continue;
        }
        const int taken = popc64(take);
        int pairs = __builtin_amdgcn_readlane(incl, taken - 1);
        if (!FORCE && count < 64 && pairs < 64) break;
        // each leaf's pairs from its place on; what a lane has no pair for goes to the upper half
        const int at = in_mask(take) ? incl - c : 64, n = in_mask(take) ? c : 0, pair0 = (rc & 63) | (first << 6);
        for (int k = 0; k < 4; ++k) L->pair[k < n ? at + k : 64 + lane] = pair0 + (k << 6);
        if (NGX_UNLIKELY(ballot(n > 4) != 0))
            for (int k = 4; k < n; ++k) L->pair[at + k] = pair0 + (k << 6);
        flush_pairs(S, L, pairs, g, lo, ld, tmax, stats);
        head = (head + taken) & (LEAF_RING - 1);
        count -= taken;
    }
}

// Gives the subtree of skip node `node` to the shared stack for every ray in mask (the caller has checked the room).
__device__ __forceinline__ void share_subtree(PairLds *L, int &top, const uint64_t mask, const int node) {
    if (in_mask(mask)) L->share[top + rank_in(mask)] = lane_id() | (node << 6);
    top += popc64(mask);
}

// Walks the `top` subtrees on the shared stack (rays of instance g, whose mesh-space rays are in their own lanes).
template <class Stats>
__device__ void walk_shared(const Scene S, PairLds *L, const int g, int top, const float3 lo, const float3 ld,
                            const float3 inv_ld, float &tmax, Stats &stats) {
    const int lane = lane_id();
    int head = 0, queued = 0;
    int ray = -1, cur = -1, end = -1, oct = 0;
    const SkipNode *const skip = S.skip();
    float3 wlo = lo, wld = ld, winv = inv_ld;
    float wlim = tmax;
    while (true) {
        // idle lanes take the newest given subtrees
        const uint64_t idle = ballot(ray < 0);
        if (top > 0 && idle != 0) {
            const int n = min(popc64(idle), top);
            const int rk = rank_in(idle);
            const bool take = in_mask(idle) && rk < n;
            wave_lds_order();
            int start = 0;
            if (take) {
                const int e = L->share[top - 1 - rk];
                ray = e & 63;
                start = e >> 6;
            }
            top -= n;
            const int src = ray >= 0 ? ray : lane;
            wlo = mk3(__shfl(lo.x, src, 64), __shfl(lo.y, src, 64), __shfl(lo.z, src, 64));
            wld = mk3(__shfl(ld.x, src, 64), __shfl(ld.y, src, 64), __shfl(ld.z, src, 64));
            winv = mk3(__shfl(inv_ld.x, src, 64), __shfl(inv_ld.y, src, 64), __shfl(inv_ld.z, src, 64));
            wlim = __shfl(tmax, src, 64);
            if (take) {
                oct = (wld.x >= 0.0f ? 1 : 0) | (wld.y >= 0.0f ? 2 : 0) | (wld.z >= 0.0f ? 4 : 0);
                cur = start;
                end = skip[start].escape[oct];
            }
        }
        const uint64_t busy = ballot(ray >= 0);
        if (busy == 0) break;
        stats.add(ST_BLAS_NODES, 1);
        stats.add(ST_BLAS_LANES, popc64(busy));
        // One step in every walking lane; the decisions are taken as wave masks, and only the node loads are
        // confined to the walking lanes (idle lanes test whatever their registers hold, and their results are masked out).
        float4 f0 = make_float4(unknown_f(), unknown_f(), unknown_f(), unknown_f());
        float4 f1 = make_float4(unknown_f(), unknown_f(), unknown_f(), unknown_f());
        int esc = unknown_i();
        if (in_mask(busy)) {
            // a 32-bit byte offset from the array's base (node indices stay below 2^25)
            const char *np = reinterpret_cast<const char *>(skip) + (uint32_t)cur * (uint32_t)sizeof(SkipNode);
            f0 = reinterpret_cast<const float4 *>(np)[0];
            f1 = reinterpret_cast<const float4 *>(np)[1];
            esc = reinterpret_cast<const SkipNode *>(np)->escape[oct];
        }
        const int a = __float_as_int(f0.w), meta = __float_as_int(f1.w);
        float tn;
        const uint64_t hm = busy & ballot(box_hit(f0.x, f0.y, f0.z, f1.x, f1.y, f1.z, wlo, winv, box_limit(wlim), tn));
        const uint64_t lm = hm & ballot(meta > 0);  // leaves entered
        const uint64_t im = hm & ~lm;               // interior nodes entered
        const int code = -meta - 1, axis = (code >> 1) & 3, flip = code & 1;
        const int near = ((oct >> axis) & 1) != flip ? a : a + 1;
        const int far = 2 * a + 1 - near;
        // a lane whose range is this node's subtree (its escape is the range's end) may give the far child away
        const uint64_t gm = im & ballot(esc == end);
        if (in_mask(busy)) cur = in_mask(im) ? near : esc;
        if (gm != 0) {
            const uint64_t given = gm & ballot(rank_in(gm) < SHARE_CAP - top);
            if (in_mask(given)) {
                L->share[top + rank_in(given)] = ray | (far << 6);
                end = far;  // after the near subtree the walk would reach the far one: stop there
            }
            top += popc64(given);
        }
        if (lm != 0) {
            if (in_mask(lm)) {
                const int slot = (head + queued + rank_in(lm)) & (LEAF_RING - 1);
                L->leaf[slot] = make_int2(a, ray | (meta << 6));
            }
            queued += popc64(lm);
        }
        if (in_mask(busy) && cur == end) ray = -1;
        if (queued >= NGX_LEAF_BATCH) {
            test_queued_leaves<false>(S, L, head, queued, g, lo, ld, tmax, stats);
            wlim = __shfl(tmax, ray >= 0 ? ray : lane, 64);
        }
    }
    test_queued_leaves<true>(S, L, head, queued, g, lo, ld, tmax, stats);
}

// The shared per-lane walk over the two-child layout the packet walk uses: a step loads one node and tests both of
// its children, as the reference does (mesh_dev.h:133-150), so a ray's chain of dependent node loads is half as long
// as in the walk above, whose arrival at a node is its box test. A work item is a subtree whose box its ray is known to
// enter. A lane entering both children of its node continues with the nearer one and gives the farther to the shared
// stack in LDS, or, when that is full, keeps it on its own stack; an idle lane first resumes its own entries, then
// takes the newest given subtree (with its ray's mesh-space data read from the ray's lane). A lane's own entries lie on
// one path down a tree, one a level at most, and the host refuses bottom-level trees of WALK_STACK levels or more, so
// WALK_STACK entries hold them. Leaves are queued and tested in batches as in the walk above.
// ORDERED: the nodes are the octant copies, an item's node in its ray's octant's, so near and far planes are known.
template <bool ORDERED, class Stats>
__device__ void walk_shared_two_child(const Scene S, PairLds *L, const int g, int top, const float3 lo,
                                      const float3 ld, const float3 inv_ld, float &tmax, Stats &stats) {
    int head = 0, queued = 0;
    // A lane's work as the stacks hold it, ray lane | node << 6 (so its upper bits are the node's byte offset), or
    // negative: idle. Lane reads take the low bits of 4 x a lane number, so work << 2 reads the ray's lane. An idle
    // lane's limit is negative, so it enters no box.
    int work = -1;
    float3 wlo = lo, winv = inv_ld;
    float wlim = -1.0f;
    int own[WALK_STACK];
    int own_n = 0, own_total = 0;  // the lane's own entries, and the wave's
    const char *const nodes = reinterpret_cast<const char *>(ORDERED ? S.blas_octants() : S.blas_wide());
    // A packet may have given more subtrees (up to SHARE_CAP) than a lowered capacity: what the first step's 64 takers leave
    // still lies on the shared stack, so its room is never negative.
    const int share_cap = max(S.share_cap(), top - 64);
    uint64_t busy = 0;
    do {
        if ((top | own_total) != 0 && ~busy != 0) {
            uint64_t takers = ~busy;
            if (NGX_UNLIKELY(own_total != 0)) {
                const uint64_t resume = takers & ballot(own_n > 0);
                if (in_mask(resume)) work = own[--own_n];
                own_total -= popc64(resume);
                takers &= ~resume;
            }
            const int n = min(popc64(takers), top);
            const int rk = rank_in(takers);
            wave_lds_order();
            if (NGX_LIKELY(in_mask(takers) && rk < n)) work = L->share[top - 1 - rk];
            top -= n;
            const int src = work << 2;
            if (!Stats::kOneOrigin) wlo = mk3(lane_read(lo.x, src), lane_read(lo.y, src), lane_read(lo.z, src));
            winv = mk3(lane_read(inv_ld.x, src), lane_read(inv_ld.y, src), lane_read(inv_ld.z, src));
            const float limit = min_quiet(lane_read(tmax, src), BELOW_NO_HIT);
            wlim = work >= 0 ? limit : -1.0f;
            busy = ballot(work >= 0);
        }
        stats.add(ST_BLAS_NODES, 1);
        stats.add(ST_BLAS_LANES, popc64(busy));
        // idle lanes test whatever their registers hold
        float4 f0 = make_float4(unknown_f(), unknown_f(), unknown_f(), unknown_f());
        float4 f1 = make_float4(unknown_f(), unknown_f(), unknown_f(), unknown_f());
        float4 f2 = make_float4(unknown_f(), unknown_f(), unknown_f(), unknown_f());
        int4 f3 = make_int4(unknown_i(), unknown_i(), unknown_i(), unknown_i());
        if (NGX_LIKELY(in_mask(busy))) {
            // a 32-bit byte offset from the array's base (node indices stay below 2^25)
            const float4 *np = reinterpret_cast<const float4 *>(nodes + ((uint32_t)work & ~63u));
            f0 = np[0];
            f1 = np[1];
            f2 = np[2];
            f3 = *reinterpret_cast<const int4 *>(np + 3);
        }
        float dl, dr;
        const uint64_t hl = ballot(ORDERED ? box_hit_ordered(f0.x, f1.x, f2.x, f0.z, f1.z, f2.z, wlo, winv, wlim, dl)
                                           : box_hit(f0.x, f1.x, f2.x, f0.z, f1.z, f2.z, wlo, winv, wlim, dl));
        const uint64_t hr = ballot(ORDERED ? box_hit_ordered(f0.y, f1.y, f2.y, f0.w, f1.w, f2.w, wlo, winv, wlim, dr)
                                           : box_hit(f0.y, f1.y, f2.y, f0.w, f1.w, f2.w, wlo, winv, wlim, dr));
        const uint64_t lleaf = ballot(f3.x < 0), rleaf = ballot(f3.y < 0);
        const uint64_t ll = hl & lleaf, rl = hr & rleaf;    // leaves entered
        const uint64_t li = hl & ~lleaf, ri = hr & ~rleaf;  // interior children entered
        const int ray = work & 63;
        if ((ll | rl) != 0) {
            // fewer than 64 wait and a step queues at most 128, so the ring holds them
            const int tail = head + queued, nl = popc64(ll), nr = popc64(rl);
            if (NGX_LIKELY(in_mask(ll))) L->leaf[(tail + rank_in(ll)) & (LEAF_RING - 1)] = make_int2(~f3.x, ray | (f3.z << 6));
            if (NGX_LIKELY(in_mask(rl))) L->leaf[(tail + nl + rank_in(rl)) & (LEAF_RING - 1)] = make_int2(~f3.y, ray | (f3.w << 6));
            queued += nl + nr;
        }
        // on to the nearer of the interior children entered (the left one when they are as near)
        const uint64_t go_left = li & (~ri | ballot(dl <= dr));
        const uint64_t both = li & ri;
        const int near = in_mask(go_left) ? f3.x : f3.y;
        if (both != 0) {
            const int far = ray | ((in_mask(go_left) ? f3.y : f3.x) << 6);
            // the lowest-ranked lanes fill the shared stack's room; the others keep their far child
            const int room = share_cap - top, rk = rank_in(both), n = popc64(both);
            const bool gives = rk < room;
            if (NGX_LIKELY(in_mask(both) && gives)) L->share[top + rk] = far;
            top += min(n, room);
            if (NGX_UNLIKELY(n > room)) {
                const bool keeps = in_mask(both) && !gives, fits = own_n < WALK_STACK;
                if (keeps && fits) own[own_n++] = far;
                if (keeps && !fits) *S.overflow() = 1;
                own_total += popc64(ballot(keeps && fits));
            }
        }
        busy = li | ri;
        work = in_mask(busy) ? ray | (near << 6) : -1;
        wlim = in_mask(busy) ? wlim : -1.0f;
        if (queued >= NGX_LEAF_BATCH) {
            test_queued_leaves<false>(S, L, head, queued, g, lo, ld, tmax, stats);
            const float limit = min_quiet(lane_read(tmax, work << 2), BELOW_NO_HIT);
            wlim = in_mask(busy) ? limit : -1.0f;
        }
    } while ((busy | (uint64_t)(uint32_t)(top | own_total)) != 0);
    test_queued_leaves<true>(S, L, head, queued, g, lo, ld, tmax, stats);
}

// The bottom level of one instance walked as a packet from its root node for the rays in root_mask. With LANES, subtrees
// entered by few rays are left on the shared stack (shared counts them).
template <bool LANES, class Stats>
__device__ __forceinline__ void walk_packet(const Scene S, PairLds *L, const int g, const int root_ref, const uint64_t root_mask,
                                            const float3 lo, const float3 ld, const float3 inv_d, float &tmax, LaneHit &h,
                                            const int octant_base, int &shared, Stats &stats) {
    int pairs = 0;
    WaveStack st;
    const WideNode *const nodes = S.blas_wide();
    const float3 lov = Stats::kOneOrigin ? in_vgpr3(lo) : lo;  // the nodes' planes are scalars too
    int cur = root_ref;
    uint64_t cm = root_mask;
    while (true) {
        const Wide w = load_wide(nodes, cur);
        stats.add(ST_BLAS_NODES, 1);
        stats.add(ST_BLAS_LANES, popc64(cm));
        // every lane runs the tests (a vector instruction costs the same for 1 lane or 64); the masks keep
        // the lanes of this node
        const float lim = box_limit(tmax);
        float dl, dr;
        const uint64_t ml = cm & ballot(box_hit(w.l_lo[0], w.l_lo[1], w.l_lo[2], w.l_hi[0], w.l_hi[1], w.l_hi[2], lov, inv_d, lim, dl));
        const uint64_t mr = cm & ballot(box_hit(w.r_lo[0], w.r_lo[1], w.r_lo[2], w.r_hi[0], w.r_hi[1], w.r_hi[2], lov, inv_d, lim, dr));
        int next_ref, next_count;
        uint64_t next_mask;
        if (ml != 0 && mr != 0) {
            // a lane is nearer the left child when it enters only the left, or the left no later than the right
            const uint64_t near_left = ml & (~mr | ballot(dl <= dr));
            const bool left_first = 2 * popc64(near_left) >= popc64(ml | mr);
            // a leaf child is pushed as its parent and side, and its run read back when popped
            if (left_first) {
                st.push(w.right >= 0 ? w.right : ~(2 * cur + 1), mr);
                next_ref = w.left; next_count = w.lcount; next_mask = ml;
            } else {
                st.push(w.left >= 0 ? w.left : ~(2 * cur), ml);
                next_ref = w.right; next_count = w.rcount; next_mask = mr;
            }
        } else if (ml != 0) {
            next_ref = w.left; next_count = w.lcount; next_mask = ml;
        } else if (mr != 0) {
            next_ref = w.right; next_count = w.rcount; next_mask = mr;
        } else {
            next_ref = 0; next_count = 0; next_mask = 0;
        }
        // Leaves are queued where they are reached; a subtree entered by few rays is given to the shared per-lane
        // walk (hybrid walk only); then the walk resumes from the stack.
        bool finished = false;
        while (true) {
            if (next_mask != 0 && next_ref >= 0) {
                const int n = popc64(next_mask);
                if (!LANES || !Stats::kHandoff || n > NGX_HANDOFF_LANES || shared + n > SHARE_CAP) break;
                share_subtree(L, shared, next_mask, Stats::kTwoChild ? octant_base + next_ref : S.blas_wide_node()[next_ref]);
            } else if (next_mask != 0) {
                add_leaf(S, L, pairs, ~next_ref, next_count, next_mask, g, lo, ld, tmax, h, stats);
            }
            if (st.sp == 0) {
                finished = true;
                break;
            }
            int r;
            st.pop(r, next_mask);
            if (r >= 0) {
                next_ref = r;
            } else {
                const int parent = (~r) >> 1, side = (~r) & 1;
                const Wide pw = load_wide(nodes, parent);
                next_ref = side ? pw.right : pw.left;
                next_count = side ? pw.rcount : pw.lcount;
            }
        }
        if (finished) break;
        cur = next_ref;
        cm = next_mask;
    }
    flush_pairs(S, L, pairs, g, lo, ld, tmax, stats);
    st.report();
}

template <class Stats>
__device__ __forceinline__ bool has_view(const Stats &stats) {
    if constexpr (Stats::kOneOrigin) return stats.inst != nullptr;
    return false;
}
template <class Stats>
__device__ __forceinline__ const float4 *view_instances(const Stats &stats) {
    if constexpr (Stats::kOneOrigin) return stats.inst;
    return nullptr;
}

// One instance for the lanes in mask: the ray moved into mesh space (mesh_dev.h:164-171, direction not
// renormalized so t is shared), then the mesh's own tree.
// BLAS: how bottom levels are walked: 0 as a packet; 1 lane by lane for meshes of lane_min_tris triangles or more,
// as a packet otherwise; 2 lane by lane for every mesh (the packet code is then not built, which frees registers; a
// mesh of a single leaf is still tested as one batch).
template <int BLAS, class Stats>
__device__ void visit_instance(const Scene S, PairLds *L, const int g, const uint64_t mask, const float3 o,
                               const float3 d, float &tmax, LaneHit &h, Stats &stats) {
    stats.add(ST_INSTANCES, 1);
    stats.add(ST_INSTANCE_LANES, popc64(mask));
    float3 lo, ld, inv_d;
    float root_t;
    uint64_t root_mask;
    int root_ref, root_count, skip_root = 0;
    bool lanes;
    if (Stats::kOneOrigin && has_view(stats)) {
        const float4 *const table = view_instances(stats);
        const uint32_t at = (uint32_t)g * (uint32_t)(VIEW_INSTANCE_FLOAT4S * sizeof(float4));
        const v16f r = sload16_at(table, at);
        const float4 m1 = sload4_at(table, at + 64);
        lo = mk3(r[3], r[7], r[11]);
        ld = mk3(dot3(mk3(r[0], r[1], r[2]), d), dot3(mk3(r[4], r[5], r[6]), d), dot3(mk3(r[8], r[9], r[10]), d));
        inv_d = safe_inverse(ld);
        root_mask = mask & ballot(box_hit(r[12], r[13], r[14], m1.x, m1.y, m1.z, mk3(0.0f, 0.0f, 0.0f), inv_d, box_limit(tmax), root_t));
        root_ref = __float_as_int(r[15]);
        root_count = __float_as_int(m1.w);
        lanes = BLAS == 2 || (BLAS == 1 && root_ref >= 0 && root_count != 0);
    } else {
        const float4 *rp = reinterpret_cast<const float4 *>((Stats::kOneOrigin ? Scene().inst() : S.inst()) + g);
        const float4 r0 = sload4(rp), r1 = sload4(rp + 1), r2 = sload4(rp + 2);
        const int4 meta = sload4i(reinterpret_cast<const int4 *>(rp + 3));
        lo = mk3(dot3(xyz(r0), o) + r0.w, dot3(xyz(r1), o) + r1.w, dot3(xyz(r2), o) + r2.w);
        if (Stats::kOneOrigin) lo = mk3(uniform_f(lo.x), uniform_f(lo.y), uniform_f(lo.z));
        ld = mk3(dot3(xyz(r0), d), dot3(xyz(r1), d), dot3(xyz(r2), d));
        inv_d = safe_inverse(ld);
        const float4 *mp = reinterpret_cast<const float4 *>((Stats::kOneOrigin ? Scene().mesh_roots() : S.mesh_roots()) + meta.x);
        const float4 m0 = sload4(mp), m1 = sload4(mp + 1);
        root_mask = mask & ballot(box_hit(m0.x, m0.y, m0.z, m1.x, m1.y, m1.z, lo, inv_d, box_limit(tmax), root_t));
        root_ref = __float_as_int(m0.w);
        root_count = __float_as_int(m1.w);
        skip_root = meta.w;
        lanes = BLAS == 2 || (BLAS == 1 && meta.z >= S.lane_min_tris());
    }
    if (root_mask == 0) return;
    stats.add(ST_INSTANCE_ROOT_LANES, popc64(root_mask));
    int shared = 0;  // subtrees given to the shared per-lane walk
    constexpr bool LANES = BLAS != 0;
    if constexpr (!Stats::kTwoChild) {
        if (lanes) {
            share_subtree(L, shared, root_mask, skip_root);
            walk_shared(S, L, g, shared, lo, ld, inv_d, tmax, stats);
            return;
        }
    }
    if (root_ref < 0) {
        // a mesh of one leaf, tested as a batch
        int pairs = 0;
        add_leaf(S, L, pairs, ~root_ref, root_count, root_mask, g, lo, ld, tmax, h, stats);
        flush_pairs(S, L, pairs, g, lo, ld, tmax, stats);
        return;
    }
    // the two-child layout starts below the root's box; with octant copies, each ray in its octant's
    const int octant_nodes = LANES && Stats::kTwoChild ? S.octant_nodes() : 0;
    const int octant_base = octant_nodes * ray_octant(inv_d);
    if (lanes) share_subtree(L, shared, root_mask, octant_base + root_ref);
    else if (BLAS != 2) walk_packet<LANES>(S, L, g, root_ref, root_mask, lo, ld, inv_d, tmax, h, octant_base, shared, stats);
    if (LANES && shared > 0) {
        if constexpr (!Stats::kTwoChild) walk_shared(S, L, g, shared, lo, ld, inv_d, tmax, stats);
        else if (octant_nodes > 0) walk_shared_two_child<true>(S, L, g, shared, lo, ld, inv_d, tmax, stats);
        else walk_shared_two_child<false>(S, L, g, shared, lo, ld, inv_d, tmax, stats);
    }
}

// From a top-level node to its nearer child, the farther one pushed, for the lanes in `mask`; l and r are the lanes whose
// rays enter each child's box, and nearer those that enter the left one no later. A lane is nearer the left child when it
// enters only the left, or the left no later than the right; the left child is first when it is nearer for half the lanes
// that enter either.
template <class Stats>
__device__ __forceinline__ void enter_children(WaveStack &st, const uint64_t l, const uint64_t r, const uint64_t nearer, const int left,
                                               const int right, int &ref, uint64_t &mask, Stats &stats) {
    stats.add(ST_TLAS_NODES, 1);
    stats.add(ST_TLAS_LANES, popc64(mask));
    const uint64_t ml = mask & l, mr = mask & r;
    const uint64_t near_left = ml & (~mr | nearer);
    const int more = as_scalar(popc64(near_left)) - as_scalar(popc64((ml | mr) & ~near_left));
    st.push_some(more >= 0 ? right : left, more >= 0 ? mr : ml);
    ref = more >= 0 ? left : right;
    mask = more >= 0 ? ml : mr;
}

// The closest instance hit in one world for the lanes in live (mesh_dev.h:177-205). tmax is each lane's
// distance to beat on entry and its closest distance on return.
template <int BLAS, class Stats>
__device__ void trace_world(const Scene S, PairLds *L, const int world, const float3 o, const float3 d,
                            const uint64_t live, float &tmax, LaneHit &h, Stats &stats) {
    if (live == 0) return;
    const int root = uniform(S.roots()[world]);
    if (root < 0) return;
    const float3 inv_d = safe_inverse(d);
    float lim = box_limit(tmax);
    // One entry is pushed per level at most. Below a world's root every level fixes at least one more bit
    // of a Morton code (30 bits) or, among equal codes, of the leaves' positions (at most ceil(log2 n) + 1
    // bits over n consecutive positions): fewer than 64 levels for any n < 2^31, so 64 entries do.
    WaveStack st;
    const WideNode *nodes = S.tlas_wide();
    int ordered = 0;  // the nodes are the view's, about its camera, for the octant all the rays have
    if constexpr (Stats::kOneOrigin) {
        if (stats.octants != VIEW_NO_OCTANTS) {
            const int octant = ray_octant(inv_d), all = __builtin_amdgcn_readlane(octant, first_lane(live));
            const int slot = (stats.octants >> (4 * all)) & 15;
            if (slot < VIEW_OCTANTS && (ballot(octant != all) & live) == 0) {
                ordered = 1;
                nodes = stats.nodes + (size_t)slot * (size_t)S.total();
            }
        }
    }
    const int first_leaf = S.total() - 1;
    // what to visit next: a node, or below zero an instance (a one-instance world's root is one)
    int next_ref = root >= first_leaf ? ~(root - first_leaf) : root;
    uint64_t next_mask = live;
    while (true) {
        // down to an instance, or to where no lane enters either child
        if (next_ref >= 0) {
            if (Stats::kOneOrigin && ordered != 0) {
                do {
                    const v16f w = sload16_at(nodes, (uint32_t)next_ref * (uint32_t)sizeof(WideNode));
                    const float3 about = mk3(0.0f, 0.0f, 0.0f);
                    float dl, dr;
                    const uint64_t l = ballot(box_hit_ordered(w[0], w[4], w[8], w[2], w[6], w[10], about, inv_d, lim, dl));
                    const uint64_t r = ballot(box_hit_ordered(w[1], w[5], w[9], w[3], w[7], w[11], about, inv_d, lim, dr));
                    enter_children(st, l, r, ballot(dl <= dr), __float_as_int(w[12]), __float_as_int(w[13]), next_ref, next_mask, stats);
                } while (as_scalar(next_mask != 0 ? next_ref : -1) >= 0);
            } else {
                const float3 ov = in_vgpr3(o);  // for camera rays the origin is scalars, as the nodes' planes are
                do {
                    const Wide w = load_wide(nodes, next_ref);
                    float dl, dr;
                    const uint64_t l = ballot(box_hit(w.l_lo[0], w.l_lo[1], w.l_lo[2], w.l_hi[0], w.l_hi[1], w.l_hi[2], ov, inv_d, lim, dl));
                    const uint64_t r = ballot(box_hit(w.r_lo[0], w.r_lo[1], w.r_lo[2], w.r_hi[0], w.r_hi[1], w.r_hi[2], ov, inv_d, lim, dr));
                    enter_children(st, l, r, ballot(dl <= dr), w.left, w.right, next_ref, next_mask, stats);
                } while (as_scalar(next_mask != 0 ? next_ref : -1) >= 0);
            }
            st.deepest = max(st.deepest, st.sp);
        }
        if (next_mask != 0) {
            visit_instance<BLAS>(S, L, ~next_ref, next_mask, o, d, tmax, h, stats);
            lim = min_quiet(tmax, BELOW_NO_HIT);
        }
        if (st.sp == 0) break;
        st.pop(next_ref, next_mask);
    }
    st.report();
}

// ------------------------------------------------------------------------------ per-lane walk --
//
// Each lane walks its own ray through both levels, in exactly the reference's order (near child first,
// mesh_dev.h:138-150, the far child visited only while its box is entered before the closest hit so far,
// :155), so ties break as the reference breaks them. No stack: a trail of bits per level remembers, for
// every node on the current path, whether its far child is still to visit and which side was near, and the
// walk climbs back through parent pointers. The top and bottom levels share one node step (the operands
// are selected per lane), so lanes working on different instances still advance together; leaves are
// postponed until every lane of the wave has one, then instance entries and triangle runs are done
// together (the "while-while" organisation of Aila and Laine, 2009).
template <class Stats>
__device__ void trace_world_lanes(const Scene S, const int world, const float3 o, const float3 d, const bool live,
                                  float &tmax, LaneHit &h, Stats &stats) {
    constexpr int NODE = 0, LEAF = 1, BACK = 2, DONE = 3;
    const WideNode *const top_nodes = S.tlas_wide(), *const bottom_nodes = S.blas_wide();
    const int *const top_parents = S.tlas_parent(), *const bottom_parents = S.blas_parent();
    const float3 inv_d = safe_inverse(d);
    int state = DONE, level = 0;
    int cur_t = -1, cur_b = -1;
    uint64_t bits_t = 0, side_t = 0, bits_b = 0, side_b = 0;
    int depth_t = 0, depth_b = 0;  // levels below the level's root: the trails hold 64 levels
    int leaf_ref = 0, leaf_count = 0, g = 0;
    float3 lo = o, ld = d, inv_ld = inv_d;
    if (live) {
        // an empty world's root is -1; test that first, since with no instances at all total - 1 is -1 too
        const int root = S.roots()[world];
        if (root < 0) {
            state = DONE;
        } else if (root >= S.total() - 1) {
            state = LEAF;
            leaf_ref = ~(root - (S.total() - 1));
        } else {
            state = NODE;
            cur_t = root;
        }
    }
    while (ballot(state != DONE)) {
        // ---- node steps until every lane waits at a leaf or is done
        while (true) {
            const bool on_node = state == NODE, on_back = state == BACK;
            const uint64_t active = ballot(on_node || on_back);
            if (active == 0) break;
            stats.add(ST_TLAS_NODES, 1);
            stats.add(ST_TLAS_LANES, popc64(active));
            if (on_node || on_back) {
                const bool bottom = level == 1;
                int cur = bottom ? cur_b : cur_t;
                uint64_t bits = bottom ? bits_b : bits_t;
                uint64_t side = bottom ? side_b : side_t;
                int depth = bottom ? depth_b : depth_t;
                const bool pending = on_back && (bits & 1ull);
                if (on_node || pending) {
                    const float4 *np = reinterpret_cast<const float4 *>((bottom ? bottom_nodes : top_nodes) + cur);
                    const float4 f0 = np[0], f1 = np[1], f2 = np[2];
                    const int4 f3 = *reinterpret_cast<const int4 *>(np + 3);
                    const float3 ro = bottom ? lo : o, ri = bottom ? inv_ld : inv_d;
                    const float dl = box_entry(f0.x, f1.x, f2.x, f0.z, f1.z, f2.z, ro, ri, tmax);
                    const float dr = box_entry(f0.y, f1.y, f2.y, f0.w, f1.w, f2.w, ro, ri, tmax);
                    const bool hl = dl < NO_HIT, hr = dr < NO_HIT;
                    int child = 0, child_count = 0;
                    bool go = false;
                    if (on_node) {
                        if (hl && hr) {
                            const bool left_first = dl <= dr;
                            bits |= 1ull;
                            side = left_first ? (side & ~1ull) : (side | 1ull);
                            child = left_first ? f3.x : f3.y;
                            child_count = left_first ? f3.z : f3.w;
                            go = true;
                        } else if (hl || hr) {
                            child = hl ? f3.x : f3.y;
                            child_count = hl ? f3.z : f3.w;
                            go = true;
                        } else {
                            state = BACK;
                        }
                    } else {
                        bits &= ~1ull;
                        const bool far_left = (side & 1ull) != 0;  // the near child was the right one
                        if (far_left ? hl : hr) {
                            child = far_left ? f3.x : f3.y;
                            child_count = far_left ? f3.z : f3.w;
                            go = true;
                        }
                    }
                    if (go) {
                        if (child >= 0) {
                            cur = child;
                            bits <<= 1;
                            side <<= 1;
                            // a 65th level would push the root's bit out of the trail
                            if (++depth >= 64) *S.overflow() = 1;
                            state = NODE;
                        } else {
                            state = LEAF;
                            leaf_ref = child;
                            leaf_count = child_count;
                        }
                    }
                } else {
                    // climb one level; a level whose root is finished hands back to the level above
                    const int parent = cur < 0 ? -1 : (bottom ? bottom_parents : top_parents)[cur];
                    if (parent < 0) {
                        if (bottom) level = 0;  // the instance is done: resume the top level where it left off
                        else state = DONE;
                    } else {
                        cur = parent;
                        bits >>= 1;
                        side >>= 1;
                        --depth;
                    }
                }
                if (bottom) {
                    cur_b = cur;
                    bits_b = bits;
                    side_b = side;
                    depth_b = depth;
                } else {
                    cur_t = cur;
                    bits_t = bits;
                    side_t = side;
                    depth_t = depth;
                }
            }
        }
        // ---- instance entries: the ray moved into mesh space, then the mesh's root box
        const bool enter = state == LEAF && level == 0;
        if (ballot(enter)) {
            stats.add(ST_INSTANCES, 1);
            stats.add(ST_INSTANCE_LANES, popc64(ballot(enter)));
            if (enter) {
                g = ~leaf_ref;
                const float4 *rp = reinterpret_cast<const float4 *>(S.inst() + g);
                const float4 r0 = rp[0], r1 = rp[1], r2 = rp[2];
                const int mesh = reinterpret_cast<const int4 *>(rp + 3)->x;
                lo = mk3(dot3(xyz(r0), o) + r0.w, dot3(xyz(r1), o) + r1.w, dot3(xyz(r2), o) + r2.w);
                ld = mk3(dot3(xyz(r0), d), dot3(xyz(r1), d), dot3(xyz(r2), d));
                inv_ld = safe_inverse(ld);
                const float4 *mp = reinterpret_cast<const float4 *>(S.mesh_roots() + mesh);
                const float4 m0 = mp[0], m1 = mp[1];
                if (box_entry(m0.x, m0.y, m0.z, m1.x, m1.y, m1.z, lo, inv_ld, tmax) < NO_HIT) {
                    level = 1;
                    bits_b = side_b = 0;
                    depth_b = 0;
                    const int root_ref = __float_as_int(m0.w);
                    if (root_ref >= 0) {
                        cur_b = root_ref;
                        state = NODE;
                    } else {
                        cur_b = -1;
                        leaf_ref = root_ref;
                        leaf_count = __float_as_int(m1.w);
                    }
                } else {
                    state = BACK;
                }
            }
        }
        // ---- triangle runs
        const bool tris = state == LEAF && level == 1;
        if (ballot(tris)) {
            stats.add(ST_TRIANGLES, 1);
            stats.add(ST_TRIANGLE_LANES, popc64(ballot(tris)));
            if (tris) {
                const int first = ~leaf_ref;
                for (int j = first; j < first + leaf_count; ++j) {
                    float3 v0, e1, e2;
                    load_tri(S.tris(), (size_t)j, v0, e1, e2);
                    float t, bu, bv;
                    if (triangle_hit(v0, e1, e2, lo, ld, tmax, t, bu, bv)) {
                        tmax = Stats::kAnyHit ? -1.0f : t;
                        h.inst = g;
                        h.tri = j;
                        h.u = bu;
                        h.v = bv;
                    }
                }
                state = BACK;
            }
        }
    }
}

// Spheres, then the floor, then the meshes with the best so far as their limit (render_core.h:78-112).
// Returns the object, or OBJECT_NONE; t and h describe the hit.
// The walks: per-lane (both levels lane by lane), packet (both levels as a packet), and hybrid (the packet
// walk with fine meshes' bottom levels walked lane by lane).
// The walks: per-lane (both levels lane by lane), packet (both levels as a packet), hybrid (the packet walk with fine
// meshes' bottom levels walked lane by lane), and shared (the packet top level, every bottom level lane by lane: what
// the hybrid walk does when every mesh is fine, built without the packet bottom level; ray queries only).
enum Walk { WALK_LANES = 0, WALK_PACKET = 1, WALK_HYBRID = 2, WALK_SHARED = 3 };
template <int WALK>
constexpr int blas_mode() { return WALK == WALK_SHARED ? 2 : WALK == WALK_HYBRID ? 1 : 0; }

template <int WALK, class Stats>
__device__ __forceinline__ int scene_hit(const Scene S, PairLds *L, const int world, const float3 o, const float3 d,
                                         const uint64_t live, float &best, LaneHit &h, Stats &stats, const float start = 1e30f) {
    best = start;
    int best_sphere = -1;
    for (int i = 0; i < S.sphere_count(); ++i) {
        const float4 sp = sload4(S.spheres() + i);
        const float3 L = sub3(xyz(sp), o);
        const float tca = dot3(L, d);
        const float r2 = sp.w * sp.w;
        const float d2 = dot3(L, L) - tca * tca;
        if (d2 > r2) continue;
        const float thc = sqrtf(r2 - d2);
        float t = tca - thc;
        if (t < 0.0f) t = tca + thc;
        if (t >= 0.0f && t < best) {
            best = t;
            best_sphere = i;
        }
    }
    bool hit_floor = false;
    if (fabsf(d.y) > 1e-3f) {
        const float dist = (S.floor_y() - o.y) / d.y;
        if (dist > 0.0f && dist < best) {
            const float3 pt = add3(o, mul3(d, dist));
            if (fabsf(pt.x) < S.floor_hx() && pt.z > S.floor_zmin() && pt.z < S.floor_zmax()) {
                best = dist;
                hit_floor = true;
            }
        }
    }
    h.inst = -1;
    h.tri = -1;
    if (WALK != WALK_LANES) {
        const int lane = lane_id();
        L->hit[lane].x = -1;
        wave_lds_order();
        trace_world<blas_mode<WALK>()>(S, L, world, o, d, live, best, h, stats);
        wave_lds_order();
        const int4 k = L->hit[lane];
        h.inst = k.x;
        if (h.inst >= 0) {
            h.tri = k.y;
            h.u = __int_as_float(k.z);
            h.v = __int_as_float(k.w);
        }
    } else trace_world_lanes(S, world, o, d, ((live >> lane_id()) & 1ull) != 0, best, h, stats);
    if (h.inst >= 0) return OBJECT_INSTANCE;
    if (hit_floor) return OBJECT_FLOOR;
    if (best_sphere >= 0) return OBJECT_SPHERE + best_sphere;
    return OBJECT_NONE;
}

// Normal and object ID of a hit (render_core.h:119-141, mesh_dev.h:238-262).
__device__ __forceinline__ void surface(const Scene S, const int kind, const float3 o, const float3 d, const float t,
                                        const LaneHit &h, float3 &normal, int &object) {
    if (kind == OBJECT_INSTANCE) {
        const InstanceRec &rec = S.inst()[h.inst];
        const float3 r0 = xyz(rec.inv[0]), r1 = xyz(rec.inv[1]), r2 = xyz(rec.inv[2]);
        float3 v0, e1, e2;
        load_tri(S.tris(), (size_t)h.tri, v0, e1, e2);
        const float3 nl = cross3(e1, e2);
        float3 geometric = normalize3(add3(add3(mul3(r0, nl.x), mul3(r1, nl.y)), mul3(r2, nl.z)));
        if (dot3(geometric, d) > 0.0f) geometric = neg3(geometric);
        normal = geometric;
        if (S.attrs() != nullptr) {
            const float4 *ap = S.attrs() + 4 * (size_t)h.tri;
            const float4 a0 = ap[0], a1 = ap[1], a2 = ap[2], a3 = ap[3];
            if (__float_as_int(a3.w) & 1) {
                const float w0 = 1.0f - h.u - h.v;
                const float3 n = add3(add3(mul3(xyz(a0), w0), mul3(xyz(a1), h.u)), mul3(xyz(a2), h.v));
                if (dot3(n, n) > 1e-12f) {
                    const float3 smooth = normalize3(add3(add3(mul3(r0, n.x), mul3(r1, n.y)), mul3(r2, n.z)));
                    normal = dot3(smooth, geometric) < 0.0f ? neg3(smooth) : smooth;
                }
            }
        }
        object = OBJECT_INSTANCE + rec.tmpl;
    } else if (kind == OBJECT_FLOOR) {
        normal = mk3(0.0f, 1.0f, 0.0f);
        object = OBJECT_FLOOR;
    } else {
        const float4 sp = S.spheres()[kind - OBJECT_SPHERE];
        normal = normalize3(sub3(add3(o, mul3(d, t)), xyz(sp)));
        object = kind;
    }
}

// The object ID surface() gives, without the normal: what a frame of depth and IDs alone needs.
__device__ __forceinline__ int object_of(const Scene S, const int kind, const LaneHit &h) {
    return kind == OBJECT_INSTANCE ? OBJECT_INSTANCE + S.inst()[h.inst].tmpl : kind;
}

struct Cam {
    float3 pos, right, up, fwd;
};

// camera_from_matrix (render_core.h:264-273): the matrix's columns, renormalized.
__device__ __forceinline__ Cam load_camera(const float *m12) {
    const float4 *p = reinterpret_cast<const float4 *>(m12);
    const float4 a = sload4(p), b = sload4(p + 1), c = sload4(p + 2);
    Cam cam;
    cam.pos = mk3(a.w, b.w, c.w);
    cam.right = normalize3(mk3(a.x, b.x, c.x));
    cam.up = normalize3(mk3(a.y, b.y, c.y));
    cam.fwd = normalize3(mk3(-a.z, -b.z, -c.z));
    return cam;
}

// A view's camera, from its tables or, where there are none, its matrix; with the tables its rays walk.
// Args: RenderArgs, or the same in the kernel arguments' segment.
template <class Args>
__device__ __forceinline__ Cam camera_of(const Args &A, const int view, const int world, ViewOfRays &rays) {
    if (A.tables.cams == nullptr) return load_camera(in_global(A.cams) + 12 * (size_t)view);
    const float4 *p = A.tables.cams + 4 * (size_t)view;
    const float4 a = sload4(p), b = sload4(p + 1), c = sload4(p + 2), e = sload4(p + 3);
    const size_t first = (size_t)(view - world * A.cameras_per_world) * (size_t)A.s.total;
    rays.octants = __float_as_int(a.w);
    rays.nodes = A.tables.nodes + VIEW_OCTANTS * first;
    rays.inst = A.tables.inst + VIEW_INSTANCE_FLOAT4S * first;
    return Cam{xyz(a), xyz(b), xyz(c), xyz(e)};
}

// camera_ray (device_scene.h:114-119) through a pixel's centre.
__device__ __forceinline__ float plane_x(const float px, const int width, const float fov_scale, const float aspect) {
    return (2.0f * px / (float)width - 1.0f) * fov_scale * aspect;
}
__device__ __forceinline__ float plane_y(const float py, const int height, const float fov_scale) {
    return -(2.0f * py / (float)height - 1.0f) * fov_scale;
}
__device__ __forceinline__ float3 plane_ray(const Cam &c, const float sx, const float sy) {
    return normalize3(add3(add3(mul3(c.right, sx), mul3(c.up, sy)), c.fwd));
}
__device__ __forceinline__ float3 pixel_ray(const Cam &c, const float fov_scale, const float aspect, const int x, const int y,
                                            const int width, const int height) {
    return plane_ray(c, plane_x((float)x + 0.5f, width, fov_scale, aspect), plane_y((float)y + 0.5f, height, fov_scale));
}
template <class Args>
__device__ __forceinline__ float3 pixel_ray_of(const Args &A, const Cam &c, const int x, const int y) {
    if (A.tables.cams == nullptr) return pixel_ray(c, A.fov_scale, A.aspect, x, y, A.width, A.height);
    const float *const px = in_global(A.tables.pixels);
    return plane_ray(c, px[(uint32_t)x], px[(uint32_t)(A.width + PIXEL_PAD + y)]);
}

// The tile of a wave: tiles are numbered view-major, and with xcd_remap consecutive workgroups, which
// the dispatcher deals round-robin over the eight XCDs, are renumbered so each XCD works through one
// contiguous range of tiles (the same views, so the same worlds' trees in its L2).
__device__ __forceinline__ long long wave_tile(const int xcd_remap, const long long waves_total) {
    const long long blocks = (long long)gridDim.x;
    long long b = blockIdx.x;
    if (xcd_remap && blocks >= 8) {
        const long long per = blocks / 8, rem = blocks % 8, xcd = b % 8, k = b / 8;
        // XCD x receives blocks x, x+8, ...: give it the x-th contiguous range
        b = xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
    }
    (void)waves_total;
    return b * (blockDim.x >> 6) + uniform(threadIdx.x >> 6);
}

// LDS of the packet walk's triangle batches: one PairLds per wavefront of a 256-thread workgroup.
#define NGX_PAIR_LDS(name) __shared__ PairLds name##_all[4]; PairLds *name = WALK != WALK_LANES ? &name##_all[threadIdx.x >> 6] : nullptr

// A lane's pixel in its wavefront's tile of one view. Args: RenderArgs, or the same in the kernel arguments' segment.
struct TilePixel {
    int view, x, y, world;
    bool valid;
    size_t index;  // into [views][H][W]
};
template <class Divide>
__device__ __forceinline__ int fast_divide(const int n, const Divide &by) { return (int)(((uint64_t)(uint32_t)n * by.mul) >> by.shift); }
template <class Args>
__device__ __forceinline__ TilePixel tile_pixel(const Args &A, const long long tile) {
    const int lane = lane_id();
    TilePixel p;
    int t, ty;
    if (A.total_tiles <= INT32_MAX) {
        p.view = fast_divide((int)tile, A.by_tiles_per_view);
        t = (int)tile - p.view * A.tiles_per_view;
        ty = fast_divide(t, A.by_tiles_x);
        p.world = fast_divide(p.view, A.by_cameras);
    } else {
        p.view = (int)(tile / A.tiles_per_view);
        t = (int)(tile - (long long)p.view * A.tiles_per_view);
        ty = t / A.tiles_x;
        p.world = p.view / A.cameras_per_world;
    }
    p.x = (t - ty * A.tiles_x) * A.tile_w + (lane & (A.tile_w - 1));
    p.y = ty * A.tile_h + (lane >> A.tile_w_log2);
    p.valid = lane < A.tile_w * A.tile_h && p.x < A.width && p.y < A.height;
    p.index = ((size_t)p.view * A.height + p.y) * A.width + p.x;
    return p;
}

// One 64-pixel tile of one view: camera ray per lane, closest hit, depth / normal / object ID.
template <int WALK>
__device__ __forceinline__ void render_tile(PairLds *L, const long long tile) {
    float3 d;
    Cam cam;
    TilePixel p;
    CameraRays stats;
    {
        const auto &A = kernel_args<RenderArgs>();
        p = tile_pixel(A, tile);
        cam = camera_of(A, p.view, p.world, stats);
        d = pixel_ray_of(A, cam, p.x, p.y);
    }
    float best;
    LaneHit h;
    const int kind = scene_hit<WALK>(Scene(), L, p.world, cam.pos, d, ballot(p.valid), best, h, stats);
    if (!p.valid) return;
    const auto &A = kernel_args<RenderArgs>();
    const size_t idx = p.index;
    const bool found = kind != OBJECT_NONE;
    float *const depth = in_global(A.depth), *const normals = in_global(A.normal);
    int32_t *const object_id = in_global(A.object_id);
    if (depth) depth[idx] = found ? best * dot3(d, cam.fwd) : __int_as_float(0x7f800000);
    if (normals) {
        float3 normal = mk3(0.0f, 0.0f, 0.0f);
        int object = OBJECT_NONE;
        if (found) surface(Scene(), kind, cam.pos, d, best, h, normal, object);
        normals[3 * idx] = normal.x;
        normals[3 * idx + 1] = normal.y;
        normals[3 * idx + 2] = normal.z;
        if (object_id) object_id[idx] = object;
    } else if (object_id) {
        object_id[idx] = found ? object_of(Scene(), kind, h) : OBJECT_NONE;
    }
}

// BLOCKS: workgroups per compute unit the kernel is built for (their registers follow: 7 gives at most 72 VGPRs,
// with more spilled; body_worlds 10.49 ms at 6, 10.20 ms at 7). The packet and hybrid walks are built at 5, 6 and 7
// and the autotuner picks one; the per-lane walk at 1.

// One tile per wavefront, tiles dealt by the dispatcher.
template <int WALK, int BLOCKS>
__global__ __launch_bounds__(256, BLOCKS) void render_kernel(const RenderArgs A) {
    NGX_PAIR_LDS(L);
    const long long tile = wave_tile(A.xcd_remap, A.total_tiles);
    if (tile >= A.total_tiles) return;
    render_tile<WALK>(L, tile);
}

// Persistent: a fixed grid whose wavefronts take tiles until none are left. The tiles are cut into eight
// contiguous ranges, one per XCD (the dispatcher deals workgroups round-robin over the XCDs, so workgroup b
// runs on XCD b mod 8), so the worlds of a range stay in one XCD's L2; each range is cut into COUNTER_SLICES
// slices with a counter each on its own cache line. A wavefront starts at the slice its index within the XCD
// picks, takes PERSISTENT_CHUNK (1) tile per counter increment until the slice is used up, then
// moves on to the XCD's next slice; it leaves once it has found every slice of its range used up, so every
// wavefront ends after at most COUNTER_SLICES empty increments. The grid is a multiple of 8 workgroups, so every
// XCD's range has wavefronts to take it.
#ifndef NGX_PERSISTENT_CHUNK
#define NGX_PERSISTENT_CHUNK 1
#endif
constexpr int PERSISTENT_CHUNK = NGX_PERSISTENT_CHUNK;

// The first workgroup zeroes `next`, the counters of the launch after this one, which spares that launch a kernel to
// do so before it (a step of one small world: 44.1 us with one, 42.1 so).
template <class Work>
__device__ __forceinline__ void take_tiles(int *counters, int *next, const long long total, Work &&work) {
    if (blockIdx.x == 0 && next != nullptr && threadIdx.x < 8 * COUNTER_SLICES) next[threadIdx.x * COUNTER_STRIDE] = 0;
    const int xcd = blockIdx.x & 7;
    const long long first = total * xcd / 8, count = total * (xcd + 1) / 8 - first;
    const int home = uniform((int)((blockIdx.x >> 3) * (blockDim.x >> 6) + (threadIdx.x >> 6)) % COUNTER_SLICES);
    for (int i = 0; i < COUNTER_SLICES; ++i) {
        const int s = (home + i) % COUNTER_SLICES;
        const long long lo = count * s / COUNTER_SLICES, n = count * (s + 1) / COUNTER_SLICES - lo;
        int *c = counters + (xcd * COUNTER_SLICES + s) * COUNTER_STRIDE;
        if (i > 0) {
            // a slice another wavefront has used up is passed over with a load rather than an increment, so the
            // end of the launch costs each wavefront one increment instead of one per slice
            int seen = 0;
            if (lane_id() == 0) seen = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_readlane(seen, 0) >= n) continue;
        }
        while (true) {
            int t = 0;
            if (lane_id() == 0) t = atomicAdd(c, PERSISTENT_CHUNK);
            t = __builtin_amdgcn_readlane(t, 0);
            if (t >= n) break;
            const int end = (int)min((long long)t + PERSISTENT_CHUNK, n);
            for (int k = t; k < end; ++k) work(first + lo + k);
        }
    }
}

template <int WALK, int BLOCKS>
__global__ __launch_bounds__(256, BLOCKS) void render_persistent_kernel(const RenderArgs A) {
    NGX_PAIR_LDS(L);
    take_tiles(A.tile_counters, A.next_counters, A.total_tiles, [&](const long long tile) { render_tile<WALK>(L, tile); });
}

// The view tables: a wavefront a view and a run of its world's instances. Bound by the copies it writes, about 340 bytes an
// instance and view (541,000 instances in 4,096 views: 80 us, 2.3 TB/s; the launch it goes before is 6.4 ms and 4 to 5%
// shorter for them). Node copies hold the lower of a pair of planes as near whatever the node holds, so that a box turned
// inside out, or one with a plane that is no number, is entered by the rays that entered it before.
__global__ __launch_bounds__(64) void view_tables_kernel(const ViewTableArgs A, const int runs) {
    const int first = blockIdx.x * 64 + threadIdx.x, step = gridDim.x * 64;
    for (int i = first; i < A.counter_sets * 8 * COUNTER_SLICES; i += step) A.counters[(size_t)i * COUNTER_STRIDE] = 0;
    if (A.t.cams == nullptr) return;
    const int columns = A.width + PIXEL_PAD;
    for (int i = first; i < columns + A.height + PIXEL_PAD; i += step)
        A.t.pixels[i] = i < columns ? plane_x((float)i + 0.5f, A.width, A.fov_scale, A.aspect)
                                    : plane_y((float)(i - columns) + 0.5f, A.height, A.fov_scale);
    const int view = blockIdx.x / runs, run = blockIdx.x % runs;
    const int world = view / A.cameras_per_world, camera = view - world * A.cameras_per_world;
    const Cam cam = load_camera(A.cams + 12 * (size_t)view);
    // The octants of the view's rays: along an axis the directions before normalization are linear over the image, so
    // the corners tell which signs it has.
    bool below[3] = {false, false, false}, above[3] = {false, false, false};
    for (int corner = 0; corner < 4; ++corner) {
        const float sx = (corner & 1 ? A.aspect : -A.aspect) * A.fov_scale, sy = corner & 2 ? A.fov_scale : -A.fov_scale;
        const float3 d = add3(add3(mul3(cam.right, sx), mul3(cam.up, sy)), cam.fwd);
        const float along[3] = {d.x, d.y, d.z};
        for (int ax = 0; ax < 3; ++ax) {
            below[ax] |= along[ax] < 0.0f;
            above[ax] |= !(along[ax] < 0.0f);
        }
    }
    int octants = 0, kept = 0, of_slot = 0;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        bool seen = kept < VIEW_OCTANTS;
        for (int ax = 0; ax < 3; ++ax) seen &= (o >> ax) & 1 ? below[ax] : above[ax];
        octants |= (seen ? kept : 15) << (4 * o);
        if (seen) of_slot |= o << (4 * kept++);
    }
    if (run == 0 && threadIdx.x < 4) {
        const float3 v = threadIdx.x == 0 ? cam.pos : threadIdx.x == 1 ? cam.right : threadIdx.x == 2 ? cam.up : cam.fwd;
        A.t.cams[4 * (size_t)view + threadIdx.x] = make_float4(v.x, v.y, v.z, threadIdx.x == 0 ? __int_as_float(octants) : 0.0f);
    }
    const int base = A.world_off[world], count = A.world_off[world + 1] - base;
    const int no_node = A.root_at_end[world] ? 0 : count - 1;  // the world's run of nodes has one unused
    const size_t at = (size_t)camera * (size_t)A.total;
    const float origin[3] = {cam.pos.x, cam.pos.y, cam.pos.z};
    for (int k = run * 64 + threadIdx.x; k < count; k += runs * 64) {
        const size_t g = (size_t)base + k;
        if (k != no_node) {
            const WideNode node = A.tlas_wide[g];
            float low[3][2], high[3][2];
            for (int ax = 0; ax < 3; ++ax)
                for (int side = 0; side < 2; ++side) {
                    const float p = node.plane[ax][side] - origin[ax], q = node.plane[ax][2 + side] - origin[ax];
                    low[ax][side] = fminf(p, q);
                    high[ax][side] = fmaxf(p, q);
                }
            for (int slot = 0; slot < kept; ++slot) {
                const int o = of_slot >> (4 * slot);
                WideNode n;
                for (int ax = 0; ax < 3; ++ax)
                    for (int side = 0; side < 2; ++side) {
                        const bool down = (o >> ax) & 1;
                        n.plane[ax][side] = down ? high[ax][side] : low[ax][side];
                        n.plane[ax][2 + side] = down ? low[ax][side] : high[ax][side];
                    }
                n.left = node.left;
                n.right = node.right;
                n.left_count = n.right_count = 1;
                A.t.nodes[VIEW_OCTANTS * at + (size_t)slot * (size_t)A.total + g] = n;
            }
        }
        const InstanceRec rec = A.inst[g];
        const MeshRoot root = A.mesh_roots[rec.mesh];
        float4 *const out = A.t.inst + VIEW_INSTANCE_FLOAT4S * (at + g);
        float lo[3];
        for (int ax = 0; ax < 3; ++ax) {
            lo[ax] = dot3(xyz(rec.inv[ax]), cam.pos) + rec.inv[ax].w;
            out[ax] = make_float4(rec.inv[ax].x, rec.inv[ax].y, rec.inv[ax].z, lo[ax]);
        }
        out[3] = make_float4(root.lo[0] - lo[0], root.lo[1] - lo[1], root.lo[2] - lo[2], __int_as_float(root.ref));
        out[4] = make_float4(root.hi[0] - lo[0], root.hi[1] - lo[1], root.hi[2] - lo[2],
                             __int_as_float(root.ref < 0 ? root.count : rec.mesh_tris >= A.lane_min_tris ? 1 : 0));
    }
}

#ifdef NGX_TRACE_STATS
// The render kernel's traversal with its counters: each wave writes ST_COUNT ints to its own slot, lane k
// storing counter k, so no atomics are involved.
static_assert(ST_COUNT == TRACE_STAT_COUNT && ST_COUNT <= 64, "one counter a lane, as many as the host reads");
template <int WALK>
__global__ __launch_bounds__(256) void render_stats_kernel(const RenderArgs A, int *out) {
    NGX_PAIR_LDS(L);
    const long long tile = wave_tile(A.xcd_remap, A.total_tiles);
    if (tile >= A.total_tiles) return;
    const int lane = lane_id();
    const TilePixel p = tile_pixel(A, tile);
    const bool valid = p.valid;
    const int world = p.world;
    WaveStats stats;
    const Cam cam = camera_of(A, p.view, world, stats);
    const float3 d = pixel_ray_of(A, cam, p.x, p.y);
    float best;
    LaneHit h;
    for (int k = 0; k < ST_COUNT; ++k) stats.c[k] = 0;
    stats.add(ST_VALID, popc64(ballot(valid)));
    scene_hit<WALK>(Scene(), L, world, cam.pos, d, ballot(valid), best, h, stats);
    int mine = 0;
    for (int k = 0; k < ST_COUNT; ++k) mine = lane == k ? stats.c[k] : mine;
    if (lane < ST_COUNT) out[(size_t)tile * ST_COUNT + lane] = mine;
}
#endif

// ------------------------------------------------------------------------------ RGB picture --
//
// The classic picture (render_core.h:146-283): per pixel, spp jittered camera rays; per ray, up to
// MAX_BOUNCES mirror bounces; at each hit, direct light from every sphere light sampled at a random point of
// the light (so shadows are soft), tested with a shadow ray, plus an ambient term; rays that leave the scene
// see the sky gradient. The random stream is the reference's: a PCG hash seeded by the pixel and the frame,
// drawn in the same order. A wavefront traces its 64 rays together with the walk of the depth image, so its
// primary rays are a packet; after a bounce the lanes' rays go their own ways and the packet walk still
// serves them (each lane tests with its own ray).
constexpr int MAX_BOUNCES = 4;
constexpr float SURFACE_EPS = 1e-3f;

__device__ __forceinline__ uint32_t pcg_hash(const uint32_t x) {
    const uint32_t state = x * 747796405u + 2891336453u;
    const uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (word >> 22u) ^ word;
}
__device__ __forceinline__ float rand01(uint32_t &state) {
    state = pcg_hash(state);
    return (float)state * 2.3283064365386963e-10f;
}
__device__ __forceinline__ float saturate(const float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }
__device__ __forceinline__ float3 mul3v(const float3 a, const float3 b) { return mk3(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ float3 reflect3(const float3 i, const float3 n) { return sub3(i, mul3(n, 2.0f * dot3(i, n))); }
__device__ __forceinline__ float3 offset_origin(const float3 p, const float3 n, const float3 dir) {
    return add3(p, mul3(n, dot3(dir, n) < 0.0f ? -SURFACE_EPS : SURFACE_EPS));
}
__device__ __forceinline__ float3 sky(const ShadeScene &E, const float3 dir) {
    const float t = saturate(dot3(dir, E.sky_up) * 0.5f + 0.5f);
    return mul3(add3(E.sky_color_down, mul3(sub3(E.sky_color_up, E.sky_color_down), t)), E.sky_intensity);
}
// geom_dev.h:141-152: a uniform direction, then a point on the light's sphere. The two random numbers are drawn
// whatever the radius; a point light (radius 0, the same for every lane) is its centre, which is what adding the
// finite unit vector times 0 gives, so its sine and cosine are not evaluated.
__device__ __forceinline__ float3 sample_sphere_light(const float3 c, const float radius, uint32_t &rng) {
    const float u = rand01(rng), v = rand01(rng);
    if (radius == 0.0f) return c;
    const float z = 1.0f - 2.0f * u;
    const float rad = sqrtf(fmaxf(0.0f, 1.0f - z * z));
    const float phi = 6.28318530718f * v;
    return add3(c, mul3(mk3(rad * cosf(phi), rad * sinf(phi), z), radius));
}
// device_scene.h:98-111
__device__ __forceinline__ float light_factor(const float4 q, const float4 dir, const float3 towards, const float d) {
    float f = 1.0f;
    if (q.y > 0.0f) {
        const float r = d / q.y;
        f = 1.0f / (1.0f + r * r);
    }
    if (q.z > -1.5f) {
        const float c = -(dir.x * towards.x + dir.y * towards.y + dir.z * towards.z);
        const float t = fminf(fmaxf((c - q.z) / fmaxf(q.w - q.z, 1e-6f), 0.0f), 1.0f);
        f *= t * t * (3.0f - 2.0f * t);
    }
    return f;
}

// Whether anything lies between o and o + max_dist d, for the lanes in live (render_core.h:146-160).
template <int WALK, class Walk>
__device__ __forceinline__ bool occluded(const Scene S, PairLds *L, const int world, const float3 o, const float3 d,
                                         const uint64_t live, const float max_dist) {
    const bool mine = in_mask(live);
    bool blocked = false;
    for (int i = 0; i < S.sphere_count(); ++i) {
        const float4 sp = sload4(S.spheres() + i);
        const float3 Lc = sub3(xyz(sp), o);
        const float tca = dot3(Lc, d);
        const float r2 = sp.w * sp.w;
        const float d2 = dot3(Lc, Lc) - tca * tca;
        if (d2 > r2) continue;
        const float thc = sqrtf(r2 - d2);
        float t = tca - thc;
        if (t < 0.0f) t = tca + thc;
        if (t >= 0.0f && t < max_dist) blocked = true;
    }
    if (fabsf(d.y) > 1e-3f) {
        const float dist = (S.floor_y() - o.y) / d.y;
        if (dist > 0.0f && dist < max_dist) {
            const float3 pt = add3(o, mul3(d, dist));
            if (fabsf(pt.x) < S.floor_hx() && pt.z > S.floor_zmin() && pt.z < S.floor_zmax()) blocked = true;
        }
    }
    // the walk limited to max_dist, stopping each ray at its first hit: it finds a hit exactly when the
    // reference's any-hit walk does (mesh_dev.h:208-227)
    const uint64_t rest = ballot(mine && !blocked);
    if (rest != 0) {
        float best = max_dist;
        LaneHit h;
        Walk stats;
        if (WALK != WALK_LANES) {
            const int lane = lane_id();
            L->hit[lane].x = -1;
            wave_lds_order();
            trace_world<blas_mode<WALK>()>(S, L, world, o, d, rest, best, h, stats);
            wave_lds_order();
            if (in_mask(rest) && L->hit[lane].x >= 0) blocked = true;
        } else {
            h.inst = -1;
            trace_world_lanes(S, world, o, d, in_mask(rest), best, h, stats);
            if (in_mask(rest) && h.inst >= 0) blocked = true;
        }
    }
    return mine && blocked;
}

__device__ __forceinline__ float3 camera_ray_at(const Cam &c, const float fov_scale, const float aspect, const float px, const float py,
                                                const int width, const int height) {
    const float sx = (2.0f * px / (float)width - 1.0f) * fov_scale * aspect;
    const float sy = -(2.0f * py / (float)height - 1.0f) * fov_scale;
    return normalize3(add3(add3(mul3(c.right, sx), mul3(c.up, sy)), c.fwd));
}

// srgb_channel (geom_dev.h:169-172). The reference's GPU path takes x^(1/2.4) with a reduced-precision pow
// (geom_dev.h:87-94); here it is 2^(log2(x) / 2.4) through the hardware base-2 logarithm and exponential, a few ulp
// from powf, so the byte it rounds to differs from powf's only for values within about 2e-4 of a rounding boundary
// (the 8-body falling-bodies scene's RGB kernel: 3.45 ms with powf, 3.08 ms so)
__device__ __forceinline__ float srgb_channel(const float v) {
    const float x = saturate(v);
    return x <= 0.0031308f ? 12.92f * x : 1.055f * exp2f(__log2f(x) * (1.0f / 2.4f)) - 0.055f;
}

// The pixel's random stream, seeded by the pixel and the frame (geom_dev.h:122-126).
__device__ __forceinline__ uint32_t pixel_stream(const RenderArgs &A, const TilePixel &p, const int frame) {
    return pcg_hash((uint32_t)(p.y * A.width + p.x) ^ pcg_hash((uint32_t)frame + 1u));
}
// The pixel's bytes from the sum of its samples (render_core.h:276-283), red in the low byte.
__device__ __forceinline__ uint32_t rgb_bytes(const RgbArgs &G, const float3 sum) {
    const float3 c = mul3(sum, 1.0f / (float)G.spp);
    const uint32_t r = (uint32_t)(saturate(srgb_channel(c.x)) * 255.0f + 0.5f);
    const uint32_t g = (uint32_t)(saturate(srgb_channel(c.y)) * 255.0f + 0.5f);
    const uint32_t b = (uint32_t)(saturate(srgb_channel(c.z)) * 255.0f + 0.5f);
    return r | g << 8 | b << 16;
}
__device__ __forceinline__ void store_rgb(const RgbArgs &G, const size_t index, const uint32_t bytes) {
    uint8_t *out = G.rgb + 3 * index;
    out[0] = (uint8_t)bytes;
    out[1] = (uint8_t)(bytes >> 8);
    out[2] = (uint8_t)(bytes >> 16);
}
__device__ __forceinline__ void write_rgb(const RgbArgs &G, const size_t index, const float3 sum) {
    store_rgb(G, index, rgb_bytes(G, sum));
}

// A hit's point, surface normal and material records (render_core.h:206-214): the instance's template material,
// the floor's checker tint, or the sphere's material.
__device__ __forceinline__ void hit_material(const RgbArgs &G, const int kind, const float3 o, const float3 d, const float best,
                                             const LaneHit &h, float3 &point, float3 &normal, float4 &m0, float4 &m1) {
    const ShadeScene &E = G.shade;
    point = add3(o, mul3(d, best));
    int object;
    surface(Scene(), kind, o, d, best, h, normal, object);
    if (kind == OBJECT_INSTANCE) {
        const float4 *mp = E.instance_materials + 2 * (size_t)Scene().inst()[h.inst].tmpl;
        m0 = mp[0];
        m1 = mp[1];
    } else if (kind == OBJECT_FLOOR) {
        m0 = E.floor_material[0];
        m1 = E.floor_material[1];
        const int cx = (int)floorf(point.x * E.floor_checker_scale), cz = (int)floorf(point.z * E.floor_checker_scale);
        const float3 tint = ((cx + cz) & 1) ? mk3(1.0f, 1.0f, 1.0f) : mk3(1.0f, 0.7f, 0.3f);
        m0.x = tint.x * 0.3f;
        m0.y = tint.y * 0.3f;
        m0.z = tint.z * 0.3f;
    } else {
        const float4 *mp = E.sphere_materials + 2 * (size_t)(kind - OBJECT_SPHERE);
        m0 = mp[0];
        m1 = mp[1];
    }
}

// Light i at a lane's hit (render_core.h:215-233): its sample point drawn from rng, the direction and distance to
// it, and the diffuse (cd) and specular (cs) light it adds if nothing blocks it. The light's terms come first:
// where both are zero (a surface facing away from the light, and no highlight) adding them changes nothing whether
// or not the light is blocked (the sums start at +0 and only grow), so the result says whether the lane needs a
// shadow ray at all.
__device__ __forceinline__ bool light_terms(const ShadeScene &E, const int i, const bool hit, const float3 point, const float3 normal,
                                            const float3 d, const float4 m1, uint32_t &rng, float3 &cd, float3 &cs,
                                            float3 &light_dir, float &light_distance) {
    const float4 lp0 = E.lights[4 * i], lq = E.lights[4 * i + 1], ldir = E.lights[4 * i + 2], lcol = E.lights[4 * i + 3];
    light_dir = mk3(0.0f, 1.0f, 0.0f);
    light_distance = 0.0f;
    float strength = 0.0f;
    if (hit) {
        const float3 lp = sample_sphere_light(xyz(lp0), lq.x, rng);
        const float3 to_light = sub3(lp, point);
        light_distance = sqrtf(dot3(to_light, to_light));
        light_dir = mul3(to_light, rcp_rn(light_distance));
        strength = lp0.w * light_factor(lq, ldir, light_dir, light_distance);
    }
    const bool test = hit && strength > 0.0f;
    cd = mk3(0.0f, 0.0f, 0.0f);
    cs = cd;
    if (test) {
        const float3 lit = mul3(xyz(lcol), strength);
        cd = mul3(lit, fmaxf(0.0f, dot3(light_dir, normal)));
        cs = mul3(lit, powf(fmaxf(0.0f, dot3(reflect3(light_dir, normal), d)), m1.z));
    }
    return test && (cd.x != 0.0f || cd.y != 0.0f || cd.z != 0.0f || cs.x != 0.0f || cs.y != 0.0f || cs.z != 0.0f);
}

// A hit's light from the summed unblocked terms and the ambient term (render_core.h:234-237), added to radiance.
__device__ __forceinline__ void add_direct(const ShadeScene &E, const float4 m0, const float4 m1, const float3 diffuse,
                                           const float3 specular, const float throughput, float3 &radiance) {
    const float3 dc = xyz(m0);
    const float3 direct = add3(mul3v(dc, mul3(diffuse, m0.w)), mul3(specular, m1.x));
    radiance = add3(radiance, mul3(add3(direct, mul3(dc, E.ambient * m0.w)), throughput));
}

// What one traced segment of a path adds (render_core.h:206-240): the lanes in active traced o + t d, and kind
// says what each hit (OBJECT_NONE: nothing, so the sky), best and h where. radiance and throughput accumulate as
// in the reference; active is cleared where the path ends, and elsewhere o and d become the mirror bounce. Every
// lane of the wavefront calls it (the shadow walk is a wavefront's); Shadow is the shadow rays' walk.
template <int WALK, class Shadow>
__device__ __forceinline__ void shade_hit(const RgbArgs &G, PairLds *L, const int world, const int kind, const float best,
                                          const LaneHit &h, bool &active, float3 &o, float3 &d, uint32_t &rng,
                                          float3 &radiance, float &throughput) {
    const ShadeScene &E = G.shade;
    const bool hit = active && kind != OBJECT_NONE;
    if (active && !hit) {
        radiance = add3(radiance, mul3(sky(E, d), throughput));
        active = false;
    }
    float3 normal = mk3(0.0f, 1.0f, 0.0f), point = o;
    float4 m0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), m1 = m0;
    if (hit) hit_material(G, kind, o, d, best, h, point, normal, m0, m1);
    float3 diffuse = mk3(0.0f, 0.0f, 0.0f), specular = mk3(0.0f, 0.0f, 0.0f);
    for (int i = 0; i < E.light_count; ++i) {
        float3 cd, cs, light_dir;
        float light_distance;
        const bool need = light_terms(E, i, hit, point, normal, d, m1, rng, cd, cs, light_dir, light_distance);
        // a wave with no lane needing a shadow ray skips the walk
        const uint64_t shadow = ballot(need);
        if (!shadow) continue;
        const bool blocked = occluded<WALK, Shadow>(Scene(), L, world, offset_origin(point, normal, light_dir), light_dir, shadow,
                                                    light_distance);
        if (need && !blocked) {
            diffuse = add3(diffuse, cd);
            specular = add3(specular, cs);
        }
    }
    if (hit) {
        add_direct(E, m0, m1, diffuse, specular, throughput, radiance);
        throughput *= m1.y;
        if (throughput < MIN_THROUGHPUT) {
            active = false;
        } else {
            d = reflect3(d, normal);
            o = offset_origin(point, normal, d);
        }
    }
}

// The packet and hybrid walks' RGB kernels are built at 4, 5, 6 and 7 workgroups per compute unit, the per-lane
// walk's at 4; the autotuner picks.
// TWO_CHILD: the paths themselves with the two-child walk below instances, as the shadow rays (OneBoxRays otherwise).
template <int WALK, bool TWO_CHILD>
__device__ __forceinline__ void rgb_tile(const RgbArgs &G, PairLds *L, const long long tile) {
    using Rays = std::conditional_t<TWO_CHILD, NoStats, OneBoxRays>;
    const RenderArgs &A = G.r;
    const TilePixel p = tile_pixel(A, tile);
    ViewOfRays view;
    const Cam cam = camera_of(A, p.view, p.world, view);
    uint32_t rng = pixel_stream(A, p, G.frame);
    float3 sum = mk3(0.0f, 0.0f, 0.0f);
    for (int sample = 0; sample < G.spp; ++sample) {
        const float jx = rand01(rng), jy = rand01(rng);
        float3 o = cam.pos;
        float3 d = camera_ray_at(cam, A.fov_scale, A.aspect, (float)p.x + jx, (float)p.y + jy, A.width, A.height);
        float3 radiance = mk3(0.0f, 0.0f, 0.0f);
        float throughput = 1.0f;
        bool active = p.valid;
        for (int depth = 0; ballot(active); ++depth) {
            float best = 0.0f;
            LaneHit h;
            Rays stats;
            int kind = OBJECT_NONE;
            if (depth <= MAX_BOUNCES) kind = scene_hit<WALK>(Scene(), L, p.world, o, d, ballot(active), best, h, stats);
            shade_hit<WALK, Occlusion>(G, L, p.world, kind, best, h, active, o, d, rng, radiance, throughput);
        }
        sum = add3(sum, radiance);
    }
    if (p.valid) write_rgb(G, p.index, sum);
}

template <int WALK, int BLOCKS, bool TWO_CHILD = false>
__global__ __launch_bounds__(256, BLOCKS) void rgb_kernel(const RgbArgs G) {
    NGX_PAIR_LDS(L);
    const long long tile = wave_tile(G.r.xcd_remap, G.r.total_tiles);
    if (tile >= G.r.total_tiles) return;
    rgb_tile<WALK, TWO_CHILD>(G, L, tile);
}

// The same tiles from a fixed grid taking them from the per-XCD slice counters, as the persistent depth
// kernel does.
template <int WALK, int BLOCKS, bool TWO_CHILD = false>
__global__ __launch_bounds__(256, BLOCKS) void rgb_persistent_kernel(const RgbArgs G) {
    NGX_PAIR_LDS(L);
    take_tiles(G.r.tile_counters, G.r.next_counters, G.r.total_tiles, [&](const long long tile) { rgb_tile<WALK, TWO_CHILD>(G, L, tile); });
}

// The picture in two passes, for one sample a pixel where no surface reflects (every reflectivity below
// MIN_THROUGHPUT, so every path ends at its first segment). The first pass traces the jittered camera rays alone,
// with the depth kernel's walk and register budget, and keeps each pixel's hit (16 bytes, and 8 more of
// barycentrics when a mesh has vertex normals); the second draws the same ray and random numbers again and shades
// the hit as the one-pass kernel does, shadow rays and all, so the bytes are the same.
template <int WALK>
__device__ __forceinline__ void rgb_hit_tile(const RgbArgs &G, PairLds *L, const long long tile) {
    const RenderArgs &A = G.r;
    const TilePixel p = tile_pixel(A, tile);
    CameraRays stats;
    const Cam cam = camera_of(A, p.view, p.world, stats);
    uint32_t rng = pixel_stream(A, p, G.frame);
    const float jx = rand01(rng), jy = rand01(rng);
    const float3 d = camera_ray_at(cam, A.fov_scale, A.aspect, (float)p.x + jx, (float)p.y + jy, A.width, A.height);
    float best;
    LaneHit h;
    const int kind = scene_hit<WALK>(Scene(), L, p.world, cam.pos, d, ballot(p.valid), best, h, stats);
    if (!p.valid) return;
    G.hits[p.index] = make_int4(__float_as_int(best), kind, h.inst, h.tri);
    if (G.hit_uv != nullptr) G.hit_uv[p.index] = kind == OBJECT_INSTANCE ? make_float2(h.u, h.v) : make_float2(0.0f, 0.0f);
}

// The ray, its random numbers and its hit as the first pass traced them.
struct ShadeStart {
    TilePixel p;
    uint32_t rng;
    float3 o, d;
    int kind;
    float best;
    LaneHit h;
};
__device__ __forceinline__ ShadeStart shade_start(const RgbArgs &G, const long long tile) {
    const RenderArgs &A = G.r;
    ShadeStart q;
    q.p = tile_pixel(A, tile);
    ViewOfRays view;
    const Cam cam = camera_of(A, q.p.view, q.p.world, view);
    q.rng = pixel_stream(A, q.p, G.frame);
    const float jx = rand01(q.rng), jy = rand01(q.rng);
    q.o = cam.pos;
    q.d = camera_ray_at(cam, A.fov_scale, A.aspect, (float)q.p.x + jx, (float)q.p.y + jy, A.width, A.height);
    q.kind = OBJECT_NONE;
    q.best = 0.0f;
    q.h.inst = -1;
    q.h.tri = -1;
    q.h.u = 0.0f;
    q.h.v = 0.0f;
    if (q.p.valid) {
        const int4 r = G.hits[q.p.index];
        q.best = __int_as_float(r.x);
        q.kind = r.y;
        q.h.inst = r.z;
        q.h.tri = r.w;
        if (G.hit_uv != nullptr) {
            const float2 uv = G.hit_uv[q.p.index];
            q.h.u = uv.x;
            q.h.v = uv.y;
        }
    }
    return q;
}

template <int WALK>
__device__ __forceinline__ void rgb_shade_tile(const RgbArgs &G, PairLds *L, const long long tile) {
    ShadeStart q = shade_start(G, tile);
    float3 radiance = mk3(0.0f, 0.0f, 0.0f);
    float throughput = 1.0f;
    bool active = q.p.valid;
    shade_hit<WALK, Occlusion>(G, L, q.p.world, q.kind, q.best, q.h, active, q.o, q.d, q.rng, radiance, throughput);
    if (q.p.valid) write_rgb(G, q.p.index, add3(mk3(0.0f, 0.0f, 0.0f), radiance));
}

// The same pass for a scene of one light. With one light and one segment a pixel takes one of two colours: the
// one with the light's terms added, if its shadow ray is not blocked, and the one without. Both are worked out
// (as shade_hit sums them) and encoded before the shadow walk, so two words, not the shading state, are what a
// lane holds across it, and the kernel fits in fewer registers.
template <int WALK>
__device__ __forceinline__ void rgb_shade_one_light_tile(const RgbArgs &G, PairLds *L, const long long tile) {
    const ShadeScene &E = G.shade;
    const ShadeStart q = shade_start(G, tile);
    const float throughput = 1.0f;
    const bool hit = q.p.valid && q.kind != OBJECT_NONE;
    float3 radiance = mk3(0.0f, 0.0f, 0.0f);
    if (q.p.valid && !hit) radiance = add3(radiance, mul3(sky(E, q.d), throughput));
    float3 normal = mk3(0.0f, 1.0f, 0.0f), point = q.o;
    float4 m0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), m1 = m0;
    if (hit) hit_material(G, q.kind, q.o, q.d, q.best, q.h, point, normal, m0, m1);
    uint32_t rng = q.rng;
    float3 cd, cs, light_dir;
    float light_distance;
    const bool need = light_terms(E, 0, hit, point, normal, q.d, m1, rng, cd, cs, light_dir, light_distance);
    const float3 zero = mk3(0.0f, 0.0f, 0.0f);
    float3 dark = radiance, lit = radiance;
    if (hit) {
        add_direct(E, m0, m1, zero, zero, throughput, dark);
        add_direct(E, m0, m1, add3(zero, cd), add3(zero, cs), throughput, lit);
    }
    const uint32_t dark_bytes = rgb_bytes(G, add3(zero, dark));
    const uint32_t lit_bytes = rgb_bytes(G, add3(zero, lit));
    const uint64_t shadow = ballot(need);
    bool blocked = false;
    if (shadow)
        blocked = occluded<WALK, Occlusion>(Scene(), L, q.p.world, offset_origin(point, normal, light_dir), light_dir, shadow,
                                                    light_distance);
    if (q.p.valid) store_rgb(G, q.p.index, need && !blocked ? lit_bytes : dark_bytes);
}

template <int WALK, int BLOCKS>
__global__ __launch_bounds__(256, BLOCKS) void rgb_hit_kernel(const RgbArgs G) {
    NGX_PAIR_LDS(L);
    take_tiles(G.r.tile_counters, G.r.next_counters, G.r.total_tiles, [&](const long long tile) { rgb_hit_tile<WALK>(G, L, tile); });
}

// ONE_LIGHT: the scene has exactly one light (the kernel built for it holds less across the shadow walk).
template <int WALK, int BLOCKS, bool ONE_LIGHT>
__global__ __launch_bounds__(256, BLOCKS) void rgb_shade_kernel(const RgbArgs G) {
    NGX_PAIR_LDS(L);
    take_tiles(G.r.tile_counters, G.r.next_counters, G.r.total_tiles, [&](const long long tile) {
        if constexpr (ONE_LIGHT) rgb_shade_one_light_tile<WALK>(G, L, tile);
        else rgb_shade_tile<WALK>(G, L, tile);
    });
}

// Ray queries (render_core.h:331-349): 64 consecutive rays a wave (with xcd_remap, each XCD takes a
// contiguous range of the waves, so the rays an XCD holds at once are neighbours in the direction order); a
// wave whose rays fall in several worlds walks each world's rays as its own packet.
// 6 workgroups (24 wavefronts) per compute unit, at most 84 VGPRs: the ray queries wait on memory more than the
// render does, and a sixth wavefront per SIMD hides more of it (lidar_sweeps 22.7 -> 21.5 ms; 7 gives 22.6)
// (built at 5, 6 and 7 for the packet and hybrid walks, the autotuner picking; the per-lane walk's at 6)
struct QueryRay {
    long long i;  // the ray's place in the caller's arrays
    float3 o, d;
    bool ok;      // its direction can be normalized
};
// The ray of a slot: the slot itself, or the world's ray at that place in the direction order. The arguments are read
// again here, so a ray is read twice, before its walk and for its results, rather than held in seven registers between.
__device__ __forceinline__ QueryRay query_ray(const long long slot, const int world) {
    const auto &A = kernel_args<RayArgs>();
    const int *const order = in_global(A.order);
    QueryRay q;
    q.i = order ? (long long)world * A.rays_per_world + order[slot] : slot;
    const float *const po = in_global(A.origins) + 3 * q.i, *const pd = in_global(A.dirs) + 3 * q.i;
    q.o = mk3(po[0], po[1], po[2]);
    q.d = mk3(pd[0], pd[1], pd[2]);
    const float len2 = dot3(q.d, q.d);
    q.ok = len2 > 1e-30f && len2 < 1e30f;
    if (q.ok) q.d = mul3(q.d, rcp_rn(sqrtf(len2)));
    return q;
}
__device__ __forceinline__ void store_ray(const long long slot, const int world, const int kind, const float best, const LaneHit &h) {
    const QueryRay q = query_ray(slot, world);
    const auto &A = kernel_args<RayArgs>();
    const bool found = kind != OBJECT_NONE && best <= A.max_distance;
    float3 normal = mk3(0.0f, 0.0f, 0.0f);
    int object = OBJECT_NONE;
    if (found) surface(Scene(), kind, q.o, q.d, best, h, normal, object);
    in_global(A.distance)[q.i] = found ? best : __int_as_float(0x7f800000);
    float *const n = in_global(A.normal) + 3 * q.i;
    n[0] = normal.x;
    n[1] = normal.y;
    n[2] = normal.z;
    in_global(A.object_id)[q.i] = object;
}

template <int WALK, int BLOCKS>
__global__ __launch_bounds__(256, BLOCKS) void ray_kernel(const RayArgs A) {
    NGX_PAIR_LDS(L);
    const long long base = wave_tile(A.xcd_remap, 0) * A.lanes;
    if (base >= A.count) return;
    const long long slot = base + lane_id();
    const bool valid = lane_id() < A.lanes && slot < A.count;
    const int world = valid ? (int)(slot / A.rays_per_world) : -1;
    float3 o = mk3(0.0f, 0.0f, 0.0f), d = mk3(0.0f, 0.0f, 1.0f);
    bool ok = false;
    LaneHit h;
    h.inst = -1;
    h.tri = -1;
    if (valid) {
        const QueryRay q = query_ray(slot, world);
        o = q.o;
        d = q.d;
        ok = q.ok;
        if (!ok) store_ray(slot, world, OBJECT_NONE, 0.0f, h);
    }
    float best;
    NoStats stats;
    if (WALK != WALK_LANES) {
        uint64_t pending = ballot(ok);
        while (pending != 0) {
            const int w = __builtin_amdgcn_readlane(world, first_lane(pending));
            const uint64_t mine = ballot(ok && world == w);
            const int kind = scene_hit<WALK>(Scene(), L, w, o, d, mine, best, h, stats);
            if (in_mask(mine)) store_ray(slot, w, kind, best, h);
            pending &= ~mine;
        }
    } else {
        // each lane walks its own world
        const int kind = scene_hit<WALK_LANES>(Scene(), L, world, o, d, ballot(ok), best, h, stats);
        if (ok) store_ray(slot, world, kind, best, h);
    }
}

// ------------------------------------------------------------------------------ backward --
//
// d(depth)/d(pose) through the fixed hit triangle: a pose change that moves the material point the ray
// hit by dX moves the hit distance by n.dX / n.d, n being the triangle's world normal (any scale). With
// X = Rb y + pb (y the point in its body's frame), dL/dpb = a and dL/dq_unit = a^T (dR/dq_unit) y, where
// a = dL/dt * n / n.d; the projection onto the raw quaternion is applied once per body afterwards.

// The 7 gradient terms of one lane's hit: returns false when the hit does not depend on a body pose.
__device__ __forceinline__ bool hit_pose_terms(const Scene S, const int world, const int bodies_per_world,
                                               const int *body_of_instance, const float *local_rot_scale, const float *body_poses,
                                               const float3 o, const float3 d, const LaneHit &h, const float dl_dt,
                                               int &body, float g[7]) {
    const InstanceRec &rec = S.inst()[h.inst];
    body = body_of_instance[rec.tmpl];
    if (body < 0) return false;
    const float3 r0 = xyz(rec.inv[0]), r1 = xyz(rec.inv[1]), r2 = xyz(rec.inv[2]);
    float3 v0, e1, e2;
    load_tri(S.tris(), (size_t)h.tri, v0, e1, e2);
    const float3 nl = cross3(e1, e2);
    const float3 n = add3(add3(mul3(r0, nl.x), mul3(r1, nl.y)), mul3(r2, nl.z));
    const float nd = dot3(n, d);
    if (nd == 0.0f) return false;
    const float s = dl_dt / nd;
    const float3 a = mul3(n, s);
    // the hit's point in mesh space, then in the body's frame: y = Rl diag(s) x + pl
    const float3 x = add3(add3(v0, mul3(e1, h.u)), mul3(e2, h.v));
    const float *L = local_rot_scale + 12 * (size_t)rec.tmpl;
    const float3 y = mk3(L[0] * x.x + L[1] * x.y + L[2] * x.z + L[3], L[4] * x.x + L[5] * x.y + L[6] * x.z + L[7],
                         L[8] * x.x + L[9] * x.y + L[10] * x.z + L[11]);
    const float *bp = body_poses + 7 * ((size_t)world * bodies_per_world + body);
    const float q0 = bp[3], q1 = bp[4], q2 = bp[5], q3 = bp[6];
    const float qn = sqrtf(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3);
    const float qx = q0 / qn, qy = q1 / qn, qz = q2 / qn, qw = q3 / qn;
    g[0] = a.x;
    g[1] = a.y;
    g[2] = a.z;
    // a^T (dR/dq_k) y for the unit quaternion's components, R as in instances.cpp:130-132
    const float ax = a.x, ay = a.y, az = a.z, yx = y.x, yy = y.y, yz = y.z;
    g[3] = ax * (2 * qy * yy + 2 * qz * yz) + ay * (2 * qy * yx - 4 * qx * yy - 2 * qw * yz) +
           az * (2 * qz * yx + 2 * qw * yy - 4 * qx * yz);
    g[4] = ax * (-4 * qy * yx + 2 * qx * yy + 2 * qw * yz) + ay * (2 * qx * yx + 2 * qz * yz) +
           az * (-2 * qw * yx + 2 * qz * yy - 4 * qy * yz);
    g[5] = ax * (-4 * qz * yx - 2 * qw * yy + 2 * qx * yz) + ay * (2 * qw * yx - 4 * qz * yy + 2 * qy * yz) +
           az * (2 * qx * yx + 2 * qy * yy);
    g[6] = ax * (-2 * qz * yy + 2 * qy * yz) + ay * (2 * qz * yx - 2 * qx * yz) + az * (-2 * qy * yx + 2 * qx * yy);
    return true;
}

// Adds each lane's 7 terms into acc[body][7] (this wave's own slice of LDS), one body at a time, with a
// fixed-order wave sum, so the result does not depend on scheduling.
__device__ __forceinline__ void wave_accumulate(const bool has, const int body, const float g[7], float *acc) {
    const int lane = lane_id();
    uint64_t pending = ballot(has);
    while (pending != 0) {
        const int b0 = __builtin_amdgcn_readlane(body, first_lane(pending));
        const bool mine = has && body == b0;
        const uint64_t m = ballot(mine);
        // the seven sums side by side, then one lane adds them in
        float s[7];
        for (int k = 0; k < 7; ++k) s[k] = wave_total(mine ? g[k] : 0.0f);
        if (lane == 0)
            for (int k = 0; k < 7; ++k) acc[7 * b0 + k] += s[k];
        pending &= ~m;
    }
}

constexpr int BWD_WAVES = 4;

// Built for 4, 5 and 6 workgroups per compute unit (BLOCKS) for the packet and hybrid walks, the autotuner picking, and the
// per-lane walk's for 5.
template <int WALK, int BLOCKS>
__global__ __launch_bounds__(64 * BWD_WAVES, BLOCKS) void depth_backward_kernel(const DepthBackwardArgs A) {
    extern __shared__ float acc_all[];  // [BWD_WAVES][bodies][7]
    NGX_PAIR_LDS(L);
    const int view = blockIdx.x / A.parts, part = blockIdx.x % A.parts;
    const int wave = uniform(threadIdx.x >> 6), lane = lane_id();
    const int B = A.bodies_per_world;
    float *acc = acc_all + (size_t)wave * B * 7;
    for (int i = lane; i < B * 7; i += 64) acc[i] = 0.0f;
    const int world = view / A.cameras_per_world;
    const Cam cam = load_camera(A.cams + 12 * (size_t)view);
    for (int t = part * BWD_WAVES + wave; t < A.tiles; t += A.parts * BWD_WAVES) {
        const int ty = t / A.tiles_x, row = lane >> A.tile_w_log2;
        const int x = ((t - ty * A.tiles_x) << A.tile_w_log2) + (lane & ((1 << A.tile_w_log2) - 1)), y = ty * A.tile_h + row;
        const bool valid = row < A.tile_h && x < A.width && y < A.height;
        const size_t idx = ((size_t)view * A.height + (valid ? y : 0)) * A.width + (valid ? x : 0);
        const float3 d = pixel_ray(cam, A.fov_scale, A.aspect, x, y, A.width, A.height);
        const float depth = valid ? A.depth[idx] : 0.0f;
        const float gd = valid ? A.grad_depth[idx] : 0.0f;
        const float cosf_ = dot3(d, cam.fwd);
        // re-trace only rays whose forward hit something, bounded just beyond the forward's distance
        const bool want = valid && gd != 0.0f && depth < __int_as_float(0x7f800000);
        const float bound = want ? (depth / cosf_) * (1.0f + 1e-5f) + 1e-6f : 0.0f;
        float best;
        LaneHit h;
        CameraRays stats;
        const int kind = scene_hit<WALK>(Scene(), L, world, cam.pos, d, ballot(want), best, h, stats, bound);
        int body = -1;
        float g[7] = {0, 0, 0, 0, 0, 0, 0};
        bool has = false;
        if (want && kind == OBJECT_INSTANCE)
            has = hit_pose_terms(Scene(), world, B, A.body_of_instance, A.local_rot_scale, A.body_poses, cam.pos, d, h, gd * cosf_, body, g);
        wave_accumulate(has, body, g, acc);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < B * 7; i += blockDim.x) {
        float s = 0.0f;
        for (int wv = 0; wv < BWD_WAVES; ++wv) s += acc_all[(size_t)wv * B * 7 + i];
        A.partial[((size_t)view * A.parts + part) * B * 7 + i] = s;
    }
}

template <int WALK>
__global__ __launch_bounds__(64 * BWD_WAVES) void range_backward_kernel(const RangeBackwardArgs A) {
    extern __shared__ float acc_all[];
    NGX_PAIR_LDS(L);
    const int piece = blockIdx.x / A.split, part = blockIdx.x % A.split;
    const int world = piece / A.chunks, chunk = piece % A.chunks;
    const int wave = uniform(threadIdx.x >> 6), lane = lane_id();
    const int B = A.bodies_per_world;
    float *acc = acc_all + (size_t)wave * B * 7;
    for (int i = lane; i < B * 7; i += 64) acc[i] = 0.0f;
    const int R = A.rays_per_world;
    const int per = (R + A.chunks - 1) / A.chunks;
    const int r0 = chunk * per, r1 = min(R, r0 + per);
    for (int r = r0 + (part * BWD_WAVES + wave) * A.lanes; r < r1; r += A.split * BWD_WAVES * A.lanes) {
        const int ri = r + lane;
        const bool valid = lane < A.lanes && ri < r1;
        const size_t i = (size_t)world * R + (valid ? ri : r0);
        float3 o = mk3(A.origins[3 * i], A.origins[3 * i + 1], A.origins[3 * i + 2]);
        float3 d = mk3(A.dirs[3 * i], A.dirs[3 * i + 1], A.dirs[3 * i + 2]);
        const float len2 = dot3(d, d);
        const bool ok = valid && len2 > 1e-30f && len2 < 1e30f;
        if (ok) d = mul3(d, rcp_rn(sqrtf(len2)));
        const float dist = valid ? A.distance[i] : 0.0f;
        const float gd = valid ? A.grad_distance[i] : 0.0f;
        const bool want = ok && gd != 0.0f && dist < __int_as_float(0x7f800000);
        const float bound = want ? dist * (1.0f + 1e-5f) + 1e-6f : 0.0f;
        float best;
        LaneHit h;
        NoStats stats;
        const int kind = scene_hit<WALK>(Scene(), L, world, o, d, ballot(want), best, h, stats, bound);
        int body = -1;
        float g[7] = {0, 0, 0, 0, 0, 0, 0};
        bool has = false;
        if (want && kind == OBJECT_INSTANCE)
            has = hit_pose_terms(Scene(), world, B, A.body_of_instance, A.local_rot_scale, A.body_poses, o, d, h, gd, body, g);
        wave_accumulate(has, body, g, acc);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < B * 7; i += blockDim.x) {
        float s = 0.0f;
        for (int wv = 0; wv < BWD_WAVES; ++wv) s += acc_all[(size_t)wv * B * 7 + i];
        A.partial[(size_t)blockIdx.x * B * 7 + i] = s;
    }
}

// Sums the parts of each body, then projects the unit-quaternion gradient onto the raw quaternion: d unit / d q =
// (I - u u^T) / |q|. Eight lanes a body, each taking every eighth part in order, their sums added pairwise: a fixed order.
constexpr int FINISH_LANES = 8;
constexpr int FINISH_BODIES = 256 / FINISH_LANES;  // a workgroup's, of as many runs of them as the grid leaves it
constexpr long long FINISH_MOST_GROUPS = 1 << 22;
__global__ __launch_bounds__(256) void pose_grad_finish_kernel(const PoseGradFinishArgs A) {
    const long long bodies = (long long)A.worlds * A.bodies_per_world;
    const int part = threadIdx.x % FINISH_LANES;
    for (long long first = (long long)blockIdx.x * FINISH_BODIES; first < bodies; first += (long long)gridDim.x * FINISH_BODIES) {
        const long long i = first + threadIdx.x / FINISH_LANES;
        float g[7] = {0, 0, 0, 0, 0, 0, 0};
        if (i < bodies) {
            const long long w = i / A.bodies_per_world;
            const int b = (int)(i - w * A.bodies_per_world);
            for (int p = part; p < A.parts; p += FINISH_LANES) {
                const float *src = A.partial + (((size_t)w * A.parts + p) * A.bodies_per_world + b) * 7;
                for (int k = 0; k < 7; ++k) g[k] += src[k];
            }
        }
        for (int o = 1; o < FINISH_LANES; o <<= 1)
            for (int k = 0; k < 7; ++k) g[k] += __shfl_xor(g[k], o, 64);
        if (i >= bodies || part != 0) continue;
        const float *bp = A.body_poses + 7 * (size_t)i;
        const float q[4] = {bp[3], bp[4], bp[5], bp[6]};
        const float qn = sqrtf(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
        const float u[4] = {q[0] / qn, q[1] / qn, q[2] / qn, q[3] / qn};
        const float ug = u[0] * g[3] + u[1] * g[4] + u[2] * g[5] + u[3] * g[6];
        float *out = A.grad + 7 * (size_t)i;
        out[0] = g[0];
        out[1] = g[1];
        out[2] = g[2];
        for (int k = 0; k < 4; ++k) out[3 + k] = (g[3 + k] - u[k] * ug) / qn;
    }
}

}  // namespace

// A kernel variant by walk and workgroups per compute unit: the per-lane walk has one variant (LANE_BLOCKS), the
// packet and hybrid walks one per value of the kernel's list; any other value takes the default.
#define NGX_BY_VARIANT3(walk, blocks, def, lane_blocks, v0, v1, v2, launch) \
    switch (walk) { \
    case WALK_LANES: launch(WALK_LANES, lane_blocks); break; \
    case WALK_HYBRID: \
        switch (blocks ? blocks : def) { case v0: launch(WALK_HYBRID, v0); break; case v1: launch(WALK_HYBRID, v1); break; \
                                         default: launch(WALK_HYBRID, v2); break; } \
        break; \
    default: \
        switch (blocks ? blocks : def) { case v0: launch(WALK_PACKET, v0); break; case v1: launch(WALK_PACKET, v1); break; \
                                         default: launch(WALK_PACKET, v2); break; } \
        break; \
    }

// The persistent grid: as many workgroups as the device holds at once (the kernel's occupancy times the
// compute units), a multiple of 8 so every XCD gets the same number.
// No more workgroups than the tiles need (4 wavefronts each), and at least 8, one per XCD.
static int capped_grid(const int resident, const long long tiles) {
    const long long need = ((tiles + 3) / 4 + 7) / 8 * 8;
    return (int)(need < resident ? need : resident);
}

template <int WALK, int BLOCKS>
static int persistent_grid(const int compute_units, const long long tiles) {
    static const int per_cu = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, render_persistent_kernel<WALK, BLOCKS>, 256, 0) != hipSuccess || n < 1) n = 1;
        return n;
    }();
    return capped_grid((per_cu * compute_units + 7) / 8 * 8, tiles);
}

// The persistent hybrid walk by default: where the bottom levels have octant copies it is built for 8 workgroups per compute
// unit (64 VGPRs, a few spilled), which hide more of each other's waits (4096 mixed worlds 128x128: 6.79 ms at 7, 6.50 at
// 8; 64x64: 1.119 and 1.088; RGB + depth + ID: 7.40 and 7.24), and where they are too large for them, and their nodes come
// from further away, for 7 (a deforming mesh of 138,000 triangles: 397 us at 7, 415 at 8).
static bool eight_blocks(const RenderArgs &a, const int blocks) { return blocks == 0 && a.walk == WALK_HYBRID && a.s.octant_nodes > 0; }

hipError_t launch_view_tables(const ViewTableArgs &a, hipStream_t stream) {
    if (a.t.cams == nullptr) {
        if (a.counters == nullptr || a.counter_sets <= 0) return hipSuccess;
        view_tables_kernel<<<std::min(a.counter_sets * 8 * COUNTER_SLICES / 64, 64), 64, 0, stream>>>(a, 1);
        return hipGetLastError();
    }
    if (a.views < 1 || a.total < 1 || (a.counter_sets > 0 && a.counters == nullptr)) return hipErrorInvalidValue;
    // a wavefront a view for every 64 instances of the largest world, and no more than fill the chip several times over
    const int runs = std::max(1, std::min((a.max_count + 63) / 64, 65536 / a.views));
    if ((long long)a.views * runs > INT32_MAX / 64) return hipErrorInvalidValue;  // thread numbers are 31 bits
    view_tables_kernel<<<a.views * runs, 64, 0, stream>>>(a, runs);
    return hipGetLastError();
}

hipError_t launch_render(const RenderArgs &a, hipStream_t stream, const int compute_units) {
    if (a.total_tiles <= 0) return hipSuccess;
    if (a.tile_counters && compute_units > 0) {
        if (a.total_tiles >= INT32_MAX / 2) return hipErrorInvalidValue;
#define NGX_LAUNCH(W, B) render_persistent_kernel<W, B><<<persistent_grid<W, B>(compute_units, a.total_tiles), 256, 0, stream>>>(a)
        if (eight_blocks(a, a.blocks)) NGX_LAUNCH(WALK_HYBRID, 8);
        else NGX_BY_VARIANT3(a.walk, a.blocks, RENDER_BLOCKS_DEFAULT, 1, 5, 6, 7, NGX_LAUNCH)
#undef NGX_LAUNCH
        return hipGetLastError();
    }
    const long long blocks = (a.total_tiles + 3) / 4;
#define NGX_LAUNCH(W, B) render_kernel<W, B><<<(unsigned)blocks, 256, 0, stream>>>(a)
    NGX_BY_VARIANT3(a.walk, a.blocks, RENDER_BLOCKS_DEFAULT, 1, 5, 6, 7, NGX_LAUNCH)
#undef NGX_LAUNCH
    return hipGetLastError();
}

#ifdef NGX_TRACE_STATS
hipError_t launch_render_stats(const RenderArgs &a, int *out, hipStream_t stream) {
    if (a.total_tiles <= 0) return hipSuccess;
    const long long blocks = (a.total_tiles + 3) / 4;
#define NGX_LAUNCH(W) render_stats_kernel<W><<<(unsigned)blocks, 256, 0, stream>>>(a, out)
    switch (a.walk) {
    case WALK_LANES: NGX_LAUNCH(WALK_LANES); break;
    case WALK_HYBRID: NGX_LAUNCH(WALK_HYBRID); break;
    default: NGX_LAUNCH(WALK_PACKET); break;
    }
#undef NGX_LAUNCH
    return hipGetLastError();
}
#endif


template <auto KERNEL>
static int resident_grid(const int compute_units, const long long tiles) {
    static const int per_cu = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, KERNEL, 256, 0) != hipSuccess || n < 1) n = 1;
        return n;
    }();
    return capped_grid((per_cu * compute_units + 7) / 8 * 8, tiles);
}

// The RGB kernels' variants: 4, 5, 6 or 7 workgroups per compute unit for the packet and hybrid walks, 4 for the per-lane
// walk; by default 4 for the packet walk, and for the hybrid walk 4, which spills least (69 of 128 vector registers, 167 of 72
// at 7), or 7 in worlds of many instances, whose walks are long and wait for each other's (two or four samples: 64 worlds of
// 64 mirrors 128x128 6.73 ms at 4, 6.75 at 5, 7.29 at 7; 256 worlds of 40 instances 2.84, 2.97, 3.07; 1,024 worlds of 256
// mirrors 219.7, 201.5, 192.2). The line lies between the sizes where one overtakes the other: 256 worlds of mirrors 96x96 of
// 64 instances 7.75 and 7.82 ms at 4 and 7, of 80 9.98 and 9.63, of 96 11.69 and 11.36, of 128 15.01 and 14.23.
static int rgb_hybrid_blocks(const RenderArgs &a) {
    return (long long)a.s.total * a.cameras_per_world > (long long)RGB_FEW_INSTANCES * a.views ? RGB_BLOCKS_DEFAULT_HYBRID : 4;
}
#define NGX_RGB_VARIANT(walk, blocks, launch) \
    switch (walk) { \
    case WALK_LANES: launch(WALK_LANES, 4); break; \
    case WALK_HYBRID: \
        switch (blocks ? blocks : rgb_hybrid_blocks(a.r)) { case 4: launch(WALK_HYBRID, 4); break; \
            case 5: launch(WALK_HYBRID, 5); break; case 6: launch(WALK_HYBRID, 6); break; default: launch(WALK_HYBRID, 7); break; } \
        break; \
    default: \
        switch (blocks ? blocks : RGB_BLOCKS_DEFAULT_PACKET) { case 5: launch(WALK_PACKET, 5); break; \
            case 6: launch(WALK_PACKET, 6); break; case 7: launch(WALK_PACKET, 7); break; default: launch(WALK_PACKET, 4); break; } \
        break; \
    }

hipError_t launch_rgb(const RgbArgs &a, hipStream_t stream, const int compute_units) {
    if (a.r.total_tiles <= 0) return hipSuccess;
    if (a.spp < 1 || a.shade.light_count < 0 || a.shade.light_count > MAX_LIGHTS) return hipErrorInvalidValue;
    // Part wavefronts take the two-child walk for the paths too (one world of 8 mirrors at 48x48: 183 us with the one-box
    // walk, 160 so). Where two surfaces meet a ray at the same distance the walks may keep different ones (20 of 16.8 M
    // pixels of 1,024 mirror worlds), so launches of full wavefronts keep the one-box walk's, and the walk follows from the
    // tile alone: whatever variant is asked for (a.blocks), part wavefronts have this one build, persistent or not.
    const bool two_child = a.r.walk == WALK_HYBRID && a.r.tile_w * a.r.tile_h < 64;
    if (a.r.tile_counters && compute_units > 0) {
        if (a.r.total_tiles >= INT32_MAX / 2) return hipErrorInvalidValue;
#define NGX_LAUNCH(W, B) rgb_persistent_kernel<W, B><<<resident_grid<rgb_persistent_kernel<W, B>>(compute_units, a.r.total_tiles), 256, 0, stream>>>(a)
        if (two_child)
            rgb_persistent_kernel<WALK_HYBRID, RGB_TWO_CHILD_BLOCKS, true>
                <<<resident_grid<rgb_persistent_kernel<WALK_HYBRID, RGB_TWO_CHILD_BLOCKS, true>>(compute_units, a.r.total_tiles), 256, 0, stream>>>(a);
        else NGX_RGB_VARIANT(a.r.walk, a.blocks, NGX_LAUNCH)
#undef NGX_LAUNCH
        return hipGetLastError();
    }
    const long long blocks = (a.r.total_tiles + 3) / 4;
#define NGX_LAUNCH(W, B) rgb_kernel<W, B><<<(unsigned)blocks, 256, 0, stream>>>(a)
    if (two_child) rgb_kernel<WALK_HYBRID, RGB_TWO_CHILD_BLOCKS, true><<<(unsigned)blocks, 256, 0, stream>>>(a);
    else NGX_RGB_VARIANT(a.r.walk, a.blocks, NGX_LAUNCH)
#undef NGX_LAUNCH
    return hipGetLastError();
}

// The two-pass picture, persistent launches of the packet and hybrid walks only: the hit pass built like the depth
// kernel (5, 6 or 7 workgroups per compute unit: hit_blocks, 0 for the default, 8 as eight_blocks says), the shading pass
// for 4 to 7 (a.blocks, 0 for the default).
// The shading pass, built for one light where the scene has one.
template <int WALK, int BLOCKS>
static void launch_shade(const RgbArgs &a, hipStream_t stream, const int compute_units) {
    if (a.shade.light_count == 1)
        rgb_shade_kernel<WALK, BLOCKS, true><<<resident_grid<rgb_shade_kernel<WALK, BLOCKS, true>>(compute_units, a.r.total_tiles), 256, 0,
                                               stream>>>(a);
    else
        rgb_shade_kernel<WALK, BLOCKS, false><<<resident_grid<rgb_shade_kernel<WALK, BLOCKS, false>>(compute_units, a.r.total_tiles), 256,
                                                0, stream>>>(a);
}

hipError_t launch_rgb_two_pass(const RgbArgs &a, const int hit_blocks, hipStream_t stream, const int compute_units, int *shade_counters,
                               int *shade_next) {
    if (a.r.total_tiles <= 0) return hipSuccess;
    if (a.spp != 1 || a.shade.light_count < 0 || a.shade.light_count > MAX_LIGHTS || a.hits == nullptr ||
        a.r.tile_counters == nullptr || compute_units <= 0 || a.r.walk == WALK_LANES || a.r.total_tiles >= INT32_MAX / 2)
        return hipErrorInvalidValue;
    const bool hybrid = a.r.walk == WALK_HYBRID;
    const bool many = (long long)a.r.s.total * a.r.cameras_per_world >= (long long)SHADE_MANY_INSTANCES * a.r.views;
#define NGX_LAUNCH(W, B) rgb_hit_kernel<W, B><<<resident_grid<rgb_hit_kernel<W, B>>(compute_units, a.r.total_tiles), 256, 0, stream>>>(a)
    switch (hit_blocks ? hit_blocks : eight_blocks(a.r, 0) ? 8 : RENDER_BLOCKS_DEFAULT) {
    case 8: NGX_LAUNCH(WALK_HYBRID, 8); break;
    case 5: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 5); else NGX_LAUNCH(WALK_PACKET, 5); break;
    case 6: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 6); else NGX_LAUNCH(WALK_PACKET, 6); break;
    default: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 7); else NGX_LAUNCH(WALK_PACKET, 7); break;
    }
#undef NGX_LAUNCH
    RgbArgs shade = a;
    shade.r.tile_counters = shade_counters;
    shade.r.next_counters = shade_next;
#define NGX_LAUNCH(W, B) launch_shade<W, B>(shade, stream, compute_units)
    switch (a.blocks ? a.blocks : a.shade.light_count != 1 ? SHADE_BLOCKS_DEFAULT : many ? SHADE_ONE_LIGHT_BLOCKS_MANY : SHADE_ONE_LIGHT_BLOCKS_FEW) {
    case 4: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 4); else NGX_LAUNCH(WALK_PACKET, 4); break;
    case 5: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 5); else NGX_LAUNCH(WALK_PACKET, 5); break;
    case 6: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 6); else NGX_LAUNCH(WALK_PACKET, 6); break;
    default: if (hybrid) NGX_LAUNCH(WALK_HYBRID, 7); else NGX_LAUNCH(WALK_PACKET, 7); break;
    }
#undef NGX_LAUNCH
    return hipGetLastError();
}

hipError_t launch_rays(const RayArgs &a, hipStream_t stream) {
    if (a.count <= 0) return hipSuccess;
    if (a.lanes < 1 || a.lanes > 64) return hipErrorInvalidValue;
    const long long waves = (a.count + a.lanes - 1) / a.lanes;
    const long long blocks = (waves + 3) / 4;
#define NGX_LAUNCH(W, B) ray_kernel<W, B><<<(unsigned)blocks, 256, 0, stream>>>(a)
    if (a.walk == WALK_SHARED) {
        switch (a.blocks ? a.blocks : RAY_BLOCKS_DEFAULT) {
        case 5: NGX_LAUNCH(WALK_SHARED, 5); break;
        case 7: NGX_LAUNCH(WALK_SHARED, 7); break;
        default: NGX_LAUNCH(WALK_SHARED, 6); break;
        }
    } else {
        NGX_BY_VARIANT3(a.walk, a.blocks, RAY_BLOCKS_DEFAULT, 6, 5, 6, 7, NGX_LAUNCH)
    }
#undef NGX_LAUNCH
    return hipGetLastError();
}

hipError_t launch_depth_backward(const DepthBackwardArgs &a, hipStream_t stream) {
    if (a.views <= 0) return hipSuccess;
    if (a.bodies_per_world <= 0 || a.bodies_per_world > BACKWARD_MAX_BODIES) return hipErrorInvalidValue;
    const size_t lds = sizeof(float) * BWD_WAVES * 7 * (size_t)a.bodies_per_world;
#define NGX_LAUNCH(W, B) depth_backward_kernel<W, B><<<a.views * a.parts, 64 * BWD_WAVES, lds, stream>>>(a)
    const int blocks = a.bodies_per_world <= BACKWARD_FEW_BODIES ? 6 : BACKWARD_BLOCKS_MOST_LDS;
    NGX_BY_VARIANT3(a.walk, a.blocks, blocks, 5, 4, 5, 6, NGX_LAUNCH)
#undef NGX_LAUNCH
    return hipGetLastError();
}

hipError_t launch_range_backward(const RangeBackwardArgs &a, hipStream_t stream) {
    if (a.worlds <= 0 || a.chunks <= 0) return hipSuccess;
    if (a.split < 1 || a.lanes < 1 || a.lanes > 64) return hipErrorInvalidValue;
    if (a.bodies_per_world <= 0 || a.bodies_per_world > BACKWARD_MAX_BODIES) return hipErrorInvalidValue;
    const size_t lds = sizeof(float) * BWD_WAVES * 7 * (size_t)a.bodies_per_world;
#define NGX_LAUNCH(W) range_backward_kernel<W><<<a.worlds * a.chunks * a.split, 64 * BWD_WAVES, lds, stream>>>(a)
    switch (a.walk) {
    case WALK_LANES: NGX_LAUNCH(WALK_LANES); break;
    case WALK_HYBRID: NGX_LAUNCH(WALK_HYBRID); break;
    case WALK_SHARED: NGX_LAUNCH(WALK_SHARED); break;
    default: NGX_LAUNCH(WALK_PACKET); break;
    }
#undef NGX_LAUNCH
    return hipGetLastError();
}

hipError_t launch_pose_grad_finish(const PoseGradFinishArgs &a, hipStream_t stream) {
    const long long n = (long long)a.worlds * a.bodies_per_world;
    if (n <= 0) return hipSuccess;
    const long long groups = std::min((n + FINISH_BODIES - 1) / FINISH_BODIES, FINISH_MOST_GROUPS);
    pose_grad_finish_kernel<<<(unsigned)groups, 256, 0, stream>>>(a);
    return hipGetLastError();
}

// The allocation-free depth backward's partial sums (ngx_pose_backward_depth_noalloc). The name `scratch` is
// a host-side stand-in: kernels and copies take the device address that noalloc_scratch() looks up, one per
// device, since each GPU holds its own copy of the array.
static constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mutex;
static float *g_scratch_ptr[MAX_DEVICES] = {};

hipError_t noalloc_scratch(float **out) {
    *out = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(::scratch));
        if (e != hipSuccess) return e;
        if (p == nullptr) return hipErrorInvalidSymbol;
        g_scratch_ptr[dev] = static_cast<float *>(p);
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

}  // namespace ngx
