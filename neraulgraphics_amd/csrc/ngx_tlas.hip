// Top-level tree build for every world of a batch, one workgroup per world, everything in LDS.
//
// The reference builds one linear BVH over all worlds at once (src/cuda_tlas.cuh:215-306): seven
// kernels plus a device-wide radix sort of (world << 32 | morton) keys, then finds each world's root in
// the global tree. Because the world number sits above the Morton code, the sort never moves an
// instance out of its world, and the Karras hierarchy (cuda_tlas.cuh:128-159) over a world's run of
// keys depends only on those keys and on the positions used to tell equal keys apart. So this kernel
// builds each world's subtree independently, in one launch for the whole batch:
//
//   place     body pose (FP64, instances.cpp:137-164) -> matrix, inverse (cuda_tlas.cuh:35-47),
//             8-corner world box, the world's centre bounds (cuda_tlas.cuh:69-96)
//   keys      30-bit Morton code of the box centre (cuda_tlas.cuh:99-115)
//   sort      stable LSD radix sort, 4-bit digits, ranks from wave ballots (multisplit), staged in LDS; worlds of
//             up to 256 instances by counting the keys before each
//   hierarchy Karras 2012 per node, equal keys told apart by their GLOBAL positions exactly as the
//             reference's common_prefix does (cuda_tlas.cuh:119-124)
//   boxes     bottom-up union with LDS arrival counters (the fit_boxes climb, cuda_tlas.cuh:179-196); in worlds
//             of up to 256 instances, of the runs of leaves that a node's children cover
//   write     the reference's node layout at the reference's node indices, plus the 64-byte wide
//             nodes the tracer reads
//
// Node numbering is the reference's: internal nodes are numbered by sorted position, leaf k is node
// N-1+k. Inside world w (positions a..b) every internal node a < i < b is the same as in the global
// tree. The world's own root covers exactly a..b; it carries index a or index b, whichever the global
// tree does not give to the ancestor that joins this world to its neighbours, which the host decides
// once from the neighbouring world numbers (root_at_end). The ancestors joining worlds are never
// traversed (a ray starts at its world's root) and are not built.
#include "ngx_kernels.h"

namespace ngx {
namespace {

__device__ __forceinline__ int to_ordered(const float f) {
    const int i = __float_as_int(f);
    return i ^ ((i >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float from_ordered(const int i) { return __int_as_float(i ^ ((i >> 31) & 0x7fffffff)); }

__device__ __forceinline__ uint32_t spread_bits(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// Rotation of a quaternion x, y, z, w in FP64, normalized first; zero gives the identity (instances.cpp:126-133).
__device__ __forceinline__ void quat_to_matrix_d(const float *q, double r[9]) {
    double x = q[0], y = q[1], z = q[2], w = q[3];
    const double n = sqrt(x * x + y * y + z * z + w * w);
    if (n > 0.0) {
        x /= n; y /= n; z /= n; w /= n;
    } else {
        x = y = z = 0.0; w = 1.0;
    }
    r[0] = 1 - 2 * (y * y + z * z); r[1] = 2 * (x * y - z * w);     r[2] = 2 * (x * z + y * w);
    r[3] = 2 * (x * y + z * w);     r[4] = 1 - 2 * (x * x + z * z); r[5] = 2 * (y * z - x * w);
    r[6] = 2 * (x * z - y * w);     r[7] = 2 * (y * z + x * w);     r[8] = 1 - 2 * (x * x + y * y);
}

// An instance's matrix from its body's pose, its own offset and its scale, in FP64 and rounded once, as the
// reference's host does (instances.cpp:137-164); the reference's GPU path composes in FP32.
__device__ void compose_body_pose(const float *body, const float *local, const float *scale, float *m) {
    double rl[9], r[9], p[3] = {local[0], local[1], local[2]};
    quat_to_matrix_d(local + 3, rl);
    if (body == nullptr) {
        for (int k = 0; k < 9; ++k) r[k] = rl[k];
    } else {
        double rb[9];
        quat_to_matrix_d(body + 3, rb);
        for (int row = 0; row < 3; ++row) {
            for (int col = 0; col < 3; ++col)
                r[3 * row + col] = rb[3 * row] * rl[col] + rb[3 * row + 1] * rl[3 + col] + rb[3 * row + 2] * rl[6 + col];
            p[row] = (double)body[row] + rb[3 * row] * (double)local[0] + rb[3 * row + 1] * (double)local[1] +
                     rb[3 * row + 2] * (double)local[2];
        }
    }
    for (int row = 0; row < 3; ++row) {
        for (int col = 0; col < 3; ++col) m[4 * row + col] = (float)(r[3 * row + col] * (double)scale[col]);
        m[4 * row + 3] = (float)p[row];
    }
}

__device__ __forceinline__ void invert_affine(const float *m, float *out) {
    const float c00 = m[5] * m[10] - m[6] * m[9];
    const float c01 = m[6] * m[8] - m[4] * m[10];
    const float c02 = m[4] * m[9] - m[5] * m[8];
    const float inv = 1.0f / (m[0] * c00 + m[1] * c01 + m[2] * c02);
    const float r[9] = {c00 * inv, (m[2] * m[9] - m[1] * m[10]) * inv, (m[1] * m[6] - m[2] * m[5]) * inv,
                        c01 * inv, (m[0] * m[10] - m[2] * m[8]) * inv, (m[2] * m[4] - m[0] * m[6]) * inv,
                        c02 * inv, (m[1] * m[8] - m[0] * m[9]) * inv, (m[0] * m[5] - m[1] * m[4]) * inv};
    for (int row = 0; row < 3; ++row) {
        for (int col = 0; col < 3; ++col) out[4 * row + col] = r[3 * row + col];
        out[4 * row + 3] = -(r[3 * row] * m[3] + r[3 * row + 1] * m[7] + r[3 * row + 2] * m[11]);
    }
}

// A wavefront's least and greatest value, every lane active: one DPP instruction a stage, as wave_prefix_sum's, and a lane
// shifted in from outside the row keeps its own.
template <class Pick>
__device__ __forceinline__ int wave_pick(int v, const Pick &pick) {
    v = pick(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false));  // row_shr:1
    v = pick(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false));  // row_shr:2
    v = pick(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false));  // row_shr:4
    v = pick(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xf, 0xf, false));  // row_shr:8
    v = pick(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = pick(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_min(const int v) { return wave_pick(v, [](const int x, const int y) { return min(x, y); }); }
__device__ __forceinline__ int wave_max(const int v) { return wave_pick(v, [](const int x, const int y) { return max(x, y); }); }

// Exclusive scan of data[0 .. count) in place, count <= blockDim.x; wave_tot has one slot per wave.
__device__ void block_exclusive_scan(int *data, const int count, int *wave_tot) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int x = tid < count ? data[tid] : 0;
    const int incl = wave_prefix_sum(x);
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += wave_tot[w];
    if (tid < count) data[tid] = base + incl - x;
    __syncthreads();
}

// ---- pieces shared by the workgroup build and the device-wide build

// Places instance i of world w (global index g): its matrix as given or composed from its body, the
// inverse the tracer reads, and its world box (the 8 corners of the mesh box, cuda_tlas.cuh:69-96).
__device__ void place_instance(const TlasBuildArgs &A, const int w, const int i, const int g, float lo[3], float hi[3]) {
    // the mesh's values first, so their loads, one after another, run beside the pose's
    const int mesh = A.tmpl_mesh[i];
    float lb[6];
    for (int k = 0; k < 6; ++k) lb[k] = A.mesh_bounds[6 * mesh + k];
    const int mesh_tris = A.mesh_tris[mesh], skip_root = A.mesh_skip_root[mesh];
    float m[12];
    if (A.source == SOURCE_BODIES) {
        const int b = A.body_of_instance[i];
        const float *body = b < 0 ? nullptr : A.body_poses + 7 * ((size_t)w * A.bodies_per_world + b);
        compose_body_pose(body, A.local_pose + 7 * i, A.scale + 3 * i, m);
    } else if (A.source == SOURCE_GEOMS) {
        // R diag(s) | p from FP32 inputs, one FP32 product an element, as the reference's MuJoCo Warp compose
        // kernel does (python/neraulgraphics/mujoco.py:276-287).
        const size_t gw = (size_t)w * A.geoms_per_world + A.geom_of_instance[i];
        const float *p = A.geom_pos + 3 * gw, *r = A.geom_mat + 9 * gw, *sc = A.geom_scale + 3 * i;
        for (int row = 0; row < 3; ++row) {
            for (int col = 0; col < 3; ++col) m[4 * row + col] = r[3 * row + col] * sc[col];
            m[4 * row + 3] = p[row];
        }
    } else {
        const float4 *mi = reinterpret_cast<const float4 *>(A.matrices_in + 12 * ((size_t)w * A.matrices_stride + i));
        const float4 r0 = mi[0], r1 = mi[1], r2 = mi[2];
        m[0] = r0.x; m[1] = r0.y; m[2] = r0.z; m[3] = r0.w;
        m[4] = r1.x; m[5] = r1.y; m[6] = r1.z; m[7] = r1.w;
        m[8] = r2.x; m[9] = r2.y; m[10] = r2.z; m[11] = r2.w;
    }
    float4 *mo = reinterpret_cast<float4 *>(A.matrices_out + 12 * (size_t)g);
    mo[0] = make_float4(m[0], m[1], m[2], m[3]);
    mo[1] = make_float4(m[4], m[5], m[6], m[7]);
    mo[2] = make_float4(m[8], m[9], m[10], m[11]);
    float inv[12];
    invert_affine(m, inv);
    InstanceRec rec;
    rec.inv[0] = make_float4(inv[0], inv[1], inv[2], inv[3]);
    rec.inv[1] = make_float4(inv[4], inv[5], inv[6], inv[7]);
    rec.inv[2] = make_float4(inv[8], inv[9], inv[10], inv[11]);
    rec.mesh = mesh;
    rec.tmpl = i;
    rec.mesh_tris = mesh_tris;
    rec.skip_root = skip_root;
    A.inst[g] = rec;

    for (int ax = 0; ax < 3; ++ax) { lo[ax] = 1e30f; hi[ax] = -1e30f; }
    for (int corner = 0; corner < 8; ++corner) {
        const float p[3] = {(corner & 1) ? lb[3] : lb[0], (corner & 2) ? lb[4] : lb[1], (corner & 4) ? lb[5] : lb[2]};
        for (int ax = 0; ax < 3; ++ax) {
            const float v = m[4 * ax] * p[0] + m[4 * ax + 1] * p[1] + m[4 * ax + 2] * p[2] + m[4 * ax + 3];
            lo[ax] = fminf(lo[ax], v);
            hi[ax] = fmaxf(hi[ax], v);
        }
    }
    if (A.dbg_aabb) {
        float *o = A.dbg_aabb + 6 * (size_t)g;
        for (int ax = 0; ax < 3; ++ax) { o[ax] = lo[ax]; o[3 + ax] = hi[ax]; }
    }
}

// 30-bit Morton code of a box centre within the world's centre bounds (ordered ints), cuda_tlas.cuh:99-115.
__device__ __forceinline__ uint32_t morton_code(const float lo[3], const float hi[3], const int *world_bounds) {
    uint32_t q[3];
    for (int ax = 0; ax < 3; ++ax) {
        const float blo = from_ordered(world_bounds[ax]), bhi = from_ordered(world_bounds[3 + ax]);
        const float centre = 0.5f * (lo[ax] + hi[ax]);
        const float extent = bhi - blo;
        const float t = extent > 1e-20f ? (centre - blo) / extent : 0.0f;
        q[ax] = (uint32_t)(fminf(fmaxf(t, 0.0f), 1.0f) * 1023.0f);
    }
    return (spread_bits(q[0]) << 2) | (spread_bits(q[1]) << 1) | spread_bits(q[2]);
}

// Karras 2012 for internal node i of a world's n sorted keys at global positions a..a+n-1 (cuda_tlas.cuh:
// 119-159): equal keys are told apart by their global positions, keys of other worlds are out of range.
// Children: local node index, or n-1+k for the k-th leaf. The node covers the leaves first .. last.
template <class Keys>
__device__ __forceinline__ void karras_node(const int i, const int n, const int a, const Keys &key, int &l, int &r, int &first, int &last) {
    auto delta = [&](const int p, const int q) -> int {
        if (q < 0 || q >= n) return -1;
        const uint32_t kp = key[p], kq = key[q];
        if (kp == kq) return 64 + __clz((a + p) ^ (a + q));
        return 32 + __clz(kp ^ kq);
    };
    const int d = delta(i, i + 1) > delta(i, i - 1) ? 1 : -1;
    const int min_prefix = delta(i, i - d);
    int max_length = 2;
    while (delta(i, i + max_length * d) > min_prefix) max_length *= 2;
    int length = 0;
    for (int t = max_length / 2; t >= 1; t /= 2)
        if (delta(i, i + (length + t) * d) > min_prefix) length += t;
    const int j = i + length * d;
    const int node_prefix = delta(i, j);
    int s = 0;
    for (int t = (length + 1) / 2;; t = (t + 1) / 2) {
        if (delta(i, i + (s + t) * d) > node_prefix) s += t;
        if (t == 1) break;
    }
    const int gamma = i + s * d + (d < 0 ? d : 0);
    first = min(i, j);
    last = max(i, j);
    l = (first == gamma) ? n - 1 + gamma : gamma;
    r = (last == gamma + 1) ? n - 1 + gamma + 1 : gamma + 1;
}

// Writes a world's internal node at global index gi (the world's run at a, n instances) in both layouts, from its
// local children l and r and their boxes (lo xyz, hi xyz); id(k) is the template index of the k-th sorted leaf.
template <class IdOf>
__device__ __forceinline__ void write_interior(const TlasBuildArgs &A, const int gi, const int n, const int a, const int l, const int r,
                                               const float lbox[6], const float rbox[6], const IdOf &id) {
    const int N = A.total;
    TlasNode node;
    WideNode wn;
    for (int ax = 0; ax < 3; ++ax) {
        node.lo[ax] = fminf(lbox[ax], rbox[ax]);
        node.hi[ax] = fmaxf(lbox[3 + ax], rbox[3 + ax]);
        wn.set_left(ax, lbox[ax], lbox[3 + ax]);
        wn.set_right(ax, rbox[ax], rbox[3 + ax]);
    }
    node.left = l >= n - 1 ? N - 1 + a + (l - (n - 1)) : a + l;
    node.right = r >= n - 1 ? N - 1 + a + (r - (n - 1)) : a + r;
    A.nodes[gi] = node;
    wn.left = l >= n - 1 ? ~(a + id(l - (n - 1))) : a + l;
    wn.right = r >= n - 1 ? ~(a + id(r - (n - 1))) : a + r;
    wn.left_count = wn.right_count = 1;
    A.wide[gi] = wn;
}

// A workgroup's stable LSD radix sort of its threads' 30-bit keys (has: this thread holds one), 4 bits a pass, ranks
// from wave ballots: from buffer 0 and, eight passes later, back to it.
template <int MAXN>
__device__ __forceinline__ void sort_keys(uint32_t (&key)[2][MAXN], uint32_t (&val)[2][MAXN], int (&hist)[MAXN / 4],
                                          int (&wave_tot)[MAXN / 64], const bool has) {
    constexpr int NW = MAXN / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int pass = 0; pass < 8; ++pass) {
        const int src = pass & 1, dst = src ^ 1, shift = 4 * pass;
        for (int i = tid; i < 16 * NW; i += MAXN) hist[i] = 0;
        __syncthreads();
        const uint32_t k = has ? key[src][tid] : 0u, v = has ? val[src][tid] : 0u;
        const uint32_t digit = (k >> shift) & 15u;
        uint64_t peers = ballot(has);
        for (int bit = 0; bit < 4; ++bit) {
            const bool set = (digit >> bit) & 1u;
            const uint64_t vote = ballot(has && set);
            peers &= set ? vote : ~vote;
        }
        const int rank = popc64(peers & below);
        if (has && rank == 0) hist[digit * NW + wave] = popc64(peers);
        __syncthreads();
        block_exclusive_scan(hist, 16 * NW, wave_tot);
        if (has) {
            const int dest = hist[digit * NW + wave] + rank;
            key[dst][dest] = k;
            val[dst][dest] = v;
        }
        __syncthreads();
    }
}

constexpr int COUNTED_BUILD_MAX = 256;

template <int MAXN>
struct BuildShared {
    static constexpr int NW = MAXN / 64;
    float box_lo[3][MAXN], box_hi[3][MAXN];    // instance boxes by template index
    float node_lo[3][MAXN], node_hi[3][MAXN];  // interior nodes by local index
    alignas(16) uint32_t key[2][MAXN];
    uint32_t val[2][MAXN];
    int left[MAXN], right[MAXN], arrivals[MAXN];
    int parent[2 * MAXN];
    int hist[16 * NW];
    int wave_tot[NW];
    int bounds[6][NW];
    int world_bounds[6];
};

// A world's build is a chain of dependent steps; what bounds it is their latency, since even thousands of worlds give a
// SIMD few wavefronts. Worlds of at most COUNTED_BUILD_MAX instances sort by counting (eight digit passes before) and make
// boxes of runs of leaves (a climb with an atomic at every node before): one world of 16 13.5 -> 7.7 us, 64 of 32 posed by
// bodies 17.3 -> 11.2, 4,096 of 32 28 -> 19; a step of one world of 100 85 -> 79, of 200 101 -> 96, of 512 of 128 392 -> 385.
// Counting takes n steps a key, so larger worlds keep the passes, and the climb.
template <int MAXN>
__global__ __launch_bounds__(MAXN) void tlas_build_kernel(const TlasBuildArgs A) {
    __shared__ BuildShared<MAXN> sh;
    constexpr int NW = MAXN / 64;
    const int w = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int a = A.world_off[w];
    const int n = A.world_off[w + 1] - a;
    const int N = A.total;
    if (n == 0) {
        if (tid == 0) A.roots[w] = -1;
        return;
    }
    if (n > MAXN) return;  // built by the device-wide path
    const bool has = tid < n;

    // ---- place: matrix, inverse, box, vote on the centre bounds
    int cen[3] = {to_ordered(1e30f), to_ordered(1e30f), to_ordered(1e30f)};
    int cmax[3] = {to_ordered(-1e30f), to_ordered(-1e30f), to_ordered(-1e30f)};
    if (has) {
        float lo[3], hi[3];
        place_instance(A, w, tid, a + tid, lo, hi);
        for (int ax = 0; ax < 3; ++ax) {
            sh.box_lo[ax][tid] = lo[ax];
            sh.box_hi[ax][tid] = hi[ax];
            const int c = to_ordered(0.5f * (lo[ax] + hi[ax]));
            cen[ax] = c;
            cmax[ax] = c;
        }
    }
    for (int ax = 0; ax < 3; ++ax) {
        const int mn = wave_min(cen[ax]), mx = wave_max(cmax[ax]);
        if (lane == 0) { sh.bounds[ax][wave] = mn; sh.bounds[3 + ax][wave] = mx; }
    }
    __syncthreads();
    if (tid < 6) {
        int v = sh.bounds[tid][0];
        for (int k = 1; k < NW; ++k) v = tid < 3 ? min(v, sh.bounds[tid][k]) : max(v, sh.bounds[tid][k]);
        sh.world_bounds[tid] = v;
        if (A.dbg_world_bounds) A.dbg_world_bounds[6 * w + tid] = from_ordered(v);
    }
    __syncthreads();

    // ---- keys
    uint32_t mine = ~0u;
    if (has) {
        const float lo[3] = {sh.box_lo[0][tid], sh.box_lo[1][tid], sh.box_lo[2][tid]};
        const float hi[3] = {sh.box_hi[0][tid], sh.box_hi[1][tid], sh.box_hi[2][tid]};
        const uint32_t morton = morton_code(lo, hi, sh.world_bounds);
        mine = morton;
        sh.key[0][tid] = morton;
        sh.val[0][tid] = (uint32_t)tid;
        if (A.dbg_keys) A.dbg_keys[a + tid] = ((uint64_t)w << 32) | morton;
    }

    // ---- sort
    // eight passes end in buffer 0
    if constexpr (MAXN > COUNTED_BUILD_MAX) sort_keys<MAXN>(sh.key, sh.val, sh.hist, sh.wave_tot, has);
    else {
        // each thread counts the keys that come before its own: from the wavefront's registers, or from LDS, four at a time
        int rank = 0;
        if constexpr (MAXN <= 64) {
            for (int j = 0; j < n; ++j)
                rank += (uint32_t)__builtin_amdgcn_readlane((int)mine, j) < mine + (j < tid ? 1u : 0u) ? 1 : 0;
        } else {
            if (!has) sh.key[0][tid] = ~0u;
            __syncthreads();
            const uint4 *const four = reinterpret_cast<const uint4 *>(sh.key[0]);
            for (int j = 0; j < n; j += 4) {
                const uint4 other = four[j / 4];
                rank += (other.x < mine + (j < tid ? 1u : 0u) ? 1 : 0) + (other.y < mine + (j + 1 < tid ? 1u : 0u) ? 1 : 0) +
                        (other.z < mine + (j + 2 < tid ? 1u : 0u) ? 1 : 0) + (other.w < mine + (j + 3 < tid ? 1u : 0u) ? 1 : 0);
            }
        }
        __syncthreads();
        if (has) {
            sh.key[0][rank] = mine;
            sh.val[0][rank] = (uint32_t)tid;
        }
        __syncthreads();
    }
    const uint32_t *key = sh.key[0];
    const uint32_t *val = sh.val[0];
    if (has) {
        if (A.dbg_sorted_keys) A.dbg_sorted_keys[a + tid] = ((uint64_t)w << 32) | key[tid];
        if (A.dbg_sorted_ids) A.dbg_sorted_ids[a + tid] = a + (int)val[tid];
    }

    // ---- leaves, and the one-instance world
    if (has) {
        const int id = (int)val[tid];
        TlasNode leaf;
        for (int ax = 0; ax < 3; ++ax) { leaf.lo[ax] = sh.box_lo[ax][id]; leaf.hi[ax] = sh.box_hi[ax][id]; }
        leaf.left = ~(a + id);
        leaf.right = -1;
        A.nodes[(size_t)(N - 1) + a + tid] = leaf;
    }
    if (n == 1) {
        if (tid == 0) A.roots[w] = N - 1 + a;
        return;
    }

    // ---- Karras hierarchy over local positions 0..n-1 (global position a + i)
    for (int i = tid; i < 2 * n - 1; i += MAXN) sh.parent[i] = -1;
    if (tid < n - 1) sh.arrivals[tid] = 0;
    __syncthreads();
    int l = 0, r = 0, first = 0, last = 0;
    if (tid < n - 1) {
        karras_node(tid, n, a, key, l, r, first, last);
        sh.left[tid] = l;
        sh.right[tid] = r;
        sh.parent[l] = tid;
        sh.parent[r] = tid;
    }
    __syncthreads();

    // ---- boxes
    const int root_index = A.root_at_end[w] ? a + n - 1 : a;
    if constexpr (MAXN <= COUNTED_BUILD_MAX) {
        // A node's children cover the leaves first .. split and split + 1 .. last, and each is the union of
        // two runs of 2^k leaves. The unions of all runs of 2^k leaves are made for one k after another, in the place of
        // the leaves' boxes, and each child taken as its k comes up: eight steps at most, whatever the tree's depth.
        float box[6], child[2][6];
        const int id = has ? (int)val[tid] : 0;
        for (int ax = 0; ax < 3; ++ax) {
            box[ax] = sh.box_lo[ax][id];
            box[3 + ax] = sh.box_hi[ax][id];
        }
        __syncthreads();
        const int split = l >= n - 1 ? l - (n - 1) : l;
        const int from[2] = {first, split + 1}, to[2] = {split, last};
        for (int k = 0; (1 << k) < n; ++k) {
            for (int ax = 0; ax < 3; ++ax) {
                sh.box_lo[ax][tid] = box[ax];
                sh.box_hi[ax][tid] = box[3 + ax];
            }
            __syncthreads();
            for (int c = 0; c < 2; ++c) {
                const int length = to[c] - from[c] + 1;
                if (tid < n - 1 && (length >> k) == 1) {
                    const int other = to[c] + 1 - (1 << k);
                    for (int ax = 0; ax < 3; ++ax) {
                        child[c][ax] = fminf(sh.box_lo[ax][from[c]], sh.box_lo[ax][other]);
                        child[c][3 + ax] = fmaxf(sh.box_hi[ax][from[c]], sh.box_hi[ax][other]);
                    }
                }
            }
            const int next = min(tid + (1 << k), n - 1);
            for (int ax = 0; ax < 3; ++ax) {
                box[ax] = fminf(box[ax], sh.box_lo[ax][next]);
                box[3 + ax] = fmaxf(box[3 + ax], sh.box_hi[ax][next]);
            }
            __syncthreads();
        }
        if (tid == 0) A.roots[w] = root_index;
        if (tid < n - 1) {
            const int gi = tid == 0 ? root_index : a + tid, parent = sh.parent[tid];
            write_interior(A, gi, n, a, l, r, child[0], child[1], [&](const int k) { return (int)val[k]; });
            A.wide_parent[gi] = parent < 0 ? -1 : (parent == 0 ? root_index : a + parent);
        }
        return;
    }
    // bottom up: the second of two children to arrive at a node computes its box
    if (has) {
        int node = n - 1 + tid;
        while (true) {
            const int p = sh.parent[node];
            if (p < 0) break;
            const int prior = __hip_atomic_fetch_add(&sh.arrivals[p], 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (prior == 0) break;
            l = sh.left[p];
            r = sh.right[p];
            for (int ax = 0; ax < 3; ++ax) {
                const float llo = l >= n - 1 ? sh.box_lo[ax][val[l - (n - 1)]] : sh.node_lo[ax][l];
                const float lhi = l >= n - 1 ? sh.box_hi[ax][val[l - (n - 1)]] : sh.node_hi[ax][l];
                const float rlo = r >= n - 1 ? sh.box_lo[ax][val[r - (n - 1)]] : sh.node_lo[ax][r];
                const float rhi = r >= n - 1 ? sh.box_hi[ax][val[r - (n - 1)]] : sh.node_hi[ax][r];
                sh.node_lo[ax][p] = fminf(llo, rlo);
                sh.node_hi[ax][p] = fmaxf(lhi, rhi);
            }
            node = p;
        }
    }
    __syncthreads();

    // ---- write the interior nodes in both layouts
    if (tid == 0) A.roots[w] = root_index;
    if (tid < n - 1) {
        l = sh.left[tid];
        r = sh.right[tid];
        const int parent = sh.parent[tid];
        float lbox[6], rbox[6];
        for (int ax = 0; ax < 3; ++ax) {
            lbox[ax] = l >= n - 1 ? sh.box_lo[ax][val[l - (n - 1)]] : sh.node_lo[ax][l];
            lbox[3 + ax] = l >= n - 1 ? sh.box_hi[ax][val[l - (n - 1)]] : sh.node_hi[ax][l];
            rbox[ax] = r >= n - 1 ? sh.box_lo[ax][val[r - (n - 1)]] : sh.node_lo[ax][r];
            rbox[3 + ax] = r >= n - 1 ? sh.box_hi[ax][val[r - (n - 1)]] : sh.node_hi[ax][r];
        }
        const int gi = tid == 0 ? root_index : a + tid;
        write_interior(A, gi, n, a, l, r, lbox, rbox, [&](const int k) { return (int)val[k]; });
        A.wide_parent[gi] = parent < 0 ? -1 : (parent == 0 ? root_index : a + parent);
    }
}

// ------------------------------------------------------------------ device-wide build of large worlds --
//
// The worlds with more instances than one workgroup sorts in LDS are built together by a few grid-wide kernels with the
// same arithmetic, a workgroup a tile of a world (BigTile):
//   place   the instances, and the centre bounds by ordered-int atomics (cuda_tlas.cuh:69-96)
//   sort    keys, and each tile of 1024 sorted as a small world is
//   merge   up to 32 sorted runs into one: an element's place is its own plus, for every other run, how many of that
//           run's keys come before it (an equal key of an earlier run does, so the sort is stable), by binary searches
//           side by side; two launches up to a million instances
//   nodes   tiles of 256 leaves: Karras per node, and the boxes of the nodes inside the tile
//   join    the nodes that span tiles
// A node's box is the union of a run of sorted leaves, and a union may count a leaf twice, so no box waits for another:
// inside a tile it is two entries of a table of the unions of 2, 4, ... 256 leaves in LDS; across tiles it is one
// tile's from the run's first leaf on, the next one's up to its last leaf, and whole tiles between.
// What bounds a build is its chain of launches and the latencies in each. One world of 20,000 instances took 30 launches
// (a radix sort of 24, and a climb with an agent-scope acquire-release at every node, 98 us alone), 250 us of kernels;
// these five take 68.

constexpr int BIG_MERGE = 32, BIG_MERGE_AT_ONCE = 16;
static_assert(BIG_SORT_TILE == WORKGROUP_BUILD_MAX, "a sort tile is sorted as the largest small world");

__global__ __launch_bounds__(BIG_NODE_TILE) void big_place_kernel(const TlasBuildArgs A, const BigBuildScratch S) {
    __shared__ int part[6][4];
    const BigTile T = S.node_tiles[blockIdx.x];
    const BigWorld W = S.worlds[T.world];
    const int i = T.first + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int cmin[3] = {to_ordered(1e30f), to_ordered(1e30f), to_ordered(1e30f)};
    int cmax[3] = {to_ordered(-1e30f), to_ordered(-1e30f), to_ordered(-1e30f)};
    if (i < W.n) {
        float lo[3], hi[3];
        place_instance(A, W.world, i, W.first + i, lo, hi);
        for (int ax = 0; ax < 3; ++ax) {
            S.box[(size_t)ax * S.capacity + W.base + i] = lo[ax];
            S.box[(size_t)(3 + ax) * S.capacity + W.base + i] = hi[ax];
            cmin[ax] = cmax[ax] = to_ordered(0.5f * (lo[ax] + hi[ax]));
        }
    }
    for (int ax = 0; ax < 3; ++ax) {
        const int mn = wave_min(cmin[ax]), mx = wave_max(cmax[ax]);
        if (lane == 0) {
            part[ax][wave] = mn;
            part[3 + ax][wave] = mx;
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int t = threadIdx.x;
        int v = part[t][0];
        for (int k = 1; k < 4; ++k) v = t < 3 ? min(v, part[t][k]) : max(v, part[t][k]);
        int *const b = S.bounds + 6 * T.world;
        if (t < 3) atomicMin(&b[t], v);
        else atomicMax(&b[t], v);
    }
}

__global__ __launch_bounds__(BIG_SORT_TILE) void big_sort_kernel(const TlasBuildArgs A, const BigBuildScratch S) {
    __shared__ uint32_t key[2][BIG_SORT_TILE], val[2][BIG_SORT_TILE];
    __shared__ int hist[BIG_SORT_TILE / 4], wave_tot[BIG_SORT_TILE / 64];
    const BigTile T = S.sort_tiles[blockIdx.x];
    const BigWorld W = S.worlds[T.world];
    const int tid = threadIdx.x, i = T.first + tid;
    const int *const bounds = S.bounds + 6 * T.world;
    if (T.first == 0 && tid < 6 && A.dbg_world_bounds) A.dbg_world_bounds[6 * W.world + tid] = from_ordered(bounds[tid]);
    const bool has = i < W.n;
    if (has) {
        float lo[3], hi[3];
        for (int ax = 0; ax < 3; ++ax) {
            lo[ax] = S.box[(size_t)ax * S.capacity + W.base + i];
            hi[ax] = S.box[(size_t)(3 + ax) * S.capacity + W.base + i];
        }
        const uint32_t morton = morton_code(lo, hi, bounds);
        key[0][tid] = morton;
        val[0][tid] = (uint32_t)i;
        if (A.dbg_keys) A.dbg_keys[W.first + i] = ((uint64_t)W.world << 32) | morton;
    }
    sort_keys<BIG_SORT_TILE>(key, val, hist, wave_tot, has);
    if (has) {
        S.key[0][W.base + i] = key[0][tid];
        S.val[0][W.base + i] = val[0][tid];
    }
}

// Merges runs of `run` elements (a power of two), BIG_MERGE of them into one, from buffer src to the other. FIRST: the
// runs are sort tiles, and a group's keys fit in LDS (128 KB at most), where the searches take half the time they take
// through the caches (20 runs: 22 us against 43).
template <bool FIRST>
__global__ __launch_bounds__(256) void big_merge_kernel(const BigBuildScratch S, const int src, const int run) {
    __shared__ uint32_t held[FIRST ? BIG_MERGE * BIG_SORT_TILE : 1];
    const BigTile T = S.node_tiles[blockIdx.x];
    const BigWorld W = S.worlds[T.world];
    // tiles do not straddle groups: a group's length is a multiple of the tile's, so group and runs are the workgroup's
    const long long group = (long long)run * BIG_MERGE;
    const int first = (int)(T.first / group * group), end = (int)min((long long)W.n, first + group);
    const int runs = (end - first + run - 1) / run;
    const uint32_t *const key = S.key[src] + W.base + first;
    if (FIRST) {
        for (int j0 = 0; j0 < end - first; j0 += 16 * 256) {
            uint32_t some[16];  // 16 loads in flight
            for (int q = 0; q < 16; ++q) some[q] = key[min(j0 + q * 256 + (int)threadIdx.x, end - first - 1)];
            for (int q = 0; q < 16; ++q) held[j0 + q * 256 + (int)threadIdx.x] = some[q];
        }
        __syncthreads();
    }
    const int i = T.first - first + (int)threadIdx.x;  // within the group
    if (first + i >= W.n) return;
    const uint32_t k = FIRST ? held[i] : key[i], v = S.val[src][W.base + first + i];
    const int mine = i / run;
    int place = i % run;
    for (int r0 = 0; r0 < runs; r0 += BIG_MERGE_AT_ONCE) {
        int at[BIG_MERGE_AT_ONCE];
        for (int j = 0; j < BIG_MERGE_AT_ONCE; ++j) at[j] = 0;
        for (int step = run; step > 0; step >>= 1) {
            for (int j = 0; j < BIG_MERGE_AT_ONCE; ++j) {
                const int r = r0 + j, start = r * run;  // below BIG_MERGE x run, at most 2^30 for the largest world there is
                const int len = r < runs && r != mine ? min(run, end - first - start) : 0;
                const int probe = at[j] + step;
                const int p = min(start + probe, end - first) - 1;  // read whether or not it counts: 16 reads side by side
                const uint32_t o = FIRST ? held[p] : key[p];
                at[j] = (probe <= len) & ((o < k) | ((o == k) & (r < mine))) ? probe : at[j];
            }
        }
        for (int j = 0; j < BIG_MERGE_AT_ONCE; ++j) place += at[j];
    }
    S.key[src ^ 1][W.base + first + place] = k;
    S.val[src ^ 1][W.base + first + place] = v;
}

// The unions of a tile's leaf boxes: entry [k][.][p] those of leaves p .. p + 2^k - 1 of the tile.
struct BigTable {
    float box[8 + 1][6][BIG_NODE_TILE];
    __device__ __forceinline__ void range(const int from, const int to, float out[6]) const {
        const int k = 31 - __clz(to - from + 1), second = to - (1 << k) + 1;
        for (int ax = 0; ax < 3; ++ax) {
            out[ax] = fminf(box[k][ax][from], box[k][ax][second]);
            out[3 + ax] = fmaxf(box[k][3 + ax][from], box[k][3 + ax][second]);
        }
    }
};

__global__ __launch_bounds__(BIG_NODE_TILE) void big_nodes_kernel(const TlasBuildArgs A, const BigBuildScratch S, const int src) {
    __shared__ BigTable table;
    const BigTile T = S.node_tiles[blockIdx.x];
    const BigWorld W = S.worlds[T.world];
    const int tid = threadIdx.x, i = T.first + tid, n = W.n, a = W.first;
    const int count = min(BIG_NODE_TILE, n - T.first);
    const uint32_t *const key = S.key[src] + W.base;
    const uint32_t *const val = S.val[src] + W.base;
    float leaf[6];
    if (tid < count) {
        const int id = (int)val[i];
        if (A.dbg_sorted_keys) A.dbg_sorted_keys[a + i] = ((uint64_t)W.world << 32) | key[i];
        if (A.dbg_sorted_ids) A.dbg_sorted_ids[a + i] = a + id;
        for (int c = 0; c < 6; ++c) table.box[0][c][tid] = leaf[c] = S.box[(size_t)c * S.capacity + W.base + id];
        TlasNode node;
        for (int ax = 0; ax < 3; ++ax) {
            node.lo[ax] = leaf[ax];
            node.hi[ax] = leaf[3 + ax];
        }
        node.left = ~(a + id);
        node.right = -1;
        A.nodes[(size_t)(A.total - 1) + a + i] = node;
    }
    __syncthreads();
    for (int k = 1; (1 << k) <= count; ++k) {
        if (tid + (1 << k) <= count)
            for (int ax = 0; ax < 3; ++ax) {
                const int other = tid + (1 << (k - 1));
                table.box[k][ax][tid] = fminf(table.box[k - 1][ax][tid], table.box[k - 1][ax][other]);
                table.box[k][3 + ax][tid] = fmaxf(table.box[k - 1][3 + ax][tid], table.box[k - 1][3 + ax][other]);
            }
        __syncthreads();
    }
    if (tid >= count) return;
    float4 span[3];
    float *const sp = reinterpret_cast<float *>(span);
    table.range(0, tid, sp);              // the tile up to this leaf
    table.range(tid, count - 1, sp + 6);  // and from it on
    float4 *const out = S.span + 3 * (size_t)(W.base + i);
    for (int c = 0; c < 3; ++c) out[c] = span[c];
    if (i >= n - 1) return;
    const int root_index = A.root_at_end[W.world] ? a + n - 1 : a;
    const int gi = i == 0 ? root_index : a + i;
    int l, r, first, last;
    karras_node(i, n, a, key, l, r, first, last);
    if (i == 0) {
        A.roots[W.world] = root_index;
        A.wide_parent[root_index] = -1;
    }
    if (l < n - 1) A.wide_parent[a + l] = gi;
    if (r < n - 1) A.wide_parent[a + r] = gi;
    const bool inside = first >= T.first && last < T.first + count;
    S.across[W.base + i] = inside ? make_int4(-1, 0, 0, 0) : make_int4(l, r, first, last);
    if (!inside) return;
    const int split = l >= n - 1 ? l - (n - 1) : l;
    float lbox[6], rbox[6];
    table.range(first - T.first, split - T.first, lbox);
    table.range(split + 1 - T.first, last - T.first, rbox);
    write_interior(A, gi, n, a, l, r, lbox, rbox, [&](const int k) { return (int)val[k]; });
}

// The box of leaves from .. to of a world, which lie in more than one tile; `whole` is how many tiles lie whole between.
__device__ __forceinline__ void big_span_ends(const BigBuildScratch &S, const BigWorld &W, const int from, const int to, float out[6]) {
    const float *const head = reinterpret_cast<const float *>(S.span + 3 * (size_t)(W.base + from)) + 6;
    const float *const tail = reinterpret_cast<const float *>(S.span + 3 * (size_t)(W.base + to));
    for (int ax = 0; ax < 3; ++ax) {
        out[ax] = fminf(head[ax], tail[ax]);
        out[3 + ax] = fmaxf(head[3 + ax], tail[3 + ax]);
    }
}
// A whole tile's box: the span up to its last leaf.
__device__ __forceinline__ void big_add_tile(const BigBuildScratch &S, const BigWorld &W, const int tile, float out[6]) {
    const float *const t = reinterpret_cast<const float *>(S.span + 3 * ((size_t)W.base + (size_t)tile * BIG_NODE_TILE + BIG_NODE_TILE - 1));
    for (int ax = 0; ax < 3; ++ax) {
        out[ax] = fminf(out[ax], t[ax]);
        out[3 + ax] = fmaxf(out[3 + ax], t[3 + ax]);
    }
}

__global__ __launch_bounds__(64) void big_bounds_kernel(const BigBuildScratch S, const int values) {
    for (int i = threadIdx.x; i < values; i += 64) S.bounds[i] = to_ordered(i % 6 < 3 ? 1e30f : -1e30f);
}

__global__ __launch_bounds__(BIG_NODE_TILE) void big_join_kernel(const TlasBuildArgs A, const BigBuildScratch S, const int src) {
    const BigTile T = S.node_tiles[blockIdx.x];
    const BigWorld W = S.worlds[T.world];
    const int tid = threadIdx.x, lane = tid & 63, i = T.first + tid, n = W.n, a = W.first;
    // the bounds as the next build expects them
    if (T.first == 0 && tid < 6) S.bounds[6 * T.world + tid] = to_ordered(tid < 3 ? 1e30f : -1e30f);
    int4 node = make_int4(-1, 0, 0, 0);
    if (i < n - 1) node = S.across[W.base + i];
    const bool mine = node.x >= 0;
    const int split = node.x >= n - 1 ? node.x - (n - 1) : node.x;
    float box[2][6];
    for (int c = 0; c < 2; ++c) {
        const int from = c == 0 ? node.z : split + 1, to = c == 0 ? split : node.w, child = c == 0 ? node.x : node.y;
        const int t0 = from / BIG_NODE_TILE, t1 = to / BIG_NODE_TILE;
        const bool across = mine && t0 != t1;
        if (mine && !across) {
            const TlasNode &k = A.nodes[child >= n - 1 ? (size_t)(A.total - 1) + a + (child - (n - 1)) : (size_t)a + child];
            for (int ax = 0; ax < 3; ++ax) {
                box[c][ax] = k.lo[ax];
                box[c][3 + ax] = k.hi[ax];
            }
        }
        if (across) big_span_ends(S, W, from, to, box[c]);
        // whole tiles between: a few by the lane itself, many by the wavefront, one node after the other
        const int whole = across ? t1 - t0 - 1 : 0;
        if (whole <= 16)
            for (int t = 0; t < whole; ++t) big_add_tile(S, W, t0 + 1 + t, box[c]);
        uint64_t many = ballot(whole > 16);
        while (many != 0) {
            const int who = first_lane(many);
            const int t_first = __builtin_amdgcn_readlane(t0, who) + 1, t_count = __builtin_amdgcn_readlane(whole, who);
            float u[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
            for (int t = lane; t < t_count; t += 64) big_add_tile(S, W, t_first + t, u);
            for (int o = 32; o >= 1; o >>= 1)
                for (int ax = 0; ax < 3; ++ax) {
                    u[ax] = fminf(u[ax], __shfl_xor(u[ax], o, 64));
                    u[3 + ax] = fmaxf(u[3 + ax], __shfl_xor(u[3 + ax], o, 64));
                }
            if (lane == who)
                for (int ax = 0; ax < 3; ++ax) {
                    box[c][ax] = fminf(box[c][ax], u[ax]);
                    box[c][3 + ax] = fmaxf(box[c][3 + ax], u[3 + ax]);
                }
            many &= many - 1;
        }
    }
    if (!mine) return;
    const int gi = i != 0 ? a + i : A.root_at_end[W.world] ? a + n - 1 : a;
    const uint32_t *const val = S.val[src] + W.base;
    write_interior(A, gi, n, a, node.x, node.y, box[0], box[1], [&](const int k) { return (int)val[k]; });
}

// ------------------------------------------------------------------ ray order for ray queries --
//
// A query's rays come in the caller's order; a LiDAR's consecutive rays fan out over many degrees, so a
// wavefront of 64 of them shares little of either tree. Each world's rays are put in a stable order of a
// 12-bit direction cell (octahedral map of the direction, 64 x 64 cells, Morton order) by a counting sort; the
// tracer then gives a wavefront 64 consecutive rays of that order, and results still go to each ray's own place.
//
// One workgroup orders a world (or a segment of one, below): each of its wavefronts takes a contiguous part of the
// rays, counts their cells into its own row of 16-bit counters in LDS (4096 cells x 16 wavefronts = 128 KB) and keeps
// each cell in 2 bytes of scratch; the counters are scanned in cell-major, wavefront-minor order, which gives each
// (cell, wavefront) its first place; each wavefront then reads its cells back and writes its rays' indices in ray
// order, a ray's rank among the equal cells of its 64 from ballots. 16 bytes a ray of traffic.
//
// Where there are fewer worlds than the chip has room for, or more rays than 16-bit places number, a world is cut into
// segments of 4096 rays: one kernel counts each segment's cells, one sums each cell's counts over the segments, and one
// orders each segment as above, from the cells' places and the segments' within them.
// One world of 262,144 rays: 21 us, where a radix sort by one workgroup took 2,000; of 65,536 rays: 20 us, where one
// workgroup takes 140. 96 worlds of 65,536 rays: 108 us against 150; at 128 worlds, half the compute units, the extra pass
// costs what the spreading saves, and every segment has 4096 cells to clear and scan, so worlds of few rays keep to one.
constexpr int RAY_ORDER_CELLS = 4096;
constexpr int RAY_ORDER_ONE_PASS_MAX_RAYS = 65536;
constexpr int RAY_ORDER_SEGMENT = 4096;
constexpr int RAY_ORDER_SEGMENTED_MIN_RAYS = 8192;
constexpr int RAY_ORDER_SEGMENTED_MAX_WORLDS = 96;
constexpr int RAY_ORDER_FEW_RAYS = 2048, RAY_ORDER_FEW_RAYS_MANY_WORLDS = 4096, RAY_ORDER_MANY_WORLDS = 512;

// tile_digit for a BITS-bit digit: the digit of each key of a 1024-key tile, its rank among the equal digits of
// its wave, and how many of its wave share the digit (valid for the rank-0 lane).
template <int BITS>
__device__ __forceinline__ void tile_digit_bits(const bool has, const uint32_t k, const int shift, uint32_t &digit, int &rank,
                                                int &count) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    digit = (k >> shift) & ((1u << BITS) - 1u);
    uint64_t peers = ballot(has);
    for (int bit = 0; bit < BITS; ++bit) {
        const bool set = (digit >> bit) & 1u;
        const uint64_t vote = ballot(has && set);
        peers &= set ? vote : ~vote;
    }
    rank = popc64(peers & below);
    count = popc64(peers);
}

__device__ __forceinline__ uint32_t spread6(uint32_t v) {
    uint32_t r = 0;
    for (int b = 0; b < 6; ++b) r |= ((v >> b) & 1u) << (2 * b);
    return r;
}

__device__ __forceinline__ uint32_t direction_cell(const float x, const float y, const float z) {
    const float s = fabsf(x) + fabsf(y) + fabsf(z);
    if (!(s > 0.0f) || !isfinite(s)) return 4095u;
    float u = x / s, v = y / s;
    if (z < 0.0f) {
        const float uu = (1.0f - fabsf(v)) * (u >= 0.0f ? 1.0f : -1.0f);
        const float vv = (1.0f - fabsf(u)) * (v >= 0.0f ? 1.0f : -1.0f);
        u = uu;
        v = vv;
    }
    const uint32_t qu = (uint32_t)fminf(63.0f, fmaxf(0.0f, (u * 0.5f + 0.5f) * 64.0f));
    const uint32_t qv = (uint32_t)fminf(63.0f, fmaxf(0.0f, (v * 0.5f + 0.5f) * 64.0f));
    return (spread6(qu) << 1) | spread6(qv);
}

// The counters of a workgroup's wavefronts: per (cell, wavefront), cell-major, first how many of the wavefront's rays
// fall in the cell, then where the next of them goes.
template <int NW>
struct RayOrderShared {
    // a count is at most 4096 and a place below 65,536, so 16 bits hold either; the scan's running sum runs in 32 bits
    // (past the last occupied slot it may reach 65,536, and those slots are never read)
    alignas(16) uint16_t slot[RAY_ORDER_CELLS * NW];
    int wave_tot[NW];
};

template <int NW>
__device__ __forceinline__ void ray_order_clear(RayOrderShared<NW> &sh) {
    uint4 *p = reinterpret_cast<uint4 *>(sh.slot);
    for (int i = threadIdx.x; i < RAY_ORDER_CELLS * NW / 8; i += 64 * NW) p[i] = make_uint4(0u, 0u, 0u, 0u);
}
// Counts a ray in its wavefront's counter of cell c: a 32-bit word holds the counters of two neighbouring wavefronts,
// and a count stays below 2^16, so adding 1 to a wavefront's own half never carries into the other.
template <int NW>
__device__ __forceinline__ void ray_order_count(RayOrderShared<NW> &sh, const uint32_t c, const int wave) {
    atomicAdd(&reinterpret_cast<uint32_t *>(sh.slot)[(c * NW + wave) >> 1], 1u << (16 * (wave & 1)));
}
// Turns a cell's counts into places from `start` on, wavefront after wavefront, and returns the cell's count. The
// counters of a cell are read and written 4 at a time: lanes take neighbouring cells.
template <int NW>
__device__ __forceinline__ int ray_order_places(RayOrderShared<NW> &sh, const int cell, const int start) {
    ushort4 *p = reinterpret_cast<ushort4 *>(sh.slot + cell * NW);
    int run = start;
    for (int k = 0; k < NW / 4; ++k) {
        ushort4 n = p[k];
        const ushort4 c = n;
        n.x = (uint16_t)run; run += c.x;
        n.y = (uint16_t)run; run += c.y;
        n.z = (uint16_t)run; run += c.z;
        n.w = (uint16_t)run; run += c.w;
        p[k] = n;
    }
    return run - start;
}
// The number of rays counted in a cell.
template <int NW>
__device__ __forceinline__ int ray_order_total(const RayOrderShared<NW> &sh, const int cell) {
    const ushort4 *p = reinterpret_cast<const ushort4 *>(sh.slot + cell * NW);
    int sum = 0;
    for (int k = 0; k < NW / 4; ++k) sum += p[k].x + p[k].y + p[k].z + p[k].w;
    return sum;
}
// The place of a ray of cell c (RAY_ORDER_CELLS: no ray) among its wavefront's, in ray order.
template <int NW>
__device__ __forceinline__ int ray_order_place(RayOrderShared<NW> &sh, const bool has, const uint32_t c, const int wave) {
    uint32_t digit;
    int rank, cnt, place = 0;
    tile_digit_bits<12>(has, c, 0, digit, rank, cnt);
    if (has) place = (int)sh.slot[c * NW + wave] + rank;
    // every lane has read its cell's place before the cell's first lane moves it on (one wavefront's LDS accesses
    // complete in order)
    if (has && rank == 0) sh.slot[c * NW + wave] = (uint16_t)(place + cnt);
    return place;
}

// The order of up to 65,536 rays a world, a workgroup of NW wavefronts a world; cells is scratch of one 16-bit cell a
// ray. What bounds it is the counters' share of LDS (one workgroup of 16 wavefronts fits a compute unit) and, for few
// rays, clearing and scanning them: there a quarter as many wavefronts take a quarter of the
// counters (64 worlds of 1,081 rays: 11 us against 15; 1,024 worlds of 4,096 rays, four workgroups a compute unit: 39 us
// against 71; but 64 such worlds 26 us against 20, each wavefront having four times the rays).
template <int NW>
__global__ __launch_bounds__(64 * NW) void ray_order_one_pass_kernel(const float *dirs, const int R, uint16_t *cells, int *order) {
    __shared__ RayOrderShared<NW> sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t base = (size_t)blockIdx.x * R;
    const int seg = (R + NW - 1) / NW;
    const int first = wave * seg, end = min(first + seg, R);
    ray_order_clear(sh);
    __syncthreads();
    for (int i = first + lane; i < end; i += 64) {
        const float *p = dirs + 3 * (base + i);
        const uint32_t c = direction_cell(p[0], p[1], p[2]);
        cells[base + i] = (uint16_t)c;
        ray_order_count(sh, c, wave);
    }
    __syncthreads();
    // the cells in order, a thread a cell, the workgroup's threads at a time
    int carry = 0;
    for (int c0 = 0; c0 < RAY_ORDER_CELLS; c0 += 64 * NW) {
        const int n = ray_order_total(sh, c0 + tid);
        const int incl = wave_prefix_sum(n);
        if (lane == 63) sh.wave_tot[wave] = incl;
        __syncthreads();
        int start = carry + incl - n;
        for (int wv = 0; wv < NW; ++wv) {
            if (wv < wave) start += sh.wave_tot[wv];
            carry += sh.wave_tot[wv];
        }
        ray_order_places(sh, c0 + tid, start);
        __syncthreads();
    }
    for (int at = first; at < end; at += 64) {
        const int i = at + lane;
        const bool has = i < end;
        const uint32_t c = has ? cells[base + i] : (uint32_t)RAY_ORDER_CELLS;
        const int place = ray_order_place(sh, has, c, wave);
        if (has) order[base + place] = i;
    }
}

// Segmented worlds, first kernel: each ray's cell, and how many of the segment's rays fall in each cell.
__global__ __launch_bounds__(1024) void ray_order_count_kernel(const float *dirs, const int R, const int segments, uint16_t *cells,
                                                               uint32_t *counts) {
    __shared__ uint32_t hist[RAY_ORDER_CELLS];
    const int world = blockIdx.x / segments, s = blockIdx.x % segments;
    const size_t base = (size_t)world * R;
    const int end = min((s + 1) * RAY_ORDER_SEGMENT, R);
    for (int c = threadIdx.x; c < RAY_ORDER_CELLS; c += 1024) hist[c] = 0u;
    __syncthreads();
    for (int i = s * RAY_ORDER_SEGMENT + threadIdx.x; i < end; i += 1024) {
        const float *p = dirs + 3 * (base + i);
        const uint32_t c = direction_cell(p[0], p[1], p[2]);
        cells[base + i] = (uint16_t)c;
        atomicAdd(&hist[c], 1u);
    }
    __syncthreads();
    uint32_t *out = counts + (size_t)blockIdx.x * RAY_ORDER_CELLS;
    for (int c = threadIdx.x; c < RAY_ORDER_CELLS; c += 1024) out[c] = hist[c];
}

// Second kernel: a world's counts [segment][cell] become how many of the cell's rays the segments before hold, and
// totals how many there are in all. A thread a cell, 16 workgroups a world.
__global__ __launch_bounds__(256) void ray_order_sum_kernel(const int segments, uint32_t *counts, uint32_t *totals) {
    const int world = blockIdx.x / (RAY_ORDER_CELLS / 256), cell = blockIdx.x % (RAY_ORDER_CELLS / 256) * 256 + threadIdx.x;
    uint32_t *c = counts + (size_t)world * segments * RAY_ORDER_CELLS + cell;
    uint32_t run = 0;
#pragma unroll 16
    for (int s = 0; s < segments; ++s) {
        const uint32_t n = c[(size_t)s * RAY_ORDER_CELLS];
        c[(size_t)s * RAY_ORDER_CELLS] = run;
        run += n;
    }
    totals[(size_t)world * RAY_ORDER_CELLS + cell] = run;
}

// Third kernel: each segment's rays to their places, 16 wavefronts of 256 rays.
__global__ __launch_bounds__(1024) void ray_order_segment_kernel(const int R, const int segments, const uint16_t *cells,
                                                                 const uint32_t *before, const uint32_t *totals, int *order) {
    constexpr int NW = 16, STEPS = RAY_ORDER_SEGMENT / (64 * NW);
    __shared__ RayOrderShared<NW> sh;
    alignas(16) __shared__ uint32_t start[RAY_ORDER_CELLS];  // the first place of the segment's rays of each cell, written four at a time
    const int world = blockIdx.x / segments, s = blockIdx.x % segments;
    const size_t base = (size_t)world * R;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int first = s * RAY_ORDER_SEGMENT + wave * 64 * STEPS + lane;
    uint32_t c[STEPS];
    for (int k = 0; k < STEPS; ++k) c[k] = first + 64 * k < R ? cells[base + first + 64 * k] : (uint32_t)RAY_ORDER_CELLS;
    const uint4 n = reinterpret_cast<const uint4 *>(totals + (size_t)world * RAY_ORDER_CELLS)[tid];
    const uint4 mine = reinterpret_cast<const uint4 *>(before + (size_t)blockIdx.x * RAY_ORDER_CELLS)[tid];
    ray_order_clear(sh);
    const int sum = (int)(n.x + n.y + n.z + n.w);
    const int incl = wave_prefix_sum(sum);
    if (lane == 63) sh.wave_tot[wave] = incl;
    __syncthreads();
    for (int k = 0; k < STEPS; ++k)
        if (c[k] < RAY_ORDER_CELLS) ray_order_count(sh, c[k], wave);
    uint32_t at = (uint32_t)(incl - sum);
    for (int wv = 0; wv < wave; ++wv) at += (uint32_t)sh.wave_tot[wv];
    reinterpret_cast<uint4 *>(start)[tid] = make_uint4(at + mine.x, at + n.x + mine.y, at + n.x + n.y + mine.z, at + n.x + n.y + n.z + mine.w);
    __syncthreads();
    for (int cell = tid; cell < RAY_ORDER_CELLS; cell += 1024) ray_order_places(sh, cell, 0);
    __syncthreads();
    for (int k = 0; k < STEPS; ++k) {
        const bool has = c[k] < RAY_ORDER_CELLS;
        const int place = ray_order_place(sh, has, c[k], wave);
        if (has) order[base + start[c[k]] + place] = first + 64 * k;
    }
}

}  // namespace

hipError_t launch_tlas_build(const TlasBuildArgs &a, const int max_count, hipStream_t stream) {
    if (a.worlds <= 0) return hipSuccess;
    if (max_count <= 64) tlas_build_kernel<64><<<a.worlds, 64, 0, stream>>>(a);
    else if (max_count <= 128) tlas_build_kernel<128><<<a.worlds, 128, 0, stream>>>(a);
    else if (max_count <= 256) tlas_build_kernel<256><<<a.worlds, 256, 0, stream>>>(a);
    else if (max_count <= 512) tlas_build_kernel<512><<<a.worlds, 512, 0, stream>>>(a);
    else tlas_build_kernel<1024><<<a.worlds, 1024, 0, stream>>>(a);  // larger worlds return at once
    return hipGetLastError();
}

hipError_t reset_big_bounds(const BigBuildScratch &s, const int worlds) {
    big_bounds_kernel<<<1, 64, 0, nullptr>>>(s, 6 * worlds);
    return hipGetLastError();
}

hipError_t launch_tlas_build_big(const TlasBuildArgs &a, const BigBuildScratch &s, hipStream_t stream) {
    if (s.node_tile_count <= 0 || s.sort_tile_count <= 0) return hipErrorInvalidValue;
    const unsigned tiles = (unsigned)s.node_tile_count;
    big_place_kernel<<<tiles, BIG_NODE_TILE, 0, stream>>>(a, s);
    big_sort_kernel<<<(unsigned)s.sort_tile_count, BIG_SORT_TILE, 0, stream>>>(a, s);
    int src = 0;
    for (long long run = BIG_SORT_TILE; run < s.largest; run *= BIG_MERGE, src ^= 1) {
        if (run == BIG_SORT_TILE) big_merge_kernel<true><<<tiles, BIG_NODE_TILE, 0, stream>>>(s, src, (int)run);
        else big_merge_kernel<false><<<tiles, BIG_NODE_TILE, 0, stream>>>(s, src, (int)run);
    }
    big_nodes_kernel<<<tiles, BIG_NODE_TILE, 0, stream>>>(a, s, src);
    big_join_kernel<<<tiles, BIG_NODE_TILE, 0, stream>>>(a, s, src);
    return hipGetLastError();
}

static bool ray_order_segmented(const int rays_per_world, const int worlds) {
    return rays_per_world > RAY_ORDER_ONE_PASS_MAX_RAYS ||
           (rays_per_world >= RAY_ORDER_SEGMENTED_MIN_RAYS && worlds <= RAY_ORDER_SEGMENTED_MAX_WORLDS);
}

size_t ray_order_scratch_words(const int rays_per_world, const int worlds) {
    // a cell in 2 bytes a ray; segmented, a word a cell for each world and for each segment, at most one of them broken
    const size_t n = (size_t)rays_per_world * worlds;
    const size_t cells = (n + 7) / 8 * 4;
    const size_t segments = ((size_t)rays_per_world + RAY_ORDER_SEGMENT - 1) / RAY_ORDER_SEGMENT;
    return ray_order_segmented(rays_per_world, worlds) ? cells + (1 + segments) * worlds * RAY_ORDER_CELLS : cells;
}

hipError_t launch_ray_order(const float *dirs, const int rays_per_world, const int worlds, uint32_t *keys, int *vals, int **order,
                            hipStream_t stream) {
    if (rays_per_world <= 0 || rays_per_world > RAY_ORDER_MAX_RAYS || worlds <= 0) return hipErrorInvalidValue;
    const size_t n = (size_t)rays_per_world * worlds;
    uint16_t *const cells = reinterpret_cast<uint16_t *>(keys);
    if (ray_order_segmented(rays_per_world, worlds)) {
        const int segments = (rays_per_world + RAY_ORDER_SEGMENT - 1) / RAY_ORDER_SEGMENT;
        uint32_t *const totals = keys + (n + 7) / 8 * 4;  // past the cells, on 16 bytes
        uint32_t *const counts = totals + (size_t)worlds * RAY_ORDER_CELLS;
        ray_order_count_kernel<<<worlds * segments, 1024, 0, stream>>>(dirs, rays_per_world, segments, cells, counts);
        ray_order_sum_kernel<<<worlds * (RAY_ORDER_CELLS / 256), 256, 0, stream>>>(segments, counts, totals);
        ray_order_segment_kernel<<<worlds * segments, 1024, 0, stream>>>(rays_per_world, segments, cells, counts, totals, vals);
    } else if (rays_per_world <= (worlds >= RAY_ORDER_MANY_WORLDS ? RAY_ORDER_FEW_RAYS_MANY_WORLDS : RAY_ORDER_FEW_RAYS)) {
        ray_order_one_pass_kernel<4><<<worlds, 256, 0, stream>>>(dirs, rays_per_world, cells, vals);
    } else {
        ray_order_one_pass_kernel<16><<<worlds, 1024, 0, stream>>>(dirs, rays_per_world, cells, vals);
    }
    *order = vals;
    return hipGetLastError();
}

}  // namespace ngx
