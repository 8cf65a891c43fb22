// Deforming meshes: a mesh's bottom level refitted on the GPU to new vertex positions, keeping its tree.
//
// The tree's topology (built once on the host with the reference's binned SAH) is kept; every node's box is
// recomputed from the new vertices exactly as the host computes a box (the min and max over the triangles'
// vertices, then unions upward), so the boxes are the ones a host refit of the same tree would give. The
// packed triangles (v0, e1, e2) are recomputed the same way. No reference counterpart: the reference builds bottom
// levels once, on the host.
//
// The tree comes cut into treelets (ngx_blas.cpp), a workgroup each: a treelet's boxes are made level by level in LDS,
// with a barrier between levels, and written once, with the wide nodes' planes and, at the mesh's root, its record and
// bounds. A launch a layer of treelets, two for a mesh of up to some hundred thousand triangles. What bounds it is
// latency: about ten levels, each an LDS round trip, after the leaves' vertex reads. The climb it replaces, in which the
// second child to arrive at a node made its box, paid an agent-scope acquire-release (a write-back and an invalidation
// of caches) at every node: 138,000 triangles 395 us, 25 us so.
#include "ngx_kernels.h"

namespace ngx {
namespace {

__global__ __launch_bounds__(256) void refit_treelet_kernel(const MeshRefitArgs A, const int first_treelet) {
    __shared__ float box[6][REFIT_TREELET_NODES];
    const RefitTreelet T = A.treelets[first_treelet + (int)blockIdx.x];
    const RefitEntry *const entries = A.entries + T.first;
    const int *const starts = A.levels + T.level_first;
    for (int level = 0; level < T.levels; ++level) {
        const int end = starts[level + 1];
        for (int k = starts[level] + (int)threadIdx.x; k < end; k += 256) {
            const RefitEntry e = entries[k];
            float lo[3], hi[3];
            if (e.wide < 0) {
                for (int ax = 0; ax < 3; ++ax) {
                    lo[ax] = INFINITY;
                    hi[ax] = -INFINITY;
                }
                for (int t = e.left; t < e.left + e.right; ++t) {
                    float p[3][3];
                    for (int c = 0; c < 3; ++c)
                        for (int ax = 0; ax < 3; ++ax) p[c][ax] = A.vertices[3 * (size_t)(A.tri_verts[3 * (size_t)t + c] - A.vertex_base) + ax];
                    float *const o = A.tris + 9 * (size_t)t;
                    for (int ax = 0; ax < 3; ++ax) {
                        o[ax] = p[0][ax];
                        o[3 + ax] = p[1][ax] - p[0][ax];
                        o[6 + ax] = p[2][ax] - p[0][ax];
                        for (int c = 0; c < 3; ++c) {
                            lo[ax] = fminf(lo[ax], p[c][ax]);
                            hi[ax] = fmaxf(hi[ax], p[c][ax]);
                        }
                    }
                }
            } else {
                float child[2][6];
                for (int c = 0; c < 2; ++c) {
                    const int ref = c == 0 ? e.left : e.right;
                    if (ref >= 0) {
                        for (int j = 0; j < 6; ++j) child[c][j] = box[j][ref];
                    } else {
                        const SkipNode &n = A.skip[~ref];
                        for (int ax = 0; ax < 3; ++ax) {
                            child[c][ax] = n.lo[ax];
                            child[c][3 + ax] = n.hi[ax];
                        }
                    }
                }
                WideNode &w = A.wide[e.wide];
                for (int ax = 0; ax < 3; ++ax) {
                    w.set_left(ax, child[0][ax], child[0][3 + ax]);
                    w.set_right(ax, child[1][ax], child[1][3 + ax]);
                    lo[ax] = fminf(child[0][ax], child[1][ax]);
                    hi[ax] = fmaxf(child[0][3 + ax], child[1][3 + ax]);
                }
                if (A.octants)
                    for (int o = 0; o < 8; ++o) A.octants[(size_t)o * A.octant_nodes + e.wide] = w.for_octant(o, o * A.octant_nodes);
            }
            SkipNode &n = A.skip[e.node];
            for (int ax = 0; ax < 3; ++ax) {
                box[ax][k] = n.lo[ax] = lo[ax];
                box[3 + ax][k] = n.hi[ax] = hi[ax];
            }
            if (T.is_root && k == starts[T.levels] - 1)
                for (int ax = 0; ax < 3; ++ax) {
                    A.mesh_root->lo[ax] = A.mesh_bounds[ax] = lo[ax];
                    A.mesh_root->hi[ax] = A.mesh_bounds[3 + ax] = hi[ax];
                }
        }
        __syncthreads();
    }
}

}  // namespace

hipError_t launch_mesh_refit(const MeshRefitArgs &a, const int first, const int count, hipStream_t stream) {
    if (count <= 0) return hipErrorInvalidValue;
    refit_treelet_kernel<<<count, 256, 0, stream>>>(a, first);
    return hipGetLastError();
}

}  // namespace ngx
