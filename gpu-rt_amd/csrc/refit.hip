// refit.hip -- BVH refit for moved vertices (same triangles, same tree).
//
// The reference only rebuilds (VK_BUILD_ACCELERATION_STRUCTURE_MODE_BUILD_KHR,
// src/vk/vulkan.cpp:832,915); an optimisation loop that moves vertices every step wants
// the cheaper update.  Steps:
//   k_refit_check   every new position finite (else the tree stays unchanged and the call
//                   returns GPURT_E_INVALID), and the new coordinate scale
//   k_refit_tris    re-gather each packed triangle from the new vertex positions (its id
//                   and leaf position are unchanged), compact copy of the positions for
//                   the backward passes, and the boxes of aligned blocks of triangles
//   k_refit_boxes   every child's box: the union of its triangles, which are contiguous,
//                   from those blocks, inflated by the new pad
// So no child waits for another and the tree takes one launch instead of one per level
// (a 252 K triangle tree's 11 took 134 us, each the latency of its nodes' loads), and the
// kernels after the check look at its flag on the device, so the host waits once.
#include <algorithm>

#include "build_common.h"
#include "index_math.h"

namespace gpurt_impl {

// tmp[0]: the coordinate scale as an ordered uint, tmp[1]: set when a position is not finite
__global__ void k_refit_init(uint32_t* tmp) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        tmp[0] = f2o(0.0f);
        tmp[1] = 0u;
    }
}

// One atomic per block: an atomic per wave on the one address took 25 us for 126 K vertices.
__global__ __launch_bounds__(kBlock) void k_refit_check(uint32_t n_verts, const float* __restrict__ v,
                                                        uint64_t stride, uint32_t* tmp) {
    __shared__ float part[kBlock / 64];
    bool bad = false;
    float amax = 0.0f;
    grid_stride(n_verts, blockIdx.x * kBlock + threadIdx.x, gridDim.x * kBlock, [&](uint32_t i) {
        const float* p = v + (size_t)i * stride;
        const float x = p[0], y = p[1], z = p[2];
        bad = bad || !(isfinite(x) && isfinite(y) && isfinite(z));
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(x), fabsf(y)), fabsf(z)));
    });
    if (__any(bad) && (threadIdx.x & 63) == 0) gatomic_or(tmp + 1, 1u);
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; w++) amax = fmaxf(amax, part[w]);
        if (amax > 0.0f) gatomic_max_u32(tmp, f2o(amax));
    }
}

__global__ __launch_bounds__(kBlock) void k_refit_tris(uint32_t n_tris, uint32_t n_verts, const float* __restrict__ v,
                                                       uint64_t stride, const uint32_t* __restrict__ leaf_order,
                                                       const uint32_t* __restrict__ tri_idx,
                                                       const uint32_t* __restrict__ tmp, float* __restrict__ compact,
                                                       float4* __restrict__ tris, float4* __restrict__ rbox) {
    __shared__ float4 part[8];
    if (tmp[1]) return;
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p < n_verts) {
        const float* q = v + (size_t)p * stride;
        compact[3 * (size_t)p] = q[0];
        compact[3 * (size_t)p + 1] = q[1];
        compact[3 * (size_t)p + 2] = q[2];
    }
    if (blockIdx.x * kBlock >= n_tris) return;  // (the whole block)
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (p < n_tris) {
        const uint32_t g = leaf_order[p];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float* q = v + (size_t)tri_idx[3 * (size_t)g + k] * stride;
            // the first vertex carries the triangle's id
            const float4 x = make_float4(q[0], q[1], q[2], k == 0 ? __uint_as_float(g) : 0.0f);
            tris[3 * (size_t)p + k] = x;
            lo = min4(lo, x);
            hi = max4(hi, x);
        }
    }
    write_range_blocks(n_tris, p, lo, hi, rbox, part);
}

// one thread per child of every node
template <int W>
__global__ __launch_bounds__(kBlock) void k_refit_boxes(uint32_t n_nodes, uint32_t n_tris, WNode<W>* nodes,
                                                        const uint32_t* __restrict__ first,
                                                        const float4* __restrict__ tris,
                                                        const float4* __restrict__ rbox,
                                                        const uint32_t* __restrict__ tmp) {
    if (tmp[1]) return;
    const uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= (uint64_t)n_nodes * W) return;
    WNode<W>& nd = nodes[k / W];
    const uint32_t j = (uint32_t)(k % W);
    const uint32_t c = nd.child[j];
    if (c == kEmpty) return;
    const float pad = o2f(tmp[0]) * 0x1p-18f;
    const uint32_t f = child_is_leaf(c) ? leaf_first(c) : first[c];
    float4 lo, hi;
    range_union(
        f, f + nd.aux[j], n_tris, rbox,
        [&](uint32_t t, float4& l, float4& h) {
#pragma unroll
            for (int v = 0; v < 3; v++) {
                const float4 p = tris[3 * (size_t)t + v];
                l = min4(l, p);
                h = max4(h, p);
            }
        },
        lo, hi);
    nd.lox[j] = lo.x - pad; nd.loy[j] = lo.y - pad; nd.loz[j] = lo.z - pad;
    nd.hix[j] = hi.x + pad; nd.hiy[j] = hi.y + pad; nd.hiz[j] = hi.z + pad;
}

template <int W>
static void refit_boxes(gpurt_bvh_s* b, const float4* rbox, const uint32_t* tmp, hipStream_t s) {
    hipLaunchKernelGGL(k_refit_boxes<W>, dim3(cdiv((size_t)b->n_nodes * W, kBlock)), dim3(kBlock), 0, s,
                       (uint32_t)b->n_nodes, (uint32_t)b->n_tris, reinterpret_cast<WNode<W>*>(b->nodes), b->node_first,
                       b->tris, rbox, tmp);
}

int launch_refit(gpurt_bvh_s* b, const float* verts, size_t vstride_floats, hipStream_t s) {
    if (!b->leaf_order || !b->tri_idx || !b->verts) return set_error(GPURT_E_INVALID, "bvh has no mesh copy");
    const uint32_t n_tris = (uint32_t)b->n_tris, n_verts = (uint32_t)b->n_verts;
    uint32_t* tmp = b->refit_tmp;
    void* mem = nullptr;
    if (const int rc = pool_alloc(b->ctx, &mem, 2 * sizeof(float4) * range_boxes(n_tris), s)) return rc;
    float4* rbox = static_cast<float4*>(mem);
    hipLaunchKernelGGL(k_refit_init, dim3(1), dim3(64), 0, s, tmp);
    // every new position must be finite; the tree is left as it was otherwise
    hipLaunchKernelGGL(k_refit_check, dim3(std::min(cdiv(n_verts, kBlock), 512u)), dim3(kBlock), 0, s, n_verts, verts,
                       (uint64_t)vstride_floats, tmp);
    hipLaunchKernelGGL(k_refit_tris, dim3(cdiv(std::max(n_tris, n_verts), kBlock)), dim3(kBlock), 0, s, n_tris, n_verts,
                       verts, (uint64_t)vstride_floats, b->leaf_order, b->tri_idx, tmp, b->verts, b->tris, rbox);
    launch_range_top(n_tris, rbox, s);
    switch (b->width) {
        case 2: refit_boxes<2>(b, rbox, tmp, s); break;
        case 4: refit_boxes<4>(b, rbox, tmp, s); break;
        case 8: refit_boxes<8>(b, rbox, tmp, s); break;
    }
    // (unchanged boxes give the same copies)
    if (has_qnodes(b->format)) launch_quantize(b->width, b->nodes, b->qnodes, (uint32_t)b->n_nodes,
                                                (uint32_t)b->n_nodes, nullptr, s);
    if (b->onodes)
        launch_orient(b->nodes, b->node_first, b->tris, b->onodes, (uint32_t)b->n_nodes, (uint32_t)b->n_nodes, nullptr,
                      tmp, 0, nullptr, tmp + 1, s);
    const hipError_t e = hipGetLastError();
    uint32_t bad = 0;
    hipError_t ce = hipMemcpyAsync(&bad, tmp + 1, sizeof(bad), hipMemcpyDeviceToHost, s);
    pool_free(b->ctx, mem, s);
    if (ce == hipSuccess) ce = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_error(e, "refit launch");
    if (ce != hipSuccess) return hip_error(ce, "refit check");
    if (bad) return set_error(GPURT_E_INVALID, "non-finite vertex position");
    return GPURT_OK;
}

}  // namespace gpurt_impl
