// backward.hip -- gradients of unsigned distance and ray hit distance (plain path).
//
// Both passes reuse the forward pass's saved primitive ids and barycentrics (no
// re-traversal; the per-query math is in backward.h).  Query / ray gradients are written
// directly.  Vertex gradients are sums over every query whose triangle uses the vertex:
//   atomic       k_cpq_bwd / k_ray_bwd add each query's three vertex terms with FP32
//                atomics: one launch, bound by the atomics (~9 random device-scope FP32
//                atomics per query; the summation order, and so the last bits, vary)
//   fixed order  k_*_bwd_terms write the terms with the vertex they belong to, a stable
//                radix sort orders them by vertex, and k_wave_segsum + k_run_sum add each
//                vertex's terms in a fixed order: the same bits on every run
// The context's mode picks one (gpurt_ctx_set_vertex_sums); by default the fixed order
// runs for calls of at least kFixedOrderMinTerms terms, where it is also the faster.
// Algorithmic bytes: a closest-point query reads q, g, prim and its triangle (12 + 4 + 4
// + 12 + 36) and writes g_q (12) and adds to three vertices (3 x 2 x 12); a ray reads its
// direction, t, uv, g and its triangle.
#include "backward.h"

namespace gpurt_impl {

// term k = 3 * item + corner: key = its vertex (n_verts when there is none, sorted last),
// terms[3k .. 3k+2] = the float3 to add
__device__ __forceinline__ void write_terms(size_t i, const CornerTerms& t, uint32_t n_verts, uint32_t* __restrict__ keys,
                                            float* __restrict__ terms) {
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const size_t k = 3 * i + j;
        keys[k] = t.v[j] == kNoVertex ? n_verts : t.v[j];
        terms[3 * k] = t.c[j][0];
        terms[3 * k + 1] = t.c[j][1];
        terms[3 * k + 2] = t.c[j][2];
    }
}

__global__ __launch_bounds__(kBlock) void k_cpq_bwd_terms(uint32_t n, const float* __restrict__ q,
                                                          const int32_t* __restrict__ prim,
                                                          const float* __restrict__ g,
                                                          const uint32_t* __restrict__ tri_idx, uint32_t n_tris,
                                                          const float* __restrict__ verts, uint32_t n_verts,
                                                          float* __restrict__ g_q, uint32_t* __restrict__ keys,
                                                          float* __restrict__ terms) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    write_terms(i, cpq_bwd_terms(i, q, prim, g, tri_idx, n_tris, verts, 3, g_q), n_verts, keys, terms);
}

__global__ __launch_bounds__(kBlock) void k_ray_bwd_terms(uint32_t n, const float4* __restrict__ rays,
                                                          const int32_t* __restrict__ prim,
                                                          const float* __restrict__ t,
                                                          const float* __restrict__ uv,
                                                          const float* __restrict__ g,
                                                          const uint32_t* __restrict__ tri_idx, uint32_t n_tris,
                                                          const float* __restrict__ verts, uint32_t n_verts,
                                                          float* __restrict__ g_o, float* __restrict__ g_d,
                                                          uint32_t* __restrict__ keys, float* __restrict__ terms) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    write_terms(i, ray_bwd_terms(i, rays, prim, t, uv, g, tri_idx, n_tris, verts, 3, g_o, g_d), n_verts, keys, terms);
}

__global__ __launch_bounds__(kBlock) void k_cpq_bwd(uint32_t n, const float* __restrict__ q,
                                                    const int32_t* __restrict__ prim, const float* __restrict__ g,
                                                    const uint32_t* __restrict__ tri_idx, uint32_t n_tris,
                                                    const float* __restrict__ verts, float* __restrict__ g_q,
                                                    float* g_verts) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    scatter_terms(cpq_bwd_terms(i, q, prim, g, tri_idx, n_tris, verts, 3, g_q), g_verts);
}

__global__ __launch_bounds__(kBlock) void k_ray_bwd(uint32_t n, const float4* __restrict__ rays,
                                                    const int32_t* __restrict__ prim, const float* __restrict__ t,
                                                    const float* __restrict__ uv, const float* __restrict__ g,
                                                    const uint32_t* __restrict__ tri_idx, uint32_t n_tris,
                                                    const float* __restrict__ verts, float* __restrict__ g_o,
                                                    float* __restrict__ g_d, float* g_verts) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    scatter_terms(ray_bwd_terms(i, rays, prim, t, uv, g, tri_idx, n_tris, verts, 3, g_o, g_d), uv ? g_verts : nullptr);
}

// a vertex's gradient
struct VertexSink {
    float* g_verts;
    __device__ float* at(uint64_t v) const { return g_verts + 3 * v; }
};

namespace {

// scratch of the vertex-gradient sum over n items (3 terms each)
struct TermScratch {
    void* mem = nullptr;
    CallScratch cs;
    uint32_t *k0 = nullptr, *k1 = nullptr, *v0 = nullptr, *v1 = nullptr, *sort = nullptr;
    float* terms = nullptr;
    WaveSums sums{};
};

int alloc_terms(gpurt_ctx_s* c, size_t n, hipStream_t s, TermScratch& t) {
    if (3 * n > 0xFFFFFFFFull - kBlock) return set_error(GPURT_E_INVALID, "too many queries for one backward call");
    const size_t m = 3 * n;
    const size_t words = radix_sort_scratch_words((uint32_t)m);
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t bytes = 4 * up(4 * m) + up(12 * m) + 2 * up(4 * wave_sum_floats(m)) + up(4 * words) + 256;
    const int rc = ctx_scratch(c, s, bytes, t.cs);
    if (rc) return rc;
    t.mem = t.cs.mem;
    char* p = static_cast<char*>(t.mem);
    t.k0 = reinterpret_cast<uint32_t*>(p);
    p += up(4 * m);
    t.k1 = reinterpret_cast<uint32_t*>(p);
    p += up(4 * m);
    t.v0 = reinterpret_cast<uint32_t*>(p);
    p += up(4 * m);
    t.v1 = reinterpret_cast<uint32_t*>(p);
    p += up(4 * m);
    t.terms = reinterpret_cast<float*>(p);
    p += up(12 * m);
    for (float** q : {&t.sums.first, &t.sums.last}) {
        *q = reinterpret_cast<float*>(p);
        p += up(4 * wave_sum_floats(m));
    }
    t.sort = reinterpret_cast<uint32_t*>(p);
    return GPURT_OK;
}

// Whether the vertex sums of n items are added in the fixed order, and then its scratch; with
// the default mode, whose atomics need none, memory that cannot be had is no error.
int plan_sums(gpurt_ctx_s* c, size_t n, hipStream_t s, TermScratch& t, bool& fixed) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    const bool recorded = hipStreamIsCapturing(s, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone;
    if (recorded) (void)hipGetLastError();
    fixed = fixed_order_sums(c, 3 * n, recorded);
    if (!fixed) return GPURT_OK;
    const int rc = alloc_terms(c, n, s, t);
    if (rc != GPURT_E_OOM || c->vertex_sums != GPURT_SUMS_AUTO) return rc;
    fixed = false;
    return GPURT_OK;
}

int bits_for(uint32_t n_verts) {
    int b = 1;
    while (b < 32 && (n_verts >> b) != 0) b++;
    return b;  // keys 0 .. n_verts (n_verts = no vertex) fit in b bits
}

// sort the terms by vertex and add each vertex's run to g_verts
void sum_terms(TermScratch& t, size_t n, uint32_t n_verts, float* g_verts, hipStream_t s) {
    const uint32_t m = (uint32_t)(3 * n);
    uint32_t* k = t.k0;
    uint32_t* v = t.v0;
    if (radix_sort_pairs(t.k0, t.v0, t.k1, t.v1, m, bits_for(n_verts), t.sort, s)) {
        k = t.k1;
        v = t.v1;
    }
    const VertexSink sink{g_verts};
    hipLaunchKernelGGL((k_wave_segsum<kBlock, uint32_t, VertexSink>), dim3(cdiv(m, kBlock)), dim3(kBlock), 0, s, m, k, v,
                       t.terms, (uint64_t)n_verts, t.sums, sink);
    hipLaunchKernelGGL((k_run_sum<kBlock, uint32_t, VertexSink>), dim3(cdiv(cdiv(m, 64), kBlock)), dim3(kBlock), 0, s, m,
                       k, (uint64_t)n_verts, t.sums, sink);
}

}  // namespace

int launch_cpq_bwd(gpurt_bvh_s* b, const float* q, size_t n, const int32_t* prim, const float* g,
                   float* g_q, float* g_verts, hipStream_t s) {
    if (n == 0) return GPURT_OK;
    TermScratch t;
    bool fixed = false;
    if (g_verts)
        if (const int rc = plan_sums(b->ctx, n, s, t, fixed)) return rc;
    if (!fixed) {
        hipLaunchKernelGGL(k_cpq_bwd, dim3(cdiv(n, kBlock)), dim3(kBlock), 0, s, (uint32_t)n, q, prim, g,
                           b->tri_idx, (uint32_t)b->n_tris, b->verts, g_q, g_verts);
        GPURT_HIP(hipGetLastError());
        return GPURT_OK;
    }
    hipLaunchKernelGGL(k_cpq_bwd_terms, dim3(cdiv(n, kBlock)), dim3(kBlock), 0, s, (uint32_t)n, q, prim, g,
                       b->tri_idx, (uint32_t)b->n_tris, b->verts, (uint32_t)b->n_verts, g_q, t.k0, t.terms);
    sum_terms(t, n, (uint32_t)b->n_verts, g_verts, s);
    const hipError_t e = hipGetLastError();
    ctx_scratch_done(b->ctx, t.cs);
    if (e != hipSuccess) return hip_error(e, "closest-point backward launch");
    return GPURT_OK;
}

int launch_ray_bwd(gpurt_bvh_s* b, const gpurt_ray* rays, size_t n, const int32_t* prim,
                   const float* t, const float* uv, const float* g, float* g_o, float* g_d,
                   float* g_verts, hipStream_t s) {
    if (n == 0) return GPURT_OK;
    TermScratch ts;
    bool fixed = false;
    if (g_verts && uv)
        if (const int rc = plan_sums(b->ctx, n, s, ts, fixed)) return rc;
    if (!fixed) {
        hipLaunchKernelGGL(k_ray_bwd, dim3(cdiv(n, kBlock)), dim3(kBlock), 0, s, (uint32_t)n,
                           reinterpret_cast<const float4*>(rays), prim, t, uv, g, b->tri_idx, (uint32_t)b->n_tris,
                           b->verts, g_o, g_d, g_verts);
        GPURT_HIP(hipGetLastError());
        return GPURT_OK;
    }
    hipLaunchKernelGGL(k_ray_bwd_terms, dim3(cdiv(n, kBlock)), dim3(kBlock), 0, s, (uint32_t)n,
                       reinterpret_cast<const float4*>(rays), prim, t, uv, g, b->tri_idx, (uint32_t)b->n_tris,
                       b->verts, (uint32_t)b->n_verts, g_o, g_d, ts.k0, ts.terms);
    sum_terms(ts, n, (uint32_t)b->n_verts, g_verts, s);
    const hipError_t e = hipGetLastError();
    ctx_scratch_done(b->ctx, ts.cs);
    if (e != hipSuccess) return hip_error(e, "ray backward launch");
    return GPURT_OK;
}

}  // namespace gpurt_impl
