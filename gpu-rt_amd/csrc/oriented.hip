// oriented.hip -- oriented 8-bit copies of the 4-wide nodes, for closest-point queries.
//
// A closest-point search visits every node whose box is nearer than the best triangle
// found so far, so it pays for the empty part of the boxes.  Around a tilted patch of a
// surface an axis-aligned box is as thick as the patch is wide however finely the mesh
// is divided, and a query at a distance has to open all patches within about the square
// root of that thickness: 401 nodes and 1106 triangles per query for points spread
// around a 1.3 M triangle blob.  A box aligned with the patch is thin: 65 nodes and 48
// triangles per query with the nodes made here (points near the surface: 15 nodes and
// 9.5 triangles instead of 15 and 14.8).
//
// Each node gets a frame R (rows = axes), the smallest rotation that takes its normal n
// to the z axis, so two numbers (n.x, n.y; n.z >= 0 follows) describe it and neighbouring
// nodes turn little against each other.  Its children's boxes are the bounds of their
// triangles in that frame, computed from the triangles for nodes of up to kOrientMax
// triangles; nodes above that (their patches are bent) and nodes whose boxes would have
// more area than the axis-aligned ones keep those: R = I, n = (0, 0, 1).  The boxes are
// stored in 8 bits about the node's origin with a power-of-two step per axis.  A rotation
// changes no distance, the boxes are inflated by the same pad as the FP32 ones (2^-18 of
// the largest coordinate, 64 ulps: the roundings of R, of the transformed points and of the
// byte grid are a few ulps each) and rounded outwards, so culls stay conservative and
// answers do not change.
#include <algorithm>

#include "build_common.h"
#include "oriented.h"

namespace gpurt_impl {

// Uniform points around a 1.3 M triangle blob visit 57 nodes without this limit, 65 with
// 4096, 85 with 1024, 128 with 256; points near its surface 16.1, 15.0, 14.4 and 14.1.
constexpr uint32_t kOrientMax = 4096;
// A node of up to kOrientQuad triangles is made by 4 lanes, up to kOrientRow by 16 and above
// by a wave: what does not depend on the triangles (frame, byte grid) is computed by all of
// a node's lanes alike and is most of the instructions, so a small node gets few lanes, and
// no lane reads more than some dozens of triangles.
constexpr uint32_t kOrientQuad = 16, kOrientRow = 64;

struct OrientArgs {
    const WNode<4>* nodes;
    const uint32_t* first;  // first packed triangle of each node's range
    const float4* tris;
    ONode* out;
    const uint32_t* n_dev;  // node count on the device (batch), or null
    uint32_t n;
    const uint32_t* scale;  // largest coordinate as an ordered uint, per mesh
    uint32_t scale_stride;
    const uint32_t* seg;    // mesh of each node, or null (one mesh)
    const uint32_t* skip;   // nothing is written when *skip (null: never)
};

__device__ __forceinline__ V3 vmin(V3 a, V3 b) { return v3(vmin(a.x, b.x), vmin(a.y, b.y), vmin(a.z, b.z)); }
__device__ __forceinline__ V3 vmax(V3 a, V3 b) { return v3(vmax(a.x, b.x), vmax(a.y, b.y), vmax(a.z, b.z)); }

// Reductions over N aligned lanes, the result in all of them: within a row of 16 lanes by
// DPP moves (no LDS round trip), across rows by shuffles.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __uint_as_float(dpp<CTRL>(__float_as_uint(v)));
}
template <int N, typename Op>
__device__ __forceinline__ float group_reduce(float v, Op op) {
    static_assert(N == 1 || N == 4 || N == 16 || N == 64, "a lane, a quad, a row or a wave");
    if constexpr (N >= 4) {
        v = op(v, dppf<0xB1>(v));  // lane ^ 1
        v = op(v, dppf<0x4E>(v));  // lane ^ 2
    }
    if constexpr (N >= 16) {
        v = op(v, dppf<0x141>(v));  // the other quad of the half row
        v = op(v, dppf<0x140>(v));  // the other half row
    }
    if constexpr (N >= 64) {
        v = op(v, __shfl_xor(v, 16));
        v = op(v, __shfl_xor(v, 32));
    }
    return v;
}
template <int N>
__device__ __forceinline__ V3 group_min(V3 v) {
    auto op = [](float x, float y) { return vmin(x, y); };
    return v3(group_reduce<N>(v.x, op), group_reduce<N>(v.y, op), group_reduce<N>(v.z, op));
}
template <int N>
__device__ __forceinline__ V3 group_max(V3 v) {
    auto op = [](float x, float y) { return vmax(x, y); };
    return v3(group_reduce<N>(v.x, op), group_reduce<N>(v.y, op), group_reduce<N>(v.z, op));
}
template <int N>
__device__ __forceinline__ float group_sum(float v) {
    return group_reduce<N>(v, [](float x, float y) { return x + y; });
}
// out[q] = the value of child q's first lane, in every lane of the group
template <int LPC>
__device__ __forceinline__ void from_children(uint32_t v, uint32_t (&out)[4]) {
    if constexpr (LPC == 1) {  // quad broadcasts
        out[0] = dpp<0x00>(v);
        out[1] = dpp<0x55>(v);
        out[2] = dpp<0xAA>(v);
        out[3] = dpp<0xFF>(v);
    } else if constexpr (LPC == 4) {  // row broadcasts
        out[0] = dpp<0x150>(v);
        out[1] = dpp<0x154>(v);
        out[2] = dpp<0x158>(v);
        out[3] = dpp<0x15C>(v);
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++) out[q] = (uint32_t)__builtin_amdgcn_readlane((int)v, 16 * q);
    }
}

// area-weighted normal of packed triangle t
__device__ __forceinline__ V3 tri_normal(const float4* __restrict__ tris, uint32_t t) {
    const size_t p = 3 * (size_t)t;
    const float4 A = tris[p], B = tris[p + 1], C = tris[p + 2];
    return cross(v3(B.x - A.x, B.y - A.y, B.z - A.z), v3(C.x - A.x, C.y - A.y, C.z - A.z));
}

// n.x, n.y of the frame that takes the direction n (or -n) to the z axis; false when n has
// no direction.  |(nx, ny)| <= 1 in the traversal's arithmetic, so that the normal it forms
// is a unit vector to an ulp.
__device__ __forceinline__ bool frame_of(V3 n, float& nx, float& ny) {
    const float m = fmaxf(fmaxf(fabsf(n.x), fabsf(n.y)), fabsf(n.z));
    nx = ny = 0.0f;
    if (!(m > 0x1p-100f && m < 0x1p100f)) return false;
    const float im = __builtin_amdgcn_rcpf(m);
    const float x = n.x * im, y = n.y * im, z = n.z * im;
    const float inv = copysignf(__builtin_amdgcn_rsqf(x * x + y * y + z * z), z);
    nx = x * inv;
    ny = y * inv;
    for (int k = 0; k < 3 && frame_z2(nx, ny) < 0.0f; k++) {
        nx *= 0.9999998f;
        ny *= 0.9999998f;
    }
    if (frame_z2(nx, ny) >= 0.0f) return true;
    nx = ny = 0.0f;
    return false;
}

// Makes node i with a group of 4 * LPC lanes (a quad, a row or a wave), LPC per child: lane
// s of child j.  All lanes of the group call it together.
template <int LPC>
__device__ __forceinline__ void orient_node(const OrientArgs& a, uint32_t i) {
    constexpr int G = 4 * LPC;
    const uint32_t l = threadIdx.x % G, j = l / LPC, s = l % LPC;
    const WNode<4>& nd = a.nodes[i];
    const uint32_t ch = nd.child[j];
    const bool empty = ch == kEmpty;
    const uint32_t cnt = nd.aux[j];  // 0 in an empty slot, whose box is [inf, -inf]
    const uint32_t f = empty ? 0u : (child_is_leaf(ch) ? leaf_first(ch) : a.first[ch]);
    const V3 alo = v3(nd.lox[j], nd.loy[j], nd.loz[j]), ahi = v3(nd.hix[j], nd.hiy[j], nd.hiz[j]);
    const V3 ulo = group_min<G>(alo), uhi = group_max<G>(ahi);
    const uint32_t total = (uint32_t)group_sum<G>(s == 0 ? (float)min(cnt, 1u << 20) : 0.0f);
    const float pad = o2f(a.scale[a.seg ? (size_t)a.seg[i] * a.scale_stride : 0]) * 0x1p-18f;
    V3 c = v3(0.5f * ulo.x + 0.5f * uhi.x, 0.5f * ulo.y + 0.5f * uhi.y, 0.5f * ulo.z + 0.5f * uhi.z);
    float nx = 0.0f, ny = 0.0f;
    bool turned = false;
    V3 blo = v3(INFINITY, INFINITY, INFINITY), bhi = v3(-INFINITY, -INFINITY, -INFINITY);
    if (total <= kOrientMax) {
        // the normal: one triangle per lane, evenly spaced, turned to the first one's side
        // (meshes of mixed winding), weighted by area
        V3 n = v3(0.f, 0.f, 0.f);
        if (s < cnt) n = tri_normal(a.tris, f + (cnt > LPC ? (2 * s + 1) * cnt / (2 * LPC) : s));
        uint32_t rx[4], ry[4], rz[4];
        from_children<LPC>(__float_as_uint(n.x), rx);
        from_children<LPC>(__float_as_uint(n.y), ry);
        from_children<LPC>(__float_as_uint(n.z), rz);
        const float side =
            dot(n, v3(__uint_as_float(rx[0]), __uint_as_float(ry[0]), __uint_as_float(rz[0]))) < 0.0f ? -1.0f : 1.0f;
        turned = frame_of(v3(group_sum<G>(n.x * side), group_sum<G>(n.y * side), group_sum<G>(n.z * side)), nx, ny);
        if (turned) {
            const Frame R(nx, ny);
#pragma unroll(LPC == 16 ? 4 : 1)
            for (uint32_t k = s; k < cnt; k += LPC) {
                const size_t p = 3 * (size_t)(f + k);
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const float4 P = a.tris[p + q];
                    const V3 y = R.to_local(v3(P.x - c.x, P.y - c.y, P.z - c.z));
                    blo = vmin(blo, y);
                    bhi = vmax(bhi, y);
                }
            }
            blo = group_min<LPC>(blo);
            bhi = group_max<LPC>(bhi);
            blo = v3(blo.x - pad, blo.y - pad, blo.z - pad);
            bhi = v3(bhi.x + pad, bhi.y + pad, bhi.z + pad);
            auto area = [&](V3 lo, V3 hi) {
                const float x = hi.x - lo.x, y = hi.y - lo.y, z = hi.z - lo.z;
                return s == 0 && !empty ? x * y + y * z + x * z : 0.0f;
            };
            turned = group_sum<G>(area(blo, bhi)) < group_sum<G>(area(alo, ahi));  // (false for a NaN)
        }
    }
    if (!turned) {
        nx = ny = 0.0f;
        blo = v3(alo.x - c.x, alo.y - c.y, alo.z - c.z);
        bhi = v3(ahi.x - c.x, ahi.y - c.y, ahi.z - c.z);
    }
    const Frame R(nx, ny);
    // move the origin to the middle of the boxes, so that the byte grid is centred on them
    const V3 lo = group_min<G>(blo), hi = group_max<G>(bhi);
    const V3 mid = R.to_world(v3(0.5f * (lo.x + hi.x), 0.5f * (lo.y + hi.y), 0.5f * (lo.z + hi.z)));
    const V3 c0 = c;
    c = v3(c0.x + mid.x, c0.y + mid.y, c0.z + mid.z);
    const V3 sh = R.to_local(v3(c.x - c0.x, c.y - c0.y, c.z - c0.z));
    const float l3[3] = {blo.x - sh.x, blo.y - sh.y, blo.z - sh.z}, h3[3] = {bhi.x - sh.x, bhi.y - sh.y, bhi.z - sh.z};
    const float ext[3] = {fmaxf(fabsf(lo.x - sh.x), fabsf(hi.x - sh.x)), fmaxf(fabsf(lo.y - sh.y), fabsf(hi.y - sh.y)),
                          fmaxf(fabsf(lo.z - sh.z), fabsf(hi.z - sh.z))};
    // coordinates beyond 2^100 (or overflowed ones): boxes that contain every point
    const bool huge = !(ext[0] < 0x1p100f && ext[1] < 0x1p100f && ext[2] < 0x1p100f);
    if (huge) {
        c = v3(0.f, 0.f, 0.f);
        nx = ny = 0.0f;
    }
    uint32_t exps = 0, plo = 0, phi = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        // the smallest step with ext <= 126 steps (ext / 126 with a margin for its
        // rounding, up to the next power of two), at least 2^-60 (a query's offset in
        // steps overflows only where its square does)
        const uint32_t step = (__float_as_uint(ext[k] * (1.00001f / 126.0f)) + 0x7FFFFFu) >> 23;
        const uint32_t e = huge ? 253u : max(step, 67u);
        exps |= e << (8 * k);
        const float inv = __uint_as_float((254u - e) << 23);
        uint32_t ql = (uint32_t)__builtin_amdgcn_fmed3f(floorf(fmaf(l3[k], inv, 128.0f)), 0.0f, 255.0f);
        uint32_t qh = (uint32_t)__builtin_amdgcn_fmed3f(ceilf(fmaf(h3[k], inv, 128.0f)), 0.0f, 255.0f);
        if (huge || empty) {
            ql = empty ? 255u : 0u;
            qh = 255u - ql;
        }
        plo |= ql << (8 * k);
        phi |= qh << (8 * k);
    }
    // rows of bytes gathered from the four children; the first four lanes write a quarter
    // of the node each
    uint32_t vl[4], vh[4], kid[4], row[6];
    from_children<LPC>(plo, vl);
    from_children<LPC>(phi, vh);
    from_children<LPC>(ch, kid);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        row[k] = row[3 + k] = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            row[k] |= ((vl[q] >> (8 * k)) & 0xFFu) << (8 * q);
            row[3 + k] |= ((vh[q] >> (8 * k)) & 0xFFu) << (8 * q);
        }
    }
    if (l < 4) {
        uint4 w = make_uint4(__float_as_uint(c.x), __float_as_uint(c.y), __float_as_uint(c.z), exps);
        if (l == 1) w = make_uint4(__float_as_uint(nx), __float_as_uint(ny), kid[0], kid[1]);
        if (l == 2) w = make_uint4(kid[2], kid[3], row[0], row[1]);
        if (l == 3) w = make_uint4(row[2], row[3], row[4], row[5]);
        reinterpret_cast<uint4*>(a.out + i)[l] = w;
    }
}

__device__ __forceinline__ uint32_t node_tris(const WNode<4>* __restrict__ nodes, uint32_t i) {
    const uint4 v = *reinterpret_cast<const uint4*>(nodes[i].aux);
    return v.x + v.y + v.z + v.w;  // 0 for empty slots
}

// Wave w of nw makes the large nodes among w, w + nw, w + 2 nw, ... (nodes lie in level
// order, large ones first: 16 consecutive ones per wave took 164 us for the 44 K nodes of a
// refit, the root's neighbours being made in turn by one wave), then the others of its 16
// consecutive ones, which share triangles in the caches.  Making a node is a chain of
// dependent loads (node, child's range, triangles), so as many as the lanes allow are made
// side by side.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_orient(OrientArgs a) {
    if (a.skip && *a.skip) return;
    const uint32_t n = a.n_dev ? a.n_dev[0] : a.n;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nw = gridDim.x * (kBlock / 64);
    const uint32_t w = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6));
    for (uint32_t k0 = 0; (uint64_t)k0 * nw + w < n; k0 += 64) {
        const uint64_t i = (uint64_t)(k0 + lane) * nw + w;
        const uint32_t t = i < n ? node_tris(a.nodes, (uint32_t)i) : 0u;
        uint64_t large = __ballot(t > kOrientRow && t <= kOrientMax);
        while (large) {
            orient_node<16>(a, (k0 + (uint32_t)__builtin_ctzll(large)) * nw + w);
            large &= large - 1;
        }
    }
    for (uint32_t base = w * 16u; base < n; base += nw * 16u) {
        const uint32_t i = base + (lane >> 2);
        const uint32_t t = i < n ? node_tris(a.nodes, i) : 0u;
        uint64_t rows = __ballot(t > kOrientQuad && t <= kOrientRow) & 0x1111111111111111ull;
        while (rows) {  // four at a time, one per row of lanes
            const uint32_t g = lane >> 4;
            if (g < (uint32_t)__popcll(rows)) orient_node<4>(a, base + (nth_set_bit(rows, g) >> 2));
            for (uint32_t r = 0; r < 4; r++) rows &= rows - 1;  // (0 stays 0)
        }
        if (i < n && (t <= kOrientQuad || t > kOrientMax)) orient_node<1>(a, i);
    }
}

void launch_orient(const void* nodes, const uint32_t* first, const float4* tris, void* onodes, uint32_t n_host,
                   uint32_t capacity, const uint32_t* n_dev, const uint32_t* scale, uint32_t scale_stride,
                   const uint32_t* seg, const uint32_t* skip, hipStream_t s) {
    const uint32_t n = n_dev ? capacity : n_host;
    if (n == 0) return;
    OrientArgs a{static_cast<const WNode<4>*>(nodes), first, tris, static_cast<ONode*>(onodes), n_dev, n_host,
                 scale, scale_stride, seg, skip};
    hipLaunchKernelGGL(k_orient, dim3(std::min(cdiv(n, 4 * (kBlock / 64)), 4096u)), dim3(kBlock), 0, s, a);
}

}  // namespace gpurt_impl
