// treelet.hip -- SAH treelet restructuring of the binary LBVH (Karras & Aila, "Fast
// Parallel Construction of High-Quality Bounding Volume Hierarchies", HPG 2013).
//
// For every internal node r with more than 2 leaf_size triangles, bottom-up:
//   1. form a treelet: start from r's two children and repeatedly open the treelet leaf
//      (an internal node) with the largest surface area, up to N leaves (N = 5..7), one
//      candidate per lane;
//   2. find the binary topology over those leaves with the least SAH cost by dynamic
//      programming over all 2^N - 1 leaf subsets (one 64-lane wave per treelet: each
//      subset tries every split that keeps its lowest leaf on one side);
//   3. if it is cheaper than the current one, rewrite the treelet's N - 1 internal nodes
//      (r keeps its index, so ancestors are untouched) with their new children, boxes,
//      triangle counts and costs.
// Bottom-up order: one launch per Karras prefix length, largest first (the roots are bucketed
// by it).  Two roots of one launch have equal prefix length, so neither is an
// ancestor of the other and their treelets are disjoint; everything below a root was
// finished by earlier launches.  (That argument holds for the tree as Karras built it,
// so one round is supported.)  Subtrees of <= leaf_size triangles become single leaves
// in the wide collapse and are priced as leaves, so they are never restructured.
#include <algorithm>
#include <type_traits>

#include "build_common.h"

namespace gpurt_impl {

// What each lane does in the dynamic programme is the same for every treelet, so it is a
// table: subsets of one size k are dealt to groups of lanes(N, k) lanes, and a lane's
// splits P (the side that holds the subset's lowest leaf) are the bytes of its words, in
// descending order.
constexpr int choose(int n, int k) {
    int c = 1;
    for (int j = 1; j <= k; j++) c = c * (n - j + 1) / j;
    return c;
}
constexpr int splits(int k) { return (1 << (k - 1)) - 1; }
constexpr int lanes(int n, int k) {  // per subset: a power of two, at most one split each
    int l = 1;
    while (2 * l * choose(n, k) <= 64 && l < splits(k)) l *= 2;
    return l;
}
constexpr int rounds(int n, int k) { return (splits(k) + lanes(n, k) - 1) / lanes(n, k); }
constexpr int words(int n, int k) { return (rounds(n, k) + 3) / 4; }
constexpr int first_word(int n, int k) {  // word 0, 1: the lane's subsets of sizes 2..7
    int w = 2;
    for (int j = 2; j < k; j++) w += words(n, j);
    return w;
}
template <int N>
struct TreeletTab {
    static constexpr int kWords = first_word(N, N + 1);
    uint32_t w[64][kWords];
};
template <int N>
constexpr TreeletTab<N> make_treelet_tab() {
    TreeletTab<N> t{};
    for (int k = 2; k <= N; k++) {
        const int L = lanes(N, k);
        int idx = 0;
        for (int sub = 1; sub < (1 << N); sub++) {
            int bits = 0;
            for (int j = 0; j < N; j++) bits += (sub >> j) & 1;
            if (bits != k) continue;
            for (int l = 0; l < L; l++) t.w[idx * L + l][(k - 2) / 4] |= (uint32_t)sub << (8 * ((k - 2) % 4));
            const int low = sub & -sub;
            int s = 0;  // splits in descending order, dealt to the group's lanes in turn
            for (int P = (sub - 1) & sub; P; P = (P - 1) & sub) {
                if (!(P & low)) continue;
                const int lane = idx * L + s % L, r = s / L;
                t.w[lane][first_word(N, k) + r / 4] |= (uint32_t)P << (8 * (r % 4));
                s++;
            }
            idx++;
        }
    }
    return t;
}
template <int N>
__device__ const TreeletTab<N> kTreeletTab = make_treelet_tab<N>();

// minimum / maximum of a lane's value and a wave-uniform one, as the instruction (fminf and
// fmaxf quiet signalling NaNs before it)
__device__ __forceinline__ float min_u(float v, float u) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "s"(u), "v"(v));
    return r;
}
__device__ __forceinline__ float max_u(float v, float u) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "s"(u), "v"(v));
    return r;
}
__device__ __forceinline__ float read_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
// the value of a lane of the other half of an aligned group of 2 o lanes whose halves are
// uniform below o
template <int O>
__device__ __forceinline__ int other_half(int v) {
    if constexpr (O == 1) return dpp<0xB1>(v);
    else if constexpr (O == 2) return dpp<0x4E>(v);
    else if constexpr (O == 4) return dpp<0x141>(v);   // half-row mirror
    else if constexpr (O == 8) return dpp<0x140>(v);   // row mirror
    else return __shfl_xor(v, O);
}

// Least-cost split of the lane's subset of size K; the group's first lane writes it.
// copt[0] = inf stands for the splits a lane does not have.
template <int N, int K>
__device__ __forceinline__ void dp_step(const uint32_t (&tab)[TreeletTab<N>::kWords], int full, const float* base,
                                        float* copt, uint8_t* part) {
    constexpr int L = lanes(N, K), R = rounds(N, K), W0 = first_word(N, K);
    const int sub = (int)((tab[(K - 2) / 4] >> (8 * ((K - 2) % 4))) & 0xFFu);
    float best = INFINITY;
    int bp = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int P = (int)((tab[W0 + r / 4] >> (8 * (r % 4))) & 0xFFu);
        const float c = copt[P] + copt[sub ^ P];
        if (c < best) {
            best = c;
            bp = P;
        }
    }
    // over the group's lanes; ties go to the larger P
    auto fold = [&](auto tag) {
        constexpr int O = decltype(tag)::value;
        if constexpr (O < L) {
            const float oc = __int_as_float(other_half<O>(__float_as_int(best)));
            const int op = other_half<O>(bp);
            if (oc < best || (oc == best && op > bp)) {
                best = oc;
                bp = op;
            }
        }
    };
    fold(std::integral_constant<int, 1>{});
    fold(std::integral_constant<int, 2>{});
    fold(std::integral_constant<int, 4>{});
    fold(std::integral_constant<int, 8>{});
    fold(std::integral_constant<int, 16>{});
    fold(std::integral_constant<int, 32>{});
    if (sub && !(sub & ~full) && (int)(threadIdx.x % L) == 0) {
        const float b = base[sub];
        copt[sub] = __float_as_uint(b) >> 31 ? -b : b + best;
        part[sub] = (uint8_t)bp;
    }
    __syncthreads();
    if constexpr (K < N) dp_step<N, K + 1>(tab, full, base, copt, part);
}

// A treelet is a chain -- opening a node waits for its children's records, a subset's cost
// for the smaller ones' -- so what counts is the length of the chain and, on levels with
// many roots, the instructions.  With the lane's part of the programme in registers, the
// treelet's boxes as wave-uniform operands and one box per lane and subset a treelet takes
// about a quarter of the instructions of a version that enumerated submasks as it went
// (3800), and the treelet passes of a 2.3 M triangle build 1.6 instead of 3.8 ms.
template <int N>
__global__ __launch_bounds__(64) void k_treelet(int level, const uint32_t* __restrict__ lvl_begin,
                                                const uint32_t* __restrict__ lvl_order, int leaf_size,
                                                float4* bnode, const float4* __restrict__ saabb) {
    constexpr int NS = 1 << N;
    constexpr int kWords = TreeletTab<N>::kWords;
    __shared__ uint32_t s_int[N];
    // per subset: kCi * area, or -(kCt * area * triangles) where it becomes one leaf
    __shared__ float s_base[NS];
    __shared__ float s_copt[NS];
    __shared__ uint32_t s_cnt[NS];
    __shared__ float4 s_lo[NS], s_hi[NS];
    __shared__ uint8_t s_part[NS];
    const int lane = threadIdx.x;
    // one wave per treelet root of this prefix length: the roots with more than
    // 2 leaf_size triangles (the others become at most two leaves of one
    // wide node, where a new topology gains nothing measurable -- rays_scene: skipping them
    // builds in 10.7 instead of 13.4 ms with the same ray times; skipping up to 16 or 32
    // triangles builds faster still but costs 2-5% in ray time)
    const uint32_t beg = lvl_begin[level], end = lvl_begin[level + 1];
    if (beg + blockIdx.x >= end) return;
    uint32_t tab[kWords];
#pragma unroll
    for (int k = 0; k < kWords; k++) tab[k] = kTreeletTab<N>.w[lane][k];
    if (lane == 0) s_copt[0] = INFINITY;
    for (uint32_t k = beg + blockIdx.x; k < end; k += gridDim.x) {
        const int r = (int)lvl_order[k];
        // Form the treelet with one candidate (treelet leaf) per lane: a lane that takes a
        // candidate loads its record (for a triangle its box), so opening a node costs one
        // round of loads by the two lanes that receive its children.  The node opened is
        // the internal candidate with the largest surface area, the lowest slot on ties.
        uint32_t x = kEmpty, xl = 0, xr = 0, xc = 0;
        float4 xlo = make_float4(0.f, 0.f, 0.f, 0.f), xhi = xlo;
        float xcost = 0.0f, xarea = -1.0f;
        auto take = [&](uint32_t ref) {
            x = ref;
            ref_box(ref, saabb, bnode, xlo, xhi);
            const float a = box_area(xlo, xhi);
            if (ref & kLeafBit) {
                xc = 1u;
                xcost = kCt * a;
                xarea = -1.0f;  // not openable
            } else {
                const float4 y = bnode[3 * (size_t)ref + 2];
                xc = __float_as_uint(y.x);
                xcost = y.y;
                xl = __float_as_uint(xlo.w);
                xr = __float_as_uint(xhi.w);
                xarea = a > -1.0f ? a : -1.0f;  // (a NaN area is never opened)
            }
        };
        const float4 rlo = bnode[3 * (size_t)r], rhi = bnode[3 * (size_t)r + 1];
        const float4 rx = bnode[3 * (size_t)r + 2];
        const uint32_t rc = __float_as_uint(rx.x);
        if (lane < 2) take(__float_as_uint(lane ? rhi.w : rlo.w));
        // the root's cost, refreshed from its (finished) children, the first two candidates
        const float cur = sah_node_cost(rlo, rhi, rc, read_lane(xcost, 0), read_lane(xcost, 1), leaf_size);
        if (lane == 0) {
            bnode[3 * (size_t)r + 2].y = cur;
            s_int[0] = (uint32_t)r;
        }
        int nl = 2, ni = 1;
        while (nl < N) {
            const float a = lane < nl ? xarea : -1.0f;
            float m = a;  // N <= 7: lanes 0..7 hold every candidate
            m = fmaxf(m, __int_as_float(dpp<0xB1>(__float_as_int(m))));
            m = fmaxf(m, __int_as_float(dpp<0x4E>(__float_as_int(m))));
            m = fmaxf(m, __int_as_float(dpp<0x141>(__float_as_int(m))));
            m = read_lane(m, 0);
            if (m < 0.0f) break;  // no internal candidate left
            const int jb = (int)__builtin_ctzll(__ballot(lane < nl && a == m));
            const uint32_t ob = __builtin_amdgcn_readlane(x, jb), lb = __builtin_amdgcn_readlane(xl, jb),
                           rb = __builtin_amdgcn_readlane(xr, jb);
            if (lane == 0) s_int[ni] = ob;
            ni++;
            if (lane == jb || lane == nl) take(lane == jb ? lb : rb);
            nl++;
        }
        const int full = (1 << nl) - 1;
        // Boxes and counts: lane s makes subset s of the first six leaves, and with the
        // seventh (N = 7) subset 64 + s.  (Leaves past nl belong to no subset of full.)
        float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.0f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
        uint32_t c = 0;
        auto add_leaf = [&](int j) {
            const float lx = read_lane(xlo.x, j), ly = read_lane(xlo.y, j), lz = read_lane(xlo.z, j);
            const float hx = read_lane(xhi.x, j), hy = read_lane(xhi.y, j), hz = read_lane(xhi.z, j);
            const uint32_t n = __builtin_amdgcn_readlane(xc, j);
            if (j == 6 || (lane & (1 << j))) {
                lo.x = min_u(lo.x, lx); lo.y = min_u(lo.y, ly); lo.z = min_u(lo.z, lz);
                hi.x = max_u(hi.x, hx); hi.y = max_u(hi.y, hy); hi.z = max_u(hi.z, hz);
                c += n;
            }
        };
        auto put = [&](int sub) {
            const float a = box_area(lo, hi);
            s_lo[sub] = lo;
            s_hi[sub] = hi;
            s_cnt[sub] = c;
            s_base[sub] = c <= (uint32_t)leaf_size ? -(kCt * a * (float)c) : kCi * a;
        };
#pragma unroll
        for (int j = 0; j < (N < 6 ? N : 6); j++) add_leaf(j);
        if (lane < NS) put(lane);
        if constexpr (N == 7) {
            add_leaf(6);
            put(64 + lane);
        }
        if (lane < nl) {
            s_copt[1 << lane] = xcost;
        }
        __syncthreads();
        dp_step<N, 2>(tab, full, s_base, s_copt, s_part);
        // Rebuild the treelet top-down from the optimal partitions, reusing its internal node
        // indices (r first).  The walk over the partitions is a serial chain, so it only
        // deals the subsets: it runs in scalar registers, with the partitions of all subsets
        // in vector ones, and lane t keeps subset t; then every lane writes the record of
        // its own.  (One lane that read a partition from LDS and wrote a record in turn was
        // a third of the time, and its stacks cost the registers of a fourth wave per SIMD:
        // a 2.3 M triangle build 2.83 -> 2.33 ms.)
        if (nl >= 3 && s_copt[full] < cur * (1.0f - 1e-5f)) {
            const uint32_t parts_lo = lane < NS ? s_part[lane] : 0u;
            const uint32_t parts_hi = NS > 64 ? s_part[64 + lane] : 0u;
            int made = 1;                // subsets dealt; subset t's node is s_int[t]
            uint32_t mine = (uint32_t)full, k0 = 0, k1 = 0;
            for (int t = 0; t < made; t++) {
                const uint32_t sub = __builtin_amdgcn_readlane(mine, t);
                const uint32_t P = sub < 64 ? __builtin_amdgcn_readlane(parts_lo, sub)
                                            : __builtin_amdgcn_readlane(parts_hi, sub - 64);
                uint32_t ref[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint32_t part = h ? sub ^ P : P;
                    if ((part & (part - 1)) == 0) {
                        ref[h] = __builtin_amdgcn_readlane(x, __builtin_ctz(part));
                    } else {
                        ref[h] = s_int[made];
                        if (lane == made) mine = part;
                        made++;
                    }
                }
                if (lane == t) {
                    k0 = ref[0];
                    k1 = ref[1];
                }
            }
            // (a rewritten node's sorted primitives are no longer one range: its first
            // field is unused, the leaves are re-packed)
            if (lane < made) {
                const uint32_t node = s_int[lane];
                const float4 l = s_lo[mine], h = s_hi[mine];
                bnode[3 * (size_t)node] = make_float4(l.x, l.y, l.z, __uint_as_float(k0));
                bnode[3 * (size_t)node + 1] = make_float4(h.x, h.y, h.z, __uint_as_float(k1));
                bnode[3 * (size_t)node + 2] = make_float4(__uint_as_float(s_cnt[mine]), s_copt[mine], 0.0f, 0.0f);
            }
        }
        __syncthreads();
    }
}

template <int N>
static void launch_treelet_levels(BuildBufs& b, int key_bits, int nbits, hipStream_t s) {
    const unsigned grid = std::min(cdiv(b.N, 64), 8192u);
    for (int level = 95; level >= 64 - key_bits; level--) {
        if (level >= 64 && level < 96 - nbits) continue;
        hipLaunchKernelGGL(k_treelet<N>, dim3(grid), dim3(64), 0, s, level, b.lvl_begin, b.lvl_order, b.leaf_size,
                           b.bnode, b.saabb);
    }
}

int run_treelets(BuildBufs& b, int treelet_size, int rounds, int key_bits, int nbits, hipStream_t s) {
    // buckets (b.lvl_begin / b.lvl_order) were filled by k_level_hist, scan and scatter
    if (rounds > 1)
        return set_error(GPURT_E_UNSUPPORTED, "treelet_rounds > 1 is not supported (one bottom-up round)");
    if (b.N < 3) return GPURT_OK;
    switch (treelet_size) {
        case 5: launch_treelet_levels<5>(b, key_bits, nbits, s); break;
        case 6: launch_treelet_levels<6>(b, key_bits, nbits, s); break;
        case 7: launch_treelet_levels<7>(b, key_bits, nbits, s); break;
        default: return set_error(GPURT_E_UNSUPPORTED, "treelet_size must be 5..7");
    }
    GPURT_HIP(hipGetLastError());
    return GPURT_OK;
}

}  // namespace gpurt_impl
