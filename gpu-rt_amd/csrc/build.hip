// build.hip -- GPU BVH builder for gfx950.
//
// Replaces the driver build behind VK::Accel::recreate(const Mesh&)
// (src/vk/vulkan.cpp:881-936 -> vkCmdBuildAccelerationStructuresKHR at :877).
//
// Pipeline (every stage is one launch over ALL meshes of the build; a plain build is a
// batch of one mesh):
//   k_prep         centroid bounds and coordinate scale per mesh (wave-reduced,
//                  ordered-uint atomics), triangle box centres
//   k_morton       key = mesh_id << 30 | 30-bit Morton code of the box centre over the
//                  mesh's centroid bounds; value = triangle index
//   radix sort     LSD, 8-bit digits, LDS histograms + LDS ranking by wave ballots
//                  (stable, so equal codes stay in triangle order); one block up to 8192
//   k_pack         triangles and boxes gathered into sorted (leaf) order
//   k_tree_local   Karras (HPG 2012) binary radix tree over the sorted keys; because the
//                  mesh id is in the high key bits every mesh is one subtree, whose root
//                  is recorded.  With it the boxes of nodes inside a chunk of 256 leaves,
//                  bottom-up by one block
//   k_range_top, k_boxes_cross
//                  the other nodes' boxes, as unions over their leaf range (no atomics, no
//                  order)
//   k_treelet      optional SAH treelet restructuring (treelet.hip), roots bucketed by
//                  k_level_hist / scan / scatter
//   k_collapse_head, k_collapse, k_collapse_tail
//                  the first levels in one launch, one launch per wide level, the last
//                  levels in one: a node opens the child with the largest surface area
//                  until it has W children; subtrees of <= leaf_size triangles become
//                  leaves (contiguous ranges of packed triangles, gathered by k_repack
//                  after treelets)
#include <algorithm>
#include <cstring>
#include <vector>

#include "build_common.h"
#include "index_math.h"

namespace gpurt_impl {

// ------------------------------------------------------------------------------------
// helpers
// ------------------------------------------------------------------------------------

__device__ __forceinline__ uint32_t expand_bits10(uint32_t x) {
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000FFu;
    x = (x | (x << 8)) & 0x0300F00Fu;
    x = (x | (x << 4)) & 0x030C30C3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

__device__ __forceinline__ uint32_t quant10(float c, float lo, float inv) {
    float f = ((c - lo) * inv) * 1024.0f;
    int v = (int)floorf(f);
    if (!(f >= 0.0f)) v = 0;
    if (v > 1023) v = 1023;
    return (uint32_t)v;
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}

__device__ __forceinline__ int find_seg(const SegDesc* segs, int n_seg, uint32_t g) {
    int lo = 0, hi = n_seg - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (segs[mid].tri_offset <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}


// Clears what the build accumulates into.  A plain build hands its one mesh over as an
// argument (no copy to the device to wait for).
__global__ void k_init_build(SegDesc* segs, int n_seg, SegDesc one, int has_one, uint32_t* segstat_rep, uint32_t* seg_root,
                             uint32_t* report, uint32_t* lvl_hist) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_seg * kRep) {
        uint32_t* st = segstat_rep + (size_t)i * kStat;
        for (int k = 0; k < 3; k++) {
            st[k] = 0xFFFFFFFFu;
            st[3 + k] = 0u;
        }
        st[6] = 0u;
        st[7] = 0u;
    }
    if (i == 0 && has_one) segs[0] = one;
    // single-triangle mesh: leaf root
    if (i < n_seg) seg_root[i] = kLeafBit | (has_one ? one.tri_offset : segs[i].tri_offset);
    // level 0 and the wide nodes start with one node per mesh; everything else is zero
    if (i < kReportWords) report[i] = (i == kReportLvl || i == kReportCounters) ? (uint32_t)n_seg : 0u;
    if (i < (int)kLevelBuckets) lvl_hist[i] = 0u;
}

// folds the kRep replicas of every mesh's statistics into segstat
__global__ void k_reduce_stats(int n_seg, const uint32_t* __restrict__ segstat_rep,
                               uint32_t* __restrict__ segstat) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_seg * kStat) return;
    const int sgi = i / kStat, k = i % kStat;
    const bool is_min = k < 3;
    uint32_t v = is_min ? 0xFFFFFFFFu : 0u;
#pragma unroll 16
    for (int r = 0; r < kRep; r++) {
        uint32_t x = segstat_rep[((size_t)r * n_seg + sgi) * kStat + k];
        v = is_min ? min(v, x) : max(v, x);
    }
    segstat[i] = v;
}

// ------------------------------------------------------------------------------------
// k_prep: box centres + per-mesh centroid bounds
// ------------------------------------------------------------------------------------

// A mesh's running bounds in the lanes of a wave (ordered uints): centroid minimum and
// maximum, largest |coordinate|.
struct WaveStats {
    uint32_t o[7];
    __device__ __forceinline__ void reset() {
        for (int a = 0; a < 3; a++) {
            o[a] = 0xFFFFFFFFu;
            o[3 + a] = 0u;
        }
        o[6] = 0u;
    }
    // wave-reduced into mesh s of a replica, one atomic per word (all lanes call it)
    __device__ __forceinline__ void flush(uint32_t* segstat, int s) {
        for (int a = 0; a < 3; a++) {
            o[a] = wave_min_u32(o[a]);
            o[3 + a] = wave_max_u32(o[3 + a]);
        }
        o[6] = wave_max_u32(o[6]);
        if ((threadIdx.x & 63) == 0) {
            for (int a = 0; a < 3; a++) {
                atomicMin(&segstat[s * kStat + a], o[a]);
                atomicMax(&segstat[s * kStat + 3 + a], o[3 + a]);
            }
            atomicMax(&segstat[s * kStat + 6], o[6]);
        }
        reset();
    }
};

// Each wave takes `rounds` x 64 consecutive triangles and keeps its mesh's bounds in
// registers until the mesh ends: one set of atomics per wave and mesh.  (With a set per 64
// triangles the same-address atomics were most of the kernel: 182 us for 2.3 M triangles.)
__global__ __launch_bounds__(kBlock) void k_prep(const SegDesc* __restrict__ segs, int n_seg,
                                                 uint32_t N, int rounds, float4* __restrict__ cen,
                                                 uint32_t* __restrict__ segstat,
                                                 uint32_t* __restrict__ counters) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    const uint32_t beg = wave * (uint32_t)rounds * 64u;
    if (beg >= N) return;
    segstat += (size_t)(wave % kRep) * n_seg * kStat;
    WaveStats ws;
    ws.reset();
    int s = find_seg(segs, n_seg, beg);  // mesh of the wave's running bounds
    SegDesc sd = segs[s];
    for (int r = 0; r < rounds; r++) {
        const uint32_t g0 = beg + (uint32_t)r * 64u, g = g0 + lane;
        if (g0 >= N) break;
        const bool valid = g < N;
        const uint32_t last = min(g0 + 63u, N - 1u);
        // most rounds lie in one mesh; the others search per lane
        if (g0 >= sd.tri_offset + sd.n_tris) {
            ws.flush(segstat, s);
            s = find_seg(segs, n_seg, g0);
            sd = segs[s];
        }
        const bool uniform = last < sd.tri_offset + sd.n_tris;
        const int sl = uniform || !valid ? s : find_seg(segs, n_seg, g);
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        float c[3] = {0.f, 0.f, 0.f};
        float amax = 0.0f;
        if (valid) {
            const SegDesc d = uniform ? sd : segs[sl];
            const uint32_t t = g - d.tri_offset;
            uint32_t vi[3];
            bool bad = false;
            for (int k = 0; k < 3; k++) {
                vi[k] = d.idx[3 * (size_t)t + k];
                if (vi[k] >= d.n_verts) { bad = true; vi[k] = 0; }
            }
            if (bad) atomicOr(&counters[1], 1u);
            float v[3][3];
            bool finite = true;
            for (int k = 0; k < 3; k++) {
                const float* p = d.verts + (size_t)vi[k] * d.vstride;
                v[k][0] = p[0]; v[k][1] = p[1]; v[k][2] = p[2];
                finite = finite && isfinite(v[k][0]) && isfinite(v[k][1]) && isfinite(v[k][2]);
            }
            // a non-finite position is reported (the build fails with GPURT_E_INVALID); the
            // triangle's box is then the origin so every later stage works on finite boxes
            if (!finite) atomicOr(&counters[1], 4u);
            for (int a = 0; a < 3; a++) {
                for (int k = 0; k < 3; k++) {
                    const float x = finite ? v[k][a] : 0.0f;
                    lo[a] = fminf(lo[a], x);
                    hi[a] = fmaxf(hi[a], x);
                    amax = fmaxf(amax, fabsf(x));
                }
                c[a] = (lo[a] + hi[a]) * 0.5f;
            }
            cen[g] = make_float4(c[0], c[1], c[2], __uint_as_float((uint32_t)sl));
        }
        if (uniform) {
            if (valid) {
                for (int a = 0; a < 3; a++) {
                    ws.o[a] = min(ws.o[a], f2o(c[a]));
                    ws.o[3 + a] = max(ws.o[3 + a], f2o(c[a]));
                }
                ws.o[6] = max(ws.o[6], f2o(amax));
            }
        } else if (valid) {
            for (int a = 0; a < 3; a++) {
                atomicMin(&segstat[sl * kStat + a], f2o(c[a]));
                atomicMax(&segstat[sl * kStat + 3 + a], f2o(c[a]));
            }
            atomicMax(&segstat[sl * kStat + 6], f2o(amax));
        }
    }
    ws.flush(segstat, s);
}

__global__ __launch_bounds__(kBlock) void k_morton(uint32_t N, const float4* __restrict__ cen,
                                                   const uint32_t* __restrict__ segstat,
                                                   uint64_t* __restrict__ keys) {
    uint32_t g = blockIdx.x * kBlock + threadIdx.x;
    if (g >= N) return;
    const float4 c4 = cen[g];
    const uint32_t s = __float_as_uint(c4.w);
    const uint32_t* st = segstat + s * kStat;
    const float c[3] = {c4.x, c4.y, c4.z};
    uint32_t q[3];
    for (int a = 0; a < 3; a++) {
        float l = o2f(st[a]), h = o2f(st[3 + a]);
        float inv = h > l ? 1.0f / (h - l) : 0.0f;
        q[a] = quant10(c[a], l, inv);
    }
    uint32_t code = (expand_bits10(q[0]) << 2) | (expand_bits10(q[1]) << 1) | expand_bits10(q[2]);
    keys[g] = ((uint64_t)s << 30) | code;
}

// ------------------------------------------------------------------------------------
// LSD radix sort of (uint64 or uint32 key, uint32 index), 8-bit digits, stable
// ------------------------------------------------------------------------------------

constexpr int kSortItems = 16;
constexpr int kSortTile = kBlock * kSortItems;
constexpr int kSortThreads = 512;  // of the scatter

template <typename K>
__global__ __launch_bounds__(kBlock) void k_radix_hist(const K* __restrict__ keys, uint32_t n,
                                                       int shift, uint32_t* __restrict__ hist,
                                                       uint32_t nblocks) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t base = blockIdx.x * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortItems; r++) {
        uint32_t i = base + r * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Exclusive scan of each digit's counts over the blocks (block d scans row d); the row's
// total goes to row_total[d].  The scatter adds the digits before its own from the 256
// totals, so the counts need one launch between histogram and scatter (tile sums, a scan
// of the sums and their application were three: 16 us of a pass on 2.3 M pairs, all
// launch and round trip).
__global__ __launch_bounds__(kBlock) void k_scan_rows(uint32_t* __restrict__ hist, uint32_t nblocks,
                                                      uint32_t* __restrict__ row_total) {
    __shared__ uint32_t wsum[kBlock / 64];
    uint32_t* row = hist + (size_t)blockIdx.x * nblocks;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t run = 0;
    for (uint32_t b0 = 0; b0 < nblocks; b0 += kBlock) {
        const uint32_t b = b0 + tid;
        const uint32_t v = b < nblocks ? row[b] : 0u;
        uint32_t x = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d);
            if (lane >= (uint32_t)d) x += y;
        }
        __syncthreads();  // the last round's sums have been read
        if (lane == 63u) wsum[wave] = x;
        __syncthreads();
        uint32_t before = run;
#pragma unroll
        for (uint32_t w = 0; w < kBlock / 64; w++) {
            if (w < wave) before += wsum[w];
            run += wsum[w];
        }
        if (b < nblocks) row[b] = before + x - v;
    }
    if (tid == 0) row_total[blockIdx.x] = run;
}

// Scatter of one radix pass.  The block's tile (kSortTile pairs) is first ordered by
// digit in LDS, stably, and then written out in that order, so each digit's run of the
// tile (16 pairs on average) leaves as one contiguous stretch of the output instead of
// one isolated write per pair.  Each wave ranks its own 512 consecutive pairs: per round
// of 64, an 8-ballot multisplit ranks the lanes of equal digit, and a wave-private LDS
// counter per digit (read by all lanes, advanced by each group's first lane; a wave's LDS
// operations complete in order) carries the rank across rounds, so the rounds need no
// block barrier.  One scan over (digit, wave) counts then gives every wave's first slot
// per digit.  Bound by the latency of that chain, not by memory, so what counts is waves in
// flight: the values pass through the LDS that the keys have left, and with 16-bit counts
// a CU holds 3-4 blocks of 8 waves (2 of 4 waves with keys and values side by side): 2.3 M
// pairs of 12 bytes 30.5 -> 16.5 us a pass, 3.1 M of 8 bytes (33 us as 12) 17 us, 3.5 TB/s.
template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_radix_scatter(const K* __restrict__ kin,
                                                                const uint32_t* __restrict__ vin,
                                                                K* __restrict__ kout, uint32_t* __restrict__ vout,
                                                                uint32_t n, int shift,
                                                                const uint32_t* __restrict__ offs,
                                                                const uint32_t* __restrict__ row_total,
                                                                uint32_t nblocks) {
    constexpr int kWaves = kSortThreads / 64;
    constexpr int kItems = kSortTile / kSortThreads;
    constexpr uint32_t kWaveItems = 64 * kItems;  // consecutive pairs per wave
    static_assert(kSortTile <= 65535, "16-bit slots");
    __shared__ K skey[kSortTile];            // keys in slot order, then the values
    __shared__ uint32_t gofs[256];           // output slot of digit d less its first LDS slot
    __shared__ uint16_t wcnt[kWaves][256];   // a wave's pairs of digit d, then its first slot
    __shared__ uint32_t wsum[2][4];
    uint32_t* const sval = reinterpret_cast<uint32_t*>(skey);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t tile = blockIdx.x * kSortTile;
    const uint32_t m = min((uint32_t)kSortTile, n - tile);
    const uint32_t wbase = (uint32_t)wave * kWaveItems + (uint32_t)lane;
    K key[kItems];
    uint32_t val[kItems], rank[kItems];
#pragma unroll
    for (int r = 0; r < kItems; r++) {
        const uint32_t i = wbase + (uint32_t)r * 64u;
        key[r] = i < m ? kin[tile + i] : (K)0;
        val[r] = !vin ? tile + i : i < m ? vin[tile + i] : 0u;
    }
    // this block's first output slot of digit tid: the digits before it, then its row
    uint32_t dtot = 0, dincl = 0, row = 0;
    if (tid < 256) {
        dtot = dincl = row_total[tid];
        row = offs[(size_t)tid * nblocks + blockIdx.x];
    }
    for (int k = tid; k < kWaves * 256; k += kSortThreads) wcnt[k >> 8][k & 255] = 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t x = __shfl_up(dincl, off);
        if (lane >= off) dincl += x;
    }
    if (tid < 256 && lane == 63) wsum[0][wave] = dincl;
    __syncthreads();
    uint16_t* const mycnt = wcnt[wave];
    const uint64_t lt_mask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
#pragma unroll
    for (int r = 0; r < kItems; r++) {
        const bool valid = wbase + (uint32_t)r * 64u < m;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint64_t bb = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bb : ~bb;
        }
        const uint32_t rk = (uint32_t)__popcll(peers & lt_mask);
        const uint32_t before = mycnt[d];
        rank[r] = before + rk;
        if (valid && rk == 0) mycnt[d] = (uint16_t)(before + (uint32_t)__popcll(peers));
    }
    __syncthreads();
    // digit tid: the tile's count and every wave's first slot inside the digit's run, from
    // an exclusive scan of the 256 totals within each wave by shuffles, then across
    uint32_t tot = 0, incl = 0;
    if (tid < 256) {
#pragma unroll
        for (int w = 0; w < kWaves; w++) tot += wcnt[w][tid];
        incl = tot;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t x = __shfl_up(incl, off);
            if (lane >= off) incl += x;
        }
        if (lane == 63) wsum[1][wave] = incl;
    }
    __syncthreads();
    if (tid < 256) {
        uint32_t start = incl - tot, base = dincl - dtot + row;
        for (int w = 0; w < wave; w++) {
            start += wsum[1][w];
            base += wsum[0][w];
        }
        gofs[tid] = base - start;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const uint32_t c = wcnt[w][tid];
            wcnt[w][tid] = (uint16_t)start;
            start += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; r++) {
        rank[r] += mycnt[(uint32_t)(key[r] >> shift) & 255u];  // the pair's slot
        if (wbase + (uint32_t)r * 64u < m) skey[rank[r]] = key[r];
    }
    __syncthreads();
    uint32_t out[kItems];
#pragma unroll
    for (int r = 0; r < kItems; r++) {
        const uint32_t j = (uint32_t)tid + (uint32_t)r * kSortThreads;
        if (j < m) {
            const K k = skey[j];
            out[r] = gofs[(uint32_t)(k >> shift) & 255u] + j;
            kout[out[r]] = k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; r++)
        if (wbase + (uint32_t)r * 64u < m) sval[rank[r]] = val[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; r++) {
        const uint32_t j = (uint32_t)tid + (uint32_t)r * kSortThreads;
        if (j < m) vout[out[r]] = sval[j];
    }
}

// Up to kSmallSort pairs are sorted by one block in LDS, all passes in one launch: a pass
// over two tiles is five launches' latency (108 us of a 5 K triangle build for its four).
// Wave w holds pairs [512 w, 512 w + 512), 8 per lane, and ranks them as k_radix_scatter.
constexpr uint32_t kSmallSort = 8192;
constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64, kSmallItems = kSmallSort / kSmallThreads;

template <typename K>
__global__ __launch_bounds__(kSmallThreads) void k_sort_small(const K* __restrict__ kin,
                                                              K* __restrict__ kout,
                                                              uint32_t* __restrict__ vout, uint32_t n,
                                                              int key_bits) {
    __shared__ K skey[kSmallSort];
    __shared__ uint32_t sval[kSmallSort];
    __shared__ uint32_t wcnt[kSmallWaves][256];
    __shared__ uint32_t wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t lt_mask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    const uint32_t wbase = (uint32_t)wave * 64u * kSmallItems;
    K key[kSmallItems];
    uint32_t val[kSmallItems], rank[kSmallItems];
#pragma unroll
    for (int r = 0; r < kSmallItems; r++) {
        const uint32_t i = wbase + (uint32_t)r * 64u + (uint32_t)lane;
        key[r] = i < n ? kin[i] : (K)0;
        val[r] = i;
    }
    for (int shift = 0; shift < key_bits; shift += 8) {
        for (int k = tid; k < kSmallWaves * 256; k += kSmallThreads) wcnt[k >> 8][k & 255] = 0;
        __syncthreads();
        uint32_t* const mycnt = wcnt[wave];
#pragma unroll
        for (int r = 0; r < kSmallItems; r++) {
            const bool valid = wbase + (uint32_t)r * 64u + (uint32_t)lane < n;
            const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const uint64_t bb = __ballot((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? bb : ~bb;
            }
            const uint32_t rk = (uint32_t)__popcll(peers & lt_mask);
            const uint32_t before = mycnt[d];
            rank[r] = before + rk;
            if (valid && rk == 0) mycnt[d] = before + (uint32_t)__popcll(peers);
        }
        __syncthreads();
        // first slot of every (digit, wave): scan over the digits by the first 256 threads
        uint32_t tot = 0, incl = 0;
        if (tid < 256) {
            for (int w = 0; w < kSmallWaves; w++) tot += wcnt[w][tid];
            incl = tot;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t x = __shfl_up(incl, off);
                if (lane >= off) incl += x;
            }
            if (lane == 63) wsum[wave] = incl;
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t start = incl - tot;
            for (int w = 0; w < wave; w++) start += wsum[w];
            for (int w = 0; w < kSmallWaves; w++) {
                const uint32_t c = wcnt[w][tid];
                wcnt[w][tid] = start;
                start += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSmallItems; r++) {
            if (wbase + (uint32_t)r * 64u + (uint32_t)lane < n) {
                const uint32_t pos = mycnt[(uint32_t)(key[r] >> shift) & 255u] + rank[r];
                skey[pos] = key[r];
                sval[pos] = val[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSmallItems; r++) {
            const uint32_t i = wbase + (uint32_t)r * 64u + (uint32_t)lane;
            if (i < n) {
                key[r] = skey[i];
                val[r] = sval[i];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kSmallItems; r++) {
        const uint32_t i = wbase + (uint32_t)r * 64u + (uint32_t)lane;
        if (i < n) {
            kout[i] = key[r];
            vout[i] = val[r];
        }
    }
}

size_t radix_sort_scratch_words(uint32_t n) {
    return 256 * (size_t)cdiv(n, kSortTile) + 256;
}

template <typename K>
bool radix_sort_pairs(K* k0, uint32_t* v0, K* k1, uint32_t* v1, uint32_t n, int key_bits,
                      uint32_t* scratch, hipStream_t s) {
    if (n <= kSmallSort) {
        hipLaunchKernelGGL((k_sort_small<K>), dim3(1), dim3(kSmallThreads), 0, s, k0, k1, v1, n, key_bits);
        return true;
    }
    const uint32_t nblocks = cdiv(n, kSortTile);
    uint32_t* hist = scratch;  // 256 digit counts per block, digit-major
    uint32_t* totals = scratch + 256 * (size_t)nblocks;
    K *kin = k0, *kout = k1;
    uint32_t *vin = nullptr, *vout = v1;  // the first pass's values are the indices
    bool in1 = false;
    for (int shift = 0; shift < key_bits; shift += 8) {
        hipLaunchKernelGGL((k_radix_hist<K>), dim3(nblocks), dim3(kBlock), 0, s, kin, n, shift, hist, nblocks);
        hipLaunchKernelGGL(k_scan_rows, dim3(256), dim3(kBlock), 0, s, hist, nblocks, totals);
        hipLaunchKernelGGL((k_radix_scatter<K>), dim3(nblocks), dim3(kSortThreads), 0, s, kin, vin, kout, vout, n, shift, hist,
                           totals, nblocks);
        std::swap(kin, kout);
        vin = vout;
        vout = in1 ? v1 : v0;
        in1 = !in1;
    }
    return in1;
}
template bool radix_sort_pairs<uint64_t>(uint64_t*, uint32_t*, uint64_t*, uint32_t*, uint32_t, int, uint32_t*,
                                         hipStream_t);
template bool radix_sort_pairs<uint32_t>(uint32_t*, uint32_t*, uint32_t*, uint32_t*, uint32_t, int, uint32_t*,
                                         hipStream_t);

// ------------------------------------------------------------------------------------
// k_pack: gather triangles and AABBs into sorted order
// ------------------------------------------------------------------------------------

// Triangles in sorted order: sorted primitive p is triangle t = vals[p] - tri_offset of
// mesh s = keys[p] >> 30.  Its vertices are read from the mesh itself (neighbours in
// Morton order share vertices, so these reads mostly hit the caches) rather than
// gathered from a per-triangle copy in input order (two box rows and three vertex rows
// at a random index each), and its box is rebuilt from them exactly as k_prep built it.
__global__ __launch_bounds__(kBlock) void k_pack(uint32_t N, const uint64_t* __restrict__ keys,
                                                 const uint32_t* __restrict__ vals,
                                                 const SegDesc* __restrict__ segs,
                                                 float4* __restrict__ saabb,
                                                 float4* __restrict__ tris,
                                                 uint32_t* __restrict__ leaf_order) {
    uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= N) return;
    const uint32_t g = vals[p];
    const uint32_t s = (uint32_t)(keys[p] >> 30);
    const SegDesc sd = segs[s];
    const uint32_t t = g - sd.tri_offset;
    float v[3][3];
    bool finite = true;
    for (int k = 0; k < 3; k++) {
        uint32_t vi = sd.idx[3 * (size_t)t + k];
        if (vi >= sd.n_verts) vi = 0;  // reported by k_prep (the build fails)
        const float* q = sd.verts + (size_t)vi * sd.vstride;
        v[k][0] = q[0]; v[k][1] = q[1]; v[k][2] = q[2];
        finite = finite && isfinite(v[k][0]) && isfinite(v[k][1]) && isfinite(v[k][2]);
    }
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int a = 0; a < 3; a++) {
        for (int k = 0; k < 3; k++) {
            const float x = finite ? v[k][a] : 0.0f;
            lo[a] = fminf(lo[a], x);
            hi[a] = fmaxf(hi[a], x);
        }
    }
    saabb[2 * (size_t)p] = make_float4(lo[0], lo[1], lo[2], __uint_as_float(s));
    saabb[2 * (size_t)p + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    tris[3 * (size_t)p + 0] = make_float4(v[0][0], v[0][1], v[0][2], __uint_as_float(t));
    tris[3 * (size_t)p + 1] = make_float4(v[1][0], v[1][1], v[1][2], 0.0f);
    tris[3 * (size_t)p + 2] = make_float4(v[2][0], v[2][1], v[2][2], 0.0f);
    if (leaf_order) leaf_order[p] = g;
}

// ------------------------------------------------------------------------------------
// internal node boxes and SAH costs
// ------------------------------------------------------------------------------------

// Treelet builds: the internal nodes of more than 2 leaf_size triangles, which are the
// treelet roots, bucketed by prefix length (a counting sort, order within a bucket
// arbitrary).  lvl_hist[256] counts, lvl_begin[257] prefix sums, lvl_order the nodes.  Each
// block counts a contiguous range of nodes in LDS and adds to the global counts once per
// bucket it saw: with one block per 256 nodes, the same-address device atomics alone took
// over 1 ms per pass for a 25 M-node batch.  Within a block's range a bucket keeps roughly
// node order, so the per-level passes read neighbouring nodes.
constexpr unsigned kLevelBlocks = 1024;

__device__ __forceinline__ void level_range(int n_int, uint32_t& lo, uint32_t& hi) {
    const uint32_t per = (((uint32_t)n_int + gridDim.x - 1) / gridDim.x + kBlock - 1) / kBlock * kBlock;
    lo = min((uint32_t)n_int, blockIdx.x * per);
    hi = min((uint32_t)n_int, lo + per);
}

static_assert(kLevelBuckets == kBlock, "one bucket per thread in the level kernels");
constexpr uint32_t kNoBucket = 255;  // small nodes and nodes above the mesh roots (0xFF)

__device__ __forceinline__ uint32_t level_bucket(uint8_t dlev, uint2 range, uint32_t small_max) {
    return range.y - range.x + 1u > small_max ? dlev : kNoBucket;
}

__global__ __launch_bounds__(kBlock) void k_level_hist(int n_int, const uint8_t* __restrict__ dlev,
                                                       const uint2* __restrict__ range, uint32_t small_max,
                                                       uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[kLevelBuckets];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t lo, hi;
    level_range(n_int, lo, hi);
    for (uint32_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const uint32_t l = level_bucket(dlev[i], range[i], small_max);
        if (l != kNoBucket) atomicAdd(&h[l], 1u);
    }
    __syncthreads();
    if (h[threadIdx.x]) gatomic_add(&hist[threadIdx.x], h[threadIdx.x]);
}

__global__ __launch_bounds__(kBlock) void k_level_scan(const uint32_t* __restrict__ hist, uint32_t* __restrict__ begin,
                                                       uint32_t* __restrict__ fill) {
    __shared__ uint32_t wsum[kBlock / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t v = hist[tid];
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if (lane >= (uint32_t)d) x += y;
    }
    if (lane == 63u) wsum[wave] = x;
    __syncthreads();
    for (uint32_t w = 0; w < wave; w++) x += wsum[w];
    begin[tid] = x - v;
    fill[tid] = x - v;
    if (tid == kBlock - 1) begin[kBlock] = x;
}

__global__ __launch_bounds__(kBlock) void k_level_scatter(int n_int, const uint8_t* __restrict__ dlev,
                                                          const uint2* __restrict__ range, uint32_t small_max,
                                                          uint32_t* __restrict__ fill,
                                                          uint32_t* __restrict__ order) {
    __shared__ uint32_t h[kLevelBuckets], base[kLevelBuckets];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t lo, hi;
    level_range(n_int, lo, hi);
    for (uint32_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const uint32_t l = level_bucket(dlev[i], range[i], small_max);
        if (l != kNoBucket) atomicAdd(&h[l], 1u);
    }
    __syncthreads();
    // reserve this block's part of every bucket, then place its nodes there
    base[threadIdx.x] = h[threadIdx.x] ? gatomic_add(&fill[threadIdx.x], h[threadIdx.x]) : 0u;
    h[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const uint32_t l = level_bucket(dlev[i], range[i], small_max);
        if (l != kNoBucket) order[base[l] + atomicAdd(&h[l], 1u)] = i;
    }
}

// Node boxes without atomics, fences or an order between launches.
//
// k_tree_local: block c owns internal nodes [256c, 256c + 256).  A node whose leaf range
// lies in one such chunk has its whole subtree there (a Karras node's index is an end of
// its range, so the subtree's internal nodes lie inside the range), so the block computes
// all of these bottom up by itself: rounds in which every node whose children are done
// merges their boxes, with the chunk's boxes and costs kept in LDS (its own global writes
// are not read back, so no cache can hand a lane a stale box) until no node is left.  A
// round always finishes the deepest pending node, so the loop ends.  This covers ~90% of
// the nodes.
//
// The others (ranges across chunks) are unions over their leaf range.  The leaves' boxes
// are merged in aligned blocks of 4, 16, 64, ... leaves (rbox, level after level: the
// local pass makes the blocks up to its chunk, k_range_top the rest), and k_boxes_cross
// covers a node's range with at most 6 blocks per level.  Minima and maxima are exact, so
// the boxes are the ones a bottom-up pass gives; one launch per prefix length in use (43 to
// 61 of them) gave them before: 110 us of GPU time and 40 launches' gaps in a 5 K triangle
// build, 235 us at 2.3 M, 390 us in a 7 M triangle batch.
__device__ __forceinline__ bool box_in_chunk(uint2 r) { return (r.x >> 8) == (r.y >> 8); }
static_assert(kBlock == 256, "k_tree_local chunks are 256 nodes");

__device__ __forceinline__ void write_bnode(float4* __restrict__ bnode, uint32_t i, float4 lo, float4 hi, uint2 kid,
                                            uint2 range, float cost) {
    lo.w = __uint_as_float(kid.x);
    hi.w = __uint_as_float(kid.y);
    bnode[3 * (size_t)i] = lo;
    bnode[3 * (size_t)i + 1] = hi;
    bnode[3 * (size_t)i + 2] = make_float4(__uint_as_float(range.y - range.x + 1u), cost, __uint_as_float(range.x), 0.0f);
}

// Karras' binary radix tree over the sorted 64-bit keys (Karras 2012, Algorithm 2) and the
// boxes of its in-chunk nodes, thread i of the grid making node i.  The searches compare a
// node's key with ones mostly near it, so the chunk's keys and a chunk's either side are held
// in LDS (as a launch of its own that read every key from memory: 76 us on 2.3 M triangles,
// and 88 us for the boxes; 132 us together).  binary references: internal node i -> i; leaf
// (sorted primitive p) -> kLeafBit | p
__global__ __launch_bounds__(kBlock) void k_tree_local(uint32_t N, const uint64_t* __restrict__ keys,
                                                       const SegDesc* __restrict__ segs,
                                                       const float4* __restrict__ saabb, uint2* __restrict__ kids,
                                                       uint2* __restrict__ range, uint32_t* __restrict__ seg_root,
                                                       uint8_t* __restrict__ dlev, float4* __restrict__ bnode,
                                                       float4* __restrict__ rbox, uint8_t* __restrict__ xlist,
                                                       uint32_t* __restrict__ xcount, int leaf_size) {
    __shared__ float4 slo[kBlock], shi[kBlock];  // the chunk's leaf boxes
    __shared__ float4 box[2 * kBlock];           // the keys, then the in-chunk nodes' boxes
    __shared__ float bcost[kBlock];
    __shared__ uint8_t done[kBlock];
    __shared__ uint32_t xwave[kBlock / 64];
    constexpr uint32_t kWindow = 3 * kBlock;
    static_assert(sizeof(uint64_t) * kWindow <= sizeof(box), "the keys fit");
    uint64_t* const skey = reinterpret_cast<uint64_t*>(box);
    float4 *const blo = box, *const bhi = box + kBlock;
    const uint32_t c0 = blockIdx.x * kBlock, tid = threadIdx.x;
    const uint32_t i = c0 + tid;
    const int w0 = (int)c0 - kBlock;
#pragma unroll
    for (uint32_t k = tid; k < kWindow; k += kBlock) {
        const int j = w0 + (int)k;
        skey[k] = j >= 0 && j < (int)N ? keys[j] : 0ull;
    }
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (i < N) {
        lo = saabb[2 * (size_t)i];
        hi = saabb[2 * (size_t)i + 1];
    }
    slo[tid] = lo;
    shi[tid] = hi;
    done[tid] = 0;
    __syncthreads();
    bool todo = false, cross = false;
    uint32_t L = 0, R = 0;
    uint2 rg = make_uint2(0u, 0u);
    if (i < N - 1) {
        auto key = [&](int j) { return (uint32_t)(j - w0) < kWindow ? skey[j - w0] : keys[j]; };
        const uint64_t mine = skey[tid + kBlock];
        const int n = (int)i;
        // common prefix of keys n and j (equal keys: of the indices, behind 64 bits)
        auto delta = [&](int j) {
            if (j < 0 || j >= (int)N) return -1;
            const uint64_t x = mine ^ key(j);
            return x ? __clzll(x) : 64 + __clz((uint32_t)(n ^ j));
        };
        const int dir = delta(n + 1) - delta(n - 1) >= 0 ? 1 : -1;
        const int dmin = delta(n - dir);
        int lmax = 2;
        while (delta(n + lmax * dir) > dmin) lmax *= 2;
        int l = 0;
        for (int t = lmax / 2; t >= 1; t /= 2)
            if (delta(n + (l + t) * dir) > dmin) l += t;
        const int j = n + l * dir;
        const int dnode = delta(j);
        int s = 0, t = l;
        do {
            t = (t + 1) / 2;
            if (delta(n + (s + t) * dir) > dnode) s += t;
        } while (t > 1);
        const int split = n + s * dir + min(dir, 0);
        const int first = min(n, j), last = max(n, j);
        L = first == split ? (kLeafBit | (uint32_t)split) : (uint32_t)split;
        R = last == split + 1 ? (kLeafBit | (uint32_t)(split + 1)) : (uint32_t)(split + 1);
        rg = make_uint2((uint32_t)first, (uint32_t)last);
        kids[i] = make_uint2(L, R);
        range[i] = rg;
        const uint32_t sf = (uint32_t)(key(first) >> 30), sl = (uint32_t)(key(last) >> 30);
        if (sf == sl) {
            const SegDesc sd = segs[sf];
            if ((uint32_t)first == sd.tri_offset && (uint32_t)last == sd.tri_offset + sd.n_tris - 1u) seg_root[sf] = i;
        }
        // nodes above the mesh roots (their range spans several meshes) belong to no BVH:
        // prefix length 0xFF keeps the box and treelet passes away from them
        dlev[i] = sf == sl ? (uint8_t)dnode : (uint8_t)0xFF;
        todo = sf == sl && box_in_chunk(rg);
        cross = sf == sl && !todo;
    }
    const uint64_t xmask = __ballot(cross);
    if ((tid & 63u) == 0) xwave[tid >> 6] = (uint32_t)__popcll(xmask);
    __syncthreads();  // (the keys have been read, too)
    if (rbox) {  // the chunk's other nodes, for k_boxes_cross
        uint32_t at = (uint32_t)__popcll(xmask & ((1ull << (tid & 63u)) - 1ull));
        for (uint32_t w = 0; w < tid >> 6; w++) at += xwave[w];
        if (cross) xlist[c0 + at] = (uint8_t)tid;
        if (tid == 0) xcount[blockIdx.x] = xwave[0] + xwave[1] + xwave[2] + xwave[3];
    }
    if (rbox) write_range_blocks(N, i, lo, hi, rbox, blo);
    const bool mine_to_write = todo;
    float cost = 0.f;
    while (__syncthreads_or(todo)) {
        const bool ready = todo && ((L & kLeafBit) || done[L - c0]) && ((R & kLeafBit) || done[R - c0]);
        if (ready) {
            // a leaf of an in-chunk node lies in the chunk
            const uint32_t l = (L & ~kLeafBit) - c0, r = (R & ~kLeafBit) - c0;
            const bool ll = (L & kLeafBit) != 0u, rl = (R & kLeafBit) != 0u;
            const float4 al = ll ? slo[l] : blo[l], ah = ll ? shi[l] : bhi[l];
            const float4 bl = rl ? slo[r] : blo[r], bh = rl ? shi[r] : bhi[r];
            const float cl = ll ? kCt * box_area(al, ah) : bcost[l], cr = rl ? kCt * box_area(bl, bh) : bcost[r];
            lo = min4(al, bl);
            hi = max4(ah, bh);
            cost = sah_node_cost(lo, hi, rg.y - rg.x + 1u, cl, cr, leaf_size);
        }
        __syncthreads();  // every read of this round before any write
        if (ready) {
            blo[tid] = lo;
            bhi[tid] = hi;
            bcost[tid] = cost;
            done[tid] = 1;
            todo = false;
        }
    }
    // (all at once at the end: a store per round had few lanes in it)
    if (mine_to_write) write_bnode(bnode, i, lo, hi, make_uint2(L, R), rg, cost);
}

// The aligned blocks above the chunks, five levels per launch: a block of threads reduces 1024
// boxes by shuffles and a last step through LDS.  (One block for all levels, reading each
// level back, took 20 us for 9 K chunks and 63 us for 27 K; now 5 and 10 us.)
constexpr int kRangeTop = 1024, kRangeLevels = 5;  // a block makes 5 levels of 1024 boxes

__global__ __launch_bounds__(kRangeTop) void k_range_top(uint32_t cnt, const float4* __restrict__ src,
                                                      float4* __restrict__ dst) {
    __shared__ float4 part[2][kRangeTop / 64];
    const uint32_t tid = threadIdx.x, i = blockIdx.x * kRangeTop + tid;
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (i < cnt) {
        lo = src[2 * (size_t)i];
        hi = src[2 * (size_t)i + 1];
    }
#pragma unroll
    for (int lvl = 1; lvl <= 3; lvl++) {
        if (cnt == 1) return;
        const int o = 1 << (2 * (lvl - 1));
        lo = min4(lo, shfl_xor4(lo, o));
        hi = max4(hi, shfl_xor4(hi, o));
        lo = min4(lo, shfl_xor4(lo, 2 * o));
        hi = max4(hi, shfl_xor4(hi, 2 * o));
        cnt = (cnt + 3) / 4;
        const uint32_t e = i >> (2 * lvl);
        if ((tid & (4u * o - 1u)) == 0 && e < cnt) {
            dst[2 * (size_t)e] = lo;
            dst[2 * (size_t)e + 1] = hi;
        }
        dst += 2 * (size_t)cnt;
    }
    if (cnt == 1) return;
    if ((tid & 63u) == 0) {
        part[0][tid >> 6] = lo;
        part[1][tid >> 6] = hi;
    }
    __syncthreads();
    if (tid >= 16) return;
    lo = part[0][tid];
    hi = part[1][tid];
#pragma unroll
    for (int o = 1; o <= 4; o *= 4) {  // 16 boxes to 4, then to 1
        lo = min4(lo, shfl_xor4(lo, o));
        hi = max4(hi, shfl_xor4(hi, o));
        lo = min4(lo, shfl_xor4(lo, 2 * o));
        hi = max4(hi, shfl_xor4(hi, 2 * o));
        if (cnt == 1) return;
        cnt = (cnt + 3) / 4;
        const uint32_t e = (blockIdx.x * 16 + tid) / (4 * o);
        if (tid % (4 * o) == 0 && e < cnt) {
            dst[2 * (size_t)e] = lo;
            dst[2 * (size_t)e + 1] = hi;
        }
        dst += 2 * (size_t)cnt;
    }
}

// four levels up to the chunks and those above down to one entry
size_t range_boxes(uint32_t N) {
    size_t total = 0;
    uint32_t cnt = N;
    for (int lvl = 1; lvl <= 4 || cnt > 1; lvl++) {
        cnt = (cnt + 3) / 4;
        total += cnt;
    }
    return total;
}

void launch_range_top(uint32_t N, float4* rbox, hipStream_t s) {
    uint32_t cnt = N;
    for (int lvl = 1; lvl <= 4; lvl++) {  // past the local pass's levels, to the chunks
        if (lvl > 1) rbox += 2 * (size_t)cnt;
        cnt = (cnt + 3) / 4;
    }
    while (cnt > 1) {
        float4* dst = rbox + 2 * (size_t)cnt;
        hipLaunchKernelGGL(k_range_top, dim3(cdiv(cnt, kRangeTop)), dim3(kRangeTop), 0, s, cnt, rbox, dst);
        for (int lvl = 1; lvl <= kRangeLevels && cnt > 1; lvl++) {
            rbox += 2 * (size_t)cnt;
            cnt = (cnt + 3) / 4;
        }
    }
}

// A subtree of at most 2 leaf_size triangles that crosses a chunk: its SAH cost, by a walk
// (larger nodes' costs are formed by the treelet pass, from their children's).
__device__ float small_cost(uint32_t root, const uint2* __restrict__ kids, const uint2* __restrict__ range,
                            const float4* __restrict__ saabb, int leaf_size) {
    float c = 0.0f;
    uint32_t stack[16];
    int sp = 0;
    stack[sp++] = root;
    while (sp > 0) {
        const uint32_t r = stack[--sp];
        const bool leaf = (r & kLeafBit) != 0u;
        const uint2 rg = leaf ? make_uint2(r & ~kLeafBit, r & ~kLeafBit) : range[r];
        float4 lo = saabb[2 * (size_t)rg.x], hi = saabb[2 * (size_t)rg.x + 1];
        for (uint32_t p = rg.x + 1; p <= rg.y; p++) {
            lo = min4(lo, saabb[2 * (size_t)p]);
            hi = max4(hi, saabb[2 * (size_t)p + 1]);
        }
        const uint32_t n = rg.y - rg.x + 1u;
        if (n <= (uint32_t)leaf_size) {
            c += kCt * box_area(lo, hi) * (float)n;
        } else {
            c += kCi * box_area(lo, hi);
            if (sp + 2 <= 16) {
                const uint2 k = kids[r];
                stack[sp++] = k.y;
                stack[sp++] = k.x;
            }
        }
    }
    return c;
}

// kCrossLanes lanes per chunk share its list: ~10 of a chunk's 256 nodes are here, each a
// chain of dependent loads (a thread per node of the tree, 10 of 256 with work: 48 us on
// 2.3 M triangles, 137 us on a 6.9 M triangle batch; now 29 and ~60).
constexpr uint32_t kCrossLanes = 16;

__global__ __launch_bounds__(kBlock) void k_boxes_cross(uint32_t N, const uint2* __restrict__ range,
                                                        const uint2* __restrict__ kids,
                                                        const uint8_t* __restrict__ xlist,
                                                        const uint32_t* __restrict__ xcount,
                                                        const float4* __restrict__ saabb,
                                                        const float4* __restrict__ rbox, float4* __restrict__ bnode,
                                                        int leaf_size, int costs) {
    const uint32_t chunk = (blockIdx.x * kBlock + threadIdx.x) / kCrossLanes;
    if (chunk * kBlock >= N) return;
    const uint32_t n = xcount[chunk];
    for (uint32_t k = threadIdx.x % kCrossLanes; k < n; k += kCrossLanes) {
        const uint32_t i = chunk * kBlock + xlist[chunk * kBlock + k];
        const uint2 rg = range[i];
        float4 lo, hi;
        range_union(
            rg.x, rg.y + 1u, N, rbox,
            [&](uint32_t k, float4& l, float4& h) {
                l = min4(l, saabb[2 * (size_t)k]);
                h = max4(h, saabb[2 * (size_t)k + 1]);
            },
            lo, hi);
        float c = 0.0f;
        if (costs && rg.y - rg.x + 1u <= 2u * (uint32_t)leaf_size) c = small_cost(i, kids, range, saabb, leaf_size);
        write_bnode(bnode, i, lo, hi, kids[i], rg, c);
    }
}

// ------------------------------------------------------------------------------------
// k_collapse: binary tree -> W-wide nodes, one launch per wide level
// ------------------------------------------------------------------------------------

struct CollapseArgs {
    const float4* bnode;  // binary nodes (build_common.h)
    const float4* saabb;
    const uint32_t* segstat;
    uint2* wsrc;     // wide node -> the two binary refs it starts from (root_kids)
    uint32_t* wseg;  // wide node -> mesh
    uint32_t* wfirst;  // wide node -> first packed triangle of its range
    uint32_t* lvl_cnt;
    uint32_t* counters;  // [0] wide nodes (set at the end), [1] error bits
    void* nodes;
    uint32_t capacity;
    int leaf_size;
    int level;
    // re-pack (after treelet restructuring a leaf's triangles are no longer one sorted
    // range): a node's range is dealt to its children in slot order, so every subtree's
    // triangles are contiguous again; perm[slot] = sorted position, gathered by k_repack
    int repack;
    uint32_t* perm;
};

// The sorted positions of the <= leaf_size triangles under binary ref r, to slots from `out`.
__device__ void list_leaf(const CollapseArgs& a, uint32_t r, uint32_t out) {
    uint32_t stack[8];
    int sp = 0;
    stack[sp++] = r;
    while (sp > 0) {
        const uint32_t x = stack[--sp];
        if (x & kLeafBit) {
            a.perm[out++] = x & ~kLeafBit;
        } else if (sp + 2 <= 8) {
            stack[sp++] = __float_as_uint(a.bnode[3 * (size_t)x + 1].w);
            stack[sp++] = __float_as_uint(a.bnode[3 * (size_t)x].w);
        }
    }
}

// Triangles copied to their slots after all leaves have theirs: a thread per float4, so the
// writes are contiguous (copied inside the collapse, a node's 16 triangles one after the
// other were most of its 730 us on 2.3 M triangles).
__global__ __launch_bounds__(kBlock) void k_repack(uint32_t N, const uint32_t* __restrict__ perm,
                                                   const float4* __restrict__ tris_in,
                                                   const uint32_t* __restrict__ order_in,
                                                   float4* __restrict__ tris_out,
                                                   uint32_t* __restrict__ order_out) {
    const size_t k = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= 3 * (size_t)N) return;
    const uint32_t out = (uint32_t)(k / 3), v = (uint32_t)(k - 3 * (size_t)out);
    // (a tree deeper than kMaxLevels, which is refused, leaves slots without a position)
    const uint32_t in = min(perm[out], N - 1u);
    tris_out[k] = tris_in[3 * (size_t)in + v];
    if (v == 0) order_out[out] = order_in[in];
}

constexpr int kBlockLevelThreads = 512;  // of the one-block kernels: 8-wide nodes need 217 VGPRs

// Block-wide allocation: each thread asks for n slots of a counter (any may ask for 0; all
// threads of the block take part), one atomic per block (add) returns the block's slots and
// a thread gets its part in thread order.  Device atomics on one address go one after another
// at the memory side: with one per wave on the node counter and one on the level's count, the
// atomics were most of a large level (the collapse of a 256-mesh batch, 6.9 M triangles:
// 494 us with them, 315 with one per block of 256 threads).
template <typename Add>
__device__ __forceinline__ uint32_t block_alloc(Add add, uint32_t n) {
    __shared__ uint32_t wsum[kBlockLevelThreads / 64], first;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t x = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if (lane >= (uint32_t)d) x += y;
    }
    __syncthreads();  // the last call's sums have been read
    if (lane == 63u) wsum[wave] = x;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; w++) {
        if (w < wave) before += wsum[w];
        total += wsum[w];
    }
    if (threadIdx.x == 0) first = total ? add(total) : 0u;
    __syncthreads();
    return first + before + x - n;
}

// A level that one block makes out of LDS (k_collapse_block): its nodes' sources, meshes and
// ranges, and the next level's with their count.
constexpr uint32_t kHeadNodes = 256;
struct HeadList {
    uint2 src[kHeadNodes];
    uint32_t seg[kHeadNodes], first[kHeadNodes];
};

// The binary nodes a mesh's first wide node starts from: its root's children, or the root
// alone when that is one leaf.  (Every other wide node gets its own binary node's children
// from the level above, which has loaded that node.)
__device__ __forceinline__ uint2 root_kids(const float4* __restrict__ bnode, uint32_t root, uint32_t leaf_size) {
    if (root & kLeafBit) return make_uint2(root, kEmpty);
    const float4* p = bnode + 3 * (size_t)root;
    if (__float_as_uint(p[2].x) <= leaf_size) return make_uint2(root, kEmpty);
    return make_uint2(__float_as_uint(p[0].w), __float_as_uint(p[1].w));
}

// Collapses nodes [begin, begin + cnt) of a level, dealt to the grid's threads; all threads
// of a block call it together.  The next level's nodes, counted in *next_count, follow them.
// HEAD: read from `in`, and the next level's (with its count in LDS) listed in `next` too
// while they fit.  last: no level follows; *next_count tells that one would have to (the tree
// is refused then), and the children that it would hold are left out, so that no node of the
// tree points to one that nothing makes.
template <int W, bool HEAD = false>
__device__ __forceinline__ void collapse_level(const CollapseArgs& a, uint32_t begin, uint32_t cnt,
                                               uint32_t* next_count, const HeadList* in = nullptr,
                                               HeadList* next = nullptr, bool last = false) {
    WNode<W>* nodes = reinterpret_cast<WNode<W>*>(a.nodes);
    // every lane runs every iteration (slot allocation is block-wide); lanes past the
    // level's end take part with nothing to allocate
    for (uint32_t k0 = blockIdx.x * blockDim.x; k0 < cnt; k0 += gridDim.x * blockDim.x) {
        const uint32_t k = k0 + threadIdx.x;
        const bool act = k < cnt;
        uint32_t wi = begin + (act ? k : 0u);
        const uint2 kids = HEAD ? in->src[act ? k : 0u] : a.wsrc[wi];
        uint32_t seg = HEAD ? in->seg[act ? k : 0u] : a.wseg[wi];
        uint32_t run = HEAD ? in->first[act ? k : 0u] : a.wfirst[wi];
        float pad = o2f(a.segstat[seg * kStat + 6]) * 0x1p-18f;
        // The wide node's children, kept in registers with their triangle counts and
        // boxes: a child is loaded once, with its own children when it is an internal
        // node (one 48-byte record).  Opening one (the child with the largest area among
        // those with more than leaf_size triangles, the lowest slot on ties) loads its two
        // children side by side, whatever their kind and slot, and then selects: a branch
        // per slot and kind was a memory latency each, and lanes that open different slots
        // waited for each other's (6 levels in one block 41 -> 29 us).  Slots are addressed with compile-time
        // indices only, so nothing spills to scratch.
        struct Child {
            uint32_t ref, c, first, l, r;
            float4 lo, hi;
            float area;  // < 0: not to be opened
        };
        auto load_child = [&](uint32_t r) {
            Child x;
            const bool internal = !(r & kLeafBit);
            const uint32_t at = r & ~kLeafBit;
            const float4* p = internal ? a.bnode + 3 * (size_t)at : a.saabb + 2 * (size_t)at;
            x.lo = p[0];
            x.hi = p[1];
            const float4 w = p[internal ? 2 : 1];
            x.ref = r;
            x.l = __float_as_uint(x.lo.w);
            x.r = __float_as_uint(x.hi.w);
            x.c = internal ? __float_as_uint(w.x) : 1u;
            x.first = internal ? __float_as_uint(w.z) : at;
            x.area = x.c > (uint32_t)a.leaf_size ? box_area(x.lo, x.hi) : -1.0f;
            return x;
        };
        Child ch[W];
        int n = 0;
        if (act) {
            ch[0] = load_child(kids.x);
            n = 1;
            if (kids.y != kEmpty) {
                ch[1] = load_child(kids.y);
                n = 2;
#pragma unroll
                for (int m = 2; m < W; m++) {
                    int best = -1;
                    float best_area = -1.0f;
                    uint32_t ol = 0, orr = 0;
#pragma unroll
                    for (int j = 0; j < m; j++) {
                        const bool b = ch[j].area > best_area;
                        best = b ? j : best;
                        best_area = b ? ch[j].area : best_area;
                        ol = b ? ch[j].l : ol;
                        orr = b ? ch[j].r : orr;
                    }
                    if (best < 0) break;  // (n == m until here)
                    const Child x = load_child(ol);
                    ch[m] = load_child(orr);
#pragma unroll
                    for (int j = 0; j < m; j++)
                        if (j == best) ch[j] = x;
                    n = m + 1;
                }
            }
        }
        WNode<W> out;
        auto leave_out = [&](int j) {
            out.lox[j] = out.loy[j] = out.loz[j] = INFINITY;
            out.hix[j] = out.hiy[j] = out.hiz[j] = -INFINITY;
            out.child[j] = kEmpty;
            out.aux[j] = 0;
        };
        uint32_t n_internal = 0;
#pragma unroll
        for (int j = 0; j < W; j++)
            if (j < n && ch[j].c > (uint32_t)a.leaf_size) n_internal++;
#pragma unroll
        for (int j = 0; j < W; j++) {
            if (j < n) {
                const float4 lo = ch[j].lo, hi = ch[j].hi;
                out.lox[j] = lo.x - pad; out.loy[j] = lo.y - pad; out.loz[j] = lo.z - pad;
                out.hix[j] = hi.x + pad; out.hiy[j] = hi.y + pad; out.hiz[j] = hi.z + pad;
                const uint32_t c = ch[j].c;
                out.aux[j] = c;
                if (a.repack) ch[j].first = run;
                run += c;
                if (c <= (uint32_t)a.leaf_size) {
                    if (a.repack) list_leaf(a, ch[j].ref, ch[j].first);
                    out.child[j] = make_leaf(ch[j].first, c);
                }
            } else {
                leave_out(j);
            }
        }
        const uint32_t base =
            begin + cnt + block_alloc([&](uint32_t x) { return HEAD ? atomicAdd(next_count, x) : gatomic_add(next_count, x); },
                                      n_internal);
        if (n_internal) {
            uint32_t m = 0;
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (j < n && out.aux[j] > (uint32_t)a.leaf_size) {
                    uint32_t idx = base + m++;
                    if (last) {
                        leave_out(j);
                    } else if (idx < a.capacity) {
                        const uint2 kids = make_uint2(ch[j].l, ch[j].r);
                        a.wsrc[idx] = kids;
                        a.wseg[idx] = seg;
                        a.wfirst[idx] = ch[j].first;
                        const uint32_t at = idx - (begin + cnt);
                        if (HEAD && at < kHeadNodes) {
                            next->src[at] = kids;
                            next->seg[at] = seg;
                            next->first[at] = ch[j].first;
                        }
                        out.child[j] = idx;
                    } else {
                        gatomic_or(&a.counters[1], 2u);
                        leave_out(j);
                    }
                }
            }
        }
        if (act) nodes[wi] = out;
    }
}

// One wide level per launch: each reads the nodes that the one before it allocated.
template <int W>
__global__ __launch_bounds__(kBlock) void k_collapse(CollapseArgs a) {
    // launches past the tree's depth find an empty level, and surplus blocks leave before
    // anything else
    const uint32_t cnt = a.lvl_cnt[a.level];
    if (blockIdx.x * kBlock >= cnt) return;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t begin = lane < (uint32_t)a.level ? a.lvl_cnt[lane] : 0u;
    for (int o = 32; o > 0; o >>= 1) begin += __shfl_xor(begin, o);
    collapse_level<W>(a, begin, cnt, a.lvl_cnt + a.level + 1);
}
static_assert(kMaxLevels <= 64, "k_collapse sums the levels before its own with one wave");

// The levels from a.level on, by one block: the few nodes of levels that trees of ordinary
// depth do not reach (a launch each would be 40 empty launches per batch replay).  The
// counts are read past the L1, where the atomics left them.

template <int W>
__global__ __launch_bounds__(kBlockLevelThreads) void k_collapse_tail(CollapseArgs a) {
    auto count = [&](int l) {
        return __hip_atomic_load((global_u32*)(a.lvl_cnt + l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    uint32_t begin = 0;
    for (int l = 0; l < a.level; l++) begin += count(l);
    for (int l = a.level; l < kMaxLevels; l++) {
        const uint32_t cnt = count(l);
        if (cnt == 0) break;
        collapse_level<W>(a, begin, cnt, a.lvl_cnt + l + 1, nullptr, nullptr, l == kMaxLevels - 1);
        begin += cnt;
        __threadfence_block();
        __syncthreads();
    }
    if (threadIdx.x == 0) a.counters[0] = begin;
}

// Levels [0, last), none of more than kHeadNodes nodes, by one block.  A level of a few
// nodes is latency alone: 7-12 us as a launch that reads its count and its list and takes its
// slots through device memory, 5 us with these in LDS (a 5 K triangle build's 5 first levels
// 45 -> 24 us).  With 1024 nodes (one level more) a 2.3 M triangle build is no faster than
// with launches: its nodes are cold, and one CU waits for them longer than many.
template <int W>
__global__ __launch_bounds__(kBlockLevelThreads) void k_collapse_head(CollapseArgs a, int n_seg, int last,
                                                                      const SegDesc* __restrict__ segs,
                                                                      const uint32_t* __restrict__ seg_root) {
    __shared__ HeadList list[2];
    __shared__ uint32_t count[2];
    for (uint32_t i = threadIdx.x; i < (uint32_t)n_seg; i += kBlockLevelThreads) {
        list[0].src[i] = root_kids(a.bnode, seg_root[i], (uint32_t)a.leaf_size);
        list[0].seg[i] = i;
        list[0].first[i] = segs[i].tri_offset;
        a.wseg[i] = i;
        a.wfirst[i] = segs[i].tri_offset;
    }
    uint32_t begin = 0, cnt = (uint32_t)n_seg;
    for (int l = 0; l < last && cnt; l++) {
        uint32_t* const next_count = &count[(l + 1) & 1];
        if (threadIdx.x == 0) *next_count = 0;
        __syncthreads();
        collapse_level<W, true>(a, begin, cnt, next_count, &list[l & 1], &list[(l + 1) & 1]);
        __syncthreads();
        begin += cnt;
        cnt = *next_count;
        if (threadIdx.x == 0) a.lvl_cnt[l + 1] = cnt;
    }
}

// SAH cost of a finished wide tree: sum over nodes of kCi * area for internal children
// and kCt * count * area for leaves, accumulated in double per block, then atomically (one
// atomic per block: one per wave was 88 us on 400 K nodes); with it the mesh's scale and
// the root's box go to the build's report.
template <int W>
__global__ __launch_bounds__(kBlock) void k_sah_cost(const WNode<W>* __restrict__ nodes, const float4* __restrict__ bnode,
                                                     const uint32_t* __restrict__ segstat, uint32_t* report) {
    __shared__ double part[kBlock / 64];
    const uint32_t n_nodes = report[kReportCounters];
    double c = 0.0;
    for (uint32_t k = blockIdx.x * kBlock + threadIdx.x; k < n_nodes; k += gridDim.x * kBlock) {
        const WNode<W>& nd = nodes[k];
#pragma unroll
        for (int j = 0; j < W; j++) {
            if (nd.child[j] == kEmpty) continue;
            const float a = box_area(make_float4(nd.lox[j], nd.loy[j], nd.loz[j], 0.0f),
                                     make_float4(nd.hix[j], nd.hiy[j], nd.hiz[j], 0.0f));
            c += child_is_leaf(nd.child[j]) ? (double)kCt * leaf_count(nd.child[j]) * a : (double)kCi * a;
        }
    }
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        c = 0.0;
        for (int w = 0; w < kBlock / 64; w++) c += part[w];
        if (c != 0.0) atomicAdd(reinterpret_cast<double*>(report + kReportSah), c);
    }
    if (blockIdx.x == 0 && threadIdx.x < 7) {
        const float* root = reinterpret_cast<const float*>(bnode);  // node 0: lo, left, hi, right
        report[kReportRoot + threadIdx.x] =
            threadIdx.x < 6 ? __float_as_uint(root[threadIdx.x < 3 ? threadIdx.x : threadIdx.x + 1]) : segstat[6];
    }
}

// level 0 of the wide tree: one node per mesh root
__global__ void k_init_levels(int n_seg, const SegDesc* __restrict__ segs, const uint32_t* __restrict__ seg_root,
                              CollapseArgs a) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_seg) {
        a.wsrc[i] = root_kids(a.bnode, seg_root[i], (uint32_t)a.leaf_size);
        a.wseg[i] = (uint32_t)i;
        a.wfirst[i] = segs[i].tri_offset;
    }
}

// ------------------------------------------------------------------------------------
// host orchestration
// ------------------------------------------------------------------------------------

BuildBufs::~BuildBufs() {
    for (void* p : allocs) {
        if (ctx) pool_free(ctx, p, pool_stream);
        else (void)hipFree(p);
    }
}

hipError_t BuildBufs::alloc(void** p, size_t bytes) {
    *p = nullptr;
    const hipError_t e = ctx ? (pool_alloc(ctx, p, bytes, pool_stream) ? hipErrorOutOfMemory : hipSuccess)
                             : ctx_malloc(owner, p, bytes);
    if (e == hipSuccess) allocs.push_back(*p);
    return e;
}

// All scratch of a build lives in one allocation.
static void carve_all(BuildBufs& b, Carver& c, size_t NI) {
    const uint32_t N = b.N;
    const int n_seg = b.n_seg;
    c.take(b.report, kReportWords);
    c.take(b.segs, n_seg);
    c.take(b.cen, N);
    c.take(b.segstat_rep, (size_t)kStat * n_seg * kRep);
    c.take(b.segstat, (size_t)kStat * n_seg);
    c.take(b.keys0, N);
    c.take(b.keys1, N);
    c.take(b.vals0, N);
    c.take(b.vals1, N);
    c.take(b.hist, radix_sort_scratch_words(N));  // the sort's digit counts and totals
    c.take(b.saabb, 2 * (size_t)N);
    c.take(b.rbox, 2 * range_boxes(N));
    c.take(b.kids, NI);
    c.take(b.range, NI);
    c.take(b.seg_root, n_seg);
    c.take(b.dlev, NI);
    c.take(b.xlist, N);
    c.take(b.xcount, cdiv(N, kBlock));
    c.take(b.lvl_order, b.treelets ? NI : 1);
    c.take(b.lvl_hist, kLevelBuckets);
    c.take(b.lvl_begin, kLevelBuckets + 1);
    c.take(b.lvl_fill, kLevelBuckets);
    c.take(b.bnode, 3 * NI);
    c.take(b.wsrc, b.capacity);
    c.take(b.wseg, b.capacity);
    c.take(b.wfirst, b.capacity);
    c.take(b.perm, b.treelets ? N : 1);
    char* nodes = nullptr;  // (a plain build copies the nodes in use to the BVH)
    c.take(nodes, node_bytes(b.width) * b.capacity);
    b.nodes = nodes;
    if (b.treelets) {  // the sorted triangles, re-packed into the final ones
        c.take(b.tris, 3 * (size_t)N);
        c.take(b.leaf_order, N);
    }
    b.lvl = b.report ? b.report + kReportLvl : nullptr;
    b.counters = b.report ? b.report + kReportCounters : nullptr;
}

int build_alloc(const SegDesc* host_segs, int n_seg, int W, int leaf_size, int treelet_size, BuildBufs& b) {
    uint64_t N64 = 0;
    for (int i = 0; i < n_seg; i++) {
        if (host_segs[i].n_tris == 0) return set_error(GPURT_E_INVALID, "a mesh has no triangles");
        N64 += host_segs[i].n_tris;
    }
    if (n_seg <= 0 || N64 == 0 || N64 > kMaxLeafFirst - 8)
        return set_error(GPURT_E_INVALID, "triangle count out of range (1 .. 2^28-9)");
    const uint32_t N = (uint32_t)N64;
    b.N = N;
    b.n_seg = n_seg;
    b.width = W;
    b.leaf_size = leaf_size;
    b.treelets = treelet_size > 0;
    const size_t NI = N > 1 ? N - 1 : 1;
    b.capacity = (uint32_t)(NI + n_seg);
    Carver sizing;
    carve_all(b, sizing, NI);
    void* scratch = nullptr;
    if (b.alloc(&scratch, sizing.off) != hipSuccess) {
        (void)hipGetLastError();
        return set_error(GPURT_E_OOM, "allocation of " + std::to_string(sizing.off) + " bytes of build scratch failed");
    }
    Carver c;
    c.base = static_cast<char*>(scratch);
    carve_all(b, c, NI);
    float4*& tris = b.treelets ? b.tris2 : b.tris;
    uint32_t*& order = b.treelets ? b.leaf_order2 : b.leaf_order;
    tris = b.own_tris;
    order = b.own_order;
    if (!tris || !order) {
        void *t = nullptr, *o = nullptr;
        if (b.alloc(&t, sizeof(float4) * 3 * (size_t)N) != hipSuccess ||
            b.alloc(&o, sizeof(uint32_t) * (size_t)N) != hipSuccess) {
            (void)hipGetLastError();
            return set_error(GPURT_E_OOM, "allocation of BVH storage failed");  // b frees what it holds
        }
        tris = static_cast<float4*>(t);
        order = static_cast<uint32_t*>(o);
    }
    b.one = n_seg == 1 ? host_segs[0] : SegDesc{};
    if (n_seg > 1) {  // (a single mesh is handed over by k_init_build)
        if (b.ctx) {
            GPURT_HIP(hipMemcpyAsync(b.segs, host_segs, sizeof(SegDesc) * n_seg, hipMemcpyHostToDevice, b.pool_stream));
        } else {
            GPURT_HIP(hipMemcpy(b.segs, host_segs, sizeof(SegDesc) * n_seg, hipMemcpyHostToDevice));
        }
    }
    return GPURT_OK;
}

// Enqueues the build up to (not including) the wide collapse.  No host synchronisation
// and no memset nodes, so the sequence can be captured into a HIP graph.
int build_enqueue_binary(BuildBufs& b, int treelet_size, int treelet_rounds, hipStream_t s) {
    const uint32_t N = b.N;
    const int n_seg = b.n_seg;
    const unsigned gN = cdiv(N, kBlock);
    hipLaunchKernelGGL(k_init_build, dim3(cdiv(std::max(n_seg * kRep, (int)kLevelBuckets), kBlock)), dim3(kBlock), 0, s,
                       b.segs, n_seg, b.one, n_seg == 1 ? 1 : 0, b.segstat_rep, b.seg_root, b.report, b.lvl_hist);
    // rounds of 64 triangles per wave: enough waves to fill the chip first, then fewer
    // atomics (up to 16 rounds)
    const int rounds = (int)std::min<uint32_t>(16u, std::max<uint32_t>(1u, N / (64u * 4096u)));
    hipLaunchKernelGGL(k_prep, dim3(cdiv(N, kBlock * (size_t)rounds)), dim3(kBlock), 0, s, b.segs, n_seg, N, rounds,
                       b.cen, b.segstat_rep, b.counters);
    hipLaunchKernelGGL(k_reduce_stats, dim3(cdiv((size_t)n_seg * kStat, kBlock)), dim3(kBlock), 0, s, n_seg,
                       b.segstat_rep, b.segstat);
    hipLaunchKernelGGL(k_morton, dim3(gN), dim3(kBlock), 0, s, N, b.cen, b.segstat, b.keys0);
    // radix sort over the bits in use: 30 Morton bits + mesh-id bits
    int seg_bits = 0;
    while ((1u << seg_bits) < (uint32_t)n_seg) seg_bits++;
    const int key_bits = 30 + seg_bits;
    uint64_t* kin = b.keys0;
    uint32_t* vin = b.vals0;
    if (radix_sort_pairs(b.keys0, b.vals0, b.keys1, b.vals1, N, key_bits, b.hist, s)) {
        kin = b.keys1;
        vin = b.vals1;
    }
    hipLaunchKernelGGL(k_pack, dim3(gN), dim3(kBlock), 0, s, N, kin, vin, b.segs, b.saabb, b.tris, b.leaf_order);
    if (N > 1) {
        const uint32_t n_int = N - 1;
        const unsigned gI = cdiv(n_int, kBlock);
        const bool cross = N > kBlock;  // more than one chunk
        hipLaunchKernelGGL(k_tree_local, dim3(gN), dim3(kBlock), 0, s, N, kin, b.segs, b.saabb, b.kids, b.range,
                           b.seg_root, b.dlev, b.bnode, cross ? b.rbox : nullptr, b.xlist, b.xcount, b.leaf_size);
        if (cross) {
            launch_range_top(N, b.rbox, s);
            hipLaunchKernelGGL(k_boxes_cross, dim3(cdiv((size_t)gN * kCrossLanes, kBlock)), dim3(kBlock), 0, s, N,
                               b.range, b.kids, b.xlist, b.xcount, b.saabb, b.rbox, b.bnode, b.leaf_size,
                               b.treelets ? 1 : 0);
        }
        if (treelet_size > 0) {
            // bucket the treelet roots by prefix length; distinct keys give
            // [64 - key_bits, 63], equal keys give 64 + clz32(i ^ j) with i, j < N, i.e.
            // [96 - ceil(log2 N), 95]
            int nbits = 0;
            while ((1u << nbits) < N) nbits++;
            const unsigned gL = std::min(gI, kLevelBlocks);
            const uint32_t small_max = 2u * (uint32_t)b.leaf_size;  // subtrees no treelet restructures
            hipLaunchKernelGGL(k_level_hist, dim3(gL), dim3(kBlock), 0, s, (int)n_int, b.dlev, b.range, small_max,
                               b.lvl_hist);
            hipLaunchKernelGGL(k_level_scan, dim3(1), dim3(kBlock), 0, s, b.lvl_hist, b.lvl_begin, b.lvl_fill);
            hipLaunchKernelGGL(k_level_scatter, dim3(gL), dim3(kBlock), 0, s, (int)n_int, b.dlev, b.range, small_max,
                               b.lvl_fill, b.lvl_order);
            int trc = run_treelets(b, treelet_size, treelet_rounds, key_bits, nbits, s);
            if (trc != GPURT_OK) return trc;
            b.repacked = true;
        }
    }
    GPURT_HIP(hipGetLastError());
    return GPURT_OK;
}

template <int W>
static void launch_collapse(CollapseArgs a, int n_seg, const SegDesc* segs, const uint32_t* seg_root, int levels,
                            unsigned grid, hipStream_t s) {
    int head = 0;  // levels of at most kHeadNodes nodes
    for (size_t n = (size_t)n_seg; n <= kHeadNodes && head < levels; n *= W) head++;
    if (head)
        hipLaunchKernelGGL(k_collapse_head<W>, dim3(1), dim3(kBlockLevelThreads), 0, s, a, n_seg, head, segs, seg_root);
    else
        hipLaunchKernelGGL(k_init_levels, dim3(cdiv(n_seg, kBlock)), dim3(kBlock), 0, s, n_seg, segs, seg_root, a);
    for (int level = head; level < levels; level++) {
        a.level = level;
        hipLaunchKernelGGL(k_collapse<W>, dim3(grid), dim3(kBlock), 0, s, a);
    }
    a.level = levels;
    hipLaunchKernelGGL(k_collapse_tail<W>, dim3(1), dim3(kBlockLevelThreads), 0, s, a);
}

int build_enqueue_collapse(BuildBufs& b, int leaf_size, hipStream_t s) {
    CollapseArgs ca{};
    ca.bnode = b.bnode;
    ca.saabb = b.saabb;
    ca.segstat = b.segstat;
    ca.wsrc = b.wsrc;
    ca.wseg = b.wseg;
    ca.wfirst = b.wfirst;
    ca.lvl_cnt = b.lvl;
    ca.counters = b.counters;
    ca.nodes = b.nodes;
    ca.capacity = b.capacity;
    ca.leaf_size = leaf_size;
    ca.repack = b.repacked ? 1 : 0;
    ca.perm = b.perm;
    const int levels = std::min(kMaxLevels - 1, collapse_launches(b.N, b.width, b.treelets));
    const unsigned grid = std::min(cdiv(b.capacity, kBlock), 2048u);
    if (b.width == 2) launch_collapse<2>(ca, b.n_seg, b.segs, b.seg_root, levels, grid, s);
    else if (b.width == 4) launch_collapse<4>(ca, b.n_seg, b.segs, b.seg_root, levels, grid, s);
    else launch_collapse<8>(ca, b.n_seg, b.segs, b.seg_root, levels, grid, s);
    if (b.repacked)
        hipLaunchKernelGGL(k_repack, dim3(cdiv(3 * (size_t)b.N, kBlock)), dim3(kBlock), 0, s, b.N, b.perm, b.tris,
                           b.leaf_order, b.tris2, b.leaf_order2);
    GPURT_HIP(hipGetLastError());
    return GPURT_OK;
}

// Plain (single-mesh) build: everything is enqueued, then one read of the report gives the
// node count, the levels and the errors, and the products are handed to *out.
int build_segments(gpurt_ctx ctx, const SegDesc* host_segs, int n_seg, int W, int leaf_size,
                   int treelet_size, int treelet_rounds, int format, hipStream_t s, gpurt_bvh_s* out) {
    BuildBufs b;  // its scratch goes back to the pool, in stream order, with it
    b.ctx = ctx;
    b.pool_stream = s;
    b.own_tris = out->tris;
    b.own_order = out->leaf_order;
    int rc;
    if ((rc = build_alloc(host_segs, n_seg, W, leaf_size, treelet_size, b))) return rc;
    if ((rc = build_enqueue_binary(b, treelet_size, treelet_rounds, s))) return rc;
    if ((rc = build_enqueue_collapse(b, leaf_size, s))) return rc;
    const unsigned gsah = std::min(cdiv(b.capacity, kBlock), 512u);
    if (W == 2) hipLaunchKernelGGL(k_sah_cost<2>, dim3(gsah), dim3(kBlock), 0, s, (const WNode<2>*)b.nodes, b.bnode, b.segstat, b.report);
    else if (W == 4) hipLaunchKernelGGL(k_sah_cost<4>, dim3(gsah), dim3(kBlock), 0, s, (const WNode<4>*)b.nodes, b.bnode, b.segstat, b.report);
    else hipLaunchKernelGGL(k_sah_cost<8>, dim3(gsah), dim3(kBlock), 0, s, (const WNode<8>*)b.nodes, b.bnode, b.segstat, b.report);
    GPURT_HIP(hipGetLastError());
    uint32_t rep[kReportWords];
    GPURT_HIP(hipMemcpyAsync(rep, b.report, sizeof(rep), hipMemcpyDeviceToHost, s));
    GPURT_HIP(hipStreamSynchronize(s));
    const uint32_t* h_lvl = rep + kReportLvl;
    const uint32_t* h_counters = rep + kReportCounters;
    if (h_lvl[kMaxLevels]) return set_error(GPURT_E_UNSUPPORTED, "BVH deeper than the supported level count");
    if (h_counters[1] & 1u) return set_error(GPURT_E_INVALID, "triangle index >= n_verts");
    if (h_counters[1] & 4u) return set_error(GPURT_E_INVALID, "non-finite vertex position");
    if (h_counters[1] & 2u) return set_error(GPURT_E_DEVICE, "wide-node capacity exceeded");
    int depth = 0;
    while (depth <= kMaxLevels && h_lvl[depth] > 0) depth++;
    // the nodes in use go to the BVH's own memory
    const uint32_t n_nodes = h_counters[0];
    auto carve = [&](Carver c) {
        char *nodes = nullptr, *q = nullptr;
        c.take(nodes, node_bytes(W) * n_nodes);
        out->nodes = nodes;
        if (has_qnodes(format)) c.take(q, qnode_bytes(W) * n_nodes);
        out->qnodes = q;
        if (cpq_use_oriented(format, W)) {
            ONode* o = nullptr;
            c.take(o, n_nodes);
            out->onodes = o;
        }
        c.take(out->node_first, n_nodes);
        return c.off;
    };
    if ((rc = pool_alloc(ctx, &out->node_mem, carve(Carver{}), s))) return rc;  // the caller frees the products
    carve(Carver{0, static_cast<char*>(out->node_mem)});
    GPURT_HIP(hipMemcpyAsync(out->nodes, b.nodes, node_bytes(W) * n_nodes, hipMemcpyDeviceToDevice, s));
    uint32_t u = rep[kReportRoot + 6];
    u = (u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u;
    float scale;
    std::memcpy(&scale, &u, 4);
    // SAH cost relative to the root box area
    double sah = 0.0;
    {
        float r[6];
        std::memcpy(&sah, rep + kReportSah, sizeof(sah));
        std::memcpy(r, rep + kReportRoot, sizeof(r));
        const float ex = r[3] - r[0], ey = r[4] - r[1], ez = r[5] - r[2];
        const double root_area = 2.0 * ((double)ex * ez + (double)ex * ey + (double)ey * ez);
        sah = (b.N > 1 && root_area > 0.0) ? sah / root_area : 0.0;
    }
    out->format = format;
    if (has_qnodes(format)) {
        launch_quantize(W, out->nodes, out->qnodes, n_nodes, n_nodes, nullptr, s);
        GPURT_HIP(hipGetLastError());
    }
    if (!b.repacked && b.treelets) {  // (a single triangle) the sorted ones are final
        GPURT_HIP(hipMemcpyAsync(out->tris, b.tris, sizeof(float4) * 3 * (size_t)b.N, hipMemcpyDeviceToDevice, s));
        GPURT_HIP(hipMemcpyAsync(out->leaf_order, b.leaf_order, sizeof(uint32_t) * (size_t)b.N, hipMemcpyDeviceToDevice, s));
    }
    GPURT_HIP(hipMemcpyAsync(out->node_first, b.wfirst, sizeof(uint32_t) * n_nodes, hipMemcpyDeviceToDevice, s));
    if (cpq_use_oriented(format, W)) {
        launch_orient(out->nodes, out->node_first, out->tris, out->onodes, n_nodes, n_nodes, nullptr, b.segstat + 6, 0,
                      nullptr, nullptr, s);
        GPURT_HIP(hipGetLastError());
    }
    out->n_nodes = n_nodes;
    out->node_capacity = n_nodes;
    out->depth = depth;
    out->width = W;
    out->leaf_size = leaf_size;
    out->n_tris = b.N;
    out->scale = scale;
    out->pad = scale * 0x1p-18f;
    out->sah_cost = (float)sah;
    return GPURT_OK;
}

}  // namespace gpurt_impl
