// gpurt_internal.h -- shared types of the gfx950 BVH builder and traversal kernels.
//
// Device layout (all 128-byte aligned allocations from hipMalloc):
//   wide nodes   WNode<W>: per child slot j: box lo/hi as six W-float arrays (SoA inside
//                the node, so one node is 6*W floats of boxes + W child words + W aux
//                words = 32*W bytes: 64 B for W=2, 128 B (one L2 line) for W=4, 256 B
//                for W=8).  Boxes are inflated by `pad` so culls stay conservative.
//   quantized    QNode<W>: the same tree with 8-bit child boxes relative to the node's
//   nodes        own box (origin + per-axis power-of-two scale), 16 + 4*W + 6*W bytes
//                rounded up to 16: 48 B for W=2, 64 B for W=4, 96 B for W=8.  Each
//                decoded box contains the FP32 box it was made from (checked in FP32
//                with the decoder's own arithmetic), so culls stay conservative.
//   triangles    3 float4 per triangle in leaf order: (a.xyz, id), (b.xyz, 0),
//                (c.xyz, 0) with id = the triangle's index in its mesh (float bits).
//   child word   internal child: wide-node index (< 2^31);
//                leaf: bit31 | (count-1) << 28 | first packed triangle (count 1..8);
//                empty slot: 0xFFFFFFFF.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <utility>
#include <vector>

#include "../../include/gpurt.h"
#include "index_math.h"

namespace gpurt_impl {

constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kMaxLeafFirst = 0x0FFFFFFFu;  // 2^28 - 1 packed triangles max
// Wide-node levels the collapse can emit.  A mesh's binary radix tree is at most 58
// levels deep (30 Morton bits + 28 index tie-break bits) and every wide level consumes
// at least one binary level; treelets can make it deeper, and a tree of more wide levels than
// these is refused.
constexpr int kMaxLevels = 64;
constexpr int kBlock = 256;
// buckets of the treelet pass, one per prefix length
constexpr uint32_t kLevelBuckets = 256;
// words of a build's report: wide nodes per level, counters ([0] wide nodes, [1] error
// bits), SAH sum (double), root box and coordinate scale
constexpr int kReportLvl = 0, kReportCounters = 72, kReportSah = 80, kReportRoot = 82, kReportWords = 96;

__host__ __device__ inline uint32_t make_leaf(uint32_t first, uint32_t count) {
    return kLeafBit | ((count - 1u) << 28) | first;
}
__host__ __device__ inline bool child_is_leaf(uint32_t c) { return (c & kLeafBit) != 0u; }
__host__ __device__ inline uint32_t leaf_first(uint32_t c) { return c & kMaxLeafFirst; }
__host__ __device__ inline uint32_t leaf_count(uint32_t c) { return ((c >> 28) & 7u) + 1u; }

template <int W>
struct alignas(32 * W) WNode {
    static constexpr int kWidth = W;
    float lox[W], loy[W], loz[W];
    float hix[W], hiy[W], hiz[W];
    uint32_t child[W];
    uint32_t aux[W];  // triangles under the child (for cost estimates)
};
static_assert(sizeof(WNode<2>) == 64, "node size");
static_assert(sizeof(WNode<4>) == 128, "node size");
static_assert(sizeof(WNode<8>) == 256, "node size");

inline size_t node_bytes(int W) { return (size_t)32 * (size_t)W; }

// Quantized wide node, as 32-bit words.  Child j's box on axis a decodes as
//   lo = fmaf((float)qlo[a][j], s_a, origin_a),  hi = fmaf((float)qhi[a][j], s_a, origin_a)
// with s_a a power of two.  2- and 4-wide nodes store the three scales as floats (words
// 3..5: the traversal multiplies them in directly); 8-wide nodes, whose 96 bytes have no
// room for them, store the biased exponents e_a (s_a = 2^(e_a - 127), byte a of word 3).
//   words 0..2         origin x, y, z (float)
//   word 3 (.. 5)      scales (float) or exponent bytes
//   kChild0 ..         child[W]
//   kQ0 ..             q[6][W] bytes: qlo x, y, z, then qhi x, y, z; zero padding
// An empty child slot has qlo = 255 and qhi = 0 on every axis (an inverted box).
template <int W>
struct alignas(16) QNode {
    static constexpr int kWidth = W;
    static constexpr bool kFloatScale = W <= 4;
    static constexpr int kChild0 = kFloatScale ? 6 : 4;
    static constexpr int kQ0 = kChild0 + W;
    static constexpr int kWords = (kQ0 + (6 * W + 3) / 4 + 3) / 4 * 4;
    uint32_t w[kWords];
};
static_assert(sizeof(QNode<2>) == 48, "node size");
static_assert(sizeof(QNode<4>) == 64, "node size");
static_assert(sizeof(QNode<8>) == 96, "node size");

inline size_t qnode_bytes(int W) { return W == 2 ? 48 : (W == 4 ? 64 : 96); }

// Oriented 4-wide node of closest-point queries (oriented.hip), as 32-bit words.  The
// frame R (oriented.h) follows from n.x and n.y; a point p lies at Y = R (p - c) / s + 128
// per axis, in the units of the byte planes, with s_a = 2^(e_a - 127) and e_a byte a of
// word 3.
//   words 0..2    c (float)
//   word 3        exponent bytes
//   words 4, 5    n.x, n.y (float; 0, 0: axis-aligned boxes)
//   words 6..9    child[4]
//   words 10..15  q[6][4] bytes: qlo x, y, z, then qhi x, y, z (255 and 0 in an empty slot)
struct alignas(64) ONode {
    static constexpr int kWidth = 4;
    uint32_t w[16];
};
static_assert(sizeof(ONode) == 64, "node size");

// Node formats of gpurt_build_opts::node_format (0 selects the library default, mixed).
constexpr int kFormatF32 = 1;    // FP32 boxes for every query
constexpr int kFormatQ8 = 2;     // 8-bit boxes for every query
constexpr int kFormatMixed = 3;  // 8-bit boxes for rays; for closest points oriented 8-bit
                                 // boxes (4-wide nodes) or FP32 boxes (2- and 8-wide nodes)
inline bool has_qnodes(int f) { return f != kFormatF32; }
inline bool rays_use_q8(int f) { return f == kFormatQ8 || f == kFormatMixed; }
inline bool cpq_use_q8(int f) { return f == kFormatQ8; }
inline bool cpq_use_oriented(int f, int width) { return f == kFormatMixed && width == 4; }
// node encodings that a traversal kernel is compiled for (NodeOf)
constexpr int kEncF32 = 0, kEncQ8 = 1, kEncOriented = 2;

// position of the n-th (from 0) set bit of m; n < popcount(m)
__device__ __forceinline__ uint32_t nth_set_bit(uint64_t m, uint32_t n) {
    uint32_t pos = 0;
#pragma unroll
    for (uint32_t w = 32; w >= 1; w >>= 1) {
        const uint32_t c = (uint32_t)__popcll((m >> pos) & ((1ull << w) - 1ull));
        if (n >= c) {
            n -= c;
            pos += w;
        }
    }
    return pos;
}

// Atomics on global memory through a global-address-space pointer: no flat-address
// (LDS / scratch aperture) checks are generated around them.
typedef __attribute__((address_space(1))) uint32_t global_u32;
__device__ __forceinline__ uint32_t gatomic_add(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_add((global_u32*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t gatomic_or(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_or((global_u32*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t gatomic_max_u32(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_max((global_u32*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One mesh of a (possibly single-mesh) build.
struct SegDesc {
    const float* verts;
    uint64_t vstride;  // in floats
    uint32_t n_verts;
    uint32_t n_tris;
    const uint32_t* idx;
    uint32_t tri_offset;  // first triangle of this mesh in the concatenated order
    uint32_t pad_;
};

// Build products that the traversal kernels read.
struct DeviceBvh {
    const void* nodes;   // WNode<W>[]
    const float4* tris;  // 3 per triangle
    uint32_t root;       // wide-node index of the root
    uint32_t n_tris;
};

// An event, destroyed with its last holder: points of streams that a BVH's memory waits for
// outlive the BVH.
struct Event {
    hipEvent_t e = nullptr;
    Event() = default;
    Event(const Event&) = delete;
    Event& operator=(const Event&) = delete;
    ~Event() {
        if (e) (void)hipEventDestroy(e);
    }
};
using EventRef = std::shared_ptr<Event>;
EventRef make_event();  // without timing; null when HIP cannot create one
// points of streams, each the last use of something there
using Uses = std::vector<std::pair<hipStream_t, EventRef>>;

}  // namespace gpurt_impl

struct gpurt_ctx_s {
    int device = 0;
    int n_cu = 256;
    int lds_per_cu = 160 * 1024;
    uint32_t* err = nullptr;  // sticky device error bits (bit 0: traversal stack overflow)
    // GPURT_SUMS_* mode of the backward passes' vertex-gradient sums
    int vertex_sums = 0;
    // stream on which memory that leaves the pool is freed, and which stands for the uses of a
    // destroyed TLAS (stream-ordered, no host wait)
    hipStream_t release = nullptr;
    hipMemPool_t mem = nullptr;  // HIP's pool under the context's (its freed memory goes back at
                                 // the next synchronisation)
    // BVHs and TLASes still open on the context: gpurt_ctx_destroy releases their device
    // memory, and destroying such a handle afterwards frees only its host part
    std::mutex live_mu;
    std::set<gpurt_bvh_s*> bvhs;
    std::set<gpurt_tlas_s*> tlases;
    // device scratch of the query and backward calls, one buffer per stream (ctx_scratch)
    struct StreamBuf {
        hipStream_t s = nullptr;
        void* mem = nullptr;
        size_t bytes = 0;
        hipEvent_t last = nullptr;  // recorded after the buffer's last use
        bool busy = false;          // a call is between ctx_scratch and ctx_scratch_done
    };
    std::mutex scratch_mu;
    std::vector<StreamBuf> scratch;
    // device memory of builds and BVHs (pool_alloc)
    struct PoolBlock {
        void* mem = nullptr;
        size_t bytes = 0;
        bool used = false;
        gpurt_impl::EventRef own;  // recorded where a stream gives the block back
        gpurt_impl::Uses after;    // the work an idle block waits for
        uint64_t when = 0;         // order of giving back
    };
    std::mutex pool_mu;
    std::vector<PoolBlock> pool;
    size_t pool_idle = 0, pool_limit = size_t(1) << 30;
    uint64_t pool_clock = 0;
};

namespace gpurt_impl {
// recorded: the call goes into a HIP graph and takes its scratch there
inline bool fixed_order_sums(const gpurt_ctx_s* c, size_t terms, bool recorded = false) {
    return fixed_order_rule(c->vertex_sums, terms, recorded);
}
}  // namespace gpurt_impl

struct gpurt_bvh_s {
    gpurt_ctx ctx = nullptr;
    int width = 4;
    int leaf_size = 4;
    int depth = 0;
    int64_t n_tris = 0;
    int64_t n_verts = 0;
    int64_t n_nodes = 0;
    int64_t node_capacity = 0;
    float scale = 0.f;
    float pad = 0.f;
    float sah_cost = 0.f;
    // two blocks of the context's pool hold all of these: the mesh copy, triangles and leaf
    // order, and the nodes
    void *mesh_mem = nullptr, *node_mem = nullptr;
    void* nodes = nullptr;        // WNode<W>[node_capacity] (boxes in FP32; refit updates these)
    void* qnodes = nullptr;       // QNode<W>[n_nodes] when has_qnodes(format)
    void* onodes = nullptr;       // ONode[n_nodes] when cpq_use_oriented(format, width)
    uint32_t* node_first = nullptr;  // first packed triangle of each node's (contiguous) range
    int format = 1;
    float4* tris = nullptr;       // 3 * n_tris
    uint32_t* tri_idx = nullptr;  // 3 * n_tris, original order (for backward / refit)
    float* verts = nullptr;       // 3 * n_verts compact positions, original order
    uint32_t* leaf_order = nullptr;  // packed position -> original triangle (refit)
    uint32_t* refit_tmp = nullptr;   // two words of a refit
    // gpurt_bvh_destroy gives the blocks back after the last use recorded on each stream that
    // used the handle.
    std::mutex use_mu;
    gpurt_impl::Uses uses;
    bool uses_lost = false;  // an event could not be recorded: destroy waits for the device
};

namespace gpurt_impl {

// error plumbing (abi.hip)
int set_error(int code, const std::string& msg);
int hip_error(hipError_t e, const char* what);

// use tracking of a BVH handle (abi.hip): note_use records, after work that reads `b`
// was enqueued on `s`, an event there (one event per stream, re-recorded); wait_uses
// makes stream `s` wait for every recorded use
void note_use(gpurt_bvh_s* b, hipStream_t s);
void wait_uses(gpurt_bvh_s* b, hipStream_t s);
// the recorded uses; waits for the device first when there may be others
Uses uses_of(gpurt_bvh_s* b);

// Device memory of builds and BVHs, kept by the context: a block given back after some points
// of streams is handed out again once they are reached (or, in order, to the one stream that
// they are on), so any stream and thread may take it and none waits for another's work.  Idle blocks are bounded (1/16 of the device's memory; the
// longest idle go first) and all are freed with the context.  Taking each buffer of a build as one (hipMallocAsync and
// hipFreeAsync) cost a small build about 100 us for its ten buffers, and after a hundred
// builds of 2.3 M triangles each hipFreeAsync took 10 ms (a build 27 ms instead of 8); and
// memory freed there in order behind a query was handed out before that query had run.
int pool_alloc(gpurt_ctx_s* c, void** p, size_t bytes, hipStream_t s);
void pool_free(gpurt_ctx_s* c, void* p, hipStream_t s);        // after what s holds now
void pool_free(gpurt_ctx_s* c, void* p, const Uses& after);
// hipMalloc; when memory is short the pool's idle blocks are freed and it is tried again
hipError_t ctx_malloc(gpurt_ctx_s* c, void** p, size_t bytes);
void pool_release(gpurt_ctx_s* c);  // after the device is idle (context destroy)

// Lays buffers out in one allocation, 256-byte aligned: a first pass without a base gives
// the size.
struct Carver {
    size_t off = 0;
    char* base = nullptr;
    template <typename T>
    void take(T*& p, size_t count) {
        const size_t bytes = count * sizeof(T) < 256 ? 256 : count * sizeof(T);
        off = (off + 255) & ~size_t(255);
        p = base ? reinterpret_cast<T*>(base + off) : nullptr;
        off += bytes;
    }
};

#define GPURT_HIP(call)                                            \
    do {                                                           \
        hipError_t e_ = (call);                                    \
        if (e_ != hipSuccess) return ::gpurt_impl::hip_error(e_, #call); \
    } while (0)

// validated build options (abi.hip); zero fields of the C struct select defaults
struct BuildParams {
    int width = 4, leaf_size = 4, treelet_size = 0, treelet_rounds = 0, format = 0;
};
int parse_build_opts(const gpurt_build_opts* o, BuildParams& p);

// builder (build.hip): device buffers of one build over one or more meshes
struct BuildBufs {
    uint32_t N = 0;  // triangles over all meshes
    int n_seg = 0;   // meshes
    int width = 4;
    int leaf_size = 4;
    bool repacked = false;  // treelets changed the tree: leaves re-packed into tris2
    uint32_t capacity = 0;  // wide nodes the node array can hold
    SegDesc* segs = nullptr;
    SegDesc one{};       // the mesh of a plain build
    bool treelets = false;
    float4* cen = nullptr;  // triangle box centres; w: mesh (bits)
    uint32_t* segstat_rep = nullptr;  // per-mesh statistics, replicated for atomics
    uint32_t* segstat = nullptr;      // per-mesh statistics, reduced
    uint64_t *keys0 = nullptr, *keys1 = nullptr;
    uint32_t *vals0 = nullptr, *vals1 = nullptr, *hist = nullptr;
    float4* saabb = nullptr;  // sorted triangle boxes (lo, hi)
    float4* rbox = nullptr;   // boxes of aligned blocks of 4, 16, ... sorted triangles
    uint2 *kids = nullptr, *range = nullptr;  // binary tree: children, leaf range
    uint8_t* xlist = nullptr;    // per chunk of 256 nodes, the ones whose range crosses chunks
    uint32_t* xcount = nullptr;  // and their number
    uint32_t* seg_root = nullptr;
    uint8_t* dlev = nullptr;  // common-prefix length (Karras delta) of each internal node
    // treelet roots bucketed by prefix length
    uint32_t* lvl_order = nullptr;
    uint32_t* lvl_hist = nullptr;   // kLevelBuckets counts
    uint32_t* lvl_begin = nullptr;  // bucket k = lvl_order[lvl_begin[k] .. lvl_begin[k+1])
    uint32_t* lvl_fill = nullptr;
    float4* bnode = nullptr;  // binary node records, 3 float4 each (build_common.h)
    uint2* wsrc = nullptr;       // wide node -> the binary refs it starts from
    uint32_t* wseg = nullptr;
    uint32_t* wfirst = nullptr;  // wide node -> first packed triangle of its (contiguous) range
    uint32_t* perm = nullptr;    // re-packed slot -> sorted position (treelet builds)
    // What the host reads of a build, in one piece (kReportWords); lvl and counters point
    // into it
    uint32_t* report = nullptr;
    uint32_t *lvl = nullptr, *counters = nullptr;
    void* nodes = nullptr;
    float4* tris = nullptr;          // triangles in sorted (Morton) order
    uint32_t* leaf_order = nullptr;  // sorted position -> triangle
    float4* tris2 = nullptr;         // re-packed leaves (treelet builds only)
    uint32_t* leaf_order2 = nullptr;
    float4* final_tris() const { return repacked ? tris2 : tris; }
    uint32_t* final_order() const { return repacked ? leaf_order2 : leaf_order; }
    // Plain builds: scratch from the context's pool, and the BVH's own buffers for the
    // triangles and their order.  Without a context everything is hipMalloc'ed (for `owner`)
    // and kept (the batch).
    gpurt_ctx_s *ctx = nullptr, *owner = nullptr;
    hipStream_t pool_stream = nullptr;
    float4* own_tris = nullptr;
    uint32_t* own_order = nullptr;
    std::vector<void*> allocs;  // freed with the object
    hipError_t alloc(void** p, size_t bytes);
    BuildBufs() = default;
    BuildBufs(const BuildBufs&) = delete;
    BuildBufs& operator=(const BuildBufs&) = delete;
    ~BuildBufs();
};
int build_alloc(const SegDesc* host_segs, int n_seg, int width, int leaf_size, int treelet_size,
                BuildBufs& b);
int build_enqueue_binary(BuildBufs& b, int treelet_size, int treelet_rounds, hipStream_t s);
int build_enqueue_collapse(BuildBufs& b, int leaf_size, hipStream_t s);
int run_treelets(BuildBufs& b, int treelet_size, int rounds, int key_bits, int nbits, hipStream_t s);
// Stable LSD radix sort (build.hip) of n uint64 or uint32 keys k0, each with its index as
// value, on the low key_bits bits, 8 bits per pass, ping-ponging between (k0, v0) and
// (k1, v1) (v0 need not be set); returns true when the sorted pairs end in (k1, v1).  scratch: radix_sort_scratch_words(n)
// words.
template <typename K>
bool radix_sort_pairs(K* k0, uint32_t* v0, K* k1, uint32_t* v1, uint32_t n, int key_bits, uint32_t* scratch,
                      hipStream_t s);
size_t radix_sort_scratch_words(uint32_t n);
int build_segments(gpurt_ctx ctx, const SegDesc* host_segs, int n_seg, int width, int leaf_size,
                   int treelet_size, int treelet_rounds, int format, hipStream_t stream, gpurt_bvh_s* out);

// boxes of aligned blocks of primitives (build_common.h): how many for N, and the levels
// above 256 from the ones below
size_t range_boxes(uint32_t N);
void launch_range_top(uint32_t N, float4* rbox, hipStream_t s);

// quantized node copies (quantize.hip): nodes [0, n) with n = *n_dev when n_dev is given
// (then `capacity` threads are launched), else n_host
void launch_quantize(int width, const void* nodes, void* qnodes, uint32_t n_host, uint32_t capacity,
                     const uint32_t* n_dev, hipStream_t s);

// oriented copies of 4-wide nodes (oriented.hip): nodes [0, n) with n = *n_dev when n_dev is
// given (at most capacity), else n_host.  first: each node's first packed triangle (its
// triangles are contiguous); scale: each mesh's largest coordinate as an ordered uint,
// scale_stride words apart, of mesh seg[node] (0 without seg); skip (or null): a device
// word that, when set, leaves everything as it is
void launch_orient(const void* nodes, const uint32_t* first, const float4* tris, void* onodes, uint32_t n_host,
                   uint32_t capacity, const uint32_t* n_dev, const uint32_t* scale, uint32_t scale_stride,
                   const uint32_t* seg, const uint32_t* skip, hipStream_t s);

// traversal launch planning (query.hip): stack depth, block size, grid, spill slots and
// leaf trigger for one launch of a query kind, and the per-call scratch (queue counters
// cleared on the stream + stack spill buffer)
enum class QKind { Cpq, Closest, Any };
struct TravPlan {
    int S = 8, BS = 256;
    unsigned grid = 1;
    uint32_t total = 256, spill_slots = 0, leaf_trigger = 32;
    size_t n = 0;     // queries of the launch
    size_t wide = 0;  // lanes up to which each query gets a wave (spread_lanes)
};
// work queues of a launch: counters at the start of the traversal scratch, kQueueStride
// words apart (traverse.h)
constexpr uint32_t kQueues = 256;
constexpr uint32_t kQueueStride = 64;
// lanes that a set of n queries is spread over: a wave per query up to `wide` lanes, 4
// lanes per query beyond (plan_traversal)
__host__ __device__ inline size_t spread_lanes(size_t n, size_t wide) {
    const size_t w = n * 64 < wide ? n * 64 : wide;
    return n * 4 > w ? n * 4 : w;
}
// Device scratch of one query or backward call.  Outside graph capture it is the
// context's buffer for the call's stream: grown when a call needs more (hipMalloc, after
// a device wait to free the old one), reused by the next call on that stream without an
// allocation, and released with the context; the stream first waits for the buffer's last recorded use,
// so a stream handle that the runtime recycles for another stream cannot overlap it.
// While the stream is being captured into a graph, or while another call on the same
// stream holds the buffer (two host threads), the call gets an allocation of its own,
// freed in stream order when it is done.  (A stream-ordered allocation per call made
// the host wait for the device on every large call: ~230 us for 1 M rays.)
struct CallScratch {
    void* mem = nullptr;
    hipStream_t s = nullptr;
    int slot = -1;  // the context's buffer index, or -1 for a call-owned allocation
};
int ctx_scratch(gpurt_ctx_s* c, hipStream_t s, size_t bytes, CallScratch& out);
void ctx_scratch_done(gpurt_ctx_s* c, CallScratch& cs);
void ctx_scratch_release(gpurt_ctx_s* c);  // after the device is idle (context destroy)

struct TravScratch {
    void* mem = nullptr;
    uint32_t* counters = nullptr;
    uint2* spill = nullptr;
    CallScratch cs;
};
// LDS per lane beyond the stack slots of the single-level kernels: the 64-bit result key
// and the member count of work donation (traverse.h)
constexpr int kGroupKeyBytes = 12;
// waves_per_simd: what the kernel is compiled for (0: the single-level kernels' WavesHint);
// lds_extra: LDS bytes per lane beyond the stack slots
int plan_traversal(gpurt_ctx ctx, int width, bool q8, QKind kind, int stack_need, const gpurt_query_opts* opts,
                   size_t n, TravPlan& p, int waves_per_simd = 0, int lds_extra = kGroupKeyBytes, bool oriented = false);
int alloc_traversal_scratch(gpurt_ctx_s* c, const TravPlan& p, hipStream_t s, TravScratch& t);
void free_traversal_scratch(gpurt_ctx_s* c, TravScratch& t);
// the same scratch in memory the caller holds
size_t traversal_scratch_bytes(const TravPlan& p);
void carve_traversal_scratch(const TravPlan& p, void* mem, TravScratch& t);
void clear_traversal_counters(const TravPlan& p, const TravScratch& t, hipStream_t s);

// traversal launchers (query.hip)
int launch_cpq(gpurt_bvh_s* b, const float* q, size_t n, int32_t* prim, float* pt, float* dist,
               float* bary, const gpurt_query_opts* opts, hipStream_t s);
int launch_ray(gpurt_bvh_s* b, const gpurt_ray* rays, size_t n, int32_t* prim, float* t,
               float* uv, uint8_t* occ, bool any, const gpurt_query_opts* opts, hipStream_t s);

// gpurt_trace_closest_noalloc (query.hip): the closest-hit launch with its traversal
// scratch in a fixed per-device array of kNoAllocScratchBytes, set up once per device by
// noalloc_scratch_init (with that device current; called by gpurt_ctx_create)
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
constexpr int kMaxDevices = 64;
int noalloc_scratch_init(int device);
int launch_ray_noalloc(gpurt_bvh_s* b, const gpurt_ray* rays, size_t n, int32_t* prim, float* t, float* uv,
                       const gpurt_query_opts* opts, hipStream_t s);

// backward (backward.hip)
int launch_cpq_bwd(gpurt_bvh_s* b, const float* q, size_t n, const int32_t* prim, const float* g,
                   float* g_q, float* g_verts, hipStream_t s);
int launch_ray_bwd(gpurt_bvh_s* b, const gpurt_ray* rays, size_t n, const int32_t* prim,
                   const float* t, const float* uv, const float* g, float* g_o, float* g_d,
                   float* g_verts, hipStream_t s);

int launch_refit(gpurt_bvh_s* b, const float* verts, size_t vstride_floats, hipStream_t s);

// host-side facts of a TLAS (tlas.hip): its context, and per instance the custom index
// and the BLAS
int tlas_host_info(gpurt_tlas t, gpurt_ctx* ctx, const std::vector<uint32_t>** custom,
                   const std::vector<gpurt_bvh_s*>** blas);
// A second ray list of a closest-hit launch, in the caller's scratch: only the object hit
// is written (-1: none).  The caller has cleared the queue counters of the scratch.
struct TlasSecond {
    const gpurt_ray* rays;
    size_t n;               // capacity of the list
    const uint32_t* n_dev;  // its length in device memory; nullptr: no list
    int32_t* obj;
};
// TLAS traversal for wavefront callers (tlas.hip): the ray count may be read from device
// memory at launch (n_dev, at most n) and the traversal scratch may be the caller's
// (scratch of >= tlas_scratch_bytes(T, n + second's n) bytes; nullptr: allocated per call)
int tlas_trace_ex(gpurt_tlas T, const gpurt_ray* rays, size_t n, const uint32_t* n_dev, int32_t* obj,
                  int32_t* prim, float* t, float* uv, uint8_t* occ, bool any, const gpurt_query_opts* opts,
                  hipStream_t s, void* scratch, size_t scratch_bytes, const TlasSecond* second = nullptr);
size_t tlas_scratch_bytes(gpurt_tlas T, size_t n);
// records a use of the TLAS (and through it of its BLASes) on stream s (tlas.hip)
void tlas_note_use(gpurt_tlas t, hipStream_t s);
// gpurt_ctx_destroy's part for a TLAS still open: frees its device memory on the
// context's release stream and detaches it from the context (tlas.hip)
void tlas_orphan(gpurt_tlas t);

inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

}  // namespace gpurt_impl
