// gps_bvh.hip — load-time Gaussian order of the reference's BVH reorder
// (GaussianBVH::build_bvh_and_reorder, src/core/rendering/occlusion/
// gaussian_bvh.cu:146-169), built on the GPU.
//
// The reference builds a tinybvh 1.6.7 binned-SAH BVH on the CPU
// (packages/tinybvh/tiny_bvh.h:2292-2420) over one flat triangle per Gaussian
// and then reorders the Gaussians by a depth-first walk of its leaves
// (gaussian_bvh.cu:14-34).  That walk pushes the leaves' primIdx *positions*
// (leftFirst + i), not the primitive ids stored there, and visits the right
// child first; reorder() (gaussian_bvh.cu:47-84) then moves Gaussian m to
// leafOrder[m].  So only the leaf ranges matter: a leaf holding positions
// [f, f + c) receives old indices [n - f - c, n - f) in order, i.e.
//     perm[q] = (n - f - c) + (q - f)      for q in [f, f + c).
// The leaf ranges depend only on the split decisions, and every quantity a
// decision reads (bin counts, bin bounds as min/max) is independent of the
// order of the Gaussians inside a node.  The build therefore runs
// level-synchronously: one pass bins every Gaussian of every open node,
// half a wave per node evaluates the SAH exactly as tinybvh does, and a
// partition pass scatters each Gaussian to its child's range (ranks in
// LDS, one cursor atomic per node side and workgroup).  Nodes of at most 32 Gaussians are
// finished after the last level by half a wave each.
//
// Float min/max go through an order-preserving integer encoding (atomic
// min/max), which orders -0 below +0 where tinybvh keeps whichever zero came
// last; a zero-sign difference in a bound cannot change a split decision
// (the decision reads extents and areas, and a zero area makes the cost
// NaN, i.e. "split", for either sign).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "../../include/gps.h"
#include "gps_detmath.h"
#include "gps_project.h"

namespace {

constexpr int BINS = 8;                  // BVHBINS (tiny_bvh.h:104-106)
constexpr float FAR = 1e30f;             // BVH_FAR (tiny_bvh.h:144)
constexpr uint32_t MT_THRESHOLD = 50000; // MT_BUILD_THRESHOLD (tiny_bvh.h:148-150)
constexpr uint32_t TASKS = 256;          // task stack of BVH::Build (tiny_bvh.h:2308)
constexpr uint32_t SMALL = 32;           // nodes this small finish in half a wave
constexpr uint32_t CHUNK = 512;          // positions per step of the bin pass
constexpr uint32_t BIN_STEPS = 8;        // steps of one workgroup of the bin pass, at most
constexpr uint32_t PCHUNK = 2048;        // positions per workgroup of the partition pass
constexpr uint32_t THREADS = 256;
// Open nodes hold more than SMALL Gaussians, so a chunk overlaps at most
// ceil(CHUNK / (SMALL + 1)) + 1 of them.
constexpr uint32_t MAXN = (CHUNK + SMALL) / (SMALL + 1) + 1;
constexpr uint32_t PMAXN = (PCHUNK + SMALL) / (SMALL + 1) + 1;
// A bin is 8 words: encoded minimum, count, encoded maximum, one unused, so that
// two 16-byte accesses move it and the eight bins of an axis lie in 64 banks.
constexpr uint32_t BINW = 3 * BINS * 8;  // words of one node's bins
constexpr uint32_t GROUPS = 8;           // nodes per workgroup where half a wave takes a node
constexpr uint32_t EMIT_BLOCK = 256;     // nodes per workgroup of the emit pass
static_assert(MAXN == 17 && PMAXN == 64, "chunk/node bound");

// A Gaussian's fragment: tinybvh's min/max of the three triangle vertices.
// The triangle is flat in z, so bmax.z == bmin.z and is not stored.
struct alignas(8) Frag {
    float lx, ly, lz, hx, hy, pad;
};

struct ONode {  // an open node: a position range and its box
    float mn[3], mx[3];
    uint32_t first, count;
    uint32_t tc;     // task-stack depth tinybvh has when it splits this node
    uint32_t depth;  // tree depth, saturated at 6
};
constexpr uint32_t SMALL_BUF = 1u << 31;  // in a small node's tc: its fragments are in buffer 1

struct Split {
    float lmn[3], lmx[3], rmn[3], rmx[3];
    float nmin, rpd;
    uint32_t axis, pos, left, kind;  // kind: 0 leaf, 1 split
    uint32_t curL, curR;             // partition cursors
};

__device__ __forceinline__ float fmin_(float a, float b) { return a < b ? a : b; }  // tiny_bvh.h:445
__device__ __forceinline__ float fmax_(float a, float b) { return a > b ? a : b; }  // tiny_bvh.h:446
__device__ __forceinline__ int32_t clampi(int32_t x, int32_t a, int32_t b) { return x > a ? (x < b ? x : b) : a; }

// x86-64 conversions (cvttss2si) as the reference host performs them.
__device__ __forceinline__ int32_t cvt_i32(float x) {
    return (x >= -2147483648.0f && x < 2147483648.0f) ? (int32_t)x : INT32_MIN;
}
__device__ __forceinline__ uint32_t cvt_u32(float x) {
    return (x >= -9223372036854775808.0f && x < 9223372036854775808.0f) ? (uint32_t)(uint64_t)(int64_t)x : 0u;
}

__device__ __forceinline__ uint32_t ford(float f) {
    const uint32_t u = gps::f2u_bits(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float fdec(uint32_t e) {
    return gps::u2f_bits((e & 0x80000000u) ? (e & 0x7fffffffu) : ~e);
}

__device__ __forceinline__ float half_area(float x, float y, float z) {  // tiny_bvh.h:460
    return x < -FAR ? 0.0f : (x * y + y * z + z * x);
}

__device__ __forceinline__ float centroid(const Frag& f, uint32_t a) {
    return a == 0 ? (f.lx + f.hx) * 0.5f : a == 1 ? (f.ly + f.hy) * 0.5f : (f.lz + f.lz) * 0.5f;
}

__device__ __forceinline__ uint32_t bin_init(uint32_t w) { return (w & 7u) < 3u ? 0xffffffffu : 0u; }

__device__ __forceinline__ void wave_sync() {  // LDS of one wave: its accesses run in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A candidate split: the boxes and counts left and right of a bin boundary.
struct Cut {
    float lmn[3], lmx[3], rmn[3], rmx[3];
    uint32_t lN, rN;
};
__device__ __forceinline__ Cut empty_cut() {
    return {{FAR, FAR, FAR}, {-FAR, -FAR, -FAR}, {FAR, FAR, FAR}, {-FAR, -FAR, -FAR}, 0u, 0u};
}

// The boundary after bin bn of an axis from the axis' eight bins in LDS, (min,
// count) and (max, -): prefix and suffix in the order of tiny_bvh.h:2336-2356.
__device__ __forceinline__ Cut cut_of_bins(const float4 (*bins)[2], uint32_t bn) {
    Cut c = empty_cut();
    float4 p[BINS], q[BINS];
#pragma unroll
    for (int i = 0; i < BINS; ++i) p[i] = bins[i][0], q[i] = bins[i][1];
#pragma unroll
    for (int i = 0; i < BINS - 1; ++i)
        if ((uint32_t)i <= bn) {
            c.lN += gps::f2u_bits(p[i].w);
            c.lmn[0] = fmin_(c.lmn[0], p[i].x), c.lmn[1] = fmin_(c.lmn[1], p[i].y), c.lmn[2] = fmin_(c.lmn[2], p[i].z);
            c.lmx[0] = fmax_(c.lmx[0], q[i].x), c.lmx[1] = fmax_(c.lmx[1], q[i].y), c.lmx[2] = fmax_(c.lmx[2], q[i].z);
        }
#pragma unroll
    for (int i = BINS - 1; i > 0; --i)
        if ((uint32_t)i > bn) {
            c.rN += gps::f2u_bits(p[i].w);
            c.rmn[0] = fmin_(c.rmn[0], p[i].x), c.rmn[1] = fmin_(c.rmn[1], p[i].y), c.rmn[2] = fmin_(c.rmn[2], p[i].z);
            c.rmx[0] = fmax_(c.rmx[0], q[i].x), c.rmx[1] = fmax_(c.rmx[1], q[i].y), c.rmx[2] = fmax_(c.rmx[2], q[i].z);
        }
    return c;
}

// The lane (8 axis + bin) of the cheapest boundary among a group's 32 lanes,
// the first of equals as the sequential search keeps it (tiny_bvh.h:2357-2369),
// or 32 if no axis has a candidate; `cost` becomes that boundary's cost.
__device__ __forceinline__ uint32_t best_cut(const Cut& c, uint32_t l, float ext, float min_dim, float* cost) {
    const float anl = c.lN == 0u ? FAR : half_area(c.lmx[0] - c.lmn[0], c.lmx[1] - c.lmn[1], c.lmx[2] - c.lmn[2]) * (float)c.lN;
    const float anr = c.rN == 0u ? FAR : half_area(c.rmx[0] - c.rmn[0], c.rmx[1] - c.rmn[1], c.rmx[2] - c.rmn[2]) * (float)c.rN;
    const float C = anl + anr;
    const bool can = l < 3u * BINS && (l & 7u) < (uint32_t)BINS - 1u && ext > min_dim && C < FAR;
    float v = can ? C : FAR;
    uint32_t at = can ? l : 32u;
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) {
        const float ov = __shfl_xor(v, d, 32);
        const uint32_t oa = __shfl_xor(at, d, 32);
        if (ov < v || (ov == v && oa < at)) v = ov, at = oa;
    }
    *cost = v;
    return at;
}

__device__ __forceinline__ float node_area(const float mn[3], const float mx[3]) {  // BVHBase::SA, tiny_bvh.h:8437-8441
    const float ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
    return ex * ey + ey * ez + ez * ex;
}

// Child task-stack depth (tiny_bvh.h:2393-2400): subtrees of nodes above
// depth 5 start on fresh threads (empty stack) in a threaded build; otherwise
// the left child runs with the right one pushed.
__device__ __forceinline__ uint32_t child_tc(uint32_t tc, uint32_t depth, bool threaded, bool left) {
    if (threaded && depth < 5) return 0u;
    return left ? tc + 1u : tc;
}

// ------------------------------------------------------------------ kernels
// gaussian_bvh.cu:150-155 + gaussian_bvh.cuh:20-26 + tiny_bvh.h:2256-2266.
__global__ __launch_bounds__(256) void bvh_frag_kernel(const float* __restrict__ means, const float* __restrict__ rots,
                                                       const float* __restrict__ scales, uint32_t n,
                                                       Frag* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float C[9];
    gps::scale_rot_to_cov(scales[3 * i], scales[3 * i + 1], scales[3 * i + 2], rots[4 * i], rots[4 * i + 1],
                          rots[4 * i + 2], rots[4 * i + 3], C);
    const float ex = 3.0f * gps::det_sqrt(C[0]), ey = 3.0f * gps::det_sqrt(C[4]), ez = 3.0f * gps::det_sqrt(C[8]);
    const float lx = means[3 * i] - ex, ly = means[3 * i + 1] - ey, lz = means[3 * i + 2] - ez;
    const float hx = means[3 * i] + ex, hy = means[3 * i + 1] + ey;
    // vertices (lx, ly, lz), (hx, ly, lz), (lx, hy, lz)
    Frag f;
    f.lx = fmin_(lx, fmin_(hx, lx));
    f.ly = fmin_(ly, fmin_(ly, hy));
    f.lz = lz;
    f.hx = fmax_(lx, fmax_(hx, lx));
    f.hy = fmax_(ly, fmax_(ly, hy));
    f.pad = 0.0f;
    out[i] = f;
}

// Root box: encoded min of bmin, max of bmax over all fragments.
__global__ __launch_bounds__(256) void bvh_root_kernel(const Frag* __restrict__ fr, uint32_t n, uint32_t* __restrict__ box) {
    uint32_t mn[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, mx[3] = {0u, 0u, 0u};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const Frag f = fr[i];
        mn[0] = min(mn[0], ford(f.lx)), mn[1] = min(mn[1], ford(f.ly)), mn[2] = min(mn[2], ford(f.lz));
        mx[0] = max(mx[0], ford(f.hx)), mx[1] = max(mx[1], ford(f.hy)), mx[2] = max(mx[2], ford(f.lz));
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
        for (int m = 32; m >= 1; m >>= 1) {
            mn[c] = min(mn[c], (uint32_t)__shfl_xor((int)mn[c], m, 64));
            mx[c] = max(mx[c], (uint32_t)__shfl_xor((int)mx[c], m, 64));
        }
    // one atomic per word and workgroup (one per wave, on six words: 292 us at 4M)
    __shared__ uint32_t s_box[6];
    if (threadIdx.x < 6) s_box[threadIdx.x] = threadIdx.x < 3 ? 0xffffffffu : 0u;
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        for (int c = 0; c < 3; ++c) {
            atomicMin(&s_box[c], mn[c]);
            atomicMax(&s_box[3 + c], mx[c]);
        }
    __syncthreads();
    if (threadIdx.x < 3) atomicMin(&box[threadIdx.x], s_box[threadIdx.x]);
    else if (threadIdx.x < 6) atomicMax(&box[threadIdx.x], s_box[threadIdx.x]);
}

// Root node and the build constants (PrepareBuild, tiny_bvh.h:2253-2266;
// minDim, tiny_bvh.h:2310).
__global__ __launch_bounds__(BINW) void bvh_root_node_kernel(const uint32_t* __restrict__ box, uint32_t n,
                                                             ONode* __restrict__ root, float* __restrict__ min_dim,
                                                             uint32_t* __restrict__ bins, uint2* __restrict__ sums,
                                                             uint32_t* __restrict__ err) {
    bins[threadIdx.x] = bin_init(threadIdx.x);
    if (threadIdx.x != 0) return;
    *sums = make_uint2(0u, 0u);
    *err = 0u;
    ONode r;
    for (int c = 0; c < 3; ++c) {
        r.mn[c] = fmin_(FAR, fdec(box[c]));
        r.mx[c] = fmax_(-FAR, fdec(box[3 + c]));
        min_dim[c] = (r.mx[c] - r.mn[c]) * 1e-20f;
    }
    r.first = 0, r.count = n, r.tc = 0, r.depth = 0;
    *root = r;
}

// The first open node that ends after position s (the list is in position
// order), by one wave: 64 probes a round.
__device__ uint32_t first_node(const ONode* __restrict__ nodes, uint32_t nn, uint32_t s) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lo = 0, len = nn;
    while (len > 0u) {
        const uint32_t step = (len + 63u) >> 6, e = lane * step + step - 1u;
        const bool before = e < len && nodes[lo + e].first + nodes[lo + e].count <= s;
        const uint32_t c = (uint32_t)__popcll(__ballot(before));
        lo += c * step;
        len = min(step - 1u, len - c * step);
    }
    return lo;
}

// How many open nodes from k on begin before position e, up to `most` (<= 64), by one wave.
__device__ uint32_t nodes_before(const ONode* __restrict__ nodes, uint32_t nn, uint32_t k, uint32_t e, uint32_t most) {
    const uint32_t lane = threadIdx.x & 63u;
    return (uint32_t)__popcll(__ballot(lane < most && k + lane < nn && nodes[k + lane].first < e));
}

// The slot of position p among m position-ordered nodes, or -1.
__device__ __forceinline__ int find_slot(const uint32_t* s_first, const uint32_t* s_count, uint32_t m, uint32_t p) {
    uint32_t lo = 0, hi = m;  // last node with first <= p
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_first[mid] <= p)
            lo = mid;
        else
            hi = mid;
    }
    return p >= s_first[lo] && p - s_first[lo] < s_count[lo] ? (int)lo : -1;
}

// Bins of every open node (tiny_bvh.h:2315-2331), LDS-aggregated.  A
// workgroup takes `steps` steps of CHUNK positions and adds its bins to the
// nodes' when the nodes change: inside one large node that is once, where
// thousands of workgroups add to the same words.  A bound is only sent to the
// bin where it moves it, and a wave inside one node counts its bins with
// ballots: an LDS atomic on a shared word runs lane after lane.  4M, a launch:
// 56 us on average over 23 levels (94 without these; the fragments' reads are 21).
__global__ __launch_bounds__(THREADS) void bvh_bin_kernel(const Frag* __restrict__ fr, uint32_t n,
                                                          const ONode* __restrict__ nodes, uint32_t nn,
                                                          uint32_t steps, uint32_t* __restrict__ bins) {
    __shared__ uint32_t s_k0, s_m;
    __shared__ uint32_t s_first[MAXN], s_count[MAXN];
    __shared__ float s_nmin[MAXN][3], s_rpd[MAXN][3];
    __shared__ alignas(16) uint32_t s_bins[MAXN * BINW];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    uint32_t k0 = 0u, m = 0u;  // nodes whose bins are in LDS
    auto flush = [&]() {
        for (uint32_t i = tid; i < m * BINW; i += THREADS) {
            const uint32_t w = i & 7u, v = s_bins[i];
            uint32_t* g = bins + (uint64_t)k0 * BINW + i;
            if (w < 3u) {
                if (v != 0xffffffffu) atomicMin(g, v);
            } else if (v) {
                if (w == 3u)
                    atomicAdd(g, v);
                else
                    atomicMax(g, v);
            }
        }
    };
    for (uint32_t step = 0; step < steps; ++step) {
        const uint32_t s = (blockIdx.x * steps + step) * CHUNK;
        if (s >= n) break;  // uniform
        if (tid < 64) {
            // after the first step: the last node of the step before, or the one after it
            uint32_t k = step == 0 ? first_node(nodes, nn, s) : s_k0 + (s_m ? s_m - 1u : 0u);
            if (step != 0 && k < nn && nodes[k].first + nodes[k].count <= s) ++k;
            const uint32_t mm = nodes_before(nodes, nn, k, s + CHUNK, MAXN);
            if (tid == 0) s_k0 = k, s_m = mm;
        }
        __syncthreads();
        const uint32_t nm = s_m, nk = s_k0;
        if (nm == 0u) {  // uniform
            __syncthreads();
            continue;
        }
        if (!(nm == 1u && m == 1u && nk == k0)) {
            flush();
            __syncthreads();
            m = nm;
            k0 = nk;
            if (tid < m) {
                const ONode& nd = nodes[k0 + tid];
                s_first[tid] = nd.first;
                s_count[tid] = nd.count;
                for (int c = 0; c < 3; ++c) {
                    s_nmin[tid][c] = nd.mn[c];
                    s_rpd[tid][c] = (float)BINS / (nd.mx[c] - nd.mn[c]);
                }
            }
            for (uint32_t i = tid; i < m * BINW; i += THREADS) s_bins[i] = bin_init(i);
            __syncthreads();
        }
        for (uint32_t r = 0; r < CHUNK / THREADS; ++r) {
            const uint32_t p = s + r * THREADS + tid;
            const int j = p < n ? find_slot(s_first, s_count, m, p) : -1;
            uint32_t bi[3] = {0u, 0u, 0u};
            if (j >= 0) {
                const Frag f = fr[p];
                const uint32_t emn[3] = {ford(f.lx), ford(f.ly), ford(f.lz)};
                const uint32_t emx[3] = {ford(f.hx), ford(f.hy), ford(f.lz)};
#pragma unroll
                for (uint32_t a = 0; a < 3; ++a) {
                    bi[a] = (uint32_t)clampi(cvt_i32((centroid(f, a) - s_nmin[j][a]) * s_rpd[j][a]), 0, BINS - 1);
                    uint32_t* b = s_bins + (uint32_t)j * BINW + (a * BINS + bi[a]) * 8u;
                    // bounds only move outwards, so an old value only sends too many
                    const uint4 lo = *(const uint4*)b, hi = *(const uint4*)(b + 4);
                    if (emn[0] < lo.x) atomicMin(&b[0], emn[0]);
                    if (emn[1] < lo.y) atomicMin(&b[1], emn[1]);
                    if (emn[2] < lo.z) atomicMin(&b[2], emn[2]);
                    if (emx[0] > hi.x) atomicMax(&b[4], emx[0]);
                    if (emx[1] > hi.y) atomicMax(&b[5], emx[1]);
                    if (emx[2] > hi.z) atomicMax(&b[6], emx[2]);
                }
            }
            const uint64_t in = __ballot(j >= 0);
            if (in == 0ull) continue;
            const int j0 = __builtin_amdgcn_readlane(j, __builtin_ctzll(in));
            if (__ballot(j >= 0 && j != j0) == 0ull) {
                uint64_t v[3][3];
#pragma unroll
                for (int a = 0; a < 3; ++a)
#pragma unroll
                    for (int c = 0; c < 3; ++c) v[a][c] = __ballot((bi[a] >> c) & 1u);
                const uint32_t a = lane >> 3, q = lane & 7u;
                uint64_t mask = in;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const uint64_t w = a == 0u ? v[0][c] : a == 1u ? v[1][c] : v[2][c];
                    mask &= (q >> c) & 1u ? w : ~w;
                }
                const uint32_t cnt = (uint32_t)__popcll(mask);
                if (lane < 3u * BINS && cnt) atomicAdd(&s_bins[(uint32_t)j0 * BINW + lane * 8u + 3u], cnt);
            } else if (j >= 0) {
#pragma unroll
                for (uint32_t a = 0; a < 3; ++a) atomicAdd(&s_bins[(uint32_t)j * BINW + (a * BINS + bi[a]) * 8u + 3u], 1u);
            }
        }
        __syncthreads();
    }
    flush();
}

// 32 lanes per open node: tinybvh's decision (tiny_bvh.h:2333-2391) from the
// node's bins, lane 8 a + b for bin b of axis a.  Writes the split record and
// the number of children that stay open (x) and that wait as small (y), and
// adds these to the sum of the node's emit workgroup.
__global__ __launch_bounds__(32 * GROUPS) void bvh_split_kernel(const ONode* __restrict__ nodes, uint32_t nn,
                                                                const uint32_t* __restrict__ bins,
                                                                const float* __restrict__ min_dim,
                                                                Split* __restrict__ splits, uint2* __restrict__ counts,
                                                                uint2* __restrict__ sums, uint32_t* __restrict__ err) {
    __shared__ float4 s_bin[GROUPS][3 * BINS][2];
    __shared__ uint32_t s_sum[2];
    const uint32_t l = threadIdx.x & 31u, g = threadIdx.x >> 5, k = blockIdx.x * GROUPS + g;
    const uint32_t ax = min(l >> 3, 2u), bn = l & 7u;
    if (threadIdx.x < 2) s_sum[threadIdx.x] = 0u;
    __syncthreads();
    const bool have = k < nn;
    ONode nd{};
    if (have) nd = nodes[k];
    if (l < 3u * BINS) {
        uint4 lo = make_uint4(0u, 0u, 0u, 0u), hi = lo;
        if (have) {
            const uint4* b = (const uint4*)(bins + (uint64_t)k * BINW) + 2u * l;
            lo = b[0], hi = b[1];
        }
        const bool any = lo.w != 0u;
        s_bin[g][l][0] = make_float4(any ? fmin_(FAR, fdec(lo.x)) : FAR, any ? fmin_(FAR, fdec(lo.y)) : FAR,
                                     any ? fmin_(FAR, fdec(lo.z)) : FAR, gps::u2f_bits(lo.w));
        s_bin[g][l][1] = make_float4(any ? fmax_(-FAR, fdec(hi.x)) : -FAR, any ? fmax_(-FAR, fdec(hi.y)) : -FAR,
                                     any ? fmax_(-FAR, fdec(hi.z)) : -FAR, 0.0f);
    }
    wave_sync();
    const Cut c = cut_of_bins(&s_bin[g][ax * BINS], bn);
    const float ext = ax == 0u ? nd.mx[0] - nd.mn[0] : ax == 1u ? nd.mx[1] - nd.mn[1] : nd.mx[2] - nd.mn[2];
    float cost;
    const uint32_t at = best_cut(c, l, ext, min_dim[ax], &cost);
    const bool found = at < 32u;
    if (have && l == (found ? at : 0u)) {  // axis 0, bin 0 where there is no candidate: ax and bn are these too
        const float rSAV = 1.0f / node_area(nd.mn, nd.mx);
        const float splitCost = 1.0f + 1.0f * rSAV * cost;
        Split sp;
        for (int i = 0; i < 3; ++i) {
            sp.lmn[i] = found ? c.lmn[i] : 0.0f, sp.lmx[i] = found ? c.lmx[i] : 0.0f;
            sp.rmn[i] = found ? c.rmn[i] : 0.0f, sp.rmx[i] = found ? c.rmx[i] : 0.0f;
        }
        sp.axis = ax, sp.pos = bn;
        sp.nmin = ax == 0u ? nd.mn[0] : ax == 1u ? nd.mn[1] : nd.mn[2];
        sp.rpd = (float)BINS / ext;
        sp.left = c.lN;
        sp.curL = 0, sp.curR = 0;
        const uint32_t left = c.lN, right = nd.count - c.lN;
        bool split = !(splitCost >= (float)nd.count * 1.0f) && left != 0u && right != 0u && nd.tc != TASKS;
        // With no candidate on any axis tinybvh may still split on axis 0 when
        // the node area exceeds ~1e30 / count; its partition then converts
        // out-of-range bin values differently from the binning, so the counts
        // above do not apply.  Such scenes are reported, not built.
        if (split && !(ext > min_dim[ax])) {
            atomicOr(err, 1u);
            split = false;
        }
        sp.kind = split ? 1u : 0u;
        splits[k] = sp;
        uint2 c2 = make_uint2(0u, 0u);
        if (split) {
            c2.x = (left > SMALL ? 1u : 0u) + (right > SMALL ? 1u : 0u);
            c2.y = 2u - c2.x;
            atomicAdd(&s_sum[0], c2.x);
            atomicAdd(&s_sum[1], c2.y);
        }
        counts[k] = c2;
    }
    __syncthreads();
    if (threadIdx.x < 2 && s_sum[threadIdx.x])  // a workgroup's nodes lie in one emit workgroup
        atomicAdd((uint32_t*)&sums[blockIdx.x * GROUPS / EMIT_BLOCK] + threadIdx.x, s_sum[threadIdx.x]);
}

__device__ __forceinline__ uint2 add2(uint2 a, uint2 b) { return make_uint2(a.x + b.x, a.y + b.y); }

__device__ uint2 block_exclusive(uint2 v, uint2* s_tmp, uint2* total) {
    // 256 threads; wave scans then a scan of the four wave totals.
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint2 x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t tx = (uint32_t)__shfl_up((int)x.x, d, 64), ty = (uint32_t)__shfl_up((int)x.y, d, 64);
        if ((int)lane >= d) x.x += tx, x.y += ty;
    }
    if (lane == 63) s_tmp[wave] = x;
    __syncthreads();
    uint2 off = make_uint2(0u, 0u);
    for (uint32_t w = 0; w < wave; ++w) off = add2(off, s_tmp[w]);
    *total = add2(add2(s_tmp[0], s_tmp[1]), add2(s_tmp[2], s_tmp[3]));
    __syncthreads();
    return make_uint2(off.x + x.x - v.x, off.y + x.y - v.y);
}

// Children of split nodes into the next open list and the small list, in
// position order (left before right, nodes in order), with the next level's
// bins and sums cleared.  A workgroup takes EMIT_BLOCK nodes and begins after
// the sum of the workgroups before it; the last one writes the totals.
static_assert(EMIT_BLOCK == 256 && EMIT_BLOCK % GROUPS == 0, "one node per thread");
__global__ __launch_bounds__(256) void bvh_emit_kernel(const ONode* __restrict__ nodes, uint32_t nn,
                                                       const Split* __restrict__ splits, const uint2* __restrict__ counts,
                                                       const uint2* __restrict__ sums, uint2* __restrict__ next_sums,
                                                       int threaded, ONode* __restrict__ next, ONode* __restrict__ small,
                                                       uint32_t buf, uint32_t* __restrict__ bins,
                                                       uint2* __restrict__ grand) {
    __shared__ uint2 s_tmp[4];
    const uint32_t tid = threadIdx.x;
    uint2 v = make_uint2(0u, 0u), carry;
    for (uint32_t b = tid; b < blockIdx.x; b += 256) v = add2(v, sums[b]);
    (void)block_exclusive(v, s_tmp, &carry);
    const uint32_t open0 = carry.x;
    const uint32_t k = blockIdx.x * EMIT_BLOCK + tid;
    const uint2 mine = k < nn ? counts[k] : make_uint2(0u, 0u);
    uint2 total;
    uint2 o = add2(carry, block_exclusive(mine, s_tmp, &total));
    carry = add2(carry, total);
    if (mine.x + mine.y != 0u) {
        const uint32_t in = buf ? SMALL_BUF : 0u;  // the buffer that this level's partition fills
        const ONode nd = nodes[k];
        const Split& sp = splits[k];
        ONode L, R;
        for (int c = 0; c < 3; ++c) {
            L.mn[c] = sp.lmn[c], L.mx[c] = sp.lmx[c];
            R.mn[c] = sp.rmn[c], R.mx[c] = sp.rmx[c];
        }
        L.first = nd.first, L.count = sp.left;
        R.first = nd.first + sp.left, R.count = nd.count - sp.left;
        L.tc = child_tc(nd.tc, nd.depth, threaded != 0, true);
        R.tc = child_tc(nd.tc, nd.depth, threaded != 0, false);
        L.depth = R.depth = nd.depth < 6 ? nd.depth + 1 : 6;
        if (L.count > SMALL) {
            next[o.x++] = L;
        } else {
            L.tc |= in;
            small[o.y++] = L;
        }
        if (R.count > SMALL) {
            next[o.x++] = R;
        } else {
            R.tc |= in;
            small[o.y++] = R;
        }
    }
    const uint64_t end = (uint64_t)carry.x * (BINW / 4);
    for (uint64_t i = (uint64_t)open0 * (BINW / 4) + tid; i < end; i += 256) {
        const uint32_t e = bin_init((uint32_t)i * 4u);
        ((uint4*)bins)[i] = make_uint4(e, e, e, 0u);
    }
    if (tid < 2) next_sums[2 * blockIdx.x + tid] = make_uint2(0u, 0u);  // one level at most doubles the nodes
    if (tid == 0 && blockIdx.x == gridDim.x - 1) *grand = carry;
}

// Moves each Gaussian of a split node into its child's range; leaves write
// their final indices (tiny_bvh.h:2372-2380 with any order inside a range).
// 2048 positions per workgroup: the cursors of a large node are two words that
// every workgroup adds to (first level at 4M: 233 us at 512 positions).
__global__ __launch_bounds__(THREADS) void bvh_partition_kernel(const Frag* __restrict__ src, Frag* __restrict__ dst,
                                                                uint32_t n, const ONode* __restrict__ nodes,
                                                                uint32_t nn, Split* __restrict__ splits,
                                                                uint32_t* __restrict__ perm, uint32_t* __restrict__ err) {
    __shared__ uint32_t s_k0, s_m;
    __shared__ uint32_t s_first[PMAXN], s_count[PMAXN], s_axis[PMAXN], s_pos[PMAXN], s_left[PMAXN], s_kind[PMAXN];
    __shared__ float s_nmin[PMAXN], s_rpd[PMAXN];
    __shared__ uint32_t s_cnt[2 * PMAXN], s_base[2 * PMAXN];
    const uint32_t s = blockIdx.x * PCHUNK, tid = threadIdx.x;
    if (tid < 64) {
        const uint32_t k = first_node(nodes, nn, s), mm = nodes_before(nodes, nn, k, s + PCHUNK, PMAXN);
        if (tid == 0) s_k0 = k, s_m = mm;
    }
    __syncthreads();
    const uint32_t m = s_m;
    if (m == 0) return;  // uniform
    if (tid < m) {
        const ONode& nd = nodes[s_k0 + tid];
        const Split& sp = splits[s_k0 + tid];
        s_first[tid] = nd.first, s_count[tid] = nd.count;
        s_axis[tid] = sp.axis, s_pos[tid] = sp.pos, s_left[tid] = sp.left, s_kind[tid] = sp.kind;
        s_nmin[tid] = sp.nmin, s_rpd[tid] = sp.rpd;
    }
    for (uint32_t i = tid; i < 2 * PMAXN; i += THREADS) s_cnt[i] = 0u;
    __syncthreads();
    // ranks inside the workgroup per (node, side), then one global cursor
    // bump per (node, side) for the whole workgroup
    constexpr uint32_t R = PCHUNK / THREADS;
    int key[R];
    uint32_t rank[R];
    Frag f[R];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        const uint32_t p = s + r * THREADS + tid;
        const int j = p < n ? find_slot(s_first, s_count, m, p) : -1;
        key[r] = -1;
        if (j < 0) continue;
        if (!s_kind[j]) {
            // leaf: positions [f, f + c) take old indices n - f - c + (q - f)
            perm[p] = (n - s_first[j] - s_count[j]) + (p - s_first[j]);
            continue;
        }
        f[r] = src[p];
        const uint32_t a = s_axis[j];
        const float c = centroid(f[r], a);
        const int32_t bi = clampi((int32_t)cvt_u32((c - s_nmin[j]) * s_rpd[j]), 0, BINS - 1);
        key[r] = 2 * j + ((uint32_t)bi <= s_pos[j] ? 0 : 1);
        rank[r] = atomicAdd(&s_cnt[key[r]], 1u);
    }
    __syncthreads();
    if (tid < 2 * m && s_cnt[tid]) {
        Split& sp = splits[s_k0 + (tid >> 1)];
        s_base[tid] = atomicAdd((tid & 1) ? &sp.curR : &sp.curL, s_cnt[tid]);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        if (key[r] < 0) continue;
        const uint32_t jj = (uint32_t)(key[r] >> 1);
        const uint32_t slot = s_base[key[r]] + rank[r];
        const uint32_t cap = (key[r] & 1) ? s_count[jj] - s_left[jj] : s_left[jj];
        if (slot < cap)
            dst[s_first[jj] + ((key[r] & 1) ? s_left[jj] + slot : slot)] = f[r];
        else
            atomicOr(err, 2u);
    }
}

// Nodes of at most SMALL Gaussians, 32 lanes each: the builder of
// tiny_bvh.h:2292-2420 on the node's range with the decisions of the level
// passes.  Lane i holds the fragment at position i; lane 8 a + b evaluates the
// boundary after bin b of axis a straight from the fragments, each of which
// lies on one side of it, and the fragments move to their side by rank.  Nodes
// wait in LDS; leaves write their final indices.  One launch takes the small
// nodes of all levels: 1.7 ms for the 186k nodes of a 4M scene, bound by the
// serial chain of each node's splits; one thread per node, launched after each
// level, took 24.7 ms.
// With a NaN among the fragments the order of the minima decides which bounds
// survive (a < b ? a : b), so such nodes keep the builder's order: bins first,
// then prefix and suffix, and the order that its in-place partition leaves.
__device__ __forceinline__ float min_num(float a, float b) {  // no NaN: one instruction
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max_num(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
struct SmallLds {
    float4 lo[SMALL];             // lx, ly, lz, hx
    uint2 hi[SMALL];              // hy, the three bins in 4 bits each
    float4 bin[3 * BINS][2];      // (min, count), (max, -)
    // waiting nodes, of two Gaussians or more each, then the left child of the
    // last split: (min, first | count << 8), (max, tc | depth << 16)
    float4 node[SMALL / 2 + 1][2];
};
template <bool NAN_ORDER>
__device__ __forceinline__ void small_node(SmallLds& s, ONode t, Frag f, bool busy, uint32_t n,
                                           const float* __restrict__ min_dim, bool threaded,
                                           uint32_t* __restrict__ perm) {
    const uint32_t l = threadIdx.x & 31u, half = threadIdx.x & 32u;
    const uint32_t ax = min(l >> 3, 2u), bn = l & 7u;  // lanes 24..31 decide nothing
    const float md = min_dim[ax];
    const uint32_t base = t.first;  // this group owns [base, base + count)
    t.first = 0u;
    uint32_t sp = 0u;  // waiting nodes
    // Both groups of a wave go round until both are done; t, sp and busy are
    // the same in all lanes of a group.
    while (__ballot(busy) != 0ull) {
        const bool mine = busy && l >= t.first && l - t.first < t.count;
        float rpd[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) rpd[c] = (float)BINS / (t.mx[c] - t.mn[c]);
        uint32_t key = 0u;
#pragma unroll
        for (uint32_t a = 0; a < 3; ++a)
            key |= (uint32_t)clampi(cvt_i32((centroid(f, a) - t.mn[a]) * rpd[a]), 0, BINS - 1) << (4 * a);
        s.lo[l] = make_float4(f.lx, f.ly, f.lz, f.hx);
        s.hi[l] = make_uint2(gps::f2u_bits(f.hy), key);
        wave_sync();
        const uint32_t todo = busy && t.count > 1u ? t.count : 0u;
        Cut c = empty_cut();
        if constexpr (NAN_ORDER) {
            uint32_t cnt = 0u;
            float mn[3] = {FAR, FAR, FAR}, mx[3] = {-FAR, -FAR, -FAR};
            for (uint32_t i = 0; i < todo; ++i) {
                const float4 lo = s.lo[t.first + i];
                const uint2 hi = s.hi[t.first + i];
                if (((hi.y >> (4u * ax)) & 15u) == bn) {
                    ++cnt;
                    mn[0] = fmin_(mn[0], lo.x), mn[1] = fmin_(mn[1], lo.y), mn[2] = fmin_(mn[2], lo.z);
                    mx[0] = fmax_(mx[0], lo.w), mx[1] = fmax_(mx[1], gps::u2f_bits(hi.x)), mx[2] = fmax_(mx[2], lo.z);
                }
            }
            if (l < 3u * BINS) {
                s.bin[l][0] = make_float4(mn[0], mn[1], mn[2], gps::u2f_bits(cnt));
                s.bin[l][1] = make_float4(mx[0], mx[1], mx[2], 0.0f);
            }
            wave_sync();
            c = cut_of_bins(&s.bin[ax * BINS], bn);
        } else {
            for (uint32_t i = 0; i < todo; ++i) {
                const float4 lo = s.lo[t.first + i];
                const uint2 hi = s.hi[t.first + i];
                const float hy = gps::u2f_bits(hi.x);
                if (((hi.y >> (4u * ax)) & 15u) <= bn) {
                    ++c.lN;
                    c.lmn[0] = min_num(c.lmn[0], lo.x), c.lmx[0] = max_num(c.lmx[0], lo.w);
                    c.lmn[1] = min_num(c.lmn[1], lo.y), c.lmx[1] = max_num(c.lmx[1], hy);
                    c.lmn[2] = min_num(c.lmn[2], lo.z), c.lmx[2] = max_num(c.lmx[2], lo.z);
                } else {
                    c.rmn[0] = min_num(c.rmn[0], lo.x), c.rmx[0] = max_num(c.rmx[0], lo.w);
                    c.rmn[1] = min_num(c.rmn[1], lo.y), c.rmx[1] = max_num(c.rmx[1], hy);
                    c.rmn[2] = min_num(c.rmn[2], lo.z), c.rmx[2] = max_num(c.rmx[2], lo.z);
                }
            }
            c.rN = todo - c.lN;
        }
        const float ext = ax == 0u ? t.mx[0] - t.mn[0] : ax == 1u ? t.mx[1] - t.mn[1] : t.mx[2] - t.mn[2];
        float cost;
        const uint32_t at = best_cut(c, l, ext, md, &cost);
        const bool found = at < 32u;
        const uint32_t axis = found ? at >> 3 : 0u, pos = found ? at & 7u : 0u;
        const float rSAV = 1.0f / node_area(t.mn, t.mx);
        const float splitCost = 1.0f + 1.0f * rSAV * cost;
        const bool want = todo != 0u && !(splitCost >= (float)t.count * 1.0f);
        // sides, by the partition's own conversion (tiny_bvh.h:2372-2380)
        const float nmin = axis == 0u ? t.mn[0] : axis == 1u ? t.mn[1] : t.mn[2];
        const float rp = axis == 0u ? rpd[0] : axis == 1u ? rpd[1] : rpd[2];
        const int32_t bi = clampi((int32_t)cvt_u32((centroid(f, axis) - nmin) * rp), 0, BINS - 1);
        const bool goes_left = (uint32_t)bi <= pos;
        const uint32_t ml = (uint32_t)(__ballot(mine && goes_left) >> half);
        const uint32_t mr = (uint32_t)(__ballot(mine && !goes_left) >> half);
        const uint32_t left = (uint32_t)__popc(ml), right = (uint32_t)__popc(mr);
        const bool split = want && left != 0u && right != 0u && t.tc != TASKS;
        // the lane that the fragment moves to: its rank on its side, others stay
        const uint32_t below = (1u << l) - 1u;
        uint32_t to = l;
        if (split && mine)
            to = t.first + (goes_left ? (uint32_t)__popc(ml & below) : left + (uint32_t)__popc(mr & below));
        if constexpr (NAN_ORDER) {
            uint32_t who = l, src = t.first, j = t.first + t.count;
            for (uint32_t i = 0; i < SMALL; ++i) {
                const uint32_t x = __shfl(who, src & 31u, 32);
                const bool on = split && i < t.count, lft = ((ml >> (x & 31u)) & 1u) != 0u;
                if (on && !lft) --j;
                const uint32_t y = __shfl(who, j & 31u, 32);
                if (on && !lft) {
                    if (l == j) who = x;
                    if (l == src) who = y;
                }
                if (on && lft) ++src;
            }
            to = (uint32_t)__builtin_amdgcn_ds_permute((int)((half + who) * 4u), (int)l);
        }
        const int dst = (int)((half + to) * 4u);
        f.lx = gps::u2f_bits((uint32_t)__builtin_amdgcn_ds_permute(dst, (int)gps::f2u_bits(f.lx)));
        f.ly = gps::u2f_bits((uint32_t)__builtin_amdgcn_ds_permute(dst, (int)gps::f2u_bits(f.ly)));
        f.lz = gps::u2f_bits((uint32_t)__builtin_amdgcn_ds_permute(dst, (int)gps::f2u_bits(f.lz)));
        f.hx = gps::u2f_bits((uint32_t)__builtin_amdgcn_ds_permute(dst, (int)gps::f2u_bits(f.hx)));
        f.hy = gps::u2f_bits((uint32_t)__builtin_amdgcn_ds_permute(dst, (int)gps::f2u_bits(f.hy)));
        uint32_t slot = SMALL / 2;  // where the next node is
        bool pop = busy && !split;
        const uint32_t f0 = base + t.first;
        if (split) {
            if (l == (found ? at : 0u)) {
                const uint32_t dp = (t.depth < 6 ? t.depth + 1 : 6) << 16;
                const float z = 0.0f;
                s.node[SMALL / 2][0] = make_float4(found ? c.lmn[0] : z, found ? c.lmn[1] : z, found ? c.lmn[2] : z,
                                                   gps::u2f_bits(t.first | left << 8));
                s.node[SMALL / 2][1] = make_float4(found ? c.lmx[0] : z, found ? c.lmx[1] : z, found ? c.lmx[2] : z,
                                                   gps::u2f_bits(child_tc(t.tc, t.depth, threaded, true) | dp));
                s.node[sp][0] = make_float4(found ? c.rmn[0] : z, found ? c.rmn[1] : z, found ? c.rmn[2] : z,
                                            gps::u2f_bits((t.first + left) | right << 8));
                s.node[sp][1] = make_float4(found ? c.rmx[0] : z, found ? c.rmx[1] : z, found ? c.rmx[2] : z,
                                            gps::u2f_bits(child_tc(t.tc, t.depth, threaded, false) | dp));
                // a single Gaussian is a leaf
                if (left == 1u) perm[f0] = n - f0 - 1u;
                if (right == 1u) perm[f0 + left] = n - f0 - left - 1u;
            }
            if (left > 1u)
                sp += right > 1u ? 1u : 0u;
            else if (right > 1u)
                slot = sp;
            else
                pop = true;
        } else if (busy && l < t.count) {
            perm[f0 + l] = (n - f0 - t.count) + l;
        }
        if (pop) {
            busy = sp != 0u;
            if (busy) slot = --sp;
        }
        wave_sync();
        if (busy) {
            const float4 a = s.node[slot][0], b = s.node[slot][1];
            const uint32_t r = gps::f2u_bits(a.w), d = gps::f2u_bits(b.w);
            t.mn[0] = a.x, t.mn[1] = a.y, t.mn[2] = a.z, t.mx[0] = b.x, t.mx[1] = b.y, t.mx[2] = b.z;
            t.first = r & 255u, t.count = r >> 8, t.tc = d & 0xffffu, t.depth = d >> 16;
        }
        wave_sync();
    }
}
__global__ __launch_bounds__(32 * GROUPS) void bvh_small_kernel(const Frag* __restrict__ fr0,
                                                                const Frag* __restrict__ fr1, uint32_t n,
                                                                const ONode* __restrict__ small, uint32_t ns,
                                                                const float* __restrict__ min_dim, int threaded,
                                                                uint32_t* __restrict__ perm) {
    __shared__ SmallLds s_lds[GROUPS];
    const uint32_t l = threadIdx.x & 31u, g = threadIdx.x >> 5, k = blockIdx.x * GROUPS + g;
    const bool have = k < ns;
    ONode t{};
    if (have) t = small[k];
    const Frag* fr = (t.tc & SMALL_BUF) ? fr1 : fr0;
    t.tc &= ~SMALL_BUF;
    Frag f{};
    if (have && l < t.count) f = fr[t.first + l];
    const bool nan = f.lx != f.lx || f.ly != f.ly || f.lz != f.lz || f.hx != f.hx || f.hy != f.hy;
    if (__ballot(nan) != 0ull)
        small_node<true>(s_lds[g], t, f, have, n, min_dim, threaded != 0, perm);
    else
        small_node<false>(s_lds[g], t, f, have, n, min_dim, threaded != 0, perm);
}

struct DevBuf {
    void* p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
};

}  // namespace

extern "C" gps_status gps_bvh_order(const float* means, const float* rotations, const float* scales, uint64_t n,
                                    uint32_t* perm) {
    if ((!means || !rotations || !scales || !perm) && n) return GPS_ERR_INVALID_ARG;
    if (n == 0) return GPS_OK;
    if (n > 0x7fffffffull) return GPS_ERR_UNSUPPORTED;
    const uint32_t N = (uint32_t)n;
    const uint32_t maxOpen = N / (SMALL + 1) + 1;  // open nodes are disjoint and hold > SMALL each
    const uint32_t maxSmall = 4 * maxOpen + 1;     // small nodes that wait; one level adds up to 2 * maxOpen
    const uint32_t nchunks = (N + CHUNK - 1) / CHUNK, npart = (N + PCHUNK - 1) / PCHUNK;
    // Steps per workgroup of the bin pass: at least 1024 workgroups while there
    // are chunks for them, and no more steps than the mean node has chunks, as
    // where every step changes the nodes there is nothing to save (4M, the
    // level with the most nodes: 106 us in steps of eight, 80 us in single ones).
    const uint32_t most_steps = nchunks / 1024u < BIN_STEPS ? nchunks / 1024u : BIN_STEPS;
    const uint32_t maxSums = 2 * ((maxOpen + EMIT_BLOCK - 1) / EMIT_BLOCK);  // emit clears two entries per workgroup
    DevBuf arena;
#define GPS_BVH_HIP(call)                              \
    do {                                               \
        if ((call) != hipSuccess) return GPS_ERR_HIP;  \
    } while (0)
    // One allocation, cut up: each hipFree of a large one waits 0.4 ms.
    uint64_t bytes = 0;
    auto take = [&](uint64_t size) {
        const uint64_t at = bytes;
        bytes += (size + 255) / 256 * 256;
        return at;
    };
    const uint64_t oFrag[2] = {take((uint64_t)N * sizeof(Frag)), take((uint64_t)N * sizeof(Frag))};
    const uint64_t oPerm = take((uint64_t)N * 4);
    const uint64_t oNodes[2] = {take((uint64_t)maxOpen * sizeof(ONode)), take((uint64_t)maxOpen * sizeof(ONode))};
    const uint64_t oSmall = take((uint64_t)maxSmall * sizeof(ONode));
    const uint64_t oBins = take((uint64_t)maxOpen * BINW * 4);
    const uint64_t oSplit = take((uint64_t)maxOpen * sizeof(Split));
    const uint64_t oCnt = take((uint64_t)maxOpen * sizeof(uint2));
    const uint64_t oSums[2] = {take((uint64_t)maxSums * sizeof(uint2)), take((uint64_t)maxSums * sizeof(uint2))};
    const uint64_t oMisc = take(256);
    // the inputs' slices lie where everything but the fragments comes later
    const uint32_t SLICE = 1u << 23;
    const uint64_t oIn = oFrag[1], in_end = oIn + (uint64_t)(N < SLICE ? N : SLICE) * 40;
    GPS_BVH_HIP(hipMalloc(&arena.p, bytes > in_end ? bytes : in_end));
    char* ar = (char*)arena.p;
    Frag* frag[2] = {(Frag*)(ar + oFrag[0]), (Frag*)(ar + oFrag[1])};
    ONode* open[2] = {(ONode*)(ar + oNodes[0]), (ONode*)(ar + oNodes[1])};
    ONode* small = (ONode*)(ar + oSmall);
    uint32_t* bins = (uint32_t*)(ar + oBins);
    Split* splits = (Split*)(ar + oSplit);
    uint2* cnt = (uint2*)(ar + oCnt);
    uint2* sums[2] = {(uint2*)(ar + oSums[0]), (uint2*)(ar + oSums[1])};
    uint32_t* box = (uint32_t*)(ar + oMisc);             // 6 words
    float* min_dim = (float*)(ar + oMisc + 64);          // 3 floats
    uint2* grand = (uint2*)(ar + oMisc + 128);           // 1 pair
    uint32_t* err = (uint32_t*)(ar + oMisc + 192);       // 1 word
    uint32_t* dperm = (uint32_t*)(ar + oPerm);
    const int threaded = N >= MT_THRESHOLD ? 1 : 0;

    // fragments, uploaded in slices
    for (uint32_t s0 = 0; s0 < N; s0 += SLICE) {
        const uint32_t c = N - s0 < SLICE ? N - s0 : SLICE;
        float* dm = (float*)(ar + oIn);
        float* dr = dm + 3ull * c;
        float* ds = dr + 4ull * c;
        GPS_BVH_HIP(hipMemcpy(dm, means + 3ull * s0, 12ull * c, hipMemcpyHostToDevice));
        GPS_BVH_HIP(hipMemcpy(dr, rotations + 4ull * s0, 16ull * c, hipMemcpyHostToDevice));
        GPS_BVH_HIP(hipMemcpy(ds, scales + 3ull * s0, 12ull * c, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(bvh_frag_kernel, dim3((c + 255) / 256), dim3(256), 0, 0, dm, dr, ds, c, frag[0] + s0);
        GPS_BVH_HIP(hipGetLastError());
    }

    const uint32_t boxInit[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
    GPS_BVH_HIP(hipMemcpy(box, boxInit, sizeof(boxInit), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(bvh_root_kernel, dim3(512), dim3(256), 0, 0, frag[0], N, box);
    hipLaunchKernelGGL(bvh_root_node_kernel, dim3(1), dim3(BINW), 0, 0, box, N, open[0], min_dim, bins, sums[0], err);
    GPS_BVH_HIP(hipGetLastError());

    int cur = 0, lv = 0;
    uint32_t nopen = 1, nsmall = 0;
    // Small nodes of all levels wait for one launch: each keeps its fragments in
    // the buffer that its level's partition filled, and no later level writes
    // outside its open nodes' ranges.  Splits that cut off a few Gaussians at a
    // time can make more than the list holds, so it is also emptied before a
    // level whose children might not fit.
    auto finish_small = [&]() {
        if (nsmall)
            hipLaunchKernelGGL(bvh_small_kernel, dim3((nsmall + GROUPS - 1) / GROUPS),
                               dim3(32 * GROUPS), 0, 0, frag[0], frag[1], N, small, nsmall, min_dim, threaded,
                               dperm);
        nsmall = 0;
    };
    if (N <= SMALL) {
        GPS_BVH_HIP(hipMemcpy(small, open[0], sizeof(ONode), hipMemcpyDeviceToDevice));
        nopen = 0;
        nsmall = 1;
    }
    while (nopen > 0) {
        if (nsmall + 2 * nopen > maxSmall) finish_small();
        const uint32_t mean = N / nopen / CHUNK, few = mean < most_steps ? mean : most_steps, steps = few > 1u ? few : 1u;
        hipLaunchKernelGGL(bvh_bin_kernel, dim3((nchunks + steps - 1) / steps), dim3(THREADS), 0, 0, frag[cur], N, open[lv], nopen, steps, bins);
        hipLaunchKernelGGL(bvh_split_kernel, dim3((nopen + GROUPS - 1) / GROUPS), dim3(32 * GROUPS), 0, 0, open[lv],
                           nopen, bins, min_dim, splits, cnt, sums[lv], err);
        hipLaunchKernelGGL(bvh_emit_kernel, dim3((nopen + EMIT_BLOCK - 1) / EMIT_BLOCK), dim3(256), 0, 0, open[lv],
                           nopen, splits, cnt, sums[lv], sums[lv ^ 1], threaded, open[lv ^ 1], small + nsmall,
                           (uint32_t)(cur ^ 1), bins, grand);
        hipLaunchKernelGGL(bvh_partition_kernel, dim3(npart), dim3(THREADS), 0, 0, frag[cur], frag[cur ^ 1], N,
                           open[lv], nopen, splits, dperm, err);
        GPS_BVH_HIP(hipGetLastError());
        uint2 g;
        GPS_BVH_HIP(hipMemcpy(&g, grand, sizeof(g), hipMemcpyDeviceToHost));
        if (g.x > maxOpen || g.y > 2 * nopen) return GPS_ERR_HIP;  // cannot happen: children are disjoint ranges
        nsmall += g.y;
        cur ^= 1;
        lv ^= 1;
        nopen = g.x;
    }
    finish_small();
    GPS_BVH_HIP(hipGetLastError());
    uint32_t herr = 0;
    GPS_BVH_HIP(hipMemcpy(&herr, err, 4, hipMemcpyDeviceToHost));
    if (herr) return GPS_ERR_UNSUPPORTED;
    GPS_BVH_HIP(hipMemcpy(perm, dperm, 4ull * N, hipMemcpyDeviceToHost));
#undef GPS_BVH_HIP
    return GPS_OK;
}
