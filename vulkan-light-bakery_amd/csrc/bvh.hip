// bvh.hip -- GPU BVH build for the probe baker (replaces the Vulkan BLAS/TLAS
// build of src/scene_manager.cpp:339-443; the reference hands triangles to
// the driver with ePreferFastTrace and culling disabled).
//
// 30-bit Morton codes of triangle centroids, a stable radix sort, then a
// PLOC hierarchy (agglomerative clustering over the Morton order, below)
// with one triangle per leaf, collapsed to the 4-wide BVH the traversal
// kernels walk.  Node boxes are unions of their children's boxes, i.e. the
// exact min/max of their triangles' vertices (conservative for the
// watertight test), and every step is deterministic.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "vlb_internal.hpp"

namespace vlb {
namespace {

// First index out of range and first vertex coordinate that is not finite or
// beyond 2^100 (bad[0], bad[1]; 0xffffffffffffffff: none).  On the host these
// loops took 0.45 of the 2.95 ms of opening a 0.5M-triangle terrain.
__global__ void k_check(const uint32_t* __restrict__ idx, unsigned long long nidx, uint32_t nverts,
                        const float* __restrict__ xyz, unsigned long long ncoords,
                        unsigned long long* __restrict__ bad)
{
    const unsigned long long step = (unsigned long long)gridDim.x * blockDim.x;
    const unsigned long long t = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long bi = ~0ull, bc = ~0ull;
    for (unsigned long long i = t; i < nidx; i += step)
        if (idx[i] >= nverts) bi = i < bi ? i : bi;
    for (unsigned long long i = t; i < ncoords; i += step)
        if (!(fabsf(xyz[i]) <= 0x1p100f)) bc = i < bc ? i : bc;
    if (bi != ~0ull) atomicMin(&bad[0], bi);
    if (bc != ~0ull) atomicMin(&bad[1], bc);
}

// Gather triangles, per-prim boxes and centroids, shading records.
__global__ void k_gather(const float* __restrict__ xyz, const uint32_t* __restrict__ idx,
                         const float* __restrict__ normals, const float* __restrict__ albedo,
                         int ntris, int nverts, float4* __restrict__ tri_raw,
                         float4* __restrict__ lo, float4* __restrict__ hi,
                         float4* __restrict__ cen, float4* __restrict__ shade)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntris) return;
    uint32_t i0 = idx[3 * i], i1 = idx[3 * i + 1], i2 = idx[3 * i + 2];
    if (i0 >= (uint32_t)nverts) i0 = 0;
    if (i1 >= (uint32_t)nverts) i1 = 0;
    if (i2 >= (uint32_t)nverts) i2 = 0;
    float3 v0 = make_float3(xyz[3 * i0], xyz[3 * i0 + 1], xyz[3 * i0 + 2]);
    float3 v1 = make_float3(xyz[3 * i1], xyz[3 * i1 + 1], xyz[3 * i1 + 2]);
    float3 v2 = make_float3(xyz[3 * i2], xyz[3 * i2 + 1], xyz[3 * i2 + 2]);
    tri_raw[3 * i + 0] = make_float4(v0.x, v0.y, v0.z, __int_as_float(i));
    tri_raw[3 * i + 1] = make_float4(v1.x, v1.y, v1.z, 0.0f);
    tri_raw[3 * i + 2] = make_float4(v2.x, v2.y, v2.z, 0.0f);
    float4 l = make_float4(fminf(v0.x, fminf(v1.x, v2.x)), fminf(v0.y, fminf(v1.y, v2.y)),
                           fminf(v0.z, fminf(v1.z, v2.z)), 0.0f);
    float4 h = make_float4(fmaxf(v0.x, fmaxf(v1.x, v2.x)), fmaxf(v0.y, fmaxf(v1.y, v2.y)),
                           fmaxf(v0.z, fmaxf(v1.z, v2.z)), 0.0f);
    lo[i] = l;
    hi[i] = h;
    cen[i] = make_float4(0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z), 0.0f);
    float3 n0, n1, n2;
    if (normals) {
        n0 = make_float3(normals[3 * i0], normals[3 * i0 + 1], normals[3 * i0 + 2]);
        n1 = make_float3(normals[3 * i1], normals[3 * i1 + 1], normals[3 * i1 + 2]);
        n2 = make_float3(normals[3 * i2], normals[3 * i2 + 1], normals[3 * i2 + 2]);
    } else {
        // geometric normal, same operation sequence as the host helper
        float3 e1 = make_float3(v1.x - v0.x, v1.y - v0.y, v1.z - v0.z);
        float3 e2 = make_float3(v2.x - v0.x, v2.y - v0.y, v2.z - v0.z);
        float3 n = make_float3(e1.y * e2.z - e1.z * e2.y, e1.z * e2.x - e1.x * e2.z,
                               e1.x * e2.y - e1.y * e2.x);
        float l2 = sqrtf(n.x * n.x + n.y * n.y + n.z * n.z);
        float3 g = l2 > 0.0f ? make_float3(n.x / l2, n.y / l2, n.z / l2)
                             : make_float3(0.0f, 1.0f, 0.0f);
        n0 = n1 = n2 = g;
    }
    float ar = albedo ? albedo[3 * i] : 1.0f;
    float ag = albedo ? albedo[3 * i + 1] : 1.0f;
    float ab = albedo ? albedo[3 * i + 2] : 1.0f;
    shade[3 * i + 0] = make_float4(n0.x, n0.y, n0.z, ar);
    shade[3 * i + 1] = make_float4(n1.x, n1.y, n1.z, ag);
    shade[3 * i + 2] = make_float4(n2.x, n2.y, n2.z, ab);
}

// Bounds reduction: centroid box (for Morton), scene box, max |coordinate|.
// Stage 1: one partial of 13 floats per block; stage 2: one block.
__device__ __forceinline__ void red13(float* v, float* sh)
{
    // v[0..2] min, v[3..5] max, v[6..8] min, v[9..11] max, v[12] max
    const int t = threadIdx.x;
    for (int k = 0; k < 13; ++k) sh[k * 256 + t] = v[k];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) {
            for (int k = 0; k < 13; ++k) {
                float a = sh[k * 256 + t], b = sh[k * 256 + t + s];
                bool is_min = (k < 3) || (k >= 6 && k < 9);
                sh[k * 256 + t] = is_min ? fminf(a, b) : fmaxf(a, b);
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_bounds1(const float4* __restrict__ lo,
                                                 const float4* __restrict__ hi,
                                                 const float4* __restrict__ cen, int n,
                                                 float* __restrict__ part)
{
    __shared__ float sh[13 * 256];
    float v[13];
    for (int k = 0; k < 3; ++k) {
        v[k] = v[6 + k] = __builtin_huge_valf();
        v[3 + k] = v[9 + k] = -__builtin_huge_valf();
    }
    v[12] = 0.0f;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        float4 c = cen[i], l = lo[i], h = hi[i];
        v[0] = fminf(v[0], c.x);
        v[1] = fminf(v[1], c.y);
        v[2] = fminf(v[2], c.z);
        v[3] = fmaxf(v[3], c.x);
        v[4] = fmaxf(v[4], c.y);
        v[5] = fmaxf(v[5], c.z);
        v[6] = fminf(v[6], l.x);
        v[7] = fminf(v[7], l.y);
        v[8] = fminf(v[8], l.z);
        v[9] = fmaxf(v[9], h.x);
        v[10] = fmaxf(v[10], h.y);
        v[11] = fmaxf(v[11], h.z);
        float m = fmaxf(fmaxf(fabsf(l.x), fabsf(l.y)), fmaxf(fabsf(l.z), fabsf(h.x)));
        m = fmaxf(m, fmaxf(fabsf(h.y), fabsf(h.z)));
        v[12] = fmaxf(v[12], m);
    }
    red13(v, sh);
    if (threadIdx.x < 13) part[blockIdx.x * 13 + threadIdx.x] = sh[threadIdx.x * 256];
}

__global__ __launch_bounds__(256) void k_bounds2(const float* __restrict__ part, int nb,
                                                 float* __restrict__ out)
{
    __shared__ float sh[13 * 256];
    float v[13];
    for (int k = 0; k < 3; ++k) {
        v[k] = v[6 + k] = __builtin_huge_valf();
        v[3 + k] = v[9 + k] = -__builtin_huge_valf();
    }
    v[12] = 0.0f;
    for (int b = threadIdx.x; b < nb; b += 256)
        for (int k = 0; k < 13; ++k) {
            float x = part[b * 13 + k];
            bool is_min = (k < 3) || (k >= 6 && k < 9);
            v[k] = is_min ? fminf(v[k], x) : fmaxf(v[k], x);
        }
    red13(v, sh);
    if (threadIdx.x < 13) out[threadIdx.x] = sh[threadIdx.x * 256];
}

__device__ __forceinline__ uint32_t expand_bits(uint32_t v)
{
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// 30-bit Morton code of each triangle's box centre on a grid of cubic cells:
// 1024 cells along the longest extent of the centre bounds, the same cell
// size on the other axes.  With cells stretched to 1024 per axis (2.5-6x
// finer vertically on the flat terrains and rooms) the PLOC pass built
// trees that traced 2-6% slower on three of the four scenes of the batched
// jobs and the same on the fourth (208.3 against 202.4 ms per batch); the
// 11k-triangle room bake of 2048 probes traces 2% faster with them (0.99
// against 1.01 ms).
__global__ void k_morton(const float4* __restrict__ cen, int n, const float* __restrict__ bounds,
                         uint32_t* __restrict__ keys, uint32_t* __restrict__ vals)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 c = cen[i];
    float q[3];
    const float cc[3] = {c.x, c.y, c.z};
    const float ext = fmaxf(fmaxf(bounds[3] - bounds[0], bounds[4] - bounds[1]), bounds[5] - bounds[2]);
    for (int a = 0; a < 3; ++a) {
        float x = ext > 0.0f ? (cc[a] - bounds[a]) / ext * 1024.0f : 0.0f;
        q[a] = fminf(fmaxf(x, 0.0f), 1023.0f);
    }
    keys[i] = (expand_bits((uint32_t)q[0]) << 2) | (expand_bits((uint32_t)q[1]) << 1) |
              expand_bits((uint32_t)q[2]);
    vals[i] = (uint32_t)i;
}

// ------------------------------------------------------------- PLOC
// Meister and Bittner, "Parallel Locally-Ordered Clustering for Bounding
// Volume Hierarchy Construction", IEEE TVCG 24(3), 2018.  Clusters start as
// the Morton-ordered leaves; each pass every cluster finds the neighbour
// within kPlocRadius positions whose union box has the least surface area,
// mutual pairs merge into a new inner node at the lower position, and the
// cluster list is compacted.  Candidate pairs are ordered by (area, distance
// in positions, parity of the lower position, lower position): a strict total
// order, so the least pair of a pass is always mutual and every pass merges
// at least once; and where areas tie (coincident or degenerate triangles),
// neighbours pair up as (0,1), (2,3), ... instead of chaining, so such runs
// halve each pass.  The build is deterministic (no atomics; positions and
// node ids come from one scan).  Node ids are handed out downward, so the
// final merge -- the root -- is node 0.  Search radius 32: on the batched
// jobs (rooms and terrains of 11k-1.15M triangles) 1.5% fewer node visits
// than radius 16 and a 1.3% shorter trace stage; 24 and 48 were no better,
// and the 11k-triangle room and the 1.15M-triangle terrain bakes trace in
// the same time at 16-64.
constexpr int kPlocRadius = 32;

// The initial clusters (leaf j = ~j; no inner node below).
__global__ void k_leaves(const uint32_t* __restrict__ order, int n, const float4* __restrict__ lo,
                         const float4* __restrict__ hi, float4* __restrict__ clo,
                         float4* __restrict__ chi, int* __restrict__ cid)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    uint32_t p = order[j];
    const float4 l = lo[p];
    clo[j] = make_float4(l.x, l.y, l.z, 0.0f);
    chi[j] = hi[p];
    cid[j] = ~j;
}

// fminf/fmaxf of numbers that were loaded get a canonicalizing instruction
// per operand first (12 of the 24 of a union's box); these do not.
__device__ __forceinline__ float min_f32(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max_f32(float a, float b)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Surface area (its half) of the union of two boxes, each axis as (lower,
// upper).  One fixed operation order: both clusters of a pair, on whichever
// path, see the same bits.
__device__ __forceinline__ float ploc_area(float2 ax, float2 ay, float2 az, float2 bx, float2 by,
                                           float2 bz)
{
    const float dx = max_f32(ax.y, bx.y) - min_f32(ax.x, bx.x);
    const float dy = max_f32(ay.y, by.y) - min_f32(ay.x, by.x);
    const float dz = max_f32(az.y, bz.y) - min_f32(az.x, bz.x);
    return dx * dy + dy * dz + dz * dx;
}

// Candidate j = i + o of area `ar` as a sort key: the area's bits, then the
// tie key (distance, then the lower position's parity, then the lower
// position: the left candidate is the lower one), unique per candidate, so
// the pair order is total.  A NaN area (non-finite input) counts as +inf.
// The key is also a positive finite double of the same order (v_min_f64), and
// kNoKey, +inf, is above all of them.
constexpr unsigned long long kNoKey = 0x7ff0000000000000ull;
__device__ __forceinline__ unsigned long long ploc_key(float ar, int i, int o)
{
    const int k = 4 * abs(o) + 2 * (min(i, i + o) & 1) + (o > 0 ? 1 : 0);
    const float a = min_f32(ar, __builtin_huge_valf());
    return ((unsigned long long)__float_as_uint(a) << 32) | (unsigned)k;
}
__device__ __forceinline__ unsigned long long min_key(unsigned long long a, unsigned long long b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(__longlong_as_double((long long)a)), "v"(__longlong_as_double((long long)b)));
    return (unsigned long long)__double_as_longlong(r);
}
// The candidate of a key.
__device__ __forceinline__ int ploc_neighbour(unsigned long long key, int i)
{
    const int k = (int)(uint32_t)key;
    return (k & 1) ? i + (k >> 2) : i - (k >> 2);
}

// Where a pass stands: `m` clusters in list `cur`.  Pass p reads state p and
// writes state p + 1, so passes are queued without waiting for their counts:
// a launch covers the clusters the host last knew of, and blocks past the
// current count return.
struct PlocState {
    int m, cur;
    int depth;  // of the whole tree, once m is 1
};
struct PlocBufs {
    float4 *lo[2], *hi[2];  // cluster boxes; lo.w: inner nodes on the longest path down
    int* id[2];             // inner node, or ~leaf
    int* nn;
    unsigned long long* counts;
    PlocState* state;
    BNode* nodes;
    int *iparent, *lparent;
};

// Clusters of a block of the windowed search.  Its 256 threads also find the
// neighbours of the kPlocRadius clusters on each side, which decide whether
// its own are mutual, so that the flags need no launch between.  Blocks of
// 1024 waste less on that (6% against a third) but leave CUs idle: the search
// of 8 passes from 0.5M clusters took 125 us in them, 115 in blocks of 256;
// of the 8 from 55k clusters 88 against 68.
constexpr int kPlocThreads = 256;
constexpr int kPlocOwn = kPlocThreads - 2 * kPlocRadius;
// Blocks whose counts each block of the second half adds up by itself; above,
// a launch between does it once (the build over 2M triangles, 10,300 blocks:
// 1.95 ms against 1.89; the adding grows with the square of the count).
constexpr int kPlocSums = 8192;
// The passes at up to kPlocFull clusters (the top of the tree) search all
// clusters; from kPlocTop down all of them run in one launch of one block.
constexpr int kPlocFull = 1024;
constexpr int kPlocTop = 256;
// From here down one wave does it all (its share of the launch below: 10 us
// less than with every wave to the end; at 64 the same).
constexpr int kPlocWave = 32;
// Windowed passes queued before the host looks at the count.
constexpr int kPlocQueue = 8;

__device__ __forceinline__ int lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Of the block: its clusters that survive the pass (unpaired, or the lower of
// a mutual pair) before this thread's, in the low word, and its pairs before
// this thread's in the high word; `total` the block's sums.
__device__ __forceinline__ unsigned long long ploc_rank(bool survives, bool pair,
                                                        unsigned long long* waves,
                                                        unsigned long long& total)
{
    const unsigned long long ms = __ballot(survives), mp = __ballot(pair);
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0)
        waves[w] = ((unsigned long long)__popcll(mp) << 32) | (unsigned long long)__popcll(ms);
    __syncthreads();
    unsigned long long before = 0;
    total = 0;
    for (int k = 0; k < nw; ++k) {
        const unsigned long long v = waves[k];
        if (k < w) before += v;
        total += v;
    }
    return before + (((unsigned long long)lanes_below(mp) << 32) | (unsigned long long)lanes_below(ms));
}

// The inner node `id` of a mutual pair, and its cluster.
__device__ __forceinline__ void ploc_pair(const PlocBufs& B, int id, float4& l, float4& h, int c0,
                                          const float4& l1, const float4& h1, int c1)
{
    BNode n;
    n.a = make_float4(l.x, l.y, l.z, h.x);
    n.b = make_float4(h.y, h.z, l1.x, l1.y);
    n.c = make_float4(l1.z, h1.x, h1.y, h1.z);
    n.d = make_int4(c0, c1, 0, 0);
    B.nodes[id] = n;
    if (c0 >= 0) B.iparent[c0] = 2 * id + 0;
    else B.lparent[~c0] = 2 * id + 0;
    if (c1 >= 0) B.iparent[c1] = 2 * id + 1;
    else B.lparent[~c1] = 2 * id + 1;
    l = make_float4(fminf(l.x, l1.x), fminf(l.y, l1.y), fminf(l.z, l1.z), fmaxf(l.w, l1.w) + 1.0f);
    h = make_float4(fmaxf(h.x, h1.x), fmaxf(h.y, h1.y), fmaxf(h.z, h1.z), 0.0f);
}

// Windowed pass, first half: every cluster's partner (-1: none) within
// kPlocRadius positions and each block's counts.  The block's window of
// boxes is staged in LDS as (lower, upper) per axis, three 8-byte reads per
// candidate; the reads and the vector ALUs take about as long.
__global__ __launch_bounds__(kPlocThreads) void k_ploc_find(PlocBufs B, int in)
{
    constexpr int T = kPlocThreads, W = T + 2 * kPlocRadius;
    __shared__ float2 sx[W], sy[W], sz[W];
    __shared__ int snn[T];
    __shared__ unsigned long long waves[T / 64];
    const int m = B.state[in].m, cur = B.state[in].cur;
    const int base = blockIdx.x * kPlocOwn;
    if (m <= kPlocFull || base >= m) return;
    const int t = threadIdx.x;
    const float inf = __builtin_huge_valf();
    for (int k = t; k < W; k += T) {
        const int g = base - 2 * kPlocRadius + k;
        // no cluster there: a box whose unions have infinite area
        float4 l = make_float4(-inf, -inf, -inf, 0.0f), h = make_float4(inf, inf, inf, 0.0f);
        if (g >= 0 && g < m) {
            l = B.lo[cur][g];
            h = B.hi[cur][g];
        }
        sx[k] = make_float2(l.x, h.x);
        sy[k] = make_float2(l.y, h.y);
        sz[k] = make_float2(l.z, h.z);
    }
    __syncthreads();
    const int i = base - kPlocRadius + t;
    int bj = -1;
    if (i >= 0 && i < m) {
        const int li = t + kPlocRadius;
        const float2 ax = sx[li], ay = sy[li], az = sz[li];
        // candidates in the order of their tie keys, two distances at a time:
        // the left one first, but the right one at odd distances from an even
        // position; a later one has to be less
        const bool right_first = (i & 1) == 0;
        float best = inf;
        int bo = 0;
#pragma unroll 4
        for (int d = 1; d <= kPlocRadius; d += 2) {
            const float l1 = ploc_area(ax, ay, az, sx[li - d], sy[li - d], sz[li - d]);
            const float r1 = ploc_area(ax, ay, az, sx[li + d], sy[li + d], sz[li + d]);
            const float l2 = ploc_area(ax, ay, az, sx[li - d - 1], sy[li - d - 1], sz[li - d - 1]);
            const float r2 = ploc_area(ax, ay, az, sx[li + d + 1], sy[li + d + 1], sz[li + d + 1]);
            const bool take_r1 = r1 < l1 || (right_first && r1 == l1);
            const float v1 = take_r1 ? r1 : l1;
            if (v1 < best) {
                best = v1;
                bo = take_r1 ? d : -d;
            }
            const bool take_r2 = r2 < l2;
            const float v2 = take_r2 ? r2 : l2;
            if (v2 < best) {
                best = v2;
                bo = take_r2 ? d + 1 : -d - 1;
            }
        }
        bj = i + bo;
        if (bo == 0) {  // no finite area: the clusters that are there, one by one
            unsigned long long key = kNoKey;
            for (int o = max(-kPlocRadius, -i); o <= min(kPlocRadius, m - 1 - i); ++o)
                if (o != 0)
                    key = min_key(key, ploc_key(ploc_area(ax, ay, az, sx[li + o], sy[li + o],
                                                          sz[li + o]), i, o));
            bj = ploc_neighbour(key, i);
        }
    }
    snn[t] = bj;
    __syncthreads();
    const bool own = t >= kPlocRadius && t < kPlocRadius + kPlocOwn && i < m;
    // an own cluster's neighbour is among the block's threads
    const bool mutual = own && snn[t + (bj - i)] == i;
    unsigned long long total;
    ploc_rank(own && !(mutual && bj < i), mutual && i < bj, waves, total);
    if (own) B.nn[i] = mutual ? bj : -1;
    if (t == 0) B.counts[blockIdx.x] = total;
}

// The blocks' counts made exclusive sums, the total behind them.  One block.
__global__ __launch_bounds__(1024) void k_ploc_sums(PlocBufs B, int in)
{
    __shared__ unsigned long long part[1024];
    const int m = B.state[in].m, t = threadIdx.x;
    if (m <= kPlocFull) return;
    const int nb = (m + kPlocOwn - 1) / kPlocOwn, per = (nb + 1023) / 1024;
    const int k0 = min(nb, t * per), k1 = min(nb, k0 + per);
    unsigned long long sum = 0;
    for (int k = k0; k < k1; ++k) sum += B.counts[k];
    part[t] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const unsigned long long v = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    unsigned long long run = part[t] - sum;
    for (int k = k0; k < k1; ++k) {
        const unsigned long long v = B.counts[k];
        B.counts[k] = run;
        run += v;
    }
    if (t == 1023) B.counts[nb] = run;
}

// Windowed pass, second half: compaction and merge.  With M merges in a pass
// over m clusters, the pass's nodes are [m - 1 - M, m - 1).
template <bool SUMMED>
__global__ __launch_bounds__(kPlocOwn) void k_ploc_join(PlocBufs B, int in, int out)
{
    constexpr int T = kPlocOwn;
    __shared__ unsigned long long waves[T / 64], sums[2][T / 64];
    const int m = B.state[in].m, cur = B.state[in].cur;
    const int t = threadIdx.x, base = blockIdx.x * T;
    if (m <= kPlocFull) {
        if (blockIdx.x == 0 && t == 0) B.state[out] = B.state[in];
        return;
    }
    if (base >= m) return;
    // the counts of the blocks before this one, and of all
    const int nb = (m + kPlocOwn - 1) / kPlocOwn;
    unsigned long long before = 0, all = 0;
    if (!SUMMED) {
        for (int k = t; k < nb; k += T) {
            const unsigned long long v = B.counts[k];
            all += v;
            if (k < (int)blockIdx.x) before += v;
        }
    } else if (t == 0) {
        before = B.counts[blockIdx.x];
        all = B.counts[nb];
    }
    for (int d = 32; d > 0; d >>= 1) {
        before += __shfl_xor(before, d);
        all += __shfl_xor(all, d);
    }
    if ((t & 63) == 0) {
        sums[0][t >> 6] = before;
        sums[1][t >> 6] = all;
    }
    const int i = base + t;
    const bool have = i < m;
    const int j = have ? B.nn[i] : -1;
    const bool survives = have && (j < 0 || i < j), pair = survives && j >= 0;
    unsigned long long total;
    unsigned long long ex = ploc_rank(survives, pair, waves, total);
    all = 0;
    for (int k = 0; k < T / 64; ++k) {
        ex += sums[0][k];
        all += sums[1][k];
    }
    if (blockIdx.x == 0 && t == 0) B.state[out] = PlocState{(int)(uint32_t)all, cur ^ 1, 0};
    if (!survives) return;
    float4 l = B.lo[cur][i], h = B.hi[cur][i];
    int id = B.id[cur][i];
    if (pair) {
        const int node = m - 1 - (int)(all >> 32) + (int)(ex >> 32);
        ploc_pair(B, node, l, h, id, B.lo[cur][j], B.hi[cur][j], B.id[cur][j]);
        id = node;
    }
    const int pos = (int)(uint32_t)ex;
    B.lo[cur ^ 1][pos] = l;
    B.hi[cur ^ 1][pos] = h;
    B.id[cur ^ 1][pos] = id;
}

// Key of the least candidate of cluster i among j0, j0 + dj, ... below j1;
// kNoKey when there is none.
__device__ __forceinline__ unsigned long long ploc_least(const float4* slo, const float4* shi, int i,
                                                         int j0, int j1, int dj)
{
    const float4 a = slo[i], b = shi[i];
    const float2 ax = make_float2(a.x, b.x), ay = make_float2(a.y, b.y), az = make_float2(a.z, b.z);
    unsigned long long best = kNoKey;
    // four candidates in flight, without branches: a lone wave waits for
    // every read and every result
    for (; j0 < j1; j0 += 4 * dj) {
        float4 l[4], h[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = min(j0 + u * dj, kPlocFull - 1);
            l[u] = slo[j];
            h[u] = shi[j];
        }
        unsigned long long k[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = j0 + u * dj;
            k[u] = ploc_key(ploc_area(ax, ay, az, make_float2(l[u].x, h[u].x),
                                      make_float2(l[u].y, h[u].y), make_float2(l[u].z, h[u].z)),
                            i, j - i);
            k[u] = j < j1 && j != i ? k[u] : kNoKey;
        }
        best = min_key(best, min_key(min_key(k[0], k[1]), min_key(k[2], k[3])));
    }
    return best;
}

// First half of a pass over kPlocTop < m <= kPlocFull clusters: each block
// takes 16 clusters, each of its 64 sixteenths of a wave one part of the
// candidates.  One thread per cluster in a single block is bound by that
// CU's vector ALUs (46.7 us a pass over the 37 passes of a 0.5M-triangle
// terrain; 5.4 a pass here, 3.8 for its second half).
__global__ __launch_bounds__(1024) void k_ploc_find_all(PlocBufs B, int in)
{
    __shared__ float4 slo[kPlocFull], shi[kPlocFull];
    __shared__ unsigned long long key[16];
    const int m = B.state[in].m, cur = B.state[in].cur;
    const int t = threadIdx.x;
    if (m <= kPlocTop || m > kPlocFull || (int)blockIdx.x * 16 >= m) return;
    if (t < m) {
        slo[t] = B.lo[cur][t];
        shi[t] = B.hi[cur][t];
    }
    if (t < 16) key[t] = kNoKey;
    __syncthreads();
    const int i = blockIdx.x * 16 + (t & 15);
    if (i < m) atomicMin(&key[t & 15], ploc_least(slo, shi, i, t >> 4, m, 64));
    __syncthreads();
    if (t < 16 && i < m) B.nn[i] = ploc_neighbour(key[t], i);
}

// One block over the last clusters.  LAST: all remaining passes, the clusters
// in LDS throughout; each wave a share of the candidates of 64 clusters, and
// from kPlocWave clusters down one wave does it all without barriers, its lanes
// shared out over clusters and candidates.  Otherwise the second half of one
// pass after k_ploc_find_all.  The loops end: a pass over two clusters or
// more merges at least the least pair of all (its candidates are totally
// ordered), and one that did not would stop them.
template <bool LAST>
__global__ __launch_bounds__(1024) void k_ploc_top(PlocBufs B, int in, int out)
{
    __shared__ float4 slo[kPlocFull], shi[kPlocFull];
    __shared__ int sid[kPlocFull], snn[kPlocFull];
    __shared__ unsigned long long key[kPlocFull];
    __shared__ unsigned long long waves[16];
    int m = B.state[in].m;
    const int cur = B.state[in].cur, t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (m > kPlocFull || (!LAST && m <= kPlocTop)) {
        if (t == 0) B.state[out] = B.state[in];
        return;
    }
    if (t < m) {
        slo[t] = B.lo[cur][t];
        shi[t] = B.hi[cur][t];
        sid[t] = B.id[cur][t];
    }
    __syncthreads();
    bool stuck = false;
    while (m > (LAST ? kPlocWave : 1) && !stuck) {
        int j = -1;
        if (LAST) {
            key[t] = kNoKey;
            __syncthreads();
            const int groups = (m + 63) >> 6, parts = 16 / groups;
            const int g = w % groups, p = w / groups, i = g * 64 + lane;
            if (p < parts && i < m) atomicMin(&key[i], ploc_least(slo, shi, i, p, m, parts));
            __syncthreads();
            if (t < m) j = ploc_neighbour(key[t], t);
        } else if (t < m) {
            j = B.nn[t];
        }
        snn[t] = j;
        __syncthreads();
        const bool mutual = t < m && snn[j] == t;
        const bool survives = t < m && !(mutual && j < t), pair = mutual && t < j;
        unsigned long long total;
        const unsigned long long ex = ploc_rank(survives, pair, waves, total);
        float4 l, h;
        int id = 0;
        if (survives) {
            l = slo[t];
            h = shi[t];
            id = sid[t];
            if (pair) {
                const int node = m - 1 - (int)(total >> 32) + (int)(ex >> 32);
                ploc_pair(B, node, l, h, id, slo[j], shi[j], sid[j]);
                id = node;
            }
        }
        __syncthreads();
        const int pos = (int)(uint32_t)ex;
        if (survives) {
            slo[pos] = l;
            shi[pos] = h;
            sid[pos] = id;
        }
        __syncthreads();
        const int m2 = (int)(uint32_t)total;
        stuck = m2 >= m;
        m = m2;
        if (!LAST) break;
    }
    if (!LAST) {
        if (t < m) {
            B.lo[cur ^ 1][t] = slo[t];
            B.hi[cur ^ 1][t] = shi[t];
            B.id[cur ^ 1][t] = sid[t];
        }
        if (t == 0) B.state[out] = PlocState{m, cur ^ 1, 0};
        return;
    }
    if (w != 0) return;
    while (m > 1 && !stuck) {
        const int span = 1 << (32 - __builtin_clz(m - 1));  // lanes per part: m or more
        const int i = lane & (span - 1);
        unsigned long long k = kNoKey;
        if (i < m) k = ploc_least(slo, shi, i, lane / span, m, 64 / span);
        for (int d = span; d < 64; d <<= 1) k = min_key(k, __shfl_xor(k, d));
        const int j = lane < m ? ploc_neighbour(k, lane) : lane;
        const bool mutual = lane < m && __shfl(j, j) == lane;
        const bool survives = lane < m && !(mutual && j < lane), pair = mutual && lane < j;
        const unsigned long long ms = __ballot(survives), mp = __ballot(pair);
        float4 l = slo[lane], h = shi[lane];
        int id = sid[lane];
        if (pair) {
            const int node = m - 1 - (int)__popcll(mp) + lanes_below(mp);
            ploc_pair(B, node, l, h, id, slo[j], shi[j], sid[j]);
            id = node;
        }
        // one wave: its LDS operations complete in order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int pos = lanes_below(ms);
        if (survives) {
            slo[pos] = l;
            shi[pos] = h;
            sid[pos] = id;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        stuck = mp == 0;
        m = (int)__popcll(ms);
    }
    if (t == 0) {
        B.state[out] = PlocState{m, cur ^ 1, (int)slo[0].w};
        B.iparent[0] = -1;  // node 0 is the root
    }
}

// One triangle: a root whose two children are the same leaf; testing it
// twice cannot change a result.
__global__ void k_single(const float4* __restrict__ clo, const float4* __restrict__ chi,
                         BNode* __restrict__ nodes, int* __restrict__ iparent,
                         int* __restrict__ lparent)
{
    const float4 l = clo[0], h = chi[0];
    BNode n;
    n.a = make_float4(l.x, l.y, l.z, h.x);
    n.b = make_float4(h.y, h.z, l.x, l.y);
    n.c = make_float4(l.z, h.x, h.y, h.z);
    n.d = make_int4(~0, ~0, 0, 0);
    nodes[0] = n;
    iparent[0] = -1;
    lparent[0] = 0;
}

// Deepest tree (inner-node levels) a scene may have.
constexpr int kMaxDepth = 4096;

// BVH2 -> BVH4: every even-depth BVH2 node becomes a BVH4 node whose
// children are its grandchildren through inner children, or the child itself
// when that is a leaf (2 to 4 entries).  Per BVH2 node: its BVH4 node's inner
// children (low word) and leaves (high word), or 0 for an odd-depth node.
__global__ void k_count4(const BNode* __restrict__ n2, const int* __restrict__ iparent, int nin,
                         unsigned long long* __restrict__ count)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nin) return;
    int d = 0, p = i;
    while (p != 0 && d <= kMaxDepth) {  // a deeper tree is refused before its counts are used
        p = iparent[p] >> 1;
        ++d;
    }
    unsigned long long c = 0;
    if ((d & 1) == 0) {
        const int4 a = n2[i].d;
        const int kid[2] = {a.x, a.y};
        for (int k = 0; k < 2; ++k) {
            if (kid[k] < 0) {
                c += 1ull << 32;
                continue;
            }
            const int4 g = n2[kid[k]].d;
            c += g.x < 0 ? 1ull << 32 : 1ull;
            c += g.y < 0 ? 1ull << 32 : 1ull;
        }
    }
    count[i] = c;
}

// BVH4 node ids: the inner children of a node are consecutive, after those of
// the nodes before it (base = exclusive sum of the counts); the root is 0.
__global__ void k_number4(const BNode* __restrict__ n2, const unsigned long long* __restrict__ count,
                          const unsigned long long* __restrict__ base, int nin, int* __restrict__ id4)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) id4[0] = 0;
    if (i >= nin || count[i] == 0) return;
    int next = 1 + (int)(uint32_t)base[i];
    const int4 a = n2[i].d;
    const int kid[2] = {a.x, a.y};
    for (int k = 0; k < 2; ++k) {
        if (kid[k] < 0) continue;
        const int4 g = n2[kid[k]].d;
        if (g.x >= 0) id4[g.x] = next++;
        if (g.y >= 0) id4[g.y] = next++;
    }
}

__device__ __forceinline__ void child_box(const BNode& a, int k, float b[6])
{
    if (k == 0) {
        b[0] = a.a.x; b[1] = a.a.y; b[2] = a.a.z; b[3] = a.a.w; b[4] = a.b.x; b[5] = a.b.y;
    } else {
        b[0] = a.b.z; b[1] = a.b.w; b[2] = a.c.x; b[3] = a.c.y; b[4] = a.c.z; b[5] = a.c.w;
    }
}

// FP16 x rounded towards -inf or +inf of the double v, never subnormal (so
// no flush of subnormals anywhere can move a plane inwards).  |v| <= 65504.
__host__ __device__ uint32_t half_outward(double v, bool up)
{
    const _Float16 h0 = (_Float16)(float)v;  // nearest (twice), then stepped
    uint16_t u = __builtin_bit_cast(uint16_t, h0);
    for (int i = 0; i < 4; ++i) {
        const double x = (double)(float)__builtin_bit_cast(_Float16, u);
        if (up ? x >= v : x <= v) break;
        // next half towards +inf (up) or -inf
        const bool neg = (u & 0x8000u) != 0;
        if ((u & 0x7FFFu) == 0) u = up ? 0x0001u : 0x8001u;
        else u = (uint16_t)(neg == up ? u - 1 : u + 1);
    }
    if ((u & 0x7C00u) == 0 && (u & 0x03FFu) != 0) {
        const bool neg = (u & 0x8000u) != 0;
        u = up ? (neg ? 0x0000u : 0x0400u) : (neg ? 0x8400u : 0x0000u);
    }
    return u;
}

// Writes the BVH4 nodes (Node4) and their leaf triangles.  Boxes are widened
// by `margin` (box_margin), taken relative to the node's origin (FP16) in
// double, where the differences are exact, and rounded outwards: offsets of at
// most 2^15 units (the scene's largest coordinate is at most 2^14).
__global__ void k_collapse(const BNode* __restrict__ n2, const unsigned long long* __restrict__ count,
                           const unsigned long long* __restrict__ base, const int* __restrict__ id4,
                           int nin, int ntris, float margin, double per_unit,
                           const uint32_t* __restrict__ order, const float4* __restrict__ tri_raw,
                           Node4* __restrict__ n4, float4* __restrict__ tris)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nin || count[i] == 0) return;
    float bi[4][6], bl[4][6], b[6];
    int leaf[4], ni = 0, nl = 0;
    const BNode a = n2[i];
    for (int k = 0; k < 2; ++k) {
        const int c = k == 0 ? a.d.x : a.d.y;
        if (c < 0) {
            child_box(a, k, b);
            for (int t = 0; t < 6; ++t) bl[nl][t] = b[t];
            leaf[nl++] = ~c;
            continue;
        }
        const BNode g = n2[c];
        for (int q = 0; q < 2; ++q) {
            const int gc = q == 0 ? g.d.x : g.d.y;
            child_box(g, q, b);
            if (gc < 0) {
                for (int t = 0; t < 6; ++t) bl[nl][t] = b[t];
                leaf[nl++] = ~gc;
            } else {
                for (int t = 0; t < 6; ++t) bi[ni][t] = b[t];
                ++ni;
            }
        }
    }
    if (ntris == 1) nl = 1;  // the root's two children are the same leaf
    const int first = (int)(base[i] >> 32);
    for (int k = 0; k < nl; ++k) {
        const uint32_t p = order[leaf[k]];
        float4* out = tris + (size_t)(first + k) * (kTriWords / 4);
        const float4 u = tri_raw[3 * (size_t)p], v = tri_raw[3 * (size_t)p + 1], w = tri_raw[3 * (size_t)p + 2];
        out[0] = make_float4(u.x, u.y, u.z, u.x);
        out[1] = make_float4(u.y, v.x, v.y, v.z);
        out[2] = make_float4(v.x, v.y, w.x, w.y);
        out[3] = make_float4(w.z, w.x, w.y, u.w);
        for (int t = 0; t < 6; ++t) bi[ni + k][t] = bl[k][t];
    }
    const int used = ni + nl;
    uint32_t org[3], lo[3][4], hi[3][4];
    for (int x = 0; x < 3; ++x) {
        float blo = bi[0][x], bhi = bi[0][3 + x];
        for (int k = 1; k < used; ++k) {
            blo = fminf(blo, bi[k][x]);
            bhi = fmaxf(bhi, bi[k][3 + x]);
        }
        // origin: the node's centre or a child's, whichever lets the rounding
        // (about 2^-11 of a plane's offset) thicken the children least in
        // proportion.  Flat children decide: a wall's box must stay thinner
        // than the offset a shadow ray leaves it with, or every such ray
        // tests the wall again (centres alone: 19% more triangle tests in a
        // room of boxes)
        double best = 0.0, bo = 0.0;
        for (int t = -1; t < used; ++t) {
            const double at = t < 0 ? 0.5 * ((double)blo + (double)bhi)
                                    : 0.5 * ((double)bi[t][x] + (double)bi[t][3 + x]);
            _Float16 h = (_Float16)(float)(at * per_unit);
            uint32_t u = __builtin_bit_cast(uint16_t, h);
            if ((u & 0x7C00u) == 0) u = 0;  // no subnormal origin
            const double o = (double)(float)__builtin_bit_cast(_Float16, (uint16_t)u) / per_unit;
            double cost = 0.0;
            for (int k = 0; k < used; ++k) {
                const double l = (double)bi[k][x] - margin, g = (double)bi[k][3 + x] + margin;
                cost += (fabs(l - o) + fabs(g - o)) / fmax(g - l, 1e-300);
            }
            if (t < 0 || cost < best) {
                best = cost;
                bo = o * per_unit;
                org[x] = u;
            }
        }
        for (int k = 0; k < 4; ++k) {
            // unused slots: +inf planes, which no ray hits
            lo[x][k] = k < used ? half_outward(((double)bi[k][x] - margin) * per_unit - bo, false) : 0x7C00u;
            hi[x][k] = k < used ? half_outward(((double)bi[k][3 + x] + margin) * per_unit - bo, true) : 0x7C00u;
        }
    }
    Node4 n;
    n.oxy = org[0] | org[1] << 16;
    n.ozn = org[2] | ((1u << used) - (1u << ni)) << 16 | (uint32_t)ni << 20;
    n.inner = 1 + (int)(uint32_t)base[i];
    n.leaf = first - ni;
    for (int p = 0; p < 2; ++p) {
        n.lox[p] = lo[0][2 * p] | lo[0][2 * p + 1] << 16;
        n.loy[p] = lo[1][2 * p] | lo[1][2 * p + 1] << 16;
        n.loz[p] = lo[2][2 * p] | lo[2][2 * p + 1] << 16;
        n.hix[p] = hi[0][2 * p] | hi[0][2 * p + 1] << 16;
        n.hiy[p] = hi[1][2 * p] | hi[1][2 * p + 1] << 16;
        n.hiz[p] = hi[2][2 * p] | hi[2][2 * p + 1] << 16;
    }
    n4[id4[i]] = n;
}

inline int nblk(int n, int b = 256) { return (n + b - 1) / b; }

// Refuses geometry by its first bad index, else by its first bad coordinate
// (~0: none).
void require_good(unsigned long long bad_index, unsigned long long bad_coord)
{
    VLB_REQUIRE(bad_index == ~0ull, VLB_ERR_INVALID, "index out of range at " + std::to_string(bad_index));
    // the BVH4 node grids need finite boxes of bounded magnitude
    VLB_REQUIRE(bad_coord == ~0ull, VLB_ERR_INVALID,
                "vertex coordinate not finite or beyond 2^100 at " + std::to_string(bad_coord));
}

// k_check on the host.
void require_good_host(const uint32_t* idx, unsigned long long nidx, uint32_t nverts, const float* xyz,
                       unsigned long long ncoords)
{
    unsigned long long bi = 0, bc = 0;
    while (bi < nidx && idx[bi] < nverts) ++bi;
    while (bc < ncoords && fabsf(xyz[bc]) <= 0x1p100f) ++bc;
    require_good(bi < nidx ? bi : ~0ull, bc < ncoords ? bc : ~0ull);
}

struct Event {
    hipEvent_t e = nullptr;
    Event() { VLB_HIP(hipEventCreate(&e)); }
    Event(const Event&) = delete;
    Event& operator=(const Event&) = delete;
    ~Event() { (void)hipEventDestroy(e); }
};

}  // namespace

void build_scene_bvh(Context& ctx, Scene& s, const float* xyz, uint32_t nverts,
                     const uint32_t* idx, uint32_t ntris, const float* normals,
                     const float* albedo)
{
    hipStream_t st = ctx.stream;
    const int n = (int)ntris;
    s.ntris = n;
    if (n == 0) {
        s.nnodes = 0;
        s.depth = 0;
        return;
    }
    // uploads
    const unsigned long long nidx = (unsigned long long)n * 3, ncoords = (unsigned long long)nverts * 3;
    DevBuf d_xyz, d_idx, d_nrm, d_alb, d_bad;
    unsigned long long bad[2] = {~0ull, ~0ull};
    try {
        d_xyz = dev_alloc(ctx, ncoords * sizeof(float));
        d_idx = dev_alloc(ctx, nidx * sizeof(uint32_t));
        d_bad = dev_alloc(ctx, sizeof bad);
    } catch (const Error&) {
        // bad geometry is refused as such also where it does not fit
        require_good_host(idx, nidx, nverts, xyz, ncoords);
        throw;
    }
    VLB_HIP(hipMemcpyAsync(d_xyz.p, xyz, d_xyz.bytes, hipMemcpyHostToDevice, st));
    VLB_HIP(hipMemcpyAsync(d_idx.p, idx, d_idx.bytes, hipMemcpyHostToDevice, st));
    VLB_HIP(hipMemcpyAsync(d_bad.p, bad, sizeof bad, hipMemcpyHostToDevice, st));
    k_check<<<std::min(2048, nblk(n)), 256, 0, st>>>(d_idx.as<uint32_t>(), nidx, nverts, d_xyz.as<float>(),
                                                    ncoords, d_bad.as<unsigned long long>());
    VLB_HIP(hipGetLastError());
    VLB_HIP(hipMemcpyAsync(bad, d_bad.p, sizeof bad, hipMemcpyDeviceToHost, st));
    VLB_HIP(hipStreamSynchronize(st));
    require_good(bad[0], bad[1]);
    if (normals) {
        d_nrm = dev_alloc(ctx, (size_t)nverts * 3 * sizeof(float));
        VLB_HIP(hipMemcpyAsync(d_nrm.p, normals, d_nrm.bytes, hipMemcpyHostToDevice, st));
    }
    if (albedo) {
        d_alb = dev_alloc(ctx, (size_t)n * 3 * sizeof(float));
        VLB_HIP(hipMemcpyAsync(d_alb.p, albedo, d_alb.bytes, hipMemcpyHostToDevice, st));
    }
    const Event e0, e1;
    VLB_HIP(hipEventRecord(e0.e, st));
    DevBuf tri_raw = dev_alloc(ctx, (size_t)n * 3 * sizeof(float4));
    DevBuf lo = dev_alloc(ctx, (size_t)n * sizeof(float4));
    DevBuf hi = dev_alloc(ctx, (size_t)n * sizeof(float4));
    DevBuf cen = dev_alloc(ctx, (size_t)n * sizeof(float4));
    s.shade = dev_alloc(ctx, (size_t)n * 3 * sizeof(float4));
    k_gather<<<nblk(n), 256, 0, st>>>(d_xyz.as<float>(), d_idx.as<uint32_t>(), d_nrm.as<float>(),
                                      d_alb.as<float>(), n, (int)nverts, tri_raw.as<float4>(),
                                      lo.as<float4>(), hi.as<float4>(), cen.as<float4>(),
                                      s.shade.as<float4>());
    VLB_HIP(hipGetLastError());
    const int nb = std::min(1024, nblk(n));
    DevBuf part = dev_alloc(ctx, (size_t)nb * 13 * sizeof(float));
    DevBuf bnd = dev_alloc(ctx, 16 * sizeof(float));
    k_bounds1<<<nb, 256, 0, st>>>(lo.as<float4>(), hi.as<float4>(), cen.as<float4>(), n,
                                  part.as<float>());
    k_bounds2<<<1, 256, 0, st>>>(part.as<float>(), nb, bnd.as<float>());
    VLB_HIP(hipGetLastError());
    // Morton codes + sort
    DevBuf keys = dev_alloc(ctx, (size_t)n * sizeof(uint32_t));
    DevBuf vals = dev_alloc(ctx, (size_t)n * sizeof(uint32_t));
    DevBuf keys2 = dev_alloc(ctx, (size_t)n * sizeof(uint32_t));
    s.leaf_prims = dev_alloc(ctx, (size_t)n * sizeof(uint32_t));
    k_morton<<<nblk(n), 256, 0, st>>>(cen.as<float4>(), n, bnd.as<float>(), keys.as<uint32_t>(),
                                      vals.as<uint32_t>());
    VLB_HIP(hipGetLastError());
    size_t tmp_bytes = 0;
    VLB_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys.as<uint32_t>(), keys2.as<uint32_t>(),
                                      vals.as<uint32_t>(), s.leaf_prims.as<uint32_t>(), (size_t)n, 0, 30, st));
    DevBuf tmp = dev_alloc(ctx, tmp_bytes > 0 ? tmp_bytes : 16);
    VLB_HIP(rocprim::radix_sort_pairs(tmp.p, tmp_bytes, keys.as<uint32_t>(), keys2.as<uint32_t>(),
                                      vals.as<uint32_t>(), s.leaf_prims.as<uint32_t>(), (size_t)n, 0, 30, st));
    // hierarchy (PLOC)
    const int nin = n > 1 ? n - 1 : 1;
    s.nodes = dev_alloc(ctx, (size_t)nin * sizeof(BNode));
    s.tris = dev_alloc(ctx, (size_t)n * kTriWords * sizeof(float));
    DevBuf iparent = dev_alloc(ctx, (size_t)nin * sizeof(int));
    DevBuf lparent = dev_alloc(ctx, (size_t)n * sizeof(int));
    DevBuf clo[2], chi[2], cid[2];
    for (int k = 0; k < 2; ++k) {
        clo[k] = dev_alloc(ctx, (size_t)n * sizeof(float4));
        chi[k] = dev_alloc(ctx, (size_t)n * sizeof(float4));
        cid[k] = dev_alloc(ctx, (size_t)n * sizeof(int));
    }
    k_leaves<<<nblk(n), 256, 0, st>>>(s.leaf_prims.as<uint32_t>(), n, lo.as<float4>(), hi.as<float4>(),
                                      clo[0].as<float4>(), chi[0].as<float4>(), cid[0].as<int>());
    VLB_HIP(hipGetLastError());
    DevBuf nn, counts, state;
    PlocState left{1, 0, 1};
    if (n == 1) {
        k_single<<<1, 1, 0, st>>>(clo[0].as<float4>(), chi[0].as<float4>(), s.nodes.as<BNode>(),
                                  iparent.as<int>(), lparent.as<int>());
    } else {
        nn = dev_alloc(ctx, (size_t)n * sizeof(int));
        counts = dev_alloc(ctx, (size_t)(n / kPlocOwn + 2) * sizeof(unsigned long long));
        state = dev_alloc(ctx, (kPlocQueue + 1) * sizeof(PlocState));
        PlocBufs B;
        for (int k = 0; k < 2; ++k) {
            B.lo[k] = clo[k].as<float4>();
            B.hi[k] = chi[k].as<float4>();
            B.id[k] = cid[k].as<int>();
        }
        B.nn = nn.as<int>();
        B.counts = counts.as<unsigned long long>();
        B.state = state.as<PlocState>();
        B.nodes = s.nodes.as<BNode>();
        B.iparent = iparent.as<int>();
        B.lparent = lparent.as<int>();
        int in = 0;
        left = PlocState{n, 0, 0};
        VLB_HIP(hipMemcpyAsync(&B.state[0], &left, sizeof left, hipMemcpyHostToDevice, st));
        while (left.m > kPlocFull) {
            const int before = left.m;
            const int nb = (before + kPlocOwn - 1) / kPlocOwn;
            for (int p = 0; p < kPlocQueue; ++p, in = p) {
                k_ploc_find<<<nb, kPlocThreads, 0, st>>>(B, in);
                if (nb > kPlocSums) {
                    k_ploc_sums<<<1, 1024, 0, st>>>(B, in);
                    k_ploc_join<true><<<nb, kPlocOwn, 0, st>>>(B, in, p + 1);
                } else {
                    k_ploc_join<false><<<nb, kPlocOwn, 0, st>>>(B, in, p + 1);
                }
            }
            VLB_HIP(hipGetLastError());
            VLB_HIP(hipMemcpyAsync(&left, &B.state[kPlocQueue], sizeof left, hipMemcpyDeviceToHost, st));
            VLB_HIP(hipStreamSynchronize(st));
            // a pass over several clusters merges at least one pair
            VLB_REQUIRE(left.m >= 1 && left.m < before, VLB_ERR_DEVICE, "PLOC build made no progress");
        }
        if (left.m > kPlocTop)
            for (int p = 0; p < kPlocQueue; ++p, in = p) {
                k_ploc_find_all<<<(left.m + 15) / 16, 1024, 0, st>>>(B, in);
                k_ploc_top<false><<<1, 1024, 0, st>>>(B, in, p + 1);
            }
        const int out = in == 0 ? 1 : 0;
        k_ploc_top<true><<<1, 1024, 0, st>>>(B, in, out);
        VLB_HIP(hipGetLastError());
        VLB_HIP(hipMemcpyAsync(&left, &B.state[out], sizeof left, hipMemcpyDeviceToHost, st));
    }
    VLB_HIP(hipGetLastError());
    // BVH4: even-depth BVH2 nodes; an exclusive scan of their child counts
    // places each one's inner children and leaves
    DevBuf count = dev_alloc(ctx, (size_t)nin * sizeof(unsigned long long));
    DevBuf base = dev_alloc(ctx, (size_t)nin * sizeof(unsigned long long));
    DevBuf id4 = dev_alloc(ctx, (size_t)nin * sizeof(int));
    k_count4<<<nblk(nin), 256, 0, st>>>(s.nodes.as<BNode>(), iparent.as<int>(), nin,
                                        count.as<unsigned long long>());
    VLB_HIP(hipGetLastError());
    size_t scan_bytes = 0;
    VLB_HIP(rocprim::exclusive_scan(nullptr, scan_bytes, count.as<unsigned long long>(),
                                    base.as<unsigned long long>(), 0ull, (size_t)nin,
                                    rocprim::plus<unsigned long long>(), st));
    DevBuf scan_tmp = dev_alloc(ctx, scan_bytes > 0 ? scan_bytes : 16);
    VLB_HIP(rocprim::exclusive_scan(scan_tmp.p, scan_bytes, count.as<unsigned long long>(),
                                    base.as<unsigned long long>(), 0ull, (size_t)nin,
                                    rocprim::plus<unsigned long long>(), st));
    unsigned long long last[2] = {0, 0};
    float hb[16];
    VLB_HIP(hipMemcpyAsync(&last[0], base.as<unsigned long long>() + (nin - 1), sizeof last[0],
                           hipMemcpyDeviceToHost, st));
    VLB_HIP(hipMemcpyAsync(&last[1], count.as<unsigned long long>() + (nin - 1), sizeof last[1],
                           hipMemcpyDeviceToHost, st));
    VLB_HIP(hipMemcpyAsync(hb, bnd.p, 13 * sizeof(float), hipMemcpyDeviceToHost, st));
    VLB_HIP(hipStreamSynchronize(st));
    VLB_REQUIRE(left.m == 1, VLB_ERR_DEVICE, "PLOC build made no progress");
    // before anything is numbered: k_count4 tells even from odd depths only
    // down to kMaxDepth, so a deeper tree's counts place leaves and nodes past
    // their arrays (10,000 concentric triangles make a tree of depth 9,999)
    VLB_REQUIRE(left.depth <= kMaxDepth, VLB_ERR_INVALID, "BVH build produced a malformed tree");
    VLB_REQUIRE((int)((last[0] + last[1]) >> 32) == (n == 1 ? 2 : n), VLB_ERR_DEVICE,
                "BVH build lost a leaf");
    const int n4 = 1 + (int)(uint32_t)(last[0] + last[1]);
    // node unit: the power of two that brings the largest coordinate to
    // [2^13, 2^14) units, so that offsets stay within FP16's range
    s.maxabs = hb[12];
    int e = 0;
    (void)frexpf(s.maxabs, &e);  // maxabs < 2^e; 0 gives e = 0
    s.unit = ldexpf(1.0f, std::max(e - 14, -100));
    s.nodes4 = dev_alloc(ctx, (size_t)n4 * sizeof(Node4));
    k_number4<<<nblk(nin), 256, 0, st>>>(s.nodes.as<BNode>(), count.as<unsigned long long>(),
                                         base.as<unsigned long long>(), nin, id4.as<int>());
    VLB_HIP(hipGetLastError());
    k_collapse<<<nblk(nin), 256, 0, st>>>(s.nodes.as<BNode>(), count.as<unsigned long long>(),
                                          base.as<unsigned long long>(), id4.as<int>(), nin, n,
                                          box_margin(s.maxabs), 1.0 / (double)s.unit,
                                          s.leaf_prims.as<uint32_t>(), tri_raw.as<float4>(),
                                          s.nodes4.as<Node4>(), s.tris.as<float4>());
    VLB_HIP(hipGetLastError());
    VLB_HIP(hipEventRecord(e1.e, st));
    VLB_HIP(hipStreamSynchronize(st));
    float ms = 0.0f;
    VLB_HIP(hipEventElapsedTime(&ms, e0.e, e1.e));
    s.build_ms = ms;
    s.nnodes = nin;
    s.nnodes4 = n4;
    s.depth = (uint32_t)left.depth;
    for (int a = 0; a < 3; ++a) {
        s.bmin[a] = hb[6 + a];
        s.bmax[a] = hb[9 + a];
    }
}

}  // namespace vlb
