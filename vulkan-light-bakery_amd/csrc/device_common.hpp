// device_common.hpp -- device-side building blocks of the probe baker:
// BVH node layout, watertight ray/triangle test, conservative slab test,
// LDS-stack traversal (closest hit and shadow query), sky and shading.
//
// Every translation unit that includes this file is compiled with
// -ffp-contract=off: the intersection, hit-point, normal and shadow-ray
// arithmetic below is a fixed sequence of correctly rounded IEEE operations
// (HIP's default f32 division and sqrt are correctly rounded), so hit ids and
// visibility are bit-identical to a C restatement that does the same
// operations in the same order.  Only the slab test uses explicit fmaf: it
// decides which nodes are visited, never which triangle wins.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/vlb_bake.h"
#include "probe_grid.hpp"

namespace vlb {

// ---------------------------------------------------------------- layout
// One BVH2 inner node = 64 bytes: the boxes of both children and their ids.
// child >= 0: inner node index; child < 0: leaf, ~child = leaf-order
// triangle index.  The root is node 0.
struct __align__(16) BNode {
    float4 a;  // lo0.x lo0.y lo0.z hi0.x
    float4 b;  // hi0.y hi0.z lo1.x lo1.y
    float4 c;  // lo1.z hi1.x hi1.y hi1.z
    int4   d;  // child0 child1 - -
};

// The traversal kernels walk a 4-wide BVH collapsed from it (half the
// dependent node fetches of the BVH2 per ray).  Node4 is 64 bytes, four
// 16-byte loads, because a visit's cost is its loads as much as its
// arithmetic (three more loads per divergent visit cost 18% on an 11k-triangle
// room and 41% on a 1.15M-triangle terrain):
//  - the children's boxes as FP16 offsets from the node's own origin, in
//    units of the scene's power-of-two scale.  v_fma_mix_f32 reads an FP16
//    operand inside an FP32 FMA, so a plane's ray parameter
//    t = fma(offset, inv, fma(origin, inv, -o * inv)) costs no decode.  The
//    offsets are rounded outwards from boxes already widened by the margin of
//    the slab test, so a decoded box contains its child: boxes decide which
//    nodes are visited, never which triangle is hit.
//  - children are consecutive: the inner ones first (nodes inner, inner + 1,
//    ...), then the leaves (triangle leaf + k for child k); unused slots have
//    all-+inf boxes, which no ray hits.
struct __align__(64) Node4 {
    uint32_t oxy;      // origin x, y (FP16, low half first)
    uint32_t ozn;      // origin z (FP16), leaf slots (4 bits) << 16, number
                       // of inner children << 20
    int32_t  inner;    // id of the first inner child
    int32_t  leaf;     // leaf-order triangle of child k: leaf + k
    uint32_t lox[2], loy[2], loz[2];  // FP16 offsets: children 0, 1 | 2, 3
    uint32_t hix[2], hiy[2], hiz[2];
};

// Stack entries a BVH4 traversal can hold for a BVH2 of `depth` inner
// levels: at most 3 pushes per BVH4 level, ceil(depth / 2) levels.
__host__ __device__ inline uint32_t stack_bound(uint32_t depth)
{
    return 3u * ((depth + 1u) / 2u) + 1u;
}

// Leaf-order triangle = 16 words, one 64-byte line: per vertex x y z x y, so
// that the three coordinates in any cyclic order are consecutive (the
// watertight test reads them in its ray's order with one load per vertex,
// instead of reordering them with 24 selects), and the prim id.
constexpr int kTriWords = 16;
constexpr int kTriPrim = 15;

// Shading record per prim id = 3 x float4: (n0, albedo.r) (n1, .g) (n2, .b).

struct SceneView {
    const Node4*  nodes;
    const float*  tris;       // kTriWords per leaf
    const float4* shade;
    int           ntris;
    float         maxabs;  // max |coordinate| of the scene's vertices
    float         unit;    // power of two: world length of a node's unit
};

struct ShadeParams {
    int32_t      mode;         // VLB_SHADE_*
    int32_t      nlights;
    float        shadow_bias;  // LAMBERT
    float        t_max;        // shadow extent of directional lights
    vlb_light    lights[VLB_MAX_LIGHTS];
    vlb_sky      sky;
    vlb_ref_shading ref;
    // LAMBERT multi-bounce: a baked grid whose looked-up value at the hit
    // (times scale) adds albedo x that value; ind.coeffs null: direct only
    ProbeGridView ind;
};

// Stack entries kept in LDS per lane: 16 for the fused and single-query
// kernels, 12 for the wavefront kernels, whose leaf queues take another 8 KB
// per workgroup (12 + 8 entries x 256 lanes x 4 B = 20 KB lets them run 7
// waves/SIMD: the trace stage of a 1.15M-triangle terrain bake, 16,384
// probes x 16,384 rays, 2.5% faster; the fused kernels measured 1% slower at
// 12 on an 11k-triangle room bake).  Spill areas are sized for the smaller
// depth.
constexpr int kLdsDepth = 16;
constexpr int kLdsDepthWave = 12;
constexpr int kLdsDepthMin = kLdsDepthWave < kLdsDepth ? kLdsDepthWave : kLdsDepth;
// Work counters (persistent kernels' fetch positions) sit 128 bytes apart,
// one per cache line: device-scope atomics on one line serialise.
constexpr int kCtrStride = 16;

// Work of the fused kernels: 32 64-aligned ranges of the items, range
// 4x + w owned by wave w of the workgroups on XCD x (= blockIdx % 8).  A wave
// takes 64 items at a time from its own range's counter, then from its XCD's
// other ranges, then from the other XCDs'.  (nitems is a multiple of 512: what
// is taken is whole.)  The ranges known to be used up are kept per workgroup,
// in LDS, so that its four waves look for the last work together.  Each wave
// asking all 32 counters one after the other ended a full launch with 260,000
// atomics on 32 addresses: 2048 probes x 4096 rays of the 11k-triangle room
// 0.92 ms per bake against 0.87.  Sharing what is known by more than a
// workgroup costs more than it saves (flags per XCD in memory: 1.0 ms;
// accesses to one line from all waves serialise), and looking only into some
// of the other XCDs' ranges leaves the launch unbalanced (terrain +3%).  The
// multi-job kernel took it over together with arguments read per set of rays
// (kernel_args): 24 jobs over three scenes 69.5 ms instead of 69.9, a burst of
// 20 requests 41.2 instead of 41.5.
struct WorkRanges {
    unsigned long long* ctr;
    size_t nitems, per;
    unsigned* used;  // in LDS, 0 at first
    __device__ __forceinline__ WorkRanges(unsigned long long* c, size_t n, unsigned* lds)
        : ctr(c), nitems(n), per(((n + 31) / 32 + 63) / 64 * 64), used(lds)
    {
        if (threadIdx.x == 0) *lds = 0u;
        __syncthreads();
    }
    __device__ __forceinline__ static int own()
    {
        return __builtin_amdgcn_readfirstlane((blockIdx.x & 7) * 4 + (threadIdx.x >> 6));
    }
    // First of the next 64 items (wave-uniform), or ~0.
    __device__ __forceinline__ unsigned long long take(int own) const
    {
        // a copy of the lane that nothing is computed from before the caller's
        // loop and held across its traversals
        int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        __asm__ __volatile__("" : "+v"(lane));
        for (;;) {
            const unsigned u = (unsigned)__builtin_amdgcn_readfirstlane(
                (int)__hip_atomic_load(used, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
            if (u == ~0u) return ~0ull;
            // the first open range: by XCD from the own one on, by wave from the own one on
            const unsigned r = __builtin_rotateright32(~u, (unsigned)own & ~3u);
            const int g = __builtin_ctz(r) & ~3;
            const unsigned nib = (r >> g) & 15u;
            const int w = __builtin_ctz((nib | (nib << 4)) >> (own & 3));
            const int v = ((own & ~3) + g + ((own + w) & 3)) & 31;
            const size_t beg = (size_t)v * per, end = min(nitems, beg + per);
            unsigned long long b = 0;
            if (lane == 0) b = atomicAdd(&ctr[v * kCtrStride], 64ull);
            // every lane is active here, so the first active lane is lane 0
            b = ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(b >> 32)) << 32) |
                (unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)b);
            if (beg + b < end) return beg + b;
            if (lane == 0) atomicOr(used, 1u << v);
        }
    }
};

// ---------------------------------------------------------------- helpers
// The running kernel's first argument (constant memory).  Called inside a
// persistent kernel's loop, it makes the compiler read the arguments again
// for each set of rays, where they are used; named directly they are loaded
// once before the loop and held in scalar registers, more than 8 waves/SIMD
// leave, which spill into vector registers, which spill into scratch.
template <class T>
__device__ __forceinline__ const T& kernel_args()
{
    typedef const T __attribute__((address_space(4)))* P;
    P p = (P)__builtin_amdgcn_kernarg_segment_ptr();
    __asm__ __volatile__("" : "+s"(p));
    return *(const T*)p;
}

__device__ __forceinline__ float dot3(const float3& a, const float3& b)
{
    return a.x * b.x + a.y * b.y + a.z * b.z;
}

// -------------------------------------------------------- watertight test
// Woop, Benthin, Wald, "Watertight Ray/Triangle Intersection", JCGT 2(1),
// 2013: shear the triangle into ray space along the dominant axis kz, take
// the 2D edge functions U, V, W (recomputed in double when one is zero), and
// accept when they share a sign.  The paper also exchanges kx and ky where
// d[kz] < 0, to keep the winding; without culling that only negates U, V, W,
// their sum and T together, exactly, so it is left out.
struct WtRay {
    float3   o;    // origin (kx, ky, kz)
    float    Sx, Sy, Sz;
    uint32_t rot;  // byte offset of (kx, ky, kz) in a vertex's x y z x y
};

__device__ __forceinline__ WtRay wt_setup(const float3& o, const float3& d)
{
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    const bool zx = ax > ay && ax > az;             // kz = x: order y z x
    const bool zy = !(ax > ay) && ay > az;          // kz = y: order z x y
    const float3 pd = make_float3(zx ? d.y : (zy ? d.z : d.x), zx ? d.z : (zy ? d.x : d.y),
                                  zx ? d.x : (zy ? d.y : d.z));
    WtRay w;
    w.o = make_float3(zx ? o.y : (zy ? o.z : o.x), zx ? o.z : (zy ? o.x : o.y),
                      zx ? o.x : (zy ? o.y : o.z));
    w.rot = zx ? 4u : (zy ? 8u : 0u);
    w.Sx = pd.x / pd.z;
    w.Sy = pd.y / pd.z;
    w.Sz = 1.0f / pd.z;
    return w;
}

// A ray with a direction component below 2^-16 of its largest (box_agrees).
__device__ __forceinline__ bool wt_thin(const WtRay& w)
{
    return fminf(fabsf(w.Sx), fabsf(w.Sy)) < 0x1p-16f;
}

// Edge-function part of the test.  On acceptance returns t (correctly
// rounded T / det) with the numerators V, W and det kept for the
// barycentrics, which are divided out once for the final hit only.
struct WtHit {
    float t, V, W, det;
};

// v0, v1, v2: the vertices in the ray's coordinate order.
__device__ __forceinline__ bool wt_test(const WtRay& w, const float3& v0, const float3& v1,
                                        const float3& v2, float tmin, float tmax, WtHit& h)
{
    const float3 A = make_float3(v0.x - w.o.x, v0.y - w.o.y, v0.z - w.o.z);
    const float3 B = make_float3(v1.x - w.o.x, v1.y - w.o.y, v1.z - w.o.z);
    const float3 C = make_float3(v2.x - w.o.x, v2.y - w.o.y, v2.z - w.o.z);
    const float Ax = A.x - w.Sx * A.z;
    const float Ay = A.y - w.Sy * A.z;
    const float Bx = B.x - w.Sx * B.z;
    const float By = B.y - w.Sy * B.z;
    const float Cx = C.x - w.Sx * C.z;
    const float Cy = C.y - w.Sy * C.z;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        double CxBy = (double)Cx * (double)By;
        double CyBx = (double)Cy * (double)Bx;
        U = (float)(CxBy - CyBx);
        double AxCy = (double)Ax * (double)Cy;
        double AyCx = (double)Ay * (double)Cx;
        V = (float)(AxCy - AyCx);
        double BxAy = (double)Bx * (double)Ay;
        double ByAx = (double)By * (double)Ax;
        W = (float)(BxAy - ByAx);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float Az = w.Sz * A.z;
    const float Bz = w.Sz * B.z;
    const float Cz = w.Sz * C.z;
    const float T = U * Az + V * Bz + W * Cz;
    const float t = T / det;
    if (!(t >= tmin && t <= tmax)) return false;
    h.t = t;
    h.V = V;
    h.W = W;
    h.det = det;
    return true;
}

// -------------------------------------------------------------- slab test
// Conservative: a node's planes are stored widened by box_margin (128 float
// roundings of the scene's largest coordinate), which covers the rounding of
// the plane parameters, of the watertight test and of its t for rays whose
// origin lies within several scene sizes; apad is the same margin of the
// origin's own magnitude for rays that start farther away, as a length in t
// (directions need not be unit vectors).  It widens the exit side, tbest
// included, so that neither a triangle at tmin nor one at the distance of the
// best so far is lost with its box.  Margins cost node visits, never change a
// result.  (Restated on the CPU over 1,752 triangles, origins at 1 to 30,000
// scene sizes, directions of 1e-15 to 1e6: no accepted triangle's box is
// culled; with apad as if directions were unit vectors and tbest not widened
// up to 2.6% of the hits were, and half of those at tbest.)
struct SlabRay {
    float3 inv;         // node unit / direction
    float3 oinv;        // origin / direction
    float  apad;
    bool   nx, ny, nz;  // direction component negative: hi is the near plane
};

__host__ __device__ __forceinline__ float box_margin(float maxabs)
{
    return maxabs * (64.0f * 1.1920929e-7f);
}

// Length in t of one world length along the direction's largest component, as
// a power of two (rounded down, the margin has room), not below 1.
__device__ __forceinline__ float wt_scale(const WtRay& w)
{
    return fmaxf(1.0f, fminf(0x1p100f, __uint_as_float(__float_as_uint(w.Sz) & 0x7F800000u)));
}

__device__ __forceinline__ SlabRay slab_setup(const float3& o, const float3& d, const WtRay& w, float maxabs,
                                              float unit)
{
    SlabRay s;
    const float m = fmaxf(maxabs, fmaxf(fabsf(o.x), fmaxf(fabsf(o.y), fabsf(o.z))));
    // a component this small against the largest moves the ray by less than
    // the margin over the whole scene; the second bound keeps unit / d and
    // o / d finite, the third a zero direction from meeting every box
    const float dm = fmaxf(fabsf(d.x), fmaxf(fabsf(d.y), fabsf(d.z)));
    const float dmin = fmaxf(fmaxf(fminf(1e-20f, dm * 0x1p-46f), fminf(dm * 0x1p-18f, m * 0x1p-126f)),
                             0x1p-126f);
    const float dx = fabsf(d.x) < dmin ? copysignf(dmin, d.x) : d.x;
    const float dy = fabsf(d.y) < dmin ? copysignf(dmin, d.y) : d.y;
    const float dz = fabsf(d.z) < dmin ? copysignf(dmin, d.z) : d.z;
    // hardware reciprocals (1 ulp, far inside the margin; 30 instructions fewer
    // than correctly rounded ones), but exact for the waves with a thin ray,
    // where box_agrees looks at their last bit
    float3 r = make_float3(__builtin_amdgcn_rcpf(dx), __builtin_amdgcn_rcpf(dy), __builtin_amdgcn_rcpf(dz));
    if (__any(wt_thin(w))) r = make_float3(1.0f / dx, 1.0f / dy, 1.0f / dz);
    s.oinv = make_float3(o.x * r.x, o.y * r.y, o.z * r.z);
    s.inv = make_float3(unit * r.x, unit * r.y, unit * r.z);
    s.nx = dx < 0.0f;
    s.ny = dy < 0.0f;
    s.nz = dz < 0.0f;
    s.apad = box_margin(m) * wt_scale(w);
    return s;
}

// ------------------------------------------------------------- traversal
// Stack of one lane: entries [0, depth) in LDS, 256 words apart (lane-
// interleaved, conflict-free), deeper ones in a global spill area at
// spill[(i - depth) * spill_stride].  The position is the LDS address of the
// next free entry, counted on past the last row for spilled entries.  The row
// below entry 0 holds kStackEnd, so popping an empty stack yields it and needs
// no test of its own (with addresses kept instead of indexes, 2% of every
// trace stage: 24-job batch 71.1 -> 69.3 ms).
typedef __attribute__((address_space(3))) uint32_t lds_u32;
constexpr uint32_t kStackEnd = 0xFFFFFFFFu;
constexpr int stack_words(int depth) { return (depth + 1) * 256; }  // LDS of a workgroup

struct Stack {
    lds_u32*  lds;     // entry 0
    uint32_t* spill;
    uint32_t  spill_stride;
    uint32_t  full;    // LDS address (row base) where fewer than 3 rows are left
    int       depth;   // LDS entries per lane (a constant of the kernel)
};

// `lds` is the workgroup's array of stack_words(depth) words, `spill` this
// lane's first spill entry.
__device__ __forceinline__ Stack make_stack(uint32_t* lds, int depth, uint32_t* spill, uint32_t stride)
{
    Stack st;
    lds_u32* row0 = (lds_u32*)lds;
    row0[threadIdx.x] = kStackEnd;
    st.lds = row0 + 256 + threadIdx.x;
    st.spill = spill;
    st.spill_stride = stride;
    st.full = (uint32_t)(uintptr_t)(row0 + 256 * (depth - 1));
    st.depth = depth;
    return st;
}

__device__ __forceinline__ void push(const Stack& st, lds_u32*& top, uint32_t v)
{
    const int i = (int)(top - st.lds) >> 8;
    if (i < st.depth) *top = v;
    else st.spill[(size_t)(i - st.depth) * st.spill_stride] = v;
    top += 256;
}
__device__ __forceinline__ uint32_t pop(const Stack& st, lds_u32*& top)
{
    top -= 256;
    const int i = (int)(top - st.lds) >> 8;  // -1: the kStackEnd row
    if (i < st.depth) return *top;
    return st.spill[(size_t)(i - st.depth) * st.spill_stride];
}

struct TraceCount {
    uint32_t nodes = 0;
    uint32_t tris = 0;
};

// Address of byte `byte` (< 64) of 64-byte record i (nodes and triangles).
// WIDE: any scene.  Without it the byte offset is kept in 32 bits, the form
// the vector loads take next to a scalar base (one instruction instead of
// two 64-bit ones and a register pair): for scenes with less than 2^26
// triangles (kNarrowTris), so that every offset is below 2^32.  At the 8
// waves/SIMD bound the short form spills 21 VGPRs, the wide one 24.
constexpr int kNarrowTris = 1 << 26;

template <bool WIDE>
__device__ __forceinline__ const char* record64(const void* base, uint32_t i, uint32_t byte)
{
    if (WIDE) return static_cast<const char*>(base) + (((size_t)i << 6) + byte);
    return static_cast<const char*>(base) + (size_t)((i << 6) + byte);
}

// The vertices of triangle `leaf` in the ray's coordinate order: three 12-byte
// loads from one line.
template <bool WIDE>
__device__ __forceinline__ void load_tri(const float* tris, int leaf, const WtRay& w, float3& v0,
                                         float3& v1, float3& v2)
{
    const char* p = record64<WIDE>(tris, (uint32_t)leaf, w.rot);
    v0 = *reinterpret_cast<const float3*>(p);
    v1 = *reinterpret_cast<const float3*>(p + 20);
    v2 = *reinterpret_cast<const float3*>(p + 40);
}

__device__ __forceinline__ int tri_prim(const float* tris, int leaf)
{
    return __float_as_int(tris[(size_t)leaf * kTriWords + kTriPrim]);
}

// Node fetches of a wave whose active lanes are all at the same node (about
// half of the fused kernel's visits on coherent probe rays) come through the
// scalar cache into scalar registers, leaving the vector memory path, which
// the divergent fetches keep busy, to those.  Nodes are read-only while any
// trace kernel runs.
typedef int sgpr16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void scalar_load64(unsigned long long addr, sgpr16_t& a)
{
    __asm__ __volatile__("s_load_dwordx16 %0, %1, 0x0\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=s"(a)
                         : "s"(addr)
                         : "memory");
}

template <bool WIDE>
__device__ __forceinline__ Node4 load_node(const Node4* nodes, uint32_t i)
{
    const uint4* p = reinterpret_cast<const uint4*>(record64<WIDE>(nodes, i, 0));
    const uint4 m = p[0], a = p[1], b = p[2], c = p[3];
    Node4 n;
    n.oxy = m.x;
    n.ozn = m.y;
    n.inner = (int)m.z;
    n.leaf = (int)m.w;
    n.lox[0] = a.x;
    n.lox[1] = a.y;
    n.loy[0] = a.z;
    n.loy[1] = a.w;
    n.loz[0] = b.x;
    n.loz[1] = b.y;
    n.hix[0] = b.z;
    n.hix[1] = b.w;
    n.hiy[0] = c.x;
    n.hiy[1] = c.y;
    n.hiz[0] = c.z;
    n.hiz[1] = c.w;
    return n;
}

__device__ __forceinline__ Node4 load_node_uniform(const Node4* nodes, uint32_t i)
{
    sgpr16_t w;
    scalar_load64((unsigned long long)(nodes + i), w);
    Node4 n;
    n.oxy = (uint32_t)w[0];
    n.ozn = (uint32_t)w[1];
    n.inner = w[2];
    n.leaf = w[3];
    n.lox[0] = (uint32_t)w[4];
    n.lox[1] = (uint32_t)w[5];
    n.loy[0] = (uint32_t)w[6];
    n.loy[1] = (uint32_t)w[7];
    n.loz[0] = (uint32_t)w[8];
    n.loz[1] = (uint32_t)w[9];
    n.hix[0] = (uint32_t)w[10];
    n.hix[1] = (uint32_t)w[11];
    n.hiy[0] = (uint32_t)w[12];
    n.hiy[1] = (uint32_t)w[13];
    n.hiz[0] = (uint32_t)w[14];
    n.hiz[1] = (uint32_t)w[15];
    return n;
}

// Whether the slab test of a triangle's own box, on its exact bounds, agrees
// that the ray meets it before tbest.  Asked for accepted triangles of thin
// rays: a ray that runs in the plane of an axis-aligned triangle (a probe on a
// wall) has a determinant of rounding errors only, and whether such a hit
// counts has always been decided by the box of the triangle; a widened box
// does not decide it.  All other rays meet the exact box of any triangle they
// are accepted by.
__device__ __forceinline__ void box_axis(const char* p, float per_unit, float inv, float oinv, float& tn,
                                         float& tf)
{
    // one axis at a time: the check is rare, its registers are not
    __asm__ __volatile__("" ::: "memory");
    const float a = *reinterpret_cast<const float*>(p), b = *reinterpret_cast<const float*>(p + 20),
                c = *reinterpret_cast<const float*>(p + 40);
    const float t0 = fmaf(fminf(a, fminf(b, c)) * per_unit, inv, -oinv);
    const float t1 = fmaf(fmaxf(a, fmaxf(b, c)) * per_unit, inv, -oinv);
    tn = fmaxf(tn, fminf(t0, t1));
    tf = fminf(tf, fmaxf(t0, t1));
}

template <bool WIDE>
__device__ __forceinline__ bool box_agrees(const float* tris, float unit, int leaf, const WtRay& w,
                                           const SlabRay& s, float tmin, float tbest)
{
    if (!wt_thin(w)) return true;
    __asm__ __volatile__("" : "+v"(unit));  // nothing of this block before the loop
    const float per_unit = 1.0f / unit;     // exact: a power of two
    const char* p = record64<WIDE>(tris, (uint32_t)leaf, 0);
    float tn = -__builtin_huge_valf(), tf = __builtin_huge_valf();
    box_axis(p, per_unit, s.inv.x, s.oinv.x, tn, tf);
    box_axis(p + 4, per_unit, s.inv.y, s.oinv.y, tn, tf);
    box_axis(p + 8, per_unit, s.inv.z, s.oinv.z, tn, tf);
    const float apad = s.apad * (1.0f / wt_scale(w));  // exact: a power of two
    float hi = fminf(tf, tbest);
    hi = fmaf(fabsf(hi), 4e-6f, hi) + apad;
    const float lo = fmaf(-fabsf(tn), 4e-6f, tn) - apad;
    return lo <= hi && hi >= tmin;
}

// Watertight test of triangle `leaf`.  Always through the vector path: a
// record that every active lane reads in the same order could come through
// the scalar cache, but the compare, the branch and the scalar registers cost
// more than the three 12-byte loads (24-job batch 72.5 ms with the scalar
// form, 71.0 without; 11k-triangle room plan 0.974 against 0.923 ms).
template <bool WIDE>
__device__ __forceinline__ bool fetch_wt(const float* tris, float unit, int leaf, const WtRay& w,
                                         const SlabRay& s, float tmin, float tmax, WtHit& h)
{
    float3 v0, v1, v2;
    load_tri<WIDE>(tris, leaf, w, v0, v1, v2);
    return wt_test(w, v0, v1, v2, tmin, tmax, h) && box_agrees<WIDE>(tris, unit, leaf, w, s, tmin, tmax);
}

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// FP16 value k (0 or 1) of a packed pair: an operand of v_fma_mix_f32.
__device__ __forceinline__ float half_of(uint32_t w, int k)
{
    return (float)__builtin_bit_cast(half2_t, w)[k];
}

// c ? a : b of a packed pair; the empty asm keeps the compiler from unpacking
// the halves first (two selects and two shifts instead of one select).
__device__ __forceinline__ uint32_t pick_pair(bool c, uint32_t a, uint32_t b)
{
    uint32_t r = c ? a : b;
    __asm__("" : "+v"(r));
    return r;
}

// What a visit found: entry distances e[k] of the hit inner children (+inf:
// missed, leaf or unused), their ids c[k], and the hit leaf children as a
// 4-bit mask, child k being leaf-order triangle leaf + k.
struct NodeHits {
    float    e[4];
    int      c[4];
    uint32_t leaves;
    int      leaf;
};

// The slab tests of a node's four children, their near and far planes picked.
struct NodePlanes {
    uint32_t nx[2], ny[2], nz[2], fx[2], fy[2], fz[2];
};

__device__ __forceinline__ void slab4(const SlabRay& s, const Node4& n, const NodePlanes& b, float tmin,
                                      float tbest, NodeHits& h)
{
    const float ax = fmaf(half_of(n.oxy, 0), s.inv.x, -s.oinv.x);
    const float ay = fmaf(half_of(n.oxy, 1), s.inv.y, -s.oinv.y);
    const float az = fmaf(half_of(n.ozn, 0), s.inv.z, -s.oinv.z);
    h.leaf = n.leaf;
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int p = k >> 1, q = k & 1;
        const float tn = fmaxf(fmaxf(fmaf(half_of(b.nx[p], q), s.inv.x, ax), fmaf(half_of(b.ny[p], q), s.inv.y, ay)),
                               fmaf(half_of(b.nz[p], q), s.inv.z, az));
        const float tf = fminf(fminf(fminf(fmaf(half_of(b.fx[p], q), s.inv.x, ax),
                                           fmaf(half_of(b.fy[p], q), s.inv.y, ay)),
                                     fmaf(half_of(b.fz[p], q), s.inv.z, az)), tbest) + s.apad;
        const bool hit = (tn <= tf) & (tf >= tmin);
        // inner children come first
        const bool inner = n.ozn >= (uint32_t)(k + 1) << 20;
        h.e[k] = (hit & inner) ? tn : __builtin_huge_valf();
        h.c[k] = n.inner + k;
        m |= hit ? 1u << k : 0u;
    }
    h.leaves = m & (n.ozn >> 16);
}

// Near and far planes by each lane's direction signs: 12 selects of packed
// pairs instead of a min and a max per child and axis.
__device__ __forceinline__ void slab4(const SlabRay& s, const Node4& n, float tmin, float tbest,
                                      NodeHits& h)
{
    NodePlanes b;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        b.nx[p] = pick_pair(s.nx, n.hix[p], n.lox[p]);
        b.fx[p] = pick_pair(s.nx, n.lox[p], n.hix[p]);
        b.ny[p] = pick_pair(s.ny, n.hiy[p], n.loy[p]);
        b.fy[p] = pick_pair(s.ny, n.loy[p], n.hiy[p]);
        b.nz[p] = pick_pair(s.nz, n.hiz[p], n.loz[p]);
        b.fz[p] = pick_pair(s.nz, n.loz[p], n.hiz[p]);
    }
    slab4(s, n, b, tmin, tbest, h);
}

// Visits node i: through the scalar cache when every active lane is at it
// (their base pointer is the same), else per lane.
template <bool WIDE>
__device__ __forceinline__ void fetch_slab4(const Node4* nodes, uint32_t i, const SlabRay& s,
                                            float tmin, float tbest, NodeHits& h)
{
    const uint32_t u = __builtin_amdgcn_readfirstlane(i);
    Node4 n;
    if (__all(i == u)) {
        n = load_node_uniform(nodes, u);
    } else {
        n = load_node<WIDE>(nodes, i);
    }
    slab4(s, n, tmin, tbest, h);
}

// Compare-exchange of two (entry distance, child id) pairs held as one 64-bit
// word each, distance in the high half: read as doubles, such words order as
// their float halves do (sign and exponent sit in the same place; +inf stays
// below a double's infinity, and 64-bit denormals are kept), so one v_min_f64
// and one v_max_f64 exchange distance and id together.  Both run at the rate
// of a 32-bit min (4.5 cycles per wave, measured); a compare with four selects
// took 22 (and on gfx950 a v_cndmask_b32_e32 right behind another one of the
// same SIMD takes 23 by itself, against 4.4 behind anything else).  The
// traversal is bound by VALU issue as much as by its vector loads (40 more
// VALU instructions per visit: +13% on the room, +8% on the terrain), so the 15
// instructions per visit saved show: a plan of 2048 probes x 4096 rays in the
// 11k-triangle room 1.186 -> 1.152 ms, served requests 45.9 -> 45.0 ms.
__device__ __forceinline__ void cswap(double& a, double& b)
{
    double lo, hi;
    __asm__("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    __asm__("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

// Orders next_node visits the inner children of a node in.
enum : int {
    kOrderNear = 0,  // nearest entry first (closest-hit queries)
    kOrderSlot = 1,  // slot order, no sort
    kOrderFar = 2,   // farthest entry first
};

// After the leaf tests (their e set to +inf): order the inner children, push
// all hit ones but the first (last first) and continue at the first, else
// pop.  Returns false when the stack is empty.  Closest-hit queries sort near
// first.  Shadow queries stop at any hit, so the order only moves the visit
// count: slot order drops the sort's 20 instructions per visit and visits
// about as many nodes as near first (0.1-0.3% fewer without the sort on
// rooms and terrains of 11k-1.15M triangles); far first (the sort on negated
// entries, misses staying +inf and last) reaches an occluder sooner on some
// trees and not on others, so it is a variant for the autotuners: on the
// 11k-triangle room it visited 5.1% fewer nodes and ran 4% faster, on a
// batch of 64 jobs over four scenes 1.4% fewer and 0.5% slower, both with
// trees built from per-axis Morton cells; on trees from cubic cells (the
// build's) it runs level with slot order or 1% behind.  The pushes below
// are right for any order (a missed child is written and then overwritten).
template <int ORDER = kOrderNear>
__device__ __forceinline__ bool next_node(float e[4], int c[4], const Stack& st, lds_u32*& top,
                                          uint32_t& node)
{
    if (ORDER == kOrderFar) {
        for (int k = 0; k < 4; ++k)
            if (e[k] != __builtin_huge_valf()) e[k] = -e[k];
    }
    if (ORDER != kOrderSlot) {
        double k[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) k[i] = __hiloint2double(__float_as_int(e[i]), c[i]);
        cswap(k[0], k[1]);
        cswap(k[2], k[3]);
        cswap(k[0], k[2]);
        cswap(k[1], k[3]);
        cswap(k[1], k[2]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            e[i] = __int_as_float(__double2hiint(k[i]));
            c[i] = __double2loint(k[i]);
        }
    }
    const float inf = __builtin_huge_valf();
    const bool go = e[0] != inf;
    if (__all((uint32_t)(uintptr_t)top < st.full)) {
        // Every active lane has three free LDS entries (one wave-uniform
        // test): straight-line pushes with conditional increments, and a pop
        // that every lane reads.  A write past the top lands at most where the
        // all-hit case writes, and is overwritten by the next push or left
        // unused, so the pushes are the same as below in any order.
        *top = (uint32_t)c[3];
        top += e[3] != inf ? 256 : 0;
        *top = (uint32_t)c[2];
        top += e[2] != inf ? 256 : 0;
        *top = (uint32_t)c[1];
        top += e[1] != inf ? 256 : 0;
        const uint32_t below = top[-256];
        node = go ? (uint32_t)c[0] : below;
        top -= go ? 0 : 256;
        return node != kStackEnd;
    }
    if (e[3] != inf) push(st, top, (uint32_t)c[3]);
    if (e[2] != inf) push(st, top, (uint32_t)c[2]);
    if (e[1] != inf) push(st, top, (uint32_t)c[1]);
    node = (uint32_t)c[0];
    if (!go) node = pop(st, top);
    return node != kStackEnd;
}

// Closest hit: lexicographic minimum of (t, prim id) over accepted
// triangles in [tmin, tmax].  Returns the prim id or -1.  Any BVH whose
// boxes are conservative gives the same answer: every triangle that could
// beat the current best is tested, and ties go to the lower prim id.
// The best triangle is held as its leaf; prim ids are read for the rare equal
// distances and once at the end.
template <bool COUNT, bool WIDE = true>
__device__ int trace_closest(const SceneView& sc, const float3& o, const float3& d, float tmin,
                             float tmax, float& t_out, float& u_out, float& v_out,
                             const Stack& st, TraceCount& cnt)
{
    if (sc.ntris <= 0) return -1;
    const WtRay w = wt_setup(o, d);
    const SlabRay s = slab_setup(o, d, w, sc.maxabs, sc.unit);
    float tbest = tmax, bV = 0.0f, bW = 0.0f, bdet = 1.0f;
    int best = -1;
    lds_u32* top = st.lds;
    uint32_t node = 0;
    for (;;) {
        if (COUNT) ++cnt.nodes;
        NodeHits n;
        fetch_slab4<WIDE>(sc.nodes, node, s, tmin, tbest, n);
        // leaves one at a time per lane: the wave runs as many tests as its
        // busiest lane has hit leaves, not one per child slot
        for (uint32_t leaves = n.leaves; leaves != 0; leaves &= leaves - 1) {
            if (COUNT) ++cnt.tris;
            const int leaf = n.leaf + __builtin_ctz(leaves);
            WtHit h;
            // t <= tbest holds on acceptance; an equal t keeps the lower prim id
            if (fetch_wt<WIDE>(sc.tris, sc.unit, leaf, w, s, tmin, tbest, h) &&
                (best < 0 || h.t < tbest || tri_prim(sc.tris, leaf) < tri_prim(sc.tris, best))) {
                tbest = h.t;
                best = leaf;
                bV = h.V;
                bW = h.W;
                bdet = h.det;
            }
        }
        if (!next_node(n.e, n.c, st, top, node)) break;
    }
    if (best >= 0) {
        t_out = tbest;
        u_out = bV / bdet;
        v_out = bW / bdet;
        best = tri_prim(sc.tris, best);
    }
    return best;
}

// Shadow query: true if any triangle is accepted in [tmin, tmax].  FAR: the
// inner children far first, else in slot order (same answer either way).
template <bool COUNT, bool FAR = false, bool WIDE = true>
__device__ bool trace_any(const SceneView& sc, const float3& o, const float3& d, float tmin,
                          float tmax, const Stack& st, TraceCount& cnt)
{
    if (sc.ntris <= 0) return false;
    const WtRay w = wt_setup(o, d);
    const SlabRay s = slab_setup(o, d, w, sc.maxabs, sc.unit);
    lds_u32* top = st.lds;
    uint32_t node = 0;
    for (;;) {
        if (COUNT) ++cnt.nodes;
        NodeHits n;
        fetch_slab4<WIDE>(sc.nodes, node, s, tmin, tmax, n);
        for (uint32_t leaves = n.leaves; leaves != 0; leaves &= leaves - 1) {
            if (COUNT) ++cnt.tris;
            WtHit h;
            if (fetch_wt<WIDE>(sc.tris, sc.unit, n.leaf + __builtin_ctz(leaves), w, s, tmin, tmax, h)) return true;
        }
        if (!next_node<FAR ? kOrderFar : kOrderSlot>(n.e, n.c, st, top, node)) break;
    }
    return false;
}

// ------------------------------------------------------------------- sky
__device__ __forceinline__ float3 sky_radiance(const vlb_sky& sky, const float3& d)
{
    float g = d.y > 0.0f ? d.y : 0.0f;
    float sd = d.x * sky.sun_dir[0] + d.y * sky.sun_dir[1] + d.z * sky.sun_dir[2];
    float sun = expf(sky.sun_sharpness * (sd - 1.0f));
    float3 r;
    r.x = sky.horizon_rgb[0] + (sky.zenith_rgb[0] - sky.horizon_rgb[0]) * g + sky.sun_rgb[0] * sun;
    r.y = sky.horizon_rgb[1] + (sky.zenith_rgb[1] - sky.horizon_rgb[1]) * g + sky.sun_rgb[1] * sun;
    r.z = sky.horizon_rgb[2] + (sky.zenith_rgb[2] - sky.horizon_rgb[2]) * g + sky.sun_rgb[2] * sun;
    return r;
}

// env_map.rchit:27-34
__device__ __forceinline__ float srgb(float x)
{
    if (x < 0.0031308f) return x * 12.92f;
    return 1.055f * powf(x, 1.0f / 2.4f) - 0.055f;
}
// RGBA8 storage-image store followed by a load
__device__ __forceinline__ float unorm8(float x)
{
    float c = (x > 0.0f) ? (x < 1.0f ? x : 1.0f) : 0.0f;
    return rintf(c * 255.0f) / 255.0f;
}

// ---------------------------------------------------------------- shading
// Indirect term of a multi-bounce bake at hit point P with the two-sided
// shading normal N: the grid lookup of probe_grid.hpp (visibility rays to the
// corner probes traced here, counted as shadow rays), times g.scale.
template <bool COUNT, bool FAR = false, bool WIDE = true>
__device__ float3 grid_indirect(const SceneView& sc, const ProbeGridView& g, const float3& P,
                                const float3& N, const Stack& st, TraceCount& cnt,
                                uint32_t& nshadow)
{
    const float p[3] = {P.x, P.y, P.z};
    // visibility first, as a mask of hidden corners: only the hit point and
    // the ray origin are live across the eight traversals, not the basis and
    // the running sums.  Corners are then found again (same values).
    uint32_t hidden = 0;
    if (g.vis) {
        const float3 org = make_float3(P.x + g.bias * N.x, P.y + g.bias * N.y, P.z + g.bias * N.z);
        for (int v = 0; v < 8; ++v) {
            const GridCorner c = grid_corner(g, p, v);
            if (corner_needs_ray(g, c, sc.ntris)) {
                ++nshadow;
                const float3 dir = make_float3(c.dir[0] / c.dist, c.dir[1] / c.dist, c.dir[2] / c.dist);
                if (trace_any<COUNT, FAR, WIDE>(sc, org, dir, 0.0f, c.dist, st, cnt)) hidden |= 1u << v;
            }
        }
    }
    const float n[3] = {N.x, N.y, N.z};
    float Y[16];
    grid_basis(g, n, Y);
    float sw = 0.0f, acc[3] = {0.0f, 0.0f, 0.0f};
    for (int v = 0; v < 8; ++v) {
        const GridCorner c = grid_corner(g, p, v);
        const float w = (hidden >> v) & 1u ? 0.0f : c.w;
        if (w > 0.0f) {
            float val[3];
            corner_value(g, c.row, Y, val);
            acc[0] += w * val[0];
            acc[1] += w * val[1];
            acc[2] += w * val[2];
            sw += w;
        }
    }
    if (!(sw > 0.0f)) return make_float3(0.f, 0.f, 0.f);
    return make_float3(g.scale * (acc[0] / sw), g.scale * (acc[1] / sw), g.scale * (acc[2] / sw));
}

// Direction Ld and distance of light j seen from hit point P, and its
// irradiance E there (before the cosine).
__device__ __forceinline__ void light_geom(const ShadeParams& sp, int j, const float3& P,
                                           float3& Ld, float& dist, float3& E)
{
    const vlb_light& Lj = sp.lights[j];
    if (Lj.type == VLB_LIGHT_POINT) {
        const float3 Lv = make_float3(Lj.vec[0] - P.x, Lj.vec[1] - P.y, Lj.vec[2] - P.z);
        dist = sqrtf(dot3(Lv, Lv));
        Ld = dist > 0.0f ? make_float3(Lv.x / dist, Lv.y / dist, Lv.z / dist)
                         : make_float3(0.f, 0.f, 0.f);
        const float d2 = dist * dist;
        E = make_float3(Lj.rgb[0] / d2, Lj.rgb[1] / d2, Lj.rgb[2] / d2);
    } else {
        Ld = make_float3(-Lj.vec[0], -Lj.vec[1], -Lj.vec[2]);
        dist = sp.t_max;
        E = make_float3(Lj.rgb[0], Lj.rgb[1], Lj.rgb[2]);
    }
}

// Origin of the shadow ray from hit point P with the two-sided normal N.
__device__ __forceinline__ float3 shadow_origin(const ShadeParams& sp, const float3& P, const float3& N)
{
    return make_float3(P.x + sp.shadow_bias * N.x, P.y + sp.shadow_bias * N.y,
                       P.z + sp.shadow_bias * N.z);
}

// Lambert term of light j at hit point P with the two-sided normal N: the
// contribution E cos is formed before the shadow query, so only it (not E
// and the cosine) is live across the traversal; added to acc when unoccluded.
template <bool COUNT, bool FAR = false, bool WIDE = true>
__device__ __forceinline__ void light_term(const SceneView& sc, const ShadeParams& sp, int j,
                                           const float3& P, const float3& N, float3& acc,
                                           const Stack& st, TraceCount& cnt, uint32_t& nshadow)
{
    float3 Ld, E;
    float dist;
    light_geom(sp, j, P, Ld, dist, E);
    const float cosNL = dot3(N, Ld);
    if (cosNL > 0.0f) {
        const float3 c = make_float3(E.x * cosNL, E.y * cosNL, E.z * cosNL);
        const float3 org = shadow_origin(sp, P, N);
        ++nshadow;
        if (!trace_any<COUNT, FAR, WIDE>(sc, org, Ld, 0.0f, dist, st, cnt)) {
            acc.x = acc.x + c.x;
            acc.y = acc.y + c.y;
            acc.z = acc.z + c.z;
        }
    }
}

// Hit point and interpolated shading normal (env_map.rchit:63-68).
__device__ __forceinline__ void hit_point_normal(const SceneView& sc, int prim, const float3& o,
                                                 const float3& d, float t, float u, float v,
                                                 float3& P, float3& N)
{
    const float4 s0 = sc.shade[3 * prim + 0];
    const float4 s1 = sc.shade[3 * prim + 1];
    const float4 s2 = sc.shade[3 * prim + 2];
    const float b0 = 1.0f - u - v;
    P = make_float3(o.x + d.x * t, o.y + d.y * t, o.z + d.z * t);
    float3 m;
    m.x = s0.x * b0 + s1.x * u + s2.x * v;
    m.y = s0.y * b0 + s1.y * u + s2.y * v;
    m.z = s0.z * b0 + s1.z * u + s2.z * v;
    const float ml = sqrtf(dot3(m, m));
    N = ml > 0.0f ? make_float3(m.x / ml, m.y / ml, m.z / ml) : make_float3(0.f, 0.f, 0.f);
}

// Radiance carried by one primary ray.  `nshadow` counts traced shadow rays.
// IND compiles the multi-bounce term in (used only when sp.ind.coeffs is
// set); direct-only kernels are built without it and keep its registers free.
// FAR: shadow queries visit children far first (same radiance).
template <bool COUNT, bool IND = false, bool FAR = false, bool WIDE = true>
__device__ float3 shade_ray(const SceneView& sc, const ShadeParams& sp, const float3& o,
                            const float3& d, float tmin, float tmax, const Stack& st,
                            TraceCount& cnt, uint32_t& nshadow, int& hit_prim)
{
    float t = 0.0f, u = 0.0f, v = 0.0f;
    const int prim = trace_closest<COUNT, WIDE>(sc, o, d, tmin, tmax, t, u, v, st, cnt);
    hit_prim = prim;
    const bool ref = sp.mode == VLB_SHADE_REFERENCE;
    if (prim < 0) {
        float3 s = sky_radiance(sp.sky, d);
        if (ref) {
            if (sp.ref.flags & VLB_REF_SRGB) {
                s.x = srgb(s.x);
                s.y = srgb(s.y);
                s.z = srgb(s.z);
            }
            if (sp.ref.flags & VLB_REF_UNORM8) {
                s.x = unorm8(s.x);
                s.y = unorm8(s.y);
                s.z = unorm8(s.z);
            }
        }
        return s;
    }
    float3 P, N;
    hit_point_normal(sc, prim, o, d, t, u, v, P, N);
    if (ref) {
        // env_map.rchit:73-101, main.rchit:95-116
        const vlb_ref_shading& r = sp.ref;
        const float3 L = make_float3(r.light_position[0] - P.x, r.light_position[1] - P.y,
                                     r.light_position[2] - P.z);
        const float Llen = sqrtf(dot3(L, L));
        const float3 Ln = Llen > 0.0f ? make_float3(L.x / Llen, L.y / Llen, L.z / Llen)
                                      : make_float3(0.f, 0.f, 0.f);
        const float sdn = dot3(Ln, N);
        const float sDotN = sdn > 0.0f ? sdn : 0.0f;
        const float3 org = make_float3(P.x + r.shadow_bias * N.x, P.y + r.shadow_bias * N.y,
                                       P.z + r.shadow_bias * N.z);
        bool in_shadow = true;
        if (sDotN != 0.0f) {
            ++nshadow;
            in_shadow = trace_any<COUNT, FAR, WIDE>(sc, org, Ln, 0.0f, Llen, st, cnt);
        }
        float diffuse = 0.0f, spec = 0.0f;
        if (!in_shadow) {
            diffuse = r.c_diffuse * sDotN;
            const float dnl = dot3(N, Ln);
            const float3 R = make_float3(Ln.x - 2.0f * dnl * N.x, Ln.y - 2.0f * dnl * N.y,
                                         Ln.z - 2.0f * dnl * N.z);
            const float rd = dot3(R, d);
            spec = r.c_specular * powf(rd > 0.0f ? rd : 0.0f, r.glossiness);
        }
        // albedo read after the shadow query (see the Lambert path below)
        __asm__ __volatile__("" ::: "memory");
        const float3 alb = make_float3(sc.shade[3 * prim + 0].w, sc.shade[3 * prim + 1].w,
                                       sc.shade[3 * prim + 2].w);
        const bool zero = alb.x == 0.0f && alb.y == 0.0f && alb.z == 0.0f;
        float3 c;
        c.x = (zero ? 1.0f : alb.x) * (r.ambient + diffuse + spec);
        c.y = (zero ? 1.0f : alb.y) * (r.ambient + diffuse + spec);
        c.z = (zero ? 1.0f : alb.z) * (r.ambient + diffuse + spec);
        if (r.flags & VLB_REF_SRGB) {
            c.x = srgb(c.x);
            c.y = srgb(c.y);
            c.z = srgb(c.z);
        }
        if (r.flags & VLB_REF_UNORM8) {
            c.x = unorm8(c.x);
            c.y = unorm8(c.y);
            c.z = unorm8(c.z);
        }
        return c;
    }
    // LAMBERT, two-sided
    if (dot3(N, d) > 0.0f) N = make_float3(-N.x, -N.y, -N.z);
    float3 acc = make_float3(0.f, 0.f, 0.f);
    // the last light is peeled off the loop: after its shadow ray is set up,
    // neither the hit point nor the normal is live across its traversal
    // (unless the indirect term needs them)
    const int nl = sp.nlights;
    for (int j = 0; j + 1 < nl; ++j)
        light_term<COUNT, FAR, WIDE>(sc, sp, j, P, N, acc, st, cnt, nshadow);
    if (nl > 0) light_term<COUNT, FAR, WIDE>(sc, sp, nl - 1, P, N, acc, st, cnt, nshadow);
    // albedo read after the shadow queries rather than held across them (the
    // compiler barrier keeps it from reusing the loads of the normals, which
    // it would otherwise keep in scratch across the traversals)
    __asm__ __volatile__("" ::: "memory");
    const float3 alb = make_float3(sc.shade[3 * prim + 0].w, sc.shade[3 * prim + 1].w,
                                   sc.shade[3 * prim + 2].w);
    const float kInvPi = 0.318309886183790671538f;
    if (!IND || !sp.ind.coeffs)
        return make_float3(alb.x * acc.x * kInvPi, alb.y * acc.y * kInvPi, alb.z * acc.z * kInvPi);
    const float3 E = grid_indirect<COUNT, FAR, WIDE>(sc, sp.ind, P, N, st, cnt, nshadow);
    return make_float3(alb.x * acc.x * kInvPi + alb.x * E.x, alb.y * acc.y * kInvPi + alb.y * E.y,
                       alb.z * acc.z * kInvPi + alb.z * E.z);
}

}  // namespace vlb
