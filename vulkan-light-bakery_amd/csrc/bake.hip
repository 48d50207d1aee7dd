// bake.hip -- the probe-baking hot path on gfx950.
//
// One fused, persistent kernel per bake replaces, per probe, the reference's
//   vkCmdTraceRaysKHR(3141x1000)  env_map.rgen -> env_map.rchit/shadow.rmiss
//                                 /main.rmiss -> RGBA8 image      (getMap,
//                                 src/baker/env_map_generator.cpp:325-359)
//   vkCmdDispatch(197x63) sh.comp (dispatchBakingKernel,
//                                 src/baker/light_baker.cpp:269-285)
//   mapMemory + memcpy 192 B      (light_baker.cpp:317-322)
// and its merge kernel replaces the host read-back.
//
// Two kernels per bake plus the merge:
//  k_trace   one ray per lane: closest hit, shading, shadow rays, sky; writes
//            FP32 radiance once, in the MFMA operand order of k_project.
//            Few live registers (no accumulators across the traversal), so
//            occupancy is bounded by the LDS stack, not by VGPRs.
//  k_project the SH projection as a dense contraction on MFMA with FP32
//            Kahan accumulation across chunks (HBM-bound, 12 B per ray).
//  k_merge   FP64 cross-slice merge in a fixed order (deterministic; no
//            atomics on the result path -- the reference's sh.comp:39 "+="
//            is a data race).
//
// k_trace walks its rays XCD by XCD: workgroup b runs on XCD b % 8
// (round-robin dispatch), and XCD x owns the x-th contiguous eighth of the
// rays, so neighbouring probes and directions share that XCD's L2.  Work is
// taken 64 rays at a time from the XCD's counters, then from the other XCDs'
// once they are drained, so the launch ends when the work does rather than
// when its unluckiest workgroup does.
#include "project_common.hpp"

namespace vlb {
namespace {

// Clears the 32 work counters of the fused kernel (a kernel, not a memset, so that captured graphs replay it).
__global__ void k_zero_ctr8(unsigned long long* c)
{
    if (threadIdx.x < 32) c[threadIdx.x * kCtrStride] = 0ull;
}

// ----------------------------------------------------------- trace + shade
// One ray per lane, persistent, over "trace tiles" (16 probes x 32 rays =
// 512 rays), 64 rays per wave and fetch.  Thread t of a tile traces for probe
// 16*pg + (l & 15) the ray 32*ch + 8*(l >> 4) + e, with l = t >> 3 and
// e = t & 7, and stores its radiance at rad[((tile*3 + c)*64 + l)*8 + e]: the 16x16 MFMA A-operand
// order of the projection kernel, written fully coalesced.  The lane map
// (tile_map, a.map) sets how many neighbouring probes x directions (probes
// Morton sorted, directions on a Hilbert curve) one wave covers.
// OCC > 0 asks the compiler for OCC waves per SIMD (VGPR budget 512/OCC).
// At 8 waves/SIMD the arguments read per set of rays (kernel_args) leave 11
// spilled VGPRs fewer (21 are left, 76 B of scratch per lane): 2048 probes x
// 4096 rays of the 11k-triangle room 0.855 against 0.871 ms per bake, 16,384 x
// 16,384 of a 1.15M-triangle terrain 33.8 against 34.35.
// IND: plans with the multi-bounce term.  FAR: shadow queries visit children
// far first (same radiance; fewer node visits on some scenes).
template <bool RECORD, bool COUNT, int OCC, bool IND, bool FAR = false,
          bool WIDE = RECORD || COUNT>
__global__ __launch_bounds__(256, OCC > 0 ? OCC : 1) void k_trace(BakeArgs args)
{
    __shared__ uint32_t lds[stack_words(kLdsDepth)];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    Stack st = make_stack(lds, kLdsDepth, args.spill + (size_t)blockIdx.x * 256 + tid, args.spill_stride);
    TraceCount cnt;
    uint32_t nshadow = 0;
    __shared__ unsigned used;
    const WorkRanges work(args.wctr, (size_t)args.ntrace * 512, &used);
    const int own = WorkRanges::own();
    for (;;) {
        const unsigned long long b = work.take(own);
        if (b == ~0ull) break;
        const BakeArgs& a = kernel_args<BakeArgs>();
        const size_t it = (size_t)b + lane;
        int tile, l, e;
        tile_map(a.map, it, tile, l, e);
        const int t = l * 8 + e;
        const int pg = tile / a.nchunk;
        const int ch = tile - pg * a.nchunk;
        const int probe = pg * 16 + (l & 15);
        const int r = ch * 32 + 8 * (l >> 4) + e;
        const float4 dd = a.dirs[r];
        float3 L = make_float3(0.f, 0.f, 0.f);
        if (probe < a.P && dd.w != 0.0f) {
            const float4 pp = a.probes[probe];
            int hp = -1;
            L = shade_ray<COUNT, IND, FAR, WIDE>(a.sc, a.sp, make_float3(pp.x, pp.y, pp.z),
                                 make_float3(dd.x, dd.y, dd.z), a.tmin, a.tmax, st, cnt, nshadow, hp);
            if (RECORD) {
                const size_t ri = (size_t)a.probe_perm[probe] * a.R + a.dir_perm[r];
                if (a.rad_out) {
                    a.rad_out[3 * ri + 0] = L.x;
                    a.rad_out[3 * ri + 1] = L.y;
                    a.rad_out[3 * ri + 2] = L.z;
                }
                if (a.hit_out) a.hit_out[ri] = hp;
            }
        }
        float* out = a.rad + (size_t)tile * 1536 + t;
        out[0] = L.x;
        out[512] = L.y;
        out[1024] = L.z;
    }
    if (COUNT) {
        atomicAdd(&args.counters[0], (unsigned long long)cnt.nodes);
        atomicAdd(&args.counters[1], (unsigned long long)cnt.tris);
        atomicAdd(&args.counters[2], (unsigned long long)nshadow);
    }
}

// Small launches, one fetch per wave at most: wave w takes the rays from
// w * n on, n = 64 or fewer, so that the chip has waves to run while each
// waits for its loads, and a wave's longest ray is the longest of fewer.  No
// counters, and the registers of an unbounded kernel.
__global__ __launch_bounds__(256) void k_trace_small(BakeArgs a, int n)
{
    __shared__ uint32_t lds[stack_words(kLdsDepth)];
    const int tid = threadIdx.x, lane = tid & 63;
    Stack st = make_stack(lds, kLdsDepth, a.spill + (size_t)blockIdx.x * 256 + tid, a.spill_stride);
    TraceCount cnt;
    uint32_t nshadow = 0;
    const size_t it = ((size_t)blockIdx.x * 4 + (tid >> 6)) * n + lane;
    if (lane >= n || it >= (size_t)a.ntrace * 512) return;
    int tile, l, e;
    tile_map(a.map, it, tile, l, e);
    const int pg = tile / a.nchunk;
    const int ch = tile - pg * a.nchunk;
    const int probe = pg * 16 + (l & 15);
    const float4 dd = a.dirs[ch * 32 + 8 * (l >> 4) + e];
    float3 L = make_float3(0.f, 0.f, 0.f);
    if (probe < a.P && dd.w != 0.0f) {
        const float4 pp = a.probes[probe];
        int hp = -1;
        L = shade_ray<false, false, false, false>(a.sc, a.sp, make_float3(pp.x, pp.y, pp.z),
                                                  make_float3(dd.x, dd.y, dd.z), a.tmin, a.tmax, st,
                                                  cnt, nshadow, hp);
    }
    float* out = a.rad + (size_t)tile * 1536 + l * 8 + e;
    out[0] = L.x;
    out[512] = L.y;
    out[1024] = L.z;
}

// ------------------------------------------------------------- projection
// Tile = (probe group pg, slice sl): chunks sl*nch .. sl*nch + nch - 1 of the
// group's trace tiles (consecutive in `rad`), partials of slice sl.
template <int PREC>
__global__ __launch_bounds__(256) void k_project(BakeArgs a)
{
    __shared__ float red[3 * 24 * 64];
    const int nch = a.RS >> 5;
    for (int tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
        const int pg = tile / a.nslices;
        const int sl = tile - pg * a.nslices;
        const int ch0 = sl * nch;
        const float* rad0 = a.rad + ((size_t)pg * a.nchunk + ch0) * 1536;
        float2* prow = a.partials + ((size_t)sl * a.Ppad + (size_t)pg * 16) * 48;
        project_tile<PREC>(rad0, nch, ch0, a.ytab, (size_t)a.Rpad * 2, red, prow);
    }
}

// FP64 cross-slice merge: out[p][k][c] = scale * sum_s (sum_s - comp_s).
__global__ __launch_bounds__(256) void k_merge(MergeArgs m)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= m.Ppad * 48) return;
    const int ps = idx / 48;
    const int rem = idx - ps * 48;
    const int c = rem >> 4;
    const int k = rem & 15;
    if (k >= m.K) return;
    const int op = m.probe_perm[ps];
    if (op < 0) return;
    double s = 0.0;
    for (int sl = 0; sl < m.nslices; ++sl) {
        const float2 v = m.partials[((size_t)sl * m.Ppad + ps) * 48 + rem];
        s += (double)v.x - (double)v.y;
    }
    s *= m.scale;
    const size_t o = ((size_t)op * m.K + k) * 3 + c;
    if (m.out) m.out[o] = (float)s;
    if (m.out64) m.out64[o] = s;
}

__global__ __launch_bounds__(256) void k_trace_closest(SceneView sc, const float* __restrict__ org,
                                                       const float* __restrict__ dir, int n,
                                                       float tmin, float tmax, int* prim,
                                                       float* tout, float* uout, float* vout,
                                                       uint32_t* spill, uint32_t stride)
{
    __shared__ uint32_t lds[stack_words(kLdsDepth)];
    Stack st = make_stack(lds, kLdsDepth, spill + (size_t)blockIdx.x * 256 + threadIdx.x, stride);
    TraceCount cnt;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const float3 o = make_float3(org[3 * i], org[3 * i + 1], org[3 * i + 2]);
        const float3 d = make_float3(dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]);
        float t = 0.f, u = 0.f, v = 0.f;
        const int p = trace_closest<false>(sc, o, d, tmin, tmax, t, u, v, st, cnt);
        prim[i] = p;
        tout[i] = p >= 0 ? t : 0.0f;
        uout[i] = p >= 0 ? u : 0.0f;
        vout[i] = p >= 0 ? v : 0.0f;
    }
}

__global__ __launch_bounds__(256) void k_trace_occluded(SceneView sc, const float* __restrict__ org,
                                                        const float* __restrict__ dir,
                                                        const float* __restrict__ tmax, int n,
                                                        float tmin, uint8_t* occ,
                                                        uint32_t* spill, uint32_t stride)
{
    __shared__ uint32_t lds[stack_words(kLdsDepth)];
    Stack st = make_stack(lds, kLdsDepth, spill + (size_t)blockIdx.x * 256 + threadIdx.x, stride);
    TraceCount cnt;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const float3 o = make_float3(org[3 * i], org[3 * i + 1], org[3 * i + 2]);
        const float3 d = make_float3(dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]);
        occ[i] = trace_any<false>(sc, o, d, tmin, tmax[i], st, cnt) ? 1 : 0;
    }
}

template <class K>
int occupancy_of(K kernel, int cus)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, 256, 0) != hipSuccess || nb < 1) nb = 1;
    return nb * cus;
}

}  // namespace

int trace_grid_size(Context& ctx, int occ, bool far)
{
    int g;
    if (far) {
        if (occ == 8) g = occupancy_of(k_trace<false, false, 8, false, true>, ctx.num_cus);
        else if (occ == 6) g = occupancy_of(k_trace<false, false, 6, false, true>, ctx.num_cus);
        else g = occupancy_of(k_trace<false, false, 0, false, true>, ctx.num_cus);
    } else if (occ == 8) g = occupancy_of(k_trace<false, false, 8, false>, ctx.num_cus);
    else if (occ == 6) g = occupancy_of(k_trace<false, false, 6, false>, ctx.num_cus);
    else g = occupancy_of(k_trace<false, false, 0, false>, ctx.num_cus);
    return (g + 7) & ~7;
}

// Rays per wave of k_trace_small for this many rays, or 0: k_trace.  The
// fewest of 16, 32 and 64 that make no more than 4 waves/SIMD; beyond 64 both
// kernels have the waves they can hold.  Trace, projection and merge of a
// repeated bake in us, k_trace | 16 | 32 | 64 rays per wave:
//   rays      11k-triangle room       0.5M terrain            2M city
//    65,536   106 |  91 |  97 | 100   132 | 117 | 124 | 124   100 |  91 |  84 |  91
//    98,304   123 | 112 | 114 | 120   144 | 142 | 130 | 138   107 | 110 |  96 |  98
//   131,072   110 | 117 | 110 | 101   162 | 145 | 149 | 152   115 | 128 | 104 | 105
//   196,608   121 |   - | 117 | 110   181 |   - | 172 | 169   118 |   - | 117 | 109
//   262,144   132 |   - | 138 | 115   179 |   - | 180 | 179   122 |   - | 140 | 111
int trace_small_launch(const BakeArgs& a, int num_cus)
{
    const long long rays = (long long)a.ntrace * 512, waves = 16ll * num_cus;
    if (a.sc.ntris >= kNarrowTris || a.sp.ind.coeffs) return 0;
    const int n = rays <= 16 * waves ? 16 : rays <= 32 * waves ? 32 : rays <= 64 * waves ? 64 : 0;
    return n && (rays / n + 3) / 4 <= (long long)(a.spill_stride / 256) ? n : 0;
}

// k_trace at the occupancy bound `occ`.
template <bool IND, bool FAR, bool WIDE>
static void launch_occ(const BakeArgs& a, int occ, int grid, hipStream_t st)
{
    if (occ == 8) k_trace<false, false, 8, IND, FAR, WIDE><<<grid, 256, 0, st>>>(a);
    else if (occ == 6) k_trace<false, false, 6, IND, FAR, WIDE><<<grid, 256, 0, st>>>(a);
    else k_trace<false, false, 0, IND, FAR, WIDE><<<grid, 256, 0, st>>>(a);
}

int launch_trace(const BakeArgs& a, bool record, bool count, int occ, bool far, int grid, int per,
                 hipStream_t st)
{
    VLB_REQUIRE(grid % 8 == 0, VLB_ERR_INVALID, "trace grid must be a multiple of 8");
    const bool wide = a.sc.ntris >= kNarrowTris;  // else record64's short form
    if (per && !record && !count) {
        grid = (a.ntrace * 512 / per + 3) / 4;
        k_trace_small<<<grid, 256, 0, st>>>(a, per);
        VLB_HIP(hipGetLastError());
        return grid;
    }
    k_zero_ctr8<<<1, 64, 0, st>>>(a.wctr);
    // no more workgroups than take one set of rays per wave (64 probes x 1024
    // rays in this kernel, one-shot: 230 us with a full grid asking for work,
    // 190 with 256 workgroups)
    grid = std::min(grid, std::max(8, (a.ntrace * 2 + 7) / 8 * 8));
    // recording (hit ids are the same in any shadow order) and multi-bounce
    // plans keep slot-order shadows.  The multi-bounce kernel takes the
    // variant's occupancy bound like the direct one: it is bound by the latency
    // and issue of its eight corner rays per hit, so 8 waves/SIMD with spills
    // outside the loops beat 3 without (2048 probes x 4096 rays of the
    // 11k-triangle room: 2.9 ms per bounce at 64 VGPRs against 4.1 at 144).
    const bool ind = a.sp.ind.coeffs != nullptr;
    if (record) {
        if (ind) k_trace<true, false, 0, true><<<grid, 256, 0, st>>>(a);
        else k_trace<true, false, 0, false><<<grid, 256, 0, st>>>(a);
    } else if (count) {
        if (ind) k_trace<false, true, 0, true><<<grid, 256, 0, st>>>(a);
        else if (far) k_trace<false, true, 0, false, true><<<grid, 256, 0, st>>>(a);
        else k_trace<false, true, 0, false><<<grid, 256, 0, st>>>(a);
    } else if (ind) {
        if (wide) launch_occ<true, false, true>(a, occ, grid, st);
        else launch_occ<true, false, false>(a, occ, grid, st);
    } else if (far) {
        if (wide) launch_occ<false, true, true>(a, occ, grid, st);
        else launch_occ<false, true, false>(a, occ, grid, st);
    } else {
        if (wide) launch_occ<false, false, true>(a, occ, grid, st);
        else launch_occ<false, false, false>(a, occ, grid, st);
    }
    VLB_HIP(hipGetLastError());
    return grid;
}

void launch_project(const BakeArgs& a, int precision, int grid, hipStream_t st)
{
    grid = std::max(1, std::min(grid, a.ntiles));
    switch (precision) {
    case VLB_PREC_BF16: k_project<VLB_PREC_BF16><<<grid, 256, 0, st>>>(a); break;
    case VLB_PREC_FP16: k_project<VLB_PREC_FP16><<<grid, 256, 0, st>>>(a); break;
    case VLB_PREC_BF16_FAST: k_project<VLB_PREC_BF16_FAST><<<grid, 256, 0, st>>>(a); break;
    case VLB_PREC_FP16_FAST: k_project<VLB_PREC_FP16_FAST><<<grid, 256, 0, st>>>(a); break;
    default: k_project<VLB_PREC_FP32><<<grid, 256, 0, st>>>(a); break;
    }
    VLB_HIP(hipGetLastError());
}

void launch_merge(const MergeArgs& m, hipStream_t st)
{
    const int n = m.Ppad * 48;
    k_merge<<<(n + 255) / 256, 256, 0, st>>>(m);
    VLB_HIP(hipGetLastError());
}

void launch_trace_closest(const SceneView& sc, const float* org, const float* dir, int n,
                          float tmin, float tmax, int* prim, float* t, float* u, float* v,
                          uint32_t* spill, uint32_t stride, int grid, hipStream_t st)
{
    k_trace_closest<<<grid, 256, 0, st>>>(sc, org, dir, n, tmin, tmax, prim, t, u, v, spill,
                                          stride);
    VLB_HIP(hipGetLastError());
}

void launch_trace_occluded(const SceneView& sc, const float* org, const float* dir,
                           const float* tmax, int n, float tmin, uint8_t* occ, uint32_t* spill,
                           uint32_t stride, int grid, hipStream_t st)
{
    k_trace_occluded<<<grid, 256, 0, st>>>(sc, org, dir, tmax, n, tmin, occ, spill, stride);
    VLB_HIP(hipGetLastError());
}

namespace {
__global__ void k_copy_f32(float* __restrict__ dst, const float* __restrict__ src, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}
}  // namespace

void launch_copy_f32(float* dst, const float* src, size_t n, hipStream_t st)
{
    if (n == 0) return;
    const int grid = (int)std::min<size_t>((n + 255) / 256, 4096);
    k_copy_f32<<<grid, 256, 0, st>>>(dst, src, n);
    VLB_HIP(hipGetLastError());
}

}  // namespace vlb
