// prepare.hip -- device side of the tables a bake starts from: the direction
// set on its Hilbert curve with the SH basis table (the reference generates
// both per ray, shaders/env_map.rgen:18-28, shaders/sh_common.h:8-22, 26-152)
// and the probes in Morton order.
//
// On the host these were the larger part of a one-shot bake: 97 ms of a 113 ms
// bake of 343 probes x 785,500 equirect rays (a double-precision basis of 16
// functions and a sort per ray), most of a millisecond at 4096 rays.  Here
// each is one thread per ray or probe around a library sort, bound by launch
// latency at a few thousand rays and by the sort's passes at a million: 0.18
// ms for 785,500 rays (keys 11 us, sort 150, rows 17).
//
// Every value is computed by the operation sequence of the host code it
// replaces (no contraction, correctly rounded divide and square root, the
// sines and cosines of an equirect grid from the host, W + H of each), so the
// tables are the same.  Only the sines and cosines of the Fibonacci angles are
// the device's, in double, then rounded to float.
#include <rocprim/device/device_radix_sort.hpp>

#include <math.h>

#include <vector>

#include "vlb_internal.hpp"

namespace vlb {
namespace {

// Position of a direction on a Hilbert curve over its octahedral map (pole =
// world +y), 2^16 cells per axis.
__device__ uint32_t direction_key(float x, float y, float z)
{
    const float s = fabsf(x) + fabsf(y) + fabsf(z);
    float u = s > 0.0f ? x / s : 0.0f, v = s > 0.0f ? z / s : 0.0f;
    if (y < 0.0f) {
        const float uu = (1.0f - fabsf(v)) * (u >= 0.0f ? 1.0f : -1.0f);
        const float vv = (1.0f - fabsf(u)) * (v >= 0.0f ? 1.0f : -1.0f);
        u = uu;
        v = vv;
    }
    constexpr uint32_t N = 1u << 16;
    const float fx = (u * 0.5f + 0.5f) * N, fy = (v * 0.5f + 0.5f) * N;
    uint32_t qx = (uint32_t)fminf((float)(N - 1), fmaxf(0.0f, fx));
    uint32_t qy = (uint32_t)fminf((float)(N - 1), fmaxf(0.0f, fy));
    uint32_t d = 0;
    for (uint32_t h = N / 2; h > 0; h /= 2) {
        const uint32_t rx = (qx & h) ? 1u : 0u, ry = (qy & h) ? 1u : 0u;
        d += h * h * ((3u * rx) ^ ry);
        if (ry == 0) {
            if (rx == 1) {
                qx = N - 1 - qx;
                qy = N - 1 - qy;
            }
            const uint32_t t = qx;
            qx = qy;
            qy = t;
        }
    }
    return d;
}

// How the directions of a set are made, by their canonical index.
struct DirGen {
    double golden, two_pi;                  // FIBONACCI (cols null)
    uint32_t R, W;
    const float2* cols;                     // EQUIRECT: (cos, sin) of phi_x,
    const float2* rows;                     // (sin, cos) of theta_y
};

__device__ __forceinline__ float3 direction(const DirGen& g, uint32_t i)
{
    if (!g.cols) {
        // fibonacci_dirs: y_i = 1 - (2i+1)/R, phi_i = i * pi * (3 - sqrt 5)
        const double y = 1.0 - (2.0 * i + 1.0) / (double)g.R;
        const double r = sqrt(fmax(0.0, 1.0 - y * y));
        // fmod(i * golden, two_pi): the remainder is representable, so one FMA
        // gives it exactly once the quotient is right
        const double a = (double)i * g.golden;
        const double q = trunc(a / g.two_pi);
        double phi = fma(-q, g.two_pi, a);
        if (phi < 0.0) phi = fma(-(q - 1.0), g.two_pi, a);
        else if (phi >= g.two_pi) phi = fma(-(q + 1.0), g.two_pi, a);
        return make_float3((float)(r * cos(phi)), (float)y, (float)(r * sin(phi)));
    }
    // equirect_dirs
    const uint32_t py = i / g.W;
    const float2 cp = g.cols[i - py * g.W], st = g.rows[py];
    const float a = st.x * cp.x, b = st.x * cp.y, c = st.y;
    const float l = sqrtf(a * a + b * b + c * c);
    return make_float3(a / l, c / l, b / l);
}

__global__ __launch_bounds__(256) void k_ray_keys(DirGen g, uint32_t* __restrict__ key,
                                                  uint32_t* __restrict__ val)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= g.R) return;
    const float3 d = direction(g, i);
    key[i] = direction_key(d.x, d.y, d.z);
    val[i] = i;
}

// Normalisation constants of sh_constants, in its order.
struct ShConst {
    double c0, c1, c2a, c20, c22, c33, c32, c31, c30, c3p2;
};

__device__ __forceinline__ uint16_t bf16_bits(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)(u >> 16);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// Sorted ray r (canonical index perm[r]; 0 is written for padding rays): its
// direction, made once more, and its row of the basis table ([ray octet]
// [coefficient][ray], times the ray's weight over wref); zeros for padding
// rays.
__global__ __launch_bounds__(256) void k_ray_rows(DirGen g, uint32_t Rpad, int K, int precision,
                                                  const float* __restrict__ row_weight, float weight,
                                                  double wref, ShConst c, float4* __restrict__ dirs,
                                                  int* __restrict__ perm, void* __restrict__ ytab)
{
    const uint32_t r = blockIdx.x * 256u + threadIdx.x;
    if (r >= Rpad) return;
    float4 d4 = make_float4(0.f, 0.f, 0.f, 0.f);
    double v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = 0.0;
    if (r < g.R) {
        const uint32_t i = (uint32_t)perm[r];
        const float3 d = direction(g, i);
        d4 = make_float4(d.x, d.y, d.z, 1.0f);
        const float w = row_weight ? row_weight[i / g.W] : weight;
        const double wr = (double)w / wref;
        // SH frame: world (x, z, y); order of terms as shaders/sh_common.h:26-152
        const double x = d4.x, y = d4.z, z = d4.y;
        v[0] = c.c0;
        v[1] = -c.c1 * y;
        v[2] = c.c1 * z;
        v[3] = -c.c1 * x;
        v[4] = c.c2a * x * y;
        v[5] = -c.c2a * y * z;
        v[6] = c.c20 * (-x * x - y * y + 2.0 * z * z);
        v[7] = -c.c2a * x * z;
        v[8] = c.c22 * (x * x - y * y);
        if (K > 9) {
            v[9] = -c.c33 * y * (3.0 * x * x - y * y);
            v[10] = c.c32 * x * y * z;
            v[11] = -c.c31 * y * (4.0 * z * z - x * x - y * y);
            v[12] = c.c30 * z * (2.0 * z * z - 3.0 * x * x - 3.0 * y * y);
            v[13] = -c.c31 * x * (4.0 * z * z - x * x - y * y);
            v[14] = c.c3p2 * z * (x * x - y * y);
            v[15] = -c.c33 * x * (x * x - 3.0 * y * y);
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] *= wr;
    } else {
        perm[r] = 0;
    }
    dirs[r] = d4;
    const size_t at = (size_t)(r >> 3) * 128 + (r & 7);
    const size_t lo = (size_t)Rpad * 16;
    const bool bf = precision == VLB_PREC_BF16 || precision == VLB_PREC_BF16_FAST;
    const bool split = precision == VLB_PREC_BF16 || precision == VLB_PREC_FP16;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (precision == VLB_PREC_FP32) {
            static_cast<float*>(ytab)[at + 8 * k] = (float)v[k];
            continue;
        }
        uint16_t* t = static_cast<uint16_t*>(ytab);
        if (bf) {
            const uint16_t hi = bf16_bits((float)v[k]);
            t[at + 8 * k] = hi;
            if (split)
                t[lo + at + 8 * k] = bf16_bits((float)(v[k] - (double)__uint_as_float((uint32_t)hi << 16)));
        } else {
            const _Float16 hi = (_Float16)(float)v[k];
            t[at + 8 * k] = __builtin_bit_cast(uint16_t, hi);
            if (split)
                t[lo + at + 8 * k] =
                    __builtin_bit_cast(uint16_t, (_Float16)(float)(v[k] - (double)(float)hi));
        }
    }
}

// --------------------------------------------------------- Morton order
constexpr int kBoundBlocks = 64;

// Bounds of one block's points: 3 minima, 3 maxima.
__global__ __launch_bounds__(256) void k_point_bounds(const float* __restrict__ xyz, uint32_t n,
                                                      float* __restrict__ part)
{
    __shared__ float sh[6][256];
    float b[6];
    for (int a = 0; a < 3; ++a) {
        b[a] = __builtin_huge_valf();
        b[3 + a] = -__builtin_huge_valf();
    }
    for (size_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u)
        for (int a = 0; a < 3; ++a) {
            const float x = xyz[3 * i + a];  // a NaN moves neither bound
            b[a] = x < b[a] ? x : b[a];
            b[3 + a] = b[3 + a] < x ? x : b[3 + a];
        }
    for (int a = 0; a < 6; ++a) sh[a][threadIdx.x] = b[a];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 6; ++a) {
                const float x = sh[a][threadIdx.x], y = sh[a][threadIdx.x + s];
                sh[a][threadIdx.x] = a < 3 ? (y < x ? y : x) : (x < y ? y : x);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = sh[threadIdx.x][0];
}

__device__ __forceinline__ uint32_t spread10(uint32_t v)
{
    v &= 1023u;
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// 30-bit Morton code of each point in the bounds (morton_order).
__global__ __launch_bounds__(256) void k_point_keys(const float* __restrict__ xyz, uint32_t n,
                                                    const float* __restrict__ part, int nparts,
                                                    uint32_t* __restrict__ key, uint32_t* __restrict__ val)
{
    __shared__ float b[6];
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float x = part[a];
        for (int p = 1; p < nparts; ++p) {
            const float y = part[p * 6 + a];
            x = a < 3 ? (y < x ? y : x) : (x < y ? y : x);
        }
        b[a] = x;
    }
    __syncthreads();
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
        const float ext = b[3 + a] - b[a];
        float x = ext > 0.0f ? (xyz[3 * (size_t)i + a] - b[a]) / ext * 1023.0f : 0.0f;
        x = 0.0f < x ? x : 0.0f;
        q[a] = (uint32_t)(x < 1023.0f ? x : 1023.0f);
    }
    key[i] = (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
    val[i] = i;
}

// Sorted probes, padded to npad with copies of the last.
__global__ __launch_bounds__(256) void k_probe_rows(const float* __restrict__ xyz, uint32_t n,
                                                    uint32_t npad, const uint32_t* __restrict__ order,
                                                    float4* __restrict__ probes, int* __restrict__ perm)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= npad) return;
    const uint32_t p = order[i < n ? i : n - 1];
    probes[i] = make_float4(xyz[3 * (size_t)p], xyz[3 * (size_t)p + 1], xyz[3 * (size_t)p + 2], 1.0f);
    perm[i] = i < n ? (int)p : -1;
}

inline uint32_t blocks(uint32_t n) { return (n + 255) / 256; }

// Scratch of a stable sort of n (key, index) pairs.
struct SortBufs {
    DevBuf key, val, key2, val2, tmp;
    size_t tmp_bytes = 0;
    SortBufs(Context& ctx, uint32_t n, unsigned bits)
    {
        key = dev_alloc(ctx, (size_t)n * 4);
        val = dev_alloc(ctx, (size_t)n * 4);
        key2 = dev_alloc(ctx, (size_t)n * 4);
        val2 = dev_alloc(ctx, (size_t)n * 4);
        VLB_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, key.as<uint32_t>(), key2.as<uint32_t>(),
                                          val.as<uint32_t>(), val2.as<uint32_t>(), (size_t)n, 0, bits,
                                          ctx.stream));
        tmp = dev_alloc(ctx, std::max<size_t>(tmp_bytes, 16));
    }
    void sort(uint32_t n, unsigned bits, hipStream_t st)
    {
        VLB_HIP(rocprim::radix_sort_pairs(tmp.p, tmp_bytes, key.as<uint32_t>(), key2.as<uint32_t>(),
                                          val.as<uint32_t>(), val2.as<uint32_t>(), (size_t)n, 0, bits, st));
    }
};

}  // namespace

void build_ray_table(Context& ctx, const vlb_bake_params& p, int K, uint32_t RS, RayTable& t)
{
    VLB_REQUIRE(RS >= 64 && RS % 64 == 0, VLB_ERR_INVALID, "rays per slice must be a multiple of 64");
    hipStream_t st = ctx.stream;
    const uint32_t R = rays_of(p);
    const double wref = 4.0 * M_PI / R;
    const int nslices = (int)((R + RS - 1) / RS);
    const uint32_t Rpad = (uint32_t)nslices * RS;
    const bool is16 = p.precision != VLB_PREC_FP32;
    const bool split = p.precision == VLB_PREC_BF16 || p.precision == VLB_PREC_FP16;

    t.R = R;
    t.RS = RS;
    t.Rpad = Rpad;
    t.nslices = nslices;
    t.wref = wref;
    t.K = K;
    t.precision = p.precision;
    t.dirs = dev_alloc(ctx, (size_t)Rpad * sizeof(float4));
    t.dir_perm = dev_alloc(ctx, (size_t)Rpad * sizeof(int));
    t.ytab = dev_alloc(ctx, (size_t)Rpad * 16 * (is16 ? sizeof(uint16_t) * (split ? 2 : 1) : sizeof(float)));

    // The sort's scratch is the basis table's memory, written last, and its
    // result the permutation: a table needs no more of the budget than itself
    // (but for the angles of an equirect grid).
    auto a256 = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t part = a256((size_t)R * 4);
    uint32_t *key = nullptr, *val = nullptr, *key2 = nullptr, *order = t.dir_perm.as<uint32_t>();
    size_t tmp_bytes = 0;
    VLB_HIP(rocprim::radix_sort_pairs(nullptr, tmp_bytes, key, key2, val, order, (size_t)R, 0, 32, st));
    DevBuf more;
    uint8_t* scratch = t.ytab.as<uint8_t>();
    if (3 * part + tmp_bytes > t.ytab.bytes) {  // a few dozen rays
        more = dev_alloc(ctx, 3 * part + tmp_bytes);
        scratch = more.as<uint8_t>();
    }
    key = reinterpret_cast<uint32_t*>(scratch);
    val = reinterpret_cast<uint32_t*>(scratch + part);
    key2 = reinterpret_cast<uint32_t*>(scratch + 2 * part);

    DirGen g{M_PI * (3.0 - sqrt(5.0)), 2.0 * M_PI, R, 1, nullptr, nullptr};
    DevBuf trig, roww;
    float weight = 0.0f;
    if (p.dir_mode == VLB_DIRS_FIBONACCI) {
        weight = (float)(4.0 * M_PI / R);
    } else {
        g.W = p.equirect_w;
        std::vector<float2> tab((size_t)g.W + p.equirect_h);
        std::vector<float> wrow(p.equirect_h);
        equirect_angles(g.W, p.equirect_h, tab.data(), wrow.data());
        trig = upload_vec(ctx, tab);
        roww = upload_vec(ctx, wrow);
        g.cols = trig.as<float2>();
        g.rows = g.cols + g.W;
        VLB_HIP(hipStreamSynchronize(st));  // tab and wrow are read
    }
    k_ray_keys<<<blocks(R), 256, 0, st>>>(g, key, val);
    VLB_HIP(hipGetLastError());
    VLB_HIP(rocprim::radix_sort_pairs(scratch + 3 * part, tmp_bytes, key, key2, val, order, (size_t)R, 0, 32, st));
    double c[10];
    sh_constants(p.sh_constants == VLB_SH_EXACT, c);
    const ShConst sc{c[0], c[1], c[2], c[3], c[4], c[5], c[6], c[7], c[8], c[9]};
    k_ray_rows<<<blocks(Rpad), 256, 0, st>>>(g, Rpad, K, p.precision, roww.as<float>(), weight, wref, sc,
                                             t.dirs.as<float4>(), t.dir_perm.as<int>(), t.ytab.p);
    VLB_HIP(hipGetLastError());
}

void build_probe_set(Context& ctx, const float* xyz, uint32_t P, ProbeSet& s)
{
    hipStream_t st = ctx.stream;
    const uint32_t Ppad = (P + 15) / 16 * 16;
    DevBuf raw = dev_alloc(ctx, (size_t)P * 3 * sizeof(float));
    VLB_HIP(hipMemcpyAsync(raw.p, xyz, (size_t)P * 3 * sizeof(float), hipMemcpyHostToDevice, st));
    SortBufs sb(ctx, P, 30);
    const int nb = (int)std::min<uint32_t>(kBoundBlocks, blocks(P));
    DevBuf part = dev_alloc(ctx, (size_t)nb * 6 * sizeof(float));
    k_point_bounds<<<nb, 256, 0, st>>>(raw.as<float>(), P, part.as<float>());
    k_point_keys<<<blocks(P), 256, 0, st>>>(raw.as<float>(), P, part.as<float>(), nb, sb.key.as<uint32_t>(),
                                            sb.val.as<uint32_t>());
    VLB_HIP(hipGetLastError());
    sb.sort(P, 30, st);
    s.P = (int)P;
    s.Ppad = (int)Ppad;
    s.probes = dev_alloc(ctx, (size_t)Ppad * sizeof(float4));
    s.probe_perm = dev_alloc(ctx, (size_t)Ppad * sizeof(int));
    k_probe_rows<<<blocks(Ppad), 256, 0, st>>>(raw.as<float>(), P, Ppad, sb.val2.as<uint32_t>(),
                                               s.probes.as<float4>(), s.probe_perm.as<int>());
    VLB_HIP(hipGetLastError());
}

}  // namespace vlb
