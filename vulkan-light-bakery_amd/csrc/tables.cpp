// tables.cpp -- host-side preparation shared by single bakes, batches and the
// request server: parameter validation, slice lengths, the server's probe
// order and shading parameters.  The ray and probe tables are built on the
// device (prepare.hip).
#include <math.h>
#include <string.h>

#include <algorithm>
#include <numeric>
#include <vector>

#include "vlb_internal.hpp"

namespace vlb {

namespace {

uint32_t expand10(uint32_t v)
{
    v &= 1023u;
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

}  // namespace

// Morton order of 3D points (stable on equal codes).
std::vector<uint32_t> morton_order(const float* xyz, size_t n)
{
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (size_t i = 0; i < n; ++i)
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], xyz[3 * i + a]);
            hi[a] = std::max(hi[a], xyz[3 * i + a]);
        }
    std::vector<uint32_t> code(n), order(n);
    for (size_t i = 0; i < n; ++i) {
        uint32_t q[3];
        for (int a = 0; a < 3; ++a) {
            float ext = hi[a] - lo[a];
            float x = ext > 0.0f ? (xyz[3 * i + a] - lo[a]) / ext * 1023.0f : 0.0f;
            q[a] = (uint32_t)std::min(1023.0f, std::max(0.0f, x));
        }
        code[i] = (expand10(q[0]) << 2) | (expand10(q[1]) << 1) | expand10(q[2]);
    }
    std::iota(order.begin(), order.end(), 0u);
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return code[a] < code[b]; });
    return order;
}

void validate(const vlb_bake_params& p)
{
    VLB_REQUIRE(p.num_probes >= 1 && p.probe_xyz, VLB_ERR_INVALID, "num_probes must be >= 1 with probe_xyz");
    VLB_REQUIRE(p.num_probes <= (1u << 26), VLB_ERR_INVALID, "num_probes too large");
    VLB_REQUIRE(p.sh_order == 2 || p.sh_order == 3, VLB_ERR_INVALID, "sh_order must be 2 or 3");
    VLB_REQUIRE(p.sh_constants == VLB_SH_LITERAL || p.sh_constants == VLB_SH_EXACT, VLB_ERR_INVALID,
                "bad sh_constants");
    VLB_REQUIRE(p.precision >= VLB_PREC_FP32 && p.precision <= VLB_PREC_FP16_FAST, VLB_ERR_INVALID,
                "bad precision");
    VLB_REQUIRE(p.shade_mode == VLB_SHADE_LAMBERT || p.shade_mode == VLB_SHADE_REFERENCE,
                VLB_ERR_INVALID, "bad shade_mode");
    VLB_REQUIRE(p.num_lights <= VLB_MAX_LIGHTS, VLB_ERR_INVALID, "too many lights");
    VLB_REQUIRE(p.num_lights == 0 || p.lights, VLB_ERR_INVALID, "lights pointer is NULL");
    for (uint32_t i = 0; i < p.num_lights; ++i)
        VLB_REQUIRE(p.lights[i].type == VLB_LIGHT_DIRECTIONAL || p.lights[i].type == VLB_LIGHT_POINT,
                    VLB_ERR_INVALID, "bad light type");
    if (p.dir_mode == VLB_DIRS_FIBONACCI) {
        VLB_REQUIRE(p.rays_per_probe >= 1 && p.rays_per_probe <= (1u << 26), VLB_ERR_INVALID,
                    "rays_per_probe out of range");
    } else if (p.dir_mode == VLB_DIRS_EQUIRECT) {
        VLB_REQUIRE(p.equirect_w >= 1 && p.equirect_h >= 1 &&
                        (uint64_t)p.equirect_w * p.equirect_h <= (1u << 26),
                    VLB_ERR_INVALID, "equirect size out of range");
    } else {
        throw Error{VLB_ERR_INVALID, "bad dir_mode"};
    }
    VLB_REQUIRE(p.t_min >= 0.0f && p.t_max > p.t_min, VLB_ERR_INVALID, "need 0 <= t_min < t_max");
    VLB_REQUIRE((uint64_t)p.num_probes * 48ull * 8ull < (1ull << 40), VLB_ERR_INVALID, "bake too large");
}


size_t scene_spill_bytes(const Scene& s, uint32_t stride)
{
    const uint32_t sb = stack_bound(s.depth);
    const uint32_t e = sb > (uint32_t)kLdsDepthMin ? sb - kLdsDepthMin : 0;
    return std::max<size_t>(16, (size_t)e * stride * 4);
}


Scene& find_scene(Context& ctx, uint32_t id)
{
    auto it = ctx.scenes.find(id);
    if (it == ctx.scenes.end()) throw Error{VLB_ERR_NOT_FOUND, "unknown scene id " + std::to_string(id)};
    return *it->second;
}

uint32_t rays_of(const vlb_bake_params& p)
{
    return p.dir_mode == VLB_DIRS_FIBONACCI ? p.rays_per_probe : p.equirect_w * p.equirect_h;
}

// Rays per projection slice: the caller's value rounded up to 64, else
// enough slices that a bake of npg probe groups gives the projection grid
// about two tiles per workgroup (an even chunk count per slice).
uint32_t slice_rays(const vlb_bake_params& p, uint32_t R, int npg, int pgrid)
{
    if (p.rays_per_slice) return (p.rays_per_slice + 63) & ~63u;
    uint64_t nsl = ((uint64_t)2 * pgrid + npg - 1) / npg;
    const uint64_t max_sl = (R + 31) / 32;
    nsl = std::max<uint64_t>(1, std::min(nsl, max_sl));
    return (uint32_t)(((R + nsl - 1) / nsl + 63) & ~63ull);
}

ShadeParams shade_params(const vlb_bake_params& p)
{
    ShadeParams sp;
    memset(&sp, 0, sizeof sp);
    sp.mode = p.shade_mode;
    sp.nlights = (int)p.num_lights;
    sp.shadow_bias = p.shadow_bias;
    sp.t_max = p.t_max;
    for (uint32_t i = 0; i < p.num_lights; ++i) sp.lights[i] = p.lights[i];
    sp.sky = p.sky;
    sp.ref = p.ref;
    return sp;
}

}  // namespace vlb
