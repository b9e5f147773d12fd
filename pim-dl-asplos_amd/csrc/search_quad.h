// The closest centroids of one token in the 4 codebooks (2 from 17 centroids on) that a wave's lanes hold, one centroid a lane: shared by the
// search of few pairs (ccs_kernel.hip) and the launches that search where they gather (gather_few_kernel.hip).
#pragma once
#include <type_traits>

#include "pimdl_internal.h"

namespace pimdl {
namespace {

// floats of x that a lane needs, 16 bytes at a time where the caller knows the rows to be aligned (uniform)
template <int V>
__device__ __forceinline__ void quad_row(float (&r)[V], const float* p, bool aligned)
{
    if (V % 4 == 0 && aligned) {
#pragma unroll
        for (int t = 0; t < V; t += 4) {
            const float4 f = *reinterpret_cast<const float4*>(p + t);
            r[t] = f.x;
            r[t + 1] = f.y;
            r[t + 2] = f.z;
            r[t + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int t = 0; t < V; ++t) r[t] = p[t];
    }
}

// The distances are the reference's own (src/host/index_calc_host.cpp:8-53: every operation rounded on its own, dimensions ascending).
// Where only one centroid is within the hysteresis of the smallest distance the scan returns it whatever the order -- the
// subtraction that decides is the scan's --, else every group goes through its distances in the scan's order.
// xr, cr: this lane's codebook's part of the row and its centroid (any, past C); real: codebooks of the wave that exist (index 0 for
// the others).  The result is the same in every lane: 16 / PER bits per codebook, the first lowest.
template <int V, bool WIDE>
__device__ __forceinline__ uint32_t quad_scan(const float (&xr)[V], const float (&cr)[V], uint32_t C, uint32_t lane, uint32_t real)
{
    constexpr uint32_t GROUP = WIDE ? 32 : 16, PER = 64 / GROUP;
    const bool valid = lane % GROUP < C;
    float d = 0.0f;
#pragma unroll
    for (int t = 0; t < V; ++t) {
        const float diff = __fsub_rn(xr[t], cr[t]);
        d = __fadd_rn(d, __fmul_rn(diff, diff));
    }
    auto smaller = [](float a, float b) {  // (a NaN gives way)
        float r;
        asm("v_min_f32_e32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
        return r;
    };
    auto rotate = [](float f, auto nc) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), 0x120 + decltype(nc)::value, 0xf, 0xf, true));
    };
    float best = valid ? d : __builtin_inff();
    best = smaller(best, rotate(best, std::integral_constant<int, 8>{}));
    best = smaller(best, rotate(best, std::integral_constant<int, 4>{}));
    best = smaller(best, rotate(best, std::integral_constant<int, 2>{}));
    best = smaller(best, rotate(best, std::integral_constant<int, 1>{}));
    if constexpr (WIDE) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(best), __float_as_uint(best), false, false);
        best = smaller(__uint_as_float(s[0]), __uint_as_float(s[1]));
    }
    // (a distance that is NaN counts as near: with another the group is gone through)
    const uint64_t near = __builtin_amdgcn_ballot_w64(valid && !(__fsub_rn(d, best) > 1e-6f));
    uint32_t found[PER];
    bool several = false;
#pragma unroll
    for (uint32_t g = 0; g < PER; ++g) {
        const uint32_t m = (uint32_t)(near >> (GROUP * g)) & (WIDE ? ~0u : 0xFFFFu);
        several |= (m & (m - 1)) != 0;
        found[g] = m ? (uint32_t)__builtin_ctz(m) : 0u;
    }
    if (several) {
        float b = __shfl(d, lane & ~(GROUP - 1));
        uint32_t k = 0;
        for (uint32_t i = 1; i < C; ++i) {
            const float di = __shfl(d, (lane & ~(GROUP - 1)) + i);
            const bool take = __fsub_rn(b, di) > 1e-6f;
            b = take ? di : b;
            k = take ? i : k;
        }
#pragma unroll
        for (uint32_t g = 0; g < PER; ++g) found[g] = __builtin_amdgcn_readlane(k, GROUP * g);
    }
    uint32_t word = 0;
#pragma unroll
    for (uint32_t g = 0; g < PER; ++g)
        if (g < real) word |= found[g] << (16 / PER * g);
    return word;
}

}  // namespace
}  // namespace pimdl
