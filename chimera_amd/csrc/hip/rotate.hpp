// FhtKac rotation of one 128-float row by one wave64 (rotator.hpp:281-334,
// fht_avx.cpp:396-591): lane l holds elements l and l + 64.
#pragma once

#include "common.hpp"

namespace chimera {

// One butterfly stage with stride h < 64 across the lanes of a wave: the
// lower element of each pair becomes a + b and the upper a - b (FFHT runs
// stages 1, 2, 4, ... in that order), each as its partner's value plus or
// minus its own. The exchanges run on the vector ALU (DPP within a row of 16
// lanes, the lane swaps past it), except h = 4, which no DPP pattern gives.
template <int kH>
__device__ __forceinline__ float butterfly_lanes(float x, int l) {
    const uint32_t bits = __float_as_uint(x);
    if constexpr (kH == 16 || kH == 32) {
        // the swap leaves the lower lane's value in [0] and the upper lane's in [1]
        const auto r = kH == 16 ? __builtin_amdgcn_permlane16_swap(bits, bits, false, false)
                                : __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        const float lo = __uint_as_float(r[0]), hi = __uint_as_float(r[1]);
        return (l & kH) ? lo - hi : lo + hi;
    } else {
        int p;
        if constexpr (kH == 1)
            p = __builtin_amdgcn_mov_dpp(static_cast<int>(bits), 0xB1, 0xF, 0xF, true);  // quad_perm 1 0 3 2
        else if constexpr (kH == 2)
            p = __builtin_amdgcn_mov_dpp(static_cast<int>(bits), 0x4E, 0xF, 0xF, true);  // quad_perm 2 3 0 1
        else if constexpr (kH == 4)
            p = __builtin_amdgcn_ds_swizzle(static_cast<int>(bits), 0x101F);             // lane ^ 4
        else
            p = __builtin_amdgcn_mov_dpp(static_cast<int>(bits), 0x128, 0xF, 0xF, true);  // row_ror:8
        const float s = (l & kH) ? -x : x;
        return __int_as_float(p) + s;
    }
}

__device__ __forceinline__ float fwht64_lanes(float x, int l) {
    x = butterfly_lanes<1>(x, l);
    x = butterfly_lanes<2>(x, l);
    x = butterfly_lanes<4>(x, l);
    x = butterfly_lanes<8>(x, l);
    x = butterfly_lanes<16>(x, l);
    return butterfly_lanes<32>(x, l);
}

// Element j changes sign when bit j % 8 of byte j / 8 of the round's 16
// flip bytes is set (rotator.hpp:129-172).
__device__ __forceinline__ float flip_sign(float x, const uint8_t* f, int j) {
    return ((f[j >> 3] >> (j & 7)) & 1u) ? -x : x;
}

// Rotates (x0, x1) = elements (l, l + 64) in place. `flips` holds the 64
// flip bytes (4 rounds x 16), `fac` = 1/sqrtf(trunc_dim), `pow2` is
// trunc_dim == 128 (dim == 128); otherwise the KAC-walk variant with the
// final 0.25 scale runs.
__device__ __forceinline__ void fht_kac_rotate(float& x0, float& x1, const uint8_t* flips, float fac, bool pow2,
                                               int l) {
#pragma unroll
    for (int round = 0; round < 4; ++round) {
        const uint8_t* f = flips + round * (kDim / 8);
        x0 = flip_sign(x0, f, l);
        x1 = flip_sign(x1, f, l + 64);
        if (pow2) {
            x0 = fwht64_lanes(x0, l);
            x1 = fwht64_lanes(x1, l);
            const float a = x0, b = x1;  // stride-64 stage, last
            x0 = a + b;
            x1 = a - b;
            x0 = x0 * fac;
            x1 = x1 * fac;
        } else {
            if (round & 1) {
                x1 = fwht64_lanes(x1, l) * fac;
            } else {
                x0 = fwht64_lanes(x0, l) * fac;
            }
            const float a = x0, b = x1;  // kacs_walk
            x0 = a + b;
            x1 = a - b;
        }
    }
    if (!pow2) {
        x0 = x0 * 0.25F;
        x1 = x1 * 0.25F;
    }
}

}  // namespace chimera
