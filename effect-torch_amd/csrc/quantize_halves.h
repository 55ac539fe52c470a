// The quantiser of gemm_h16's activation tiles for one (vector, 256-column stage), shared by the
// kernels that write such tiles: quantize_act.hip and the epilogue of kv_attention.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "kernels.h"

namespace et {

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}

// Activations for gemm_h16: per vector and 256-column stage, x = unit * X with unit = amax / (2^23 - 1) and
// X = 4096 * hi + lo: hi the nearest integer to X / 4096 (|hi| <= 2048: exact in a half float), lo the rest, written as the
// half float nearest to lo / 4096 - eleven significant bits of |lo| <= 2048, so off by half a unit of X at most (2^-24
// of the stage's largest value) and by less wherever lo is small. X is x / unit to within one rounding: the quotient by a multiplication with 1 / unit, corrected
// by its remainder. (A whole number lo from the product alone: relative error of a contraction with 20 vectors x 4096
// columns, 1e-7, before / now Q5_K 1.46 / 1.20, Q6_K 1.58 / 1.37, Q2_K 1.64 / 1.43; no slower.) The two products of a weight with these operands add
// up to X * w / 4096 in one accumulator. xsum[g] = unit * (sum of X over sub-block g).
// One wave per (vector, stage): lane `quad` holds columns 4 quad .. 4 quad + 3 of the stage. Blob
// layout: see tile_blob_bytes() in kernels.h.
__device__ __forceinline__ void quantize_halves_store(const float4& in, uint32_t v, uint32_t stage, uint32_t quad,
                                                      uint32_t vector_tiles, uint8_t* __restrict__ tiles) {
#pragma clang fp contract(off)  // the same bits in every file that includes this
    constexpr float kRange = 8388607.f;  // 2^23 - 1
    float amax = fmaxf(fmaxf(fabsf(in.x), fabsf(in.y)), fmaxf(fabsf(in.z), fabsf(in.w)));
    // over the wave: inside rows of 16 lanes with DPP, then the four rows through scalar registers
    amax = fmaxf(amax, dpp_f32<0xB1>(amax));   // quad_perm [1,0,3,2]
    amax = fmaxf(amax, dpp_f32<0x4E>(amax));   // quad_perm [2,3,0,1]
    amax = fmaxf(amax, dpp_f32<0x141>(amax));  // row_half_mirror
    amax = fmaxf(amax, dpp_f32<0x140>(amax));  // row_mirror
    {
        const int bits = __float_as_int(amax);
        amax = fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(bits, 0)),
                           __int_as_float(__builtin_amdgcn_readlane(bits, 16))),
                     fmaxf(__int_as_float(__builtin_amdgcn_readlane(bits, 32)),
                           __int_as_float(__builtin_amdgcn_readlane(bits, 48))));
    }
    const float inv = amax > 0.f ? kRange / amax : 0.f, unit = amax / kRange;
    const bool corrected = unit >= 1.17549435e-38f && unit < INFINITY;  // else 1 / unit or unit is no normal number
    const float values[4] = {in.x, in.y, in.z, in.w};
    float sum_hi = 0.f, sum_lo = 0.f;
    union {
        _Float16 h[4];
        uint2 words;
    } low, high;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float r = values[i] * inv;
        if (corrected) r = fmaf(fmaf(-r, unit, values[i]), inv, r);
        r = fminf(fmaxf(r, -kRange), kRange);
        const float hi = rintf(r * (1.0f / 4096.0f)), lo = fmaf(-4096.0f, hi, r);  // lo is exact
        sum_hi += hi;  // exact: whole numbers up to 2^16
        sum_lo += lo;
        constexpr int kPlace[4] = {0, 2, 1, 3};  // where the weight operands have column i of four (gemm_h16_device.h)
        low.h[kPlace[i]] = static_cast<_Float16>(lo * (1.0f / 4096.0f));
        high.h[kPlace[i]] = static_cast<_Float16>(hi);
    }
    sum_hi += dpp_f32<0xB1>(sum_hi);  // the eight lanes of a 32-column sub-block
    sum_lo += dpp_f32<0xB1>(sum_lo);
    sum_hi += dpp_f32<0x4E>(sum_hi);
    sum_lo += dpp_f32<0x4E>(sum_lo);
    sum_hi += dpp_f32<0x141>(sum_hi);
    sum_lo += dpp_f32<0x141>(sum_lo);
    uint8_t* blob = tiles + (static_cast<uint64_t>(stage) * vector_tiles + (v >> 5)) * tile_blob_bytes(2);
    // columns 4 quad .. + 3 = sub-block quad / 8, 16-column half, 8-column part, first or second four
    const uint32_t at = (quad >> 1) * 512u + (v & 31u) * 16u + (quad & 1u) * 8u;
    *reinterpret_cast<uint2*>(blob + at) = low.words;
    *reinterpret_cast<uint2*>(blob + 16384u + at) = high.words;
    float* tables = reinterpret_cast<float*>(blob + 32768u);
    if (quad == 0) tables[v & 31u] = unit;
    if ((quad & 7u) == 0) tables[32u + (quad >> 3) * 32u + (v & 31u)] = unit * fmaf(4096.0f, sum_hi, sum_lo);
}

}  // namespace et
