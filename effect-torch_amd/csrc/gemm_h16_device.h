// What the two kernels of the half-float contraction share (gemm_h16.hip, gemm_h16_wide.hip): the stage's layout in
// memory and LDS, the weight operands' arithmetic, and the matrices of a launch.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "decode_math.h"
#include "et_codecs.h"
#include "gemv_common.h"
#include "kernels.h"
#include "lds_handover.h"

namespace et {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kStageBlocks = 8;
constexpr float kPlaneRatio = 4096.0f;          // what the accumulators lack: the tiles hold hi and lo / 4096
constexpr uint32_t kBlob = tile_blob_bytes(2);  // in memory and in LDS
constexpr uint32_t kUnitAt = 32768u;            // unit[m]
constexpr uint32_t kSumsAt = 32768u + 128u;     // xsum[g][m]

// (scale, min) of Q4_K sub-block g (crates/runtime-cpu/src/quantized.rs:77-86).
__device__ __forceinline__ void q4k_scale_min(const uint4& header, uint32_t g, uint32_t& sc, uint32_t& mn) {
    const uint32_t shift = 8u * (g & 3u);
    const uint32_t s0 = (header.y >> shift) & 0xffu;
    const uint32_t s1 = (header.z >> shift) & 0xffu;
    const uint32_t s2 = (header.w >> shift) & 0xffu;
    sc = g < 4 ? (s0 & 63u) : ((s2 & 0x0fu) | ((s0 >> 6) << 4));
    mn = g < 4 ? (s1 & 63u) : ((s2 >> 4) | ((s1 >> 6) << 4));
}

// A row's share of a stage, as it lies in memory: a Q4_K super-block is d, dmin, scales[12], qs[128];
// a Q5_K one d, dmin, scales[12], qh[32] (the fifth bits: bit g of qh[c] belongs to column c of
// sub-block g), qs[128] (crates/runtime-cpu/src/quantized.rs:180-234).
// Super-blocks whose size is not a multiple of sixteen (Q6_K: 210 bytes = ql[128], qh[64], sixteen int8
// scales, d; Q3_K: 110 = hmask[32], qs[64], scales[12], d; Q2_K: 84 = scales[16], qs[64], d, dmin;
// crates/runtime-cpu/src/quantized.rs:117-176, 238-261) get an LDS row of the next multiple: every
// 16-byte chunk holds the stage's bytes at the same offset except the last one, which is taken from the
// stage's last sixteen bytes - so no copy reads past the stage (or the weight buffer). Q3_K and Q6_K
// stages start on 2-byte boundaries; global_load_lds takes such sources, more slowly.
template <int CODEC>
struct HalfStage {
    static_assert(CODEC == kQ2_K || CODEC == kQ3_K || CODEC == kQ4_K || CODEC == kQ5_K || CODEC == kQ6_K,
                  "the K-quants");
    static constexpr uint32_t kStageBytes = block_bytes(CODEC);            // in memory
    static constexpr uint32_t kRowBytes = (kStageBytes + 15u) / 16u * 16u;  // in LDS
    static constexpr uint32_t kQuantsAt = CODEC == kQ5_K ? 48u : 16u;       // Q4_K / Q5_K
    // where the stage's last sixteen bytes lie in the LDS row: d (and dmin) are read from there
    static constexpr uint32_t kTailAt = kRowBytes - 16u, kTailFrom = kStageBytes - 16u;
    // byte of the stage that LDS byte `within` (a multiple of 16) of the row holds
    static __device__ __forceinline__ uint32_t source_of(uint32_t within) {
        return kRowBytes != kStageBytes && within == kTailAt ? kTailFrom : within;
    }
    // LDS offset of stage byte `at` of the tail
    static constexpr uint32_t in_tail(uint32_t at) { return kTailAt + (at - kTailFrom); }
};

// Operands hold the columns of each four in the order 0, 2, 1, 3, as the activation tiles do (quantize_halves.h): the values
// of the even bytes of a dword fill a pair's halves without being moved, those of its odd bytes after one shift.
// Eight nibbles (two dwords of four, one per byte) as eight half floats times `scale`:
// 0x6400 | n is the half float 1024 + n, and (1024 + n) * scale - 1024 * scale, one fused
// multiply-add per pair, is n * scale exactly (1024 * scale <= 64512 is a half float).
template <int OFFSET = 0>
__device__ __forceinline__ v8h nibbles_times(uint32_t first, uint32_t second, v2h scale) {
    // OFFSET is subtracted from every byte first: (1024 + n) * scale - (1024 + OFFSET) * scale
    const v2h offset = {static_cast<_Float16>(1024.0f + OFFSET), static_cast<_Float16>(1024.0f + OFFSET)};
    union {
        uint32_t word[4];
        v2h pair[4];
        v8h all;
    } u;
    u.word[0] = __builtin_amdgcn_perm(0x64646464u, first, 0x04020400u);  // bytes 0, 2
    u.word[1] = __builtin_amdgcn_perm(0x64646464u, first, 0x04030401u);  // bytes 1, 3
    u.word[2] = __builtin_amdgcn_perm(0x64646464u, second, 0x04020400u);
    u.word[3] = __builtin_amdgcn_perm(0x64646464u, second, 0x04030401u);
#pragma unroll
    for (int i = 0; i < 4; i++) u.pair[i] = __builtin_elementwise_fma(u.pair[i], scale, -(offset * scale));
    return u.all;
}

// nibbles_times of the low (HIGH false) or high nibbles of two dwords of packed bytes: 0x6400 | n is 1024 + n, and with
// n four bits further up 0x5400 | 16 n is 64 + n; either is one v_and_or_b32 per pair. (Masks and v_perm_b32 as above: 26
// vector instructions per sixteen weights instead of 18.)
template <bool HIGH>
__device__ __forceinline__ v8h packed_nibbles_times(uint32_t first, uint32_t second, v2h scale) {
    // In registers: the instruction takes no literals, and the compiler would rather use two that do.
    uint32_t mask = HIGH ? 0x00f000f0u : 0x000f000fu, ones = HIGH ? 0x54005400u : 0x64006400u;
    asm("" : "+s"(mask));
    asm("" : "+v"(ones));
    constexpr float kOffset = HIGH ? 64.0f : 1024.0f;
    const v2h offset = {static_cast<_Float16>(kOffset), static_cast<_Float16>(kOffset)};
    union {
        uint32_t word[4];
        v2h pair[4];
        v8h all;
    } u;
    u.word[0] = (first & mask) | ones;
    u.word[1] = ((first >> 8) & mask) | ones;
    u.word[2] = (second & mask) | ones;
    u.word[3] = ((second >> 8) & mask) | ones;
#pragma unroll
    for (int i = 0; i < 4; i++) u.pair[i] = __builtin_elementwise_fma(u.pair[i], scale, -(offset * scale));
    return u.all;
}

// Eight bytes as eight half floats, (n - OFFSET) * scale in two exact steps (for offsets whose product
// with the scale a half float does not hold: 1028 * 31).
template <int OFFSET>
__device__ __forceinline__ v8h bytes_minus_times(uint32_t first, uint32_t second, v2h scale) {
#pragma clang fp contract(off)
    const v2h offset = {static_cast<_Float16>(1024.0f + OFFSET), static_cast<_Float16>(1024.0f + OFFSET)};
    union {
        uint32_t word[4];
        v2h pair[4];
        v8h all;
    } u;
    u.word[0] = __builtin_amdgcn_perm(0x64646464u, first, 0x04020400u);
    u.word[1] = __builtin_amdgcn_perm(0x64646464u, first, 0x04030401u);
    u.word[2] = __builtin_amdgcn_perm(0x64646464u, second, 0x04020400u);
    u.word[3] = __builtin_amdgcn_perm(0x64646464u, second, 0x04030401u);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const v2h centred = u.pair[i] - offset;
        u.pair[i] = centred * scale;
    }
    return u.all;
}

// Weight operands per sixteen columns: Q6_K splits its scale, Q2_K contracts its minima.
constexpr int weight_parts(int codec) { return codec == kQ6_K || codec == kQ2_K ? 2 : 1; }

// The matrices of one launch: contractions that share their activations (the q / k / v projections
// of a decode step) run as one grid over the row tiles of all of them.
struct Member {
    const uint8_t* weight;
    const float* bias;
    const float* residual;
    float* y;
    uint32_t rows;
    uint32_t first_tile;  // of the launch's row tiles
};
struct Group {
    Member member[kGemmGroupMost];
    uint32_t count;
    uint32_t row_tiles;  // of all members together
};

hipError_t gemm_h16_wide(int32_t codec, const Group& group, const uint8_t* tiles, uint32_t columns, uint32_t vectors,
                         uint32_t k_splits, float* partials, hipStream_t stream);

}  // namespace et
