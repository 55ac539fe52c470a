// What the kernels that fold weights with three-limb activations on v_dot4_i32_i8 share (gemv_limb.hip,
// gemv_step.hip): the activations' limbs and, per codec, what a lane loads of a row and how it folds it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gemv_common.h"

namespace et {
namespace {

constexpr int kChunk = 64;                       // columns a lane owns
constexpr uint32_t kSliceColumns = 64 * kChunk;  // columns a wave covers
constexpr uint32_t kSliceQuads = kSliceColumns / 4;

// Per-vector lane state: the limbs of the lane's 64 activations and their sums.
struct XLimbs {
    int limb[3][16];  // limb[k][j]: bytes = limb k of elements 4j..4j+3 of the chunk;
                      // limb 0 is the least significant (weight 1), limb 2 the most (65536)
    float s;          // value of one unit of limb 0
    float sum[2];     // exact f32 sums of elements 0..31 and 32..63
    // Codecs whose lanes own four separate 16-column runs (Q6_K) use these instead of s / sum:
    float s_pair[2];  // unit of runs 0, 1 and of runs 2, 3 (they lie in two 64-column chunks)
    int bias[4][3];   // -offset * (sum of the limb bytes of run g): where the integer dots start
    float run_sum[4]; // sum of the (quantised) activations of run g, for codecs with block minima
};

constexpr float kLimbRange = 8323072.0f;  // 127 * 2^16: |X| <= this

// LDS slot (in 16-byte units) of limb unit u = 4*chunk + j: the XOR spreads the
// eight lanes that read in one pass over all banks; writes of consecutive dwords
// stay conflict-free because it only permutes within aligned groups of four units.
__device__ __forceinline__ uint32_t limb_slot(uint32_t u) { return u ^ ((u >> 3) & 3u); }

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

struct alignas(16) StageMemory {
    uint32_t limbs[3][kSliceQuads];  // [limb][swizzled dword]
    float unit[64];
    float sum[2][64];
};

// Splits one float4 of a slice into limbs and stores them in LDS. Float4 number f
// of the slice belongs to thread f % THREADS; sixteen consecutive lanes (one DPP
// row) hold one 64-column chunk, so the chunk's maximum and its two 32-column
// sums are folded across lanes with DPP. Must be called by whole waves.
//
// X = rint(x * inv) is an exact integer of at most 24 bits. Adding 0x8080 and
// flipping the top bit of the two low bytes turns its bytes into balanced
// digits: X = 65536*x1 + 256*x2 + x3 with every x_k a signed byte.
__device__ __forceinline__ void stage_quad(StageMemory& stage, float4 v, uint32_t f) {
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = fmaxf(amax, dpp<0xB1>(amax));   // quad_perm [1,0,3,2]
    amax = fmaxf(amax, dpp<0x4E>(amax));   // quad_perm [2,3,0,1]
    amax = fmaxf(amax, dpp<0x141>(amax));  // row_half_mirror
    amax = fmaxf(amax, dpp<0x140>(amax));  // row_mirror: all 16 lanes hold the chunk's max
    float total = (v.x + v.y) + (v.z + v.w);
    total += dpp<0xB1>(total);
    total += dpp<0x4E>(total);
    total += dpp<0x141>(total);  // sum over the lane's 8-lane half = 32 columns
    // 1 ulp of the reciprocal moves |X| by at most 1, far inside the headroom of the limbs.
    const bool nonzero = amax >= 1e-30f;
    const float inv = nonzero ? kLimbRange * __builtin_amdgcn_rcpf(amax) : 0.f;
    const float unit = nonzero ? amax * (1.0f / kLimbRange) : 0.f;
    const int x0 = static_cast<int>(rintf(v.x * inv)) + 0x8080;
    const int x1 = static_cast<int>(rintf(v.y * inv)) + 0x8080;
    const int x2 = static_cast<int>(rintf(v.z * inv)) + 0x8080;
    const int x3 = static_cast<int>(rintf(v.w * inv)) + 0x8080;
    // 4x3 byte transpose: limb k of the four elements into one dword.
    const uint32_t a = __builtin_amdgcn_perm(x1, x0, 0x05010400u);  // x0.b0 x1.b0 x0.b1 x1.b1
    const uint32_t b = __builtin_amdgcn_perm(x3, x2, 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(x1, x0, 0x0c0c0602u);  // x0.b2 x1.b2 0 0
    const uint32_t d = __builtin_amdgcn_perm(x3, x2, 0x0c0c0602u);
    const uint32_t limb0 = __builtin_amdgcn_perm(b, a, 0x05040100u) ^ 0x80808080u;
    const uint32_t limb1 = __builtin_amdgcn_perm(b, a, 0x07060302u) ^ 0x80808080u;
    const uint32_t limb2 = __builtin_amdgcn_perm(d, c, 0x05040100u);
    const uint32_t slot = limb_slot(f >> 2) * 4u + (f & 3u);
    stage.limbs[0][slot] = limb0;
    stage.limbs[1][slot] = limb1;
    stage.limbs[2][slot] = limb2;
    const uint32_t chunk = f >> 4;
    if ((f & 15u) == 0u) stage.unit[chunk] = unit;
    if ((f & 7u) == 0u) stage.sum[(f >> 3) & 1u][chunk] = total;
}

__device__ __forceinline__ void load_limbs(const StageMemory& stage, uint32_t lane, bool active,
                                           XLimbs& out) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint4 v = *reinterpret_cast<const uint4*>(&stage.limbs[k][limb_slot(4u * lane + j) * 4u]);
            out.limb[k][4 * j + 0] = active ? static_cast<int>(v.x) : 0;
            out.limb[k][4 * j + 1] = active ? static_cast<int>(v.y) : 0;
            out.limb[k][4 * j + 2] = active ? static_cast<int>(v.z) : 0;
            out.limb[k][4 * j + 3] = active ? static_cast<int>(v.w) : 0;
        }
    }
    out.s = active ? stage.unit[lane] : 0.f;
    out.sum[0] = active ? stage.sum[0][lane] : 0.f;
    out.sum[1] = active ? stage.sum[1][lane] : 0.f;
}

// s * (D0 + 256*D1 + 65536*D2) for the integer dots D_k of the three limbs.
__device__ __forceinline__ float limb_value(const XLimbs& x, int d0, int d1, int d2) {
    float v = static_cast<float>(d0);
    v = fmaf(256.0f, static_cast<float>(d1), v);
    v = fmaf(65536.0f, static_cast<float>(d2), v);
    return x.s * v;
}

// ---------------------------------------------------------------------------
// Codec traits: what a lane loads per row and how it folds it with the limbs.
// ---------------------------------------------------------------------------

struct Q4KLimb {
    static constexpr uint32_t kBlockColumns = 256u, kBlockBytes = 144u;
    static constexpr bool kLdsCopies = true;     // its weights can come through LDS copies
    static constexpr bool kCopiesInTurn = true;  // ... on gemv_limb_turns_kernel
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_limbs(stage, lane, active, out);
    }
    struct Lane {
        uint32_t offset;  // byte offset of the lane's block within a row
        uint32_t p;       // pair within the block
    };
    struct Data {
        uint4 header;  // d, dmin, scales[12]
        uint4 q[2];    // the pair's 32 bytes of quants
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 8) * 144u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) {
        return Lane{(chunk >> 2) * 144u, chunk & 3u};
    }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        const uint8_t* base = row + lane.offset;
        data.header = *reinterpret_cast<const uint4*>(base);
        data.q[0] = *reinterpret_cast<const uint4*>(base + 16 + 32 * lane.p);
        data.q[1] = *reinterpret_cast<const uint4*>(base + 32 + 32 * lane.p);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane& lane,
                                                const XLimbs (&x)[M], float (&value)[M]) {
        const uint32_t w[8] = {data.q[0].x, data.q[0].y, data.q[0].z, data.q[0].w,
                               data.q[1].x, data.q[1].y, data.q[1].z, data.q[1].w};
        int lo[M][3], hi[M][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int k = 0; k < 3; k++) lo[m][k] = hi[m][k] = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // low nibbles: elements 4j..4j+3 of sub-block 2p; high nibbles: of sub-block 2p+1
            const int ql = static_cast<int>(w[j] & 0x0f0f0f0fu);
            const int qh = static_cast<int>((w[j] >> 4) & 0x0f0f0f0fu);
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    lo[m][k] = __builtin_amdgcn_sdot4(ql, x[m].limb[k][j], lo[m][k], false);
                    hi[m][k] = __builtin_amdgcn_sdot4(qh, x[m].limb[k][8 + j], hi[m][k], false);
                }
        }
        // (scale, min) of sub-blocks 2p, 2p+1: crates/runtime-cpu/src/quantized.rs:77-86
        const uint32_t shift = (lane.p & 1u) * 16u;
        const uint32_t a = data.header.y >> shift, b = data.header.z >> shift, c = data.header.w >> shift;
        uint32_t sc, mn;
        if (lane.p < 2) {
            sc = a & 0x3f3fu;
            mn = b & 0x3f3fu;
        } else {
            sc = (c & 0x0f0fu) | ((a >> 2) & 0x3030u);
            mn = ((c >> 4) & 0x0f0fu) | ((b >> 2) & 0x3030u);
        }
        const float sc_lo = static_cast<float>(sc & 0xffu), sc_hi = static_cast<float>((sc >> 8) & 0xffu);
        const float m_lo = static_cast<float>(mn & 0xffu), m_hi = static_cast<float>((mn >> 8) & 0xffu);
        const float d = half_bits_to_float(data.header.x & 0xffffu);
        const float dmin = half_bits_to_float(data.header.x >> 16);
#pragma unroll
        for (int m = 0; m < M; m++) {
            // sub-block scales first, limb weights second, one f32 scale last
            // (as floats: the dots are below 2^17 and convert exactly; a 32-bit
            // integer multiply would run at quarter rate)
            const float i1 = fmaf(sc_hi, static_cast<float>(hi[m][0]), sc_lo * static_cast<float>(lo[m][0]));
            const float i2 = fmaf(sc_hi, static_cast<float>(hi[m][1]), sc_lo * static_cast<float>(lo[m][1]));
            const float i3 = fmaf(sc_hi, static_cast<float>(hi[m][2]), sc_lo * static_cast<float>(lo[m][2]));
            const float pos = x[m].s * fmaf(65536.0f, i3, fmaf(256.0f, i2, i1));
            const float neg = fmaf(m_lo, x[m].sum[0], m_hi * x[m].sum[1]);
            value[m] = d * pos - dmin * neg;
        }
    }
};

// Q5_K (decode_q5_k, crates/runtime-cpu/src/quantized.rs:203-234): Q4_K's layout with a fifth bit per
// value in qh[32] between the scales and the nibbles - bit g of qh[i] belongs to element i of
// sub-block g. 176 bytes per block, every field 16-byte aligned.
struct Q5KLimb {
    static constexpr uint32_t kBlockColumns = 256u, kBlockBytes = 176u;
    static constexpr bool kLdsCopies = true;     // its weights can come through LDS copies
    static constexpr bool kCopiesInTurn = true;  // ... on gemv_limb_turns_kernel
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_limbs(stage, lane, active, out);
    }
    struct Lane {
        uint32_t offset;  // byte offset of the lane's block within a row
        uint32_t p;       // pair within the block
    };
    struct Data {
        uint4 header;  // d, dmin, scales[12]
        uint4 h[2];    // qh[32]: the fifth bits of all eight sub-blocks
        uint4 q[2];    // the pair's 32 bytes of nibbles
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 8) * 176u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) {
        return Lane{(chunk >> 2) * 176u, chunk & 3u};
    }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        const uint8_t* base = row + lane.offset;
        data.header = *reinterpret_cast<const uint4*>(base);
        data.h[0] = *reinterpret_cast<const uint4*>(base + 16);
        data.h[1] = *reinterpret_cast<const uint4*>(base + 32);
        data.q[0] = *reinterpret_cast<const uint4*>(base + 48 + 32 * lane.p);
        data.q[1] = *reinterpret_cast<const uint4*>(base + 64 + 32 * lane.p);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane& lane,
                                                const XLimbs (&x)[M], float (&value)[M]) {
        const uint32_t w[8] = {data.q[0].x, data.q[0].y, data.q[0].z, data.q[0].w,
                               data.q[1].x, data.q[1].y, data.q[1].z, data.q[1].w};
        const uint32_t h[8] = {data.h[0].x, data.h[0].y, data.h[0].z, data.h[0].w,
                               data.h[1].x, data.h[1].y, data.h[1].z, data.h[1].w};
        const uint32_t bit = 2u * lane.p;  // sub-blocks 2p and 2p + 1
        int lo[M][3], hi[M][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int k = 0; k < 3; k++) lo[m][k] = hi[m][k] = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // low nibbles: elements 4j..4j+3 of sub-block 2p; high nibbles: of sub-block 2p+1
            const uint32_t fifth = h[j] >> bit;
            const int ql = static_cast<int>((w[j] & 0x0f0f0f0fu) | ((fifth & 0x01010101u) << 4));
            const int qh = static_cast<int>(((w[j] >> 4) & 0x0f0f0f0fu) | ((fifth & 0x02020202u) << 3));
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    lo[m][k] = __builtin_amdgcn_sdot4(ql, x[m].limb[k][j], lo[m][k], false);
                    hi[m][k] = __builtin_amdgcn_sdot4(qh, x[m].limb[k][8 + j], hi[m][k], false);
                }
        }
        // (scale, min) of sub-blocks 2p, 2p+1: crates/runtime-cpu/src/quantized.rs:77-86
        const uint32_t shift = (lane.p & 1u) * 16u;
        const uint32_t a = data.header.y >> shift, b = data.header.z >> shift, c = data.header.w >> shift;
        uint32_t sc, mn;
        if (lane.p < 2) {
            sc = a & 0x3f3fu;
            mn = b & 0x3f3fu;
        } else {
            sc = (c & 0x0f0fu) | ((a >> 2) & 0x3030u);
            mn = ((c >> 4) & 0x0f0fu) | ((b >> 2) & 0x3030u);
        }
        const float sc_lo = static_cast<float>(sc & 0xffu), sc_hi = static_cast<float>((sc >> 8) & 0xffu);
        const float m_lo = static_cast<float>(mn & 0xffu), m_hi = static_cast<float>((mn >> 8) & 0xffu);
        const float d = half_bits_to_float(data.header.x & 0xffffu);
        const float dmin = half_bits_to_float(data.header.x >> 16);
#pragma unroll
        for (int m = 0; m < M; m++) {
            // sub-block scales first, limb weights second, one f32 scale last
            // (as floats: the dots are below 2^17 and convert exactly; a 32-bit
            // integer multiply would run at quarter rate)
            const float i1 = fmaf(sc_hi, static_cast<float>(hi[m][0]), sc_lo * static_cast<float>(lo[m][0]));
            const float i2 = fmaf(sc_hi, static_cast<float>(hi[m][1]), sc_lo * static_cast<float>(lo[m][1]));
            const float i3 = fmaf(sc_hi, static_cast<float>(hi[m][2]), sc_lo * static_cast<float>(lo[m][2]));
            const float pos = x[m].s * fmaf(65536.0f, i3, fmaf(256.0f, i2, i1));
            const float neg = fmaf(m_lo, x[m].sum[0], m_hi * x[m].sum[1]);
            value[m] = d * pos - dmin * neg;
        }
    }
};

struct __attribute__((packed, aligned(4))) Dwords9 {
    uint32_t v[9];
};
struct __attribute__((packed, aligned(4))) Dwords17 {
    uint32_t v[17];
};

// Q4_0: two 18-byte blocks = 36 bytes = 9 dwords (dword aligned when columns % 64 == 0).
struct Q40Limb {
    static constexpr uint32_t kBlockColumns = 32u, kBlockBytes = 18u;
    static constexpr bool kLdsCopies = true;     // its weights can come through LDS copies
    static constexpr bool kCopiesInTurn = true;  // ... on gemv_limb_turns_kernel
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_limbs(stage, lane, active, out);
    }
    struct Lane {
        uint32_t offset;
    };
    struct Data {
        Dwords9 raw;
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 5) * 18u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) { return Lane{chunk * 36u}; }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        data.raw = *reinterpret_cast<const Dwords9*>(row + lane.offset);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane&, const XLimbs (&x)[M],
                                                float (&value)[M]) {
        const uint32_t* w = data.raw.v;
        int da_[M][3], db_[M][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int k = 0; k < 3; k++) da_[m][k] = db_[m][k] = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // block A: bytes 2..17 of the pair (2 bytes off dword alignment); block B: bytes 20..35.
            // Byte j's low nibble is element j, its high nibble element j + 16.
            const uint32_t qa = __builtin_amdgcn_alignbit(w[i + 1], w[i], 16);
            const uint32_t qb = w[5 + i];
            const int al = static_cast<int>(qa & 0x0f0f0f0fu), ah = static_cast<int>((qa >> 4) & 0x0f0f0f0fu);
            const int bl = static_cast<int>(qb & 0x0f0f0f0fu), bh = static_cast<int>((qb >> 4) & 0x0f0f0f0fu);
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    da_[m][k] = __builtin_amdgcn_sdot4(al, x[m].limb[k][i], da_[m][k], false);
                    da_[m][k] = __builtin_amdgcn_sdot4(ah, x[m].limb[k][4 + i], da_[m][k], false);
                    db_[m][k] = __builtin_amdgcn_sdot4(bl, x[m].limb[k][8 + i], db_[m][k], false);
                    db_[m][k] = __builtin_amdgcn_sdot4(bh, x[m].limb[k][12 + i], db_[m][k], false);
                }
        }
        const float da = half_bits_to_float(w[0] & 0xffffu);
        const float db = half_bits_to_float(w[4] >> 16);
#pragma unroll
        for (int m = 0; m < M; m++) {
            // value = d * (nibble - 8): the -8 meets the chunk's activation sums once
            const float va = limb_value(x[m], da_[m][0], da_[m][1], da_[m][2]) - 8.f * x[m].sum[0];
            const float vb = limb_value(x[m], db_[m][0], db_[m][1], db_[m][2]) - 8.f * x[m].sum[1];
            value[m] = da * va + db * vb;
        }
    }
};

// Q8_0: two 34-byte blocks = 68 bytes = 17 dwords (dword aligned when columns % 64 == 0).
struct Q80Limb {
    static constexpr uint32_t kBlockColumns = 32u, kBlockBytes = 34u;
    static constexpr bool kLdsCopies = true;     // its weights can come through LDS copies
    static constexpr bool kCopiesInTurn = true;  // ... on gemv_limb_turns_kernel
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_limbs(stage, lane, active, out);
    }
    struct Lane {
        uint32_t offset;
    };
    struct Data {
        Dwords17 raw;
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 5) * 34u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) { return Lane{chunk * 68u}; }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        data.raw = *reinterpret_cast<const Dwords17*>(row + lane.offset);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane&, const XLimbs (&x)[M],
                                                float (&value)[M]) {
        const uint32_t* w = data.raw.v;
        int da_[M][3], db_[M][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int k = 0; k < 3; k++) da_[m][k] = db_[m][k] = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int qa = static_cast<int>(__builtin_amdgcn_alignbit(w[i + 1], w[i], 16));  // bytes 2..33
            const int qb = static_cast<int>(w[9 + i]);                                        // bytes 36..67
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    da_[m][k] = __builtin_amdgcn_sdot4(qa, x[m].limb[k][i], da_[m][k], false);
                    db_[m][k] = __builtin_amdgcn_sdot4(qb, x[m].limb[k][8 + i], db_[m][k], false);
                }
        }
        const float da = half_bits_to_float(w[0] & 0xffffu);
        const float db = half_bits_to_float(w[8] >> 16);
#pragma unroll
        for (int m = 0; m < M; m++)
            value[m] = da * limb_value(x[m], da_[m][0], da_[m][1], da_[m][2]) +
                       db * limb_value(x[m], db_[m][0], db_[m][1], db_[m][2]);
    }
};

// Sixteen bytes from an address that is only 2-byte aligned (odd Q6_K blocks start at 210 * b).
#pragma clang diagnostic ignored "-Walign-mismatch"
typedef uint4 __attribute__((aligned(2))) uint4_a2;
typedef uint2 __attribute__((aligned(2))) uint2_a2;

// Activations of a lane that owns four 16-column runs of a 256-column block (Q2_K, Q3_K, Q6_K):
// lane (block b, half, j) takes runs g = 0..3 = 16-column units 16b + 8*half + 2g + j of the slice.
// OFFSET is what the codec subtracts from every quant: the integer dots start at -OFFSET * (sum of
// the run's limb bytes), so that sum (q - OFFSET) x needs no per-row work.
template <int OFFSET>
__device__ __forceinline__ void load_run_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                     XLimbs& out) {
    const uint32_t first = 16u * (lane >> 2) + 8u * ((lane >> 1) & 1u) + (lane & 1u);
    int totals[4][3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint4 v = *reinterpret_cast<const uint4*>(&stage.limbs[k][limb_slot(first + 2u * g) * 4u]);
            const int words[4] = {static_cast<int>(v.x), static_cast<int>(v.y), static_cast<int>(v.z),
                                  static_cast<int>(v.w)};
            int total = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                out.limb[k][4 * g + i] = active ? words[i] : 0;
                total = __builtin_amdgcn_sdot4(0x01010101, out.limb[k][4 * g + i], total, false);
            }
            totals[g][k] = total;
            out.bias[g][k] = -OFFSET * total;
        }
    }
    const uint32_t chunk = 4u * (lane >> 2) + 2u * ((lane >> 1) & 1u);
    out.s_pair[0] = active ? stage.unit[chunk] : 0.f;
    out.s_pair[1] = active ? stage.unit[chunk + 1u] : 0.f;
#pragma unroll
    for (int g = 0; g < 4; g++)
        out.run_sum[g] = out.s_pair[g >> 1] * fmaf(65536.0f, static_cast<float>(totals[g][2]),
                                                   fmaf(256.0f, static_cast<float>(totals[g][1]),
                                                        static_cast<float>(totals[g][0])));
    out.s = 0.f;
    out.sum[0] = out.sum[1] = 0.f;
}

// Q6_K (decode_q6_k, crates/runtime-cpu/src/quantized.rs:238-261): 210 bytes per 256 values -
// ql[128] low nibbles, qh[64] two high bits, scales[16] int8 per 16 values, d. Value e = half*128 +
// quarter*32 + i of a block is d * scale[half*8 + quarter*2 + i/16] * (q - 32) with
// q = nibble(ql[half*64 + (quarter & 1)*32 + i], quarter >> 1) | ((qh[half*32 + i] >> 2*quarter) & 3) << 4.
// A lane takes (half, j = i / 16) of a block: the four 16-column runs quarter = 0..3, each with ONE
// scale, out of exactly 48 bytes of quants - three 16-byte loads, nothing read twice. Its 64 columns
// are not consecutive, so it gathers its activation limbs run by run (load_activations).
struct Q6KLimb {
    static constexpr uint32_t kBlockColumns = 256u, kBlockBytes = 210u;
    static constexpr bool kLdsCopies = false;    // gemv_limb_kernel only: a share of 14336 rows (56 x 3360 bytes) does not fit LDS
    struct Lane {
        uint32_t offset;  // byte offset of the lane's block within a row
        uint32_t half, j;
    };
    struct Data {
        uint4 qa, qb, qh;  // ql[half*64 + 16j ..], ql[half*64 + 32 + 16j ..], qh[half*32 + 16j ..]
        uint2 scales;      // scales[half*8 .. half*8 + 8]
        uint32_t d;        // f16 bits
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 8) * 210u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) {
        return Lane{(chunk >> 2) * 210u, (chunk >> 1) & 1u, chunk & 1u};
    }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        const uint8_t* base = row + lane.offset;
        data.qa = *reinterpret_cast<const uint4_a2*>(base + 64u * lane.half + 16u * lane.j);
        data.qb = *reinterpret_cast<const uint4_a2*>(base + 64u * lane.half + 32u + 16u * lane.j);
        data.qh = *reinterpret_cast<const uint4_a2*>(base + 128u + 32u * lane.half + 16u * lane.j);
        data.scales = *reinterpret_cast<const uint2_a2*>(base + 192u + 8u * lane.half);
        data.d = *reinterpret_cast<const uint16_t*>(base + 208u);
    }
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_run_activations<32>(stage, lane, active, out);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane& lane,
                                                const XLimbs (&x)[M], float (&value)[M]) {
        const uint32_t qa[4] = {data.qa.x, data.qa.y, data.qa.z, data.qa.w};
        const uint32_t qb[4] = {data.qb.x, data.qb.y, data.qb.z, data.qb.w};
        const uint32_t qh[4] = {data.qh.x, data.qh.y, data.qh.z, data.qh.w};
        int dot[M][4][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int k = 0; k < 3; k++) dot[m][g][k] = x[m].bias[g][k];  // sum (q - 32) x = sum q x - 32 sum x
#pragma unroll
        for (int g = 0; g < 4; g++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t low = (g & 1) ? qb[i] : qa[i];
                const uint32_t nibbles = ((g & 2) ? (low >> 4) : low) & 0x0f0f0f0fu;
                const uint32_t high = (qh[i] >> (2 * g)) & 0x03030303u;
                const int q = static_cast<int>((high << 4) | nibbles);  // four values 0..63
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int k = 0; k < 3; k++)
                        dot[m][g][k] = __builtin_amdgcn_sdot4(q, x[m].limb[k][4 * g + i], dot[m][g][k], false);
            }
        }
        // scale of run g: signed byte j + 2g of the eight
        const uint32_t shift = 8u * lane.j;
        const auto signed_byte = [](uint32_t word, uint32_t at) {
            return static_cast<float>(static_cast<int>(static_cast<int8_t>(word >> at)));
        };
        const float sc[4] = {signed_byte(data.scales.x, shift), signed_byte(data.scales.x, shift + 16u),
                             signed_byte(data.scales.y, shift), signed_byte(data.scales.y, shift + 16u)};
        const float d = half_bits_to_float(data.d);
#pragma unroll
        for (int m = 0; m < M; m++) {
            float part[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                // the dots are below 2^21 in magnitude and convert exactly
                float limb_sum[3];
#pragma unroll
                for (int k = 0; k < 3; k++)
                    limb_sum[k] = fmaf(sc[2 * h + 1], static_cast<float>(dot[m][2 * h + 1][k]),
                                       sc[2 * h] * static_cast<float>(dot[m][2 * h][k]));
                part[h] = fmaf(65536.0f, limb_sum[2], fmaf(256.0f, limb_sum[1], limb_sum[0]));
            }
            value[m] = d * fmaf(x[m].s_pair[1], part[1], x[m].s_pair[0] * part[0]);
        }
    }
};

// s_pair[0] * (limb-combined, scale-weighted dots of runs 0, 1) + s_pair[1] * (those of runs 2, 3)
template <int M>
__device__ __forceinline__ void combine_runs(const int (&dot)[M][4][3], const float (&sc)[4], const XLimbs (&x)[M],
                                             float (&out)[M]) {
#pragma unroll
    for (int m = 0; m < M; m++) {
        float part[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float limb_sum[3];
#pragma unroll
            for (int k = 0; k < 3; k++)
                limb_sum[k] = fmaf(sc[2 * h + 1], static_cast<float>(dot[m][2 * h + 1][k]),
                                   sc[2 * h] * static_cast<float>(dot[m][2 * h][k]));
            part[h] = fmaf(65536.0f, limb_sum[2], fmaf(256.0f, limb_sum[1], limb_sum[0]));
        }
        out[m] = fmaf(x[m].s_pair[1], part[1], x[m].s_pair[0] * part[0]);
    }
}

typedef uint4 __attribute__((aligned(4))) uint4_a4;
typedef struct __attribute__((packed, aligned(2))) { uint32_t v[3]; } Dwords3_a2;

// Q2_K (decode_q2_k, crates/runtime-cpu/src/quantized.rs:117-138): 84 bytes per 256 values - scales[16]
// (4-bit scale, 4-bit minimum per 16 values), qs[64] (2-bit quants), d, dmin. Value e = half*128 + 32g +
// 16j + i is d * (scales[8*half + 2g + j] & 15) * ((qs[32*half + 16j + i] >> 2g) & 3) - dmin *
// (scales[..] >> 4). A lane takes (half, j): runs g = 0..3, sixteen bytes of quants.
struct Q2KLimb {
    static constexpr uint32_t kBlockColumns = 256u, kBlockBytes = 84u;
    static constexpr bool kLdsCopies = true;     // gemv_limb_dma_kernel takes this codec; LDS serves the lanes' loads at any alignment
    static constexpr bool kCopiesInTurn = false; // ... on gemv_limb_dma_kernel, whose loaders fold the end of their ranges
    struct Lane {
        uint32_t offset, half, j;
    };
    struct Data {
        uint4 qs;
        uint2 scales;  // scales[8*half .. 8*half + 8]
        uint32_t dd;   // d | dmin << 16 (f16 bits)
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 8) * 84u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) {
        return Lane{(chunk >> 2) * 84u, (chunk >> 1) & 1u, chunk & 1u};
    }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        const uint8_t* base = row + lane.offset;  // 84 b: dword aligned
        data.qs = *reinterpret_cast<const uint4_a4*>(base + 16u + 32u * lane.half + 16u * lane.j);
        data.scales = *reinterpret_cast<const uint2_a2*>(base + 8u * lane.half);
        data.dd = *reinterpret_cast<const uint32_t*>(base + 80u);
    }
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_run_activations<0>(stage, lane, active, out);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane& lane,
                                                const XLimbs (&x)[M], float (&value)[M]) {
        const uint32_t qs[4] = {data.qs.x, data.qs.y, data.qs.z, data.qs.w};
        int dot[M][4][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int k = 0; k < 3; k++) dot[m][g][k] = 0;
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int q = static_cast<int>((qs[i] >> (2 * g)) & 0x03030303u);
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int k = 0; k < 3; k++)
                        dot[m][g][k] = __builtin_amdgcn_sdot4(q, x[m].limb[k][4 * g + i], dot[m][g][k], false);
            }
        // (scale, minimum) of run g: byte j + 2g of the eight
        const uint32_t shift = 8u * lane.j;
        const uint32_t bytes[4] = {(data.scales.x >> shift) & 0xffu, (data.scales.x >> (shift + 16u)) & 0xffu,
                                   (data.scales.y >> shift) & 0xffu, (data.scales.y >> (shift + 16u)) & 0xffu};
        float sc[4], mn[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            sc[g] = static_cast<float>(bytes[g] & 15u);
            mn[g] = static_cast<float>(bytes[g] >> 4);
        }
        float pos[M];
        combine_runs<M>(dot, sc, x, pos);
        const float d = half_bits_to_float(data.dd & 0xffffu), dmin = half_bits_to_float(data.dd >> 16);
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float neg = fmaf(mn[3], x[m].run_sum[3],
                                   fmaf(mn[2], x[m].run_sum[2], fmaf(mn[1], x[m].run_sum[1], mn[0] * x[m].run_sum[0])));
            value[m] = d * pos[m] - dmin * neg;
        }
    }
};

// Q3_K (decode_q3_k, crates/runtime-cpu/src/quantized.rs:142-176): 110 bytes per 256 values - hmask[32]
// (third bits), qs[64] (2-bit quants), scales[12] (sixteen 6-bit scales, packed), d. Value e = half*128 +
// 32g + 16j + i is d * (scale[8*half + 2g + j] - 32) * (((qs[32*half + 16j + i] >> 2g) & 3) -
// (hmask[16j + i] bit (4*half + g) ? 0 : 4)). A lane takes (half, j): runs g = 0..3.
struct Q3KLimb {
    static constexpr uint32_t kBlockColumns = 256u, kBlockBytes = 110u;
    // gemv_limb_kernel only. LDS serves the lanes' 2-byte-aligned 16-byte reads, but slowly: through
    // gemv_limb_dma_kernel 14336 x 4096 measured 10.5 us against 9.6.
    static constexpr bool kLdsCopies = false;
    struct Lane {
        uint32_t offset, half, j;
    };
    struct Data {
        uint4 qs, hm;
        uint32_t packed[3];  // scales[12]
        uint32_t d;
    };
    static __device__ __forceinline__ uint64_t row_bytes(uint32_t columns) {
        return static_cast<uint64_t>(columns >> 8) * 110u;
    }
    static __device__ __forceinline__ Lane lane_setup(uint32_t chunk) {
        return Lane{(chunk >> 2) * 110u, (chunk >> 1) & 1u, chunk & 1u};
    }
    static __device__ __forceinline__ void load(const uint8_t* row, const Lane& lane, Data& data) {
        const uint8_t* base = row + lane.offset;  // 110 b: odd blocks start 2 bytes off a dword
        data.hm = *reinterpret_cast<const uint4_a2*>(base + 16u * lane.j);
        data.qs = *reinterpret_cast<const uint4_a2*>(base + 32u + 32u * lane.half + 16u * lane.j);
        const Dwords3_a2 packed = *reinterpret_cast<const Dwords3_a2*>(base + 96u);
        data.packed[0] = packed.v[0];
        data.packed[1] = packed.v[1];
        data.packed[2] = packed.v[2];
        data.d = *reinterpret_cast<const uint16_t*>(base + 108u);
    }
    static __device__ __forceinline__ void load_activations(const StageMemory& stage, uint32_t lane, bool active,
                                                            XLimbs& out) {
        load_run_activations<4>(stage, lane, active, out);
    }
    template <int M>
    static __device__ __forceinline__ void fold(const Data& data, const Lane& lane,
                                                const XLimbs (&x)[M], float (&value)[M]) {
        const uint32_t qs[4] = {data.qs.x, data.qs.y, data.qs.z, data.qs.w};
        const uint32_t hm[4] = {data.hm.x, data.hm.y, data.hm.z, data.hm.w};
        int dot[M][4][3];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int k = 0; k < 3; k++) dot[m][g][k] = x[m].bias[g][k];  // sum (v - 4) x = sum v x - 4 sum x
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t low = (qs[i] >> (2 * g)) & 0x03030303u;
                const uint32_t third = (hm[i] >> (4u * lane.half + g)) & 0x01010101u;
                const int v = static_cast<int>(low | (third << 2));  // four values 0..7
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int k = 0; k < 3; k++)
                        dot[m][g][k] = __builtin_amdgcn_sdot4(v, x[m].limb[k][4 * g + i], dot[m][g][k], false);
            }
        // scale of group G = 8*half + 2g + j: low four bits = nibble `half` of byte 2g + j of scales[0..8],
        // top two bits = bits 2*(2*half + g/2) of byte 8 + 2*(g & 1) + j; minus 32
        float sc[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t word = g < 2 ? data.packed[0] : data.packed[1];
            const uint32_t low = (word >> (8u * (2u * (g & 1) + lane.j) + 4u * lane.half)) & 15u;
            const uint32_t high = (data.packed[2] >> (8u * (2u * (g & 1) + lane.j) + 2u * (2u * lane.half + (g >> 1)))) & 3u;
            sc[g] = static_cast<float>(static_cast<int>(low | (high << 4)) - 32);
        }
        float pos[M];
        combine_runs<M>(dot, sc, x, pos);
        const float d = half_bits_to_float(data.d);
#pragma unroll
        for (int m = 0; m < M; m++) value[m] = d * pos[m];
    }
};

}  // namespace
}  // namespace et
