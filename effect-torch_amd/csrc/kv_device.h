// What the kernels of paged key/value-cache attention share (kv_attention.hip, kv_chunk.hip): the launch
// arguments, a slot's span of positions, and how the slab types store and read a value.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>

#include "decode_math.h"
#include "kernels.h"
#include "quantize_halves.h"  // dpp_f32

namespace et {

constexpr uint32_t kNoBlock = 0xffffffffu;
constexpr float kLowest = -1.0e30f;  // "no score yet": finite, so that exp2(kLowest - m) = 0 without NaN

// Element types of a slab besides float and __half.
struct Bf16 {
    uint16_t bits;
};
struct U8 {  // the int8-quantized tier: byte = round(x / scale) + 128, one f32 scale per row and head
    uint8_t byte;
};

struct KvArgs {
    void* k_slab;
    void* v_slab;
    float* k_scales;  // [max_tokens, kv_heads], the U8 tier only
    float* v_scales;
    const uint32_t* table;
    const uint32_t* cursors;
    const uint32_t* advances;
    const float* q;
    const float* k;
    const float* v;
    float* out;
    float* partial;
    unsigned long long* status;
    uint32_t max_tokens, kv_heads, width, block_size;
    int32_t block_shift;  // log2(block_size), or -1 when it is not a power of two
    uint32_t table_stride, active_batch, query_heads, tokens, context_window, window;
    uint32_t splits, max_context;
    float scale_log2;  // scale * log2(e)
    uint8_t* prepared;       // see KvAttention::prepared; null = none, or a quantiser launch follows
    uint32_t vector_tiles;   // of the prepared activations: ceil(batch / 32)
    KvProjected projected;   // see KvAttention::projected; shares == null: q, k, v above
};

struct Span {
    uint32_t cursor, advance, needed, start;
    uint32_t code;   // the first check of kv_prepare that fails, 0 = none
    uint64_t value;  // what that check reports; cursor + advance needs 33 bits
    bool ok;
};

// kv_prepare (napi/mod.rs:3588-3609) on device-resident cursors.
__device__ inline Span slot_span(const KvArgs& a, uint32_t slot) {
    Span s;
    s.cursor = a.cursors[slot];
    s.advance = a.advances[slot];
    // The reference adds in usize and cannot wrap; a cursor near 2^32 (an idle slot's -1) must fail
    // a check here, before any table access, instead of wrapping to a small context.
    const uint64_t needed = static_cast<uint64_t>(s.cursor) + s.advance;
    const uint64_t start = a.context_window != 0 && needed > a.context_window ? needed - a.context_window : 0;
    s.code = 0;
    s.value = 0;
    if (s.advance == 0 || s.advance > a.tokens) {
        s.code = kKvBadAdvance;
        s.value = s.advance;
    } else if (needed - start > a.max_tokens) {
        s.code = kKvOverCapacity;
        s.value = needed - start;
    } else if ((needed + a.block_size - 1) / a.block_size > a.table_stride) {
        s.code = kKvShortTable;
        s.value = needed;
    } else if (needed > a.max_context) {  // max_context is 32 bits wide: passing means no wrap below
        s.code = kKvOverDeclared;
        s.value = needed;
    }
    s.ok = s.code == 0;
    s.needed = s.ok ? static_cast<uint32_t>(needed) : 0;
    s.start = s.ok ? static_cast<uint32_t>(start) : 0;
    return s;
}

__device__ __forceinline__ uint32_t block_of(const KvArgs& a, uint32_t position) {
    return a.block_shift >= 0 ? position >> a.block_shift : position / a.block_size;
}
__device__ __forceinline__ uint32_t within_block(const KvArgs& a, uint32_t position) {
    return a.block_shift >= 0 ? position & (a.block_size - 1) : position % a.block_size;
}

__device__ __forceinline__ void slab_store(float* slab, uint64_t at, float value) { slab[at] = value; }
__device__ __forceinline__ void slab_store(__half* slab, uint64_t at, float value) {
    slab[at] = __float2half_rn(value);
}
// the value a slab of this type holds after storing `value`
__device__ __forceinline__ float slab_round(const float*, float value) { return value; }
__device__ __forceinline__ float slab_round(const __half*, float value) {
    return __half2float(__float2half_rn(value));
}
__device__ __forceinline__ float slab_load(const float* slab, uint64_t at) { return slab[at]; }
__device__ __forceinline__ float slab_load(const __half* slab, uint64_t at) { return __half2float(slab[at]); }
// bf16::from_f32 (half 2.7.1): NaN keeps its top bits and gets a quiet bit, else round to nearest even.
__device__ __forceinline__ uint32_t bf16_bits(float value) {
    const uint32_t x = __float_as_uint(value);
    if ((x & 0x7fffffffu) > 0x7f800000u) return (x >> 16) | 0x0040u;
    return (x + 0x7fffu + ((x >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ void slab_store(Bf16* slab, uint64_t at, float value) {
    slab[at].bits = static_cast<uint16_t>(bf16_bits(value));
}
__device__ __forceinline__ float slab_round(const Bf16*, float value) { return __uint_as_float(bf16_bits(value) << 16); }
__device__ __forceinline__ float slab_load(const Bf16* slab, uint64_t at) {
    return __uint_as_float(static_cast<uint32_t>(slab[at].bits) << 16);
}
// The U8 tier (napi/mod.rs:3397-3437, :3467-3478): scale = max|x| / 127 + 1e-12 over the row of a
// head, byte = clamp(round(x / scale), +-127) + 128 (halves away from zero), value = (byte - 128) * scale.
__device__ __forceinline__ float u8_scale(float row_maximum) { return row_maximum / 127.0f + 1e-12f; }
__device__ __forceinline__ uint32_t u8_byte(float value, float scale) {
    return static_cast<uint32_t>(fminf(fmaxf(roundf(value / scale), -127.0f), 127.0f) + 128.0f);
}
__device__ __forceinline__ float u8_value(uint32_t byte, float scale) {
    return (static_cast<float>(byte) - 128.0f) * scale;
}

// The status word of a slot: 0, or code << 56 | value. Written by one wave per slot, which also
// checks that the rows of the new positions lie inside the pool.
__device__ inline void write_slot_status(const KvArgs& a, uint32_t slot, const Span& s, int lane) {
    uint32_t code = s.code;
    uint64_t value = s.value;
    if (s.ok) {
        uint32_t worst = 0;
        for (uint32_t token = lane; token < s.advance; token += 64) {
            const uint32_t position = s.cursor + token;
            const uint64_t row = static_cast<uint64_t>(a.table[static_cast<uint64_t>(slot) * a.table_stride +
                                                               block_of(a, position)]) * a.block_size +
                                 within_block(a, position);
            if (row >= a.max_tokens) worst = max(worst, static_cast<uint32_t>(min(row, uint64_t{0xffffffffu})));
        }
        for (int offset = 32; offset > 0; offset >>= 1) worst = max(worst, __shfl_xor(worst, offset));
        if (worst != 0) {
            code = kKvBlockOutside;
            value = worst;
        }
    }
    if (lane == 0) a.status[slot] = (static_cast<unsigned long long>(code) << 56) | value;
}

// Positions a query attends to (napi/mod.rs:3481-3483).
__device__ __forceinline__ void query_range(const KvArgs& a, const Span& s, uint32_t token,
                                            uint32_t& begin, uint32_t& end) {
    end = min(s.cursor + token + 1, s.needed);
    begin = s.start;
    if (a.window != 0) begin = max(end > a.window ? end - a.window : 0u, s.start);
    begin = min(begin, end);
}

// q of the workgroup's G heads, then k and v of its kv head, for one slot, from the K shares of the
// projection: the sums in share order, the bias, the rotary pairs of q and k - what
// reduce_group_rotary_kernel (gemm_h16.hip) stores. out: [(G + 2)][width] floats in LDS.
__device__ __forceinline__ void project_rows(const KvArgs& a, uint32_t slot, uint32_t G, uint32_t head0, uint32_t kv_head,
                                             float* out, uint32_t threads) {
    const KvProjected& s = a.projected;
    const uint32_t width = a.width, half = width / 2;
    const uint64_t share_stride = s.launch_rows * s.vectors;
    const auto summed = [&](uint32_t first_row, const float* bias, uint32_t row) {
        const float* first = s.shares + static_cast<uint64_t>(slot) * s.launch_rows + first_row + row;
        float total = first[0];
        for (uint32_t k = 1; k < s.count; k++) total += first[k * share_stride];
        return bias != nullptr ? total + bias[row] : total;
    };
    const uint32_t offset = s.offsets_len == 1 ? s.offsets[0] : s.offsets[slot];
    const uint32_t rotated = (G + 1) * half;  // the pairs of the G query heads, then of the key head
    for (uint32_t item = threadIdx.x; item < rotated + width; item += threads) {
        if (item < rotated) {
            const uint32_t h = item / half, index = item - h * half;
            const uint32_t head = h < G ? head0 + h : kv_head;
            const uint32_t first_row = h < G ? s.q_row : s.k_row;
            const float* bias = h < G ? s.q_bias : s.k_bias;
            const uint32_t lo = s.interleaved ? 2u * index : index, hi = s.interleaved ? lo + 1u : lo + half;
            float value_lo = summed(first_row, bias, head * width + lo);
            float value_hi = summed(first_row, bias, head * width + hi);
            rotate_pair(value_lo, value_hi, offset, 0u, index, width, s.theta, s.sign, value_lo, value_hi);
            out[h * width + lo] = value_lo;
            out[h * width + hi] = value_hi;
        } else {
            const uint32_t d = item - rotated;
            out[(G + 1) * width + d] = summed(s.v_row, s.v_bias, kv_head * width + d);
        }
    }
}

// Sum over the LANES lanes of an aligned group; every lane gets the total.
template <int LANES>
__device__ __forceinline__ float group_sum(float v) {
    if constexpr (LANES >= 2) v += dpp_f32<0xB1>(v);    // quad_perm [1,0,3,2]
    if constexpr (LANES >= 4) v += dpp_f32<0x4E>(v);    // quad_perm [2,3,0,1]
    if constexpr (LANES >= 8) v += dpp_f32<0x141>(v);   // row_half_mirror
    if constexpr (LANES >= 16) v += dpp_f32<0x140>(v);  // row_mirror
    if constexpr (LANES >= 32) v += __shfl_xor(v, 16);
    if constexpr (LANES >= 64) v += __shfl_xor(v, 32);
    return v;
}

template <int LANES>
__device__ __forceinline__ float group_max(float v) {
    if constexpr (LANES >= 2) v = fmaxf(v, dpp_f32<0xB1>(v));
    if constexpr (LANES >= 4) v = fmaxf(v, dpp_f32<0x4E>(v));
    if constexpr (LANES >= 8) v = fmaxf(v, dpp_f32<0x141>(v));
    if constexpr (LANES >= 16) v = fmaxf(v, dpp_f32<0x140>(v));
    if constexpr (LANES >= 32) v = fmaxf(v, __shfl_xor(v, 16));
    if constexpr (LANES >= 64) v = fmaxf(v, __shfl_xor(v, 32));
    return v;
}

// kv_bytes.hip: decode steps over u8 slabs on the int8 matrix cores; a.splits context splits per (slot, kv head).
hipError_t kv_bytes(const KvArgs& a, int waves, uint32_t workgroups, hipStream_t stream);
// kv_chunk.hip: calls of several tokens per slot on the matrix cores. `workgroups` = grid.units * splits.
hipError_t kv_chunk(int32_t slab_dtype, const KvArgs& a, int row_waves, uint32_t workgroups, hipStream_t stream);

}  // namespace et
