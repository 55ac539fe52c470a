// One decode step's attention (one token per slot) over slabs of the int8-quantized tier on the gfx950 int8 matrix cores;
// semantics of kv_attention_into (crates/runtime-cpu/src/napi/mod.rs:3320-3544) as in kv_attention.hip, whose streaming
// kernel this one stands in for (streaming_bytes there says where).
//
// The bytes never become floats. q enters as 31-bit fixed point in four balanced signed-byte limbs per head; a row of K
// less 128 is signed bytes as it lies in the slab, and v_mfma_i32_16x16x64_i8 contracts sixteen positions with the limbs of
// up to four query heads (rows 4 * limb + head of one operand) in exact integers. A score is the sum of its four integers
// times q's unit, the softmax scale and the row's K scale. The weights times the rows' V scales, 64 positions at a time,
// are fixed point in four limbs as well and contract with V's bytes, which ds_read_b64_tr_b8 transposes out of LDS; the sums
// of a step are added up in f32.
//
// Layout. A wave takes 64 positions a step on its own: K straight into the registers of the lanes that hold it as an
// operand (lane = position l % 16, sixteen columns per lane group l / 16), V by copies into an LDS tile of its own, both
// asked for as soon as the step before has contracted its keys. Three lane exchanges per sixteen positions sum a score's
// limbs and leave head h in lane group h, so the softmax works on four scores per lane and none twice.
// LDS: [wave: two V tiles, the weights' limbs] x WAVES, [rows of the split's blocks]; the waves meet there at the end.
//
// Precision: limbs hold 31 bits, a float's 24 and more, the integer sums are exact, and an exponent is rounded once, next to
// the row's maximum. Relative error against 64 bits (2-norm, 1e-7; streaming kernel / this), 32/8 heads x 128: 32 slots at
// 2048 3.3 / 1.3, three at 10000 to 30000 3.3 / 1.7, one at 60000 3.7 / 2.0. Three limbs (24 bits) and exponents of a rounded
// score had 4.5. The fixed point is that of the largest of a row of q, and of the largest of 64 weights: what is smaller than
// it by 2^-6 and more loses bits, which shows only where the largest meets a byte of 128, a value of zero. V scales and
// queries keep their bits down to 2^-121.
// What is not finite: a NaN or infinity in q, a K scale or a V scale makes all columns of the heads that see it NaN, as in
// the streaming kernel (whose values are byte * scale - 128 * scale).
//
// Bound: reads of 128 bytes a position and head, with the ends of a launch. Per 64 positions of 128 columns a wave issues
// about 700 vector and 16 matrix instructions (of 16 cycles) where the streaming kernel - a conversion, a scale and four
// multiply-adds per byte - issues 2000. 32 slots at 2048 (138 MB, which the Infinity Cache holds), streaming kernel / this, in a
// graph: the same inputs again 50.4 / 31.8 us (4.3 TB/s), inputs from memory 51.1 / 35.7; with the loads left out 17. K comes by
// ordinary loads: the two halves of a row are two instructions', and non-temporal ones fetched its line twice (a quarter
// more time).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <type_traits>

#include "kernels.h"
#include "kv_device.h"

namespace et {
namespace {

constexpr uint32_t kTile = 64;  // positions a wave takes per step
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4), aligned(4)));

template <int W, int WAVES>
struct BytesLds {
    static constexpr uint32_t kValueTile = kTile * W;
    static constexpr uint32_t kWave = 2 * kValueTile + 16 * kTile;  // two tiles of V, sixteen rows of weight limbs
    static constexpr uint32_t kTableAt = WAVES * kWave;
    static constexpr uint32_t kRowsAt = kTableAt + kKvTableEntries * 4;  // projected q of four heads, k and v
    static constexpr uint32_t kBytes = kRowsAt + 6 * W * 4;
    static_assert(WAVES * (W + 2) * 16 <= kTableAt, "the waves' sums meet where the tiles were");
    static_assert(4 * W * 4 <= kKvTableEntries * 4, "and the results that are quantised where the table was");
    static_assert(kBytes <= 160 * 1024, "LDS of a compute unit");
};

// A non-temporal copy of sixteen bytes per lane to LDS (lane i to `to` + 16 i) that the compiler does not see (see
// kv_chunk.hip). Its eight lanes a row take whole lines.
__device__ __forceinline__ void copy_streamed(const void* from, uint32_t to) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(from), "s"(to) : "memory", "m0");
}

// Eight rows of sixteen bytes to sixteen lanes of eight: lane i names row (i & 15) / 2, columns 8 (i & 1) .. + 7, and
// receives column i & 15 of the eight rows.
__device__ __forceinline__ v2i read_transposed(uint32_t from) {
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)from);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
    return max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true)));
}
// over the sixteen lanes of a row
__device__ __forceinline__ uint32_t row_max(uint32_t v) {
    return dpp_max_u32<0x140>(dpp_max_u32<0x141>(dpp_max_u32<0x4E>(dpp_max_u32<0xB1>(v))));
}

// The sums over the four lane groups of v[0..3], of v[g] in lane group g.
__device__ __forceinline__ float reduce_scatter(const float (&v)[4]) {
    const auto add32 = [](float a, float b) {  // lanes 0-31: a summed over the halves; 32-63: b
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(s[0]) + __uint_as_float(s[1]);
    };
    const float even = add32(v[0], v[2]), odd = add32(v[1], v[3]);
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(even), __float_as_uint(odd), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// Fixed point in units of 2^-up, `bits` being those of the largest magnitude: below 2^30 units, so that a float loses
// nothing unless it is smaller than the largest by 2^6 or more, and then what lies under 2^-30 of that. `top` is the worth
// of the top limb, 2^24 units: a normal number down to values of 2^-121, where the unit itself is not, and below that
// all floats are whole units. A NaN or infinity makes it NaN, and with it every result that the values take part in.
__device__ __forceinline__ void fixed_point(uint32_t bits, float& top, int& up) {
    const int exponent = max(static_cast<int>(bits >> 23), 7);  // the largest is below 2^(exponent - 126)
    up = 156 - exponent;
    top = bits < 0x7f800000u ? __uint_as_float(static_cast<uint32_t>(exponent - 5) << 23) : NAN;
}
// Balanced digits: X + 0x808080 with the top bits of its three low bytes flipped is sum_i 256^i x_i in signed bytes. (2^up is
// no float where the values are small.)
__device__ __forceinline__ uint32_t digits(float value, int up) {
    return static_cast<uint32_t>(static_cast<int>(rintf(__builtin_amdgcn_ldexpf(value, up)))) + 0x00808080u;
}

// PROJECTED: q, k and v arrive as the K shares of their projections (KvArgs::projected).
template <int W, int WAVES, bool PROJECTED>
__global__ __launch_bounds__(64 * WAVES, 2) void kv_bytes_kernel(const KvArgs a) {
    using L = BytesLds<W, WAVES>;
    constexpr int kHalves = W / 64;             // 64-column operands of a row
    constexpr int kDims = W / 16;               // sixteen-column operands of V
    constexpr uint32_t kPieces = W / 16;        // sixteen-byte pieces of a row
    constexpr int kCopies = kTile * W / 1024;   // of a V tile
    constexpr uint32_t kRowsPerCopy = 1024 / W;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint32_t* rows_of_block = reinterpret_cast<uint32_t*>(lds + L::kTableAt);

    // Whole slots: the heads of one run side by side on one XCD (workgroups go to the eight in turn), as a position's row holds
    // all of them and their scales share a line (32 slots at 2048, inputs from memory: 35.3 -> 34.6 us). Splits of a slot run
    // side by side instead (one slot at 60000: 39.4 -> 37.6).
    uint32_t split = 0, kv_head, slot;
    if (a.splits == 1 && blockIdx.x < a.active_batch / 8 * 8 * a.kv_heads) {
        slot = blockIdx.x / (8 * a.kv_heads) * 8 + blockIdx.x % 8;
        kv_head = blockIdx.x / 8 % a.kv_heads;
    } else {
        const uint32_t pair = blockIdx.x / a.splits;
        split = blockIdx.x % a.splits;
        kv_head = pair % a.kv_heads;
        slot = pair / a.kv_heads;
    }
    const uint32_t heads = a.query_heads / a.kv_heads, head0 = kv_head * heads;
    const int lane = threadIdx.x & 63, column = lane & 15, group = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const Span s = slot_span(a, slot);
    if (kv_head == 0 && split == 0 && wave == 0) write_slot_status(a, slot, s, lane);
    uint32_t begin, end;
    query_range(a, s, 0, begin, end);
    const uint32_t length = s.ok ? end - begin : 0;
    uint32_t share = (length + a.splits - 1) / a.splits;
    share = (share + kTile - 1) / kTile * kTile;
    const uint32_t my_begin = min(begin + split * share, begin + length);
    const uint32_t my_end = min(my_begin + share, begin + length);
    const uint32_t cached_end = min(my_end, max(my_begin, s.cursor));  // the position behind it arrives with this call
    const uint32_t first_block = block_of(a, my_begin);
    if (my_end > my_begin) {
        const uint32_t blocks = block_of(a, my_end - 1) - first_block + 1;
        for (uint32_t i = threadIdx.x; i < blocks && i < kKvTableEntries; i += 64 * WAVES) {
            const uint64_t row = static_cast<uint64_t>(a.table[static_cast<uint64_t>(slot) * a.table_stride + first_block + i]) *
                                 a.block_size;
            rows_of_block[i] = row >= a.max_tokens ? kNoBlock : static_cast<uint32_t>(row);
        }
    }

    // q as the A operand: this lane holds limb column / 4 of head column % 4, columns 16 * group + (0..15) of each half.
    const uint32_t limb = column >> 2, head = column & 3;
    float* rows = reinterpret_cast<float*>(lds + L::kRowsAt);
    const float *q_rows = rows, *k_row = rows + heads * W, *v_row = k_row + W;
    if constexpr (PROJECTED) {
        project_rows(a, slot, heads, head0, kv_head, rows, 64 * WAVES);
    } else {
        q_rows = a.q + (static_cast<uint64_t>(slot) * a.query_heads + head0) * W;
        k_row = a.k + (static_cast<uint64_t>(slot) * a.kv_heads + kv_head) * W;
        v_row = a.v + (static_cast<uint64_t>(slot) * a.kv_heads + kv_head) * W;
    }
    v4f q_in[kHalves][4];
    const auto load_q = [&]() {
#pragma unroll
        for (int h = 0; h < kHalves; h++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                q_in[h][i] = *reinterpret_cast<const v4f*>(q_rows + min(head, heads - 1) * W + 64 * h + 16 * group + 4 * i);
    };
    if constexpr (!PROJECTED) load_q();  // on their way in front of the first tile
    const float limb_weight = __uint_as_float((103u + 8u * group) << 23);  // of limb `group`, 256^(group - 3) of the top one

    const uint32_t row_bytes = a.kv_heads * W;
    const uint8_t* k_base = static_cast<const uint8_t*>(a.k_slab) + kv_head * W;
    const uint8_t* v_base = static_cast<const uint8_t*>(a.v_slab) + kv_head * W;
    // positions past the end read the last cached row
    const auto slab_row = [&](uint32_t position, auto shifts) __attribute__((always_inline)) -> uint64_t {
        position = min(position, cached_end - 1);
        const uint32_t block = shifts ? position >> a.block_shift : position / a.block_size;
        const uint32_t within = shifts ? position & (a.block_size - 1) : position - block * a.block_size;
        const uint32_t base = rows_of_block[min(block - first_block, kKvTableEntries - 1u)];
        return base == kNoBlock ? 0u : min(base + within, a.max_tokens - 1);
    };
    // Piece p of row r of a V tile lies in slot p ^ swizzle(r): the transposing reads spread over all banks.
    const auto swizzle = [](uint32_t r) { return W == 128 ? ((r >> 4) & 3u) | (((r >> 2) & 1u) << 2) : (r >> 4) & 3u; };
    const uint32_t wave_lds = __builtin_amdgcn_readfirstlane(
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds)) + wave * L::kWave);
    uint4 k_raw[4][kHalves];
    float k_scale[4], v_scale[4];
    const auto fetch_rows = [&](uint32_t tile, uint32_t buffer, auto shifts) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < kCopies; c++) {
            const uint32_t r = c * kRowsPerCopy + lane / kPieces;
            copy_streamed(v_base + slab_row(tile + r, shifts) * row_bytes + ((lane % kPieces) ^ swizzle(r)) * 16u,
                          __builtin_amdgcn_readfirstlane(wave_lds + buffer * L::kValueTile + c * 1024u));
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint64_t row = slab_row(tile + 16 * t + column, shifts);
#pragma unroll
            for (int h = 0; h < kHalves; h++) k_raw[t][h] = *reinterpret_cast<const uint4*>(k_base + row * row_bytes + 64 * h + 16 * group);
            k_scale[t] = a.k_scales[row * a.kv_heads + kv_head];
            v_scale[t] = a.v_scales[row * a.kv_heads + kv_head];
        }
    };
    // one branch on the block size, not one per row
    const auto fetch = [&](uint32_t tile, uint32_t buffer) __attribute__((always_inline)) {
        if (a.block_shift >= 0)
            fetch_rows(tile, buffer, std::true_type{});
        else
            fetch_rows(tile, buffer, std::false_type{});
    };

    // The weights' limbs: row 4 * limb + head, byte 4 * column + t for position 16 t + column of the step.
    uint8_t* weights = lds + wave * L::kWave + 2 * L::kValueTile;
    // V operand: lane group g holds bytes 4 j + t for positions 16 t + 4 g + j; this lane names row (lane & 15) / 2 of the
    // first eight (j = 0, 1), and two rows further on of the others.
    const uint32_t named = (lane & 15) >> 1, value_row = 16 * (named & 3) + 4 * group + (named >> 2);
    const uint32_t value_at = value_row * W + (lane & 1) * 8u, value_swizzle = swizzle(value_row);

    float m = kLowest, l = 0.f;  // of head `group`: its maximum, this lane's part of the sum
    float o[kDims][4];           // limb `group` of head i's sums at column 16 d + column
#pragma unroll
    for (int d = 0; d < kDims; d++)
#pragma unroll
        for (int i = 0; i < 4; i++) o[d][i] = 0.f;

    __syncthreads();  // the table is in LDS
    uint32_t buffer = 0;
    uint32_t tile = my_begin + wave * kTile;
    if (tile < cached_end) fetch(tile, 0);

    v4i q[kHalves];
    float q_unit;  // the worth of q's top limb
    {
        if constexpr (PROJECTED) load_q();
        uint32_t most = 0;
#pragma unroll
        for (int h = 0; h < kHalves; h++)
#pragma unroll
            for (int i = 0; i < 16; i++) most = max(most, __float_as_uint(q_in[h][i / 4][i % 4]) & 0x7fffffffu);
        most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), 16)));
        most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), 32)));
        float worth;
        int up;
        fixed_point(most, worth, up);
        const bool used = head < heads;
#pragma unroll
        for (int h = 0; h < kHalves; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t word = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) word |= ((digits(q_in[h][i][e], up) >> (8 * limb)) & 0xffu) << (8 * e);
                q[h][i] = used ? static_cast<int>(limb < 3 ? word ^ 0x80808080u : word) : 0;
            }
        q_unit = __shfl(worth, group) * a.scale_log2;  // of head `group`, whose scores this lane will hold
    }

    for (; tile < cached_end; tile += WAVES * kTile) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this step's rows have landed
        // A score is (high + low) * (scale + scale_rest): the sum of the top limb and those of the others, and the exact
        // product of q's unit and the K scale, so that the exponent below is rounded once, where it is small.
        float high[4], low[4], scale[4], scale_rest[4], v_now[4], seen = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            v4i sum = {0, 0, 0, 0};
#pragma unroll
            for (int h = 0; h < kHalves; h++) {
                const uint4 raw = k_raw[t][h];
                const v4i key = {static_cast<int>(raw.x ^ 0x80808080u), static_cast<int>(raw.y ^ 0x80808080u),
                                 static_cast<int>(raw.z ^ 0x80808080u), static_cast<int>(raw.w ^ 0x80808080u)};
                sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(q[h], key, sum, 0, 0, 0);
            }
            float top_parts[4], parts[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float part = static_cast<float>(sum[i]) * limb_weight;
                top_parts[i] = group == 3 ? part : 0.f;
                parts[i] = group == 3 ? 0.f : part;
            }
            high[t] = reduce_scatter(top_parts);
            low[t] = reduce_scatter(parts);
            // A K row with an infinite scale has values that are infinite or, byte 128, NaN: its score is NaN.
            const float k = fabsf(k_scale[t]) < INFINITY ? k_scale[t] : NAN;
            scale[t] = q_unit * k;
            scale_rest[t] = fmaf(q_unit, k, -scale[t]);
            v_now[t] = v_scale[t];
            if (tile + 16 * t + column < cached_end) seen = fmaxf(seen, fmaf(high[t], scale[t], low[t] * scale[t]));
        }
        if (tile + WAVES * kTile < cached_end) fetch(tile + WAVES * kTile, buffer ^ 1u);

        const float top = fmaxf(m, group_max<16>(seen));
        const float keep = __builtin_amdgcn_exp2f(m - top);
        m = top;
        float w[4], total = 0.f;
        uint32_t most = 0;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const float exponent = fmaf(high[t], scale[t], -top) + fmaf(low[t], scale[t], high[t] * scale_rest[t]);
            const bool live = tile + 16 * t + column < cached_end;
            const float p = live ? __builtin_amdgcn_exp2f(exponent) : 0.f;
            total += p;
            w[t] = live ? p * v_now[t] : 0.f;
            most = max(most, __float_as_uint(w[t]) & 0x7fffffffu);  // NaN and infinities are the largest
        }
        l = fmaf(l, keep, total);
        float worth;
        int up;
        fixed_point(row_max(most), worth, up);
        const uint32_t x0 = digits(w[0], up), x1 = digits(w[1], up), x2 = digits(w[2], up), x3 = digits(w[3], up);
        // 4x4 byte transpose: limb k of the four weights into one dword
        const uint32_t ab = __builtin_amdgcn_perm(x1, x0, 0x05010400u), cd = __builtin_amdgcn_perm(x3, x2, 0x05010400u);
        const uint32_t ah = __builtin_amdgcn_perm(x1, x0, 0x07030602u), ch = __builtin_amdgcn_perm(x3, x2, 0x07030602u);
        uint32_t* to = reinterpret_cast<uint32_t*>(weights + group * kTile + 4 * column);
        to[0] = __builtin_amdgcn_perm(cd, ab, 0x05040100u) ^ 0x80808080u;
        to[4 * kTile / 4] = __builtin_amdgcn_perm(cd, ab, 0x07060302u) ^ 0x80808080u;
        to[8 * kTile / 4] = __builtin_amdgcn_perm(ch, ah, 0x05040100u) ^ 0x80808080u;
        to[12 * kTile / 4] = __builtin_amdgcn_perm(ch, ah, 0x07060302u);
        __builtin_amdgcn_wave_barrier();
        const v4i p = *reinterpret_cast<const v4i*>(weights + column * kTile + 16 * group);

        float kept[4], units[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {  // head i's are those of lane group i
            kept[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(keep), 16 * i));
            units[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(worth), 16 * i)) * limb_weight;
        }
        if (__builtin_amdgcn_ballot_w64(keep != 1.0f) != 0) {  // some maximum moved
#pragma unroll
            for (int d = 0; d < kDims; d++)
#pragma unroll
                for (int i = 0; i < 4; i++) o[d][i] *= kept[i];
        }
        const uint32_t values = wave_lds + buffer * L::kValueTile + value_at;
#pragma unroll
        for (int d = 0; d < kDims; d++) {
            const uint32_t at = values + ((d ^ value_swizzle) << 4);
            const v2i low = read_transposed(at), high = read_transposed(at + 2 * W);
            const v4i value = {low.x ^ static_cast<int>(0x80808080u), low.y ^ static_cast<int>(0x80808080u),
                               high.x ^ static_cast<int>(0x80808080u), high.y ^ static_cast<int>(0x80808080u)};
            const v4i sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(p, value, v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) o[d][i] = fmaf(static_cast<float>(sum[i]), units[i], o[d][i]);
        }
        buffer ^= 1u;
    }

    // Head `group`'s sums over its limbs and lanes: column 16 d + column.
    l = group_sum<16>(l);
    float sums[kDims];
#pragma unroll
    for (int d = 0; d < kDims; d++) sums[d] = reduce_scatter(o[d]);

    // The row that arrives, as the slab will hold it, by the first wave of the split it belongs to, which also appends it.
    if (wave == 0 && cached_end < my_end) {
        const uint32_t position = cached_end;
        constexpr int kMine = W / 64;
        float k_in[kMine], v_in[kMine], k_most = 0.f, v_most = 0.f;
#pragma unroll
        for (int i = 0; i < kMine; i++) {
            k_in[i] = k_row[kMine * lane + i];
            v_in[i] = v_row[kMine * lane + i];
            k_most = fmaxf(k_most, fabsf(k_in[i]));
            v_most = fmaxf(v_most, fabsf(v_in[i]));
        }
        const float ks = u8_scale(group_max<64>(k_most)), vs = u8_scale(group_max<64>(v_most));
        uint32_t k_bytes[kMine], v_bytes[kMine];
#pragma unroll
        for (int i = 0; i < kMine; i++) {
            k_bytes[i] = u8_byte(k_in[i], ks);
            v_bytes[i] = u8_byte(v_in[i], vs);
        }
        const uint32_t base = rows_of_block[min(block_of(a, position) - first_block, kKvTableEntries - 1u)];
        const uint32_t row = base + within_block(a, position);
        if (base != kNoBlock && row < a.max_tokens) {
            uint8_t* k_to = static_cast<uint8_t*>(a.k_slab) + static_cast<uint64_t>(row) * row_bytes + kv_head * W + kMine * lane;
            uint8_t* v_to = static_cast<uint8_t*>(a.v_slab) + static_cast<uint64_t>(row) * row_bytes + kv_head * W + kMine * lane;
#pragma unroll
            for (int i = 0; i < kMine; i++) {
                k_to[i] = static_cast<uint8_t>(k_bytes[i]);
                v_to[i] = static_cast<uint8_t>(v_bytes[i]);
            }
            if (lane == 0) {
                a.k_scales[static_cast<uint64_t>(row) * a.kv_heads + kv_head] = ks;
                a.v_scales[static_cast<uint64_t>(row) * a.kv_heads + kv_head] = vs;
            }
        }
        // (byte - 128) * scale with one rounding; NaN where the scale is infinite
        float score = 0.f;
        for (uint32_t h = 0; h < heads; h++) {
            float part = 0.f;
#pragma unroll
            for (int i = 0; i < kMine; i++)
                part = fmaf(q_rows[h * W + kMine * lane + i] * a.scale_log2,
                            fmaf(static_cast<float>(k_bytes[i]), ks, -128.0f * ks), part);
            part = group_sum<64>(part);
            if (static_cast<uint32_t>(group) == h) score = part;
        }
        const float top = fmaxf(m, score);
        const float keep = __builtin_amdgcn_exp2f(m - top), p = __builtin_amdgcn_exp2f(score - top);
        m = top;
        l = fmaf(l, keep, p);
#pragma unroll
        for (int d = 0; d < kDims; d++) {
            const float byte = static_cast<float>(u8_byte(v_row[16 * d + column], vs));
            sums[d] = fmaf(p, fmaf(byte, vs, -128.0f * vs), sums[d] * keep);
        }
    }

    // Combine the waves' softmax states.
    __syncthreads();  // every wave is done with its tiles
    float* meet = reinterpret_cast<float*>(lds);
    float* mine = meet + (wave * 4 + group) * (W + 2);
    if (column == 0) {
        mine[0] = m;
        mine[1] = l;
    }
#pragma unroll
    for (int d = 0; d < kDims; d++) mine[2 + 16 * d + column] = sums[d];
    __syncthreads();
    // The heads' results are heads * W neighbouring columns of the slot's row of activations for the contraction that
    // follows; where they are whole 256-column stages the row's tiles are quantised here, from the values just stored (a
    // skipped slot: from what the destination holds).
    float* row_part = reinterpret_cast<float*>(lds + L::kTableAt);
    const bool quantise = a.prepared != nullptr && a.splits == 1 && (heads * W) % 256 == 0;
    for (uint32_t item = threadIdx.x; item < heads * W; item += 64 * WAVES) {
        const uint32_t h = item / W, at = item % W;
        float top = kLowest;
        for (int i = 0; i < WAVES; i++) top = fmaxf(top, meet[(i * 4 + h) * (W + 2)]);
        float total = 0.f, value = 0.f;
        for (int i = 0; i < WAVES; i++) {
            const float* state = meet + (i * 4 + h) * (W + 2);
            const float weight = __builtin_amdgcn_exp2f(state[0] - top);
            total = fmaf(weight, state[1], total);
            value = fmaf(weight, state[2 + at], value);
        }
        const uint64_t query = static_cast<uint64_t>(slot) * a.query_heads + head0 + h;
        if (a.splits == 1) {
            const float result = value / total;
            if (s.ok) a.out[query * W + at] = result;
            if (quantise) row_part[item] = s.ok ? result : a.out[query * W + at];
        } else {
            float* record = a.partial + (query * a.splits + split) * (W + 2);
            record[2 + at] = value;
            if (at == 0) {
                record[0] = top;
                record[1] = total;
            }
        }
    }
    if (quantise) {
        __syncthreads();
        if (wave < heads * W / 256u) {
            const float4 in = *reinterpret_cast<const float4*>(&row_part[wave * 256u + 4u * lane]);
            quantize_halves_store(in, slot, head0 * W / 256u + wave, lane, a.vector_tiles, a.prepared);
        }
    }
}

template <int W, int WAVES, bool PROJECTED>
hipError_t launch(const KvArgs& a, uint32_t workgroups, hipStream_t stream) {
    using L = BytesLds<W, WAVES>;
    static std::atomic<bool> allowed[64];
    int device = 0;
    if (hipError_t status = hipGetDevice(&device)) return status;
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    if (!allowed[device].load(std::memory_order_acquire)) {
        if (hipError_t status = hipFuncSetAttribute(reinterpret_cast<const void*>(&kv_bytes_kernel<W, WAVES, PROJECTED>),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, L::kBytes))
            return status;
        allowed[device].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((kv_bytes_kernel<W, WAVES, PROJECTED>), dim3(workgroups), dim3(64 * WAVES), L::kBytes, stream, a);
    return hipGetLastError();
}

}  // namespace

hipError_t kv_bytes(const KvArgs& a, int waves, uint32_t workgroups, hipStream_t stream) {
    const auto go = [&](auto eight, auto four) { return waves == 8 ? eight(a, workgroups, stream) : four(a, workgroups, stream); };
    const bool projected = a.projected.shares != nullptr;
    if (a.width == 128) return projected ? go(launch<128, 8, true>, launch<128, 4, true>) : go(launch<128, 8, false>, launch<128, 4, false>);
    if (a.width == 64) return projected ? go(launch<64, 8, true>, launch<64, 4, true>) : go(launch<64, 8, false>, launch<64, 4, false>);
    return hipErrorInvalidValue;
}

}  // namespace et
