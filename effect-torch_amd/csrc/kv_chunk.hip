// Paged key/value-cache attention for calls of several tokens per slot (a prompt's chunk, draft tokens being
// verified) on the gfx950 matrix cores; semantics of kv_attention_into (crates/runtime-cpu/src/napi/mod.rs:
// 3320-3544) as in kv_attention.hip.
//
//   1. kv_append_kernel   writes the new rows (the reference writes first and attends afterwards)
//   2. kv_chunk_kernel    one workgroup per (slot, kv head, 128 query rows, context split); a query row is one
//                         (token, query head of the group), so a K / V tile serves 128 of them where the
//                         streaming kernel reads the context again for every token
//   3. kv_merge_kernel    (kv_attention.hip) where the context is split
//
// S^T = K Q^T with v_mfma_f32_32x32x16: a lane holds the scores of ONE query row (its column) at sixteen of 32
// positions, so the softmax needs one exchange between the two lane halves per step. The same registers are the B
// operand of O^T = V^T P^T: the matrix instruction sums over k in any order, so the A operand is read from V in the
// order in which S^T leaves its positions (ds_read_b64_tr_b16 transposes four positions x sixteen columns on the way)
// and the weights never move between lanes.
//
// Precision: K and V enter the matrix cores as the slab holds them (f16, bf16, or the u8 tier's integers, all exact);
// q and the weights are f32 and enter in pieces whose sum they are: three bfloat16 (24 bits, all of an f32), or two half
// floats where K or V are half floats (23 bits: every fourth value is off by its last bit; q scaled by a power of two per
// row and the weights by 2^12, so that the pieces stay normal). Sums are f32, in short chains: four column chunks of a
// score, or a step's positions of an output, from zero and the small pieces first, then added to the total. Exponents are
// taken against the row's own maximum, so that those of the large weights are small numbers: with the 2^12 inside the
// exponent (weights up to exp2(12)) its rounding was the larger part of the error. Against 64 bits (2-norm, 1e-7;
// streaming kernel / 2^12 in the exponent / this), 32/8 heads x 128, ragged contexts, two slots of 500 tokens at context
// 2000: f16 2.1 / 2.4 / 1.7, bf16 2.1 / 2.3 / 1.5, u8 2.7 / 2.7 / 2.5; eight of 64 at 512: f16 1.9 / 2.4 / 1.6, bf16 1.9 /
// 2.2 / 1.4, u8 2.5 / 2.5 / 2.2; four of 100 at 800, 16/8 heads x 64: f16 2.3 / 2.3 / 1.6. With scores sixteen times as large
// the scores' own error rules: f16 5.4 / 5.3 / 5.3 and bf16 5.3 / 4.6 / 4.6 at 8 x 64, u8 6.6 / 7.4 / 7.3 at 5 x 12 tokens and
// context 2000. (A third half float of q takes 0.1 off the u8 tier's error at ordinary scores and costs 35 % of its time,
// f16 20 %; one chain over everything would add 1.7.)
//
// Eight waves in kGroups groups of kRowWaves: the waves of a group share 32 query rows each, the groups take tiles of
// positions in turn and meet in LDS at the end, so that each SIMD has two waves to issue from. Tiles lie in LDS as in
// the slab, [position][column], with the sixteen-byte pieces of a row swizzled, two buffers per group: the next tile
// is copied (global_load_lds; the u8 tier passes through registers, where it becomes half floats and bfloat16) while
// this one is contracted.
//
// Bound: instruction issue. A wave's scores, weights and products follow one another, and the matrix and vector instructions
// of the two waves of a SIMD hardly run side by side in such long runs (with the waves half a step apart the same time); two
// slots of 500 tokens at context 2000, 32/8 heads x 128: matrix 38 %, vector (softmax, the weights' pieces, the adds of
// the short chains) about 40 % of the cycles of busy compute units, no LDS bank conflicts, compute units busy 76 %
// of the launch (their workgroups have 1500 to 2000 positions). What a tile costs besides: its addresses, found by a lane per
// position one tile ahead and handed out with ds_bpermute; two LDS offsets per lane, from which every operand's address is
// one exclusive or; a row's maximum that is followed to within kSlack. Before these three, and now (us): two slots of 500 at
// 2000 96.7 / 93.4, bf16 115.3 / 106.2, u8 127.1 / 121.2, at 8000 289 / 280 (the streaming kernel took 1036, 1097 and 1322).
// The f16 kernel of four row waves and width 128, alone among the twelve, needs nine registers more than the 256: four of them, a query
// operand, are reloaded at the head of every tile's contraction, and the wait for them is one for the next tile's copies, too,
// which have just been asked for. (Before the three changes one was, with the same wait, and the u8 and bf16 kernels had such reloads.)
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <type_traits>

#include "et_hip.h"
#include "kernels.h"
#include "kv_device.h"

namespace et {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4), aligned(4)));  // of rows that are only whole floats aligned

// An element type of the matrix cores.
struct Half {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ v16f mfma(v8 a, v8 b, v16f c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};
struct BFloat {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ v16f mfma(v8 a, v8 b, v16f c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

// Eight f32 as N vectors of E, each the rounded rest of the ones before.
template <typename E, int N>
__device__ __forceinline__ void split(const float (&x)[8], typename E::v8 (&out)[N]) {
    union Piece {
        typename E::v8 all;
        typename E::v2 pair[4];
    } u[N];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v2f rest = {x[2 * i], x[2 * i + 1]};
#pragma unroll
        for (int p = 0; p < N; p++) {
            u[p].pair[i] = __builtin_convertvector(rest, typename E::v2);
            if (p + 1 < N) {
                rest.x -= static_cast<float>(u[p].pair[i].x);
                rest.y -= static_cast<float>(u[p].pair[i].y);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < N; p++) out[p] = u[p].all;
}

// Slab types: the elements K and V are contracted in, and eight values of a slab row as those.
template <typename T>
struct Slab;
template <>
struct Slab<__half> {
    using K = Half;
    using V = Half;
    using Raw = uint4;
    static constexpr bool kScaled = false;
    static constexpr int kBytes = 2;
    static constexpr int kQueryPieces = 2, kWeightPieces = 2;
    static constexpr float kWeightScale = 4096.0f;  // the half-float pieces of small weights stay normal
    static constexpr int kBlocksPerStep = 2;  // 32-position blocks per softmax step
    static __device__ __forceinline__ uint4 key(Raw raw) { return raw; }
    static __device__ __forceinline__ uint4 value(Raw raw) { return raw; }
};
template <>
struct Slab<Bf16> {
    using K = BFloat;
    using V = BFloat;
    using Raw = uint4;
    static constexpr bool kScaled = false;
    static constexpr int kBytes = 2;
    static constexpr int kQueryPieces = 3, kWeightPieces = 3;
    static constexpr float kWeightScale = 1.0f;
    static constexpr int kBlocksPerStep = 1;  // three pieces of q leave no registers for two
    static __device__ __forceinline__ uint4 key(Raw raw) { return raw; }
    static __device__ __forceinline__ uint4 value(Raw raw) { return raw; }
};
template <>
struct Slab<U8> {
    // byte - 128 is exact in either type; the weights carry V's scales, whose range a half float has not
    using K = Half;
    using V = BFloat;
    using Raw = uint2;
    static constexpr bool kScaled = true;
    static constexpr int kBytes = 1;
    static constexpr int kQueryPieces = 2, kWeightPieces = 3;
    static constexpr float kWeightScale = 1.0f;
    static constexpr int kBlocksPerStep = 1;
    static __device__ __forceinline__ uint4 key(Raw raw) {
        union {
            uint32_t word[4];
            Half::v2 pair[4];
            uint4 all;
        } u;
        const Half::v2 offset = {static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
        u.word[0] = __builtin_amdgcn_perm(0x64646464u, raw.x, 0x04010400u);  // 0x6400 | byte = 1024 + byte
        u.word[1] = __builtin_amdgcn_perm(0x64646464u, raw.x, 0x04030402u);
        u.word[2] = __builtin_amdgcn_perm(0x64646464u, raw.y, 0x04010400u);
        u.word[3] = __builtin_amdgcn_perm(0x64646464u, raw.y, 0x04030402u);
#pragma unroll
        for (int i = 0; i < 4; i++) u.pair[i] = u.pair[i] - offset;
        return u.all;
    }
    static __device__ __forceinline__ uint4 value(Raw raw) {
        union {
            BFloat::v2 pair[4];
            uint4 all;
        } u;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t word = i < 2 ? raw.x : raw.y;
            const v2f wide = {static_cast<float>((word >> (16 * (i & 1))) & 0xffu) - 128.0f,
                              static_cast<float>((word >> (16 * (i & 1) + 8)) & 0xffu) - 128.0f};
            u.pair[i] = __builtin_convertvector(wide, BFloat::v2);
        }
        return u.all;
    }
};

// Weights are at most exp2(kSlack), 4 * 4096 in a half float's pieces, and the rounding of a positive exponent is that of the
// exponents between -2 and 0. With a maximum that is followed exactly nearly every step of 64 positions has one row of 32 that
// moves, and all 32 pay 70 vector instructions for it.
constexpr float kSlack = 2.0f, kMostWeight = 4.0f;
constexpr int kChunkWaves = 8, kChunkThreads = 64 * kChunkWaves;

// RW row waves share a tile (32 * RW query rows per workgroup), 8 / RW groups of them take tiles in turn.
template <typename T, int W, int RW>
struct ChunkShape {
    static constexpr int kGroups = kChunkWaves / RW, kRows = 32 * RW;
    static constexpr int kTile = 16 * RW * 128 / W;        // positions per tile: 16 KiB per row wave in two buffers of K and V
    static constexpr int kPieces = W / 8;                  // sixteen-byte pieces of a row
    static constexpr int kRowsPerCopy = 64 / kPieces;      // positions one wave's copy instruction covers
    static constexpr int kCopies = kTile / (RW * kRowsPerCopy);
    static constexpr uint32_t kRowBytes = W * 2;
    static constexpr uint32_t kTileBytes = kTile * kRowBytes;
    static constexpr uint32_t kBufferBytes = 2 * kTileBytes + (Slab<T>::kScaled ? 2u * kTile * 4u : 0u);
    static constexpr uint32_t kTableAt = 2u * kGroups * kBufferBytes;
    static constexpr uint32_t kLdsBytes = kTableAt + kKvTableEntries * 4u;
    static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");
    static_assert(kTile <= 64 || (kTile == 128 && kCopies % 2 == 0 && 64 % (RW * kRowsPerCopy) == 0), "half of the copies to each 64 positions");
    static_assert(kBufferBytes % 256 == 0 && kTileBytes % 256 == 0, "rows start where the bits of their pieces are zero");
    static_assert(kChunkWaves * (W / 32) * 1024 * 4 <= kTableAt && kChunkWaves * 128 * 4 <= kKvTableEntries * 4,
                  "the waves' sums meet where the tiles and the table were");
    // Piece p of position r of a tile lies in slot p ^ swizzle(r): the 32 positions of a K operand read and the
    // 4 positions x 32 columns of a transposing V read both spread over all banks.
    static __device__ __forceinline__ uint32_t swizzle(uint32_t r) {
        return W == 128 ? ((r & 3u) << 2) | ((r >> 2) & 3u) : (((r >> 1) & 1u) << 2) | ((r >> 2) & 3u);
    }
};

__device__ __forceinline__ float other_half(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __float_as_int(v)));
}

// A copy of sixteen bytes per lane to LDS (lane i to `to` + 16 i) that the compiler does not see: one it saw would
// make it wait for every copy in flight before each LDS read, as it cannot tell their buffers apart. The waves wait
// for their copies themselves before the barrier that hands the buffer over.
__device__ __forceinline__ void copy_unseen(const void* from, uint32_t to) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(to) : "memory", "m0");
}

__device__ __forceinline__ uint2 read_transposed(const uint8_t* from) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    union {
        v4s values;
        uint2 raw;
    } u;
    u.values = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) v4s*)(reinterpret_cast<uintptr_t>(from) & 0xffffffffu));
    return u.raw;
}

// Eight values of a slab row as f32: what the slab holds.
__device__ __forceinline__ void slab_values(const __half*, const uint4& raw, float, float (&out)[8]) {
    union {
        uint4 all;
        Half::v8 half;
    } u;
    u.all = raw;
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = static_cast<float>(u.half[i]);
}
__device__ __forceinline__ void slab_values(const Bf16*, const uint4& raw, float, float (&out)[8]) {
    const uint32_t word[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = __uint_as_float(i & 1 ? word[i / 2] & 0xffff0000u : word[i / 2] << 16);
}
__device__ __forceinline__ void slab_values(const U8*, const uint2& raw, float scale, float (&out)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = u8_value(((i < 4 ? raw.x : raw.y) >> (8 * (i & 3))) & 0xffu, scale);
}

// Up to kRowsAtOnce query rows of one (slot, kv head) by one wave in plain f32, each over its own positions
// [begin, end): the streaming kernel's scheme. W / 8 lanes share a position and hold sixteen bytes of its rows each
// (eight of the u8 tier), so that a K / V row is read once for all of them; 2 * 64 / (W / 8) positions are contracted
// while the next ones are on their way. The running maximum, sum and weighted values are a lane group's own until the end.
// Bound: its vector instructions, about forty per query row and position of a lane group.
constexpr int kRowsAtOnce = 8;
template <typename T, int W>
__device__ void attend_rows(const KvArgs& a, uint32_t slot, uint32_t kv_head, uint32_t split_index, uint32_t count,
                            const uint32_t (&query)[kRowsAtOnce], const uint32_t (&begin)[kRowsAtOnce],
                            const uint32_t (&end)[kRowsAtOnce], int lane) {
    using S = Slab<T>;
    using Raw = typename S::Raw;
    constexpr int R = kRowsAtOnce, U = 2;
    constexpr uint32_t kLanes = W / 8, kAt = 64 / kLanes;
    const uint32_t column = lane % kLanes * 8, offset = lane / kLanes;
    // any position of the rows, and those that all of them see
    uint32_t lo = 0xffffffffu, hi = 0, all_lo = 0, all_hi = 0xffffffffu;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= static_cast<int>(count)) continue;
        if (begin[r] < end[r]) {
            lo = min(lo, begin[r]);
            hi = max(hi, end[r]);
        }
        all_lo = max(all_lo, begin[r]);
        all_hi = min(all_hi, end[r]);
    }
    float q[R][8], o[R][8], m[R], l[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        m[r] = kLowest;
        l[r] = 0.f;
        const v4f* source = reinterpret_cast<const v4f*>(a.q + static_cast<uint64_t>(query[r]) * W + column);
        const v4f low = source[0], high = source[1];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            q[r][i] = (i < 4 ? low[i & 3] : high[i & 3]) * a.scale_log2;
            o[r][i] = 0.f;
        }
    }
    // slab row of a position: first its block's row, which has to arrive before the row itself can be asked for
    const uint32_t* table = a.table + static_cast<uint64_t>(slot) * a.table_stride;
    const auto position_of = [&](uint32_t first, int u) { return min(first + u * kAt + offset, hi - 1); };
    const auto load = [&](const uint32_t (&block)[U], uint32_t first, Raw (&k)[U], Raw (&v)[U], float (&k_scale)[U], float (&v_scale)[U]) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t base = static_cast<uint64_t>(block[u]) * a.block_size;
            const uint32_t at = base >= a.max_tokens ? 0u
                                                     : min(static_cast<uint32_t>(base) + within_block(a, position_of(first, u)), a.max_tokens - 1);
            const uint64_t row = static_cast<uint64_t>(at) * a.kv_heads + kv_head;
            k[u] = *reinterpret_cast<const Raw*>(static_cast<const char*>(a.k_slab) + (row * W + column) * S::kBytes);
            v[u] = *reinterpret_cast<const Raw*>(static_cast<const char*>(a.v_slab) + (row * W + column) * S::kBytes);
            if constexpr (S::kScaled) {
                k_scale[u] = a.k_scales[row];
                v_scale[u] = a.v_scales[row];
            }
        }
    };
    const auto blocks = [&](uint32_t first, uint32_t (&block)[U]) {
#pragma unroll
        for (int u = 0; u < U; u++) block[u] = table[block_of(a, position_of(first, u))];
    };
    uint32_t block[U];
    Raw k_next[U], v_next[U];
    float k_scale[U] = {}, v_scale[U] = {};
    if (lo < hi) {
        blocks(lo, block);
        load(block, lo, k_next, v_next, k_scale, v_scale);
        blocks(lo + U * kAt, block);
    }
    for (uint32_t first = lo; first < hi; first += U * kAt) {
        float key[U][8], value[U][8];
#pragma unroll
        for (int u = 0; u < U; u++) {
            slab_values(static_cast<const T*>(nullptr), k_next[u], k_scale[u], key[u]);
            slab_values(static_cast<const T*>(nullptr), v_next[u], v_scale[u], value[u]);
        }
        if (first + U * kAt < hi) {
            load(block, first + U * kAt, k_next, v_next, k_scale, v_scale);
            blocks(first + 2 * U * kAt, block);
        }
        const bool whole = first >= all_lo && first + U * kAt <= all_hi;  // every row sees all of these
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r >= static_cast<int>(count)) continue;
            float score[U], top = m[r], total = 0.f;
            bool seen[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t position = first + u * kAt + offset;
                seen[u] = whole || (position >= begin[r] && position < end[r]);
                float part = 0.f;
#pragma unroll
                for (int i = 0; i < 8; i++) part = fmaf(q[r][i], key[u][i], part);
                part = group_sum<kLanes>(part);
                score[u] = seen[u] ? part : -INFINITY;
                top = fmaxf(top, score[u]);
            }
            const float keep = __builtin_amdgcn_exp2f(m[r] - top);
#pragma unroll
            for (int u = 0; u < U; u++) {
                score[u] = __builtin_amdgcn_exp2f(score[u] - top);
                total += score[u];
            }
            m[r] = top;
            l[r] = fmaf(l[r], keep, total);
#pragma unroll
            for (int i = 0; i < 8; i++) o[r][i] *= keep;
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                // a weight of zero does not hide an infinite value: positions that are not seen add nothing
                for (int i = 0; i < 8; i++) o[r][i] = fmaf(score[u], seen[u] ? value[u][i] : 0.f, o[r][i]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r >= static_cast<int>(count)) continue;
        float top = m[r];
#pragma unroll
        for (uint32_t step = kLanes; step < 64; step *= 2) top = fmaxf(top, __shfl_xor(top, step));
        const float share = __builtin_amdgcn_exp2f(m[r] - top);
        float total = l[r] * share;
#pragma unroll
        for (int i = 0; i < 8; i++) o[r][i] *= share;
#pragma unroll
        for (uint32_t step = kLanes; step < 64; step *= 2) {
            total += __shfl_xor(total, step);
#pragma unroll
            for (int i = 0; i < 8; i++) o[r][i] += __shfl_xor(o[r][i], step);
        }
        float* record = a.partial + (static_cast<uint64_t>(query[r]) * a.splits + split_index) * (W + 2);
        if (a.splits != 1 && lane == 0) {
            record[0] = top;
            record[1] = total;
        }
        if (offset == 0) {
            float* to = (a.splits == 1 ? a.out + static_cast<uint64_t>(query[r]) * W : record + 2) + column;
            const float divisor = a.splits == 1 ? total : 1.0f;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                v4f joined;
#pragma unroll
                for (int i = 0; i < 4; i++) joined[i] = o[r][4 * j + i] / divisor;
                *reinterpret_cast<v4f*>(to + 4 * j) = joined;
            }
        }
    }
}

template <typename T, int W, int RW>
__global__ __launch_bounds__(kChunkThreads, 2) void kv_chunk_kernel(const KvArgs a) {
    using S = Slab<T>;
    using KE = typename S::K;
    using VE = typename S::V;
    using Raw = typename S::Raw;
    using Shape = ChunkShape<T, W, RW>;
    constexpr int kGroups = Shape::kGroups, kRows = Shape::kRows, kTile = Shape::kTile, kCopies = Shape::kCopies;
    constexpr int kKeyChunks = W / 16, kDimTiles = W / 32, kQueryPieces = S::kQueryPieces, kWeightPieces = S::kWeightPieces;
    constexpr int U = S::kBlocksPerStep < kTile / 32 ? S::kBlocksPerStep : kTile / 32;
    // A weight past that would be infinite, and its row attended to once more: right, and fifteen times slower.
    static_assert(!std::is_same<VE, Half>::value || kMostWeight * S::kWeightScale <= 65504.0f, "weights are half floats");
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];
    uint32_t* rows_of_block = reinterpret_cast<uint32_t*>(lds + Shape::kTableAt);

    // Workgroups of one (slot, kv head) share their K and V in an XCD's L2: the pair runs fastest over the
    // grid, so with eight or more pairs their workgroups go to one XCD. Last rows first: they see most positions.
    const uint32_t group_size = a.query_heads / a.kv_heads;
    const uint32_t pairs = a.active_batch * a.kv_heads;
    const uint32_t rows = a.tokens * group_size, row_tiles = (rows + kRows - 1) / kRows;
    uint32_t index = blockIdx.x;
    const uint32_t pair = index % pairs;
    index /= pairs;
    const uint32_t split_index = index % a.splits;
    const uint32_t first_row = (row_tiles - 1 - index / a.splits) * kRows;
    const uint32_t slot = pair / a.kv_heads, kv_head = pair % a.kv_heads;

    const int lane = threadIdx.x & 63, in_half = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row_wave = wave / kGroups, group = wave % kGroups;

    const Span s = slot_span(a, slot);
    // positions of the workgroup's rows, and this split's part of them in whole rounds of all groups
    uint32_t begin, end, ignored;
    query_range(a, s, first_row / group_size, begin, ignored);
    query_range(a, s, min(first_row + kRows - 1, rows - 1) / group_size, ignored, end);
    const uint32_t length = s.ok && end > begin ? end - begin : 0;
    constexpr uint32_t kRound = kGroups * kTile;
    uint32_t share = (length + a.splits - 1) / a.splits;
    share = (share + kRound - 1) / kRound * kRound;
    const uint32_t my_begin = min(begin + split_index * share, begin + length);
    const uint32_t my_end = min(my_begin + share, begin + length);
    const uint32_t first_block = block_of(a, my_begin);
    if (my_end > my_begin) {
        const uint32_t blocks = block_of(a, my_end - 1) - first_block + 1;
        for (uint32_t i = threadIdx.x; i < blocks && i < kKvTableEntries; i += kChunkThreads) {
            const uint64_t row = static_cast<uint64_t>(a.table[static_cast<uint64_t>(slot) * a.table_stride +
                                                               first_block + i]) * a.block_size;
            rows_of_block[i] = row >= a.max_tokens ? kNoBlock : static_cast<uint32_t>(row);
        }
    }

    // This lane's query row: its column of S^T and O^T.
    const uint32_t row = first_row + 32 * row_wave + in_half;
    const uint32_t live_row = min(row, rows - 1), token = live_row / group_size;
    const uint64_t query = (static_cast<uint64_t>(slot) * a.query_heads + kv_head * group_size + live_row % group_size) *
                               a.tokens + token;
    uint32_t row_begin, row_end;
    query_range(a, s, token, row_begin, row_end);
    // the wave's rows all see [all_begin, all_end), none sees a position outside [any_begin, any_end)
    const uint32_t wave_first = min(first_row + 32 * row_wave, rows - 1), wave_last = min(wave_first + 31, rows - 1);
    uint32_t any_begin, any_end, all_begin, all_end;
    query_range(a, s, wave_first / group_size, any_begin, all_end);
    query_range(a, s, wave_last / group_size, all_begin, any_end);
    const bool has_rows = first_row + 32 * row_wave < rows;

    uint8_t* buffers = lds + group * 2u * Shape::kBufferBytes;
    // Copy i of this wave covers the tile's positions (i * RW + row_wave) * kRowsPerCopy + lane / kPieces, and of those
    // the piece whose slot is lane % kPieces.
    const uint64_t slab_row = static_cast<uint64_t>(a.kv_heads) * W * S::kBytes;
    const char* k_base = static_cast<const char*>(a.k_slab) + static_cast<uint64_t>(kv_head) * W * S::kBytes;
    const char* v_base = static_cast<const char*>(a.v_slab) + static_cast<uint64_t>(kv_head) * W * S::kBytes;
    Raw k_raw[S::kScaled ? kCopies : 1], v_raw[S::kScaled ? kCopies : 1];
    float k_scale[S::kScaled ? kCopies : 1], v_scale[S::kScaled ? kCopies : 1];
    const auto tile_row = [&](int i) { return static_cast<uint32_t>((i * RW + row_wave) * Shape::kRowsPerCopy + lane / Shape::kPieces); };
    // Slab rows of a tile's positions, found a tile ahead, a lane to a position.
    constexpr int kPlaces = (kTile + 63) / 64;
    uint32_t place[kPlaces];
    const auto locate = [&](uint32_t tile_begin) {
        uint32_t block[kPlaces], within[kPlaces];
        // positions past the end read the last row again; their weights are zero
        const auto position = [&](int i) { return min(tile_begin + 64 * i + lane, my_end - 1); };
#pragma unroll
        for (int i = 0; i < kPlaces; i++) {
            if (a.block_shift >= 0) {
                block[i] = position(i) >> a.block_shift;
                within[i] = position(i) & (a.block_size - 1);
            } else {
                block[i] = position(i) / a.block_size;
                within[i] = position(i) - block[i] * a.block_size;
            }
        }
#pragma unroll
        for (int i = 0; i < kPlaces; i++) {
            const uint32_t base = rows_of_block[min(block[i] - first_block, kKvTableEntries - 1u)];
            const uint32_t at = min(base + within[i], a.max_tokens - 1);
            place[i] = base == kNoBlock ? 0u : at;
        }
    };
    const auto fetch = [&](uint32_t buffer) {
#pragma unroll
        for (int i = 0; i < kCopies; i++) {
            const uint32_t r = tile_row(i), piece = (lane % Shape::kPieces) ^ Shape::swizzle(r);
            const uint32_t at = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute((r & 63u) << 2, place[i * kPlaces / kCopies]));
            const uint64_t from = static_cast<uint64_t>(at) * slab_row + piece * (8 * S::kBytes);
            if constexpr (S::kScaled) {
                k_raw[i] = *reinterpret_cast<const Raw*>(k_base + from);
                v_raw[i] = *reinterpret_cast<const Raw*>(v_base + from);
                if (lane % Shape::kPieces == 0) {
                    k_scale[i] = a.k_scales[static_cast<uint64_t>(at) * a.kv_heads + kv_head];
                    v_scale[i] = a.v_scales[static_cast<uint64_t>(at) * a.kv_heads + kv_head];
                }
            } else {
                const uint32_t to = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
                    buffers + buffer * Shape::kBufferBytes + (i * RW + row_wave) * 1024u)));
                copy_unseen(k_base + from, to);
                copy_unseen(v_base + from, to + Shape::kTileBytes);
            }
        }
    };
    const auto deposit = [&](uint32_t buffer) {
        if constexpr (S::kScaled) {
            uint8_t* tile = buffers + buffer * Shape::kBufferBytes;
            float* scales = reinterpret_cast<float*>(tile + 2 * Shape::kTileBytes);
#pragma unroll
            for (int i = 0; i < kCopies; i++) {
                uint8_t* to = tile + (i * RW + row_wave) * 1024u + lane * 16u;
                *reinterpret_cast<uint4*>(to) = S::key(k_raw[i]);
                *reinterpret_cast<uint4*>(to + Shape::kTileBytes) = S::value(v_raw[i]);
                if (lane % Shape::kPieces == 0) {
                    // Of a K row with an infinite scale every value is infinite or, byte 128, NaN, and so are its products with q:
                    // NaN, not the infinity that the scale makes of the whole sum (-inf would pass for a weight of zero).
                    scales[tile_row(i)] = fabsf(k_scale[i]) < INFINITY ? k_scale[i] : NAN;
                    scales[kTile + tile_row(i)] = v_scale[i];
                }
            }
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies have landed
        }
    };

    __syncthreads();  // the table is in LDS
    const uint32_t rounds = (my_end - my_begin + kRound - 1) / kRound;
    uint32_t tile_begin = my_begin + group * kTile;
    if (rounds != 0) {
        locate(tile_begin);
        fetch(0);
        locate(tile_begin + kRound);
    }

    // q in pieces, scaled so that the row's largest component lies in [2^9, 2^10); the score's unit undoes it.
    typename KE::v8 q[kQueryPieces][kKeyChunks];
    float unit;
    {
        const auto load = [&](int c, float (&x)[8]) {
            const v4f* source = reinterpret_cast<const v4f*>(a.q + query * W + 16 * c + 8 * half);
            const v4f low = source[0], high = source[1];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                x[i] = low[i];
                x[4 + i] = high[i];
            }
        };
        float x[8], top = 0.f;
#pragma unroll
        for (int c = 0; c < kKeyChunks; c++) {
            load(c, x);
#pragma unroll
            for (int i = 0; i < 8; i++) top = fmaxf(top, fabsf(x[i]));
        }
        top = fmaxf(top, other_half(top, lane));
        int exponent;
        (void)frexpf(top, &exponent);
        exponent = max(exponent, -100);
        const float up = a.scale_log2 == 0.f ? 0.f : copysignf(ldexpf(1.0f, 10 - exponent), a.scale_log2);
        unit = a.scale_log2 == 0.f ? 1.0f : ldexpf(fabsf(a.scale_log2), exponent - 10);
#pragma unroll
        for (int c = 0; c < kKeyChunks; c++) {
            load(c, x);
#pragma unroll
            for (int i = 0; i < 8; i++) x[i] *= up;
            typename KE::v8 pieces[kQueryPieces];
            split<KE, kQueryPieces>(x, pieces);
#pragma unroll
            for (int p = 0; p < kQueryPieces; p++) q[p][c] = pieces[p];
        }
    }

    float m = kLowest, l = 0.f;
    v16f o[kDimTiles], zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.f;
#pragma unroll
    for (int t = 0; t < kDimTiles; t++) o[t] = zero;

    // K operand of a 32-position block: position in_half, pieces 2c + half. V operand: positions
    // 16c + 8h + 4 half + (0..3), of which this lane's address names row (lane & 15) / 4 and four of sixteen columns.
    // A row's pieces fill the bits of the address that the swizzle changes, so c, h and the column tile come in with one
    // exclusive or each, and no lane keeps more than these two offsets.
    const uint32_t key_at = in_half * Shape::kRowBytes + ((half ^ Shape::swizzle(in_half)) << 4);
    const uint32_t value_row = 4 * half + ((lane & 15) >> 2), value_piece = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    const uint32_t value_at = Shape::kTileBytes + value_row * Shape::kRowBytes +
                              ((value_piece ^ Shape::swizzle(value_row)) << 4) + (lane & 1) * 8;
    const auto contract = [&](uint32_t buffer, uint32_t tile) {
        const uint32_t keys = buffer + key_at, values = buffer + value_at;
        const float* scales = reinterpret_cast<const float*>(lds + buffer + 2 * Shape::kTileBytes);
#pragma unroll
        for (int b = 0; b < kTile / 32; b += U) {
            const uint32_t step = tile + 32 * b;
            if (step >= any_end || step + 32 * U <= any_begin) continue;  // uniform in the wave
            v16f score[U];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int first = 0; first < kKeyChunks; first += 4) {
                    typename KE::v8 key[4];
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        key[c] = *reinterpret_cast<const typename KE::v8*>(lds + (keys ^ ((first + c) << 5)) + 32 * (b + u) * Shape::kRowBytes);
                    v16f sum = zero;
#pragma unroll
                    for (int p = kQueryPieces - 1; p >= 0; p--)
#pragma unroll
                        for (int c = 0; c < 4; c++) sum = KE::mfma(key[c], q[p][first + c], sum);
                    score[u] = first == 0 ? sum : score[u] + sum;
                }
            if constexpr (S::kScaled) {
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float4 k4 = *reinterpret_cast<const float4*>(scales + 32 * (b + u) + 8 * j + 4 * half);
                        score[u][4 * j] *= k4.x;
                        score[u][4 * j + 1] *= k4.y;
                        score[u][4 * j + 2] *= k4.z;
                        score[u][4 * j + 3] *= k4.w;
                    }
            }
            if (step < all_begin || step + 32 * U > all_end) {  // some row of the wave does not see all of these
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const uint32_t position = step + 32 * u + 8 * (r / 4) + 4 * half + (r & 3);
                        if (position < row_begin || position >= row_end) score[u][r] = -INFINITY;
                    }
            }
            float top = score[0][0];
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int r = 0; r < 16; r++) top = fmaxf(top, score[u][r]);
            top = fmaxf(top, other_half(top, lane));
            // The reference point of a row's exponents may lie up to kSlack below its maximum.
            const float next = fmaxf(m, top * unit);
            if (__builtin_amdgcn_ballot_w64(next > m + kSlack) != 0) {
                const float keep = __builtin_amdgcn_exp2f(m - next);
                m = next;
                l *= keep;
#pragma unroll
                for (int t = 0; t < kDimTiles; t++)
#pragma unroll
                    for (int r = 0; r < 16; r++) o[t][r] *= keep;
            }
            // The weights of the whole step, then the values 32 columns at a time.
            typename VE::v8 pieces[2 * U][kWeightPieces];
            float step_sum = 0.f;
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    float weight[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        weight[i] = __builtin_amdgcn_exp2f(fmaf(score[u][8 * c + i], unit, -m));
                        if constexpr (S::kWeightScale != 1.0f) weight[i] *= S::kWeightScale;
                        step_sum += weight[i];
                    }
                    if constexpr (S::kScaled) {
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            const float4 v4 = *reinterpret_cast<const float4*>(scales + kTile + 32 * (b + u) + 16 * c + 8 * j +
                                                                               4 * half);
                            weight[4 * j] *= v4.x;
                            weight[4 * j + 1] *= v4.y;
                            weight[4 * j + 2] *= v4.z;
                            weight[4 * j + 3] *= v4.w;
                        }
                    }
                    split<VE, kWeightPieces>(weight, pieces[2 * u + c]);
                }
            }
            l += step_sum;
#pragma unroll
            for (int t = 0; t < kDimTiles; t++) {
                union {
                    uint2 raw[2];
                    typename VE::v8 all;
                } value[2 * U];
#pragma unroll
                for (int c = 0; c < 2 * U; c++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        value[c].raw[h] = read_transposed(lds + (values ^ (t * 64 + h * 32)) + (32 * b + 16 * c + 8 * h) * Shape::kRowBytes);
                v16f sum = zero;
#pragma unroll
                for (int p = kWeightPieces - 1; p >= 0; p--)
#pragma unroll
                    for (int c = 0; c < 2 * U; c++) sum = VE::mfma(value[c].all, pieces[c][p], sum);
                o[t] += sum;
            }
        }
    };

    if (rounds != 0) {
        // all groups run the same number of rounds; a group whose tile lies past the end reads the last row
        deposit(0);
        __syncthreads();
        for (uint32_t round = 0; round < rounds; round++, tile_begin += kRound) {
            const bool more = round + 1 < rounds;
            if (more) {
                fetch((round + 1) & 1);
                locate(tile_begin + 2 * kRound);
            }
            if (has_rows && tile_begin < my_end) contract((2u * group + (round & 1)) * Shape::kBufferBytes, tile_begin);
            if (more) deposit((round + 1) & 1);
            __syncthreads();
        }
    }
    // NaN where a sum is not finite
#pragma unroll
    for (int t = 0; t < kDimTiles; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) l = fmaf(o[t][r], 0.f, l);
    l += other_half(l, lane);

    // All groups leave their sums in LDS (the tiles and the table are read no more); each group's wave then joins a
    // share of the 32-column tiles of its rows, in group order.
    float* sums = reinterpret_cast<float*>(lds) + lane;
    float* weights = reinterpret_cast<float*>(lds + Shape::kTableAt) + lane;
    const auto sums_of = [&](int g, int t) { return sums + ((g * RW + row_wave) * kDimTiles + t) * 1024; };
    const auto weights_of = [&](int g) { return weights + (g * RW + row_wave) * 128; };
    weights_of(group)[0] = m;
    weights_of(group)[64] = l;
#pragma unroll
    for (int t = 0; t < kDimTiles; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) sums_of(group, t)[64 * r] = o[t][r];
    __syncthreads();
    float share_of[kGroups], top = kLowest, total = 0.f;
#pragma unroll
    for (int g = 0; g < kGroups; g++) top = fmaxf(top, weights_of(g)[0]);
#pragma unroll
    for (int g = 0; g < kGroups; g++) {
        share_of[g] = __builtin_amdgcn_exp2f(weights_of(g)[0] - top) * (1.0f / S::kWeightScale);
        total = fmaf(share_of[g], weights_of(g)[64], total);
    }
    const bool live = row < rows && s.ok, again = live && !(fabsf(total) < INFINITY);
    if (live && !again) {
        float* record = a.partial + (query * a.splits + split_index) * (W + 2);
        if (a.splits != 1 && group == 0 && half == 0) {
            record[0] = top;
            record[1] = total;
        }
        float* to = (a.splits == 1 ? a.out + query * W : record + 2) + 4 * half;
        const float divisor = a.splits == 1 ? total : 1.0f;
        for (int t = group; t < kDimTiles; t += kGroups) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v4f joined;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float value = 0.f;
#pragma unroll
                    for (int g = 0; g < kGroups; g++) value = fmaf(share_of[g], sums_of(g, t)[64 * (4 * j + i)], value);
                    joined[i] = value / divisor;
                }
                *reinterpret_cast<v4f*>(to + 32 * t + 8 * j) = joined;
            }
        }
    }
    // An infinity or NaN in a K or V row spoils the matrix products of every query row it shares a tile with, also of those
    // that do not see its position, and a product of pieces overflows or meets inf - inf before the product itself does.
    // Such rows are attended to once more, without pieces and over their own positions alone. Two slots of 500 tokens at
    // context 2000 with a NaN at position 0 of one, which all its rows see: f16 1337 us, u8 1494 (all finite 93 and 126; row
    // after row, a lane to a position, 6617 and 7408; the streaming kernel 1036 and 1322 whatever the values); eight slots
    // of 64 tokens at context 512, f16, 363 (1691); a NaN in one row of q of the former 178 (332).
    uint32_t left = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(again));
    const uint32_t begin_here = max(row_begin, my_begin), end_here = min(row_end, my_end);
    for (int turn = 0; left != 0; turn++) {
        uint32_t query_of[kRowsAtOnce], begin_of[kRowsAtOnce], end_of[kRowsAtOnce], count = 0;
#pragma unroll
        for (int r = 0; r < kRowsAtOnce; r++) {
            const int which = left != 0 ? __builtin_ctz(left) : 0;
            count += left != 0 ? 1 : 0;
            left &= left - 1;
            query_of[r] = __builtin_amdgcn_readlane(static_cast<uint32_t>(query), which);
            begin_of[r] = __builtin_amdgcn_readlane(begin_here, which);
            end_of[r] = __builtin_amdgcn_readlane(end_here, which);
        }
        if (turn % kGroups == group) attend_rows<T, W>(a, slot, kv_head, split_index, count, query_of, begin_of, end_of, lane);
    }
}

// A wave per (slot, token, kv head): the token's K and V row as the slab stores them, and the slot's status.
template <typename T>
__global__ __launch_bounds__(256) void kv_append_kernel(const KvArgs a, uint32_t count) {
    const uint32_t item = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (item >= count) return;
    const uint32_t kv_head = item % a.kv_heads, token = item / a.kv_heads % a.tokens, slot = item / a.kv_heads / a.tokens;
    const Span s = slot_span(a, slot);
    if (token == 0 && kv_head == 0) write_slot_status(a, slot, s, lane);
    if (!s.ok || token >= s.advance) return;
    const uint32_t position = s.cursor + token;
    const uint64_t row = static_cast<uint64_t>(a.table[static_cast<uint64_t>(slot) * a.table_stride + block_of(a, position)]) *
                             a.block_size + within_block(a, position);
    if (row >= a.max_tokens) return;  // reported by the slot's status
    const uint64_t at = (row * a.kv_heads + kv_head) * a.width;
    const uint64_t source = ((static_cast<uint64_t>(slot) * a.kv_heads + kv_head) * a.tokens + token) * a.width;
#pragma unroll
    for (int which = 0; which < 2; which++) {
        const float* from = (which == 0 ? a.k : a.v) + source;
        T* to = static_cast<T*>(which == 0 ? a.k_slab : a.v_slab) + at;
        if constexpr (std::is_same<T, U8>::value) {
            float top = 0.f;
            for (uint32_t column = lane; column < a.width; column += 64) top = fmaxf(top, fabsf(from[column]));
            const float scale = u8_scale(group_max<64>(top));
            if (lane == 0) (which == 0 ? a.k_scales : a.v_scales)[row * a.kv_heads + kv_head] = scale;
            for (uint32_t column = lane; column < a.width; column += 64)
                to[column].byte = static_cast<uint8_t>(u8_byte(from[column], scale));
        } else {
            for (uint32_t column = lane; column < a.width; column += 64) slab_store(to, column, from[column]);
        }
    }
}

template <typename T, int W, int RW>
hipError_t launch_chunk(const KvArgs& a, uint32_t workgroups, hipStream_t stream) {
    using Shape = ChunkShape<T, W, RW>;
    auto* kernel = kv_chunk_kernel<T, W, RW>;
    // More than 64 KiB of dynamic LDS has to be allowed once per kernel and device.
    constexpr int kDevices = 64;
    static std::atomic<bool> allowed[kDevices] = {};
    int device = 0;
    if (hipError_t error = hipGetDevice(&device); error != hipSuccess) return error;
    if (device < 0 || device >= kDevices || !allowed[device].load(std::memory_order_acquire)) {
        const hipError_t error = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, Shape::kLdsBytes);
        if (error != hipSuccess) return error;
        if (device >= 0 && device < kDevices) allowed[device].store(true, std::memory_order_release);
    }
    const uint32_t count = a.active_batch * a.tokens * a.kv_heads;
    hipLaunchKernelGGL(kv_append_kernel<T>, dim3((count + 3) / 4), dim3(256), 0, stream, a, count);
    if (hipError_t error = hipGetLastError(); error != hipSuccess) return error;
    hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(kChunkThreads), Shape::kLdsBytes, stream, a);
    return hipGetLastError();
}

template <typename T, int W>
hipError_t launch_chunk_rows(const KvArgs& a, int row_waves, uint32_t workgroups, hipStream_t stream) {
    return row_waves == 4 ? launch_chunk<T, W, 4>(a, workgroups, stream) : launch_chunk<T, W, 2>(a, workgroups, stream);
}

template <typename T>
hipError_t launch_chunk_width(const KvArgs& a, int row_waves, uint32_t workgroups, hipStream_t stream) {
    return a.width == 128 ? launch_chunk_rows<T, 128>(a, row_waves, workgroups, stream)
                          : launch_chunk_rows<T, 64>(a, row_waves, workgroups, stream);
}

}  // namespace

bool kv_chunk_supported(const KvAttention& p) {
    return (p.width == 64 || p.width == 128) && p.tokens > 1 &&
           (p.slab_dtype == ET_DTYPE_F16 || p.slab_dtype == ET_DTYPE_BF16 || p.slab_dtype == ET_DTYPE_U8);
}

KvChunkGrid kv_chunk_grid(const KvAttention& p) {
    KvChunkGrid grid{};
    const uint64_t rows = static_cast<uint64_t>(p.tokens) * (p.query_heads / p.kv_heads);
    grid.row_waves = rows <= 64 ? 2 : 4;
    grid.units = static_cast<uint64_t>(p.active_batch) * p.kv_heads * ((rows + 32 * grid.row_waves - 1) / (32 * grid.row_waves));
    grid.round = kChunkWaves * 16 * 128 / p.width;
    return grid;
}

hipError_t kv_chunk(int32_t slab_dtype, const KvArgs& a, int row_waves, uint32_t workgroups, hipStream_t stream) {
    switch (slab_dtype) {
        case ET_DTYPE_F16: return launch_chunk_width<__half>(a, row_waves, workgroups, stream);
        case ET_DTYPE_BF16: return launch_chunk_width<Bf16>(a, row_waves, workgroups, stream);
        case ET_DTYPE_U8: return launch_chunk_width<U8>(a, row_waves, workgroups, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace et
