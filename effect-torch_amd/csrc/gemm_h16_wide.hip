// gemm_h16.hip's contraction (the same operands in half floats) for prompts. A workgroup contracts 128
// vectors with 256 weight rows (Q2_K, Q6_K: 128), so that weights are unpacked once for 128 (64) vectors instead of for
// every 32, and an activation tile is copied for 256 rows instead of 64 or 128.
//
// Bound: matrix instructions together with the LDS reads of their operands. Eight waves, two per SIMD, each 128 vectors x 32 rows
// (Q2_K, Q6_K, which contract two operands per weight: 64 x 32). A Q4_K wave's stage of 256 columns is 128 half-float matrix
// instructions, eight bfloat16 ones for the minima (32 cycles each), 165 LDS instructions, as an activation operand (16 bytes a
// lane, about eight cycles of the compute unit's LDS) serves one matrix instruction, and about 520 vector instructions. 14336 x
// 4096 with 1000 vectors: 240 us, 27.6 ns per matrix instruction of a SIMD, matrix pipes busy 68 % of the cycles of busy compute units at 1.93
// GHz. Loops on random operands, two waves per SIMD: matrix instructions alone 21.3 ns (zeros 14.3: their power takes the
// clock down), with six, ten and twelve LDS reads to ten of them 25.0, 27.5 and 30.8. Left: operands that serve two matrix
// instructions (64 x 64 per wave, every weight unpacked twice), and 448 workgroups on 256 compute units, an eighth of them idle.
// Vector instructions, up to seven for a matrix instruction, cost next to nothing where they lie evenly between them (loops of
// both, two waves per SIMD): the next sub-block's operands are made between this one's matrix instructions, and a stage's sums
// are folded into the accumulators tile by tile between the next tile's. The minima were f32 matrix instructions (16 of 64
// cycles per stage, a fifth of the pipe's time); now a sub-block's sum, an f32, is divided by the vector's unit and the
// quotient, rounded to 24 bits, is cut into three bfloat16 pieces that add up to it exactly, once per workgroup; their products are
// exact. Clocks of busy compute units before these steps, with them, and with the nibbles' eight instructions less per sub-block
// (packed_nibbles_times): 122.5, 99.6 and 92.2 million.
// Every wave unpacks its own weight rows from the packed bytes in LDS. There are no loader waves (a third wave per SIMD
// would leave 168 registers each): the waves ask for the next sub-blocks' activations and the next stage's weights
// themselves, through inline assembly, because any LDS read next to a copy that the compiler can see waits for it.
// Q4_K and Q5_K have all 256 registers and spill 12 and 16, in the last stage and the stores.
//
// Whole calls (us, gemm_h16_kernel / this before those steps / this): 14336 x 4096 with 1000 vectors Q4_K 415 / 294 / 259 (453
// TFLOP/s), Q5_K 445 / 301 / 266, Q6_K 730 / 474 / 437, Q3_K 434 / 268 / 254, Q2_K 534 / 426 / 399; Q4_K 4096 x 14336 with 1000
// 390 / 293 / 266, 14336 x 4096 with 256 121 / 95 / 88. In launches of one stage per workgroup the separate last stage is no gain: Q6_K
// 622 x 3584 with 371 vectors 42.0 / 34.3 / 35.2 (one loop for all stages: 35.7, and 1000 vectors 447 instead of 418).
// Relative error against 64 bits there (2-norm, 1e-7): Q4_K 1.75 / 1.69 / 1.66, Q6_K 1.66 / 1.63 / 1.63, Q2_K 1.84 / 1.76 / 1.76:
// one chain of sums over the stage's eight sub-blocks instead of two or four, from activations that are rounded less (quantize_halves.h).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <type_traits>

#include "gemm_h16_device.h"

namespace et {
namespace {

typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8;
constexpr int kTiles = kGemmWideVectors / 32;        // activation tiles per workgroup
constexpr int kSlots = 4;                            // sub-blocks of activations in LDS: two landed, two on their way
constexpr uint32_t kSlotBytes = kTiles * 2 * 2048u;  // per tile and plane four 8-column parts of 512 bytes
constexpr int kCutAt = 3;                            // the sub-block in which the stage's sums are cut: they have landed by then
constexpr int kActivationCopies = 2;                 // per wave and sub-block: one plane of one tile
static_assert(kTiles * 2 == kWaves && kStageBlocks % kSlots == 0, "a wave copies one plane of one tile; slots start anew per stage");

template <int CODEC>
struct Wide {
    static constexpr bool kMinima = CODEC == kQ4_K || CODEC == kQ5_K;  // a minimum per sub-block, against xsum
    static constexpr int kParts = weight_parts(CODEC);
    static constexpr int kMT = kParts == 2 ? 2 : 4;  // 32-vector tiles per wave, against 32 rows
    static constexpr int kWavesM = kTiles / kMT, kWavesN = kWaves / kWavesM;
    static constexpr uint32_t kRows = 32u * kWavesN;
    static constexpr uint32_t kRowBytes = HalfStage<CODEC>::kRowBytes;
    static constexpr uint32_t kWeightBytes = kRows * kRowBytes;
    static constexpr int kWeightJobs = kWeightBytes / 1024;
    static_assert(kWeightBytes % 1024 == 0, "whole copy instructions");
    static constexpr int kRounds = (kWeightJobs + kWaves - 1) / kWaves;  // weight copies per wave and stage, one per sub-block
    static_assert(kRounds <= kStageBlocks - 2, "landed before the last sub-block");
    // the activation slots; one stage of unit[m] (512 bytes, copied twice) and of xsum; two stages of weights
    // (and, in their place, the sums cut into three bfloat16 pieces, [tile][piece][vector][sub-block])
    static constexpr uint32_t kUnitsAt = kSlots * kSlotBytes, kSumsAt = kUnitsAt + 1024u,
                              kWeightsAt = kSumsAt + (kMinima ? kTiles * 1536u : 0u), kLdsBytes = kWeightsAt + 2 * kWeightBytes;
    static_assert(kLdsBytes <= 160 * 1024, "LDS of a gfx950 CU: 160 KiB, all of it dynamic here");
    // copies that a wave asks for in front of the activations during sub-block b: the stage's tables, next weights
    static constexpr int ahead(int b, bool last) { return (b == 0 ? 1 : 0) + (!last && b < kRounds ? 1 : 0); }
};

// 1 KiB from `base` + a byte offset per lane to LDS address `to` + 16 bytes per lane.
__device__ __forceinline__ void copy_to_lds(const uint8_t* base, uint32_t lane_offset, uint32_t to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(to)), "v"(lane_offset), "s"(base)
                 : "m0", "memory");
}

// The packed bytes of one lane's columns 32 b + 16 half .. + 16 of a row, as they come out of LDS.
struct Raw {
    uint4 low, high;
    uint32_t scale, scale_top;
};
// What all of a row's sub-blocks share: d, dmin and the scales (Q4_K, Q5_K); the fifth (Q5_K) or top (Q3_K) bits.
struct Shared {
    uint4 header, bits;
};
template <int CODEC>
__device__ __forceinline__ Shared fetch_shared(const uint8_t* row, uint32_t half) {
    Shared s = {};
    if constexpr (CODEC == kQ4_K || CODEC == kQ5_K) s.header = *reinterpret_cast<const uint4*>(row);
    if constexpr (CODEC == kQ5_K) s.bits = *reinterpret_cast<const uint4*>(row + 16u + 16u * half);
    if constexpr (CODEC == kQ3_K) s.bits = *reinterpret_cast<const uint4*>(row + 16u * half);
    return s;
}
template <int CODEC>
__device__ __forceinline__ Raw fetch(const uint8_t* row, int b, uint32_t half) {
    const uint32_t n = b >> 2, t = b & 3;
    Raw r = {};
    if constexpr (CODEC == kQ4_K || CODEC == kQ5_K) {
        r.low = *reinterpret_cast<const uint4*>(row + HalfStage<CODEC>::kQuantsAt + 32u * (b >> 1) + 16u * half);
    } else if constexpr (CODEC == kQ6_K) {
        r.low = *reinterpret_cast<const uint4*>(row + 64u * n + 32u * (t & 1u) + 16u * half);
        r.high = *reinterpret_cast<const uint4*>(row + 128u + 32u * n + 16u * half);
        r.scale = row[192u + 8u * n + 2u * t + half];
    } else if constexpr (CODEC == kQ3_K) {
        r.low = *reinterpret_cast<const uint4*>(row + 32u + 32u * n + 16u * half);
        r.scale = row[HalfStage<CODEC>::in_tail(96u) + 2u * t + half];
        r.scale_top = row[HalfStage<CODEC>::in_tail(104u) + 2u * (t & 1u) + half];
    } else {
        r.low = *reinterpret_cast<const uint4*>(row + 16u + 32u * n + 16u * half);
        r.scale = row[2u * b + half];
    }
    return r;
}
__device__ __forceinline__ v2h twice(int value) {
    const _Float16 h = static_cast<_Float16>(static_cast<float>(value));
    return v2h{h, h};
}
// The weight operands of those columns, eight by eight: gemm_h16_kernel's values.
template <int CODEC>
__device__ __forceinline__ void operands(const Raw& raw, const Shared& shared, int b, v8h out[2][weight_parts(CODEC)]) {
    const uint32_t n = b >> 2, t = b & 3;
    const uint32_t low[4] = {raw.low.x, raw.low.y, raw.low.z, raw.low.w}, high[4] = {raw.high.x, raw.high.y, raw.high.z, raw.high.w};
    const uint32_t bits[4] = {shared.bits.x, shared.bits.y, shared.bits.z, shared.bits.w};
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if constexpr (CODEC == kQ4_K || CODEC == kQ5_K) {
            w[i] = (low[i] >> ((b & 1) * 4)) & 0x0f0f0f0fu;
            if constexpr (CODEC == kQ5_K) w[i] |= ((bits[i] >> b) & 0x01010101u) << 4;
        } else if constexpr (CODEC == kQ6_K) {
            w[i] = ((low[i] >> ((t >> 1) * 4u)) & 0x0f0f0f0fu) | (((high[i] >> (2u * t)) & 0x03030303u) << 4);
        } else {
            w[i] = (low[i] >> (2u * t)) & 0x03030303u;
            if constexpr (CODEC == kQ3_K) w[i] |= ((bits[i] >> (4u * n + t)) & 0x01010101u) << 2;
        }
    }
    if constexpr (CODEC == kQ4_K || CODEC == kQ5_K) {
        uint32_t sc, mn;
        q4k_scale_min(shared.header, b, sc, mn);
        const v2h scale = twice(sc);
        if (CODEC == kQ4_K && (b & 1)) {
            out[0][0] = packed_nibbles_times<true>(low[0], low[1], scale);
            out[1][0] = packed_nibbles_times<true>(low[2], low[3], scale);
        } else if (CODEC == kQ4_K) {
            out[0][0] = packed_nibbles_times<false>(low[0], low[1], scale);
            out[1][0] = packed_nibbles_times<false>(low[2], low[3], scale);
        } else {
            out[0][0] = nibbles_times(w[0], w[1], scale);
            out[1][0] = nibbles_times(w[2], w[3], scale);
        }
    } else if constexpr (CODEC == kQ6_K) {
        const int sc = static_cast<int8_t>(raw.scale);
        const v2h scale_low = twice(sc & 15), scale_high = twice(sc >> 4);
        out[0][0] = nibbles_times<32>(w[0], w[1], scale_low);
        out[1][0] = nibbles_times<32>(w[2], w[3], scale_low);
        out[0][1] = nibbles_times<32>(w[0], w[1], scale_high);
        out[1][1] = nibbles_times<32>(w[2], w[3], scale_high);
    } else if constexpr (CODEC == kQ3_K) {
        const int sc = static_cast<int>(((raw.scale >> (4u * n)) & 15u) |
                                        (((raw.scale_top >> (2u * (2u * n + (t >> 1)))) & 3u) << 4)) - 32;
        const v2h scale = twice(sc);
        out[0][0] = bytes_minus_times<4>(w[0], w[1], scale);
        out[1][0] = bytes_minus_times<4>(w[2], w[3], scale);
    } else {
        const v2h scale = twice(raw.scale & 15u), m = twice(raw.scale >> 4);
        out[0][0] = nibbles_times(w[0], w[1], scale);
        out[1][0] = nibbles_times(w[2], w[3], scale);
        out[0][1] = out[1][1] = v8h{m.x, m.x, m.x, m.x, m.x, m.x, m.x, m.x};
    }
}

// f32 bits as three bfloat16 numbers that add up to it, eight significant bits each: the top halves of `x`, of
// what is left of it, and of what is left then (nothing is lost above 2^-110). Of an infinity nothing is left.
struct Pieces {
    uint32_t high, mid, low;  // in the upper sixteen bits
};
__device__ __forceinline__ Pieces cut(float x) {
    Pieces p;
    p.high = __float_as_uint(x) & 0xffff0000u;
    const float rest = __builtin_isinf(x) ? 0.f : x - __uint_as_float(p.high);
    p.mid = __float_as_uint(rest) & 0xffff0000u;
    p.low = __float_as_uint(rest - __uint_as_float(p.mid));
    return p;
}
__device__ __forceinline__ v8bf as_bf16(const v8s& bits) { return __builtin_bit_cast(v8bf, bits); }
// The eight minima of this lane's row, against the high (lane half 0) and middle pieces, and against the low ones
// (half 0 alone: the operand's other eight columns are zero).
__device__ __forceinline__ void minimum_operands(const uint4& header, uint32_t half, v8s out[2]) {
#pragma unroll
    for (uint32_t g = 0; g < kStageBlocks; g++) {
        uint32_t sc, mn;
        q4k_scale_min(header, g, sc, mn);
        out[0][g] = static_cast<short>(__float_as_uint(static_cast<float>(mn)) >> 16);  // at most 63: exact
    }
    out[1] = half == 0 ? out[0] : v8s{0, 0, 0, 0, 0, 0, 0, 0};
}

template <int CODEC>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_h16_wide_kernel(const Group group, const uint8_t* __restrict__ tiles,
                                                                       uint32_t vector_tiles, uint32_t columns,
                                                                       uint32_t vectors, uint32_t k_splits,
                                                                       float* __restrict__ partials) {
    using W = Wide<CODEC>;
    constexpr uint32_t kRowBytes = W::kRowBytes, kStageBytes = HalfStage<CODEC>::kStageBytes;
    constexpr int MT = W::kMT, P = W::kParts;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    // Workgroups go to the eight XCDs round-robin: the vector groups of one (row tile, K share) run on the same XCD, next
    // to each other in time, so the later ones find the weights in its L2. (Row tiles whole to an XCD each, as in
    // gemm_h16.hip, leave some XCDs a second turn: 5000 x 3072 with 333 vectors 72 us.)
    const uint32_t xcd = blockIdx.x & 7u, turn = blockIdx.x >> 3;
    const uint32_t vector_groups = (vector_tiles + kTiles - 1u) / kTiles;
    const uint32_t vector_group = turn % vector_groups, pair = (turn / vector_groups) * 8u + xcd;
    const uint32_t row_tile = pair / k_splits, k_share = pair % k_splits;
    if (row_tile >= group.row_tiles) return;
    uint32_t which = 0;
    for (uint32_t i = 1; i < group.count; i++)
        if (row_tile >= group.member[i].first_tile) which = i;
    const Member& member = group.member[which];
    const uint32_t rows = member.rows;

    const uint32_t lane = threadIdx.x & 63u, half = lane >> 5, in_half = lane & 31u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wave_n = wave % W::kWavesN, wave_m = wave / W::kWavesN;
    const uint32_t all_stages = columns / 256u, share = (all_stages + k_splits - 1u) / k_splits;
    const uint32_t first_stage = k_share * share;  // < all_stages: the launcher leaves no share empty
    const uint32_t stages = min(share, all_stages - first_stage);
    const uint32_t row_bytes = all_stages * kStageBytes;
    const uint32_t row0 = (row_tile - member.first_tile) * W::kRows;  // in the member's own rows
    const uint32_t first_vector_tile = vector_group * kTiles + wave_m * MT;
    const bool working = first_vector_tile < vector_tiles;  // else every vector of this wave is padding

    // ---- copies ----
    const uint32_t lds0 = lds_address(lds);
    // activations: wave w copies plane w & 1 of tile w / 2 (of the last tile where there are no more)
    const uint32_t copied_tile = min(vector_group * kTiles + (wave >> 1), vector_tiles - 1u);
    const uint8_t* const blobs = tiles + (static_cast<uint64_t>(first_stage) * vector_tiles + copied_tile) * kBlob + (wave & 1u) * 16384u;
    const uint64_t blob_stride = static_cast<uint64_t>(vector_tiles) * kBlob;
    const auto copy_activations = [&](uint32_t stage, int b) {
        const uint8_t* from = blobs + stage * blob_stride + b * 2048u;
        const uint32_t to = lds0 + (b % kSlots) * kSlotBytes + wave * 2048u;
#pragma unroll
        for (uint32_t i = 0; i < kActivationCopies; i++) copy_to_lds(from + i * 1024u, lane * 16u, to + i * 1024u);
    };
    // weights: the stage's bytes of the rows, row after row, as HalfStage lays them out
    uint32_t weight_from[W::kRounds];
#pragma unroll
    for (int i = 0; i < W::kRounds; i++) {
        const uint32_t at = (i * kWaves + wave) % W::kWeightJobs * 1024u + lane * 16u;
        weight_from[i] = min(at / kRowBytes, rows - 1u - row0) * row_bytes + HalfStage<CODEC>::source_of(at % kRowBytes);
    }
    const uint8_t* const weights = member.weight + static_cast<uint64_t>(row0) * row_bytes + static_cast<uint64_t>(first_stage) * kStageBytes;
    const auto copy_weights = [&](uint32_t stage, int round) {
        copy_to_lds(weights + static_cast<uint64_t>(stage) * kStageBytes, weight_from[round],
                    lds0 + W::kWeightsAt + (stage & 1u) * W::kWeightBytes + (round * kWaves + wave) % W::kWeightJobs * 1024u);
    };
    // xsum[g][m], 1 KiB per tile (waves 0 to 3), and the units of all tiles (the others, each the same bytes: every wave
    // asks for one copy, so that all of them count alike)
    const auto copy_tables = [&](uint32_t stage) {
        const uint8_t* base = tiles + static_cast<uint64_t>(first_stage + stage) * blob_stride + static_cast<uint64_t>(vector_group) * kTiles * kBlob;
        const uint32_t tiles_left = vector_tiles - 1u - vector_group * kTiles;
        if (W::kMinima && wave < kTiles)
            copy_to_lds(base + min(wave, tiles_left) * kBlob + ::et::kSumsAt, lane * 16u, lds0 + W::kSumsAt + wave * 1024u);
        else
            copy_to_lds(base + kUnitAt, min((lane >> 3) & 3u, tiles_left) * kBlob + (lane & 7u) * 16u, lds0 + W::kUnitsAt);
    };

    // Between the barriers of sub-blocks kCutAt and kCutAt + 1 every thread reads and cuts the sums of two sub-blocks of one
    // vector, in units of the vector (pieces of numbers around 10^-35 would not be normal); behind the second one the
    // pieces take the sums' place; they are read in the last sub-block.
    uint32_t piece[3];
    const uint32_t cut_vector = threadIdx.x & 31u, cut_group = ((threadIdx.x >> 5) & 3u) * 2u;
    const auto cut_sums = [&] {
        const float* sums = reinterpret_cast<const float*>(lds + W::kSumsAt + (wave >> 1) * 1024u) + cut_group * 32u + cut_vector;
        const float unit = *reinterpret_cast<const float*>(lds + W::kUnitsAt + (wave >> 1) * 128u + cut_vector * 4u);
        const auto in_units = [&](float sum) { return unit != 0.f ? sum / unit : 0.f; };
        const Pieces a = cut(in_units(sums[0])), b = cut(in_units(sums[32]));
        piece[0] = __builtin_amdgcn_perm(b.high, a.high, 0x07060302u);
        piece[1] = __builtin_amdgcn_perm(b.mid, a.mid, 0x07060302u);
        piece[2] = __builtin_amdgcn_perm(b.low, a.low, 0x07060302u);
    };
    const auto put_pieces = [&] {
#pragma unroll
        for (int i = 0; i < 3; i++)
            *reinterpret_cast<uint32_t*>(lds + W::kSumsAt + (wave >> 1) * 1536u + i * 512u + cut_vector * 16u + cut_group * 2u) = piece[i];
    };

    v16f acc[MT], zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.f;
#pragma unroll
    for (int m = 0; m < MT; m++) acc[m] = zero;

    const auto row_of = [&](uint32_t stage) {  // this lane's row in LDS
        return lds + W::kWeightsAt + (stage & 1u) * W::kWeightBytes + (wave_n * 32u + in_half) * kRowBytes;
    };
    const uint8_t* const activations = lds + wave_m * MT * 4096u + half * 1024u + in_half * 16u;
    const auto operand = [&](int b, int m, int turn) {  // turn: low and high plane of one sixteen-column chunk, then of the other
        return *reinterpret_cast<const v8h*>(activations + (b % kSlots) * kSlotBytes + m * 4096u + (turn & 1) * 2048u + (turn >> 1) * 512u);
    };

    // Sub-block b of a stage begins. Landed behind its barrier: the activations of sub-block b + 1, and whatever was
    // asked for before them two sub-blocks ago. Free: the slot of sub-block b - 1, in a stage's first sub-block also the
    // other stage's weights and the tables of the stage before.
    const auto begin = [&](uint32_t stage, auto is_last, int b) {
        constexpr bool last = decltype(is_last)::value;
        if (!last) wait_copies_in_flight(kActivationCopies + (b > 0 ? W::ahead(b - 1, false) : 0));
        else wait_copies_in_flight(b < 6 ? kActivationCopies + (b > 0 ? W::ahead(b - 1, true) : 0) : 0);
        if (W::kMinima && b == kCutAt + 1) asm volatile("" : "+v"(piece[0]), "+v"(piece[1]), "+v"(piece[2]));  // read before others write
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (b == 0) copy_tables(stage);
        if (!last && b < W::kRounds) copy_weights(stage + 1u, b);
        if (b + kSlots - 1 < kStageBlocks) copy_activations(stage, b + kSlots - 1);
        else if (!last) copy_activations(stage + 1u, b + kSlots - 1 - kStageBlocks);
        if (W::kMinima && b == kCutAt) cut_sums();
        if (W::kMinima && b == kCutAt + 1) put_pieces();
    };
#pragma unroll
    for (int i = 0; i < W::kRounds; i++) copy_weights(0, i);
#pragma unroll
    for (int b = 0; b < kSlots - 1; b++) copy_activations(0, b);
    wait_copies_in_flight(kActivationCopies);  // all but the last sub-block's
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (!working) {
        const auto pass = [&](uint32_t stage, auto is_last) {
#pragma unroll
            for (int b = 0; b < kStageBlocks; b++) {
                begin(stage, is_last, b);
                // The pieces are in LDS before this wave's next barrier. (Waves with vectors wait for operands that they read
                // behind these writes, and LDS answers in order.)
                if (W::kMinima && b == kCutAt + 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        };
        for (uint32_t stage = 0; stage + 1u < stages; stage++) pass(stage, std::false_type{});
        pass(stages - 1u, std::true_type{});
        return;
    }
    Shared shared = fetch_shared<CODEC>(row_of(0), half);
    v8h w[2][P], x[2][4];  // x: the operands of MT tiles in one turn, in the last sub-block of one tile in four turns
    operands<CODEC>(fetch<CODEC>(row_of(0), 0, half), shared, 0, w);
    const auto load_turn = [&](int b, int turn, v8h to[4]) {
#pragma unroll
        for (int m = 0; m < MT; m++) to[m] = operand(b, m, turn);
    };
    const auto load_tile = [&](int b, int m, v8h to[4]) {
#pragma unroll
        for (int turn = 0; turn < 4; turn++) to[turn] = operand(b, m, turn);
    };
    load_turn(0, 0, x[0]);

    // One stage. A wave issues in order and a matrix instruction keeps its pipe busy for eight issue cycles, so what keeps the
    // pipe fed is that no run of vector instructions stands alone: the sums of one tile of vectors are finished before the
    // next tile's begin, the packed bytes of the next sub-block become operands between the matrix instructions of
    // this one, and a tile's sums of the stage are folded into acc between the last matrix instructions of the next tile.
    // The last stage is compiled apart: a branch between sub-blocks would let the compiler move that arithmetic behind it.
    const auto contract = [&](uint32_t stage, auto is_last) {
        constexpr bool last = decltype(is_last)::value;
        v16f p[P][MT];
        Shared shared_next;
        // what the fold needs of this lane's row
        float d = 0.f, dmin = 0.f;
        v8s minima[2];
#pragma unroll
        for (int b = 0; b < kStageBlocks; b++) {
            begin(stage, is_last, b);
            const bool more = !last || b + 1 < kStageBlocks;
            const int bn = (b + 1) % kStageBlocks;
            const uint8_t* const row_n = row_of(b + 1 < kStageBlocks ? stage : stage + 1u);
            Raw raw;
            v8h next[2][P];
            if (b + 1 == kStageBlocks) {
                const uint8_t* row = row_of(stage);
                uint32_t dd = 0;
                if constexpr (W::kMinima) dd = shared.header.x;
                else if constexpr (CODEC == kQ3_K) dd = *reinterpret_cast<const uint16_t*>(row + HalfStage<CODEC>::in_tail(108u));
                else if constexpr (CODEC == kQ6_K) dd = *reinterpret_cast<const uint16_t*>(row + HalfStage<CODEC>::in_tail(208u));
                else dd = *reinterpret_cast<const uint32_t*>(row + HalfStage<CODEC>::in_tail(80u));
                d = kPlaneRatio * half_bits_to_float(dd & 0xffffu), dmin = half_bits_to_float(dd >> 16);
                if constexpr (W::kMinima) minimum_operands(shared.header, half, minima);
            }
            // acc += unit[m] * (p * d[n] - (sum_g xsum[m, g] / unit[m] * m_g[n]) * dmin[n]); vectors of a lane: 8 (r / 4) + 4 half + r % 4
            v16f below;
            const auto units_of = [&](int m, int j) {
                return *reinterpret_cast<const float4*>(lds + W::kUnitsAt + (wave_m * MT + m) * 128u + (8u * j + 4u * half) * 4u);
            };
            const auto fold = [&](int m, int j, const float4& units) {
                const float unit[4] = {units.x, units.y, units.z, units.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int r = 4 * j + i;
                    if constexpr (W::kMinima) acc[m][r] = fmaf(fmaf(p[0][m][r], d, -dmin * below[r]), unit[i], acc[m][r]);
                    else if constexpr (CODEC == kQ6_K) acc[m][r] = fmaf(fmaf(16.0f, p[P - 1][m][r], p[0][m][r]), unit[i] * d, acc[m][r]);
                    else if constexpr (CODEC == kQ2_K)
                        acc[m][r] = fmaf(fmaf(p[0][m][r], d, -p[P - 1][m][r] * (kPlaneRatio * dmin)), unit[i], acc[m][r]);
                    else acc[m][r] = fmaf(p[0][m][r], unit[i] * d, acc[m][r]);
                }
            };
            float4 units = {};
            if (b + 1 < kStageBlocks) {
                // four turns; x[0] holds the first one's operands
#pragma unroll
                for (int turn = 0; turn < 4; turn++) {
                    if (turn < 3) load_turn(b, turn + 1, x[(turn + 1) & 1]);
                    else if (b + 2 < kStageBlocks) load_turn(bn, 0, x[0]);
                    else load_tile(bn, 0, x[0]);
                    if (turn == 0) raw = fetch<CODEC>(row_n, bn, half);
                    if (turn == 1) operands<CODEC>(raw, shared, bn, next);
#pragma unroll
                    for (int m = 0; m < MT; m++)
#pragma unroll
                        for (int k = 0; k < P; k++)
                            p[k][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[turn & 1][m], w[turn >> 1][k], b + turn == 0 ? zero : p[k][m], 0, 0, 0);
                    // reads first, then the matrix instructions, from the second turn on with the next operands' arithmetic between them
                    __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
                    if (turn == 0) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 4 * P * MT / 4, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    } else {
#pragma unroll
                        for (int i = 0; i < P * MT; i++) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, P == 1 ? 3 : 5, 0);
                        }
                    }
                }
            } else {
                // tile after tile; x[0] holds the first one's operands
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    if (m + 1 < MT) load_tile(b, m + 1, x[(m + 1) & 1]);
                    else if (more) load_turn(bn, 0, x[(m + 1) & 1]);
                    if (m == 0 && more) {
                        shared_next = fetch_shared<CODEC>(row_n, half);
                        raw = fetch<CODEC>(row_n, bn, half);
                    }
                    if (m == MT / 2 && more) operands<CODEC>(raw, shared_next, bn, next);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float4 units_next = units;
                        if (m + (i + 1) / 4 > 0) units_next = units_of(m - 1 + (i + 1) / 4, (i + 1) % 4);
#pragma unroll
                        for (int k = 0; k < P; k++)
                            p[k][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[m & 1][i], w[i >> 1][k], p[k][m], 0, 0, 0);
                        if (m > 0) fold(m - 1, i, units);
                        units = units_next;
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (W::kMinima) {
                        const uint8_t* pieces = lds + W::kSumsAt + (wave_m * MT + m) * 1536u + in_half * 16u;
                        below = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(*reinterpret_cast<const v8s*>(pieces + half * 512u)),
                                                                        as_bf16(minima[0]), zero, 0, 0, 0);
                        below = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(*reinterpret_cast<const v8s*>(pieces + 1024u)),
                                                                        as_bf16(minima[1]), below, 0, 0, 0);
                    }
                }
            }
            if (b + 1 == kStageBlocks) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 now = units;
                    if (j < 3) units = units_of(MT - 1, j + 1);
                    fold(MT - 1, j, now);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (more) {
#pragma unroll
                for (int chunk = 0; chunk < 2; chunk++)
#pragma unroll
                    for (int k = 0; k < P; k++) w[chunk][k] = next[chunk][k];
            }
        }
        if (!last) shared = shared_next;
    };
    for (uint32_t stage = 0; stage + 1u < stages; stage++) contract(stage, std::false_type{});
    contract(stages - 1u, std::true_type{});

    // ---- add bias, store: y, or this K share's sums ----
    const uint64_t launch_rows = static_cast<uint64_t>(group.row_tiles) * W::kRows;
    const uint32_t in_tile = wave_n * 32u + in_half, n_out = row0 + in_tile;
    if (n_out >= rows) return;
    const bool direct = k_splits == 1;
    const float bias = direct && member.bias != nullptr ? member.bias[n_out] : 0.f;
    const uint64_t stride = direct ? rows : launch_rows;  // of a vector; row_tile * kRows + in_tile is among the rows of all members
    float* const out = direct ? member.y + n_out : partials + k_share * (vectors * launch_rows) + row_tile * W::kRows + in_tile;
    const float* const residual = direct && member.residual != nullptr ? member.residual + n_out : nullptr;
    const auto store = [&](auto all_vectors) {
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t v = (first_vector_tile + m) * 32u + 8u * (r >> 2) + 4u * half + (r & 3u);
                if (!decltype(all_vectors)::value && v >= vectors) continue;
                // residual may be y itself: every output is read, then written, by this lane only
                const float value = acc[m][r] + bias;
                out[v * stride] = residual != nullptr ? value + residual[v * stride] : value;
            }
        }
    };
    if ((first_vector_tile + MT) * 32u <= vectors && residual == nullptr) store(std::true_type{});
    else store(std::false_type{});
}

template <int CODEC>
hipError_t launch(const Group& group, const uint8_t* tiles, uint32_t columns, uint32_t vectors, uint32_t k_splits,
                  float* partials, hipStream_t stream) {
    using W = Wide<CODEC>;
    static_assert(W::kRows == gemm_h16_wide_rows(CODEC), "the planner's tile height");
    const auto kernel = gemm_h16_wide_kernel<CODEC>;
    // More than 64 KiB of dynamic LDS has to be allowed once per kernel and device.
    static std::atomic<bool> allowed[64] = {};  // callers may enqueue from several threads; setting twice is harmless
    int device = 0;
    if (hipError_t status = hipGetDevice(&device)) return status;
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    if (!allowed[device].load(std::memory_order_acquire)) {
        if (hipError_t status = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, W::kLdsBytes))
            return status;
        allowed[device].store(true, std::memory_order_release);
    }
    const uint32_t vector_tiles = (vectors + 31u) / 32u, vector_groups = (vector_tiles + kTiles - 1u) / kTiles;
    const uint64_t grid = (static_cast<uint64_t>(group.row_tiles) * k_splits + 7u) / 8u * 8u * vector_groups;
    if (grid > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(grid)), dim3(64 * kWaves), W::kLdsBytes, stream, group, tiles,
                       vector_tiles, columns, vectors, k_splits, partials);
    return hipGetLastError();
}
}  // namespace

hipError_t gemm_h16_wide(int32_t codec, const Group& group, const uint8_t* tiles, uint32_t columns, uint32_t vectors,
                         uint32_t k_splits, float* partials, hipStream_t stream) {
    switch (codec) {
        case kQ2_K: return launch<kQ2_K>(group, tiles, columns, vectors, k_splits, partials, stream);
        case kQ3_K: return launch<kQ3_K>(group, tiles, columns, vectors, k_splits, partials, stream);
        case kQ4_K: return launch<kQ4_K>(group, tiles, columns, vectors, k_splits, partials, stream);
        case kQ5_K: return launch<kQ5_K>(group, tiles, columns, vectors, k_splits, partials, stream);
        case kQ6_K: return launch<kQ6_K>(group, tiles, columns, vectors, k_splits, partials, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace et
