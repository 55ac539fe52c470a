// Dequant-GEMV for a few activation vectors (2..8) on the int8 matrix cores of gfx950 (Q4_K, Q5_K, Q4_0, Q8_0):
//     y[v, r] = sum_k x[v, k] * decode(W[r])[k] (+ bias[r])
//
// Same contraction as linear_into (crates/runtime-cpu/src/quantized.rs:419-499) with decode_q4_k
// (:180-199) and decode_q5_k (:203-234) in factored form; Q4_0 and Q8_0 follow the public ggml block layouts. The reference's own GPU
// backend keeps 2..8 vectors in its GEMV family (crates/runtime-metal/src/quantized.rs:1204-1220).
// f32-accurate (23-bit fixed-point activations per 256 columns, exact integer dots).
//
// The kernel is HBM-bound and streams W exactly once, whatever the number of vectors. What a few
// vectors cost on v_dot4 (gemv_limb.hip: 48 dots per vector, row and lane) is here one matrix
// instruction per 32-column block and sixteen rows: v_mfma_i32_16x16x32_i8 with the weights' quants
// as its B operand (sixteen rows of W) and, as its A operand, the three signed-byte limbs of four
// activation vectors in rows 4v + limb (row 4v + 3 is zero, or a limb of a fifth vector). A lane of the result then holds,
// for its weight row and its vector, the three limb dots of the block side by side.
//
// Work split. A workgroup owns a contiguous range of rows (one per compute unit when the matrix
// fits). LOADER waves copy that range into LDS as it lies in memory, with 1 KiB global-to-LDS copies
// taken in turn, a few in flight per wave, and publish how many have landed. Eight CONSUMER waves
// each own one eighth of the columns (two 256-column units at 4096 columns): a consumer quantises its
// own slice of the activation vectors once, keeps the A operands of all its blocks in registers for
// its whole life and walks the rows in groups of sixteen as they land; the eight partial sums of a
// group meet in LDS and the consumer that arrives last adds them in wave order (the same bits on
// every run) and stores y.
//
// LDS image of the weights: rows `pitch` bytes apart, pitch = row bytes + the padding that makes it
// 16 (mod 256), so that the sixteen rows a matrix instruction reads at one column offset lie in
// sixteen different groups of four banks. A copy instruction writes 1 KiB of the image; the lanes
// whose 16 bytes are padding are switched off.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>

#include "et_codecs.h"
#include "gemv_common.h"
#include "kernels.h"
#include "lds_handover.h"

namespace et {
namespace {

constexpr int kConsumers = 8;
constexpr uint32_t kLdsBytes = 160u * 1024u;
constexpr uint32_t kGroupRows = 16u;    // rows of W per matrix instruction
constexpr uint32_t kNarrowColumns = 4096u;  // wider rows: gemv_mma_wide_kernel
// Activations as fixed point: X = rint(x * kLimbRange / max|x|), |X| < 2^22. Adding kLimbMagic to the
// scaled value makes the float's mantissa the integer X + 0x408080 (the sum lies in [2^23, 2^24), where
// floats are the integers): one fused multiply-add quantises, rounds to nearest even and offsets.
constexpr float kLimbRange = 4161000.0f;                // X + 0x8080 stays below 2^22 with room for the reciprocal's ulp
constexpr float kLimbMagic = 12582912.0f + 32896.0f;    // 1.5 * 2^23 + 0x8080

constexpr uint32_t kMostGroups = 4u;    // groups of a range: its rows' partial sums wait in LDS for the end

// Per consumer wave: [limb planes of one vector, 544 bytes apart][sums and unit per vector and 256 columns]. Once the A operands are in registers the first part holds the
// wave's partial sums: [group][vector group][lane].
constexpr uint32_t kSumsFloats = 12u;  // of one (vector, unit): eight sums, one or four units of limb 0, whole float4s
constexpr uint32_t kLimbPitch = 544u;  // 512 bytes of a limb plane + 32: the three planes start in different banks
constexpr uint32_t kSumsAt = 2048u, kWaveScratch = 2048u + 8u * 2u * kSumsFloats * 4u;
static_assert(3u * kLimbPitch <= kSumsAt && kMostGroups * 2u * 256u <= kSumsAt, "planes and partial sums share the first part");
struct Control {
    uint32_t landed[8];  // copies of loader w that have landed
    uint32_t summed;     // consumers that have left the partial sums of all their groups
    uint32_t pad[7];
};
static_assert(sizeof(Control) == 64, "sixteen words, zeroed by sixteen lanes");
constexpr uint32_t kControlAt = kLdsBytes - 64u;
constexpr uint32_t kScratchAt = kControlAt - kConsumers * kWaveScratch;  // the image ends below this

__host__ __device__ constexpr uint32_t image_pitch(uint32_t row_bytes) {
    return row_bytes + ((16u - (row_bytes & 255u)) & 255u);
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ long pack(uint32_t low, uint32_t high) {
    return static_cast<long>((static_cast<uint64_t>(high) << 32) | low);
}

// 4x3 byte transpose: limb k of four 23-bit values X + 0x408080 (the low three bytes of the words) into
// one dword each. With X = 65536 l2 + 256 l1 + l0 in balanced digits (l0, l1 in [-128, 127], l2 in
// [-64, 63]) the bytes are l0 + 128, l1 + 128 and l2 + 64: flipping the top bit gives the signed limb,
// for the third after another 64 (no byte carries: it is below 128).
__device__ __forceinline__ void split_quad(int x0, int x1, int x2, int x3, uint32_t (&limb)[3]) {
    const uint32_t a = __builtin_amdgcn_perm(x1, x0, 0x05010400u);  // x0.b0 x1.b0 x0.b1 x1.b1
    const uint32_t b = __builtin_amdgcn_perm(x3, x2, 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(x1, x0, 0x0c0c0602u);  // x0.b2 x1.b2 0 0
    const uint32_t d = __builtin_amdgcn_perm(x3, x2, 0x0c0c0602u);
    limb[0] = __builtin_amdgcn_perm(b, a, 0x05040100u) ^ 0x80808080u;
    limb[1] = __builtin_amdgcn_perm(b, a, 0x07060302u) ^ 0x80808080u;
    limb[2] = (__builtin_amdgcn_perm(d, c, 0x05040100u) + 0x40404040u) ^ 0x80808080u;
}

// sum += unit * (the value of three limb sums), which start anew.
__device__ __forceinline__ void scaled_limbs(int (&acc)[3], float unit, float& sum) {
    float f = static_cast<float>(acc[0]);
    f = fmaf(256.0f, static_cast<float>(acc[1]), f);
    f = fmaf(65536.0f, static_cast<float>(acc[2]), f);
    sum = fmaf(unit, f, sum);
    acc[0] = acc[1] = acc[2] = 0;
}

// A fifth vector (FIFTH): its three limbs are the rows 4v + 3 that four vectors leave empty, limb i in the fourth result of
// lane group i (row 15 stays zero). Once per unit the groups' parts are put together, in every lane: limb i's `pos` is worth
// 256^i, `neg` is the group's share of the minima. (Kept apart until the end of the row, positive and negative sums cost
// two instructions less and a sixth more error where activations do not cancel.)
__device__ __forceinline__ void join_groups(uint32_t q, float& pos, float& neg) {
    pos = q == 3u ? 0.f : pos * __uint_as_float((127u + 8u * q) << 23);
    // the two small limbs first: one rounding of the whole sum's size, as in scaled_limbs
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(pos), __float_as_uint(neg), false, false);
    const uint32_t two = __float_as_uint(__uint_as_float(rows[0]) + __uint_as_float(rows[1]));  // pos in even groups, neg in odd
    const auto halves = __builtin_amdgcn_permlane32_swap(two, two, false, false);
    const uint32_t four = __float_as_uint(__uint_as_float(halves[0]) + __uint_as_float(halves[1]));
    const auto both = __builtin_amdgcn_permlane16_swap(four, four, false, false);
    pos = __uint_as_float(both[0]);
    neg = __uint_as_float(both[1]);
}

// ---------------------------------------------------------------------------
// Codec traits: one 256-column unit (kUnitBytes) of sixteen rows against the A operands.
//   rp     the unit in the lane's row of the LDS image
//   q      the lane's K index: which 8 of a block's 32 columns its operand registers hold
//   a      A operands of the wave's sixteen 32-column blocks, per group of four vectors
//   sums   f32 sums of the lane's vector over the unit's eight blocks, then the value of one unit of limb 0:
//          SCALES = 1 for all of the unit's columns, SCALES = 4 for every 64 of them
//          (next vector group: + sums_step floats)
//   fifth_sums  the same of a fifth vector, whose part is added to total[VG]
// ---------------------------------------------------------------------------
struct Q4KMma {
    static constexpr uint32_t kUnitBytes = 144u;  // one super-block
    static constexpr bool kTakesFifth = true;
    static __device__ __forceinline__ uint32_t chunk(uint32_t q) { return q; }
    template <int VG, int UNIT, int SCALES, bool FIFTH, int BLOCKS>
    static __device__ __forceinline__ void contract(const uint8_t* rp, uint32_t q, const long (&a)[VG][BLOCKS], const float* sums,
                                                    uint32_t sums_step, const float* fifth_sums, float (&total)[VG + FIFTH]) {
        const uint4 h = *reinterpret_cast<const uint4*>(rp);
        const float d = half_bits_to_float(h.x & 0xffffu), dmin = half_bits_to_float(h.x >> 16);
        // (scale, min) of the eight sub-blocks, a byte each: crates/runtime-cpu/src/quantized.rs:77-86
        const uint32_t sc[2] = {h.y & 0x3f3f3f3fu, (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u)};
        uint32_t mn[2] = {h.z & 0x3f3f3f3fu, ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u)};
        // keeps the minima packed, a byte-to-float conversion each, instead of a mask per byte
        asm volatile("" : "+v"(mn[0]), "+v"(mn[1]));
        int acc[VG][3], fifth_acc = 0;
        float pos[VG], fifth_pos = 0.f;
#pragma unroll
        for (int g = 0; g < VG; g++) acc[g][0] = acc[g][1] = acc[g][2] = 0, pos[g] = 0.f;
        const v4i zero = {0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < 4; p++) {
            // bytes 8q..8q+7 of the pair: low nibbles = columns 8q.. of sub-block 2p, high = of 2p + 1
            const uint2 w = *reinterpret_cast<const uint2*>(rp + 16 + 32 * p + 8 * q);
            const long lo = pack(w.x & 0x0f0f0f0fu, w.y & 0x0f0f0f0fu);
            const long hi = pack((w.x >> 4) & 0x0f0f0f0fu, (w.y >> 4) & 0x0f0f0f0fu);
            const int s_lo = static_cast<int>((sc[p >> 1] >> (16 * (p & 1))) & 0xffu);
            const int s_hi = static_cast<int>((sc[p >> 1] >> (16 * (p & 1) + 8)) & 0xffu);
#pragma unroll
            for (int g = 0; g < VG; g++) {
                const v4i c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * p], lo, zero, 0, 0, 0);
                const v4i c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * p + 1], hi, zero, 0, 0, 0);
                // block dots are below 2^17, scales below 2^6: 24-bit multiplies, exact int32 sums
#pragma unroll
                for (int k = 0; k < 3; k++) acc[g][k] += __mul24(c0[k], s_lo) + __mul24(c1[k], s_hi);
                if constexpr (SCALES == 4) scaled_limbs(acc[g], sums[sums_step * g + 8 + p], pos[g]);
                if constexpr (FIFTH) {
                    fifth_acc += __mul24(c0[3], s_lo) + __mul24(c1[3], s_hi);
                    if constexpr (SCALES == 4) fifth_pos = fmaf(fifth_sums[8 + p], static_cast<float>(fifth_acc), fifth_pos), fifth_acc = 0;
                }
            }
        }
        // (the compiler turns these into v_cvt_f32_ubyte0..3)
        const float m0 = static_cast<float>(mn[0] & 0xffu), m1 = static_cast<float>((mn[0] >> 8) & 0xffu);
        const float m2 = static_cast<float>((mn[0] >> 16) & 0xffu), m3 = static_cast<float>(mn[0] >> 24);
        const float m4 = static_cast<float>(mn[1] & 0xffu), m5 = static_cast<float>((mn[1] >> 8) & 0xffu);
        const float m6 = static_cast<float>((mn[1] >> 16) & 0xffu), m7 = static_cast<float>(mn[1] >> 24);
#pragma unroll
        for (int g = 0; g < VG; g++) {
            const float4 s0 = *reinterpret_cast<const float4*>(sums + sums_step * g);
            const float4 s1 = *reinterpret_cast<const float4*>(sums + sums_step * g + 4);
            float neg = m0 * s0.x;
            neg = fmaf(m1, s0.y, neg);
            neg = fmaf(m2, s0.z, neg);
            neg = fmaf(m3, s0.w, neg);
            neg = fmaf(m4, s1.x, neg);
            neg = fmaf(m5, s1.y, neg);
            neg = fmaf(m6, s1.z, neg);
            neg = fmaf(m7, s1.w, neg);
            if constexpr (SCALES == 1) scaled_limbs(acc[g], sums[sums_step * g + 8], pos[g]);
            total[g] += d * pos[g] - dmin * neg;
        }
        // The minima of sub-blocks 2q and 2q + 1 are this lane's part. (Written out here and in Q5KMma: as a function of both, Q4_K
        // 4096 x 14336 takes 16.5 us for 15.4.)
        if constexpr (FIFTH) {
            const uint32_t mine = (q & 2u ? mn[1] : mn[0]) >> (16 * (q & 1u));
            const float2 s = *reinterpret_cast<const float2*>(fifth_sums + 2 * q);
            float neg = fmaf(static_cast<float>((mine >> 8) & 0xffu), s.y, static_cast<float>(mine & 0xffu) * s.x);
            if constexpr (SCALES == 1) fifth_pos = static_cast<float>(fifth_acc);
            join_groups(q, fifth_pos, neg);
            if constexpr (SCALES == 1) fifth_pos *= fifth_sums[8];
            total[VG] += d * fifth_pos - dmin * neg;
        }
    }
};

// Q4_0: a unit is four pairs of 18-byte blocks, 36 bytes = 9 dwords each. Block: half-float d, then
// sixteen bytes whose low nibbles are columns 0..15 and whose high nibbles are columns 16..31. The
// lanes with K index q take bytes 8 * (q >> 1) .. + 7, low (q even) or high nibbles: columns
// 16 * (q & 1) + 8 * (q >> 1) .. + 7. value = d * (nibble - 8): the - 8 meets the f32 sums of the
// activations once per block.
struct Q40Mma {
    static constexpr uint32_t kUnitBytes = 144u;  // eight blocks of 18 bytes
    static constexpr bool kTakesFifth = false;
    static __device__ __forceinline__ uint32_t chunk(uint32_t q) { return ((q & 1u) << 1) | (q >> 1); }
    template <int VG, int UNIT, int SCALES, bool FIFTH, int BLOCKS>
    static __device__ __forceinline__ void contract(const uint8_t* rp, uint32_t q, const long (&a)[VG][BLOCKS], const float* sums,
                                                    uint32_t sums_step, const float* fifth_sums, float (&total)[VG + FIFTH]) {
        const uint32_t half = q >> 1, shift = (q & 1u) * 4u;
        static_assert(!FIFTH, "scales by the block: see launch_vectors");
        float pos[VG], corr[VG], s[VG][8];
#pragma unroll
        for (int g = 0; g < VG; g++) {
            pos[g] = corr[g] = 0.f;
            const float4 s0 = *reinterpret_cast<const float4*>(sums + sums_step * g);
            const float4 s1 = *reinterpret_cast<const float4*>(sums + sums_step * g + 4);
            s[g][0] = s0.x, s[g][1] = s0.y, s[g][2] = s0.z, s[g][3] = s0.w;
            s[g][4] = s1.x, s[g][5] = s1.y, s[g][6] = s1.z, s[g][7] = s1.w;
        }
        const v4i zero = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint32_t* pair = reinterpret_cast<const uint32_t*>(rp + 36 * c);
            const uint32_t* mine = pair + 2 * half;
            // even block: quants at bytes 2..17 of the pair (2 bytes off dword alignment); odd: 20..35
            const uint32_t e0 = mine[0], e1 = mine[1], e2 = mine[2], o0 = mine[5], o1 = mine[6];
            const uint32_t qa0 = __builtin_amdgcn_alignbit(e1, e0, 16), qa1 = __builtin_amdgcn_alignbit(e2, e1, 16);
            const long even = pack((qa0 >> shift) & 0x0f0f0f0fu, (qa1 >> shift) & 0x0f0f0f0fu);
            const long odd = pack((o0 >> shift) & 0x0f0f0f0fu, (o1 >> shift) & 0x0f0f0f0fu);
            const float da = half_bits_to_float(pair[0] & 0xffffu), db = half_bits_to_float(pair[4] >> 16);
#pragma unroll
            for (int g = 0; g < VG; g++) {
                const v4i c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * c], even, zero, 0, 0, 0);
                const v4i c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * c + 1], odd, zero, 0, 0, 0);
                float f0 = static_cast<float>(c0[0]);
                f0 = fmaf(256.0f, static_cast<float>(c0[1]), f0);
                f0 = fmaf(65536.0f, static_cast<float>(c0[2]), f0);
                float f1 = static_cast<float>(c1[0]);
                f1 = fmaf(256.0f, static_cast<float>(c1[1]), f1);
                f1 = fmaf(65536.0f, static_cast<float>(c1[2]), f1);
                if constexpr (SCALES == 4) pos[g] = fmaf(sums[sums_step * g + 8 + c], fmaf(db, f1, da * f0), pos[g]);
                else pos[g] = fmaf(db, f1, fmaf(da, f0, pos[g]));
                corr[g] = fmaf(db, s[g][2 * c + 1], fmaf(da, s[g][2 * c], corr[g]));
            }
        }
#pragma unroll
        for (int g = 0; g < VG; g++) total[g] += (SCALES == 4 ? pos[g] : sums[sums_step * g + 8] * pos[g]) - 8.0f * corr[g];
    }
};

// Q5_K (decode_q5_k, crates/runtime-cpu/src/quantized.rs:203-234): Q4_K's layout with a fifth bit per
// value in qh[32] between the scales and the nibbles - bit g of qh[i] belongs to column i of sub-block g.
struct Q5KMma {
    static constexpr uint32_t kUnitBytes = 176u;
    static constexpr bool kTakesFifth = true;
    static __device__ __forceinline__ uint32_t chunk(uint32_t q) { return q; }
    template <int VG, int UNIT, int SCALES, bool FIFTH, int BLOCKS>
    static __device__ __forceinline__ void contract(const uint8_t* rp, uint32_t q, const long (&a)[VG][BLOCKS], const float* sums,
                                                    uint32_t sums_step, const float* fifth_sums, float (&total)[VG + FIFTH]) {
        const uint4 h = *reinterpret_cast<const uint4*>(rp);
        const float d = half_bits_to_float(h.x & 0xffffu), dmin = half_bits_to_float(h.x >> 16);
        const uint32_t sc[2] = {h.y & 0x3f3f3f3fu, (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u)};
        uint32_t mn[2] = {h.z & 0x3f3f3f3fu, ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u)};
        asm volatile("" : "+v"(mn[0]), "+v"(mn[1]));
        const uint2 fifth = *reinterpret_cast<const uint2*>(rp + 16 + 8 * q);  // columns 8q..8q+7, all sub-blocks
        int acc[VG][3], fifth_acc = 0;
        float pos[VG], fifth_pos = 0.f;
#pragma unroll
        for (int g = 0; g < VG; g++) acc[g][0] = acc[g][1] = acc[g][2] = 0, pos[g] = 0.f;
        const v4i zero = {0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const uint2 w = *reinterpret_cast<const uint2*>(rp + 48 + 32 * p + 8 * q);
            const uint32_t fx = fifth.x >> (2 * p), fy = fifth.y >> (2 * p);
            const long lo = pack((w.x & 0x0f0f0f0fu) | ((fx & 0x01010101u) << 4), (w.y & 0x0f0f0f0fu) | ((fy & 0x01010101u) << 4));
            const long hi = pack(((w.x >> 4) & 0x0f0f0f0fu) | ((fx & 0x02020202u) << 3),
                                 ((w.y >> 4) & 0x0f0f0f0fu) | ((fy & 0x02020202u) << 3));
            const int s_lo = static_cast<int>((sc[p >> 1] >> (16 * (p & 1))) & 0xffu);
            const int s_hi = static_cast<int>((sc[p >> 1] >> (16 * (p & 1) + 8)) & 0xffu);
#pragma unroll
            for (int g = 0; g < VG; g++) {
                const v4i c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * p], lo, zero, 0, 0, 0);
                const v4i c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * p + 1], hi, zero, 0, 0, 0);
                // block dots are below 2^18, scales below 2^6
#pragma unroll
                for (int k = 0; k < 3; k++) acc[g][k] += __mul24(c0[k], s_lo) + __mul24(c1[k], s_hi);
                if constexpr (SCALES == 4) scaled_limbs(acc[g], sums[sums_step * g + 8 + p], pos[g]);
                if constexpr (FIFTH) {
                    fifth_acc += __mul24(c0[3], s_lo) + __mul24(c1[3], s_hi);
                    if constexpr (SCALES == 4) fifth_pos = fmaf(fifth_sums[8 + p], static_cast<float>(fifth_acc), fifth_pos), fifth_acc = 0;
                }
            }
        }
        const float m0 = static_cast<float>(mn[0] & 0xffu), m1 = static_cast<float>((mn[0] >> 8) & 0xffu);
        const float m2 = static_cast<float>((mn[0] >> 16) & 0xffu), m3 = static_cast<float>(mn[0] >> 24);
        const float m4 = static_cast<float>(mn[1] & 0xffu), m5 = static_cast<float>((mn[1] >> 8) & 0xffu);
        const float m6 = static_cast<float>((mn[1] >> 16) & 0xffu), m7 = static_cast<float>(mn[1] >> 24);
#pragma unroll
        for (int g = 0; g < VG; g++) {
            const float4 s0 = *reinterpret_cast<const float4*>(sums + sums_step * g);
            const float4 s1 = *reinterpret_cast<const float4*>(sums + sums_step * g + 4);
            float neg = m0 * s0.x;
            neg = fmaf(m1, s0.y, neg);
            neg = fmaf(m2, s0.z, neg);
            neg = fmaf(m3, s0.w, neg);
            neg = fmaf(m4, s1.x, neg);
            neg = fmaf(m5, s1.y, neg);
            neg = fmaf(m6, s1.z, neg);
            neg = fmaf(m7, s1.w, neg);
            if constexpr (SCALES == 1) scaled_limbs(acc[g], sums[sums_step * g + 8], pos[g]);
            total[g] += d * pos[g] - dmin * neg;
        }
        if constexpr (FIFTH) {  // the minima of sub-blocks 2q and 2q + 1 are this lane's part
            const uint32_t mine = (q & 2u ? mn[1] : mn[0]) >> (16 * (q & 1u));
            const float2 s = *reinterpret_cast<const float2*>(fifth_sums + 2 * q);
            float neg = fmaf(static_cast<float>((mine >> 8) & 0xffu), s.y, static_cast<float>(mine & 0xffu) * s.x);
            if constexpr (SCALES == 1) fifth_pos = static_cast<float>(fifth_acc);
            join_groups(q, fifth_pos, neg);
            if constexpr (SCALES == 1) fifth_pos *= fifth_sums[8];
            total[VG] += d * fifth_pos - dmin * neg;
        }
    }
};

// Q8_0: a unit is four pairs of 34-byte blocks, 68 bytes = 17 dwords each. Block: half-float d, then
// 32 signed bytes. The lanes with K index q take columns 8q..8q+7.
struct Q80Mma {
    static constexpr uint32_t kUnitBytes = 272u;
    static constexpr bool kTakesFifth = false;
    static __device__ __forceinline__ uint32_t chunk(uint32_t q) { return q; }
    template <int VG, int UNIT, int SCALES, bool FIFTH, int BLOCKS>
    static __device__ __forceinline__ void contract(const uint8_t* rp, uint32_t q, const long (&a)[VG][BLOCKS], const float* sums,
                                                    uint32_t sums_step, const float* fifth_sums, float (&total)[VG + FIFTH]) {
        static_assert(!FIFTH, "scales by the block: see launch_vectors");
        float pos[VG];
#pragma unroll
        for (int g = 0; g < VG; g++) pos[g] = 0.f;
        const v4i zero = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint32_t* pair = reinterpret_cast<const uint32_t*>(rp + 68 * c);
            const uint32_t* mine = pair + 2 * q;
            // even block: quants at bytes 2..33 of the pair (2 bytes off dword alignment); odd: 36..67
            const uint32_t e0 = mine[0], e1 = mine[1], e2 = mine[2], o0 = mine[9], o1 = mine[10];
            const long even = pack(__builtin_amdgcn_alignbit(e1, e0, 16), __builtin_amdgcn_alignbit(e2, e1, 16));
            const long odd = pack(o0, o1);
            const float da = half_bits_to_float(pair[0] & 0xffffu), db = half_bits_to_float(pair[8] >> 16);
#pragma unroll
            for (int g = 0; g < VG; g++) {
                const v4i c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * c], even, zero, 0, 0, 0);
                const v4i c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g][UNIT * 8 + 2 * c + 1], odd, zero, 0, 0, 0);
                float f0 = static_cast<float>(c0[0]);
                f0 = fmaf(256.0f, static_cast<float>(c0[1]), f0);
                f0 = fmaf(65536.0f, static_cast<float>(c0[2]), f0);
                float f1 = static_cast<float>(c1[0]);
                f1 = fmaf(256.0f, static_cast<float>(c1[1]), f1);
                f1 = fmaf(65536.0f, static_cast<float>(c1[2]), f1);
                if constexpr (SCALES == 4) pos[g] = fmaf(sums[sums_step * g + 8 + c], fmaf(db, f1, da * f0), pos[g]);
                else pos[g] = fmaf(db, f1, fmaf(da, f0, pos[g]));
            }
        }
#pragma unroll
        for (int g = 0; g < VG; g++) total[g] += SCALES == 4 ? pos[g] : sums[sums_step * g + 8] * pos[g];
    }
};

template <class T, int VG, bool FIFTH, int LOADERS, int DEPTH>
__global__ __launch_bounds__(64 * (kConsumers + LOADERS)) void gemv_mma_kernel(
    const uint8_t* __restrict__ weight, const float* __restrict__ x, uint64_t x_row_stride,
    const float* __restrict__ bias, float* __restrict__ y, uint32_t rows, uint32_t columns, uint32_t rows_per_wg,
    uint32_t vectors, uint32_t spin_limit, uint32_t* timeouts) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    static_assert(DEPTH >= 1 && DEPTH <= 8 && LOADERS >= 1 && LOADERS <= 8, "wait_copies_in_flight counts to seven");
    static_assert(!FIFTH || VG == 1, "a fifth vector takes the rows of four");
    constexpr int VEC = 4 * VG + FIFTH, kSlots = VG + FIFTH;
    Control* control = reinterpret_cast<Control*>(lds + kControlAt);

    const uint32_t lane_id = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wg_row0 = blockIdx.x * rows_per_wg;
    if (wg_row0 >= rows) return;
    const uint32_t wg_rows = min(rows_per_wg, rows - wg_row0);
    const uint32_t row_units = columns >> 8;
    const uint32_t row_bytes = row_units * T::kUnitBytes;
    const uint32_t pitch = image_pitch(row_bytes);
    const uint32_t image_bytes = (wg_rows - 1u) * pitch + row_bytes;  // ends with the last row's last byte

    if (wave >= static_cast<uint32_t>(kConsumers)) {
        // ---- loaders ----------------------------------------------------------------------------
        const uint32_t loader = wave - kConsumers;
        const uint32_t copies = (image_bytes + 1023u) >> 10;
        const uint32_t mine = copies > loader ? (copies - loader + LOADERS - 1u) / LOADERS : 0u;
        // where this lane's 16 bytes of the wave's next copy lie in the image, and in W (from the range's first byte)
        uint32_t at = loader * 1024u + lane_id * 16u;
        uint32_t row = at / pitch, column = at - row * pitch;
        uint32_t from = row * row_bytes + column;
        constexpr uint32_t kStep = LOADERS * 1024u;  // between two copies of a wave
        const uint32_t step_rows = kStep / pitch, step_columns = kStep - step_rows * pitch;
        const uint32_t step_from = step_rows * row_bytes + step_columns;
        const uint32_t end = wg_rows * row_bytes;  // rows past the range start there
        const uint8_t* source = weight + static_cast<uint64_t>(wg_row0) * row_bytes;
        const uint32_t landed_address = lds_address(&control->landed[loader]);
        uint32_t next = loader;  // number of the wave's next copy
        const auto copy = [&]() {
            // never a copy without a lane: the image ends with bytes of W and padding is shorter than a copy
            if (column < row_bytes && from < end)
                // streamed once: non-temporal (aux bit 1), the caches keep nothing of it
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint4*>(source + from),
                                                 reinterpret_cast<uint4*>(lds + next * 1024u), 16, 0, 2);
            next += LOADERS;
            column += step_columns;
            from += step_from;
            if (column >= pitch) {  // into the next row: its padding is not in W
                column -= pitch;
                from += row_bytes - pitch;
            }
        };
        // The first copies wait for the barrier, i.e. until the consumers have issued their activation
        // loads: issued ahead of it they delay those loads, and with them everything else.
        // (measured: issued ahead of the barrier, 0.9 to 1.5 us per launch slower)
        __syncthreads();
        const uint32_t head = min(mine, static_cast<uint32_t>(DEPTH));
        for (uint32_t i = 0; i < head; i++) copy();
        uint32_t landed = 0;
        for (uint32_t i = head; i < mine; i++) {  // only with DEPTH copies in flight
            // the oldest copy in flight has landed: say so, then take its place in the queue
            __builtin_amdgcn_s_waitcnt(vmcnt_only(DEPTH - 1));
            lds_store_unseen(landed_address, ++landed);
            copy();
        }
        for (uint32_t left = head; left > 0u; left--) {
            wait_copies_in_flight(left - 1u);
            lds_store_unseen(landed_address, ++landed);
        }
        return;
    }

    // ---- consumers --------------------------------------------------------------------------------
    Patience patience{spin_limit, timeouts};
    const uint32_t first_unit = 2u * wave;  // the wave's columns: units first_unit, first_unit + 1
    const uint32_t my_units = row_units > first_unit ? min(2u, row_units - first_unit) : 0u;
    uint8_t* scratch = lds + kScratchAt + wave * kWaveScratch;
    float* sums = reinterpret_cast<float*>(scratch + kSumsAt);    // [vector][unit of the slice][kSumsFloats]

    // Activation loads first: nothing of the consumers' may queue behind a copy. Lane j holds columns
    // 8j .. 8j+7 of the slice: chunk j % 4 of block j / 4.
    float4 xv[VEC][2];
    {
        const uint32_t column = first_unit * 256u + lane_id * 8u;
#pragma unroll
        for (int v = 0; v < VEC; v++) {
            xv[v][0] = xv[v][1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (static_cast<uint32_t>(v) < vectors && column < columns) {
                const float4* p = reinterpret_cast<const float4*>(x + v * x_row_stride + column);
                xv[v][0] = p[0];
                xv[v][1] = p[1];
            }
        }
    }
    if (threadIdx.x < 16) reinterpret_cast<uint32_t*>(control)[threadIdx.x] = 0u;
    __syncthreads();  // the only barrier: the counters are zero before anybody counts

    // 23-bit fixed point per vector and 256-column unit, X = rint(x * kLimbRange / max|x|), in three
    // balanced signed-byte limbs; the limbs go through the wave's scratch into the lanes that hold
    // them as A operands: lane l, as row l % 16 = 4 * vector + limb, K index l / 16.
    long a[VG][16];
#pragma unroll
    for (int g = 0; g < VG; g++)
#pragma unroll
        for (int s = 0; s < 16; s++) a[g][s] = 0;
#pragma unroll
    for (int v = 0; v < VEC; v++) {
        if (static_cast<uint32_t>(v) >= vectors) break;
        const float4 f0 = xv[v][0], f1 = xv[v][1];
        float amax = fmaxf(fmaxf(fabsf(f0.x), fabsf(f0.y)), fabsf(f0.z));  // three-input maxima
        amax = fmaxf(fmaxf(amax, fabsf(f0.w)), fabsf(f1.x));
        amax = fmaxf(fmaxf(amax, fabsf(f1.y)), fabsf(f1.z));
        amax = fmaxf(amax, fabsf(f1.w));
        amax = fmaxf(amax, dpp<0xB1>(amax));   // quad_perm [1,0,3,2]
        amax = fmaxf(amax, dpp<0x4E>(amax));   // quad_perm [2,3,0,1]
        amax = fmaxf(amax, dpp<0x141>(amax));  // row_half_mirror
        amax = fmaxf(amax, dpp<0x140>(amax));  // row_mirror: sixteen lanes = 128 columns
        amax = fmaxf(amax, __shfl_xor(amax, 16));  // the unit's 256 columns
        float total = ((f0.x + f0.y) + (f0.z + f0.w)) + ((f1.x + f1.y) + (f1.z + f1.w));
        total += dpp<0xB1>(total);
        total += dpp<0x4E>(total);  // the block's 32 columns
        // 1 ulp of the reciprocal moves |X| by at most 1, far inside the headroom of the range.
        const bool nonzero = amax >= 1e-30f;
        const float inv = nonzero ? kLimbRange * __builtin_amdgcn_rcpf(amax) : 0.f;
        const float unit = nonzero ? amax * (1.0f / kLimbRange) : 0.f;
        uint32_t low[3], high[3];
        split_quad(__float_as_int(fmaf(f0.x, inv, kLimbMagic)), __float_as_int(fmaf(f0.y, inv, kLimbMagic)),
                   __float_as_int(fmaf(f0.z, inv, kLimbMagic)), __float_as_int(fmaf(f0.w, inv, kLimbMagic)), low);
        split_quad(__float_as_int(fmaf(f1.x, inv, kLimbMagic)), __float_as_int(fmaf(f1.y, inv, kLimbMagic)),
                   __float_as_int(fmaf(f1.z, inv, kLimbMagic)), __float_as_int(fmaf(f1.w, inv, kLimbMagic)), high);
        asm volatile("" ::: "memory");  // the reads of the vector before are done with the planes
#pragma unroll
        for (int k = 0; k < 3; k++)
            *reinterpret_cast<uint2*>(scratch + k * kLimbPitch + lane_id * 8u) = make_uint2(low[k], high[k]);
        float* of_unit = sums + (2u * v + (lane_id >> 5)) * kSumsFloats;
        if ((lane_id & 3u) == 0u) of_unit[(lane_id & 31u) >> 2] = total;
        if ((lane_id & 31u) == 0u) of_unit[8] = unit;
        asm volatile("" ::: "memory");  // LDS serves a wave in order: written above, read below
        // row 4 * vector + limb; of a fifth vector row 4 * limb + 3
        const uint32_t upper = (lane_id & 15u) >> 2, lower = lane_id & 3u;
        const bool is_fifth = FIFTH && v == 4;
        const uint32_t limb = is_fifth ? upper : lower;
        if (is_fifth ? lower == 3u && upper < 3u : upper == static_cast<uint32_t>(v & 3) && lower != 3u) {
            const uint8_t* plane = scratch + limb * kLimbPitch + T::chunk(lane_id >> 4) * 8u;
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const uint2 w = *reinterpret_cast<const uint2*>(plane + s * 32);
                a[is_fifth ? 0 : v >> 2][s] = pack(w.x, w.y);
            }
        }
    }
    asm volatile("" ::: "memory");

    const uint32_t n = lane_id & 15u, q = lane_id >> 4;
    const uint32_t groups = (wg_rows + kGroupRows - 1u) / kGroupRows;
    float* partial = reinterpret_cast<float*>(scratch);  // [group][vector group][lane]
    for (uint32_t group = 0; group < groups; group++) {
        const uint32_t last_row = min(group * kGroupRows + kGroupRows, wg_rows) - 1u;
        const bool landed = await_copies_in_turn<LOADERS>(control->landed, lane_id, (last_row * pitch + row_bytes + 1023u) >> 10, patience);
        float total[kSlots];
#pragma unroll
        for (int g = 0; g < kSlots; g++) total[g] = 0.f;
        if (landed && my_units != 0u) {
            // rows past the end of the range read its last row again and are not stored
            const uint8_t* rp = lds + min(group * kGroupRows + n, wg_rows - 1u) * pitch + first_unit * T::kUnitBytes;
            const float* of_vector = sums + 2u * q * kSumsFloats;
            constexpr uint32_t kStep = 4u * 2u * kSumsFloats;  // to the next vector group
            const float* of_fifth = sums + 8u * kSumsFloats;
            T::template contract<VG, 0, 1, FIFTH>(rp, q, a, of_vector, kStep, of_fifth, total);
            // in one block with the first: the second unit's LDS reads overtake the first's arithmetic
            if (my_units > 1u)
                T::template contract<VG, 1, 1, FIFTH>(rp + T::kUnitBytes, q, a, of_vector + kSumsFloats, kStep, of_fifth + kSumsFloats, total);
        }
#pragma unroll
        for (int g = 0; g < kSlots; g++) partial[(group * kSlots + g) * 64u + lane_id] = total[g];
    }
    // The eight partial sums of every (group, vector group) meet here: each consumer adds those of one
    // pair in wave order (the same bits on every run) and stores sixteen rows of four vectors.
    const uint32_t summed_address = lds_address(&control->summed);
    lds_arrive(summed_address, lane_id == 0);
    if (!lds_await(summed_address, kConsumers, patience)) return;
    for (uint32_t pair = wave; pair < groups * kSlots; pair += kConsumers) {
        const uint32_t group = pair / kSlots, g = pair - group * kSlots;
        float value = 0.f;
#pragma unroll
        for (int w = 0; w < kConsumers; w++)
            value += reinterpret_cast<const float*>(lds + kScratchAt + w * kWaveScratch)[pair * 64u + lane_id];
        const uint32_t vector = 4u * g + q, row = group * kGroupRows + n;
        if (vector < vectors && row < wg_rows) {
            if (bias != nullptr) value += bias[wg_row0 + row];
            y[static_cast<uint64_t>(vector) * rows + wg_row0 + row] = value;
        }
    }
}

// ---------------------------------------------------------------------------
// Rows wider than 4096 columns. The A operands of a whole row no longer fit the consumers' registers, and a workgroup
// holds few rows (sixteen of 14336 columns fill LDS), so that quantising the activations once per workgroup would cost
// more than everything else: gemv_mma_prepare_kernel does it once per call and leaves A operands in the order of the
// lanes that take them. The row is then walked in SLICES of eight 256-column units, one per consumer wave, whose operands
// arrive from L2 a slice ahead; one or two groups of sixteen rows are contracted and their sums stay in registers. The
// image of W lies slice after slice - [slice][row][slice bytes, padded to an odd number of 16-byte pieces so that
// sixteen rows at one column offset spread over the banks] - and lands in that order, so the first slices are
// contracted while the last ones are still in flight.
// Activations are 24-bit fixed point per vector and 64 columns, as in gemv_limb.hip, whose launches this replaces:
// X = rint(x * 127 * 2^16 / max|x|), limbs in [-128, 127]. One unit per 256 columns would let a single large activation
// coarsen 255 others instead of 63.
// ---------------------------------------------------------------------------
constexpr uint32_t kSliceUnits = kConsumers;
constexpr int kWideGroups = 2;
// Per consumer wave: the sums of its units, [slice][vector][kSumsFloats], and at the end its partial sums,
// [group][vector group][lane]. The image ends below the waves' scratch.
constexpr uint32_t kWidePartials = kWideGroups * 2u * 256u;
__host__ __device__ constexpr uint32_t wide_scratch(uint32_t row_units, uint32_t vectors) {
    const uint32_t sums = (row_units + kSliceUnits - 1u) / kSliceUnits * vectors * kSumsFloats * 4u;
    return sums > kWidePartials ? sums : kWidePartials;
}
constexpr float kWideRange = 8323072.0f;  // 127 * 2^16

// One (unit, vector) of the prepared activations: the three rows of the A operand that are the vector's,
// [block pair][limb][K index][16 bytes], then the f32 sums of the unit's eight blocks and the four units of limb 0. Nothing is
// kept for the zero rows and absent vectors: every workgroup reads all of this from L2.
constexpr uint32_t kWideRecordSumsAt = 768u, kWideRecord = 768u + kSumsFloats * 4u;

__host__ __device__ constexpr uint32_t slice_pitch(uint32_t slice_bytes) { return slice_bytes + (slice_bytes / 16u % 2u == 0 ? 16u : 0u); }

// Limb k of four 24-bit values X + 0x808080 into one dword each, as split_quad.
__device__ __forceinline__ void split_quad_24(int x0, int x1, int x2, int x3, uint32_t (&limb)[3]) {
    const uint32_t a = __builtin_amdgcn_perm(x1, x0, 0x05010400u), b = __builtin_amdgcn_perm(x3, x2, 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(x1, x0, 0x0c0c0602u), d = __builtin_amdgcn_perm(x3, x2, 0x0c0c0602u);
    limb[0] = __builtin_amdgcn_perm(b, a, 0x05040100u) ^ 0x80808080u;
    limb[1] = __builtin_amdgcn_perm(b, a, 0x07060302u) ^ 0x80808080u;
    limb[2] = __builtin_amdgcn_perm(d, c, 0x05040100u) ^ 0x80808080u;
}

// A wave per (unit, vector).
template <class T>
__global__ __launch_bounds__(64) void gemv_mma_prepare_kernel(const float* __restrict__ x, uint64_t x_row_stride,
                                                              uint8_t* __restrict__ prepared) {
    __shared__ uint32_t planes[3][64];
    const uint32_t unit = blockIdx.x, v = blockIdx.y, lane_id = threadIdx.x;
    uint8_t* out = prepared + (static_cast<uint64_t>(unit) * gridDim.y + v) * kWideRecord;
    const float4 f = *reinterpret_cast<const float4*>(x + v * x_row_stride + unit * 256u + lane_id * 4u);
    float amax = fmaxf(fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fabsf(f.z)), fabsf(f.w));
    float sum = (f.x + f.y) + (f.z + f.w);
    sum += dpp<0xB1>(sum);
    sum += dpp<0x4E>(sum);
    sum += dpp<0x141>(sum);  // eight lanes: the block's 32 columns
    amax = fmaxf(amax, dpp<0xB1>(amax));
    amax = fmaxf(amax, dpp<0x4E>(amax));
    amax = fmaxf(amax, dpp<0x141>(amax));
    amax = fmaxf(amax, dpp<0x140>(amax));  // sixteen lanes: 64 columns
    const bool nonzero = amax >= 1e-30f;
    const float inv = nonzero ? kWideRange / amax : 0.f;
    // to nearest even: a rounding with a bias would meet the mean of W's quants, which is not zero
    const auto fixed = [&](float value) { return static_cast<int>(rintf(value * inv)) + 0x808080; };
    uint32_t limb[3];
    split_quad_24(fixed(f.x), fixed(f.y), fixed(f.z), fixed(f.w), limb);
#pragma unroll
    for (int k = 0; k < 3; k++) planes[k][lane_id] = limb[k];
    float* sums = reinterpret_cast<float*>(out + kWideRecordSumsAt);
    if ((lane_id & 7u) == 0u) sums[lane_id >> 3] = sum;
    if ((lane_id & 15u) == 0u) sums[8u + (lane_id >> 4)] = nonzero ? amax * (1.0f / kWideRange) : 0.f;
    __syncthreads();
    if (lane_id < 48u) {  // lane: block pair, limb k, K index q
        const uint32_t pair = lane_id / 12u, k = lane_id % 12u >> 2, q = lane_id & 3u;
        const uint32_t* plane = planes[k] + pair * 16u + T::chunk(q) * 2u;  // block 2 pair; the next one 8 words on
        *reinterpret_cast<uint4*>(out + lane_id * 16u) = make_uint4(plane[0], plane[1], plane[8], plane[9]);
    }
}

template <class T, int VG, bool FIFTH, int LOADERS, int DEPTH, int AHEAD>
__global__ __launch_bounds__(64 * (kConsumers + LOADERS)) void gemv_mma_wide_kernel(
    const uint8_t* __restrict__ weight, const uint8_t* __restrict__ prepared, const float* __restrict__ bias,
    float* __restrict__ y, uint32_t rows, uint32_t columns, uint32_t rows_per_wg, uint32_t vectors, uint32_t spin_limit,
    uint32_t* timeouts) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    static_assert(DEPTH >= 1 && DEPTH <= 8 && LOADERS >= 1 && LOADERS <= 8, "wait_copies_in_flight counts to seven");
    static_assert(!FIFTH || VG == 1, "a fifth vector takes the rows of four");
    constexpr int kSlots = VG + FIFTH;
    Control* control = reinterpret_cast<Control*>(lds + kControlAt);

    const uint32_t lane_id = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wg_row0 = blockIdx.x * rows_per_wg;
    if (wg_row0 >= rows) return;
    const uint32_t wg_rows = min(rows_per_wg, rows - wg_row0);
    const uint32_t row_units = columns >> 8, row_bytes = row_units * T::kUnitBytes;
    // whole slices, then one of the remaining units (its rows closer together)
    constexpr uint32_t kSliceBytes = kSliceUnits * T::kUnitBytes, kPitch = slice_pitch(kSliceBytes);
    const uint32_t whole = row_units / kSliceUnits, rest_units = row_units % kSliceUnits;
    const uint32_t rest_bytes = rest_units * T::kUnitBytes, rest_pitch = slice_pitch(rest_bytes);
    const uint32_t rest_at = whole * wg_rows * kPitch;

    if (wave >= static_cast<uint32_t>(kConsumers)) {
        // ---- loaders: 1 KiB copies in turn, front to back over the image ------------------------
        const uint32_t loader = wave - kConsumers;
        // the image ends with the last byte of the last row of the last slice
        const uint32_t image_bytes = rest_units != 0u ? rest_at + (wg_rows - 1u) * rest_pitch + rest_bytes
                                                      : rest_at - kPitch + kSliceBytes;
        const uint32_t copies = (image_bytes + 1023u) >> 10;
        const uint32_t mine = copies > loader ? (copies - loader + LOADERS - 1u) / LOADERS : 0u;
        const uint8_t* source = weight + static_cast<uint64_t>(wg_row0) * row_bytes;
        const uint32_t landed_address = lds_address(&control->landed[loader]);
        // where this lane's 16 bytes of the wave's next copy lie: image byte `at`, in a whole slice byte `column` of
        // its row (a step at a time: two divisions per copy kept the loaders from filling their queues)
        constexpr uint32_t kStep = LOADERS * 1024u, kStepRows = kStep / kPitch, kStepColumns = kStep % kPitch;
        uint32_t next = loader, at = loader * 1024u + lane_id * 16u;
        uint32_t row = at / kPitch, column = at % kPitch, slice = row / wg_rows;
        row -= slice * wg_rows;
        const auto copy = [&]() {
            const uint8_t* from = source + row * row_bytes + slice * kSliceBytes + column;
            bool live = column < kSliceBytes && at < image_bytes;
            if (at >= rest_at) {
                const uint32_t line = (at - rest_at) / rest_pitch, byte = (at - rest_at) - line * rest_pitch;
                from = source + line * row_bytes + whole * kSliceBytes + byte;
                live = byte < rest_bytes && at < image_bytes;
            }
            // padding is shorter than a copy and the image ends with bytes of W: never a copy without a lane
            if (live)
                // streamed once: non-temporal (aux bit 1), the caches keep nothing of it
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint4*>(from), reinterpret_cast<uint4*>(lds + next * 1024u),
                                                 16, 0, 2);
            next += LOADERS;
            at += kStep;
            column += kStepColumns;
            row += kStepRows;
            if (column >= kPitch) {
                column -= kPitch;
                row++;
            }
            while (row >= wg_rows) {
                row -= wg_rows;
                slice++;
            }
        };
        __syncthreads();  // the consumers' first operand loads go ahead of the copies
        const uint32_t head = min(mine, static_cast<uint32_t>(DEPTH));
        for (uint32_t i = 0; i < head; i++) copy();
        uint32_t landed = 0;
        for (uint32_t i = head; i < mine; i++) {  // only with DEPTH copies in flight
            __builtin_amdgcn_s_waitcnt(vmcnt_only(DEPTH - 1));
            lds_store_unseen(landed_address, ++landed);
            copy();
        }
        for (uint32_t left = head; left > 0u; left--) {
            wait_copies_in_flight(left - 1u);
            lds_store_unseen(landed_address, ++landed);
        }
        return;
    }

    // ---- consumers --------------------------------------------------------------------------------
    Patience patience{spin_limit, timeouts};
    const uint32_t n = lane_id & 15u, q = lane_id >> 4;
    const uint32_t scratch_bytes = wide_scratch(row_units, vectors);
    uint8_t* scratch = lds + kControlAt - (kConsumers - wave) * scratch_bytes;
    const uint8_t* my_units = prepared + static_cast<uint64_t>(wave) * vectors * kWideRecord;
    const uint64_t slice_stride = static_cast<uint64_t>(kSliceUnits) * vectors * kWideRecord;
    // the wave's own slices: the row's last slice may have no unit for it
    const uint32_t my_slices = (row_units + kSliceUnits - 1u - wave) / kSliceUnits;
    union Operands {
        uint4 raw[VG][4];
        long a[VG][8];
    };
    // as A operand: row n = 4 * vector + limb; of a fifth vector 4 * limb + 3
    const bool in_fifth = FIFTH && (n & 3u) == 3u;
    const uint32_t limb = in_fifth ? n >> 2 : n & 3u;
    const auto load = [&](Operands& operands, uint32_t slice) {
#pragma unroll
        for (int g = 0; g < VG; g++) {
            const uint32_t vector = in_fifth ? 4u : 4u * g + (n >> 2);
            const uint8_t* from = my_units + slice * slice_stride + vector * kWideRecord + (limb * 4u + q) * 16u;
#pragma unroll
            for (int p = 0; p < 4; p++) {
                operands.raw[g][p] = make_uint4(0u, 0u, 0u, 0u);
                if (vector < vectors && limb != 3u) operands.raw[g][p] = *reinterpret_cast<const uint4*>(from + p * 192);
            }
        }
    };
    // AHEAD slices of operands are in flight while one is contracted: an L2 read takes longer than a slice
    Operands operands[AHEAD + 1];
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
        if (static_cast<uint32_t>(i) < my_slices) load(operands[i], i);
    float* sums = reinterpret_cast<float*>(scratch);
    for (uint32_t i = lane_id; i < my_slices * vectors * 3u; i += 64u) {
        const uint32_t record = i / 3u, slice = record / vectors, vector = record - slice * vectors;
        *reinterpret_cast<float4*>(sums + 4u * i) = *reinterpret_cast<const float4*>(
            my_units + slice * slice_stride + vector * kWideRecord + kWideRecordSumsAt + (i - 3u * record) * 16u);
    }
    if (threadIdx.x < 16) reinterpret_cast<uint32_t*>(control)[threadIdx.x] = 0u;
    __syncthreads();  // the only barrier: the counters are zero before anybody counts

    const uint32_t groups = (wg_rows + kGroupRows - 1u) / kGroupRows;
    const float* of_result = sums + min(q, vectors - 1u) * kSumsFloats;  // result rows past `vectors` are not stored
    const uint32_t sums_step = (min(q + 4u, vectors - 1u) - min(q, vectors - 1u)) * kSumsFloats;
    float total[kWideGroups][kSlots];
#pragma unroll
    for (int i = 0; i < kWideGroups; i++)
#pragma unroll
        for (int g = 0; g < kSlots; g++) total[i][g] = 0.f;
    for (uint32_t first = 0; first < my_slices; first += AHEAD + 1) {
#pragma unroll
        for (int i = 0; i <= AHEAD; i++) {  // unrolled: operand sets change their roles, not their registers
            const uint32_t slice = first + i;
            if (slice >= my_slices) break;
            if (slice + AHEAD < my_slices) load(operands[(i + AHEAD) % (AHEAD + 1)], slice + AHEAD);
            const bool in_rest = slice == whole;
            const uint32_t pitch = in_rest ? rest_pitch : kPitch, bytes = in_rest ? rest_bytes : kSliceBytes;
            const uint32_t slice_at = slice * wg_rows * kPitch;
#pragma unroll
            for (int group = 0; group < kWideGroups; group++) {
                if (static_cast<uint32_t>(group) >= groups) break;
                const uint32_t last_row = min(group * kGroupRows + kGroupRows, wg_rows) - 1u;
                if (!await_copies_in_turn<LOADERS>(control->landed, lane_id, (slice_at + last_row * pitch + bytes + 1023u) >> 10, patience))
                    continue;
                // rows past the end of the range read its last row again and are not stored
                const uint8_t* rp = lds + slice_at + min(group * kGroupRows + n, wg_rows - 1u) * pitch + wave * T::kUnitBytes;
                T::template contract<VG, 0, 4, FIFTH>(rp, q, operands[i].a, of_result + slice * vectors * kSumsFloats, sums_step,
                                                      sums + (slice * vectors + 4u) * kSumsFloats, total[group]);
            }
        }
    }
    asm volatile("" ::: "memory");  // the sums are read no more
    float* partial = reinterpret_cast<float*>(scratch);
#pragma unroll
    for (int group = 0; group < kWideGroups; group++)
#pragma unroll
        for (int g = 0; g < kSlots; g++) partial[(group * kSlots + g) * 64u + lane_id] = total[group][g];
    // as in gemv_mma_kernel: the eight partial sums of a pair are added in wave order
    const uint32_t summed_address = lds_address(&control->summed);
    lds_arrive(summed_address, lane_id == 0);
    if (!lds_await(summed_address, kConsumers, patience)) return;
    for (uint32_t pair = wave; pair < groups * kSlots; pair += kConsumers) {
        const uint32_t group = pair / kSlots, g = pair - group * kSlots;
        float value = 0.f;
#pragma unroll
        for (int w = 0; w < kConsumers; w++)
            value += reinterpret_cast<const float*>(lds + kControlAt - (kConsumers - w) * scratch_bytes)[pair * 64u + lane_id];
        const uint32_t vector = 4u * g + q, row = group * kGroupRows + n;
        if (vector < vectors && row < wg_rows) {
            if (bias != nullptr) value += bias[wg_row0 + row];
            y[static_cast<uint64_t>(vector) * rows + wg_row0 + row] = value;
        }
    }
}

// Rows of W whose slices fit a workgroup's LDS.
uint32_t wide_rows_that_fit(uint64_t columns, uint32_t vectors, uint32_t unit_bytes) {
    const uint32_t units = static_cast<uint32_t>(columns >> 8), whole = units / kSliceUnits, rest = units % kSliceUnits;
    const uint32_t scratch = kConsumers * wide_scratch(units, vectors);
    if (scratch >= kControlAt) return 0;
    const uint32_t per_row = whole * slice_pitch(kSliceUnits * unit_bytes) + (rest != 0 ? slice_pitch(rest * unit_bytes) : 0u);
    return std::min((kControlAt - scratch) / per_row, kWideGroups * kGroupRows);
}

// Rows of a workgroup's range: a two-hundred-fifty-sixth of the matrix when `most` rows (what fits LDS and the
// partial sums' slots) hold it; else the matrix is cut into the fewest rounds of 256 ranges that do.
uint32_t range_rows(uint32_t rows, uint32_t most) {
    const uint32_t share = (rows + 255u) / 256u;
    if (share <= most) return share;
    const uint32_t rounds = (share + most - 1u) / most;
    return (rows + 256u * rounds - 1u) / (256u * rounds);
}
uint32_t rows_that_fit(uint32_t row_bytes) {
    return std::min((kScratchAt - row_bytes) / image_pitch(row_bytes) + 1u, kMostGroups * kGroupRows);
}

// The whole LDS of a compute unit has to be allowed once per kernel and device.
template <typename Kernel>
hipError_t allow_lds(Kernel kernel, std::atomic<bool> (&allowed)[64]) {
    int device = 0;
    if (hipError_t status = hipGetDevice(&device)) return status;
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    if (!allowed[device].load(std::memory_order_acquire)) {
        if (hipError_t status = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes))
            return status;
        allowed[device].store(true, std::memory_order_release);
    }
    return hipSuccess;
}

template <class T, int VG, bool FIFTH, int LOADERS, int DEPTH>
hipError_t launch(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias, float* y,
                  uint32_t rows, uint32_t columns, uint32_t vectors, hipStream_t stream) {
    static std::atomic<bool> allowed[64];
    const auto kernel = gemv_mma_kernel<T, VG, FIFTH, LOADERS, DEPTH>;
    if (hipError_t status = allow_lds(kernel, allowed)) return status;
    HandoverState handover;
    if (hipError_t status = handover_state(&handover)) return status;
    const uint32_t rows_per_wg = range_rows(rows, rows_that_fit((columns >> 8) * T::kUnitBytes));
    const uint32_t grid = (rows + rows_per_wg - 1u) / rows_per_wg;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * (kConsumers + LOADERS)), kLdsBytes, stream, weight, x, x_row_stride,
                       bias, y, rows, columns, rows_per_wg, vectors, handover.limit, handover.timeouts);
    return hipGetLastError();
}

template <class T, int VG, bool FIFTH, int LOADERS, int DEPTH, int AHEAD>
hipError_t launch_wide(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias, float* y,
                       uint32_t rows, uint32_t columns, uint32_t vectors, uint8_t* prepared, hipStream_t stream) {
    static std::atomic<bool> allowed[64];
    const auto kernel = gemv_mma_wide_kernel<T, VG, FIFTH, LOADERS, DEPTH, AHEAD>;
    if (hipError_t status = allow_lds(kernel, allowed)) return status;
    HandoverState handover;
    if (hipError_t status = handover_state(&handover)) return status;
    hipLaunchKernelGGL(gemv_mma_prepare_kernel<T>, dim3(columns >> 8, vectors), dim3(64), 0, stream, x, x_row_stride, prepared);
    if (hipError_t status = hipGetLastError()) return status;
    const uint32_t rows_per_wg = range_rows(rows, wide_rows_that_fit(columns, vectors, T::kUnitBytes));
    const uint32_t grid = (rows + rows_per_wg - 1u) / rows_per_wg;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * (kConsumers + LOADERS)), kLdsBytes, stream, weight, prepared, bias, y,
                       rows, columns, rows_per_wg, vectors, handover.limit, handover.timeouts);
    return hipGetLastError();
}

template <class T>
hipError_t launch_vectors(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias, float* y,
                          uint32_t rows, uint32_t columns, uint32_t vectors, uint8_t* prepared, hipStream_t stream) {
    // Two vector groups keep 64 registers of A operands: twelve waves leave each 168. Five vectors are fifteen limbs and fit
    // one operand: half the matrix instructions of two groups, a multiply-add per block and eight instructions per unit more
    // than four vectors. In a graph, two groups / one (us; the same inputs again | inputs from memory): Q4_K 4096 x 14336 17.9 /
    // 15.7 | 18.0 / 16.6, 14336 x 4096 12.0 / 11.2 | 12.9 / 12.0, 4096 x 4096 7.4 / 7.0 | 7.3 / 6.9; Q5_K 31.6 / 27.2 | 31.1 / 27.3, 17.2 /
    // 16.3 | 17.3 / 16.4, 7.4 / 6.9 | 7.5 / 7.2. The fifth vector's error against 64 bits is what it was. Not Q4_0 and Q8_0: a
    // scale per block would have to meet the limbs' sums one by one, where an infinite one makes NaN of two signs, or the
    // groups be put together for every block.
    if (columns > kNarrowColumns) {
        if (prepared == nullptr) return hipErrorInvalidValue;
        if (vectors <= 4) return launch_wide<T, 1, false, 8, 4, 2>(weight, x, x_row_stride, bias, y, rows, columns, vectors, prepared, stream);
        if constexpr (T::kTakesFifth)
            if (vectors == 5) return launch_wide<T, 1, true, 8, 4, 2>(weight, x, x_row_stride, bias, y, rows, columns, vectors, prepared, stream);
        return launch_wide<T, 2, false, 4, 8, 1>(weight, x, x_row_stride, bias, y, rows, columns, vectors, prepared, stream);
    }
    if (vectors <= 4) return launch<T, 1, false, 8, 4>(weight, x, x_row_stride, bias, y, rows, columns, vectors, stream);
    if constexpr (T::kTakesFifth)
        if (vectors == 5) return launch<T, 1, true, 8, 4>(weight, x, x_row_stride, bias, y, rows, columns, vectors, stream);
    return launch<T, 2, false, 4, 8>(weight, x, x_row_stride, bias, y, rows, columns, vectors, stream);
}

}  // namespace

bool gemv_mma_supported(int32_t codec, uint64_t rows, uint64_t columns, uint32_t vectors) {
    if (codec != kQ4_K && codec != kQ4_0 && codec != kQ5_K && codec != kQ8_0) return false;
    if (vectors < 2 || vectors > kGemvMmaMaxVectors) return false;
    // the copies are 16 bytes wide (a unit is a multiple of 16 bytes)
    if (columns == 0 || columns % 256 != 0) return false;
    // with less than a group of rows to a compute unit most of every matrix instruction is padding
    if (rows < 256u * 8u || rows > 0xffffffffull) return false;
    if (columns <= kNarrowColumns) return true;
    // Wider rows, against the launches of gemv_limb.hip (two or three vectors each), us, this / those: Q4_K 4096 x 14336 with
    // 2 / 3 / 5 vectors 12.9 / 13.2 / 17.2 against 17.1 / 22.3 / 39.7; Q8_0 3072 x 12800, whose ranges take two rounds of
    // workgroups, 3 vectors 19.9 (23.9), 2 vectors slower: a second round of ranges is worth it from three vectors on where
    // LDS holds less than a group of sixteen rows.
    // Two vectors on at most 8192 columns are one launch there, without the preparing one: 2048 x 7936 Q4_K 10.2 (8.0), Q8_0
    // 10.0 (7.7), 4096 x 8192 Q8_0 11.3 (9.7); 5120 x 4608 Q4_K 10.6 (11.2) is the most that is given away. Wider ones take
    // twice the launches' slices: 3072 x 8704 Q4_K 10.6 (14.3).
    // Not taken up: from seven vectors on the batch kernels' plans hold prepared inputs, which callers may share between
    // plans; more rounds of ranges, although they would be faster at least once (14336 x 5120, 4 vectors 18.2 against 41.4).
    if (vectors == 2u && columns <= 8192u) return false;
    if (vectors > 6u || columns > (1u << 20)) return false;
    const uint32_t unit_bytes = static_cast<uint32_t>(256 / block_values(codec) * block_bytes(codec));
    const uint32_t fit = wide_rows_that_fit(columns, vectors, unit_bytes);
    return rows <= 256u * fit || (vectors > 2u && fit >= 8u && fit < kGroupRows && rows <= 512u * fit);
}

uint64_t gemv_mma_prepared_bytes(uint64_t columns, uint32_t vectors) {
    if (columns <= kNarrowColumns) return 0;
    return (columns >> 8) * vectors * kWideRecord;
}

hipError_t gemv_mma(int32_t codec, const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias,
                    float* y, uint64_t rows, uint64_t columns, uint32_t vectors, uint8_t* prepared, hipStream_t stream) {
    const uint32_t n = static_cast<uint32_t>(rows), k = static_cast<uint32_t>(columns);
    if (!gemv_mma_supported(codec, rows, columns, vectors)) return hipErrorInvalidValue;
    switch (codec) {
        case kQ4_K: return launch_vectors<Q4KMma>(weight, x, x_row_stride, bias, y, n, k, vectors, prepared, stream);
        case kQ5_K: return launch_vectors<Q5KMma>(weight, x, x_row_stride, bias, y, n, k, vectors, prepared, stream);
        case kQ4_0: return launch_vectors<Q40Mma>(weight, x, x_row_stride, bias, y, n, k, vectors, prepared, stream);
        case kQ8_0: return launch_vectors<Q80Mma>(weight, x, x_row_stride, bias, y, n, k, vectors, prepared, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace et
