// One-vector contractions of a decode step with the small operators around them in the same launch:
//     y_i[r] = sum_k f(x)[k] * decode(W_i[r])[k] (+ residual_i[r])
// for up to four matrices W_i of one codec and width, f(x) = x or rms_norm(x) * w; or, for two matrices of the same
// rows, y[r] = silu(gate[r]) * up[r] from the rows of both (PAIR).
//
// Bound: launches. At one vector a layer's weights are 123 MB (25 us at the rate of a large copy) in contractions of 4
// to 12 us, and every launch next to them - norm, rotary, SiLU, residual sum - lasts 2 to 5 us for a few KB: 17 launches a
// layer of 4096 columns and 14336 feed-forward rows. Here the norm's squares are summed by the eight waves that hold the
// activations anyway, in front of their folds, the residual and SiLU ride on the stores, and one grid over several matrices
// saves the ramp of all but one. Traced, Q4_K (us): norm + q + k + v 16.6 in four launches -> 6.0; norm + gate + up + SiLU
// 25.9 in four -> 16.2; down + residual 14.0 in two -> 10.7; a step of four layers at context 1000 399 -> 290.
//
// The contraction is gemv_limb_kernel's (gemv_limb.hip) for one vector: the same limbs, the same folds, the same sums in
// the same order. All slices of a wide row are staged at once (13 KiB of LDS each, behind one barrier and one round trip
// to L2) instead of one after the other.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "decode_math.h"
#include "et_codecs.h"
#include "gemv_common.h"
#include "gemv_limb_device.h"
#include "kernels.h"

namespace et {
namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves;

struct StepArgs {
    const float* x;
    const void* norm;  // [columns] floats or halves, or null: ones; used when `normed`
    int32_t normed, norm_half;
    double eps;
    // launch rows: the members' rows one after the other; PAIR: rows 2 r and 2 r + 1 are row r of members 0 and 1
    uint32_t rows, columns, rows_per_wg;
    // Where launch row r's weights, result and residual are: that many bytes (floats) past those of member 0's row 0 plus
    // r rows, a sum over the members that start at or in front of r. Sums of steps and not a choice of pointers: the
    // compiler turns that into a load from the chosen place in the arguments, a round trip to memory in front of each row.
    uint32_t first[kGemvStepMost];  // first launch row; unused members start past the end
    int64_t weight_step[kGemvStepMost], y_step[kGemvStepMost], residual_step[kGemvStepMost];
    uint32_t residuals;  // bit i: member i has one
    const uint8_t* weight;
    const float* residual;
    float* y;
};

// Sum over the 64 lanes of a wave, in every lane: wave_sum of gemv_common.h in f64 (a sum through ds_bpermute takes six
// round trips to LDS).
__device__ __forceinline__ double wave_sum_f64(double v) {
    const auto moved = [](double value, auto move) {
        const uint64_t bits = __double_as_longlong(value);
        const uint32_t low = move(static_cast<uint32_t>(bits)), high = move(static_cast<uint32_t>(bits >> 32));
        return __longlong_as_double(static_cast<long long>(static_cast<uint64_t>(high) << 32 | low));
    };
    v += moved(v, [](uint32_t w) { return __builtin_amdgcn_update_dpp(0, w, 0xB1, 0xF, 0xF, true); });
    v += moved(v, [](uint32_t w) { return __builtin_amdgcn_update_dpp(0, w, 0x4E, 0xF, 0xF, true); });
    v += moved(v, [](uint32_t w) { return __builtin_amdgcn_update_dpp(0, w, 0x141, 0xF, 0xF, true); });
    v += moved(v, [](uint32_t w) { return __builtin_amdgcn_update_dpp(0, w, 0x140, 0xF, 0xF, true); });
    const double r0 = moved(v, [](uint32_t w) { return __builtin_amdgcn_readlane(w, 0); });
    const double r1 = moved(v, [](uint32_t w) { return __builtin_amdgcn_readlane(w, 16); });
    const double r2 = moved(v, [](uint32_t w) { return __builtin_amdgcn_readlane(w, 32); });
    const double r3 = moved(v, [](uint32_t w) { return __builtin_amdgcn_readlane(w, 48); });
    return (r0 + r1) + (r2 + r3);
}

// R rows of a wave per turn, NK waves per row. LOOP = false: R covers all of a wave's rows, each requested before
// the one in front of it is folded; LOOP = true: two buffers of R rows in turn.
template <class T, int R, int NK, bool PAIR, bool LOOP>
__global__ __launch_bounds__(kThreads) void gemv_step_kernel(const StepArgs a) {
    constexpr int RG = kWaves / NK;
    constexpr int NI = NK * static_cast<int>(kSliceQuads) / kThreads;  // float4s per thread
    static_assert(!PAIR || R % 2 == 0, "a wave folds whole pairs");
    __shared__ StageMemory stage[NK];
    __shared__ float partial[2][RG][NK][R];
    __shared__ double squares[kWaves];
    const uint32_t lane_id = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t slice = wave % NK, group = wave / NK;
    const uint32_t quads = a.columns >> 2;

    // Activations first: L2 serves them and they must not queue behind weights (a wave's loads return in order). The norm's
    // weights are asked for next and looked at only when the squares have been summed.
    float4 xv[NI];
    uint4 wv[NI];
#pragma unroll
    for (int i = 0; i < NI; i++)
        xv[i] = reinterpret_cast<const float4*>(a.x)[min(threadIdx.x + i * kThreads, quads - 1u)];
    if (a.normed && a.norm != nullptr) {  // any alignment its elements have
        if (a.norm_half) {
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint2 two = static_cast<const uint2_a2*>(a.norm)[min(threadIdx.x + i * kThreads, quads - 1u)];
                wv[i].x = two.x;
                wv[i].y = two.y;
            }
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++)
                wv[i] = static_cast<const uint4_a4*>(a.norm)[min(threadIdx.x + i * kThreads, quads - 1u)];
        }
    }

    const uint32_t chunk = slice * 64u + lane_id;  // which 64-column stretch of the row
    const bool active = chunk < a.columns / kChunk;
    const typename T::Lane lane = T::lane_setup(active ? chunk : 0u);
    const uint64_t row_bytes = T::row_bytes(a.columns);
    const uint32_t wg_row0 = blockIdx.x * a.rows_per_wg;
    const uint32_t wg_row_end = min(wg_row0 + a.rows_per_wg, a.rows);

    const auto load_row = [&](uint32_t it, int r, typename T::Data& data) {
        uint32_t row = wg_row0 + (it * RG + group) * R + r;
        row = min(row, a.rows - 1);  // rows past the end re-read a valid row and are discarded
        int64_t at = 0;
        if constexpr (PAIR) {
            at = row & 1u ? a.weight_step[1] : 0;
            row >>= 1;
        } else {
#pragma unroll
            for (uint32_t i = 1; i < kGemvStepMost; i++) at += row >= a.first[i] ? a.weight_step[i] : 0;
        }
        T::load(a.weight + (at + static_cast<int64_t>(row * row_bytes)), lane, data);
    };

    // One row of weights travels while the activations are prepared; the others, which may stall on a full queue,
    // are asked for behind the barrier (gemv_limb_kernel).
    typename T::Data current[R];
    load_row(0, 0, current[0]);
    __builtin_amdgcn_sched_barrier(0);

#pragma unroll
    for (int i = 0; i < NI; i++)
        if (threadIdx.x + i * kThreads >= quads) xv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.normed) {  // rms_norm's arithmetic (decode_math.h): squares summed in f64, one rounding per element
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < NI; i++)
            sum += (static_cast<double>(xv[i].x) * xv[i].x + static_cast<double>(xv[i].y) * xv[i].y) +
                   (static_cast<double>(xv[i].z) * xv[i].z + static_cast<double>(xv[i].w) * xv[i].w);
        sum = wave_sum_f64(sum);
        if (lane_id == 0) squares[wave] = sum;
        __syncthreads();
        double total = squares[0];
#pragma unroll
        for (int w = 1; w < kWaves; w++) total += squares[w];
        const double scale = 1.0 / sqrt(total / static_cast<double>(a.columns) + a.eps);
#pragma unroll
        for (int i = 0; i < NI; i++) {
            float4 w = make_float4(1.f, 1.f, 1.f, 1.f);
            if (a.norm != nullptr)
                w = a.norm_half ? make_float4(half_bits_to_float(wv[i].x & 0xffffu), half_bits_to_float(wv[i].x >> 16),
                                              half_bits_to_float(wv[i].y & 0xffffu), half_bits_to_float(wv[i].y >> 16))
                                : make_float4(__uint_as_float(wv[i].x), __uint_as_float(wv[i].y), __uint_as_float(wv[i].z),
                                              __uint_as_float(wv[i].w));
            xv[i] = rms_four(xv[i], scale, w);
        }
#pragma unroll
        for (int i = 0; i < NI; i++)  // a row that is all infinities or NaN does not reach the columns past its end
            if (threadIdx.x + i * kThreads >= quads) xv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < NI; i++)
        stage_quad(stage[i * kThreads / kSliceQuads], xv[i], (threadIdx.x + i * kThreads) % kSliceQuads);
    __syncthreads();
    XLimbs xr[1];
    T::load_activations(stage[slice], lane_id, active, xr[0]);

    // Lane r of the wave that writes a group's results writes launch row r of it (PAIR: r / 2).
    struct Target {
        bool mine, add;
        int64_t y, residual;
    };
    const auto target = [&](uint32_t it) {
        uint32_t row = wg_row0 + (it * RG + group) * R + (PAIR ? 2u * lane_id : lane_id);
        Target t;
        t.mine = lane_id < (PAIR ? R / 2 : R) && row < wg_row_end && (NK == 1 || slice == 0);
        t.add = !PAIR && (a.residuals & 1u);
        if (PAIR) row >>= 1;
        t.y = row;
        t.residual = row + a.residual_step[0];
        if constexpr (!PAIR) {
#pragma unroll
            for (uint32_t i = 1; i < kGemvStepMost; i++) {
                const bool behind = row >= a.first[i];
                t.y += behind ? a.y_step[i] : 0;
                t.residual += behind ? a.residual_step[i] : 0;
                t.add = behind ? (a.residuals >> i) & 1u : t.add;
            }
        }
        t.add = t.add && t.mine;
        return t;
    };
    const auto write_rows = [&](uint32_t it, const float (&total)[R], const Target& t, float added) {
        float value = 0.f, second = 0.f;
        if constexpr (NK == 1) {
            // the totals are the same in all lanes; lane r (PAIR: lane r / 2) takes the one it writes
            const auto lane_value = [&](float into, float from, uint32_t lane) {
                asm("" : "+v"(from));  // a select, not an array in LDS that the lane indexes
                return lane_id == lane ? from : into;
            };
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (!PAIR)
                    value = lane_value(value, total[r], r);
                else if (r % 2 == 0)
                    value = lane_value(value, total[r], r / 2);
                else
                    second = lane_value(second, total[r], r / 2);
            }
        } else {
            const uint32_t parity = it & 1u;
            if (lane_id == 0) {
#pragma unroll
                for (int r = 0; r < R; r++) partial[parity][group][slice][r] = total[r];
            }
            __syncthreads();
            if (t.mine) {
                const uint32_t r = PAIR ? 2u * lane_id : lane_id;
                value = 0.f;
                for (int s = 0; s < NK; s++) value += partial[parity][group][s][r];
                if constexpr (PAIR)
                    for (int s = 0; s < NK; s++) second += partial[parity][group][s][r + 1u];
            }
        }
        if (!t.mine) return;
        if constexpr (PAIR) value = silu_mul_one(value, second);
        a.y[t.y] = t.add ? added + value : value;
    };
    const auto fold_row = [&](const typename T::Data& data) {
        float value[1];
        T::template fold<1>(data, lane, xr, value);
        return wave_sum(active ? value[0] : 0.f);
    };

    float total[R];
    if constexpr (!LOOP) {
        // the residuals travel in front of the weights, not behind them
        const Target t = target(0);
        const float added = t.add ? a.residual[t.residual] : 0.f;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r + 1 < R) load_row(0, r + 1, current[r + 1]);
            __builtin_amdgcn_sched_barrier(0);
            total[r] = fold_row(current[r]);
            __builtin_amdgcn_sched_barrier(0);
        }
        write_rows(0, total, t, added);
    } else {
        const uint32_t turns = (wg_row_end - wg_row0 + RG * R - 1) / (RG * R);
        typename T::Data other[R];
#pragma unroll
        for (int r = 1; r < R; r++) load_row(0, r, current[r]);
        const auto finish = [&](uint32_t it, const typename T::Data (&data)[R]) {
            const Target t = target(it);
            const float added = t.add ? a.residual[t.residual] : 0.f;
#pragma unroll
            for (int r = 0; r < R; r++) total[r] = fold_row(data[r]);
            write_rows(it, total, t, added);
        };
        for (uint32_t it = 0; it < turns; it += 2) {
            if (it + 1 < turns) {
#pragma unroll
                for (int r = 0; r < R; r++) load_row(it + 1, r, other[r]);
            }
            finish(it, current);
            if (it + 1 < turns) {
                if (it + 2 < turns) {
#pragma unroll
                    for (int r = 0; r < R; r++) load_row(it + 2, r, current[r]);
                }
                finish(it + 1, other);
            }
        }
    }
}

template <class T, int R, int NK, bool PAIR, bool LOOP>
hipError_t launch(StepArgs a, uint32_t rows_per_wg, hipStream_t stream) {
    a.rows_per_wg = rows_per_wg;
    hipLaunchKernelGGL((gemv_step_kernel<T, R, NK, PAIR, LOOP>), dim3((a.rows + rows_per_wg - 1) / rows_per_wg),
                       dim3(kThreads), 0, stream, a);
    return hipGetLastError();
}

// One contiguous range of launch rows per compute unit; up to eight rows of a wave fit its registers.
template <class T, int NK, bool PAIR>
hipError_t launch_rows(const StepArgs& a, hipStream_t stream) {
    constexpr uint32_t RG = kWaves / NK;
    const uint32_t share = (a.rows + 255u) / 256u;
    uint32_t depth = (share + RG - 1) / RG;
    if (PAIR) depth = (depth + 1u) / 2u * 2u;
#define ET_SHOT(D) \
    case D: return launch<T, D, NK, PAIR, false>(a, RG * D, stream)
    if constexpr (PAIR) {
        switch (depth) {
            ET_SHOT(2);
            ET_SHOT(4);
            ET_SHOT(6);
            ET_SHOT(8);
            default: break;
        }
    } else {
        switch (depth) {
            ET_SHOT(1);
            ET_SHOT(2);
            ET_SHOT(3);
            ET_SHOT(4);
            ET_SHOT(5);
            ET_SHOT(6);
            ET_SHOT(7);
            ET_SHOT(8);
            default: break;
        }
    }
#undef ET_SHOT
    return launch<T, 2, NK, PAIR, true>(a, (share + RG * 2 - 1) / (RG * 2) * (RG * 2), stream);
}

template <class T>
hipError_t launch_slices(const StepArgs& a, bool pair, hipStream_t stream) {
    const uint32_t slices = (a.columns + kSliceColumns - 1) / kSliceColumns;
    if (slices <= 1) return pair ? launch_rows<T, 1, true>(a, stream) : launch_rows<T, 1, false>(a, stream);
    if (slices <= 2) return pair ? launch_rows<T, 2, true>(a, stream) : launch_rows<T, 2, false>(a, stream);
    if (slices <= 4 && !pair) return launch_rows<T, 4, false>(a, stream);
    return hipErrorInvalidValue;
}

}  // namespace

bool gemv_step_supported(int32_t codec, uint64_t columns, bool pair) {
    return gemv_limb_supported(codec, columns, 1) && columns <= (pair ? 2u : 4u) * kSliceColumns;
}

hipError_t gemv_step(int32_t codec, const GemvStep& s, hipStream_t stream) {
    if (s.count == 0 || s.count > kGemvStepMost || !gemv_step_supported(codec, s.columns, s.silu_mul) ||
        (s.silu_mul && (s.count != 2 || s.rows[0] != s.rows[1])))
        return hipErrorInvalidValue;
    StepArgs a{};
    a.x = s.x;
    a.norm = s.norm_weight;
    a.normed = s.normed;
    a.norm_half = s.norm_weight_is_half;
    a.eps = s.eps;
    a.columns = static_cast<uint32_t>(s.columns);
    a.weight = s.weight[0];
    a.y = s.y[0];
    a.residual = s.y[0];  // residuals by their distance from there
    const auto floats_from_y0 = [&](const float* p) {
        return (static_cast<int64_t>(reinterpret_cast<uintptr_t>(p)) - static_cast<int64_t>(reinterpret_cast<uintptr_t>(s.y[0]))) / 4;
    };
    const int64_t row_bytes = static_cast<int64_t>(s.row_bytes);
    uint64_t rows = 0;
    int64_t weight_at = 0, y_at = 0, residual_at = 0;  // of the member in front, less its first row
    for (uint32_t i = 0; i < kGemvStepMost; i++) {
        a.first[i] = i < s.count ? static_cast<uint32_t>(rows) : 0xffffffffu;
        if (i >= s.count) continue;
        const int64_t first = s.silu_mul ? 0 : static_cast<int64_t>(rows);
        const int64_t weight = static_cast<int64_t>(reinterpret_cast<uintptr_t>(s.weight[i])) -
                               static_cast<int64_t>(reinterpret_cast<uintptr_t>(s.weight[0])) - first * row_bytes;
        a.weight_step[i] = weight - weight_at;
        weight_at = weight;
        rows += s.rows[i];
        if (s.silu_mul) continue;
        const int64_t y = floats_from_y0(s.y[i]) - first;
        a.y_step[i] = y - y_at;
        y_at = y;
        if (s.residual[i] != nullptr) {
            const int64_t residual = floats_from_y0(s.residual[i]) - first;
            a.residual_step[i] = residual - residual_at;
            residual_at = residual;
            a.residuals |= 1u << i;
        }
    }
    if (rows == 0) return hipSuccess;
    if (rows > 0x7fffffffull) return hipErrorInvalidValue;
    a.rows = static_cast<uint32_t>(rows);
    switch (codec) {
        case kQ2_K: return launch_slices<Q2KLimb>(a, s.silu_mul, stream);
        case kQ3_K: return launch_slices<Q3KLimb>(a, s.silu_mul, stream);
        case kQ4_K: return launch_slices<Q4KLimb>(a, s.silu_mul, stream);
        case kQ5_K: return launch_slices<Q5KLimb>(a, s.silu_mul, stream);
        case kQ6_K: return launch_slices<Q6KLimb>(a, s.silu_mul, stream);
        case kQ4_0: return launch_slices<Q40Limb>(a, s.silu_mul, stream);
        case kQ8_0: return launch_slices<Q80Limb>(a, s.silu_mul, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace et
