// Dequant-GEMV on integer dot products for gfx950 (the five K-quants, Q4_0, Q8_0; 1-3 vectors):
//     y[v, r] = sum_k x[v, k] * decode(W[r])[k] (+ bias[r])
//
// Same contraction as linear_into (crates/runtime-cpu/src/quantized.rs:419-499)
// with decode_q4_k (:180-199) in factored form; Q4_0 / Q8_0 follow the public
// ggml block layouts. f32-accurate: the result agrees with the scalar f32 loop
// within 1e-3 (in fact to a few 1e-6 relative).
//
// Why integers. The kernel is HBM-bound (0.56 - 1.06 bytes per weight), and on
// CDNA4 the obvious f32 formulation (byte -> float convert + FMA per weight) is
// VALU-bound before it is HBM-bound: ~2.4 vector ops per weight. Here each f32
// activation is converted ONCE per workgroup to a 24-bit fixed-point integer
// with a shared scale per 64 columns, X = rint(x * 127 * 2^16 / max|x|), and X
// is cut into three signed 8-bit limbs,
//     x ~= s * (65536*x1 + 256*x2 + x3),   |residual| <= 6.0e-8 * max|x|,
// i.e. to f32 precision. The weights' quants - already small integers - meet
// the limbs in v_dot4_i32_i8: 4 multiply-adds per op, three ops per four
// weights, exact int32 accumulation. Block scales are applied to the integer
// sums in f32 afterwards. ~1.3 vector ops per weight.
//
// Work split (activation-stationary): a lane owns 64 consecutive columns (one
// 32-byte pair of a Q4_K super-block, or two Q4_0 / Q8_0 blocks), keeps their
// limbs in registers for its whole life, and streams weight rows past them with
// 16-byte loads. A wave covers 4096 columns, NK waves a row; their partial sums
// meet in LDS. A workgroup walks a contiguous range of rows.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdlib>

#include "et_codecs.h"
#include "gemv_common.h"
#include "gemv_limb_device.h"
#include "kernels.h"
#include "lds_handover.h"

namespace et {
namespace {

// ---------------------------------------------------------------------------
// The kernel. M vectors, R rows per wave iteration, WAVES waves per workgroup,
// NK waves per row (so WAVES / NK row groups per workgroup).
//
// A 33 MB GEMV lasts only a few microseconds, comparable to a handful of HBM
// round trips, so what counts is how early the whole weight matrix is in
// flight. LOOP = false is the single-shot form: every wave requests ALL its rows
// (R <= 8) as its very first instructions after the activation loads, then
// prepares the activations while the weights travel, then folds the rows as
// they arrive. LOOP = true keeps two R-row buffers in ping-pong for shapes
// whose rows per wave do not fit registers.
// ---------------------------------------------------------------------------
template <class T, int M, int R, int WAVES, int NK, bool LOOP>
__global__ __launch_bounds__(64 * WAVES) void gemv_limb_kernel(
    const uint8_t* __restrict__ weight, const float* __restrict__ x, uint64_t x_row_stride,
    const float* __restrict__ bias, float* __restrict__ y, uint32_t rows, uint32_t columns,
    uint32_t rows_per_wg) {
    constexpr int RG = WAVES / NK;
    constexpr int THREADS = 64 * WAVES;
    constexpr int NI = (kSliceQuads + THREADS - 1) / THREADS;  // float4s per thread and slice
    __shared__ StageMemory stage[M];
    __shared__ float partial[2][RG][NK][R][M];
    const uint32_t lane_id = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t slice = wave % NK;
    const uint32_t group = wave / NK;
    const uint32_t all_quads = columns >> 2;

    // Activation loads first: they are served by L2 and must not queue behind
    // the weight loads (a wave's loads complete in order).
    auto load_x = [&](uint32_t s, float4 (&xv)[M][NI]) {
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t f = threadIdx.x + i * THREADS;
                const uint32_t quad = s * kSliceQuads + f;
                xv[m][i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (f < kSliceQuads && quad < all_quads)
                    xv[m][i] = reinterpret_cast<const float4*>(x + m * x_row_stride)[quad];
            }
    };
    float4 xv[M][NI];
    load_x(0, xv);

    const uint32_t chunk = slice * 64u + lane_id;  // which 64-column stretch of the row
    const bool active = chunk < columns / kChunk;
    const typename T::Lane lane = T::lane_setup(active ? chunk : 0u);
    const uint64_t row_bytes = T::row_bytes(columns);

    const uint32_t wg_row0 = blockIdx.x * rows_per_wg;
    const uint32_t wg_row_end = min(wg_row0 + rows_per_wg, rows);
    const uint32_t iterations = LOOP ? (wg_row_end - wg_row0 + RG * R - 1) / (RG * R) : 1u;

    auto load_row = [&](uint32_t it, int r, typename T::Data& data) {
        uint32_t row = wg_row0 + (it * RG + group) * R + r;
        row = min(row, rows - 1);  // rows past the end re-read a valid row and are discarded
        T::load(weight + row * row_bytes, lane, data);
    };
    auto load_rows = [&](uint32_t it, typename T::Data (&data)[R]) {
#pragma unroll
        for (int r = 0; r < R; r++) load_row(it, r, data[r]);
    };

    // Order of the prologue. A wave that issues a load while the CU's memory
    // queue is full stalls, and so does everything behind the load in program
    // order; once the weights of a whole CU are requested the queue stays full
    // for microseconds. The activations, which the whole workgroup needs before
    // the first multiply, therefore go first: (1) activation loads, (2) ONE row
    // of weights, so that HBM has work during the activation round trip,
    // (3) split the activations as soon as they are back, (4) barrier, (5) only
    // then the rest of the rows, which may stall freely.
    typename T::Data current[R];
    load_row(0, 0, current[0]);
    __builtin_amdgcn_sched_barrier(0);

    // Activations: limbs in LDS -> registers, one 4096-column slice at a time.
    XLimbs xr[M];
    for (uint32_t s = 0; s < NK; s++) {
        if (s != 0) {
            __syncthreads();
            load_x(s, xv);
        }
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t f = threadIdx.x + i * THREADS;
                if (f < kSliceQuads) stage_quad(stage[m], xv[m][i], f);  // wave-uniform condition
            }
        __syncthreads();
        if (s == slice) {
#pragma unroll
            for (int m = 0; m < M; m++) T::load_activations(stage[m], lane_id, active, xr[m]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // Writes the outputs of iteration `it` from the per-row totals.
    auto write_rows = [&](uint32_t it, const float (&total)[R][M]) {
        const uint32_t row0 = wg_row0 + (it * RG + group) * R;
        if (NK == 1) {
            if (lane_id == 0) {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const uint32_t row = row0 + r;
                    if (row < wg_row_end) {
                        const float b = bias != nullptr ? bias[row] : 0.f;
#pragma unroll
                        for (int m = 0; m < M; m++)
                            y[static_cast<uint64_t>(m) * rows + row] =
                                bias != nullptr ? total[r][m] + b : total[r][m];
                    }
                }
            }
        } else {
            const uint32_t parity = it & 1u;
            if (lane_id == 0) {
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int m = 0; m < M; m++) partial[parity][group][slice][r][m] = total[r][m];
            }
            __syncthreads();
            if (slice == 0 && lane_id < R * M) {
                const uint32_t r = lane_id / M, m = lane_id - r * M;
                const uint32_t row = row0 + r;
                if (row < wg_row_end) {
                    float value = 0.f;
                    for (int s = 0; s < NK; s++) value += partial[parity][group][s][r][m];
                    if (bias != nullptr) value += bias[row];
                    y[static_cast<uint64_t>(m) * rows + row] = value;
                }
            }
        }
    };
    auto fold_row = [&](const typename T::Data& data, float (&total)[M]) {
        float value[M];
        T::template fold<M>(data, lane, xr, value);
#pragma unroll
        for (int m = 0; m < M; m++) total[m] = wave_sum(active ? value[m] : 0.f);
    };

    if (!LOOP) {
        // Request row r+1, then fold row r: a request that stalls on a full
        // queue stalls behind useful work, and rows are folded as they arrive.
        float total[R][M];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r + 1 < R) load_row(0, r + 1, current[r + 1]);
            __builtin_amdgcn_sched_barrier(0);
            fold_row(current[r], total[r]);
            __builtin_amdgcn_sched_barrier(0);
        }
        write_rows(0, total);
    } else {
        // Two R-row buffers in ping-pong. Row 0 of the first is already on its way.
        typename T::Data other[R];
#pragma unroll
        for (int r = 1; r < R; r++) load_row(0, r, current[r]);
        float total[R][M];
        for (uint32_t it = 0; it < iterations; it += 2) {
            if (it + 1 < iterations) load_rows(it + 1, other);
#pragma unroll
            for (int r = 0; r < R; r++) fold_row(current[r], total[r]);
            write_rows(it, total);
            if (it + 1 < iterations) {
                if (it + 2 < iterations) load_rows(it + 2, current);
#pragma unroll
                for (int r = 0; r < R; r++) fold_row(other[r], total[r]);
                write_rows(it + 1, total);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// The same GEMV with the weights brought in by global-to-LDS copies (one slice: columns <= 4096).
//
// What bounds gemv_limb_kernel is how many bytes a compute unit keeps in flight: a wave requests
// the next row only after it has folded the one before, because a wave that issues a load into a
// full memory queue stalls with all the arithmetic behind it. Here the two jobs are split between
// waves. The workgroup's share of W - a contiguous range of rows, at most 158 KiB - is cut into
// eight contiguous ranges, one per CONSUMER wave; consumer w's range is copied into LDS, as it lies
// in memory, by LOADER wave w with 1 KiB global_load_lds copies (no registers; a loader that stalls
// on a full queue holds nothing up), while the consumers prepare the activations and then fold
// their rows out of LDS as they land. A consumer issues no global load after its activation loads.
//
// Hand-over without barriers (s_barrier would tie the loaders to the consumers' prologue): a
// loader keeps DEPTH copies in flight; before it issues the next one it waits for the oldest
// (loads return in order per wave: one counted s_waitcnt) and publishes in LDS how many of its
// copies have landed; its consumer polls that one word until it covers the next row.
// This kernel serves the 2-bit codec, whose folds are long against its bytes: a loader has issued its
// few copies early and would idle, so once they have all landed it folds the last quarter of its range.
// The other codecs run on gemv_limb_turns_kernel below.
// The consumers meet each other through one LDS counter (`staged`).
// LDS: [the ranges, whole KiB each][...][StageMemory x M][control]; shapes whose ranges would reach
// into the stages stay on gemv_limb_kernel.
// ---------------------------------------------------------------------------
// ET_HIP_GEMV_LDS_COPIES=0 in the environment keeps every shape on gemv_limb_kernel (for A/B timing).
bool gemv_limb_dma_enabled() {
    static const bool enabled = [] {
        const char* value = std::getenv("ET_HIP_GEMV_LDS_COPIES");
        return value == nullptr || value[0] != '0';
    }();
    return enabled;
}

constexpr int kDmaPairs = 8;  // ranges of a share: one loader and one consumer wave each (a workgroup has at most
                              // sixteen waves)
constexpr int kDmaConsumers = kDmaPairs;
constexpr int kDmaDepth = 4;  // copies a loader keeps in flight: more only lengthen the queue, and a loader says that a
                              // copy has landed only when it may issue the copy DEPTH places later
constexpr int kDmaHead = kDmaDepth;  // copies a loader issues before it does anything else, at most eight
                                     // (wait_copies_in_flight). Six and eight measured slower when the 4-bit codec ran
                                     // on this kernel (14336 x 4096: 7.9 and 8.2 against 7.7 us).
constexpr uint32_t kDmaLateEighths = 2;  // share of a range that a loader which only copies folds at the end
constexpr int kDmaThreads = 64 * (kDmaConsumers + kDmaPairs);
constexpr int kTurnConsumers = 11, kTurnLoaders = 5, kTurnDepth = 6;  // gemv_limb_turns_kernel: waves that fold, waves that
                                                                      // copy, copies in flight per loader
static_assert(64 * (kTurnConsumers + kTurnLoaders) == kDmaThreads, "sixteen waves either way");
constexpr uint32_t kDmaLdsBytes = 160u * 1024u;
struct DmaControl {
    uint32_t landed[kDmaPairs];  // copies of loader w that have landed
    uint32_t staged;             // consumers that have written their part of the stages
    uint32_t pad[7];
};
constexpr uint32_t kDmaControlAt = kDmaLdsBytes - 1024u;
static_assert(sizeof(DmaControl) == 64, "sixteen words, zeroed by sixteen lanes");

template <class T, int M, int DEPTH>
__global__ __launch_bounds__(kDmaThreads) void gemv_limb_dma_kernel(
    const uint8_t* __restrict__ weight, const float* __restrict__ x, uint64_t x_row_stride,
    const float* __restrict__ bias, float* __restrict__ y, uint32_t rows, uint32_t columns,
    uint32_t rows_per_wg, uint32_t spin_limit, uint32_t* timeouts) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    Patience patience{spin_limit, timeouts};  // every wait on another wave is bounded (lds_handover.h)
    constexpr uint32_t kStageAt = kDmaControlAt - M * static_cast<uint32_t>(sizeof(StageMemory));
    constexpr int NI = kSliceQuads / (64 * kDmaConsumers);  // float4s per consumer thread and vector
    static_assert(DEPTH <= kDmaHead && kDmaHead <= 8, "the steady loop starts with DEPTH copies in flight; wait_copies_in_flight counts to seven");
    static_assert(!T::kCopiesInTurn, "the other codecs run on gemv_limb_turns_kernel");
    DmaControl* control = reinterpret_cast<DmaControl*>(lds + kDmaControlAt);
    StageMemory* stage = reinterpret_cast<StageMemory*>(lds + kStageAt);

    const uint32_t lane_id = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wg_row0 = blockIdx.x * rows_per_wg;
    if (wg_row0 >= rows) return;
    const uint32_t wg_rows = min(rows_per_wg, rows - wg_row0);
    const uint32_t row_bytes = static_cast<uint32_t>(T::row_bytes(columns));
    const bool consumer = wave < static_cast<uint32_t>(kDmaConsumers);
    // the range this wave works on: rows [first, first + count) of the share, `range_kib` KiB of LDS each
    const uint32_t pair = consumer ? wave : wave - kDmaConsumers;
    const uint32_t per_pair = (rows_per_wg + kDmaPairs - 1u) / kDmaPairs;
    const uint32_t first = min(pair * per_pair, wg_rows);
    const uint32_t count = min(per_pair, wg_rows - first);
    const uint32_t range_kib = (per_pair * row_bytes + 1023u) >> 10;
    uint8_t* range = lds + pair * (range_kib << 10);
    const uint32_t late = count * kDmaLateEighths / 8u;  // rows the loader folds after its last copy

    const uint32_t chunk = lane_id;  // one slice: the lane's 64-column stretch of the row
    const bool active = chunk < columns / kChunk;
    const typename T::Lane lane = T::lane_setup(active ? chunk : 0u);
    XLimbs xr[M];
    // Folds a row of the range that is in registers and stores the result. The loaders keep few copies
    // in flight, so a store finds room in the memory queue.
    const auto fold_row = [&](uint32_t r, const typename T::Data& data) {
        float value[M];
        T::template fold<M>(data, lane, xr, value);
        const uint32_t row = wg_row0 + first + r;
        const float b = bias != nullptr ? bias[row] : 0.f;
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float total = wave_sum(active ? value[m] : 0.f);
            if (lane_id == 0) y[static_cast<uint64_t>(m) * rows + row] = bias != nullptr ? total + b : total;
        }
    };

    float4 xv[M][NI];
    if (consumer) {
        // Activation loads go first in the consumers: nothing of theirs may queue behind a copy.
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t quad = threadIdx.x + i * 64u * kDmaConsumers;
                xv[m][i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (quad < (columns >> 2)) xv[m][i] = reinterpret_cast<const float4*>(x + m * x_row_stride)[quad];
            }
        if (threadIdx.x < 16) reinterpret_cast<uint32_t*>(control)[threadIdx.x] = 0u;
        __syncthreads();  // the only barrier: the counters are zero before anybody counts
    } else {
        // ---- loaders ------------------------------------------------------------------------
        const uint32_t bytes = count * row_bytes;
        const uint32_t copies = (bytes + 1023u) >> 10;
        const uint8_t* source = weight + (static_cast<uint64_t>(wg_row0) + first) * row_bytes;
        const uint32_t landed_address = lds_address(&control->landed[pair]);
        const auto copy = [&](uint32_t i) {
            const uint32_t at = i * 1024u + lane_id * 16u;
            if (at < bytes)  // the last copy of a range stops where the range ends
                // streamed once: non-temporal (aux bit 1), the caches keep nothing of it
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint4*>(source + at),
                                                 reinterpret_cast<uint4*>(range + i * 1024u), 16, 0, 2);
        };
        // The first copies wait for the barrier, i.e. until the consumers have issued their activation
        // loads: issued ahead of it they delay those loads, and with them every fold, by half a microsecond.
        __syncthreads();
        const uint32_t head = min(copies, static_cast<uint32_t>(kDmaHead));
        for (uint32_t i = 0; i < head; i++) copy(i);
        uint32_t landed = 0, in_flight = head;
        if (in_flight > static_cast<uint32_t>(DEPTH)) {  // down to the steady depth
            __builtin_amdgcn_s_waitcnt(vmcnt_only(DEPTH));
            landed = in_flight - DEPTH;
            in_flight = DEPTH;
            lds_store_unseen(landed_address, landed);
        }
        for (uint32_t i = head; i < copies; i++) {  // only with DEPTH copies in flight (head = kDmaHead < copies)
            // the oldest copy in flight has landed: say so, then take its place in the queue
            __builtin_amdgcn_s_waitcnt(vmcnt_only(DEPTH - 1));
            lds_store_unseen(landed_address, ++landed);
            copy(i);
        }
        for (uint32_t left = in_flight; left > 0u; left--) {
            wait_copies_in_flight(left - 1u);
            lds_store_unseen(landed_address, ++landed);
        }
        // nothing of this wave is in flight any more: ordinary LDS reads from here on
        if (late != 0u) {
            lds_await(lds_address(&control->staged), kDmaConsumers, patience);
#pragma unroll
            for (int m = 0; m < M; m++) T::load_activations(stage[m], lane_id, active, xr[m]);
            for (uint32_t r = count - late; r < count; r++) {
                typename T::Data data;
                T::load(range + r * row_bytes, lane, data);
                fold_row(r, data);
            }
        }
        return;
    }

    // ---- consumers ------------------------------------------------------------------------------
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int i = 0; i < NI; i++) stage_quad(stage[m], xv[m][i], threadIdx.x + i * 64u * kDmaConsumers);
    lds_arrive(lds_address(&control->staged), lane_id == 0);
    lds_await(lds_address(&control->staged), kDmaConsumers, patience);
#pragma unroll
    for (int m = 0; m < M; m++) T::load_activations(stage[m], lane_id, active, xr[m]);

    const uint32_t landed_address = lds_address(&control->landed[pair]);
    // Row r needs the copies that hold bytes [0, (r + 1) * row_bytes) of the range. (Reading row r + 1
    // out of LDS ahead of the fold of row r, when it has landed by then, measured slower: the consumers
    // are bound by their arithmetic, two of them and two loaders to a SIMD, not by LDS latency.)
    const uint32_t mine = count - late;  // the last rows are the loader's
    for (uint32_t r = 0; r < mine; r++) {
        lds_await(landed_address, ((r + 1u) * row_bytes + 1023u) >> 10, patience);
        typename T::Data data;
        T::load(range + r * row_bytes, lane, data);
        fold_row(r, data);
    }
}

// The same split of the work with the copies taken in turn (the 4-, 5- and 8-bit codecs): the
// workgroup's share of W is ONE image in LDS, exactly as it lies in memory, whose 1 KiB copies the
// loaders take in turn (copy i is loader i % LOADERS's), so the image lands front to back at the rate of
// all loaders together. Rows are not tied to waves: a consumer that is free takes the next row from a
// counter in LDS, waits until the row's last byte has landed (one poll reads all the loaders' words) and
// folds it. The loaders do nothing but copy: a launch whose loaders read the staged activations while
// their first copies are on the way, to fold a row each at the end, measured half a microsecond slower
// than one whose loaders only copy - and such a launch, with its consumers switched off, runs as fast
// as the same copies alone (Q4_K 14336 x 4096: 6.2 - 6.6 us). What the launch waits for is its folds:
// they start when the activations are in registers (1.3 us after the barrier) and then keep the vector
// ALU busy for about 70 % of the time, so eleven of the sixteen waves fold and five copy, six copies in
// flight each (8 + 8 x 4: 8.2 - 8.4 us, 11 + 5 x 6: 7.9 - 8.1 on the same box; Q4_0 11008 x 4096: 7.1 -> 6.5).
template <class T, int M, int CONSUMERS, int LOADERS, int DEPTH>
__global__ __launch_bounds__(64 * (CONSUMERS + LOADERS)) void gemv_limb_turns_kernel(
    const uint8_t* __restrict__ weight, const float* __restrict__ x, uint64_t x_row_stride,
    const float* __restrict__ bias, float* __restrict__ y, uint32_t rows, uint32_t columns,
    uint32_t rows_per_wg, uint32_t spin_limit, uint32_t* timeouts) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr uint32_t kStageAt = kDmaControlAt - M * static_cast<uint32_t>(sizeof(StageMemory));
    constexpr int kStagers = 8;                            // consumer waves that prepare the activations
    constexpr int NI = kSliceQuads / (64 * kStagers);      // float4s per such thread and vector
    static_assert(DEPTH >= 1 && DEPTH <= 8, "wait_copies_in_flight counts to seven");
    static_assert(CONSUMERS >= kStagers && LOADERS <= kDmaPairs, "eight waves stage; DmaControl has eight loader words");
    DmaControl* control = reinterpret_cast<DmaControl*>(lds + kDmaControlAt);
    StageMemory* stage = reinterpret_cast<StageMemory*>(lds + kStageAt);
    Patience patience{spin_limit, timeouts};  // every wait on another wave is bounded (lds_handover.h)

    const uint32_t lane_id = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wg_row0 = blockIdx.x * rows_per_wg;
    if (wg_row0 >= rows) return;
    const uint32_t wg_rows = min(rows_per_wg, rows - wg_row0);
    const uint32_t row_bytes = static_cast<uint32_t>(T::row_bytes(columns));
    const uint32_t bytes = wg_rows * row_bytes;
    const uint32_t chunk = lane_id;  // one slice: the lane's 64-column stretch of the row
    const bool active = chunk < columns / kChunk;
    const uint32_t staged_address = lds_address(&control->staged);
    const uint32_t next_row_address = lds_address(&control->pad[0]);

    if (wave >= static_cast<uint32_t>(CONSUMERS)) {
        // ---- loaders ------------------------------------------------------------------------
        const uint32_t loader = wave - CONSUMERS;
        const uint32_t copies = (bytes + 1023u) >> 10;
        const uint32_t mine = copies > loader ? (copies - loader + LOADERS - 1u) / LOADERS : 0u;
        const uint8_t* source = weight + static_cast<uint64_t>(wg_row0) * row_bytes + lane_id * 16u;
        const uint32_t landed_address = lds_address(&control->landed[loader]);
        uint32_t at = loader * 1024u;  // of this loader's next copy in the image
        const auto copy = [&]() {
            if (at + lane_id * 16u < bytes)  // the last copy of the image stops where the share ends
                // streamed once: non-temporal (aux bit 1), the caches keep nothing of it
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint4*>(source + at),
                                                 reinterpret_cast<uint4*>(lds + at), 16, 0, 2);
            at += LOADERS * 1024u;
        };
        // The first copies wait for the barrier, i.e. until the consumers have issued their activation
        // loads: issued ahead of it they delay those loads, and with them every fold.
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

    // ---- consumers ------------------------------------------------------------------------------
    {
        // Activation loads go first: nothing of the consumers' may queue behind a copy.
        float4 xv[M][NI];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const uint32_t quad = threadIdx.x + i * 64u * kStagers;
                xv[m][i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (wave < kStagers && quad < (columns >> 2))
                    xv[m][i] = reinterpret_cast<const float4*>(x + m * x_row_stride)[quad];
            }
        if (threadIdx.x < 16) reinterpret_cast<uint32_t*>(control)[threadIdx.x] = 0u;
        __syncthreads();  // the only barrier: the counters are zero before anybody counts
        if (wave < kStagers) {
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int i = 0; i < NI; i++) stage_quad(stage[m], xv[m][i], threadIdx.x + i * 64u * kStagers);
            lds_arrive(staged_address, lane_id == 0);
        }
        if (!lds_await(staged_address, kStagers, patience)) return;
    }

    // ---- take a row, wait for it, fold it -------------------------------------------------------
    const typename T::Lane lane = T::lane_setup(active ? chunk : 0u);
    XLimbs xr[M];
#pragma unroll
    for (int m = 0; m < M; m++) T::load_activations(stage[m], lane_id, active, xr[m]);
    for (;;) {
        const uint32_t r = lds_take(next_row_address, lane_id == 0);
        if (r >= wg_rows) break;
        if (!await_copies_in_turn<LOADERS>(control->landed, lane_id, ((r + 1u) * row_bytes + 1023u) >> 10, patience)) break;
        typename T::Data data;
        T::load(lds + r * row_bytes, lane, data);
        float value[M];
        T::template fold<M>(data, lane, xr, value);
        const uint32_t row = wg_row0 + r;
        const float b = bias != nullptr ? bias[row] : 0.f;
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float total = wave_sum(active ? value[m] : 0.f);
            if (lane_id == 0) y[static_cast<uint64_t>(m) * rows + row] = bias != nullptr ? total + b : total;
        }
    }
}

// Whether gemv_limb_dma_kernel takes this shape: one slice of columns, a share per compute unit that
// fits LDS below the activation stages, enough rows per share to occupy the consumers.
template <class T, int M>
bool dma_takes(uint32_t rows, uint32_t columns, uint32_t* rows_per_wg) {
    if (columns > kSliceColumns) return false;
    const uint32_t share = (rows + 255u) / 256u;
    // With fewer than four rows to a range gemv_limb_kernel, which has all of them in flight from its
    // first instructions, is the faster one (Q8_0 4096 x 4096, two rows to a range: 5.1 against 5.5 us).
    if (share < 4u * kDmaPairs) return false;
    const uint64_t row_bytes = (static_cast<uint64_t>(columns) / T::kBlockColumns) * T::kBlockBytes;
    // A loader lane copies 16 bytes: rows that are not whole 16-byte pieces (Q2_K unless columns % 1024 == 0,
    // Q4_0 / Q8_0 unless columns % 256 == 0) would let the last lane of a range read up to 12 bytes past it -
    // for the last range of the matrix, past the weight buffer. Those widths stay on gemv_limb_kernel,
    // which reads exact dwords.
    if (row_bytes % 16u != 0u) return false;
    const uint64_t per_pair = (share + kDmaPairs - 1u) / kDmaPairs;
    const uint64_t range_bytes = ((per_pair * row_bytes + 1023u) / 1024u) * 1024u;  // as laid out in LDS
    const uint64_t stage_at = kDmaControlAt - M * sizeof(StageMemory);
    if (range_bytes * kDmaPairs > stage_at) return false;
    *rows_per_wg = share;
    return true;
}

template <class T, int M>
hipError_t launch_dma(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias,
                      float* y, uint32_t rows, uint32_t columns, uint32_t rows_per_wg, hipStream_t stream) {
    static std::atomic<bool> allowed[64];
    int device = 0;
    if (hipError_t status = hipGetDevice(&device)) return status;
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    HandoverState handover;
    if (hipError_t status = handover_state(&handover)) return status;
    const uint32_t grid = (rows + rows_per_wg - 1) / rows_per_wg;
    const auto go = [&](auto kernel, uint32_t threads) -> hipError_t {
        if (!allowed[device].load(std::memory_order_acquire)) {
            if (hipError_t status = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, kDmaLdsBytes))
                return status;
            allowed[device].store(true, std::memory_order_release);
        }
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), kDmaLdsBytes, stream, weight, x, x_row_stride, bias, y,
                           rows, columns, rows_per_wg, handover.limit, handover.timeouts);
        return hipGetLastError();
    };
    if constexpr (T::kCopiesInTurn)
        return go(gemv_limb_turns_kernel<T, M, kTurnConsumers, kTurnLoaders, kTurnDepth>, kDmaThreads);
    else
        return go(gemv_limb_dma_kernel<T, M, kDmaDepth>, kDmaThreads);
}

template <class T, int M, int R, int WAVES, int NK, bool LOOP>
hipError_t launch(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias,
                  float* y, uint32_t rows, uint32_t columns, uint32_t rows_per_wg, hipStream_t stream) {
    const uint32_t grid = (rows + rows_per_wg - 1) / rows_per_wg;
    hipLaunchKernelGGL((gemv_limb_kernel<T, M, R, WAVES, NK, LOOP>), dim3(grid), dim3(64 * WAVES), 0,
                       stream, weight, x, x_row_stride, bias, y, rows, columns, rows_per_wg);
    return hipGetLastError();
}

// Picks rows per workgroup and the single-shot depth for WAVES / NK row groups.
template <class T, int M, int WAVES, int NK>
hipError_t launch_rows(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias,
                       float* y, uint32_t rows, uint32_t columns, hipStream_t stream) {
    constexpr uint32_t RG = WAVES / NK;
    // One contiguous range of rows per CU; a wave takes ceil(range / RG) of them.
    const uint32_t share = (rows + 255u) / 256u;
    const uint32_t depth = (share + RG - 1) / RG;
    // Registers bound the single-shot depth: 4 rows with more than 8 waves (128 VGPRs), else 8.
    constexpr uint32_t kMaxDepth = (WAVES > 8 || M > 1) ? 4 : 8;
#define ET_SHOT(D)                                                                               \
    case D:                                                                                      \
        return launch<T, M, D, WAVES, NK, false>(weight, x, x_row_stride, bias, y, rows, columns, \
                                                 RG * D, stream)
    if (depth <= kMaxDepth) {
        switch (depth) {
            ET_SHOT(1);
            ET_SHOT(2);
            ET_SHOT(3);
            ET_SHOT(4);
            default: break;
        }
        if (kMaxDepth == 8) {
            switch (depth) {
                case 5: return launch<T, M, (kMaxDepth == 8 ? 5 : 1), WAVES, NK, false>(weight, x, x_row_stride, bias, y, rows, columns, RG * 5, stream);
                case 6: return launch<T, M, (kMaxDepth == 8 ? 6 : 1), WAVES, NK, false>(weight, x, x_row_stride, bias, y, rows, columns, RG * 6, stream);
                case 7: return launch<T, M, (kMaxDepth == 8 ? 7 : 1), WAVES, NK, false>(weight, x, x_row_stride, bias, y, rows, columns, RG * 7, stream);
                case 8: return launch<T, M, (kMaxDepth == 8 ? 8 : 1), WAVES, NK, false>(weight, x, x_row_stride, bias, y, rows, columns, RG * 8, stream);
                default: break;
            }
        }
    }
#undef ET_SHOT
    // Too many rows per wave for registers: loop with two 2-row buffers.
    const uint32_t rows_per_wg = ((share + RG * 2 - 1) / (RG * 2)) * (RG * 2);
    return launch<T, M, 2, WAVES, NK, true>(weight, x, x_row_stride, bias, y, rows, columns,
                                            rows_per_wg, stream);
}

template <class T, int M>
hipError_t launch_slices(const uint8_t* weight, const float* x, uint64_t x_row_stride,
                         const float* bias, float* y, uint32_t rows, uint32_t columns,
                         hipStream_t stream) {
    const uint32_t slices = (columns + kSliceColumns - 1) / kSliceColumns;
    if constexpr (T::kLdsCopies && M == 1) {  // more vectors need more registers than sixteen waves leave
        uint32_t rows_per_wg = 0;
        if (gemv_limb_dma_enabled() && dma_takes<T, M>(rows, columns, &rows_per_wg))
            return launch_dma<T, M>(weight, x, x_row_stride, bias, y, rows, columns, rows_per_wg, stream);
    }
    if (slices <= 1) {
        return launch_rows<T, M, 8, 1>(weight, x, x_row_stride, bias, y, rows, columns, stream);
    }
    if (slices <= 2) return launch_rows<T, M, 8, 2>(weight, x, x_row_stride, bias, y, rows, columns, stream);
    if (slices <= 4) return launch_rows<T, M, 8, 4>(weight, x, x_row_stride, bias, y, rows, columns, stream);
    if (slices <= 8) return launch_rows<T, M, 8, 8>(weight, x, x_row_stride, bias, y, rows, columns, stream);
    return launch_rows<T, M, 16, 16>(weight, x, x_row_stride, bias, y, rows, columns, stream);
}

template <class T>
hipError_t launch_vectors(const uint8_t* weight, const float* x, uint64_t x_row_stride,
                          const float* bias, float* y, uint32_t rows, uint32_t columns,
                          uint32_t vectors, hipStream_t stream) {
    switch (vectors) {
        case 1: return launch_slices<T, 1>(weight, x, x_row_stride, bias, y, rows, columns, stream);
        case 2: return launch_slices<T, 2>(weight, x, x_row_stride, bias, y, rows, columns, stream);
        case 3: return launch_slices<T, 3>(weight, x, x_row_stride, bias, y, rows, columns, stream);
        default: return hipErrorInvalidValue;
    }
}

// One or two vectors per launch (the codecs whose lanes own four runs).
template <class T>
hipError_t launch_pair(const uint8_t* weight, const float* x, uint64_t x_row_stride, const float* bias, float* y,
                       uint32_t rows, uint32_t columns, uint32_t vectors, hipStream_t stream) {
    if (vectors == 1) return launch_slices<T, 1>(weight, x, x_row_stride, bias, y, rows, columns, stream);
    if (vectors == 2) return launch_slices<T, 2>(weight, x, x_row_stride, bias, y, rows, columns, stream);
    return hipErrorInvalidValue;
}

}  // namespace

uint32_t gemv_limb_max_vectors(int32_t codec) {
    // Q2_K, Q3_K and Q6_K keep 62 and more registers of activation state per vector (48 limb words,
    // 12 dot offsets, 2 units, run sums): three vectors do not fit next to the rows in flight.
    return codec == kQ6_K || codec == kQ3_K || codec == kQ2_K ? 2u : kGemvLimbMaxVectors;
}

bool gemv_limb_copies_through_lds(int32_t codec, uint64_t rows, uint64_t columns, uint32_t vectors) {
    if (vectors != 1 || rows > 0xffffffffull || columns > kSliceColumns || !gemv_limb_dma_enabled()) return false;
    const uint32_t n = static_cast<uint32_t>(rows), k = static_cast<uint32_t>(columns);
    uint32_t rows_per_wg = 0;
    switch (codec) {
        case kQ4_K: return dma_takes<Q4KLimb, 1>(n, k, &rows_per_wg);
        case kQ5_K: return dma_takes<Q5KLimb, 1>(n, k, &rows_per_wg);
        case kQ4_0: return dma_takes<Q40Limb, 1>(n, k, &rows_per_wg);
        case kQ8_0: return dma_takes<Q80Limb, 1>(n, k, &rows_per_wg);
        case kQ2_K: return dma_takes<Q2KLimb, 1>(n, k, &rows_per_wg);
        default: return false;
    }
}

bool gemv_limb_supported(int32_t codec, uint64_t columns, uint32_t vectors) {
    if (vectors == 0 || vectors > gemv_limb_max_vectors(codec) || columns == 0 || columns > 65536u) return false;
    if (codec == kQ2_K || codec == kQ3_K || codec == kQ4_K || codec == kQ5_K || codec == kQ6_K) return columns % 256 == 0;
    if (codec == kQ4_0 || codec == kQ8_0) return columns % 64 == 0;
    return false;
}

hipError_t gemv_limb(int32_t codec, const uint8_t* weight, const float* x, uint64_t x_row_stride,
                     const float* bias, float* y, uint64_t rows, uint64_t columns, uint32_t vectors,
                     hipStream_t stream) {
    const uint32_t n = static_cast<uint32_t>(rows), k = static_cast<uint32_t>(columns);
    switch (codec) {
        case kQ4_K: return launch_vectors<Q4KLimb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        case kQ5_K: return launch_vectors<Q5KLimb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        case kQ6_K: return launch_pair<Q6KLimb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        case kQ3_K: return launch_pair<Q3KLimb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        case kQ2_K: return launch_pair<Q2KLimb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        case kQ4_0: return launch_vectors<Q40Limb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        case kQ8_0: return launch_vectors<Q80Limb>(weight, x, x_row_stride, bias, y, n, k, vectors, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace et
