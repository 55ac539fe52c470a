// Bit-exact dequantisation of packed GGUF rows on gfx950.
//
// out[p, :] = decode(W[index[p], :]) with every f32 operation rounded exactly
// as the reference's scalar decoders do (crates/runtime-cpu/src/quantized.rs:
// decode_q2_k :117-138, decode_q3_k :142-176, decode_q4_k :180-199,
// decode_q5_k :203-234, decode_q6_k :238-261): `d * scale`, `dmin * min`, then
// `dl * q` and `- ml` as separate multiply and subtract. This translation unit
// is compiled with -ffp-contract=off and carries the pragma below so that no
// multiply-subtract pair is ever fused into an FMA.
//
// The kernel is store-bound (4 output bytes per 0.56-1.06 input bytes), so the
// work split is chosen for the stores: one lane produces four consecutive
// output floats and writes them with a single 16-byte store, which makes every
// wave write 1 KiB of contiguous output. Packed bytes are read through the
// vector L1, where the eight lanes that share a 32-value group hit the same line.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "et_codecs.h"
#include "kernels.h"

#pragma clang fp contract(off)

#include "decode_device.h"

namespace et {
namespace {

// crates/runtime-cpu/src/tensor.rs:940-953, for the index tensor.
__device__ __forceinline__ uint64_t source_index(const IndexLayout& layout, uint64_t logical) {
    if (layout.contiguous) return layout.offset + logical;
    uint64_t source = layout.offset;
    uint64_t remainder = logical;
    for (int d = layout.rank - 1; d >= 0; d--) {
        const uint64_t width = layout.shape[d] > 1 ? layout.shape[d] : 1;
        source += (remainder % width) * layout.strides[d];
        remainder /= width;
    }
    return source;
}

constexpr uint64_t kNoBadIndex = ~0ull;
template <int CODEC>
constexpr uint32_t kSpansPerThread = 4 / Span<CODEC>::kGroups;  // sixteen values

// The value of an index as 64 bits, and whether the table has such a row.
__device__ __forceinline__ uint64_t index_value(const void* indexes, int index_is_i64, uint64_t source, uint64_t table_rows, bool& bad) {
    if (index_is_i64) {
        const long long value = static_cast<const long long*>(indexes)[source];
        bad = value < 0 || static_cast<uint64_t>(value) >= table_rows;
        return static_cast<uint64_t>(value);
    }
    const uint64_t value = static_cast<const uint32_t*>(indexes)[source];
    bad = value >= table_rows;
    return value;
}

// The status block is the lowest position of a bad index and its VALUE, so the host can word the error like
// crates/runtime-cpu/src/quantized.rs:570-583; or kNoBadIndex and 0. Two ways to write it:
//
// Few indexes (lookup_checks_itself): an extra workgroup of the lookup's own launch checks all of them and writes the
// block while the others decode.
// Many, or strided: the block is cleared first, the workgroups that decode check their own index, and a third launch
// adds the value.
constexpr uint32_t kChecksInFlight = 16;                        // loads in flight per thread of the checking workgroup
constexpr uint64_t kMostSelfChecked = 2 * 256u * kChecksInFlight;  // indexes it takes in two rounds

// Two launches less (contiguous ids in a captured graph, three launches / one in us: one id of 4096 Q4_K columns 6.9 / 4.8,
// 1000 ids 10.6 / 7.7, 4096 ids 22.1 / 20.1; 4096 ids of 32 Q8_0 columns 8.2 / 5.7, 8192 ids 10.0 / 7.0). One workgroup takes
// more than 4096 ids in rounds, each a memory latency: the second is hidden also by the narrowest rows, further ones are not
// (100 000 ids of 256 columns took 73 in three launches and 97 in one), and strided ids cost each of its threads sixteen
// times a division per dimension (1000 ids 7.1 / 11.4).
bool lookup_checks_itself(const IndexLayout& layout, uint64_t count) { return layout.contiguous && count <= kMostSelfChecked; }

__device__ void report_bad_index(const void* indexes, int index_is_i64, uint64_t offset, uint32_t count, uint64_t table_rows,
                                 unsigned long long* status) {
    __shared__ unsigned long long lowest[256];
    unsigned long long position = kNoBadIndex;
    for (uint32_t first = threadIdx.x; first < count && position == kNoBadIndex; first += 256u * kChecksInFlight) {
        bool bad[kChecksInFlight];
#pragma unroll
        for (uint32_t i = 0; i < kChecksInFlight; i++) {
            const uint32_t p = first + 256u * i;
            index_value(indexes, index_is_i64, offset + (p < count ? p : 0u), table_rows, bad[i]);
        }
#pragma unroll
        for (int i = kChecksInFlight - 1; i >= 0; i--)
            if (bad[i] && first + 256u * i < count) position = first + 256u * i;
    }
    lowest[threadIdx.x] = position;
    __syncthreads();
    for (uint32_t step = 128; step > 0; step >>= 1) {
        if (threadIdx.x < step && lowest[threadIdx.x + step] < lowest[threadIdx.x]) lowest[threadIdx.x] = lowest[threadIdx.x + step];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        bool ignored;
        status[0] = lowest[0];
        status[1] = lowest[0] == kNoBadIndex ? 0ull : index_value(indexes, index_is_i64, offset + lowest[0], table_rows, ignored);
    }
}

__global__ void status_init_kernel(unsigned long long* status) {
    if (threadIdx.x == 0) {
        status[0] = kNoBadIndex;
        status[1] = 0;
    }
}

__global__ void status_finalize_kernel(const void* indexes, int index_is_i64, IndexLayout layout, uint64_t table_rows,
                                       unsigned long long* status) {
    if (threadIdx.x != 0 || status[0] == kNoBadIndex) return;
    bool ignored;
    status[1] = index_value(indexes, index_is_i64, source_index(layout, status[0]), table_rows, ignored);
}

// Q4_0: the two runs of a lane lie in the two halves of a block's 128-byte line. The lanes of two blocks swap runs, lane i
// with lane i ^ 4, so that a store of eight lanes fills a line, in order. In a graph, inputs from memory, half / whole lines (us):
// 5000 ids of 4096 columns 22.3 / 21.0, 20 000 94.4 / 82.4, 9000 of 11008 columns 119.5 / 103.1.
__device__ __forceinline__ void store_two_blocks(float* blocks, uint32_t lane, const float (&values)[2][4]) {
    const bool second = lane >= 4;
    float first_block[4], second_block[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int given = __float_as_int(second ? values[0][i] : values[1][i]);
        int got = __builtin_amdgcn_update_dpp(given, given, 0x104, 0xF, 0x5, false);  // row_shl:4 in lanes 0..3 of eight,
        got = __builtin_amdgcn_update_dpp(got, given, 0x114, 0xF, 0xA, false);        // row_shr:4 in the others
        first_block[i] = second ? __int_as_float(got) : values[0][i];
        second_block[i] = second ? values[1][i] : __int_as_float(got);
    }
    float* to = blocks + 4u * lane;
    *reinterpret_cast<float4*>(to) = make_float4(first_block[0], first_block[1], first_block[2], first_block[3]);
    *reinterpret_cast<float4*>(to + 32) = make_float4(second_block[0], second_block[1], second_block[2], second_block[3]);
}

// A workgroup decodes one output row, or sixteen values per thread of a wider one, or (SHORT_ROWS) as many rows as its
// threads hold. The row's index is read once, and its address held, by the workgroup or by each thread of a short row (per thread
// for all rows: 20 000 ids of 4096 columns, inputs from memory, Q8_0 101.5 us for 98.2, Q4_K 86.5 for 80.1); everything else is
// 32-bit arithmetic. A thread takes spans (decode_device.h) of sixteen values in all and decodes them before its first
// store, so that their loads are in flight together; the stores of a wave are whole 128-byte lines (of short Q4_0 rows:
// halves). CHECKER: workgroup (0, 0) checks all the indexes.
//
// Bound: stores (4 bytes out per 0.3 to 1.1 in) now that the loads are few. With a load per header field and dword of
// quants (24 a thread for Q4_K) the address path of a compute unit alone took half the time. In a graph, before / after (us):
// 5000 ids of 4096 columns Q4_K 24.3 / 17.3 (5.4 TB/s), Q5_K 24.9 / 17.9, Q3_K 23.8 / 17.1, Q2_K 19.7 / 17.2, Q6_K 21.3 / 18.8, Q8_0
// 21.2 / 18.5, Q4_0 20.3 / 17.4; inputs and outputs from memory Q4_K 33.6 / 21.3, Q6_K 29.7 / 23.0, Q8_0 28.2 / 25.8; 20 000 Q4_K
// 124 / 80; rows that left threads idle: 100 000 ids of 256 columns 73 / 25.
template <int CODEC, bool CHECKER, bool SHORT_ROWS>
__global__ __launch_bounds__(256) void dequant_rows_kernel(
    const uint8_t* __restrict__ weight, const void* __restrict__ indexes, int index_is_i64,
    IndexLayout layout, uint64_t out_rows, uint64_t table_rows, uint32_t columns, uint32_t rows_per_wg,
    uint64_t row_bytes, float* __restrict__ out, unsigned long long* status) {
    using S = Span<CODEC>;
    constexpr uint32_t kBytes = block_bytes(CODEC);
    constexpr uint32_t kSpans = kSpansPerThread<CODEC>;
    constexpr uint32_t kCheckers = CHECKER ? 1u : 0u;
    if (blockIdx.x < kCheckers) {
        if (blockIdx.y == 0) report_bad_index(indexes, index_is_i64, layout.offset, static_cast<uint32_t>(out_rows), table_rows, status);
        return;
    }
    const uint32_t spans = columns / (4 * S::kGroups);  // of a row
    const uint32_t my_rows = SHORT_ROWS ? rows_per_wg : 1u;
    const uint32_t sub_row = SHORT_ROWS ? threadIdx.x / spans : 0u;
    const uint32_t thread = threadIdx.x - sub_row * spans;  // among those of its row
    if (sub_row >= my_rows) return;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x - kCheckers) * my_rows;
    for (uint64_t p = static_cast<uint64_t>(blockIdx.x - kCheckers) * my_rows + sub_row; p < out_rows; p += stride) {
        uint64_t row = p;
        if (indexes != nullptr) {
            bool bad;
            row = index_value(indexes, index_is_i64, source_index(layout, p), table_rows, bad);
            if (bad) {  // skipped, like the reference's Metal kernel
                if (!CHECKER && blockIdx.y == 0 && thread == 0) atomicMin(status, static_cast<unsigned long long>(p));
                continue;
            }
        }
        const uint8_t* packed_row = weight + row * row_bytes;
        float* out_row = out + p * columns;
        for (uint32_t at = blockIdx.y * (256u * kSpans); at < spans; at += gridDim.y * (256u * kSpans)) {
            float values[kSpans][S::kGroups][4];
#pragma unroll
            for (uint32_t u = 0; u < kSpans; u++) {
                const uint32_t span = at + 256u * u + thread;
                if (span < spans) S::decode(packed_row + static_cast<uint64_t>(span / S::kLanes) * kBytes, span % S::kLanes, values[u]);
            }
#pragma unroll
            for (uint32_t u = 0; u < kSpans; u++) {
                const uint32_t span = at + 256u * u + thread;
                if (span >= spans) continue;
                float* to = out_row + span / S::kLanes * block_values(CODEC) + S::first(span % S::kLanes);
                if constexpr (CODEC == kQ4_0 && !SHORT_ROWS) {
                    if ((span | 7u) < spans) {  // both blocks of these eight lanes are there
                        store_two_blocks(out_row + (span >> 3) * 64u, span & 7u, values[u]);
                        continue;
                    }
                }
#pragma unroll
                for (int g = 0; g < S::kGroups; g++)
                    *reinterpret_cast<float4*>(to + g * S::kStride) =
                        make_float4(values[u][g][0], values[u][g][1], values[u][g][2], values[u][g][3]);
            }
        }
    }
}

template <int CODEC, bool SHORT_ROWS>
hipError_t launch_rows(const uint8_t* weight, const void* indexes, int index_is_i64,
                       const IndexLayout& layout, uint64_t out_rows, uint64_t table_rows,
                       uint64_t columns, float* out, void* status, hipStream_t stream) {
    const uint64_t row_bytes = columns / block_values(CODEC) * block_bytes(CODEC);
    // The loops in the kernel take what the grid limits leave over.
    const uint64_t spans = columns / (4 * Span<CODEC>::kGroups);
    const uint32_t rows_per_wg = SHORT_ROWS ? static_cast<uint32_t>(256 / spans) : 1u;
    const uint64_t parts = (spans + 256 * kSpansPerThread<CODEC> - 1) / (256 * kSpansPerThread<CODEC>);
    const uint64_t groups = (out_rows + rows_per_wg - 1) / rows_per_wg;
    const uint32_t grid_x = static_cast<uint32_t>(groups < (1u << 24) ? groups : (1u << 24));
    const uint32_t grid_y = static_cast<uint32_t>(parts < 1024 ? parts : 1024);
    auto* status_words = static_cast<unsigned long long*>(status);
    if (indexes != nullptr && lookup_checks_itself(layout, out_rows)) {
        hipLaunchKernelGGL((dequant_rows_kernel<CODEC, true, SHORT_ROWS>), dim3(grid_x + 1, grid_y), dim3(256), 0,
                           stream, weight, indexes, index_is_i64, layout, out_rows, table_rows,
                           static_cast<uint32_t>(columns), rows_per_wg, row_bytes, out, status_words);
        return hipGetLastError();
    }
    if (indexes != nullptr) {
        hipLaunchKernelGGL(status_init_kernel, dim3(1), dim3(64), 0, stream, status_words);
    }
    hipLaunchKernelGGL((dequant_rows_kernel<CODEC, false, SHORT_ROWS>), dim3(grid_x, grid_y), dim3(256), 0,
                       stream, weight, indexes, index_is_i64, layout, out_rows, table_rows,
                       static_cast<uint32_t>(columns), rows_per_wg, row_bytes, out, status_words);
    if (indexes != nullptr) {
        hipLaunchKernelGGL(status_finalize_kernel, dim3(1), dim3(64), 0, stream, indexes,
                           index_is_i64, layout, table_rows, status_words);
    }
    return hipGetLastError();
}

template <int CODEC>
hipError_t launch_dequant(const uint8_t* weight, const void* indexes, int index_is_i64,
                          const IndexLayout& layout, uint64_t out_rows, uint64_t table_rows,
                          uint64_t columns, float* out, void* status, hipStream_t stream) {
    if (out_rows == 0 || columns == 0) return hipSuccess;
    const bool short_rows = columns / (4 * Span<CODEC>::kGroups) <= 128;  // a workgroup holds two or more
    return (short_rows ? launch_rows<CODEC, true> : launch_rows<CODEC, false>)(
        weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
}

}  // namespace

hipError_t dequantize_rows(int32_t codec, const uint8_t* weight, const void* indexes,
                           int index_is_i64, const IndexLayout& layout, uint64_t out_rows,
                           uint64_t table_rows, uint64_t columns, float* out, void* status,
                           hipStream_t stream) {
    switch (codec) {
        case kQ4_0: return launch_dequant<kQ4_0>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        case kQ8_0: return launch_dequant<kQ8_0>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        case kQ2_K: return launch_dequant<kQ2_K>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        case kQ3_K: return launch_dequant<kQ3_K>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        case kQ4_K: return launch_dequant<kQ4_K>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        case kQ5_K: return launch_dequant<kQ5_K>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        case kQ6_K: return launch_dequant<kQ6_K>(weight, indexes, index_is_i64, layout, out_rows, table_rows, columns, out, status, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace et
