// The NF4 quantizer on the device: pack_nf4 and double_quantize_scales of the
// reference (src/core/quantization/quantized_weight.cpp:176-206 and :208-254,
// nearest_nf4_code src/core/quantization/nf4.cpp:55-68, under /root/reference),
// bit for bit.
//
//   block scale   s_b = max |w| over the block (fp32; max is order-free)
//   code          7 for a zero block, else the codebook entry nearest to w / s_b
//                 -- the reference's linear scan with a strict '<', so the
//                 lowest index wins a tie; the division is correctly rounded
//   packing       even flat index in the low nibble, an unused high nibble of
//                 the last byte stays zero
//   double quantisation of the scales
//                 offset = (float)(sum of the scales in double, in index
//                 order, / count);  per group of C scales t = max |s - offset|,
//                 code = 128 + clamp(round-half-away(127 (s - offset) / t)),
//                 every operation rounded on its own
//
// The one step whose result depends on evaluation order is the double sum.
// It is evaluated in parallel only where that provably cannot matter: the
// scales are non-negative fp32 values, all of them multiples of u, the
// smallest unit in the last place among the non-zero ones, so every partial
// sum below 2^53 u is exact in double.  A sum that comes out below 2^53 u had
// no partial sum that reached it (sums of non-negative values do not shrink,
// and 2^53 u itself is representable), so every order gives it.  Otherwise one
// thread adds the scales in index order, as the reference does.
//
// What bounds it: memory; the weight is read once, its scales stay in
// registers between the maximum and the codes, and the sum of the scales is
// taken on the way.  11008 x 4096, block 64, nested: 37 us for the pass over
// the weight (5.5 TB/s) and 9 us for the scales, 79 us for the whole call with
// its wait.  A pass for the scales (70 us), one for the codes by sixteen
// distances each (94 us) and one workgroup for the mean (229 us) took 435 us.

#include "kernels.hpp"
#include "nf4_decode.hpp"

#include <bit>
#include <cfloat>
#include <climits>

namespace rthip {
namespace {

// Bits of the status word the kernels report through.
constexpr unsigned kNonFiniteSource = 1U;
constexpr unsigned kOffsetOverflow = 2U;
constexpr unsigned kInfinityBits = 0x7F800000U;

// The linear scan's result only grows with the normalised value: between two
// neighbouring entries the rounded distance to the lower one does not shrink
// and that to the upper one does not grow.  kThresholds[i] is the smallest
// value at which the scan prefers entry i + 1 to entry i.
struct Thresholds {
    float at[15];
};
consteval Thresholds find_thresholds() {
    // floats in ascending order as integers, and back
    const auto order = [](float value) {
        const int bits = std::bit_cast<int>(value);
        return bits < 0 ? INT_MIN - bits : bits;
    };
    const auto value_of = [](int place) {
        return std::bit_cast<float>(place < 0 ? INT_MIN - place : place);
    };
    Thresholds out{};
    for (int i = 0; i < 15; ++i) {
        const float lower = kNf4Codebook[i];
        const float upper = kNf4Codebook[i + 1];
        int below = order(lower);  // prefers i
        int above = order(upper);  // prefers i + 1
        while (above - below > 1) {
            const int middle = below + (above - below) / 2;
            const float value = value_of(middle);
            if (upper - value < value - lower) {
                above = middle;
            } else {
                below = middle;
            }
        }
        out.at[i] = value_of(above);
    }
    return out;
}
constexpr Thresholds kThresholds = find_thresholds();

// [-1, 1] in 31 intervals, narrower than the distance between two thresholds
// (0.0646 against 0.0804): the codes of an interval are those from `code` on,
// one more from `threshold` on.  One LDS read (32 entries in 64 banks: no
// conflicts) and one comparison in place of sixteen distances.
struct Interval {
    float threshold;
    unsigned code;
};
constexpr int kIntervals = 32;  // the first is for values that are no numbers
__device__ __forceinline__ unsigned interval_of(float normalized) {
    // 1..31 in the low bits: the sum's unit in the last place is one
    return __float_as_uint(
               __builtin_fmaf(normalized, 15.49F, 0x1p23F + 16.0F)) %
           kIntervals;
}
__device__ __forceinline__ Interval make_interval(unsigned interval) {
    Interval out{INFINITY, 0};
#pragma unroll
    for (int i = 0; i < 15; ++i) {
        const unsigned place = interval_of(kThresholds.at[i]);
        out.code += place < interval ? 1U : 0U;
        out.threshold = place == interval ? kThresholds.at[i] : out.threshold;
    }
    return out;
}

// What a workgroup of pack_kernel found: the sum of its scales, the biased
// exponent of the smallest non-zero one (INT_MAX: none), status bits.
struct ScaleRecord {
    double sum;
    int least_exponent;
    unsigned status;
};
__device__ __forceinline__ ScaleRecord combine(const ScaleRecord& a,
                                               const ScaleRecord& b) {
    return {a.sum + b.sum, min(a.least_exponent, b.least_exponent),
            a.status | b.status};
}

constexpr int kPackThreads = 512;
constexpr std::size_t kPackValues = kPackThreads * 8;
// Enough for every workgroup the device holds at once.
constexpr unsigned kMaxRecords = 1024;
static_assert(kMaxRecords * sizeof(ScaleRecord) <= kStreamWorkspaceBytes);

// A thread takes eight consecutive weights, a workgroup 4096 at a time; the
// threads of a quantisation block (4 to 512 neighbours) exchange their largest
// magnitude.  kWide: a block spans wavefronts (block sizes from 1024 on).
// records null: fp32 scales, status bits go to *status.
template <bool kWide>
__global__ __launch_bounds__(kPackThreads) void pack_kernel(
    const float* __restrict__ values, std::size_t element_count,
    unsigned block_shift, bool aligned, float* __restrict__ scales,
    std::uint8_t* __restrict__ codes, ScaleRecord* __restrict__ records,
    unsigned* __restrict__ status
) {
    constexpr unsigned kWaves = kPackThreads / 64;
    __shared__ Interval intervals[kIntervals];
    __shared__ unsigned wave_largest[2][kWaves];
    __shared__ ScaleRecord wave_records[kWaves];
    if (threadIdx.x < kIntervals) {
        intervals[threadIdx.x] = make_interval(threadIdx.x);
    }
    __syncthreads();

    const unsigned wave = threadIdx.x / 64;
    const unsigned block_threads = 1U << (block_shift - 3);
    const unsigned block_lanes = min(block_threads, 64U);
    const std::size_t byte_count = (element_count + 1) / 2;
    ScaleRecord record{0.0, INT_MAX, 0U};
    unsigned turn = 0;
    for (std::size_t tile = blockIdx.x; tile * kPackValues < element_count;
         tile += gridDim.x) {
        const std::size_t first = tile * kPackValues + threadIdx.x * 8;
        float value[8];
        if (aligned && first + 8 <= element_count) {
            const float4 low =
                *reinterpret_cast<const float4*>(values + first);
            const float4 high =
                *reinterpret_cast<const float4*>(values + first + 4);
            value[0] = low.x;
            value[1] = low.y;
            value[2] = low.z;
            value[3] = low.w;
            value[4] = high.x;
            value[5] = high.y;
            value[6] = high.z;
            value[7] = high.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                value[i] =
                    first + i < element_count ? values[first + i] : 0.0F;
            }
        }
        // magnitudes compare like their bits; above infinity: not a number
        unsigned largest = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            largest = max(largest, __float_as_uint(value[i]) & 0x7FFFFFFFU);
        }
        for (unsigned step = 1; step < block_lanes; step *= 2) {
            largest = max(largest, static_cast<unsigned>(__shfl_xor(
                                       static_cast<int>(largest),
                                       static_cast<int>(step), 64)));
        }
        if constexpr (kWide) {
            // (two arrays in turn: one barrier a tile)
            if (threadIdx.x % 64 == 0) {
                wave_largest[turn][wave] = largest;
            }
            __syncthreads();
            const unsigned block_waves = block_threads / 64;
            const unsigned first_wave = wave / block_waves * block_waves;
            for (unsigned other = 0; other < block_waves; ++other) {
                largest =
                    max(largest, wave_largest[turn][first_wave + other]);
            }
            turn ^= 1U;
        }
        const float scale = __uint_as_float(largest);
        if (largest >= kInfinityBits) {
            record.status = kNonFiniteSource;
        }
        if (first >= element_count) {
            continue;  // (kWide: the tile is the last one, see the loop)
        }
        if (threadIdx.x % block_threads == 0) {
            scales[first >> block_shift] = scale;
            record.sum += static_cast<double>(scale);
            if (largest != 0) {
                record.least_exponent =
                    min(record.least_exponent,
                        max(static_cast<int>(largest >> 23), 1));
            }
        }
        unsigned packed = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float normalized = value[i] / scale;
            const Interval interval = intervals[interval_of(normalized)];
            const unsigned code =
                interval.code + (normalized >= interval.threshold ? 1U : 0U);
            packed |= code << (4 * i);
        }
        if (largest == 0) {
            packed = 0x77777777U;
        }
        const std::size_t first_byte = first / 2;
        if (first + 8 <= element_count) {
            // four-byte groups start at multiples of four bytes
            *reinterpret_cast<unsigned*>(codes + first_byte) = packed;
        } else {
            // an unused nibble stays zero
            packed &= (1U << (4 * (element_count - first))) - 1U;
            for (unsigned i = 0; first_byte + i < byte_count; ++i) {
                codes[first_byte + i] =
                    static_cast<std::uint8_t>((packed >> (8 * i)) & 0xFFU);
            }
        }
    }
    if (records == nullptr) {
        if (record.status != 0) {
            atomicOr(status, record.status);
        }
        return;
    }
#pragma unroll
    for (int step = 32; step >= 1; step /= 2) {
        record = combine(
            record,
            {__shfl_xor(record.sum, step, 64),
             __shfl_xor(record.least_exponent, step, 64),
             static_cast<unsigned>(__shfl_xor(
                 static_cast<int>(record.status), step, 64))});
    }
    if (threadIdx.x % 64 == 0) {
        wave_records[wave] = record;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned other = 1; other < kWaves; ++other) {
            record = combine(record, wave_records[other]);
        }
        records[blockIdx.x] = record;
    }
}

// The scales' mean, then their codes; one wavefront per group of
// second-level-block scales.  Every workgroup adds the records for itself, in
// the same order (at most 16 KB from L2, where a launch of one workgroup
// between the two kernels took longer); the first one reports the mean and the
// status.
constexpr int kEncodeThreads = 256;

__global__ __launch_bounds__(kEncodeThreads) void scale_encode_kernel(
    const float* __restrict__ scales, std::size_t count, unsigned group_shift,
    std::size_t group_count, const ScaleRecord* __restrict__ records,
    unsigned record_count, float* __restrict__ offset_out,
    unsigned* __restrict__ status, std::uint8_t* __restrict__ scale_codes,
    float* __restrict__ second_level
) {
#pragma clang fp contract(off)
    __shared__ ScaleRecord sums[kEncodeThreads];
    constexpr unsigned kStaged = 1024;
    __shared__ float staged[kStaged];
    ScaleRecord record{0.0, INT_MAX, 0U};
    for (unsigned index = threadIdx.x; index < record_count;
         index += kEncodeThreads) {
        record = combine(record, records[index]);
    }
    sums[threadIdx.x] = record;
    __syncthreads();
    for (unsigned width = kEncodeThreads / 2; width >= 1; width /= 2) {
        if (threadIdx.x < width) {
            sums[threadIdx.x] =
                combine(sums[threadIdx.x], sums[threadIdx.x + width]);
        }
        __syncthreads();
    }
    record = sums[0];
    // 2^53 units in the last place of the smallest scale: the exponent of
    // that unit is least_exponent - 127 - 23
    const bool order_free =
        record.status != 0 || record.least_exponent == INT_MAX ||
        record.sum < ldexp(1.0, 53 - 127 - 23 + record.least_exponent);
    if (!order_free) {  // uniform
        double total = 0.0;
        for (std::size_t first = 0; first < count; first += kStaged) {
            __syncthreads();
            for (unsigned i = threadIdx.x; i < kStaged; i += kEncodeThreads) {
                staged[i] = first + i < count ? scales[first + i] : 0.0F;
            }
            __syncthreads();
            if (threadIdx.x == 0) {
                // (zeros past the end change no sum)
#pragma unroll 16
                for (unsigned i = 0; i < kStaged; ++i) {
                    total += static_cast<double>(staged[i]);
                }
            }
        }
        if (threadIdx.x == 0) {
            sums[0].sum = total;
        }
        __syncthreads();
        record.sum = sums[0].sum;
    }
    const float offset =
        static_cast<float>(record.sum / static_cast<double>(count));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *offset_out = offset;
        *status = record.status | (isfinite(offset) ? 0U : kOffsetOverflow);
    }

    const std::size_t waves_per_grid =
        static_cast<std::size_t>(gridDim.x) * (kEncodeThreads / 64);
    const unsigned lane = threadIdx.x % 64;
    const std::size_t group_size = std::size_t{1} << group_shift;
    for (std::size_t group =
             static_cast<std::size_t>(blockIdx.x) * (kEncodeThreads / 64) +
             threadIdx.x / 64;
         group < group_count; group += waves_per_grid) {
        const std::size_t begin = group << group_shift;
        const std::size_t end =
            begin + group_size < count ? begin + group_size : count;
        float absmax = 0.0F;
        for (std::size_t index = begin + lane; index < end; index += 64) {
            const float distance = fabsf(scales[index] - offset);
            absmax = absmax < distance ? distance : absmax;
        }
#pragma unroll
        for (int step = 32; step >= 1; step /= 2) {
            const float other = __shfl_xor(absmax, step, 64);
            absmax = absmax < other ? other : absmax;
        }
        if (lane == 0) {
            second_level[group] = absmax;
        }
        for (std::size_t index = begin + lane; index < end; index += 64) {
            unsigned code = 128;
            if (absmax != 0.0F) {
                const float normalized = (scales[index] - offset) / absmax;
                const float scaled = normalized * 127.0F;
                const float rounded = scaled >= 0.0F ? floorf(scaled + 0.5F)
                                                     : ceilf(scaled - 0.5F);
                int centered = static_cast<int>(rounded);
                centered =
                    centered < -127 ? -127 : (centered > 127 ? 127 : centered);
                code = static_cast<unsigned>(centered + 128);
            }
            scale_codes[index] = static_cast<std::uint8_t>(code);
        }
    }
}

unsigned grid_for(std::size_t items, std::size_t per_block, unsigned most) {
    const std::size_t blocks = (items + per_block - 1) / per_block;
    return static_cast<unsigned>(blocks < most ? blocks : most);
}

}  // namespace

void launch_quantize(const QuantizeProblem& p, hipStream_t stream) {
    const bool nested = p.scale_codes != nullptr;
    const std::size_t block_count =
        (p.element_count + (std::size_t{1} << p.block_shift) - 1) >>
        p.block_shift;
    ScaleRecord* const records =
        nested ? static_cast<ScaleRecord*>(p.workspace) : nullptr;
    if (!nested) {
        launch_fill(reinterpret_cast<float*>(p.status), 0.0F, 1, stream);
    }
    const unsigned groups =
        grid_for(p.element_count, kPackValues, kMaxRecords);
    const auto kernel =
        p.block_shift > 9 ? pack_kernel<true> : pack_kernel<false>;
    kernel<<<groups, kPackThreads, 0, stream>>>(
        p.values, p.element_count, p.block_shift,
        reinterpret_cast<std::uintptr_t>(p.values) % 16 == 0, p.fp32_scales,
        p.codes, records, p.status);
    if (!nested) {
        return;
    }
    const std::size_t group_count =
        (block_count + (std::size_t{1} << p.second_level_shift) - 1) >>
        p.second_level_shift;
    constexpr unsigned kEncodeGroups = 512;
    scale_encode_kernel<<<
        grid_for(group_count, kEncodeThreads / 64, kEncodeGroups),
        kEncodeThreads, 0, stream>>>(
        p.fp32_scales, block_count, p.second_level_shift, group_count,
        records, groups, p.offset, p.status, p.scale_codes, p.second_level);
}

}  // namespace rthip
