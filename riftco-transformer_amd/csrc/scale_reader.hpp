// Block scales read through buffer descriptors, for the matrix-core kernels of
// the packed weight: requested as they lie in memory and decoded when the
// load has returned.
#pragma once

#include "gemv_shared.hpp"
#include "nf4_decode.hpp"

namespace rthip {
namespace {

constexpr unsigned kOutside = 0xFFFFFFFFU;  // past every descriptor's extent

// A block scale as it was loaded: the fp32 scale, or the second-level scale
// with the block's scale code beside it.
struct LoadedScale {
    float value;
    unsigned code;
};

template <bool kDoubleQuantized>
class ScaleReader {
public:
    __device__ __forceinline__ ScaleReader(const Nf4WeightView& weight,
                                           unsigned weights,
                                           unsigned block_shift)
        : block_shift_(block_shift),
          second_level_shift_(weight.second_level_shift),
          offset_(weight.offset) {
        const unsigned blocks = ((weights - 1U) >> block_shift) + 1U;
        primary_ = make_buffer(
            weight.primary_scales,
            kDoubleQuantized ? blocks
                             : blocks * static_cast<unsigned>(sizeof(float)));
        secondary_ = make_buffer(
            weight.secondary_scales,
            kDoubleQuantized
                ? (((blocks - 1U) >> second_level_shift_) + 1U) *
                      static_cast<unsigned>(sizeof(float))
                : 0U);
    }
    // The scale of flat weight `flat`; zero where it is not `inside`.
    __device__ __forceinline__ LoadedScale load(unsigned flat,
                                                bool inside) const {
        const unsigned block = inside ? flat >> block_shift_ : kOutside / 4;
        LoadedScale out{0.0F, 0U};
        if constexpr (kDoubleQuantized) {
            out.code = __builtin_amdgcn_raw_buffer_load_b8(primary_, block, 0,
                                                           0);
            out.value = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           secondary_, (block >> second_level_shift_) * 4, 0,
                           0));
        } else {
            out.value = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(primary_,
                                                            block * 4, 0, 0));
        }
        return out;
    }
    __device__ __forceinline__ float decode(const LoadedScale& loaded,
                                            const float* factors) const {
        if constexpr (kDoubleQuantized) {
            return double_quantized_scale_from_factor(factors[loaded.code],
                                                      loaded.value, offset_);
        } else {
            return loaded.value;
        }
    }

private:
    __amdgpu_buffer_rsrc_t primary_;
    __amdgpu_buffer_rsrc_t secondary_;
    unsigned block_shift_;
    unsigned second_level_shift_;
    float offset_;
};

}  // namespace
}  // namespace rthip
