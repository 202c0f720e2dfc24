// Device-side pieces shared by the fused attention kernels: the head width, V's
// transposing fragment reads out of LDS, masked loads of the packed projection
// and the exchanges between the lanes that hold one query's row.
#pragma once

#include "device_common.hpp"
#include "gemm_kernel.hpp"

namespace cuvit::detail::attention {

using namespace cuvit::device;

constexpr int kHeadDim = 64;  // head_dim the fused kernels handle

/// Elements per LDS row of K ([key][head_dim + 8]).
constexpr int kKeyPitch = kHeadDim + 8;

/// Element offset of V[key][dim] in its LDS tile: 16-byte chunk dim / 8 of
/// the key's row sits at chunk (dim / 8) ^ 4 ((key >> 1) & 1).
__device__ __forceinline__ int value_slot(int key, int dim) {
    return key * kHeadDim + 8 * ((dim >> 3) ^ (4 * ((key >> 1) & 1))) + (dim & 7);
}

/// Four 16-bit elements in LDS, the operand type of ds_read_b64_tr_b16.
typedef short Short4 __attribute__((vector_size(4 * sizeof(short))));
using Lds4x16 = __attribute__((address_space(3))) Short4;

/// The weights.V B fragment of k-block @p kb, dims @p d0 + 0..31: lane l
/// holds dim d0 + l % 32, keys 16 kb + 8 (l / 32) + 0..7, the layout a
/// 16-byte row of transposed V would give it.
__device__ __forceinline__ Vec16 value_fragment(const std::uint16_t* values, int kb, int d0,
                                                int lane) {
    const int j = lane & 15;
    const int dim = d0 + 16 * ((lane >> 4) & 1) + 4 * (j & 3);
    Vec16 fragment;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int key = kb * 16 + 8 * (lane >> 5) + 4 * s + (j >> 2);
        // `values` points into LDS; the C-style cast is the address-space
        // conversion the builtin's operand needs.
        const auto part =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds4x16*)(values + value_slot(key, dim)));
        fragment.w[2 * s] = static_cast<std::uint16_t>(part[0]) |
                            (static_cast<std::uint32_t>(static_cast<std::uint16_t>(part[1])) << 16);
        fragment.w[2 * s + 1] = static_cast<std::uint16_t>(part[2]) |
                                (static_cast<std::uint32_t>(static_cast<std::uint16_t>(part[3])) << 16);
    }
    return fragment;
}

/// 16 bytes at @p element of the pair's packed projection, through the
/// buffer resource @p resource (based at that element 0), or zero when
/// @p inside is false: the offset is then one the resource drops, so the load
/// needs no branch. The launches hold an image's rows to 0x7FFFFFF0 bytes, so
/// an element's byte offset fits the 32 bits the load takes.
__device__ __forceinline__ Vec16 load_or_zero(__amdgpu_buffer_rsrc_t resource, std::int64_t element,
                                              bool inside) {
    return gemm::buffer_load16(resource, inside ? static_cast<unsigned int>(element * 2) : gemm::kOutside);
}

/// op(value of lanes 16 k + i, value of lanes 16 (k + 1) + i) for k = 0 and
/// k = 2, in both lanes of each pair (@p kRows 16: rows of 16 lanes, by
/// v_permlane16_swap), or op(lower half, upper half) (@p kRows 32, by
/// v_permlane32_swap): a swap of the value with itself leaves each lane its
/// own value and its partner's, the lower one first in both lanes, with no LDS
/// round trip. op is max or + here, which give the same bits as
/// op(own, partner) in either order.
template <int kRows, typename Op> __device__ __forceinline__ float combine_rows(float value, Op op) {
    const std::uint32_t bits = __float_as_uint(value);
    if constexpr (kRows == 16) {
        const auto swapped = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
        return op(__uint_as_float(swapped[0]), __uint_as_float(swapped[1]));
    } else {
        static_assert(kRows == 32, "rows of 16 or halves of 32 lanes");
        const auto swapped = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        return op(__uint_as_float(swapped[0]), __uint_as_float(swapped[1]));
    }
}

/// op over the two lanes l and l ^ 32, the lower half's value first.
template <typename Op> __device__ __forceinline__ float combine_halves(float value, Op op) {
    return combine_rows<32>(value, op);
}

} // namespace cuvit::detail::attention
