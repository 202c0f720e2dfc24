// Launch of the LDS-ring GEMM (gemm_ring.hpp): its instances, one translation
// unit of their own.
#include "gemm_choice.hpp"
#include "gemm_ring.hpp"

namespace cuvit::detail {
namespace {

/// Launches @p Kernel over the tile grid, one workgroup per tile (per slot of
/// the largest XCD block with a split) and batch entry.
template <typename S, auto Kernel, typename T>
hipError_t run_tiles(const T* a, const T* b, const float* bias, T* c, const GemmArgs& args,
                     const gemm::TileMap& map, int c_run, hipStream_t stream) {
    const std::int64_t tiles_m = (args.m + S::kBM - 1) / S::kBM;
    const std::int64_t tiles_n = (args.n + S::kBN - 1) / S::kBN;
    const std::int64_t tiles = map.px > 0 ? 8 * ((tiles_m + map.px - 1) / map.px) *
                                                ((tiles_n + map.py - 1) / map.py)
                                          : tiles_m * tiles_n;
    if (tiles > 0x7FFFFFFF) {
        return hipErrorInvalidConfiguration;
    }
    if (const hipError_t opted = allow_lds<Kernel>(S::kLdsBytes); opted != hipSuccess) {
        return opted;
    }
    return for_entries(args.count, [&](int first, int entries) -> hipError_t {
        const dim3 grid = map.px < 0 ? dim3(kXcds, static_cast<unsigned int>(tiles),
                                            static_cast<unsigned int>((entries + kXcds - 1) / kXcds))
                                     : dim3(static_cast<unsigned int>(tiles), static_cast<unsigned int>(entries));
        Kernel<<<grid, S::kThreads, S::kLdsBytes, stream>>>(a, b, bias, c, args, map, c_run, first);
        return hipGetLastError();
    });
}

template <typename S>
hipError_t launch(const std::uint16_t* a, const std::uint16_t* b, const float* bias, std::uint16_t* c,
                  const GemmArgs& args, const gemm::TileMap& map, int c_run, hipStream_t stream) {
    auto run = [&](auto kernel) -> hipError_t {
        return run_tiles<S, decltype(kernel)::kValue>(a, b, bias, c, args, map, c_run, stream);
    };
    if (args.addend != nullptr) {
        return run(KernelConstant<gemm::gemm_ring_kernel<S, true, false, false, true>>{});
    }
    auto with_gelu = [&](auto with_bias) -> hipError_t {
        constexpr bool kB = decltype(with_bias)::value;
        if (args.gelu) {
            return args.accumulate ? run(KernelConstant<gemm::gemm_ring_kernel<S, kB, true, true>>{})
                                   : run(KernelConstant<gemm::gemm_ring_kernel<S, kB, true, false>>{});
        }
        return args.accumulate ? run(KernelConstant<gemm::gemm_ring_kernel<S, kB, false, true>>{})
                               : run(KernelConstant<gemm::gemm_ring_kernel<S, kB, false, false>>{});
    };
    return bias != nullptr ? with_gelu(std::true_type{}) : with_gelu(std::false_type{});
}

} // namespace

hipError_t gemm_ring_bf16(RingTile tile, const std::uint16_t* a, const std::uint16_t* b,
                          const float* bias, std::uint16_t* c, const GemmArgs& args,
                          const gemm::TileMap& map, int c_run, hipStream_t stream) {
    using T = std::uint16_t;
    switch (tile) {
    case RingTile::k64x64: return launch<gemm::RingShape<T, 2, 2, 1, 1, 2>>(a, b, bias, c, args, map, c_run, stream);
    case RingTile::k64x32Alone:
        return launch<gemm::RingShape<T, 2, 1, 1, 1, 4, true, true>>(a, b, bias, c, args, map, c_run, stream);
    case RingTile::k64x64Alone:
        return launch<gemm::RingShape<T, 2, 2, 1, 1, 3, true, true>>(a, b, bias, c, args, map, c_run, stream);
    case RingTile::k64x64Deep:
        return launch<gemm::RingShape<T, 2, 2, 1, 1, 3, true>>(a, b, bias, c, args, map, c_run, stream);
    case RingTile::k128x64:
        return launch<gemm::RingShape<T, 4, 2, 1, 1, 2>>(a, b, bias, c, args, map, c_run, stream);
    case RingTile::k128x128:
        return launch<gemm::RingShape<T, 4, 2, 1, 2, 2>>(a, b, bias, c, args, map, c_run, stream);
    default: return launch<gemm::RingShape<T, 4, 2, 1, 2, 3>>(a, b, bias, c, args, map, c_run, stream);
    }
}

hipError_t gemm_ring_f32(RingTileF32 tile, const float* a, const float* b, const float* bias, float* c,
                         const GemmArgs& args, const gemm::TileMap& map, hipStream_t stream) {
    auto launch_f32 = [&](auto shape) -> hipError_t {
        using S = decltype(shape);
        return run_tiles<S, gemm::gemm_ring_f32_kernel<S>>(a, b, bias, c, args, map, 4, stream);
    };
    switch (tile) {
    case RingTileF32::k32x16Alone: return launch_f32(gemm::RingShape<float, 2, 1, 1, 1, 3, true, true>{});
    case RingTileF32::k32x32: return launch_f32(gemm::RingShape<float, 2, 2, 1, 1, 2, true>{});
    case RingTileF32::k32x32Deep: return launch_f32(gemm::RingShape<float, 2, 2, 1, 1, 3, true>{});
    case RingTileF32::k64x32: return launch_f32(gemm::RingShape<float, 2, 2, 2, 1, 2, true>{});
    default: return launch_f32(gemm::RingShape<float, 2, 2, 2, 2, 2, true>{});
    }
}

} // namespace cuvit::detail
