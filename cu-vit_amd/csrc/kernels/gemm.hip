// Host dispatch of the batched GEMM. The kernels, all measured on MI355X at
// the ViT shapes and picked in this order:
//   fp32 (16 x 16 MFMA): the resident-panel kernel (gemm_panel.hpp) for
//        tall products with B as [N, K] and K of 192, or 768 into up to 1024 columns
//        (the ViT-Tiny linear layers and patch embedding); the ring kernel
//        (gemm_ring.hpp) for the others with B as [N, K] and 16-byte rows, but
//        for some of the largest; else the tiled kernel (gemm_kernel.hpp), 32 x
//        32 tiles, 64 x 64 once a problem has work for more than 32 small tiles
//        per compute unit.
//   bf16 (32 x 32 MFMA): B as [N, K] with 16-byte rows runs on direct-to-LDS
//        loads, in the persistent kernel (gemm_dma.hpp, up to 320 x 256 tiles)
//        where its tiles fill the chip and in the ring kernel (gemm_ring.hpp,
//        64 x 64 to 128 x 128 tiles) otherwise, by a cost fitted to both; else
//        (B as [K, N], odd rows) the tiled kernel, 128 x 128 once a problem
//        fills every compute unit twice with it (32-deep stages up to K =
//        1024), else 64 x 64.
// Every kernel of a type runs the same MFMA over K in the same order, so the
// choice never changes a result.
#include "gemm_choice.hpp"
#include "gemm_dma.hpp"
#include "gemm_kernel.hpp"
#include "gemm_panel.hpp"

namespace cuvit::detail {
namespace {

using cuvit::device::aligned16;
using gemm::Shape;

/// True when every row of an operand starts on a 16-byte boundary and rows
/// of @p depth elements (the vector direction) hold whole 16-byte chunks.
template <typename T>
bool vector_operand(const T* base, int ld, int depth, std::int64_t stride, std::int64_t outer_stride,
                    bool split) {
    constexpr int V = gemm::Mma<T>::kPerVec;
    return aligned16(base) && ld % V == 0 && depth % V == 0 && stride % V == 0 &&
           (!split || outer_stride % V == 0);
}

/// True when the epilogue may store four results at once: floats always (a
/// dwordx4 store needs 4-byte alignment; the logits product of 24 heads at 577
/// tokens, odd rows of C: 34.3 -> 28.1, the tile kernel before it included us), bf16 on 8-byte rows.
template <typename T> bool vector_output(const T* c, const GemmArgs& args) {
    if (sizeof(T) == 4) {
        return true;
    }
    const bool split = args.inner > 0;
    return (reinterpret_cast<std::uintptr_t>(c) % (4 * sizeof(T))) == 0 && args.ldc % 4 == 0 &&
           args.stride_c % 4 == 0 && (!split || args.outer_stride_c % 4 == 0);
}

template <typename T, int WM, int WN, int TM, int TN, int BK, int MinWaves, bool VecA, bool VecB,
          bool TransB, bool Unaligned>
hipError_t launch(const T* a, const T* b, const float* bias, T* c, const GemmArgs& args,
                  bool vector_c, hipStream_t stream) {
    using S = Shape<T, WM, WN, TM, TN, BK>;
    const gemm::TileMap map = tile_map(args, S::kBM, S::kBN, sizeof(T));
    const std::int64_t tiles_m = (args.m + S::kBM - 1) / S::kBM;
    const std::int64_t tiles_n = (args.n + S::kBN - 1) / S::kBN;
    // With the XCD split every block gets a workgroup slot per tile of the
    // largest block.
    const std::int64_t tiles = map.px > 0
                                   ? 8 * ((tiles_m + map.px - 1) / map.px) * ((tiles_n + map.py - 1) / map.py)
                                   : tiles_m * tiles_n;
    if (tiles > 0x7FFFFFFF) {
        return hipErrorInvalidConfiguration;
    }
    // The occupancy hint caps registers; the element-wise operand paths need
    // more than it leaves, so they take the default.
    constexpr int kMinWaves = VecA && VecB ? MinWaves : 1;
    constexpr auto kernel = gemm::gemm_kernel<T, WM, WN, TM, TN, BK, VecA, VecB, TransB, kMinWaves, Unaligned>;
    // Above 64 KiB of LDS a kernel has to opt in, once per device.
    if (const hipError_t opted = allow_lds<kernel>(S::kLdsBytes); opted != hipSuccess) {
        return opted;
    }
    const dim3 grid(static_cast<unsigned int>(tiles),
                    static_cast<unsigned int>(args.count < kMaxGridY ? args.count : kMaxGridY));
    kernel<<<grid, S::kThreads, S::kLdsBytes, stream>>>(a, b, bias, c, args, map, vector_c);
    return hipGetLastError();
}

template <typename T, int WM, int WN, int TM, int TN, int BK, int MinWaves = 1>
hipError_t pick_flags(const T* a, const T* b, const float* bias, T* c, const GemmArgs& args,
                      hipStream_t stream) {
    using S = Shape<T, WM, WN, TM, TN, BK>;
    const bool split = args.inner > 0;
    // Buffer offsets of a tile stay inside the span one descriptor addresses.
    const bool spans_a = static_cast<std::int64_t>(S::kBM) * args.lda * sizeof(T) < gemm::kMaxSpan;
    const bool spans_b = (args.transposed ? static_cast<std::int64_t>(S::kBN) : static_cast<std::int64_t>(args.k)) *
                             args.ldb * sizeof(T) <
                         gemm::kMaxSpan;
    const bool vec_a =
        spans_a && vector_operand(a, args.lda, args.k, args.stride_a, args.outer_stride_a, split);
    const bool vec_b = spans_b && vector_operand(b, args.ldb, args.transposed ? args.k : args.n, args.stride_b,
                                                 args.outer_stride_b, split);
    const bool vec_c = vector_output(c, args);
#define CUVIT_GEMM_LAUNCH(VA, VB, U)                                                               \
    (args.transposed ? launch<T, WM, WN, TM, TN, BK, MinWaves, VA, VB, true, U>(a, b, bias, c, args, vec_c, stream) \
                     : launch<T, WM, WN, TM, TN, BK, MinWaves, VA, VB, false, U>(a, b, bias, c, args, vec_c, stream))
    if (vec_a && vec_b) {
        return CUVIT_GEMM_LAUNCH(true, true, false);
    }
    if constexpr (sizeof(T) == 4) {
        // fp32 rows that start at any float, through the resources all the same
        // (577 x 64 x 577 in 24 entries 25 us element by element, 20 so). Not where
        // neither operand has aligned rows, most of a short K is a cut stage's four
        // loads a chunk, and enough workgroups share a CU to hide the element-wise
        // loads: 577 x 98 x 50 in 96 entries 28.5 us element by element, 36 so;
        // 12000 x 577 x 65 38.5 and 43.
        const bool element_wise = !vec_a && !vec_b && args.k < (args.transposed ? 64 : 128) &&
                                  tile_count(args, 32, 32) > 20 * static_cast<std::int64_t>(compute_units());
        if (spans_a && spans_b && !element_wise) {
            return vec_a   ? CUVIT_GEMM_LAUNCH(true, false, true)
                   : vec_b ? CUVIT_GEMM_LAUNCH(false, true, true)
                           : CUVIT_GEMM_LAUNCH(false, false, true);
        }
        return CUVIT_GEMM_LAUNCH(false, false, false);
    } else {
        return vec_a   ? CUVIT_GEMM_LAUNCH(true, false, false)
               : vec_b ? CUVIT_GEMM_LAUNCH(false, true, false)
                       : CUVIT_GEMM_LAUNCH(false, false, false);
    }
#undef CUVIT_GEMM_LAUNCH
}

/// @p args with a batch whose entries share B (stride 0) and whose A rows
/// follow one another run as one problem of all the entries' rows
/// (rows_per_entry: each output row goes back to its entry); @p args itself
/// otherwise. Every output is computed by the same operations either way.
GemmArgs as_one_problem(const GemmArgs& args) {
    GemmArgs whole = args;
    if (args.count > 1 && args.inner == 0 && args.stride_b == 0 && args.m > 0 &&
        args.stride_a == static_cast<std::int64_t>(args.m) * args.lda &&
        static_cast<std::int64_t>(args.m) * args.count <= 0x7FFFFFFF) {
        whole.m = args.m * args.count;
        whole.count = 1;
        whole.rows_per_entry = args.m;
    }
    return whole;
}

} // namespace

/// The resident-panel kernel (gemm_panel.hpp) for a problem it covers: one
/// batch entry (or entries run as one, rows_per_entry), B as [N, K], K equal
/// to 16 KB, vector A and B, C written in 16-byte runs (N, ldc and the entry
/// stride multiples of 4, C 16-byte aligned), an addend only without GELU or
/// accumulation (and in 16-byte runs), every operand within one descriptor's
/// span, and at least eight wavefront items per compute unit. Returns
/// hipErrorNotSupported otherwise.
template <int KB, int BN, int TN, int KG, int W>
hipError_t launch_panel(const float* a, const float* b, const float* bias, float* c,
                        const GemmArgs& args, hipStream_t stream) {
    using S = gemm::PanelShape<KB, BN, TN, KG, W>;
    const std::int64_t tiles_m = (args.m + 15) / 16;
    const std::int64_t panels = (args.n + BN - 1) / BN;
    const bool with_addend = args.addend != nullptr;
    const std::int64_t c_span =
        args.rows_per_entry > 0
            ? ((args.m - 1) / args.rows_per_entry + 1) * args.stride_c
            : static_cast<std::int64_t>(args.m) * args.ldc;
    const bool eligible =
        args.count == 1 && args.transposed &&
        (!with_addend || (!args.gelu && !args.accumulate && aligned16(args.addend) &&
                          args.ld_addend % 4 == 0 &&
                          static_cast<std::int64_t>(args.m) * args.ld_addend * 4 < gemm::kMaxSpan)) &&
        args.k == 16 * KB && vector_operand(a, args.lda, args.k, 0, 0, false) &&
        vector_operand(b, args.ldb, args.k, 0, 0, false) && aligned16(c) && args.ldc % 4 == 0 && args.stride_c % 4 == 0 &&
        args.n % 4 == 0 && static_cast<std::int64_t>(args.m) * args.lda * 4 < gemm::kMaxSpan &&
        c_span * 4 < gemm::kMaxSpan &&
        static_cast<std::int64_t>(BN) * args.ldb * 4 < gemm::kMaxSpan &&
        tiles_m * panels * S::kParts >= 8 * static_cast<std::int64_t>(compute_units());
    if (!eligible) {
        return hipErrorNotSupported;
    }
    // One workgroup per compute unit: the row tiles of a panel split into
    // as many ranges as there are compute units per panel.
    std::int64_t groups = compute_units() / panels;
    groups = groups < 1 ? 1 : groups > tiles_m ? tiles_m : groups;
    const dim3 grid(static_cast<unsigned int>(panels * groups));
    const int groups_argument = static_cast<int>(groups);
    auto run = [&](auto chosen) -> hipError_t {
        constexpr auto kernel = decltype(chosen)::kValue;
        if (const hipError_t opted = allow_lds<kernel>(S::kLdsBytes); opted != hipSuccess) {
            return opted;
        }
        kernel<<<grid, S::kThreads, S::kLdsBytes, stream>>>(a, b, bias, c, args, groups_argument);
        return hipGetLastError();
    };
    // The epilogue's parts as template flags: alpha (when not 1), bias, GELU,
    // accumulate; the addend alone (the patch embedding's positional add).
    auto with_alpha = [&](auto alpha, auto with_bias, auto gelu, auto accumulate) -> hipError_t {
        return run(KernelConstant<gemm::gemm_panel_kernel<KB, BN, TN, KG, W, decltype(alpha)::value,
                                                          decltype(with_bias)::value, decltype(gelu)::value,
                                                          decltype(accumulate)::value>>{});
    };
    if (with_addend) {
        auto with_bias = [&](auto alpha) -> hipError_t {
            constexpr bool kAlpha = decltype(alpha)::value;
            return bias != nullptr
                       ? run(KernelConstant<gemm::gemm_panel_kernel<KB, BN, TN, KG, W, kAlpha, true, false, false, true>>{})
                       : run(KernelConstant<gemm::gemm_panel_kernel<KB, BN, TN, KG, W, kAlpha, false, false, false, true>>{});
        };
        return args.alpha == 1.0F ? with_bias(std::false_type{}) : with_bias(std::true_type{});
    }
    auto with_accumulate = [&](auto with_bias, auto gelu) -> hipError_t {
        if (args.accumulate) {
            return args.alpha == 1.0F ? with_alpha(std::false_type{}, with_bias, gelu, std::true_type{})
                                      : with_alpha(std::true_type{}, with_bias, gelu, std::true_type{});
        }
        return args.alpha == 1.0F ? with_alpha(std::false_type{}, with_bias, gelu, std::false_type{})
                                  : with_alpha(std::true_type{}, with_bias, gelu, std::false_type{});
    };
    auto with_gelu = [&](auto with_bias) -> hipError_t {
        return args.gelu ? with_accumulate(with_bias, std::true_type{})
                         : with_accumulate(with_bias, std::false_type{});
    };
    return bias != nullptr ? with_gelu(std::true_type{}) : with_gelu(std::false_type{});
}

hipError_t gemm_f32(const float* a, const float* b, const float* bias, float* c,
                    const GemmArgs& args, hipStream_t stream) {
    // Tall single products with B as [N, K] (the model's linear layers): the
    // resident-panel kernel, bitwise equal to the tiles below. Measured at
    // ViT-Tiny batch 32 (6304 rows), against the tiled kernel: QKV 21.4 ->
    // 17.8 us, FC1 + GELU 27.9 -> 24.2, projection 10.7 -> 8.4, FC2 25.7 ->
    // 22.7. Wide panels with three wavefronts per SIMD suit the wide outputs,
    // 32-column panels the 192-wide ones.
    // A batch whose entries share B and whose A rows follow one another (the
    // patch embedding: 196 rows per image into rows 1.. of its 197) runs as
    // one problem of all its rows (ViT-Tiny b32 embedding 27 -> 22 us).
    const GemmArgs whole = as_one_problem(args);
    if (whole.n >= 512) {
        if (const hipError_t panel = launch_panel<12, 64, 2, 4, 12>(a, b, bias, c, whole, stream);
            panel != hipErrorNotSupported) {
            return panel;
        }
    } else if (const hipError_t panel = launch_panel<12, 32, 2, 4, 8>(a, b, bias, c, whole, stream);
               panel != hipErrorNotSupported) {
        return panel;
    }
    // K = 768: the panels into few columns (192 of 6304 rows: 23.1 us against the
    // ring kernel's 25.0) and, with many tiles, into up to 1024 (768 of 4616 rows
    // accumulating 51 against 55 to 58, of 3152 37 against 39 to 41, of 2364 31.6
    // against 31). Wider ones, and with GELU, are the ring kernel's (3152 x 2304
    // 101 against 101, 4616 x 3072 with GELU 216 against 190).
    if (whole.n < 512 || (whole.n <= 1024 && !whole.gelu &&
                          tile_count(whole, 32, 32) > 8 * static_cast<std::int64_t>(compute_units()))) {
        if (const hipError_t panel = launch_panel<48, 32, 2, 4, 12>(a, b, bias, c, whole, stream);
            panel != hipErrorNotSupported) {
            return panel;
        }
    }
    const bool split = whole.inner > 0;
    if (whole.transposed && vector_operand(a, whole.lda, whole.k, whole.stride_a, whole.outer_stride_a, split) &&
        vector_operand(b, whole.ldb, whole.k, whole.stride_b, whole.outer_stride_b, split) &&
        static_cast<std::int64_t>(64) * whole.lda * 4 < gemm::kMaxSpan &&
        static_cast<std::int64_t>(64) * whole.ldb * 4 < gemm::kMaxSpan && !tiled_beats_ring_f32(whole, compute_units())) {
        const RingChoiceF32 ring = choose_ring_f32(whole, compute_units());
        return gemm_ring_f32(ring.tile, a, b, bias, c, whole, ring.map, stream);
    }
    if (tile_count(args, 32, 32) > static_cast<std::int64_t>(compute_units()) * 32) {
        return pick_flags<float, 2, 2, 2, 2, 32>(a, b, bias, c, args, stream);
    }
    return pick_flags<float, 2, 2, 1, 1, 32>(a, b, bias, c, args, stream);
}

/// The direct-to-LDS kernel (gemm_dma.hpp) for a problem it covers: one batch
/// entry, B as [N, K], N a multiple of 256, K of at least 256, no addend,
/// vector A and B, C written in 16-byte pieces, every operand tile within one
/// descriptor's span, the CUs a multiple of 8 (one persistent workgroup per
/// CU, the same number on every XCD), tiles for at least half the CUs, and no
/// @p ring tile that is the better choice. Returns hipErrorNotSupported
/// otherwise.
hipError_t launch_dma(const std::uint16_t* a, const std::uint16_t* b, const float* bias,
                      std::uint16_t* c, const GemmArgs& args, const RingChoice& ring, hipStream_t stream) {
    const int units = compute_units();
    // Entries run as one problem, each row stored back in its entry: the patch
    // embedding, with its positional addend (the instance that takes entries).
    const bool with_addend = args.addend != nullptr;
    const bool entries = args.rows_per_entry > 0;
    // The addend only in the combination the model uses (bias, no alpha, no
    // GELU, no accumulation), 16-byte runs of it per lane.
    const bool addend_ok =
        !with_addend ||
        (bias != nullptr && args.alpha == 1.0F && !args.gelu && !args.accumulate && aligned16(args.addend) &&
         args.ld_addend % 4 == 0);
    const bool eligible =
        args.transposed && args.count == 1 && addend_ok && (!entries || (with_addend && args.stride_c % 8 == 0)) &&
        args.n % 256 == 0 && args.k >= 256 && units % 8 == 0 &&
        vector_operand(a, args.lda, args.k, 0, 0, false) && vector_operand(b, args.ldb, args.k, 0, 0, false) &&
        static_cast<std::int64_t>(320) * args.lda * 2 < gemm::kMaxSpan &&
        static_cast<std::int64_t>(256) * args.ldb * 2 < gemm::kMaxSpan && aligned16(c) &&
        args.ldc % 8 == 0 && static_cast<std::int64_t>(args.n) * 4 < gemm::kMaxSpan;
    if (!eligible) {
        return hipErrorNotSupported;
    }
    const DmaChoice choice = choose_dma(args, units);
    if (ring_beats_dma(args, ring, choice)) {
        return hipErrorNotSupported;
    }
    auto run = [&](auto chosen, std::size_t lds_bytes) -> hipError_t {
        constexpr auto kernel = decltype(chosen)::kValue;
        if (const hipError_t opted = allow_lds<kernel>(lds_bytes); opted != hipSuccess) {
            return opted;
        }
        kernel<<<units, 512, lds_bytes, stream>>>(a, b, bias, c, args, choice.map);
        return hipGetLastError();
    };
    // The epilogue's parts as template flags: bias, GELU, alpha (when not 1),
    // accumulate.
    auto pick = [&](auto height) -> hipError_t {
        constexpr int BM = decltype(height)::value;
        constexpr std::size_t kLds = gemm::DmaShape<BM>::kLdsBytes;
        if (with_addend) {
            if constexpr (BM == 320) {
                return hipErrorNotSupported;  // not chosen for an addend (see above)
            } else {
                return run(KernelConstant<gemm::gemm_dma_kernel<BM, true, false, false, false, true>>{}, kLds);
            }
        }
        auto with_flags = [&](auto with_bias, auto with_gelu, auto with_alpha) -> hipError_t {
            constexpr bool kB = decltype(with_bias)::value;
            constexpr bool kG = decltype(with_gelu)::value;
            constexpr bool kA = decltype(with_alpha)::value;
            return args.accumulate ? run(KernelConstant<gemm::gemm_dma_kernel<BM, kB, kG, kA, true>>{}, kLds)
                                   : run(KernelConstant<gemm::gemm_dma_kernel<BM, kB, kG, kA, false>>{}, kLds);
        };
        auto with_alpha = [&](auto with_bias, auto with_gelu) -> hipError_t {
            return args.alpha == 1.0F ? with_flags(with_bias, with_gelu, std::false_type{})
                                      : with_flags(with_bias, with_gelu, std::true_type{});
        };
        auto with_gelu = [&](auto with_bias) -> hipError_t {
            return args.gelu ? with_alpha(with_bias, std::true_type{}) : with_alpha(with_bias, std::false_type{});
        };
        return bias != nullptr ? with_gelu(std::true_type{}) : with_gelu(std::false_type{});
    };
    switch (choice.rows) {
    case 192: return pick(std::integral_constant<int, 192>{});
    case 256: return pick(std::integral_constant<int, 256>{});
    default: return pick(std::integral_constant<int, 320>{});
    }
}

hipError_t gemm_bf16(const std::uint16_t* a, const std::uint16_t* b, const float* bias,
                     std::uint16_t* c, const GemmArgs& args, hipStream_t stream) {
    // B as [N, K] with 16-byte rows: the persistent kernel (ViT-Base b64: FC1 +
    // GELU 78 us, QKV 52, FC2 accumulating 68, the projection 27) or the ring
    // kernel, whichever the costs above say is faster. A batch whose entries'
    // A rows follow one another and share B (the patch embedding) runs as one
    // problem of all the rows, so tiles do not stop at entry boundaries.
    const GemmArgs whole = as_one_problem(args);
    const bool split = whole.inner > 0;
    const bool vector_c = aligned16(c) && whole.n % 8 == 0 && whole.ldc % 8 == 0 && whole.stride_c % 8 == 0 &&
                          (!split || whole.outer_stride_c % 8 == 0);
    const int c_run = vector_c ? 8 : whole.n % 4 == 0 && vector_output(c, whole) ? 4 : 1;
    const bool addend_ok = whole.addend == nullptr ||
                           (vector_c && bias != nullptr && !whole.gelu && !whole.accumulate &&
                            aligned16(whole.addend) && whole.ld_addend % 4 == 0);
    if (whole.transposed && addend_ok &&
        vector_operand(a, whole.lda, whole.k, whole.stride_a, whole.outer_stride_a, split) &&
        vector_operand(b, whole.ldb, whole.k, whole.stride_b, whole.outer_stride_b, split) &&
        static_cast<std::int64_t>(128) * whole.lda * 2 < gemm::kMaxSpan &&
        static_cast<std::int64_t>(128) * whole.ldb * 2 < gemm::kMaxSpan) {
        const RingChoice ring = choose_ring(whole, compute_units());
        if (const hipError_t dma = launch_dma(a, b, bias, c, whole, ring, stream); dma != hipErrorNotSupported) {
            return dma;
        }
        return gemm_ring_bf16(ring.tile, a, b, bias, c, whole, ring.map, c_run, stream);
    }
    const std::int64_t units = compute_units();
    if (tile_count(args, 128, 128) >= units * 2) {
        // Up to K = 1024, 32-deep stages with registers for three workgroups
        // per CU; 64-deep stages beyond.
        if (args.k <= 1024) {
            return pick_flags<std::uint16_t, 2, 2, 2, 2, 32, 3>(a, b, bias, c, args, stream);
        }
        return pick_flags<std::uint16_t, 2, 2, 2, 2, 64>(a, b, bias, c, args, stream);
    }
    // 64 x 64: 32-deep stages for short K, 64-deep beyond.
    if (args.k <= 512) {
        return pick_flags<std::uint16_t, 2, 2, 1, 1, 32>(a, b, bias, c, args, stream);
    }
    return pick_flags<std::uint16_t, 2, 2, 1, 1, 64>(a, b, bias, c, args, stream);
}

} // namespace cuvit::detail
