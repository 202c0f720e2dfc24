// Internals for the Python tests: the GEMM dispatch rules (gemm_choice.hpp) for
// test_gemm_choice_cpu.py, which kernel and tile a problem takes on a card of
// `units` compute units, and how a batch is spread over launches; and the
// model's attention beyond 256 tokens by itself for test_long_attention_gpu.py.
#include "capi/status.hpp"
#include "kernels/gemm_choice.hpp"

using namespace cuvit::detail;

namespace {

GemmArgs problem(int m, int n, int k, int count, int gelu) {
    GemmArgs args{};
    args.m = m;
    args.n = n;
    args.k = k;
    args.count = count;
    args.transposed = true;
    args.alpha = 1.0F;
    args.gelu = gelu != 0;
    return args;
}

} // namespace

extern "C" {

/// A RingTile's number, or 100 + the tile height of the persistent kernel, for
/// operands that @p persistent_fits.
int bf16_choice(int m, int n, int k, int count, int gelu, int persistent_fits, int units) {
    const GemmArgs args = problem(m, n, k, count, gelu);
    const RingChoice ring = choose_ring(args, units);
    if (persistent_fits != 0) {
        const DmaChoice dma = choose_dma(args, units);
        if (!ring_beats_dma(args, ring, dma)) {
            return 100 + dma.rows;
        }
    }
    return static_cast<int>(ring.tile);
}

/// A RingTileF32's number, or 5 for the tiled kernel; @p rows_per_entry > 0:
/// entries run as one problem.
int f32_choice(int m, int n, int k, int count, int units, int rows_per_entry) {
    GemmArgs args = problem(m, n, k, count, 0);
    args.rows_per_entry = rows_per_entry;
    return tiled_beats_ring_f32(args, units) ? 5 : static_cast<int>(choose_ring_f32(args, units).tile);
}

int whole_entries(int count, long long tiles) { return entries_by_xcd(count, tiles) ? 1 : 0; }

/// The launches that a batch of @p count entries takes, or -1 if they don't
/// cover it in order, each within a grid (or are more than they can be).
int batch_launches(int count) {
    int launches = 0;
    long long covered = 0;
    const hipError_t status = for_entries(count, [&](int first, int entries) -> hipError_t {
        ++launches;
        if (first != covered || entries < 1 || entries > kMaxGridY || launches > 40000) {
            return hipErrorInvalidValue;
        }
        covered += entries;
        return hipSuccess;
    });
    return status == hipSuccess && covered == count ? launches : -1;
}

int long_attention_f32(const void* qkv, void* context, int images, int heads, int tokens, void* stream) {
    return cuvit::capi::attention_long(static_cast<const float*>(qkv), static_cast<float*>(context), images, heads,
                                       tokens, static_cast<hipStream_t>(stream));
}

int long_attention_bf16(const void* qkv, void* context, int images, int heads, int tokens, void* stream) {
    return cuvit::capi::attention_long(static_cast<const std::uint16_t*>(qkv), static_cast<std::uint16_t*>(context),
                                       images, heads, tokens, static_cast<hipStream_t>(stream));
}
}
