// Internals for the Python tests: the GEMM dispatch rules (gemm_choice.hpp) for
// test_gemm_choice_cpu.py, which kernel and tile a problem takes on a card of
// `units` compute units.
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
}
