"""The LDS-ring GEMM in every tile that the dispatch takes (bf16 64 x 32 to 128
x 128, fp32 32 x 16 to 64 x 64; test_gemm_choice_cpu.py checks that each case
below reaches the tile it names), which products with B as [N, K] and 16-byte
operand rows take where the persistent kernel and the panels do not.

The tiled kernel, which B as [K, N] takes, runs the same MFMA over the same
k-blocks in the same order and rounds every step of the epilogue alike, so the
two layouts of one B must give the same bits. Each result is also judged
against float64, and what lies past N in C's rows must keep its values.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def normal(seed, shape, stddev, device, dtype=torch.bfloat16):
    generator = torch.Generator(device="cpu").manual_seed(seed)
    return (torch.randn(shape, generator=generator) * stddev).to(dtype).to(device)


def run(cuvit, a, b, bias, c, problem, transposed):
    problem.layout = cuvit.TRANSPOSED if transposed else cuvit.NO_TRANSPOSE
    cuvit.gemm(a, b, bias, c, problem)
    torch.cuda.synchronize()


CASES = [
    # m, n, k, bias, gelu, accumulate, alpha, C's padding, tile
    (1, 8, 8, True, False, False, 1.0, 0, "64x32 alone"),            # one row, one chunk of K
    (63, 64, 64, True, True, False, 1.0, 0, "64x32 alone"),          # a row short of a tile
    (65, 72, 136, True, False, True, 1.0, 8, "64x32 alone"),         # a row and a chunk past; K past one span
    (64, 65, 128, True, False, True, 1.0, 0, "64x32 alone"),         # odd N: element-wise C, accumulating
    (65, 76, 136, True, False, True, 1.0, 0, "64x32 alone"),         # C in 8-byte pieces, half a chunk at N
    (130, 132, 72, True, True, False, 1.0, 4, "64x32 alone"),        # the same, padded rows
    (130, 199, 72, False, True, False, -0.5, 3, "64x32 alone"),      # odd rows of C, GELU without bias, alpha
    (197, 768, 3080, True, False, True, 1.0, 0, "64x32 alone"),      # long K
    (65, 2304, 128, True, True, True, 1.0, 0, "64x32 alone"),        # one span of K
    (197, 2304, 776, True, False, False, 1.0, 0, "64x64 alone"),     # loading wavefronts
    (1576, 1536, 200, True, False, True, 1.0, 0, "64x64"),           # several tiles a CU
    (4616, 1540, 384, True, False, True, 1.0, 0, "64x64"),           # C in 8-byte pieces
    (3152, 776, 1032, True, False, True, 1.0, 0, "64x64"),           # N and K off the grid
    (1576, 768, 1032, True, False, True, 1.0, 0, "64x64 deep"),      # three stages
    (1576, 2304, 200, True, False, False, 1.0, 0, "128x64"),
    (1571, 3064, 64, True, True, True, 1.0, 1, "128x64"),            # odd rows of C
    (6304, 1152, 384, True, False, False, 1.0, 0, "128x128"),
    (6301, 1145, 200, True, False, True, 1.0, 1, "128x128"),         # accumulating, odd N and rows of C
    (6304, 1148, 384, False, False, True, 0.5, 0, "128x128"),        # C in 8-byte pieces, accumulating
    (4616, 1536, 384, True, True, False, 1.0, 0, "128x128"),         # where the persistent kernel could run
    (4616, 768, 1032, True, False, True, 1.0, 0, "128x128 deep"),    # three stages, accumulating
    (4611, 757, 1032, False, True, False, 1.0, 3, "128x128 deep"),   # tails, odd rows of C
]


@pytest.mark.parametrize("m,n,k,with_bias,gelu,accumulate,alpha,pad", [case[:-1] for case in CASES])
def test_ring_equals_the_tiled_kernel(cuvit, device, m, n, k, with_bias, gelu, accumulate, alpha, pad):
    a = normal(m + k, (m, k), 1.0, device)
    b = normal(n + k, (n, k), 0.05, device)
    bias = normal(n, (n,), 0.5, device, torch.float32) if with_bias else None
    start = normal(7, (m, n + pad), 1.0, device) if accumulate else \
        torch.full((m, n + pad), float("nan"), dtype=torch.bfloat16, device=device)
    results = []
    for transposed in (True, False):
        problem = cuvit.gemm_problem(m, n, k, cuvit.TRANSPOSED)
        problem.alpha, problem.ldc = alpha, n + pad
        problem.epilogue.gelu, problem.epilogue.accumulate = int(gelu), int(accumulate)
        c = start.clone()
        run(cuvit, a, b if transposed else b.t().contiguous(), bias, c, problem, transposed)
        results.append(c.cpu().view(torch.int16))
    assert torch.equal(results[0], results[1])
    assert torch.equal(results[0][:, n:], start.cpu().view(torch.int16)[:, n:])

    a64, b64 = a.cpu().double(), b.cpu().double()
    expected = alpha * (a64 @ b64.t())
    scale = abs(alpha) * (a64.abs() @ b64.abs().t())
    if with_bias:
        expected = expected + bias.cpu().double()
    if gelu:
        expected = torch.nn.functional.gelu(expected)
    if accumulate:
        expected = expected + start.cpu().double()[:, :n]
    actual = results[0].view(torch.bfloat16)[:, :n].double()
    # One rounding to bf16 (2^-9, doubled), fp32 sums of k terms (k 2^-24 of
    # their sizes at most, GELU's slope at most 1.13) and the GELU's own 4e-7.
    limit = 2.0 ** -8 * expected.abs() + 1.2 * (k + 4) * 2.0 ** -24 * (scale + 1.0) + 1e-6
    assert bool(((actual - expected).abs() <= limit).all())


@pytest.mark.parametrize("count,inner,m,n,k", [(3, 0, 70, 72, 64), (6, 3, 33, 64, 72), (6, 2, 65, 65, 64),
                                                (65537, 0, 2, 8, 8), (8, 0, 70, 136, 64), (16, 4, 130, 65, 72),
                                                (75, 5, 33, 76, 64), (80, 0, 257, 168, 128)])
def test_ring_batches(cuvit, device, count, inner, m, n, k):
    """Batch entries of their own A, B and C, flat and split, more than one
    launch's, and dealt to the XCDs whole (from 8 on, evenly or nearly so)."""
    a, b = normal(1, (count, m, k), 1.0, device), normal(2, (count, n, k), 0.1, device)
    results = []
    for transposed in (True, False):
        problem = cuvit.gemm_problem(m, n, k, cuvit.TRANSPOSED)
        problem.batch.count, problem.batch.inner = count, inner
        problem.batch.stride_a, problem.batch.stride_b, problem.batch.stride_c = m * k, n * k, m * n
        if inner:
            problem.batch.outer_stride_a = inner * m * k
            problem.batch.outer_stride_b = inner * n * k
            problem.batch.outer_stride_c = inner * m * n
        c = torch.full((count, m, n), float("nan"), dtype=torch.bfloat16, device=device)
        operand = b if transposed else b.transpose(1, 2).contiguous()
        run(cuvit, a, operand, None, c, problem, transposed)
        results.append(c.cpu().view(torch.int16))
    assert torch.equal(results[0], results[1])
    assert not bool(results[0].view(torch.bfloat16).isnan().any())


def test_ring_runs_a_shared_weight_batch_as_one_problem(cuvit, device):
    """Entries that share B and follow one another in A, stored back apart."""
    count, m, n, k, gap = 5, 49, 72, 64, 3
    a, b = normal(3, (count, m, k), 1.0, device), normal(4, (n, k), 0.1, device)
    bias = normal(5, (n,), 0.5, device, torch.float32)
    start = normal(6, (count, (m + gap) * n), 1.0, device)
    for accumulate in (0, 1):
        c = start.clone()
        problem = cuvit.gemm_problem(m, n, k, cuvit.TRANSPOSED)
        problem.batch.count = count
        problem.batch.stride_a, problem.batch.stride_c = m * k, (m + gap) * n
        problem.epilogue.accumulate = accumulate
        run(cuvit, a, b, bias, c, problem, True)
        one = cuvit.gemm_problem(m, n, k, cuvit.NO_TRANSPOSE)
        one.epilogue.accumulate = accumulate
        for i in range(count):
            expected = start[i].clone()
            run(cuvit, a[i], b.t().contiguous(), bias, expected, one, False)
            assert np.array_equal(c[i].cpu().view(torch.int16).numpy(), expected.cpu().view(torch.int16).numpy())


F32_CASES = [
    # m, n, k, bias, gelu, accumulate, alpha, C's padding, tile
    (1, 8, 4, True, False, False, 1.0, 0, "32x16 alone"),            # one chunk of K
    (31, 33, 64, True, True, False, 1.0, 3, "32x16 alone"),          # odd rows of C
    (33, 65, 68, True, False, True, 1.0, 0, "32x16 alone"),          # past a tile, past a span of K; a run that N cuts
    (197, 192, 772, False, False, True, -0.5, 4, "32x16 alone"),
    (230, 640, 772, True, False, False, 1.0, 0, "32x32 deep"),       # three stages
    (788, 384, 320, True, True, True, 1.0, 0, "32x32 deep"),         # several tiles a CU
    (3151, 1540, 196, False, True, False, 2.0, 0, "32x32"),          # many tiles a CU, GELU without bias
    (1003, 1152, 100, True, False, False, 1.0, 0, "32x32"),          # two stages, tails
    (394, 2302, 100, True, True, True, 0.5, 1, "64x32"),             # tails, odd rows of C
    (3151, 1541, 100, False, False, True, 1.0, 0, "64x64"),          # tails, odd N
    (5001, 1540, 1028, True, False, False, 1.0, 0, "64x64"),         # a long K
]


@pytest.mark.parametrize("m,n,k,with_bias,gelu,accumulate,alpha,pad", [case[:-1] for case in F32_CASES])
def test_f32_ring_equals_the_tiled_kernel(cuvit, device, m, n, k, with_bias, gelu, accumulate, alpha, pad):
    a = normal(m + k, (m, k), 1.0, device, torch.float32)
    b = normal(n + k, (n, k), 0.05, device, torch.float32)
    bias = normal(n, (n,), 0.5, device, torch.float32) if with_bias else None
    start = normal(7, (m, n + pad), 1.0, device, torch.float32) if accumulate else \
        torch.full((m, n + pad), float("nan"), device=device)
    results = []
    for transposed in (True, False):
        problem = cuvit.gemm_problem(m, n, k, cuvit.TRANSPOSED)
        problem.alpha, problem.ldc = alpha, n + pad
        problem.epilogue.gelu, problem.epilogue.accumulate = int(gelu), int(accumulate)
        c = start.clone()
        run(cuvit, a, b if transposed else b.t().contiguous(), bias, c, problem, transposed)
        results.append(c.cpu().view(torch.int32))
    assert torch.equal(results[0], results[1])
    assert torch.equal(results[0][:, n:], start.cpu().view(torch.int32)[:, n:])

    a64, b64 = a.cpu().double(), b.cpu().double()
    expected = alpha * (a64 @ b64.t())
    scale = abs(alpha) * (a64.abs() @ b64.abs().t())
    if with_bias:
        expected = expected + bias.cpu().double()
    if gelu:
        expected = torch.nn.functional.gelu(expected)
    if accumulate:
        expected = expected + start.cpu().double()[:, :n]
    actual = results[0].view(torch.float32)[:, :n].double()
    # fp32 sums of k terms (k 2^-24 of their sizes at most, GELU's slope at
    # most 1.13), a few roundings of the result and the GELU's own 4e-7.
    limit = 2.0 ** -22 * expected.abs() + 1.2 * (k + 4) * 2.0 ** -24 * (scale + 1.0) + 1e-6
    assert bool(((actual - expected).abs() <= limit).all())


@pytest.mark.parametrize("count,inner,m,n,k", [(3, 0, 33, 36, 68), (6, 3, 50, 50, 64), (4, 2, 17, 65, 64),
                                                (65537, 0, 2, 8, 4), (8, 0, 70, 136, 64), (16, 4, 50, 65, 68),
                                                (75, 5, 33, 76, 64), (80, 0, 257, 168, 128)])
def test_f32_ring_batches(cuvit, device, count, inner, m, n, k):
    a, b = normal(1, (count, m, k), 1.0, device, torch.float32), normal(2, (count, n, k), 0.1, device, torch.float32)
    results = []
    for transposed in (True, False):
        problem = cuvit.gemm_problem(m, n, k, cuvit.TRANSPOSED)
        problem.batch.count, problem.batch.inner = count, inner
        problem.batch.stride_a, problem.batch.stride_b, problem.batch.stride_c = m * k, n * k, m * n
        if inner:
            problem.batch.outer_stride_a = inner * m * k
            problem.batch.outer_stride_b = inner * n * k
            problem.batch.outer_stride_c = inner * m * n
        c = torch.full((count, m, n), float("nan"), device=device)
        run(cuvit, a, b if transposed else b.transpose(1, 2).contiguous(), None, c, problem, transposed)
        results.append(c.cpu().view(torch.int32))
    assert torch.equal(results[0], results[1])
    assert not bool(results[0].view(torch.float32).isnan().any())
