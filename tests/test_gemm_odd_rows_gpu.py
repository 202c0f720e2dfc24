"""fp32 products whose operand rows start at any float, in the tiled kernel's
ways of loading them: 16 bytes at once through the buffer resources, with a
stage that K or N cuts element by element, and element by element throughout
(a short K and many tiles). The same operands with K and N padded by zeros to
whole 16-byte rows take the vector loads, and a zero more in a sum of products
changes no bit.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transposed", [False, True], ids=["no_transpose", "transposed"])
@pytest.mark.parametrize("m,n,k,count", [
    (1, 1, 1, 1),
    (33, 37, 18, 3),          # both cut, below one stage
    (70, 64, 50, 2),          # N whole: vector B as [K, N]
    (70, 31, 64, 2),          # K whole: vector A
    (65, 98, 577, 2),         # many stages, the last one cut
    (31, 130, 35, 4),         # three elements past a stage
    (197, 130, 197, 60),      # 64 x 64 tiles
    (577, 98, 50, 96),        # many tiles, short K: element by element
    (3001, 577, 127, 4),      # the longest K of those with B as [K, N]
    (3001, 577, 63, 4),       # and as [N, K]
])
def test_odd_rows_equal_padded_rows(cuvit, device, m, n, k, count, transposed):
    generator = torch.Generator(device="cpu").manual_seed(m + n + k)
    a = torch.randn((count, m, k), generator=generator).to(device)
    b = torch.randn((count, n, k) if transposed else (count, k, n), generator=generator).to(device)
    start = torch.randn((count, m, n), generator=generator).to(device)

    def run(a, b, c, n, k, accumulate):
        problem = cuvit.gemm_problem(m, n, k, cuvit.TRANSPOSED if transposed else cuvit.NO_TRANSPOSE)
        batch = problem.batch
        batch.count, batch.stride_a, batch.stride_b, batch.stride_c = count, m * k, n * k, m * n
        problem.epilogue.accumulate = accumulate
        cuvit.gemm(a, b, None, c, problem)
        torch.cuda.synchronize()

    pad_n, pad_k = -n % 4, -k % 4
    pad = torch.nn.functional.pad
    padded_a = pad(a, (0, pad_k)).contiguous()
    padded_b = pad(b, (0, pad_k, 0, pad_n) if transposed else (0, pad_n, 0, pad_k)).contiguous()
    for accumulate in (0, 1):
        c = start.clone() if accumulate else torch.full_like(start, float("nan"))
        padded_c = pad(c, (0, pad_n)).contiguous()
        run(a, b, c, n, k, accumulate)
        run(padded_a, padded_b, padded_c, n + pad_n, k + pad_k, accumulate)
        assert torch.equal(c.view(torch.int32), padded_c[:, :, :n].contiguous().view(torch.int32))
    a64, b64 = a[-1].cpu().double(), b[-1].cpu().double()
    b64 = b64.t().contiguous() if transposed else b64
    # fp32 sums of k terms and the sum with C.
    limit = (k + 2) * 2.0 ** -24 * (a64.abs() @ b64.abs() + start[-1].cpu().double().abs())
    assert bool(((c[-1].cpu().double() - (start[-1].cpu().double() + a64 @ b64)).abs() <= limit).all())
