"""The native half of the Python binding: it takes every launcher's plain case
itself, and a GEMM only where the Python checks let it through."""

from __future__ import annotations

import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_plain_calls_are_taken(cuvit, device):
    native = cuvit._native_calls
    for dtype in (torch.float32, torch.bfloat16):
        x, out = torch.randn(6, 8, device=device).to(dtype), torch.empty(6, 8, dtype=dtype, device=device)
        row = torch.ones(8, device=device)
        problem = cuvit.gemm_problem(6, 6, 8, cuvit.TRANSPOSED)
        square = torch.empty(6, 6, dtype=dtype, device=device)
        qkv = torch.randn(1, 5, 3, 2, 64, device=device).to(dtype)
        context = torch.empty(1, 5, 2, 64, dtype=dtype, device=device)
        images = torch.randn(1, 3, 8, 8, device=device).to(dtype)
        for stream in (None, torch.cuda.Stream()):
            assert native.layer_norm(x, row, row, out, 6, 8, 1e-6, stream, None) == 0
            assert native.softmax(x, out, 6, 8, stream, dtype == torch.bfloat16) == 0
            assert native.gemm(x, x, row, square, problem, stream, None) == 0
            assert native.attention(qkv, context, 1, 2, 5, 64, stream) == 0
            assert native.extract_patches(images, torch.empty_like(images), 1, 3, 8, 8, 4, stream, None) == 0
    pixels = torch.zeros(1, 9, 7, 3, dtype=torch.uint8, device=device)
    assert native.preprocess(pixels, torch.empty(1, 3, 4, 4, device=device), 1, 7, 9, cuvit.Preprocessing(4), None) == 0
    torch.cuda.synchronize()


def test_what_is_not_plain_is_left_to_python(cuvit, device):
    class Sub(torch.Tensor):
        pass

    x = torch.randn(4, 8, device=device)
    native = cuvit._native_calls
    for operand in (x.data_ptr(), None, x.cpu(), x.double(), x.t(), x[:3], x.as_subclass(Sub)):
        assert native.softmax(operand, x, 4, 8, None, False) == -1
        assert native.softmax(x, operand, 4, 8, None, False) == -1
    # An address and a subclass are the Python code's to take; the rest it refuses.
    expected = torch.softmax(x, -1)
    for operand in (x.data_ptr(), x.as_subclass(Sub)):
        out = torch.empty_like(x)
        cuvit.softmax(operand, out, 4, 8, bf16=False)
        torch.cuda.synchronize()
        assert torch.allclose(out, expected, atol=1e-6)
    for operand in (None, x.cpu(), x.double(), x.t(), x[:3]):
        with pytest.raises(cuvit.InvalidArgument):
            cuvit.softmax(operand, torch.empty_like(x), 4, 8, bf16=False)


@pytest.mark.parametrize("layout", [0, 1], ids=["no_transpose", "transposed"])
def test_gemm_checks_agree(cuvit, device, layout):
    """One element short of what a problem reaches, in each operand, over flat,
    split and shared batches, padded rows and bad strides."""
    m, n, k = 3, 5, 4
    b_rows, b_columns = (n, k) if layout == cuvit.TRANSPOSED else (k, n)
    batches = [(1, 0), (4, 0), (6, 3), (6, 6), (6, 8), (4, 1)]  # (count, inner)
    for (count, inner), pad, stride, short in itertools.product(batches, (0, 3), (0, 40, -1), "-abc"):
        problem = cuvit.gemm_problem(m, n, k, layout)
        problem.lda, problem.ldb, problem.ldc = k + pad, b_columns + pad, n + pad
        batch = problem.batch
        batch.count, batch.inner = count, inner
        batch.stride_a = batch.stride_b = stride
        batch.stride_c = 40
        batch.outer_stride_a, batch.outer_stride_b, batch.outer_stride_c = stride, 2 * stride, 120
        sizes = {}
        for name, rows, ld, columns in (("a", m, k + pad, k), ("b", b_rows, b_columns + pad, b_columns),
                                        ("c", m, n + pad, n)):
            _, high = cuvit._offset_range(count, inner, getattr(batch, "stride_" + name),
                                          getattr(batch, "outer_stride_" + name))
            sizes[name] = max(1, high + (rows - 1) * ld + columns) - (short == name)
        a, b, c = (torch.zeros(max(0, sizes[name]), device=device) for name in "abc")
        try:
            cuvit._gemm_operands(a, b, None, c, problem, False)
            refused = False
        except cuvit.InvalidArgument:
            refused = True
        status = cuvit._native_calls.gemm(a, b, None, c, problem, None, None)
        # A negative stride that no entry reaches with is legal, and Python's to take.
        taken = status >= 0
        assert taken == (not refused and stride >= 0), (count, inner, pad, stride, short, status)
    torch.cuda.synchronize()
