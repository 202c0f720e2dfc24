"""The model's attention beyond 256 tokens (attention_long.hip) against the
oracle's forward, at token counts around its block edges: one key past a block
(257 = 4 x 64 + 1, also past a 32-key block), tails up to 16, 32, 48 and 64
keys, the 384-pixel count (577), and query tiles that leave wavefronts idle.
Two blocks deep, so that every query's row reaches the logits; two heads and
three images, so that the pairs (6) do not fill the eight XCDs. Then the kernel
by itself against float64: more pairs than XCDs, more tokens, and the values at
which its running softmax takes another way than the launches do.

Tolerances: fp32 rtol = atol = 1e-4, the model tests' (vit_test.cu:128-130).
bf16: the error against the fp32 oracle over the three images' logits, at most
twice the bf16 oracle's own. The two round at the same points but for the
attention logits, which only the oracle rounds, so their errors are two draws
of the same size (about 3e-2 here: weights of standard deviation 0.2 at 128
columns amplify every rounding) and a norm over 21 logits spreads by well under
a factor of two, where a wrong row or key is an error near 1. Images of a batch
are bitwise the same images run alone.
"""

from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

from conftest import ROOT, to_device, to_host
from numerics import TestFailure, require_close, require_exact
from vit_support import random_image, random_weights, small_config, write_weights

pytestmark = pytest.mark.gpu

BF16_FACTOR = 2.0


def long_config(cuvit, side: int):
    config = small_config(cuvit)
    config.image_size = 4 * side
    config.patch_size = 4
    config.channels = 1
    config.embed_dim = 128
    config.depth = 2
    config.heads = 2
    config.mlp_hidden = 64
    config.classes = 7
    return config


@pytest.mark.parametrize("side", [16, 17, 18, 19, 20, 24], ids=lambda s: f"{s * s + 1}_tokens")
@pytest.mark.parametrize("precision", [0, 1], ids=["f32", "bf16"])
def test_model_beyond_256_tokens(cuvit, oracle, device, tmp_path, side, precision):
    config = long_config(cuvit, side)
    assert not cuvit.attention_supported(config.token_count(), config.head_dim())
    tensors = random_weights(cuvit, oracle, config, 900 + side)
    path = os.path.join(tmp_path, "long.cvw")
    write_weights(cuvit, tensors, path)
    model = cuvit.VisionTransformer(config, cuvit.WeightFile(path), 3, precision)
    images = [random_image(oracle, config, 70 + i) for i in range(3)]

    def forward(chosen):
        logits = torch.empty(len(chosen) * config.classes, device=device)
        model.forward(to_device(np.concatenate(chosen), device), logits, len(chosen))
        return to_host(logits).reshape(len(chosen), config.classes)

    together = forward(images)
    values = [t for _, t in tensors]
    full = np.stack([oracle.vit_forward(config, values, image) for image in images])
    for i, image in enumerate(images):
        require_exact(together[i], forward([image])[0], "an image in a batch differs from the image alone")
    if precision == 0:
        require_close(together, full, "forward beyond 256 tokens", 1.0e-4, 1.0e-4)
        return
    reduced = np.stack([oracle.vit_forward(config, values, image, bf16=True) for image in images])
    error = np.linalg.norm(together.astype(np.float64) - full)
    bound = BF16_FACTOR * np.linalg.norm(reduced.astype(np.float64) - full)
    print(f"{config.token_count()} tokens: error {error:.2e}, bound {bound:.2e}, logits {np.linalg.norm(full):.2e}")
    if not error <= bound:
        raise TestFailure(f"bf16 forward beyond 256 tokens: error {error:.3e} above {bound:.3e}")


@pytest.fixture(scope="module")
def internals():
    library = os.path.join(ROOT, "tests", "cpp", "bin", "libinternals.so")
    if not os.path.exists(library):
        subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "tests", "cpp")], check=True)
    library = ctypes.CDLL(library)
    for entry in (library.long_attention_f32, library.long_attention_bf16):
        entry.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int] * 3 + [ctypes.c_void_p]
    return library


def attend(internals, qkv, device):
    """[images, tokens, 3, heads, 64] on the CPU -> the kernel's context there."""
    images, tokens, _, heads, _ = qkv.shape
    source = qkv.to(device)
    context = torch.full((images, tokens, heads, 64), -7.0, dtype=qkv.dtype, device=device)
    entry = internals.long_attention_bf16 if qkv.dtype == torch.bfloat16 else internals.long_attention_f32
    assert entry(source.data_ptr(), context.data_ptr(), images, heads, tokens,
                 torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    return context.cpu()


def require_attention(actual, qkv, exact_logits=False):
    """Against float64, NaN where it has NaN.

    With x the logits and A = sum w |v|: an fp32 logit is off by 66 roundings of
    its 64 terms' sizes and the exponent's product and sum by two of its own
    (all over 8), which shifts weights and their sum alike, so twice that times
    A; the sums of fp32 weights and products add a rounding a block and a few
    for the exponential and the division. bf16, with 8 significant bits, adds a
    rounding of the weights and one of the result, 2^-8 of their sizes each.
    With @p exact_logits (one term each, the largest ones alike) none is off."""
    q, k, v = (qkv[:, :, i].double().transpose(1, 2) for i in range(3))
    x = q @ k.transpose(2, 3).contiguous() / 8
    sizes = q.abs() @ k.abs().transpose(2, 3).contiguous() / 8
    w = torch.softmax(x, -1)
    expected = w @ v
    magnitude = w @ v.abs()
    tokens = qkv.shape[1]
    # Keys without weight do not matter, however large their terms.
    shift = torch.where(w > 1e-30, 68 * 2.0 ** -24 * sizes, torch.zeros(())).amax(-1, keepdim=True)
    if exact_logits:
        shift = torch.zeros_like(shift)
    relative = 2 * shift + (tokens / 32 + 16) * 2.0 ** -24
    if qkv.dtype == torch.bfloat16:
        relative = relative + 2.0 ** -7
    got = actual.double().transpose(1, 2)
    differing = got.isnan() != expected.isnan()
    assert int(differing.sum()) == 0, differing.nonzero()[0].tolist()
    limit = relative * magnitude + 1e-37
    bad = ~((got - expected).abs() <= limit) & ~expected.isnan()
    assert int(bad.sum()) == 0, (bad.nonzero()[0].tolist(), float(got[bad][0]), float(expected[bad][0]))


def random_qkv(seed, images, tokens, heads, dtype):
    generator = torch.Generator().manual_seed(seed)
    return torch.randn((images, tokens, 3, heads, 64), generator=generator).to(dtype)


TYPES = pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])


@TYPES
@pytest.mark.parametrize("images,heads,tokens", [(1, 9, 257), (3, 4, 300), (5, 5, 289), (1, 2, 1025), (1, 1, 2100)])
def test_kernel_against_float64(internals, device, images, heads, tokens, dtype):
    """Second and third pairs of an XCD, a last XCD without one, more tokens."""
    qkv = random_qkv(tokens + heads, images, tokens, heads, dtype)
    require_attention(attend(internals, qkv, device), qkv)


@TYPES
@pytest.mark.parametrize("step", [0.05, 0.5, -0.5], ids=["some", "every_block", "first_block"])
def test_maximum_that_rises_along_the_keys(internals, device, step, dtype):
    """Logits that grow with the key: the accumulated sums are rescaled in later
    blocks, in both halves of a block and where the halves are added up."""
    qkv = random_qkv(11, 2, 333, 2, dtype)
    qkv[:, :, 0, :, 0] = 8.0
    qkv[:, :, 1, :, 0] = (step * torch.arange(333.0)).to(dtype)[None, :, None]
    require_attention(attend(internals, qkv, device), qkv)


@TYPES
def test_infinite_and_missing_logits(internals, device, dtype):
    """Queries whose logits are -inf for whole blocks, for all keys but one, for
    all keys (NaN), +inf for one key (NaN), NaN, or the type's lowest value."""
    tokens, lowest = 300, torch.finfo(dtype).min
    qkv = random_qkv(12, 1, tokens, 1, dtype)
    qkv[:, :, :2, :, 0] = 0  # the masks' dim
    # Whole blocks first, all keys but the last, all of them, a block in the
    # middle, one half of every block.
    masks = [lambda key: key < 200, lambda key: key != 299, lambda key: key >= 0, lambda key: (key >= 64) & (key < 128),
             lambda key: (key // 32) % 2 == 0]
    keys = torch.arange(tokens)
    for value in (-float("inf"), lowest):
        batch = qkv.repeat(len(masks), 1, 1, 1, 1)
        batch[:, :, 0, :, 0] = 1
        for i, mask in enumerate(masks):
            batch[i, mask(keys), 1, :, 0] = value
        require_attention(attend(internals, batch, device), batch)
    for value in (float("inf"), float("nan")):
        batch = qkv.clone()
        batch[:, :, 0, :, 0] = 1
        batch[0, 40, 0, 0, 0] = value  # one query only
        batch[:, :, 1, :, 0] = 1
        require_attention(attend(internals, batch, device), batch)


@TYPES
def test_values_near_the_largest(internals, device, dtype):
    """Sums of unnormalised weights times V overflow where the context does not."""
    tokens = 300
    qkv = random_qkv(15, 2, tokens, 3, dtype)
    qkv[0, :, 2] = 3e38  # every query of image 0
    qkv[1, 17:20, 2, 1] = -3.2e38  # three keys of one pair
    qkv[1, 100, 2, 1, :32] = 3.2e38
    require_attention(attend(internals, qkv, device), qkv)
    # An infinite value stays one.
    qkv[1, 30, 2, 2, 5] = float("inf")
    context = attend(internals, qkv, device)
    assert bool(torch.isinf(context[1, :, 2, 5]).all())
    assert bool(torch.isfinite(context[1, :, 2, 6:]).all())


@TYPES
@pytest.mark.parametrize("size", [1e3, 1e7, 1e10, 1e15, 1e30, -1e10, -1e30])
def test_large_logits(internals, device, size, dtype):
    """Where the exponent's shift is rounded by more than the weights differ.
    Every key has the same large logit, or half of them -size."""
    for second in (1.0, -1.0):
        qkv = random_qkv(16, 1, 290, 2, dtype)
        qkv[:, :, :2] = 0
        qkv[:, :, 0, :, 3] = 2.0 ** round(np.log2(abs(size)) / 2)
        qkv[:, :, 1, :, 3] = size / 2.0 ** round(np.log2(abs(size)) / 2)
        qkv[:, 100:245, 1, :, 3] *= second
        require_attention(attend(internals, qkv, device), qkv, exact_logits=True)
