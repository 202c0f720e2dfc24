"""The model's attention beyond 256 tokens (attention_long.hip) against the
oracle's forward, at token counts around its block edges: one key past a block
(257 = 4 x 64 + 1, also past a 32-key block), tails up to 16, 32, 48 and 64
keys, the 384-pixel count (577), and query tiles that leave wavefronts idle.
Two blocks deep, so that every query's row reaches the logits; two heads and
three images, so that the pairs (6) do not fill the eight XCDs.

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

import os

import numpy as np
import pytest
import torch

from conftest import to_device, to_host
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
