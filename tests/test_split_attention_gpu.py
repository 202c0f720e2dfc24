"""Fused fp32 attention of few (image, head) pairs, which runs one query tile
per workgroup, against the whole-tile kernel that many pairs take: the same
bits for every count of key tiles, full and ragged."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key_tiles", range(1, 17))
def test_few_pairs_equal_many_pairs(cuvit, device, key_tiles):
    heads, images = 12, 80  # 960 pairs: beyond the line at every count of key tiles
    for tokens in sorted({16 * key_tiles - 15, 16 * key_tiles - 7, 16 * key_tiles}):
        generator = torch.Generator(device="cpu").manual_seed(tokens)
        qkv = torch.randn((images, tokens, 3, heads, 64), generator=generator).to(device)
        many = torch.full((images, tokens, heads, 64), float("nan"), device=device)
        cuvit.attention(qkv, many, images, heads, tokens, 64)
        for image in (0, images - 1):  # 12 pairs at a time
            few = torch.full((1, tokens, heads, 64), float("nan"), device=device)
            cuvit.attention(qkv[image:image + 1].contiguous(), few, 1, heads, tokens, 64)
            torch.cuda.synchronize()
            assert torch.equal(few.view(torch.int32), many[image:image + 1].view(torch.int32))
        assert not bool(many.isnan().any())
