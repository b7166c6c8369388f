"""The 64-row prepack (token groups of 8 to 128 tokens) against the oracle,
bit for bit, at the edges of its row blocks and groups."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import core
from popkv_amd import popkv_cuda

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _bits(t: torch.Tensor) -> np.ndarray:
    t = t.cpu().contiguous()
    return t.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.float16 else t.numpy()


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16, torch.float16))
@pytest.mark.parametrize("tg,g", [(tg, g) for tg in (8, 16, 32, 64, 128) for g in (16, 32, 64)])
def test_pack_row_blocks_bit_exact(tg, g, dtype):
    """One row, a block short of / at / past its 64 (128) rows, a last group
    of one row behind whole blocks; every form is exact, so no tolerance."""
    rows = max(64, tg)
    for tokens in (1, rows - 1, rows, rows + 1, 2 * rows + tg + 1):
        gen = torch.Generator().manual_seed(tokens + tg + g)
        keys = torch.randn(3, tokens, 128, generator=gen).to(dtype)
        keys[:, ::5, 3] *= 10.0
        packed = popkv_cuda.pack_keys(keys.to(DEV), token_capacity=tokens + 7, token_group_size=tg, dim_group_size=g)
        want = core.pack_keys(keys.float().numpy(), token_group_size=tg, dim_group_size=g)
        for got, expected in zip(packed, want):
            assert np.array_equal(_bits(got)[:, :tokens], expected), (tokens, got.dtype)
