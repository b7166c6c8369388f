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


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16, torch.float16))
@pytest.mark.parametrize("tg,g", [(tg, g) for tg in (8, 16, 32, 64, 128) for g in (16, 32, 64)])
def test_pack_of_one_group_bit_exact(tg, g, dtype):
    """One token group, the line between its own workgroup and a row block
    (64 rows) among its lengths, encoded in place behind two sealed groups."""
    for tokens in sorted({1, tg // 2 + 1, min(tg, 63), min(tg, 64), min(tg, 65), tg}):
        gen = torch.Generator().manual_seed(tokens + tg + g)
        keys = torch.randn(3, tokens, 128, generator=gen).to(dtype)
        cap, offset = 4 * tg, 2 * tg
        packed = popkv_cuda.pack_keys(torch.zeros(3, cap, 128, dtype=dtype, device=DEV), token_group_size=tg,
                                      dim_group_size=g)
        before = [_bits(p) for p in packed]
        popkv_cuda.pack_keys_into(keys.to(DEV), packed, token_offset=offset, token_group_size=tg, dim_group_size=g)
        want = core.pack_keys(keys.float().numpy(), token_group_size=tg, dim_group_size=g)
        for got, expected, old in zip(packed, want, before):
            old[:, offset:offset + tokens] = expected
            assert np.array_equal(_bits(got), old), (tokens, got.dtype)


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16, torch.float16))
@pytest.mark.parametrize("dim,tg,g", [(32, 8, 16), (64, 32, 32), (64, 24, 32), (64, 64, 64), (64, 8, 16), (96, 32, 16),
                                      (96, 64, 32), (160, 40, 32), (192, 64, 64), (256, 16, 16), (256, 64, 32)])
def test_pack_rows_of_other_head_sizes_bit_exact(dim, tg, g, dtype):
    """Row blocks of head sizes other than 128 (fp32 rows of 192 and 256 dimensions
    do not fit them): one row, the edges of stripes, groups and blocks, an
    offset into a larger cache, the largest values and zeros of both
    signs in the keys; exact."""
    rows = 64 // tg * tg
    for tokens in (1, 7, 9, rows - 1, rows, rows + 1, 2 * rows + tg + 1):
        gen = torch.Generator().manual_seed(tokens + tg + g + dim)
        keys = torch.randn(3, tokens, dim, generator=gen)
        keys[:, ::5, 3] *= 10.0
        keys[:, ::3, 5] = 0.0
        keys[:, 1::3, 5] = -0.0
        keys[1, tokens // 2, 7] = torch.finfo(dtype).max
        keys[2, tokens // 2, 9] = -torch.finfo(dtype).max
        keys = keys.to(dtype)
        cap, offset = tokens + 2 * tg + 3, 2 * tg
        packed = popkv_cuda.pack_keys(torch.zeros(3, cap, dim, dtype=dtype, device=DEV), token_group_size=tg,
                                      dim_group_size=g)
        before = [_bits(p) for p in packed]
        popkv_cuda.pack_keys_into(keys.to(DEV), packed, token_offset=offset, token_group_size=tg, dim_group_size=g)
        want = core.pack_keys(keys.float().numpy(), token_group_size=tg, dim_group_size=g)
        for got, expected, old in zip(packed, want, before):
            bits = _bits(got)
            assert np.array_equal(bits[:, offset:offset + tokens], expected), (tokens, got.dtype)
            assert np.array_equal(bits[:, :offset], old[:, :offset])
            assert np.array_equal(bits[:, offset + tokens:], old[:, offset + tokens:])
