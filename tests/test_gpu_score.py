"""The matrix-core scorer against the oracle, bit for bit: ragged ends of its
64-token groups, waves and spans, every representative size, and the batched
step whose sequences end inside other spans."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import core
from popkv_amd import batch as pb
from popkv_amd import popkv, popkv_cuda

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _u16(t: torch.Tensor) -> np.ndarray:
    return t.cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _planes(packed):
    return (packed[0].cpu().numpy(), packed[1].cpu().numpy(), _u16(packed[2]), _u16(packed[3]))


@pytest.mark.parametrize("g", (16, 32, 64))
@pytest.mark.parametrize("kv_heads,qpk,tokens", [(2, 8, 1), (3, 8, 63), (2, 8, 65), (1, 8, 513), (5, 8, 1999),
                                                 (2, 4, 577), (8, 4, 49217)])
def test_scores_bit_exact_at_group_and_span_edges(kv_heads, qpk, tokens, g):
    """Groups of four heads at G64 and G32 take the matrix cores only from
    384K (row, token) pairs on (the last shape); integer counts and one fp32
    chain, so the comparison is exact.  Two batches, a mapping that is not the
    standard one, and rows of infinite and NaN keys."""
    gen = torch.Generator().manual_seed(tokens + g + qpk)
    keys = torch.randn(kv_heads, tokens, 128, generator=gen)
    keys[:, :, 5] *= 10.0
    if tokens > 64:
        keys[0, 17], keys[0, 33, 2] = float("inf"), float("nan")
    packed = popkv_cuda.pack_keys(keys.to(DEV), token_group_size=32 if g == 32 else 64, dim_group_size=g)
    q = torch.randn(2, kv_heads * qpk, 128, generator=gen).to(DEV)
    mapping = (kv_heads - 1 - torch.arange(kv_heads * qpk) // qpk).to(DEV)
    enc = popkv_cuda.query_encode(q, dim_group_size=g)
    got = _u16(popkv_cuda.score_encoded(enc, packed, head_to_kv=mapping, tokens=tokens, dim_group_size=g))
    want = core.score_encoded([e.cpu().numpy() for e in enc], _planes(packed), head_to_kv=mapping.cpu().numpy(),
                              tokens=tokens, dim_group_size=g)
    nan = (want & 0x7C00 == 0x7C00) & (want & 0x03FF != 0)
    assert np.array_equal(got[~nan], want[~nan])
    assert np.all((got[nan] & 0x7C00 == 0x7C00) & (got[nan] & 0x03FF != 0))


@pytest.mark.parametrize("method", ("popkv-s", "popkv-q", "popkv-normal"))
def test_ragged_batch_selects_as_the_oracle(method):
    """Sequences from one token to several spans in one launch (spans past a
    sequence's end return at once): the selected indices of every sequence."""
    tg, g = popkv.POPKV_PRESETS[method]
    lengths, budget, kvh, qpk = [9001, 1, 2048, 700, 4097], 256, 2, 8
    gen = torch.Generator().manual_seed(g)
    rows = max(lengths) + 1
    kc = torch.randn(len(lengths), kvh, rows, 128, generator=gen).half().to(DEV)
    q = torch.randn(len(lengths), kvh * qpk, 128, generator=gen).half().to(DEV)
    k = torch.randn(len(lengths), kvh, 128, generator=gen).half().to(DEV)
    mapping = torch.arange(kvh * qpk, device=DEV) // qpk
    seq = pb.SequenceLengths.create(lengths, DEV)
    cache = pb.build_batched_popkv_cache(kc, kc.clone(), seq, group_size=tg, dim_group_size=g)
    ws = popkv.LayerStepWorkspace()
    for _ in range(2):  # the histograms are zero again after the first
        _, idx = pb.popkv_layer_step_batched(q, cache, seq, k, k, mapping, budget=budget, workspace=ws,
                                             return_indices=True)
    for i, n in enumerate(lengths):
        enc = core.query_encode(q[i:i + 1].float().cpu().numpy(), g, order="fold")
        planes = core.pack_keys(kc[i, :, :n].float().cpu().numpy(), token_group_size=tg, dim_group_size=g)
        scores = core.score_encoded(enc, planes, head_to_kv=mapping.cpu().numpy(), tokens=n, dim_group_size=g)
        kk = min(budget - 1, n)
        assert np.array_equal(idx[i, :, :kk + 1].cpu().numpy(), core.select(scores[0], kk, n)), n
