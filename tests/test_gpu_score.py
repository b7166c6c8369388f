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


def _ragged(method, lengths, budget, kvh, qpk):
    """A batched layer step of `lengths` selects in every sequence what the
    oracle does; twice, as the histograms are zero again after the first."""
    tg, g = popkv.POPKV_PRESETS[method]
    gen = torch.Generator().manual_seed(g)
    draw = lambda *shape: torch.randn(*shape, generator=gen).half().to(DEV)  # noqa: E731
    kc, q = draw(len(lengths), kvh, max(lengths) + 1, 128), draw(len(lengths), kvh * qpk, 128)
    k = draw(len(lengths), kvh, 128)
    mapping = torch.arange(kvh * qpk, device=DEV) // qpk
    seq = pb.SequenceLengths.create(lengths, DEV)
    cache = pb.build_batched_popkv_cache(kc, kc.clone(), seq, group_size=tg, dim_group_size=g)
    ws = popkv.LayerStepWorkspace()
    for _ in range(2):
        _, idx = pb.popkv_layer_step_batched(q, cache, seq, k, k, mapping, budget=budget, workspace=ws,
                                             return_indices=True)
    for i, n in enumerate(lengths):
        enc = core.query_encode(q[i:i + 1].float().cpu().numpy(), g, order="fold")
        planes = core.pack_keys(kc[i, :, :n].float().cpu().numpy(), token_group_size=tg, dim_group_size=g)
        scores = core.score_encoded(enc, planes, head_to_kv=mapping.cpu().numpy(), tokens=n, dim_group_size=g)
        kk = min(budget - 1, n)
        assert np.array_equal(idx[i, :, :kk + 1].cpu().numpy(), core.select(scores[0], kk, n)), n


@pytest.mark.parametrize("method", ("popkv-s", "popkv-q", "popkv-normal"))
def test_ragged_batch_selects_as_the_oracle(method):
    """Sequences from one token to several spans in one launch (spans past a
    sequence's end return at once); a span is one round of 512 tokens here."""
    _ragged(method, [9001, 1, 2048, 700, 4097], 256, 2, 8)


@pytest.mark.parametrize("qpk", (4, 8))
@pytest.mark.parametrize("method", ("popkv-q", "popkv-normal"))
def test_ragged_batch_with_spans_of_two_rounds(method, qpk):
    """40 rows of 20001 tokens make spans of two rounds (1024 tokens): each
    wave's next group in flight behind its first, sequences that end in the
    second round, in the first, at a round's and at a span's end."""
    _ragged(method, [20001, 9400, 700, 2560, 8192], 1024, 8, qpk)


@pytest.mark.parametrize("kv_heads,qpk,tokens,method", [(1, 8, 140001, "popkv-q"), (2, 4, 200003, "popkv-q"),
                                                        (2, 8, 131600, "popkv-s"), (8, 8, 40001, "popkv-q"),
                                                        (8, 4, 70001, "popkv-normal")])
def test_step_with_spans_of_several_rounds(kv_heads, qpk, tokens, method):
    """One layer step of few rows (256 workgroups), of G16 groups of 8 (256)
    and of others (512): spans of 2 to 4 rounds, the last one short."""
    tg, g = popkv.POPKV_PRESETS[method]
    gen = torch.Generator(DEV).manual_seed(tokens)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device=DEV).half()  # noqa: E731
    keys, q, k = draw(kv_heads, tokens, 128), draw(kv_heads * qpk, 128), draw(kv_heads, 128)
    mapping = torch.arange(kv_heads * qpk, device=DEV) // qpk
    cache = popkv.build_popkv_cache(keys, group_size=tg, dim_group_size=g, reserve_tokens=64)
    _, idx = popkv.popkv_layer_step(q, cache, keys, keys, k, k, mapping, budget=2048, return_indices=True)
    enc = core.query_encode(q[None].float().cpu().numpy(), g, order="fold")
    planes = core.pack_keys(keys.float().cpu().numpy(), token_group_size=tg, dim_group_size=g)
    scores = core.score_encoded(enc, planes, head_to_kv=mapping.cpu().numpy(), tokens=tokens, dim_group_size=g)
    assert np.array_equal(idx.cpu().numpy(), core.select(scores[0], 2047, tokens))
