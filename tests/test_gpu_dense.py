"""Dense decode attention at the edges of its tiles, waves and splits against
float64."""
from __future__ import annotations

import math

import pytest
import torch

from popkv_amd import popkv

pytestmark = pytest.mark.gpu

DEV = "cuda"
# Largest error allowed per element: one unit in the last place of the output
# type (its rounding, and a neighbour where the fp32 result sits on a tie)
# plus 4e-5: fp32 sums and exponentials of logits up to about 30 in
# magnitude, relative error about 30 * 2^-23 of values up to about 5.
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -23}


def _reference(q, pk, pv, k, v):
    group = q.shape[0] // pk.shape[0]
    out = []
    for h in range(q.shape[0]):
        g = h // group
        keys = torch.cat([pk[g], k[g, None]]).double()
        values = torch.cat([pv[g], v[g, None]]).double()
        out.append(torch.softmax(keys @ q[h].double() / math.sqrt(128), 0) @ values)
    return torch.stack(out)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("group", (1, 2, 4, 8))
@pytest.mark.parametrize("kv_heads,tokens", [(1, 0), (2, 1), (3, 15), (2, 17), (1, 127), (3, 129), (2, 2049), (40, 1301),
                                             (1, 40007), (300, 200)])
def test_dense_attention_tile_and_split_edges(kv_heads, tokens, group, dtype):
    """No token, a ragged tile, a split of fewer tiles than waves, several
    splits with a short last one, KV heads that do not divide the workgroup
    target and more KV heads than it; one workspace used twice (the merge
    tickets go back to zero)."""
    gen = torch.Generator().manual_seed(tokens + group)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(dtype)  # noqa: E731
    q, k, v = draw(kv_heads * group, 128) * 3, draw(kv_heads, 128), draw(kv_heads, 128)
    rows = draw(2, kv_heads, tokens + 3, 128)  # a head stride wider than the prefix
    pk, pv = rows[0].to(DEV)[:, :tokens], rows[1].to(DEV)[:, :tokens]
    ws = popkv.LayerStepWorkspace()
    want = _reference(q, rows[0][:, :tokens], rows[1][:, :tokens], k, v)
    for _ in range(2):
        got = popkv.dense_attention_step(q.to(DEV), pk, pv, k.to(DEV), v.to(DEV), workspace=ws)
        err = (got.cpu().double() - want).abs()
        assert (err <= ULP[dtype] * want.abs() + 4e-5).all(), float((err - ULP[dtype] * want.abs()).max())


def _attend_nonfinite(kv_heads, group, tokens, dtype, spoil):
    """dense_attention_step after `spoil(keys, values)`, and float64: (got,
    want).  Small queries, so that no weight of any row underflows."""
    gen = torch.Generator().manual_seed(tokens + group)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(dtype)  # noqa: E731
    q, k, v = draw(kv_heads * group, 128) * 0.1, draw(kv_heads, 128), draw(kv_heads, 128)
    pk, pv = draw(kv_heads, tokens, 128), draw(kv_heads, tokens, 128)
    spoil(pk, pv)
    got = popkv.dense_attention_step(q.to(DEV), pk.to(DEV), pv.to(DEV), k.to(DEV), v.to(DEV))
    return got.cpu().double(), _reference(q, pk, pv, k, v)


def _same_nonfinite(got, want, dtype):
    assert torch.equal(got.isnan(), want.isnan())
    inf = want.isinf()
    assert torch.equal(got[inf], want[inf])
    ok = want.isfinite()
    assert ((got[ok] - want[ok]).abs() <= ULP[dtype] * want[ok].abs() + 4e-5).all()


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("group", (1, 2, 4, 8))
@pytest.mark.parametrize("kv_heads,tokens", [(2, 100), (2, 1024), (1, 4240), (1, 8191), (1, 40007)])
def test_dense_attention_infinite_value_in_the_last_split(kv_heads, tokens, group, dtype):
    """An infinite value element in the last row: infinite in that output
    dimension however many splits the merge folds, finite in the others."""
    def spoil(pk, pv):
        pv[0, -1, 3], pv[-1, -1, 77] = float("inf"), float("-inf")

    _same_nonfinite(*_attend_nonfinite(kv_heads, group, tokens, dtype, spoil), dtype)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("group", (1, 2, 4, 8))
@pytest.mark.parametrize("kv_heads,tokens", [(2, 1), (2, 1000), (3, 2001), (1, 40007), (300, 200)])
def test_dense_attention_infinite_value_at_a_splits_first_row(kv_heads, tokens, group, dtype):
    """Infinite value elements in every row a split can start at (multiples
    of 16, dimension row / 16): a pass that reaches past its split's end has
    no live row to take there, and must not fold another's value."""
    def spoil(pk, pv):
        rows = torch.arange(0, tokens, 16)
        pv[:, rows, rows // 16 % 96] = float("inf")

    _same_nonfinite(*_attend_nonfinite(kv_heads, group, tokens, dtype, spoil), dtype)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("group", (1, 2, 4, 8))
@pytest.mark.parametrize("first,tokens", [(0, 300), (112, 300), (288, 300), (0, 2049)])
def test_dense_attention_tile_of_nan_keys(first, tokens, group, dtype):
    """NaN keys in 16 rows of the second KV head that make up one tile of the
    matrix-core kernel, the first a wave folds: NaN in every output of that
    head's group, none elsewhere."""
    def spoil(pk, pv):
        pk[1, first:first + 16] = float("nan")

    _same_nonfinite(*_attend_nonfinite(2, group, tokens, dtype, spoil), dtype)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("group", (1, 2, 4, 8))
@pytest.mark.parametrize("kv_heads,tokens", [(1, 4096), (1, 4112), (1, 8192), (1, 8193), (1, 12288), (1, 32768),
                                             (2, 16383), (3, 11000), (150, 1000), (300, 1301)])
def test_dense_attention_merge_levels(kv_heads, tokens, group, dtype):
    """32, 33 and 64 splits (one level of one and two bursts), 65, 96, 128
    and 256, and the 77 of three KV heads (sets of 32, then the sets); three
    splits of KV heads that fill one and a half rounds of the CUs.  Against
    float64, equal bits from the same workspace again, tickets back at zero."""
    gen = torch.Generator().manual_seed(tokens + group)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(dtype)  # noqa: E731
    q, k, v = draw(kv_heads * group, 128) * 3, draw(kv_heads, 128), draw(kv_heads, 128)
    pk, pv = draw(kv_heads, tokens, 128), draw(kv_heads, tokens, 128)
    want = _reference(q, pk, pv, k, v)
    ws, args = popkv.LayerStepWorkspace(), [t.to(DEV) for t in (q, pk, pv, k, v)]
    got = popkv.dense_attention_step(*args, workspace=ws)
    err = (got.cpu().double() - want).abs()
    assert (err <= ULP[dtype] * want.abs() + 4e-5).all(), float((err - ULP[dtype] * want.abs()).max())
    assert torch.equal(popkv.dense_attention_step(*args, workspace=ws), got)
    assert not ws.buffer[:max(256, 4 * q.shape[0])].any()
