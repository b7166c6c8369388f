"""append_retrieval_caches' one-launch append against the per-layer append it
replaces, bit for bit, and the calls that keep to the general path."""
from __future__ import annotations

import io

import pytest
import torch

from popkv_amd import _native, popkv

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _caches(layers, tokens, tg, g, dtype, reserve=64):
    gen = torch.Generator().manual_seed(layers + tokens + tg)
    keys = [torch.randn(3, tokens, 128, generator=gen).to(dtype).to(DEV) for _ in range(layers)]
    return {i: popkv.build_popkv_cache(k, group_size=tg, dim_group_size=g, reserve_tokens=reserve)
            for i, k in enumerate(keys)}


def _same(a, b):
    for i in a:
        n = a[i].token_count
        assert (n, a[i].sealed_tokens) == (b[i].token_count, b[i].sealed_tokens)
        assert torch.equal(a[i].active_keys, b[i].active_keys)
        for x, y in zip(a[i].packed, b[i].packed):
            assert torch.equal(x[:, :n].view(torch.int16), y[:, :n].view(torch.int16))


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("layers,tokens,tg,g", [(1, 61, 64, 64), (3, 127, 128, 16), (33, 30, 32, 32), (2, 13, 8, 64),
                                                (2, 141, 150, 32)])
def test_one_launch_append_equals_the_layers_own(layers, tokens, tg, g, dtype, monkeypatch):
    """Tokens that fill, seal and start groups, more layers than one launch
    takes, a group size of no preset."""
    one, each = _caches(layers, tokens, tg, g, dtype), _caches(layers, tokens, tg, g, dtype)
    calls = []
    real = _native.call
    monkeypatch.setattr(_native, "call", lambda name, *args: (calls.append(name), real(name, *args))[1])
    for step in range(12):
        gen = torch.Generator().manual_seed(1000 + step)
        new = [torch.randn(1, 3, 1, 128, generator=gen).to(dtype).to(DEV) for _ in range(layers)]
        calls.clear()
        popkv.append_retrieval_caches(popkv.RetrievalCaches("popkv-s", one), new)
        assert calls == ["popkv_stage_append"]
        for i in each:
            popkv.append_popkv(each[i], new[i][0])
        _same(one, each)


def test_unequal_caches_take_the_general_path(monkeypatch):
    """Layers at different points of their groups, a key that is not
    contiguous and one cache listed twice, as the per-layer appends do."""
    one, each = _caches(3, 40, 64, 64, torch.bfloat16), _caches(3, 40, 64, 64, torch.bfloat16)
    extra = torch.randn(3, 1, 128).bfloat16().to(DEV)
    popkv.append_popkv(one[1], extra)
    popkv.append_popkv(each[1], extra)
    wide = torch.randn(1, 3, 2, 128).bfloat16().to(DEV)
    new = [wide[:, :, :1] for _ in range(3)]
    calls = []
    real = _native.call
    monkeypatch.setattr(_native, "call", lambda name, *args: (calls.append(name), real(name, *args))[1])
    popkv.append_retrieval_caches(popkv.RetrievalCaches("popkv-s", one), new)
    assert calls == ["popkv_pack"] * 3
    for i in each:
        popkv.append_popkv(each[i], new[i][0])
    _same(one, each)
    cache = one[0]
    before = cache.token_count
    popkv.append_retrieval_caches(popkv.RetrievalCaches("popkv-s", {0: cache, 1: cache}), [extra[None], extra[None]])
    assert cache.token_count == before + 2 and int(cache.active_keys.shape[1]) == before + 2


def test_exhausted_reserve_is_refused_as_before():
    caches = _caches(2, 64, 64, 64, torch.bfloat16, reserve=0)
    with pytest.raises(RuntimeError, match="Pop-KV cache reserve exhausted"):
        popkv.append_retrieval_caches(popkv.RetrievalCaches("popkv-s", caches), [torch.zeros(1, 3, 1, 128, device=DEV,
                                                                                            dtype=torch.bfloat16)] * 2)


def test_staged_keys_are_each_layers_own():
    """A layer's staged keys keep no other layer's rows alive, and saving
    them writes that layer's rows alone."""
    caches = _caches(5, 61, 64, 64, torch.bfloat16)
    new = [torch.randn(1, 3, 1, 128).bfloat16().to(DEV) for _ in range(5)]
    for _ in range(2):
        popkv.append_retrieval_caches(popkv.RetrievalCaches("popkv-s", caches), new)
        for cache in caches.values():
            keys = cache.active_keys
            assert keys.untyped_storage().nbytes() == keys.numel() * keys.element_size()
            saved = io.BytesIO()
            torch.save(keys, saved)
            assert saved.getbuffer().nbytes < 2 * keys.numel() * keys.element_size()
