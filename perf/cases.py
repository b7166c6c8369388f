"""The work that the speed of this framework is measured on.

Each case is one call, or one step of calls, that a decode or prefill loop
makes through the package's public entry points (``popkv_amd.popkv``,
``.batch``, ``.popkv_cuda``, ``.sparse_kernels``), with the operands such a
loop has in hand.  Kinds:

  step     one sparse layer of a decode step, called eagerly (popkv_layer_step)
  stack    a whole decode step over a layer stack, captured once in a HIP
           graph and replayed token after token (SparseDecodeStack)
  decode   one layer of a batched decode step with the append of the new
           token (popkv_layer_step_batched(append=True)), replayed from a
           graph (equal lengths) or called eagerly (ragged lengths, a batch
           whose members come and go)
  ops      the layer as the separate operations of the reference's decode
           loop (popkv_retrieval_step: encode, score, select, attend, merge)
  dense    a full layer (dense_attention_step)
  prefill  the prefix prepack (build_popkv_cache, build_batched_popkv_cache)
  append   the per-token metadata append of every sparse layer
           (append_retrieval_caches)
  head     head dimensions other than 128 (pack_keys, score and
           indexed_attention_split)

Keys carry four outlier channels per KV head and queries lean on a few of
the cached keys, as in ``popkv_amd.workloads``; everything is drawn on the
GPU from the seed.
"""
from __future__ import annotations

import dataclasses
import math

import torch

from popkv_amd import batch as pb
from popkv_amd import popkv, popkv_cuda, sparse_kernels

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed() -> list[dict]:
    return [
        # the smallest call: one layer of a small fp32 model at a 4K context
        dict(name="step-normal-4k", kind="step", method="popkv-normal", q_heads=8, kv_heads=2, tokens=4095,
             budget=512, dtype="fp32"),
        # one layer of an 8B-shaped model at a long context, no graph
        dict(name="step-s-128k", kind="step", method="popkv-s", q_heads=32, kv_heads=8, tokens=131071, budget=4096,
             dtype="bf16"),
        # the whole decode step of a 32-layer model at 32K, two dense layers
        dict(name="stack-q-32k", kind="stack", method="popkv-q", layers=32, q_heads=32, kv_heads=8, tokens=32767,
             budget=4096, dtype="bf16"),
        # batched serving: eight sequences of 64K, one graph for all tokens
        dict(name="decode-s-8x64k", kind="decode", method="popkv-s", batch=8, ragged=False, q_heads=32, kv_heads=8,
             tokens=65535, budget=4096, dtype="bf16"),
        # continuous batching: sequences of different lengths, 8 queries per KV head
        dict(name="decode-normal-ragged", kind="decode", method="popkv-normal", batch=5, ragged=True, q_heads=64,
             kv_heads=8, tokens=20001, budget=1024, dtype="fp16"),
        # the reference's decode loop with only its imports changed, an ordinary odd-sized context
        dict(name="ops-s-16k", kind="ops", method="popkv-s", q_heads=32, kv_heads=8, tokens=16001, budget=1001,
             dtype="fp16"),
        # a full layer of a 70B-shaped model
        dict(name="dense-gqa8-50k", kind="dense", q_heads=64, kv_heads=8, tokens=50001, dtype="bf16"),
        # a full layer of a model without grouped heads
        dict(name="dense-mha-8k", kind="dense", q_heads=32, kv_heads=32, tokens=8191, dtype="fp16"),
        # prefix prepack of one layer, the default preset
        dict(name="prefill-normal-32k", kind="prefill", method="popkv-normal", batch=1, kv_heads=8, tokens=32767,
             dtype="bf16"),
        # prefix prepack of one layer for a batch of long prompts
        dict(name="prefill-s-8x64k", kind="prefill", method="popkv-s", batch=8, kv_heads=8, tokens=65535,
             dtype="bf16"),
        # the metadata of one new token in all thirty sparse layers
        dict(name="append-q-30-layers", kind="append", method="popkv-q", layers=30, kv_heads=8, tokens=8269,
             dtype="bf16"),
        # a model with 64-dimension heads, operation by operation
        dict(name="head64-8k", kind="head", head_dim=64, token_group=32, dim_group=32, q_heads=32, kv_heads=8,
             tokens=8191, selected=1024, dtype="fp16"),
    ]


def _log(rng, lo: int, hi: int) -> int:
    """An odd or even size spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng, kv=(2, 4, 8), group=(1, 2, 4, 8)) -> dict:
    kv_heads = rng.choice(kv)
    return dict(q_heads=kv_heads * rng.choice(group), kv_heads=kv_heads)


def draw(rng) -> dict:
    kind = rng.choice(("step", "step", "stack", "decode", "decode", "ops", "dense", "dense", "prefill", "prefill",
                       "append", "head"))
    method = rng.choice(("popkv-normal", "popkv-q", "popkv-s"))
    half = rng.choice(("bf16", "fp16"))
    any_dtype = rng.choice(("bf16", "fp16", "fp32"))
    if kind == "step":
        return dict(kind=kind, method=method, **_heads(rng), tokens=_log(rng, 700, 262144),
                    budget=_log(rng, 256, 8192), dtype=any_dtype)
    if kind == "stack":
        return dict(kind=kind, method=method, layers=rng.randrange(4, 17), q_heads=32, kv_heads=8,
                    tokens=_log(rng, 4096, 49152), budget=_log(rng, 512, 4096), dtype=half)
    if kind == "decode":
        return dict(kind=kind, method=method, batch=rng.randrange(2, 9), ragged=rng.random() < 0.5,
                    **_heads(rng, group=(4, 8)), tokens=_log(rng, 2048, 65535), budget=_log(rng, 512, 4096), dtype=half)
    if kind == "ops":
        return dict(kind=kind, method=method, **_heads(rng), tokens=_log(rng, 1000, 65536),
                    budget=_log(rng, 256, 4096), dtype=any_dtype)
    if kind == "dense":
        return dict(kind=kind, **_heads(rng, kv=(2, 4, 8, 32)), tokens=_log(rng, 500, 65536), dtype=any_dtype)
    if kind == "prefill":
        return dict(kind=kind, method=method, batch=rng.choice((1, 1, 2, 4)), kv_heads=rng.choice((2, 4, 8)),
                    tokens=_log(rng, 1000, 131072), dtype=any_dtype)
    if kind == "append":
        return dict(kind=kind, method=method, layers=rng.randrange(8, 33), kv_heads=rng.choice((2, 4, 8)),
                    tokens=_log(rng, 500, 16384), dtype=any_dtype)
    return dict(kind=kind, head_dim=rng.choice((64, 96)), token_group=rng.choice((32, 64)),
                dim_group=rng.choice((16, 32)), **_heads(rng, group=(2, 4)), tokens=_log(rng, 1000, 16384),
                selected=_log(rng, 128, 900), dtype=half)


# ------------------------------------------------------------------ operands

def _device() -> torch.device:
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=_device()).manual_seed(seed)


def _keys(gen, heads: int, rows: int, dtype: torch.dtype, dim: int = 128) -> torch.Tensor:
    """[heads, rows, dim] N(0, 1) keys with four channels per head ten times larger."""
    keys = torch.randn(heads, rows, dim, device=_device(), generator=gen, dtype=torch.float32)
    loud = torch.rand(heads, dim, device=_device(), generator=gen).argsort(-1)[:, :4]
    scale = torch.ones(heads, dim, device=_device()).scatter_(1, loud, 10.0)
    return keys.mul_(scale[:, None]).to(dtype)


def _values(gen, heads: int, rows: int, dtype: torch.dtype, dim: int = 128) -> torch.Tensor:
    return torch.randn(heads, rows, dim, device=_device(), generator=gen, dtype=torch.float32).to(dtype)


def _queries(gen, keys: torch.Tensor, q_heads: int, tokens: int) -> torch.Tensor:
    """[q_heads, D]: half the mean of 64 cached keys of the head's KV head plus N(0, 1)."""
    kv_heads, _, dim = keys.shape
    rows = torch.randint(0, tokens, (q_heads, 64), device=_device(), generator=gen)
    group = _mapping(q_heads, kv_heads)
    lean = keys[group[:, None], rows].float().mean(1)
    return (0.5 * lean + torch.randn(q_heads, dim, device=_device(), generator=gen)).to(keys.dtype)


def _mapping(q_heads: int, kv_heads: int) -> torch.Tensor:
    return torch.arange(q_heads, device=_device()) // (q_heads // kv_heads)


def _layer(case: dict, seed: int) -> dict:
    """One layer of one sequence: K/V storage [KVH, tokens + 1, 128] whose
    last row is the current token, and its queries."""
    gen, n = _generator(seed), case["tokens"]
    dtype = _DTYPES[case["dtype"]]
    keys = _keys(gen, case["kv_heads"], n + 1, dtype)
    values = _values(gen, case["kv_heads"], n + 1, dtype)
    return dict(q=_queries(gen, keys, case["q_heads"], n), pk=keys[:, :n], pv=values[:, :n],
                k=keys[:, n].contiguous(), v=values[:, n].contiguous())


def _lengths(case: dict) -> list[int]:
    """The batch's cached tokens: all alike, or from the longest down to a tenth of it."""
    n, b = case["tokens"], case["batch"]
    if not case["ragged"]:
        return [n] * b
    return [max(1, int(n * 10.0 ** (-i / (b - 1)))) for i in range(b)]


def _batch(case: dict, seed: int) -> dict:
    gen, dtype = _generator(seed), _DTYPES[case["dtype"]]
    b, kvh, rows = case["batch"], case["kv_heads"], case["tokens"] + 1
    key_cache = torch.empty(b, kvh, rows, 128, device=_device(), dtype=dtype)
    value_cache = torch.empty_like(key_cache)
    queries, lengths = [], _lengths(case)
    for i in range(b):
        key_cache[i] = _keys(gen, kvh, rows, dtype)
        value_cache[i] = _values(gen, kvh, rows, dtype)
        queries.append(_queries(gen, key_cache[i], case["q_heads"], lengths[i]))
    k, v = _values(gen, b * kvh, 1, dtype).view(b, kvh, 128), _values(gen, b * kvh, 1, dtype).view(b, kvh, 128)
    return dict(key_cache=key_cache, value_cache=value_cache, q=torch.stack(queries), k=k, v=v, lengths=lengths)


def _capture(call):
    """`call` recorded into a HIP graph after one warm-up call, with what it returned."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = call()
    return graph, outs


def prepare(case: dict, seed: int) -> dict:
    return {"step": _prepare_step, "ops": _prepare_step, "stack": _prepare_stack, "decode": _prepare_decode,
            "dense": _prepare_dense, "prefill": _prepare_prefill, "append": _prepare_append,
            "head": _prepare_head}[case["kind"]](case, seed)


def _prepare_step(case, seed):
    s = _layer(case, seed)
    tg, g = popkv.POPKV_PRESETS[case["method"]]
    cache = popkv.build_popkv_cache(s["pk"], group_size=tg, dim_group_size=g, reserve_tokens=256)
    return dict(s, kind=case["kind"], cache=cache, mapping=_mapping(case["q_heads"], case["kv_heads"]),
                budget=case["budget"], workspace=popkv.LayerStepWorkspace())


_FULL_LAYERS = (0, 1)


def _prepare_stack(case, seed):
    tg, g = popkv.POPKV_PRESETS[case["method"]]
    operands, caches = [], {}
    for i in range(case["layers"]):
        s = _layer(case, seed * 1000 + i)
        operands.append((s["q"], s["pk"], s["pv"], s["k"], s["v"]))
        if i not in _FULL_LAYERS:
            caches[i] = popkv.build_popkv_cache(s["pk"], group_size=tg, dim_group_size=g, reserve_tokens=256)
    stack = popkv.SparseDecodeStack(caches, _mapping(case["q_heads"], case["kv_heads"]), budget=case["budget"],
                                    full_layers=_FULL_LAYERS)
    graph, outs = _capture(lambda: stack.step(operands))
    return dict(kind="stack", stack=stack, operands=operands, graph=graph, outs=outs)


def _prepare_decode(case, seed):
    s = _batch(case, seed)
    tg, g = popkv.POPKV_PRESETS[case["method"]]
    lengths = pb.SequenceLengths.create(s["lengths"], _device())
    cache = pb.build_batched_popkv_cache(s["key_cache"], s["value_cache"], lengths, group_size=tg, dim_group_size=g)
    s = dict(s, kind="decode", cache=cache, lengths=lengths, budget=case["budget"],
             mapping=_mapping(case["q_heads"], case["kv_heads"]), workspace=popkv.LayerStepWorkspace())
    if not case["ragged"]:
        s["graph"], s["outs"] = _capture(lambda: _decode(s))
    return s


def _prepare_dense(case, seed):
    return dict(_layer(case, seed), kind="dense", workspace=popkv.LayerStepWorkspace())


def _prepare_prefill(case, seed):
    tg, g = popkv.POPKV_PRESETS[case["method"]]
    gen, dtype, b, n = _generator(seed), _DTYPES[case["dtype"]], case["batch"], case["tokens"]
    if b == 1:
        return dict(kind="prefill", keys=_keys(gen, case["kv_heads"], n, dtype), tg=tg, g=g)
    key_cache = torch.empty(b, case["kv_heads"], n + 1, 128, device=_device(), dtype=dtype)
    for i in range(b):
        key_cache[i] = _keys(gen, case["kv_heads"], n + 1, dtype)
    return dict(kind="prefill", key_cache=key_cache, value_cache=torch.zeros_like(key_cache),
                lengths=pb.SequenceLengths.create([n] * b, _device()), tg=tg, g=g)


def _append_keys(case, seed):
    gen, dtype = _generator(seed), _DTYPES[case["dtype"]]
    shape = (case["layers"], case["kv_heads"])
    keys = _keys(gen, shape[0] * shape[1], case["tokens"], dtype).view(*shape, -1, 128)
    return keys, _values(gen, shape[0] * shape[1], 1, dtype).view(*shape, 1, 128)


def _prepare_append(case, seed):
    tg, g = popkv.POPKV_PRESETS[case["method"]]
    keys, new = _append_keys(case, seed)
    built = [popkv.build_popkv_cache(k, group_size=tg, dim_group_size=g, reserve_tokens=256) for k in keys]
    # every layer's planes side by side, so that they can be handed back whole
    planes = [torch.stack([c.packed[p] for c in built]) for p in range(4)]
    caches = {i: dataclasses.replace(c, packed=tuple(p[i] for p in planes)) for i, c in enumerate(built)}
    return dict(kind="append", method=case["method"], caches=caches, new=list(new), planes=planes,
                rows=case["tokens"] + 1)


def _head_operands(case, seed):
    gen, dtype, n, dim = _generator(seed), _DTYPES[case["dtype"]], case["tokens"], case["head_dim"]
    keys, values = _keys(gen, case["kv_heads"], n + 1, dtype, dim), _values(gen, case["kv_heads"], n + 1, dtype, dim)
    picked = torch.rand(case["q_heads"], n, device=_device(), generator=gen).argsort(-1)[:, :case["selected"]]
    current = torch.full((case["q_heads"], 1), n, device=_device())
    return dict(q=_queries(gen, keys, case["q_heads"], n), keys=keys[:, :n].contiguous(), values=values[:, :n],
                k=keys[:, n].contiguous(), v=values[:, n].contiguous(),
                indices=torch.cat([picked.sort(-1).values, current], -1))


def _prepare_head(case, seed):
    return dict(_head_operands(case, seed), kind="head", tg=case["token_group"], g=case["dim_group"],
                mapping=_mapping(case["q_heads"], case["kv_heads"]))


# ---------------------------------------------------------------------- pass

def _decode(s):
    return pb.popkv_layer_step_batched(s["q"], s["cache"], s["lengths"], s["k"], s["v"], s["mapping"],
                                       budget=s["budget"], workspace=s["workspace"], append=True)


def run(s: dict):
    kind = s["kind"]
    if kind == "step":
        return popkv.popkv_layer_step(s["q"], s["cache"], s["pk"], s["pv"], s["k"], s["v"], s["mapping"],
                                      budget=s["budget"], workspace=s["workspace"])
    if kind == "ops":
        return popkv.popkv_retrieval_step(s["q"], s["pk"], s["pv"], s["k"], s["v"], s["cache"], s["mapping"],
                                          budget=s["budget"])
    if kind == "stack":
        s["graph"].replay()
        return s["outs"]
    if kind == "decode":
        if "graph" in s:
            s["graph"].replay()
            out = s["outs"]
        else:
            out = _decode(s)
        return dict(out=out, packed=s["cache"].packed, keys=s["key_cache"], values=s["value_cache"])
    if kind == "dense":
        return popkv.dense_attention_step(s["q"], s["pk"], s["pv"], s["k"], s["v"], workspace=s["workspace"])
    if kind == "prefill":
        if "keys" in s:  # rows past the prefix are reserve, not written
            n = s["keys"].shape[1]
            cache = popkv.build_popkv_cache(s["keys"], group_size=s["tg"], dim_group_size=s["g"], reserve_tokens=256)
            return [p[:, :n] for p in cache.packed]
        return pb.build_batched_popkv_cache(s["key_cache"], s["value_cache"], s["lengths"], group_size=s["tg"],
                                            dim_group_size=s["g"]).packed
    if kind == "append":
        # the loop's caches before this token (the planes are shared, the
        # staged keys are replaced by the append)
        caches = popkv.RetrievalCaches(s["method"], {i: dataclasses.replace(c) for i, c in s["caches"].items()})
        popkv.append_retrieval_caches(caches, s["new"])
        return [p[:, :, :s["rows"]] for p in s["planes"]]
    packed = popkv_cuda.pack_keys(s["keys"], token_group_size=s["tg"], dim_group_size=s["g"])
    scores = popkv_cuda.score(s["q"][None], packed, head_to_kv=s["mapping"], tokens=int(s["keys"].shape[1]),
                              dim_group_size=s["g"])
    out = sparse_kernels.indexed_attention_split(s["q"], s["keys"], s["values"], s["k"], s["v"], s["indices"],
                                                 s["mapping"])
    return dict(packed=packed, scores=scores, out=out)


# ---------------------------------------------------------------- what it costs

def _step_work(q_heads, kv_heads, tokens, budget, g, esize):
    """Bytes and operations one sparse layer cannot do without: the planes
    scored once, K/V rows the heads of a group select counted once as if
    they agreed on them, the agreement counts and the attention."""
    k = min(budget - 1, tokens)
    planes = kv_heads * tokens * (32 + 4 * (128 // g)) if k < tokens else 0
    rows = kv_heads * (k + 1) * 2 * 128 * esize
    return dict(bytes=planes + rows + 2 * q_heads * 128 * esize,
                flops=q_heads * ((tokens * 128 * 2 if k < tokens else 0) + (k + 1) * 128 * 4))


def _plane_bytes(heads, tokens, g, dim=128):
    return heads * tokens * (8 * math.ceil(dim / 32) + 4 * math.ceil(dim / g))


def work(case: dict) -> dict:
    kind, n = case["kind"], case["tokens"]
    esize = 4 if case["dtype"] == "fp32" else 2
    g = popkv.POPKV_PRESETS[case["method"]][1] if "method" in case else None
    tg = popkv.POPKV_PRESETS[case["method"]][0] if "method" in case else None
    if kind in ("step", "ops"):
        return _step_work(case["q_heads"], case["kv_heads"], n, case["budget"], g, esize)
    dense = dict(bytes=case["kv_heads"] * (n + 1) * 2 * 128 * esize, flops=case.get("q_heads", 0) * (n + 1) * 128 * 4)
    if kind == "dense":
        return dense
    if kind == "stack":
        one = _step_work(case["q_heads"], case["kv_heads"], n, case["budget"], g, esize)
        full = len(_FULL_LAYERS)
        return {x: one[x] * (case["layers"] - full) + dense[x] * full for x in one}
    if kind == "decode":
        each = [_step_work(case["q_heads"], case["kv_heads"], x, case["budget"], g, esize) for x in _lengths(case)]
        heads = case["batch"] * case["kv_heads"]
        append = sum(case["kv_heads"] * (x % tg + 1) * 128 * esize for x in _lengths(case)) + 4 * heads * 128 * esize
        return dict(bytes=sum(e["bytes"] for e in each) + append, flops=sum(e["flops"] for e in each))
    if kind == "prefill":
        heads = case["batch"] * case["kv_heads"]
        return dict(bytes=heads * n * 128 * esize + _plane_bytes(heads, n, g), flops=heads * n * 128 * 4)
    if kind == "append":
        heads, active = case["layers"] * case["kv_heads"], n % tg + 1
        return dict(bytes=heads * active * 128 * esize + _plane_bytes(heads, active, g), flops=heads * active * 128 * 4)
    dim, heads, sel = case["head_dim"], case["kv_heads"], case["selected"] + 1
    bits = _plane_bytes(heads, n, case["dim_group"], dim)
    return dict(bytes=heads * n * dim * esize + 2 * bits + case["q_heads"] * n * 4 + heads * sel * 2 * dim * esize
                + case["q_heads"] * sel * 8,
                flops=heads * n * dim * 4 + case["q_heads"] * (n * dim * 2 + sel * dim * 4))


def tolerance(case: dict):
    """Planes are bits and exact.  Attention rounds once to the output type;
    scores of other head dimensions are fp32 sums."""
    if case["kind"] in ("prefill", "append"):
        return "exact"
    return {"bf16": {"rel": 8e-3, "max": 2e-2}, "fp16": {"rel": 1e-3, "max": 2e-3},
            "fp32": {"rel": 1e-5, "max": 4e-5}}[case["dtype"]]


# ------------------------------------------------------------- in 64 bits

def _bits(flags: torch.Tensor) -> torch.Tensor:
    """Truth values [..., D] as int32 words, dimension 32 w + j at bit j."""
    d = flags.shape[-1]
    flags = torch.nn.functional.pad(flags, (0, -d % 32)).unflatten(-1, (-1, 32))
    word = (flags.long() << torch.arange(32, device=flags.device)).sum(-1)
    return torch.where(word >= 1 << 31, word - (1 << 32), word).to(torch.int32)


def _representatives(mag: torch.Tensor, values: torch.Tensor, g: int):
    """Mean |value| of each dimension group's small and large entries: (low, high - low)."""
    d = values.shape[-1]
    pad = -d % g
    real = torch.nn.functional.pad(torch.ones_like(mag), (0, pad)).unflatten(-1, (-1, g))
    a = torch.nn.functional.pad(values.abs(), (0, pad)).unflatten(-1, (-1, g))
    big = torch.nn.functional.pad(mag, (0, pad)).unflatten(-1, (-1, g))
    small = real & ~big
    ln, hn = small.sum(-1), big.sum(-1)
    low, high = (a * small).sum(-1) / ln.clamp(min=1), (a * big).sum(-1) / hn.clamp(min=1)
    low, high = torch.where(ln > 0, low, high), torch.where(hn > 0, high, low)
    return low, high - low


def _key_planes(keys: torch.Tensor, tg: int, g: int):
    """The packed planes of [heads, tokens, D]: signs, magnitudes, low, delta in 64 bits."""
    x = keys.double()
    n = x.shape[1]
    pad = -n % tg
    grouped = torch.nn.functional.pad(x, (0, 0, 0, pad), value=float("nan")).unflatten(1, (-1, tg))
    hi = torch.where(grouped.isnan(), -math.inf, grouped).amax(2, keepdim=True) * 0.5
    lo = torch.where(grouped.isnan(), math.inf, grouped).amin(2, keepdim=True) * 0.5
    mag = torch.where(grouped >= 0, grouped > hi, grouped < lo).flatten(1, 2)[:, :n]
    low, delta = _representatives(mag, x, g)
    return x >= 0, mag, low, delta


def _dense_values(sign, mag, low, delta, g: int, d: int) -> torch.Tensor:
    wide = lambda t: t.repeat_interleave(g, -1)[..., :d]  # noqa: E731
    return torch.where(sign, 1.0, -1.0) * (wide(low) + torch.where(mag, wide(delta), 0.0))


def _scores(q: torch.Tensor, planes, mapping: torch.Tensor, g: int) -> torch.Tensor:
    """Approximate scores [QH, tokens]: the products of the reconstructed query and keys."""
    x = q.double()
    d = x.shape[-1]
    sign = x >= 0
    mag = torch.where(sign, x > 0.5 * x.amax(-1, keepdim=True), x < 0.5 * x.amin(-1, keepdim=True))
    low, delta = _representatives(mag, x, g)
    ks, km, kl, kd = planes
    qhat = _dense_values(sign, mag, low, delta, g, d)
    khat = _dense_values(ks, km, kl.half().double(), kd.half().double(), g, d)
    heads = khat.shape[0]
    return (qhat.view(heads, -1, d) @ khat.transpose(1, 2).contiguous()).flatten(0, 1) / math.sqrt(d)


def _attend(q, pk, pv, k, v, mapping, indices=None) -> torch.Tensor:
    """Softmax attention of [QH, D] over the selected rows (None: all) and the current token."""
    out = []
    for h, kv in enumerate(mapping.tolist()):
        rows = slice(None) if indices is None else indices[h]
        keys = torch.cat([pk[kv][rows].double(), k[kv][None].double()])
        values = torch.cat([pv[kv][rows].double(), v[kv][None].double()])
        weights = torch.softmax(keys @ q[h].double() / math.sqrt(q.shape[-1]), 0)
        out.append(weights @ values)
    return torch.stack(out)


def _sparse(q, pk, pv, k, v, mapping, budget, tg, g) -> torch.Tensor:
    """One sparse layer: the k best fp16 scores (the first among equal ones) and the current token."""
    kk = min(budget - 1, pk.shape[1])
    scores = _scores(q, _key_planes(pk, tg, g), mapping, g).float().half()
    picked = scores.float().sort(dim=-1, descending=True, stable=True).indices[:, :kk]
    return _attend(q, pk, pv, k, v, mapping, picked)


def exact(case: dict, seed: int):
    kind = case["kind"]
    tg, g = popkv.POPKV_PRESETS[case["method"]] if "method" in case else (None, None)
    if kind == "dense":
        s = _layer(case, seed)
        return _attend(s["q"], s["pk"], s["pv"], s["k"], s["v"], _mapping(case["q_heads"], case["kv_heads"]))
    if kind in ("step", "ops"):
        s = _layer(case, seed)
        return _sparse(s["q"], s["pk"], s["pv"], s["k"], s["v"], _mapping(case["q_heads"], case["kv_heads"]),
                       case["budget"], tg, g)
    if kind == "stack":
        outs, mapping = [], _mapping(case["q_heads"], case["kv_heads"])
        for i in range(case["layers"]):
            s = _layer(case, seed * 1000 + i)
            ops = (s["q"], s["pk"], s["pv"], s["k"], s["v"], mapping)
            outs.append(_attend(*ops) if i in _FULL_LAYERS else _sparse(*ops, case["budget"], tg, g))
        return outs
    if kind == "decode":
        s, mapping = _batch(case, seed), _mapping(case["q_heads"], case["kv_heads"])
        out = torch.stack([_sparse(s["q"][i], s["key_cache"][i, :, :n], s["value_cache"][i, :, :n], s["k"][i],
                                   s["v"][i], mapping, case["budget"], tg, g) for i, n in enumerate(s["lengths"])])
        for i, n in enumerate(s["lengths"]):
            s["key_cache"][i, :, n] = s["k"][i]
            s["value_cache"][i, :, n] = s["v"][i]
        return dict(out=out, packed=(None, None, None, None), keys=s["key_cache"], values=s["value_cache"])
    if kind == "prefill":
        s, n = _prepare_prefill(case, seed), case["tokens"]
        if "keys" in s:
            sign, mag, low, delta = _key_planes(s["keys"], tg, g)
            return [_bits(sign), _bits(mag), low, delta]
        parts = []
        for keys in s["key_cache"]:
            sign, mag, low, delta = _key_planes(keys[:, :n], tg, g)
            cap = math.ceil(keys.shape[1] / tg) * tg
            parts.append([torch.nn.functional.pad(p, (0, 0, 0, cap - n))
                          for p in (_bits(sign), _bits(mag), low, delta)])
        return [torch.stack(p) for p in zip(*parts)]
    if kind == "append":
        keys, new = _append_keys(case, seed)
        parts = []
        for k, x in zip(keys, new):
            sign, mag, low, delta = _key_planes(torch.cat([k, x], 1), tg, g)
            parts.append((_bits(sign), _bits(mag), low, delta))
        return [torch.stack(p) for p in zip(*parts)]
    s, mapping, n = _head_operands(case, seed), _mapping(case["q_heads"], case["kv_heads"]), case["tokens"]
    sign, mag, low, delta = _key_planes(s["keys"], case["token_group"], case["dim_group"])
    scores = _scores(s["q"], (sign, mag, low, delta), mapping, case["dim_group"])[None]
    out = _attend(s["q"], s["keys"], s["values"], s["k"], s["v"], mapping, s["indices"][:, :-1])
    return dict(packed=[_bits(sign), _bits(mag), low, delta], scores=scores, out=out)
