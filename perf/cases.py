"""The calls that a program built on this package makes, for measuring them.

Each case is one call pattern of a WhiteMatter model over these operators, at
sizes of this repository's benchmark and tests or at odd ones of the same
range:

  decode     one token per row over the KV pool, launched eagerly
             (strict_causal_attention without gradients)
  loop       one token through every layer's attention and the pool store,
             replayed from a graph (DecodeLoop)
  prefill    a chunk of queries behind a ragged cached prefix, forward
  jacobi     packed documents in Jacobi mode, forward and backward, with the
             document schedule kept over calls or built for the call
  cyclic     the residue calls of a cyclic pass, with documents (kept or built
             for the call) or without, forward alone or with backward
  pool       the KV-pool write of one token group: producer, per-channel
             projections, key norm, RoPE and the store
  pool_train the producer and the key transform under autograd
  model      a cyclic prefill of a small model, and the last token's logits

Values are unit normals where a norm precedes them in the model (queries, keys,
sources) and gradients and values are unit normals too. Documents have
geometric lengths (mean a quarter of the row, at least 16 tokens). `work`
counts visible pairs for the documents of one seed; other seeds differ by some
percent.
"""

from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

from white_matter_amd import (
    DecodeLoop,
    cyclic_attention,
    kv_pool,
    prepare_feedback_metadata,
    prepare_strict_causal_metadata,
    strict_causal_attention,
)
from white_matter_amd.cyclic_pass import FeedbackConfig, FeedbackModel, document_positions, forward_cyclic, write_sources

DEV = "cuda"
BF16 = torch.bfloat16


# ------------------------------------------------------------------ cases ----
def listed() -> list[dict]:
    return [
        # an interactive request: one row, a short context, one eager call (the smallest)
        dict(name="decode_one", kind="decode", batch=1, heads=16, kv_heads=8, dim=64, capacity=1153, dummy=True, masked=False),
        # a serving batch over long ragged contexts, two query heads per KV head
        dict(name="decode_batch", kind="decode", batch=32, heads=16, kv_heads=8, dim=128, capacity=8192, dummy=False,
             masked=False),
        # the attention side of a 24-layer model's captured decode step
        dict(name="decode_loop", kind="loop", layers=24, batch=8, heads=16, kv_heads=8, channels=8, dim=64, prefix=1024),
        # the next 256 tokens of every row behind its cached prefix (the most arithmetic)
        dict(name="prefill_cached", kind="prefill", batch=32, heads=16, kv_heads=16, dim=128, queries=256, capacity=8448),
        # one layer of a training step over packed documents, the schedule kept over layers
        dict(name="jacobi_train", kind="jacobi", batch=8, heads=16, kv_heads=16, dim=128, length=2048, dummy=False,
             fresh=False, layers=1),
        # a step over new documents: the schedule, then the layers that use it
        dict(name="jacobi_fresh", kind="jacobi", batch=4, heads=16, kv_heads=8, dim=64, length=1531, dummy=True,
             fresh=True, layers=4),
        # one layer of a cyclic training pass: every residue, the metadata kept over layers
        dict(name="cyclic_train", kind="cyclic", batch=8, heads=16, kv_heads=16, dim=128, length=2048, stride=8, dummy=True,
             documents=True, fresh=False, backward=True, layers=1),
        # the attention of a prefill over new documents: metadata, then layers over pool channels
        dict(name="cyclic_fresh", kind="cyclic", batch=4, heads=16, kv_heads=8, dim=64, length=1027, stride=8, dummy=True,
             documents=True, fresh=True, backward=False, layers=4),
        # cyclic training on rows of one document
        dict(name="cyclic_dense", kind="cyclic", batch=4, heads=16, kv_heads=8, dim=96, length=1500, stride=4, dummy=False,
             documents=False, fresh=False, backward=True, layers=1),
        # the pool write of one token group of a 24-layer model
        dict(name="pool_write", kind="pool", batch=8, tokens=256, layers=24, hidden=1024, heads=16, kv_heads=8, dim=64,
             channels=8),
        # the same group's producer and key transform in training
        dict(name="pool_train", kind="pool_train", batch=4, tokens=256, layers=24, hidden=1024, heads=16, kv_heads=8, dim=64,
             channels=8),
        # a whole prefill and the next token's logits
        dict(name="model_prefill", kind="model", batch=8, length=1024, layers=4, hidden=512, heads=8, kv_heads=4, dim=64,
             channels=4, groups=8, passes=2, vocab=151936),
    ]


def draw(rng) -> dict:
    def log_int(low: int, high: int) -> int:
        return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))

    kind = rng.choice(["decode", "loop", "prefill", "jacobi", "cyclic", "pool", "pool_train", "model"])
    dim = rng.choice([64, 96, 128])
    heads, kv_heads = rng.choice([(16, 16), (16, 8), (16, 4), (8, 8), (8, 4), (12, 6)])
    case = dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim)
    flag = lambda: rng.random() < 0.5  # noqa: E731
    if kind == "decode":
        case.update(batch=log_int(1, 32), capacity=log_int(200, 8192), dummy=flag(), masked=rng.random() < 0.25)
    elif kind == "loop":
        case.update(layers=rng.randint(4, 24), batch=log_int(1, 8), kv_heads=min(kv_heads, 8), channels=rng.choice([2, 4, 8]),
                    prefix=log_int(64, 1024))
    elif kind == "prefill":
        queries = log_int(16, 256)
        case.update(batch=log_int(1, 32), queries=queries, capacity=queries + log_int(200, 8192))
    elif kind == "jacobi":
        fresh = flag()
        case.update(batch=log_int(1, 4 if fresh else 8), length=log_int(130, 1531 if fresh else 2048), dummy=flag(), fresh=fresh,
                    layers=rng.randint(1, 4) if fresh else 1)
    elif kind == "cyclic":
        documents, fresh = rng.random() < 0.7, flag()
        case.update(batch=log_int(1, 4 if fresh else 8), length=log_int(130, 1027 if fresh else 2048),
                    stride=rng.choice([2, 4, 8]), dummy=flag(), documents=documents, fresh=fresh and documents,
                    backward=not fresh, layers=rng.randint(1, 4) if fresh else 1)
    elif kind in ("pool", "pool_train"):
        case.update(batch=log_int(1, 8 if kind == "pool" else 4), tokens=log_int(16, 256), layers=rng.randint(8, 24),
                    hidden=32 * log_int(8, 32), channels=rng.choice([2, 4]) if kind == "pool_train" else rng.choice([2, 4, 8]))
        case.update(kv_heads=min(kv_heads, 8))
    else:
        case.update(batch=log_int(1, 8), length=log_int(100, 1024), layers=rng.randint(3, 4), hidden=64 * rng.randint(2, 8),
                    heads=8, kv_heads=rng.choice([4, 8]), channels=rng.choice([2, 4]), groups=rng.choice([2, 4, 8]), passes=2, vocab=32000)
    return case


# ----------------------------------------------------------------- inputs ----
def _documents(batch: int, length: int, seed: int) -> np.ndarray:
    """(B, T) document ids: geometric lengths, at least 16 tokens, filling each row."""
    rng = np.random.default_rng(seed)
    mean, rows = max(32, length // 4), []
    for _ in range(batch):
        sizes: list[int] = []
        while sum(sizes) < length:
            sizes.append(int(np.clip(rng.geometric(1.0 / mean), 16, length)))
        sizes[-1] -= sum(sizes) - length
        rows.append(np.repeat(np.arange(len(sizes)), sizes))
    return np.stack(rows)


def _lengths(case: dict, seed: int) -> np.ndarray:
    """Cached tokens per row: a sixteenth of the room to all of it."""
    room = case["capacity"] - case.get("queries", 1) - int(case.get("dummy", False))
    return np.random.default_rng(seed).integers(max(1, room // 16), room, size=case["batch"], endpoint=True)


class _Normal:
    """Unit normals on the GPU from one seed."""

    def __init__(self, seed: int) -> None:
        self.gen = torch.Generator(device=DEV).manual_seed(seed)

    def __call__(self, *shape: int, dtype: torch.dtype = BF16, scale: float = 1.0) -> torch.Tensor:
        return (torch.randn(*shape, generator=self.gen, device=DEV) * scale).to(dtype)


def _config(case: dict) -> FeedbackConfig:
    return FeedbackConfig(
        vocab_size=case.get("vocab", 256), hidden_size=case["hidden"], intermediate_size=3 * case["hidden"],
        num_layers=case["layers"], num_heads=case["heads"], num_kv_heads=case["kv_heads"], head_dim=case["dim"],
        num_kv_channels=case["channels"], cyclic_groups=case.get("groups", 8), num_passes=case.get("passes", 3),
    )


def _model(case: dict, seed: int, normal: _Normal) -> FeedbackModel:
    """A random model. The single calls get content in its routers; the whole
    prefill keeps their prior, with which the pool's feedback does not multiply
    a rounding into another result."""
    model = FeedbackModel(_config(case), device=DEV, seed=seed)
    if case["kind"] == "model":
        return model
    for side in "kv":
        weight = model.router[side][0]
        weight.copy_(normal(*weight.shape, scale=0.003))
    return model


def prepare(case: dict, seed: int) -> dict:
    kind, normal = case["kind"], _Normal(seed)
    heads, kv_heads, dim = case["heads"], case["kv_heads"], case["dim"]
    batch = case["batch"]
    state: dict = {"case": case}
    if kind in ("decode", "prefill"):
        queries, capacity = case.get("queries", 1), case["capacity"]
        state["q"] = normal(batch, heads, queries, dim)
        state["k"], state["v"] = normal(batch, kv_heads, capacity, dim), normal(batch, kv_heads, capacity, dim)
        state["lengths"] = torch.from_numpy(_lengths(case, seed)).to(DEV)
        state["mask"] = None
        if case.get("masked"):
            state["mask"] = torch.rand(batch, capacity, generator=normal.gen, device=DEV) < 0.5
            state["mask"][:, :8] = True
    elif kind == "loop":
        channels, start, capacity = case["channels"], case["prefix"] + 1, case["prefix"] + 257
        folded = channels * kv_heads
        keys, values = normal(batch, folded, capacity, dim), normal(batch, folded, capacity, dim)
        angle = torch.arange(capacity, device=DEV)[:, None] * 10000.0 ** (
            -torch.arange(0, dim, 2, device=DEV).float() / dim
        ).repeat(2)
        state.update(
            start=start, weight=1 + 0.1 * normal(channels, dim, dtype=torch.float32), cos=angle.cos(), sin=angle.sin(),
            query=normal(case["layers"], batch, heads, 1, dim), new_key=normal(batch, channels, kv_heads, 1, dim),
            new_value=normal(batch, channels, kv_heads, 1, dim), layer_channels=[i % channels for i in range(case["layers"])],
        )
        length = torch.full((1,), start, device=DEV, dtype=torch.long)
        state["loop"] = DecodeLoop(keys, values, length, state["layer_channels"], state["weight"], state["cos"], state["sin"],
                                   query_heads=heads)
    elif kind == "jacobi":
        length, slots = case["length"], case["length"] + int(case["dummy"])
        state["docs"] = torch.from_numpy(_documents(batch, length, seed)).to(DEV)
        state["leaves"] = [
            [normal(batch, h, n, dim).requires_grad_() for h, n in ((heads, length), (kv_heads, slots), (kv_heads, slots))]
            for _ in range(case["layers"])
        ]
        state["grad"] = normal(batch, length, heads, dim)
        if not case["fresh"]:
            state["metadata"] = prepare_strict_causal_metadata(state["docs"], length, use_dummy_token=case["dummy"])
    elif kind == "cyclic":
        length, stride, slots = case["length"], case["stride"], case["length"] + int(case["dummy"])
        state["groups"] = [torch.arange(r, length, stride, device=DEV) for r in range(stride)]
        if case["documents"]:
            state["docs"] = torch.from_numpy(_documents(batch, length, seed)).to(DEV)
        # keys and values are channel views of the pool, as a layer reads them
        pool = [normal(batch, case["layers"], kv_heads, slots, dim) for _ in range(2)]
        state["layers"] = []
        for layer in range(case["layers"]):
            k, v = (p[:, layer].detach().requires_grad_(case["backward"]) for p in pool)
            qs = [normal(batch, heads, g.numel(), dim).requires_grad_(case["backward"]) for g in state["groups"]]
            state["layers"].append((qs, k, v))
        if case["backward"]:
            state["grads"] = [normal(batch, g.numel(), heads, dim).transpose(1, 2) for g in state["groups"]]
        state["metadata"] = None
        if case["documents"] and not case["fresh"]:
            state["metadata"] = prepare_feedback_metadata(state["docs"], state["groups"], slots, use_dummy_token=case["dummy"])
    elif kind in ("pool", "pool_train"):
        tokens, channels = case["tokens"], case["channels"]
        model = state["model"] = _model(case, seed, normal)
        state["stacked"] = normal(batch, tokens, case["layers"] + 1, case["hidden"], dtype=torch.float32)
        state["positions"] = torch.arange(tokens, device=DEV) * 8 + 1  # a residue of a group of 8
        state["rope"] = model.rope(state["positions"].expand(batch, tokens))
        if kind == "pool":
            state["pool"] = model.new_pool(batch, 8 * tokens + 1)
        else:
            leaf = lambda t: t.detach().clone().requires_grad_()  # noqa: E731
            state["stacked"].requires_grad_()
            state["pre_mix"], state["gain"] = ([leaf(w[s]) for s in "kv"] for w in (model.pre_mix, model.gain))
            state["router"] = [tuple(leaf(t) for t in model.router[s]) for s in "kv"]
            state["key"] = normal(batch, channels, kv_heads, tokens, dim).requires_grad_()
            state["weight"] = leaf(1 + 0.1 * normal(channels, dim))
            state["grads"] = [normal(channels, batch * tokens, case["hidden"]) for _ in range(2)]
            state["grads"].append(normal(batch, channels, kv_heads, tokens, dim))
    else:
        state["model"] = _model(case, seed, normal)
        state["ids"] = torch.randint(0, case["vocab"], (batch, case["length"]), generator=normal.gen, device=DEV)
        state["docs"] = torch.from_numpy(_documents(batch, case["length"], seed)).to(DEV)
    return state


# -------------------------------------------------------------------- run ----
def _decode(s):
    with torch.no_grad():
        return strict_causal_attention(s["q"], s["k"], s["v"], query_start=s["lengths"], kv_lengths=s["lengths"],
                                       use_dummy_token=s["case"]["dummy"], key_mask=s["mask"])


def _prefill(s):
    with torch.no_grad():
        return strict_causal_attention(s["q"], s["k"], s["v"], query_start=s["lengths"])


def _loop(s):
    loop = s["loop"]
    if loop.seen >= loop.capacity:  # the request is done: the next one starts behind the same prefix
        loop.cumulative_length.fill_(s["start"])
        loop.seen = s["start"]
    return loop(s["query"], s["new_key"], s["new_value"]), loop.keys, loop.values


def _jacobi(s):
    case = s["case"]
    metadata = s.get("metadata")
    if metadata is None:
        metadata = prepare_strict_causal_metadata(s["docs"], case["length"], use_dummy_token=case["dummy"])
    outs = []
    for leaves in s["leaves"]:
        out = strict_causal_attention(*leaves, metadata=metadata, use_dummy_token=case["dummy"])
        outs.append((out.detach(), *torch.autograd.grad(out, leaves, s["grad"])))
    return outs


def _cyclic(s):
    case, metadata = s["case"], s["metadata"]
    if metadata is None and case["documents"]:
        metadata = prepare_feedback_metadata(s["docs"], s["groups"], case["length"] + int(case["dummy"]),
                                             use_dummy_token=case["dummy"])
    outs = []
    with torch.set_grad_enabled(case["backward"]):
        for qs, k, v in s["layers"]:
            for residue, q in enumerate(qs):
                out = cyclic_attention(
                    q, k, v, query_stride=case["stride"], query_offset=residue, strict_past=not case["dummy"],
                    metadata=None if metadata is None else metadata[residue], backend="tilelang",
                )
                if case["backward"]:
                    outs.append((out.detach(), *torch.autograd.grad(out, (q, k, v), s["grads"][residue])))
                else:
                    outs.append(out)
    return outs


def _pool(s):
    write_sources(s["model"], s["stacked"], *s["pool"], s["positions"], s["rope"])
    return s["pool"]


def _pool_train(s):
    (w_k, b_k), (w_v, b_v) = s["router"]
    config = s["model"].config
    mixed = kv_pool.projection_inputs(
        s["stacked"], s["pre_mix"], s["router"], s["gain"], eps=config.rms_norm_eps, mix_eps=config.mix_norm_eps,
        router_layer_stride=config.router_layer_stride,
    )
    keys = kv_pool.k_norm_rope(s["key"], s["weight"], *s["rope"], eps=config.rms_norm_eps)
    leaves = [s["stacked"], *s["pre_mix"], w_k, b_k, w_v, b_v, *s["gain"], s["key"], s["weight"]]
    grads = torch.autograd.grad([*mixed, keys], leaves, s["grads"])
    return [t.detach() for t in (*mixed, keys)], grads


def _whole(s):
    model = s["model"]
    hidden, keys, values, _ = forward_cyclic(model, s["ids"], s["docs"])
    with torch.no_grad():
        return hidden, keys, values, model.logits(hidden[:, -1:])


_RUN = dict(decode=_decode, prefill=_prefill, loop=_loop, jacobi=_jacobi, cyclic=_cyclic, pool=_pool, pool_train=_pool_train,
            model=_whole)


def run(state: dict):
    return _RUN[state["case"]["kind"]](state)


# ------------------------------------------------------------------- work ----
def _pairs(case: dict) -> int:
    """Visible (query, key) pairs of one head over a whole row set of documents."""
    batch, length = case["batch"], case["length"]
    if case["kind"] == "cyclic" and not case["documents"]:
        sizes = np.full(batch, length, dtype=np.int64)
    else:
        docs = _documents(batch, length, 1)
        sizes = np.concatenate([np.bincount(row) for row in docs]).astype(np.int64)
    return int((sizes * (sizes - 1) // 2).sum()) + (batch * length if case.get("dummy", True) else 0)


def _pool_work(case: dict, tokens: int) -> tuple[float, float]:
    """Bytes and flops of the producer over `tokens` tokens, fp32 sources read
    once, each side's mixtures written once."""
    sources, hidden, channels = case["layers"] + 1, case["hidden"], case["channels"]
    read = (sources + 1) // 2  # the router reads every second source
    logits = channels * sources
    weights = 2 * 2 * (logits * read * hidden + sources * hidden + channels * hidden)
    return (
        tokens * (4 * sources * hidden + 2 * 2 * channels * hidden) + weights,
        2.0 * 2 * tokens * (logits * read * hidden + logits * hidden),
    )


def work(case: dict) -> dict:
    kind, heads, kv_heads, dim, batch = case["kind"], case["heads"], case["kv_heads"], case["dim"], case["batch"]
    if kind in ("decode", "prefill"):
        queries, lengths = case.get("queries", 1), _lengths(case, 1).astype(np.int64)
        pairs = int((lengths * queries + queries * (queries - 1) // 2).sum())
        slots = int(lengths.sum()) + batch * (queries - 1 + int(case.get("dummy", False)))
        nbytes = 2 * 2 * slots * kv_heads * dim + 2 * 2 * batch * heads * queries * dim
        share = 0.5 if case.get("masked") else 1.0  # the masked half of the slots need not be read
        return {"bytes": share * nbytes, "flops": share * 4.0 * dim * heads * pairs}
    if kind == "loop":
        slots, layers = case["prefix"] + 1, case["layers"]
        # a channel that several layers read is read once
        reads = 2 * 2 * batch * kv_heads * slots * dim * min(layers, case["channels"])
        rows = 2 * 2 * layers * batch * heads * dim + 2 * 2 * 2 * batch * case["channels"] * kv_heads * dim
        return {"bytes": reads + rows, "flops": 4.0 * dim * heads * batch * slots * layers}
    if kind == "jacobi":
        layers, slots = case["layers"], case["length"] + int(case["dummy"])
        q, kv = 2 * batch * heads * case["length"] * dim, 2 * 2 * batch * kv_heads * slots * dim
        # q, k, v and the output's gradient in; the output and three gradients out
        return {"bytes": layers * (4 * q + 2 * kv), "flops": layers * 14.0 * dim * heads * _pairs(case)}
    if kind == "cyclic":
        layers, slots = case["layers"], case["length"] + int(case["dummy"])
        q, kv = 2 * batch * heads * case["length"] * dim, 2 * 2 * batch * kv_heads * slots * dim
        calls = case["stride"]
        if case["backward"]:  # every residue call gives whole key and value gradients
            return {"bytes": layers * (4 * q + kv + calls * kv), "flops": layers * 14.0 * dim * heads * _pairs(case)}
        return {"bytes": layers * (2 * q + kv), "flops": layers * 4.0 * dim * heads * _pairs(case)}
    tokens = batch * case.get("tokens", case.get("length", 0))
    nbytes, flops = _pool_work(case, tokens)
    hidden, channels = case["hidden"], case["channels"]
    row = channels * kv_heads * dim
    if kind == "pool":
        return {"bytes": nbytes - 4 * tokens * channels * hidden + 2 * 2 * (hidden * row + tokens * row),
                "flops": flops + 2 * 2.0 * tokens * hidden * row}
    if kind == "pool_train":
        # the sources' gradient, the mixtures' gradients, the weights' gradients; the key rows and theirs
        extra = tokens * (4 * (case["layers"] + 1) * hidden + 2 * 2 * channels * hidden) + 2 * 4 * tokens * row
        return {"bytes": nbytes + extra, "flops": 3 * flops}
    # the layers' weights are read per group and pass, activations stay on the card
    calls, layers = case["groups"] * case["passes"], case["layers"]
    per_layer = 2 * heads * dim * hidden + 9 * hidden * hidden
    weights = 2.0 * (layers * per_layer + 2 * hidden * row) + 2.0 * case["vocab"] * hidden
    runs = case["passes"] + 1  # the pool is written once before the passes
    return {
        "bytes": calls * weights + runs * (nbytes + 2 * 2 * tokens * row),
        "flops": case["passes"] * layers * (2.0 * tokens * per_layer + 4.0 * dim * heads * _pairs(case))
        + runs * (flops + 2 * 2.0 * tokens * hidden * row) + 2.0 * batch * case["vocab"] * hidden,
    }


def tolerance(case: dict) -> dict:
    """bf16 results: about four times what one rounding of probabilities,
    mixtures or score gradients in another order shows (measured against
    `exact`: attention 2e-3 to 3e-3, the pool's rows 5e-3, the whole prefill
    1e-2, where layers, groups and passes follow each other)."""
    return {"rel": 3e-2 if case["kind"] == "model" else 2e-2 if case["kind"] in ("pool", "pool_train") else 1e-2}


# ------------------------------------------------------------------ exact ----
def _attend(q, k, v, keep, scale):
    """float64 attention of (H, T, D) over (Hkv, N, D) under keep (T, N); rows that see nothing are zero."""
    group = q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(group, 0), v.repeat_interleave(group, 0)
    scores = (q @ k.transpose(1, 2).contiguous()) * scale
    scores = scores.masked_fill(~keep, -math.inf)
    top = scores.detach().amax(-1, keepdim=True).clamp_min(-1e300)
    weights = (scores - top).exp()
    return (weights @ v) / weights.sum(-1, keepdim=True).clamp_min(1e-300)


def _rows(q, k, v, keep, grad=None):
    """_attend row by row of the batch: the output (B, H, T, D), and the three gradients for `grad`."""
    outs = []
    for b in range(q.shape[0]):
        leaves = [t[b].detach().double().requires_grad_(grad is not None) for t in (q, k, v)]
        out = _attend(*leaves, keep(b), q.shape[-1] ** -0.5)
        grads = () if grad is None else torch.autograd.grad(out, leaves, grad[b].double())
        outs.append((out.detach(), *grads))
    return [torch.stack(t) for t in zip(*outs)]


def _keep(docs, slots, length: int, dummy: bool, b: int):
    """(T, N): the keys that the tokens `slots` see: earlier ones of their document, and the dummy."""
    token = torch.arange(length, device=DEV)
    keep = token[None] < slots[:, None]
    if docs is not None:
        keep = keep & (docs[b][None] == docs[b][slots][:, None])
    return torch.cat((torch.ones_like(keep[:, :1]), keep), 1) if dummy else keep


def _norm64(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _mixed64(stacked, pre_mix, router, gain, config):
    """The producer of one side in float64: (C, B*T, hidden)."""
    batch, tokens, sources, hidden = stacked.shape
    p = (_norm64(stacked, config.rms_norm_eps) * pre_mix).reshape(batch * tokens, sources, hidden)
    weight, bias = router
    logits = p[:, (sources - 1) % 2 :: 2].reshape(batch * tokens, -1) @ weight.t().contiguous() + bias
    mixed = _norm64(torch.bmm(logits.view(batch * tokens, -1, sources), p), config.mix_norm_eps) * gain
    return mixed.transpose(0, 1)


def _project64(model, stacked, rope):
    """Keys and values (B, C, Hkv, T, D) of the sources in float64."""
    c = model.config
    batch, tokens = stacked.shape[:2]
    out = []
    for side in "kv":
        rows = _mixed64(stacked, model.pre_mix[side].double(), [t.double() for t in model.router[side]],
                        model.gain[side].double(), c)
        rows = torch.bmm(rows.contiguous(), model.proj[side].double())
        out.append(rows.view(c.num_kv_channels, batch, tokens, c.num_kv_heads, c.head_dim).permute(1, 0, 3, 2, 4))
    key = _norm64(out[0], c.rms_norm_eps) * model.k_norm.double()[None, :, None, None]
    return _rope64(key, rope[0].double()[:, None, None], rope[1].double()[:, None, None]), out[1]


def _exact_model(s):
    model, docs = s["model"], s["docs"]
    c = model.config
    batch, length = s["ids"].shape
    rope = [t.double() for t in model.rope(document_positions(docs) + 1)]
    first = [t.double() for t in model.rope(torch.zeros(batch, 1, device=DEV))]
    x = model.embed.double()[s["ids"]]
    whole = torch.cat((model.dummy.double().expand(batch, 1, -1), x), 1)
    keys, values = _project64(model, whole[:, :, None].expand(-1, -1, c.num_sources, -1),
                              [torch.cat(t, 1) for t in zip(first, rope)])
    keys, values = keys.contiguous(), values.contiguous()
    groups = [torch.arange(g, length, c.cyclic_groups, device=DEV) for g in range(c.cyclic_groups)]
    weights = [{n: w.double() for n, w in p.items()} for p in model.layers]
    out = torch.empty_like(x)
    for _ in range(c.num_passes):
        for slots in groups:
            cos, sin = (t[:, slots][:, None] for t in rope)
            h, states = x[:, slots], []
            for layer, p in enumerate(weights):
                states.append(h)
                q = _norm64(h, c.rms_norm_eps) * p["input_norm"] @ p["q_proj"].t().contiguous()
                q = _norm64(q.view(batch, -1, c.num_heads, c.head_dim), c.rms_norm_eps) * p["q_norm"]
                q = _rope64(q.transpose(1, 2), cos, sin)
                ch = layer % c.num_kv_channels
                keep = lambda b: _keep(docs, slots, length, True, b)[:, :length]  # noqa: B023,E731
                a = _rows(q, keys[:, ch, :, :length], values[:, ch, :, :length], keep)[0].transpose(1, 2).flatten(2)
                h = h + a @ p["o_proj"].t().contiguous()
                m = _norm64(h, c.rms_norm_eps) * p["post_norm"]
                h = h + (F.silu(m @ p["gate"].t().contiguous()) * (m @ p["up"].t().contiguous())) @ p["down"].t().contiguous()
            states.append(h)
            out[:, slots] = h
            k, v = _project64(model, torch.stack(states, 2), [t[:, slots] for t in rope])
            keys[:, :, :, slots + 1], values[:, :, :, slots + 1] = k, v
    logits = _norm64(out[:, -1:], c.rms_norm_eps) * model.final_norm.double() @ model.embed.double().t().contiguous()
    return out, keys, values, logits


def exact(case: dict, seed: int):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "decode":
        token = torch.arange(case["capacity"], device=DEV)
        def keep(b):
            seen = token[None] < s["lengths"][b] + int(case["dummy"])
            return seen if s["mask"] is None else seen & s["mask"][b][None]
        return _rows(s["q"], s["k"], s["v"], keep)[0].transpose(1, 2)
    if kind == "prefill":
        token, query = torch.arange(case["capacity"], device=DEV), torch.arange(case["queries"], device=DEV)
        return _rows(s["q"], s["k"], s["v"], lambda b: token[None] < s["lengths"][b] + query[:, None])[0].transpose(1, 2)
    if kind == "loop":
        loop, start, h = s["loop"], s["start"], case["kv_heads"]
        every = torch.ones(1, start, device=DEV, dtype=torch.bool)
        outs = [
            _rows(q, *(t[:, c * h : (c + 1) * h, :start] for t in (loop.keys, loop.values)), lambda b: every)[0].transpose(1, 2)
            for q, c in zip(s["query"], s["layer_channels"])
        ]
        keys, values = loop.keys.double(), loop.values.double()
        new = _norm64(s["new_key"].double(), 1e-6) * s["weight"].double()[None, :, None, None]
        new = _rope64(new, s["cos"][start].double(), s["sin"][start].double())
        keys[:, :, start], values[:, :, start] = new.flatten(1, 2)[:, :, 0], s["new_value"].double().flatten(1, 2)[:, :, 0]
        return torch.stack(outs), keys, values
    if kind == "jacobi":
        slots = torch.arange(case["length"], device=DEV)
        outs = []
        for leaves in s["leaves"]:
            keep = lambda b: _keep(s["docs"], slots, case["length"], case["dummy"], b)  # noqa: E731
            out, *grads = _rows(*leaves, keep, s["grad"].transpose(1, 2))
            outs.append((out.transpose(1, 2), *grads))
        return outs
    if kind == "cyclic":
        outs = []
        for qs, k, v in s["layers"]:
            for residue, q in enumerate(qs):
                keep = lambda b: _keep(s.get("docs"), s["groups"][residue], case["length"], case["dummy"], b)  # noqa: B023,E731
                rows = _rows(q, k, v, keep, s["grads"][residue] if case["backward"] else None)
                outs.append(tuple(rows) if case["backward"] else rows[0])
        return outs
    if kind == "pool":
        keys, values = (t.double() for t in s["pool"])
        keys[:, :, :, s["positions"]], values[:, :, :, s["positions"]] = _project64(s["model"], s["stacked"].double(), s["rope"])
        return keys, values
    if kind == "pool_train":
        config = s["model"].config
        wide = lambda t: t.detach().double().requires_grad_()  # noqa: E731
        stacked, pre, gain = wide(s["stacked"]), [wide(t) for t in s["pre_mix"]], [wide(t) for t in s["gain"]]
        router = [tuple(wide(t) for t in pair) for pair in s["router"]]
        key, weight = wide(s["key"]), wide(s["weight"])
        mixed = [_mixed64(stacked, p, r, g, config) for p, r, g in zip(pre, router, gain)]
        cos, sin = (t.double()[:, None, None] for t in s["rope"])
        keys = _rope64(_norm64(key, config.rms_norm_eps) * weight[None, :, None, None], cos, sin)
        leaves = [stacked, *pre, *router[0], *router[1], *gain, key, weight]
        grads = torch.autograd.grad([*mixed, keys], leaves, [g.double() for g in s["grads"]])
        return [t.detach() for t in (*mixed, keys)], grads
    return _exact_model(s)
