"""The layer's fused steps and products (white_matter::residual_norm, query_norm_rope,
silu_mul, linear_*, pool_project) against the torch operations they replace, at the
edges of their row and lane splits, and a model layer through them against the
same layer through the torch operations.

Bounds: the kernels round where the torch operations do, so results are equal
except where the fp32 mean's summation order moves a value across a bf16
rounding boundary: one bf16 step (2^-7 relative at most), on few elements."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F

from white_matter_amd import cyclic_pass
from white_matter_amd.cyclic_pass import FeedbackConfig, FeedbackModel

pytestmark = pytest.mark.gpu
DEV = "cuda"
ops = torch.ops.white_matter


def _near(got, want, what):
    g, w = got.float(), want.float()
    assert g.shape == w.shape and got.dtype == want.dtype, what
    assert ((g == w) | ((g - w).abs() <= 2**-7 * w.abs() + 1e-6)).all(), what  # (equal infinities differ by nan)
    assert (g == w).float().mean() > 0.99, what


@pytest.mark.parametrize("weight_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(("shape", "sources"), [((1, 1, 8), 1), ((3, 5, 520), 4), ((2, 33, 1024), 1), ((1, 7, 1032), 3), ((1, 2, 4096), 2)])
@torch.no_grad()
def test_residual_norm(shape, sources, weight_dtype):
    gen = torch.Generator(device=DEV).manual_seed(sum(shape))
    stacked = torch.randn(*shape[:2], sources, shape[2], generator=gen, device=DEV)
    x = stacked[:, :, -1]  # rows a multiple of the width apart
    delta = torch.randn(shape, generator=gen, device=DEV).bfloat16()
    weight = (1 + 0.1 * torch.randn(shape[2], generator=gen, device=DEV)).to(weight_dtype)
    out = torch.full((*shape[:2], sources + 1, shape[2]), float("nan"), device=DEV)
    h = ops.residual_norm(x, delta, out[:, :, 0], weight, 1e-6)
    want = x + delta.float()
    assert torch.equal(out[:, :, 0], want) and bool(out[:, :, 1:].isnan().all())
    _near(h, (F.rms_norm(want, (shape[2],), None, 1e-6) * weight.float()).bfloat16(), "norm of the sum")
    _near(ops.residual_norm(x, None, None, weight, 1e-6), (F.rms_norm(x, (shape[2],), None, 1e-6) * weight.float()).bfloat16(), "norm")
    assert ops.residual_norm(x, delta, out[:, :, 0], None, 1e-6).numel() == 0
    # rows that are not equally spaced, and a misaligned weight
    odd = torch.randn(shape[0] + 1, shape[1] + 2, shape[2], generator=gen, device=DEV)[1:, 1:-1]
    shifted = torch.cat((weight[:1], weight))[1:]
    _near(ops.residual_norm(odd, None, None, shifted, 1e-6), (F.rms_norm(odd, (shape[2],), None, 1e-6) * weight.float()).bfloat16(), "odd rows")


@pytest.mark.parametrize(("batch", "length", "heads", "dim"), [(1, 1, 1, 64), (3, 5, 12, 96), (2, 33, 16, 128), (8, 1, 16, 64)])
@torch.no_grad()
def test_query_norm_rope(batch, length, heads, dim):
    gen = torch.Generator(device=DEV).manual_seed(dim + length)
    q = torch.randn(batch, length, heads * dim, generator=gen, device=DEV).bfloat16()
    weight = (1 + 0.1 * torch.randn(dim, generator=gen, device=DEV)).bfloat16()
    angle = torch.rand(batch, length + 2, dim // 2, generator=gen, device=DEV) * 50
    cos, sin = (torch.cat((t, t), -1)[:, 1:-1] for t in (angle.cos(), angle.sin()))
    got = ops.query_norm_rope(q, weight, cos, sin, heads, 1e-6)
    y = F.rms_norm(q.view(batch, length, heads, dim).float(), (dim,), None, 1e-6) * weight.float()
    y = y.bfloat16().float()
    rot = torch.cat((-y[..., dim // 2 :], y[..., : dim // 2]), -1)
    # (the sum of the two products may cancel: one bf16 step of the larger one)
    want = (y * cos[:, :, None] + rot * sin[:, :, None]).bfloat16()
    assert got.shape == want.shape and (got == want).float().mean() > 0.99
    assert ((got.float() - want.float()).abs() <= 2**-7 * (y.abs() + rot.abs())).all()


@pytest.mark.parametrize("n", [8, 4096 * 2048 + 8])
@torch.no_grad()
def test_silu_mul(n):
    gen = torch.Generator(device=DEV).manual_seed(n)
    gate, up = (torch.randn(n, generator=gen, device=DEV).mul(4).bfloat16() for _ in range(2))
    gate[:3] = torch.tensor([float("inf"), -200.0, 0.0])
    _near(ops.silu_mul(gate, up), F.silu(gate) * up, "silu")


@pytest.mark.parametrize("tokens", [1, 37])
def test_layer_matches_the_torch_operations(tokens):
    config = FeedbackConfig(vocab_size=64, hidden_size=136, intermediate_size=264, num_layers=2, num_heads=4, num_kv_heads=2,
                            head_dim=64, num_kv_channels=2)
    model = FeedbackModel(config, device=DEV, seed=1)
    gen = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(2, tokens, 136, generator=gen, device=DEV)
    rope = model.rope(torch.arange(tokens, device=DEV).expand(2, tokens))
    attend = lambda q: q.transpose(1, 2) * 0.5  # noqa: E731
    with torch.no_grad():
        fused = model.layer(0, x, attend, rope)
        top, states = model.layers_forward(x, lambda i, q: attend(q), rope)
        assert torch.equal(states[0], x) and torch.equal(states[1], fused) and torch.equal(states[2], top)
    with torch.enable_grad():
        eager = model.layer(0, x.requires_grad_(), attend, rope)  # differentiable: the torch operations
        eager.sum().backward()
    # a bf16 rounding moved in the norm reaches the layer's output through two products
    assert (fused - eager.detach()).norm() <= 2e-3 * (eager.detach() - x.detach()).norm()


@pytest.mark.parametrize(
    ("rows", "inner", "outer"),
    [(1, 8, 8), (33, 136, 72), (64, 128, 64), (65, 1160, 200), (513, 264, 1032), (1100, 512, 1536)],
)
@torch.no_grad()
def test_linear(rows, inner, outer):
    """Plain and gated products, either side of both row tiles, with partial
    stages and tiles, against float64. Bounds: one bf16 rounding of the result
    and the fp32 sums' error, inner * 2^-24 of the sum of magnitudes."""
    gen = torch.Generator(device=DEV).manual_seed(rows + inner)
    wide = torch.randn(1, rows + 1, inner + 3, generator=gen, device=DEV).bfloat16()
    x = wide[:, 1:, 3:]  # rows that the kernel cannot read in place
    gate, up = (torch.randn(outer, inner, generator=gen, device=DEV).mul(inner**-0.5).bfloat16() for _ in range(2))
    xd, gd, ud = x.double(), gate.double(), up.double()
    p, u = xd @ gd.t(), xd @ ud.t()
    slack = lambda w: inner * 2**-24 * (xd.abs() @ w.abs().t())  # noqa: E731
    got = ops.linear_rows(x, gate)
    assert got.shape == p.shape and ((got.double() - p).abs() <= 2**-8 * p.abs() + slack(gd)).all()
    want = F.silu(p) * u
    # both products, the activation (slope at most 1.1) and the result are rounded to bf16
    bound = 1.1 * u.abs() * (2**-8 * p.abs() + slack(gd)) + F.silu(p).abs() * slack(ud) + 3 * 2**-8 * want.abs()
    bound = 1.02 * bound + 1e-30  # (terms of second order, fp32 steps)
    assert ((ops.linear_gated(x, gate, up).double() - want).abs() <= bound).all()


@pytest.mark.parametrize(("batch", "length", "inner", "heads", "dim"), [(1, 1, 8, 1, 64), (3, 11, 200, 12, 96), (2, 33, 136, 3, 128), (5, 13, 512, 8, 64)])
@torch.no_grad()
def test_linear_query(batch, length, inner, heads, dim):
    gen = torch.Generator(device=DEV).manual_seed(dim + inner)
    x = torch.randn(batch, length, inner, generator=gen, device=DEV).bfloat16()
    proj = torch.randn(heads * dim, inner, generator=gen, device=DEV).mul(inner**-0.5).bfloat16()
    weight = (1 + 0.1 * torch.randn(dim, generator=gen, device=DEV)).bfloat16()
    angle = torch.rand(batch, length + 2, dim // 2, generator=gen, device=DEV) * 50
    cos, sin = (torch.cat((t, t), -1)[:, 1:-1] for t in (angle.cos(), angle.sin()))
    got = ops.linear_query(x, proj, weight, cos, sin, heads, 1e-6)
    q = (x.double() @ proj.double().t()).view(batch, length, heads, dim)
    y = F.rms_norm(q, (dim,), None, 1e-6) * weight.double()
    rot = torch.cat((-y[..., dim // 2 :], y[..., : dim // 2]), -1)
    want = y * cos[:, :, None].double() + rot * sin[:, :, None].double()
    # four bf16 roundings: the product, the mean through it, y and the result, 2^-8 of each term
    assert got.shape == want.shape
    assert ((got.double() - want).abs() <= (2**-6 + 2**-11) * (y.abs() + rot.abs()) + 1e-6).all()


@pytest.mark.parametrize(("channels", "rows", "inner", "outer"), [(1, 1, 8, 8), (3, 65, 136, 264), (2, 64, 128, 128), (8, 130, 1160, 512)])
@torch.no_grad()
def test_pool_project(channels, rows, inner, outer):
    gen = torch.Generator(device=DEV).manual_seed(rows + inner)
    x = [torch.randn(channels, rows, inner, generator=gen, device=DEV).bfloat16() for _ in range(2)]
    w = [torch.randn(channels, inner, outer, generator=gen, device=DEV).mul(inner**-0.5).bfloat16() for _ in range(2)]
    for got, a, b in zip(ops.pool_project(*x, *w), x, w, strict=True):
        a, b = a.double(), b.double()
        want = torch.bmm(a, b)
        # one bf16 rounding and the fp32 sums
        assert got.shape == want.shape and ((got.double() - want).abs() <= 2**-8 * want.abs() + inner * 2**-24 * torch.bmm(a.abs(), b.abs())).all()


@pytest.mark.parametrize(("tokens", "dim", "strided"), [(1, 96, False), (37, 128, True), (70, 64, True)])
@torch.no_grad()
def test_own_products_match_the_library(monkeypatch, tokens, dim, strided):
    """A layer and the pool projection on either side of the size rule, with
    weights that lie otherwise than the kernels read them."""
    config = FeedbackConfig(vocab_size=64, hidden_size=136, intermediate_size=264, num_layers=2, num_heads=4, num_kv_heads=2,
                            head_dim=dim, num_kv_channels=2)
    model = FeedbackModel(config, device=DEV, seed=3)
    if strided:
        p = model.layers[0]
        for name in ("q_proj", "o_proj", "gate", "up", "down"):
            p[name] = p[name].t().contiguous().t()
        model.proj = {side: torch.cat((w, w), -1)[..., : w.shape[-1]] for side, w in model.proj.items()}
    gen = torch.Generator(device=DEV).manual_seed(4)
    x = torch.randn(2, tokens, 136, generator=gen, device=DEV)
    stacked = torch.randn(2, tokens, 3, 136, generator=gen, device=DEV)
    rope = model.rope(torch.arange(tokens, device=DEV).expand(2, tokens))
    run = lambda: (model.layer(0, x, lambda q: q.transpose(1, 2) * 0.5, rope), *model.project(stacked))  # noqa: E731
    own = run()
    for name in ("_PLAIN_TILES", "_GATED_TILES", "_POOL_TILES"):
        monkeypatch.setattr(cyclic_pass, name, 0)
    library = run()
    # sums in another order move bf16 roundings, which reach the layer's output through two products
    assert (own[0] - library[0]).norm() <= 2e-3 * (library[0] - x).norm()
    for a, b in zip(own[1:], library[1:], strict=True):
        _near(a, b, "projection")


def _small_model(tokens, seed=5, **config):
    config = FeedbackConfig(vocab_size=64, hidden_size=136, intermediate_size=264, num_layers=2, num_heads=4, num_kv_heads=2,
                            head_dim=64, num_kv_channels=2, **config)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x, t = (torch.randn(2, tokens, 136, generator=gen, device=DEV) for _ in range(2))
    return FeedbackModel(config, device=DEV, seed=seed), x, t


def _attend(q):
    return q.transpose(1, 2) * 0.5


@pytest.mark.parametrize("call", ["layer", "layers_forward", "layers_stacked", "logits"])
def test_forward_mode_and_vmap_without_gradients(call):
    """Tangents and batched inputs pass through the model as with gradients on,
    where the torch operations run. The results are equal; a tangent and a
    vmapped call are within 2^-8, one bf16 rounding of every element: torch's
    derivative formulas and products differ in fp32 with gradients on, under
    jvp, for dual numbers and in a batch, which moves their bf16 roundings."""
    model, x, t = _small_model(5)
    rope = model.rope(torch.arange(5, device=DEV).expand(2, 5))
    fn = {
        "layer": lambda x: model.layer(0, x, _attend, rope),
        "layers_forward": lambda x: model.layers_forward(x, lambda i, q: _attend(q), rope)[0],
        "layers_stacked": lambda x: model.layers_stacked(x, lambda i, q: _attend(q), rope)[1],
        "logits": model.logits,
    }[call]
    near = lambda a, b: (a.float() - b.float()).norm() <= 2**-8 * b.float().norm()  # noqa: E731
    want, tangent = torch.func.jvp(fn, (x,), (t,))
    assert tangent.abs().max() > 0
    with torch.no_grad():
        got = torch.func.jvp(fn, (x,), (t,))
        assert torch.equal(got[0], want) and near(got[1], tangent)
        with fwAD.dual_level():
            dual = fwAD.unpack_dual(fn(fwAD.make_dual(x, t)))
            assert dual.tangent is not None, "the tangent was dropped"
            assert torch.equal(dual.primal, want) and near(dual.tangent, tangent)
        batched = torch.func.vmap(fn)(torch.stack((x, t)))
    for one, row in zip(batched, (x, t), strict=True):
        assert near(one, fn(row))


@torch.no_grad()
def test_tangents_of_weights_and_tables_without_gradients():
    """A tangent that only a weight, the RoPE tables or the attention carries."""
    model, x, _ = _small_model(5)
    cos, sin = model.rope(torch.arange(5, device=DEV).expand(2, 5))
    p = model.layers[0]
    with fwAD.dual_level():
        tangent = lambda attend, rope: fwAD.unpack_dual(model.layer(0, x, attend, rope)).tangent  # noqa: E731
        assert tangent(_attend, (cos, sin)) is None
        assert tangent(_attend, (fwAD.make_dual(cos, torch.ones_like(cos)), sin)) is not None
        assert tangent(lambda q: fwAD.make_dual(_attend(q).contiguous(), torch.ones(2, 5, 4, 64, device=DEV).bfloat16()), (cos, sin)) is not None
        kept = p["up"]
        p["up"] = fwAD.make_dual(kept, torch.ones_like(kept))
        assert tangent(_attend, (cos, sin)) is not None
        p["up"] = kept


@pytest.mark.parametrize("tokens", [1, 37])
@torch.no_grad()
def test_rope_tables_of_other_forms(tokens):
    """Tables that broadcast over rows or tokens and tables of 16-bit floats
    give what their expanded float32 form gives; float64 tables and tables of
    other shapes run the torch operations."""
    model, x, _ = _small_model(tokens)
    cos, sin = model.rope(torch.arange(tokens, device=DEV)[None] + 3)
    run = lambda c, s: model.layer(0, x, _attend, (c, s))  # noqa: E731
    expand = lambda *tables: tuple(t.float().expand(2, tokens, 64).contiguous() for t in tables)  # noqa: E731
    want = run(*expand(cos, sin))
    assert torch.equal(run(cos, sin), want)
    assert torch.equal(run(cos.expand(2, tokens, 64), sin), want)
    top, states = model.layers_forward(x, lambda i, q: _attend(q), (cos, sin))
    assert torch.equal(states[1], want)
    for one in (cos[:, :1], cos[:, :1].expand(2, 1, 64), cos[:, :, :1]):
        assert torch.equal(run(one, sin), run(*expand(one, sin)))
    for dtype in (torch.bfloat16, torch.float16):
        c, s = cos.to(dtype), sin.to(dtype)
        assert torch.equal(run(c, s), run(*expand(c, s)))
        assert torch.equal(run(c, sin), run(*expand(c, sin)))
    for c, s in ((cos.double(), sin.double()), (cos[0, :1], sin[0, :1])):
        with torch.enable_grad():
            eager = run(c, s)
        assert torch.equal(run(c, s), eager)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float64])
@torch.no_grad()
def test_norm_weights_of_other_types(dtype):
    """Norm weights are read in float32, as the torch operations cast them."""
    model, x, _ = _small_model(9)
    rope = model.rope(torch.arange(9, device=DEV).expand(2, 9))
    run = lambda: (model.layer(0, x, _attend, rope), *model.layers_forward(x, lambda i, q: _attend(q), rope)[1], model.logits(x))  # noqa: E731
    gen = torch.Generator(device=DEV).manual_seed(1)
    weights = {n: (1 + 0.1 * torch.randn(model.layers[0][n].shape, generator=gen, device=DEV)).to(dtype)
               for n in ("input_norm", "q_norm", "post_norm")}
    results = []
    for cast in (dtype, torch.float32):
        for p in model.layers:
            p.update({n: w.to(cast) for n, w in weights.items()})
        model.final_norm = weights["input_norm"].to(cast)
        results.append(run())
    for got, want in zip(*results, strict=True):
        assert torch.equal(got, want)


def test_autocast_to_another_type():
    """Under autocast to float16 the products round to float16, as with
    gradients on; under autocast to the model's own type nothing changes."""
    model, x, _ = _small_model(9)
    rope = model.rope(torch.arange(9, device=DEV).expand(2, 9))
    run = lambda: (model.layer(0, x, _attend, rope), model.logits(x))  # noqa: E731
    with torch.autocast("cuda", torch.float16):
        want = run()
        with torch.no_grad():
            got = run()
    assert all(torch.equal(g, w) and g.dtype == w.dtype for g, w in zip(got, want, strict=True))
    with torch.no_grad():
        plain = run()
        with torch.autocast("cuda", torch.bfloat16):
            same = run()
    assert all(torch.equal(g, w) and g.dtype == w.dtype for g, w in zip(same, plain, strict=True))


@torch.no_grad()
def test_layer_outputs_own_their_memory():
    """The top output and the sources are contiguous tensors of their own: a
    caller may view them flat, and keeping one does not keep the others."""
    model, x, _ = _small_model(9)
    rope = model.rope(torch.arange(9, device=DEV).expand(2, 9))
    top, states = model.layers_forward(x, lambda i, q: _attend(q), rope)
    assert states[0] is x and top is states[-1] and len(states) == 3
    for t in states:
        assert t.view(-1, 136).shape == (18, 136) and t.untyped_storage().nbytes() == t.numel() * 4
    stacked = model.layers_stacked(x, lambda i, q: _attend(q), rope)
    assert torch.equal(stacked[0], top) and torch.equal(stacked[1], torch.stack(states, 2))


@torch.no_grad()
def test_a_subclass_keeps_its_own_layers():
    """A model that redefines a layer, or how the layers follow each other,
    gets its own in the pass too."""

    class OwnLayer(FeedbackModel):
        def layer(self, index, x, attend, rope):
            return super().layer(index, x, attend, rope) + 1

    class OwnLayers(FeedbackModel):
        def layers_forward(self, x, attend_layer, rope):
            return x * 2, [x] * self.config.num_sources

    plain, x, _ = _small_model(9)
    rope = plain.rope(torch.arange(9, device=DEV).expand(2, 9))
    for kind in (OwnLayer, OwnLayers):
        model = kind(plain.config, device=DEV, seed=5)
        top, states = model.layers_forward(x, lambda i, q: _attend(q), rope)
        got = model.layers_stacked(x, lambda i, q: _attend(q), rope)
        assert torch.equal(got[0], top) and torch.equal(got[1], torch.stack(states, 2))
    plain.layer = lambda index, x, attend, rope: x + 1
    assert torch.equal(plain.layers_stacked(x, lambda i, q: _attend(q), rope)[0], x + 1 + 1)
