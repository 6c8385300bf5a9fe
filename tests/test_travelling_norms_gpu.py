"""Norms that travel with the products of up to 16 rows, and the packed product that rotates and fills the cache, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]
BITS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8}       # half a last place: 24 and 8 bits of significand


@pytest.fixture(scope="module")
def ops(device):
    from tessweave_engine_amd.kernels import ops
    return ops


def rand(shape, dtype, device, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype).to(device)


def close(got, want, sizes, dtype, rounded=True):
    """SIZES: the sum of the products' magnitudes behind each element. float32 sums of products of K are off by less than 2^-18 of it here
    (K up to 8,192 in any order: the errors' random walk, not its bound); what is rounded once more by half a last place."""
    bound = 2.0 ** -18 * sizes + (BITS[dtype] * want.abs() if rounded else 0)
    assert torch.isfinite(got.float()).all()
    assert ((got.double() - want).abs() <= 1.01 * bound + 1e-30).all(), float(((got.double() - want).abs() / (bound + 1e-30)).max())


# rows, columns, K: one and all rows of a tile; the fewest columns, sums that fill a lane's share exactly and not; K of four, eight and sixteen waves, and ragged
LEAVES = [(1, 64, 64), (16, 64, 72), (3, 896, 4864), (8, 2048, 5632), (5, 2112, 3000), (16, 4096, 1024), (1, 4096, 8192)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", LEAVES)
@pytest.mark.parametrize("form", ["plain", "two norms", "after a norm", "after rows as they are"])
def test_rows_left(ops, device, dtype, m, n, k, form):
    x, w = rand((m, k), dtype, device), rand((n, k), dtype, device, k ** -0.5, 1)
    bias, stream = rand((n,), torch.float32, device, 0.1, 2), rand((m, n), torch.float32, device, 1.0, 3)
    weight, second = 1 + rand((n,), torch.float32, device, 0.1, 4), 1 + rand((n,), torch.float32, device, 0.1, 5)
    before_weight, scale = 1 + rand((n,), torch.float32, device, 0.1, 6), 1 + rand((n,), torch.float32, device, 0.1, 7)
    rows, rows2 = (torch.full((m, n), float("nan"), dtype=dtype, device=device) for _ in range(2))
    sums, old = torch.full((m, n // 16), float("nan"), device=device), stream.double()
    product = x.double() @ w.double().T + bias.double()
    size = x.double().abs() @ w.double().abs().T + bias.abs().double()
    after = None
    if form.startswith("after"):
        before = None
        if form == "after a norm":
            before = ops.NormedRows(None, (old ** 2).view(m, n // 16, 16).sum(-1).float().contiguous(), 1e-6)
            old = old / torch.sqrt((old ** 2).mean(-1, keepdim=True) + 1e-6) * before_weight.double()
        after = (before, before_weight if before is not None else None, 0.7, scale)
        want, size = 0.7 * old + scale.double() * product, scale.abs().double() * size + old.abs()
    else:
        want, size = old + product, size + old.abs()
    left = ops.linear_leave(x, ops.shuffle_weight(w), stream, weight, 1e-6, rows, sums, bias=bias,
                            second=(second, rows2) if form == "two norms" else None, after=after)
    close(stream, want, size, torch.float32)
    close(rows, stream.double() * weight.double(), stream.abs().double(), dtype)         # of the stream as it was written
    assert left.rows is rows and (left.second is not None) == (form == "two norms")
    if left.second is not None:
        close(left.second.rows, stream.double() * second.double(), stream.abs().double(), dtype)
    else:
        assert torch.isnan(rows2.float()).all()
    torch.testing.assert_close(sums.double(), (stream.double() ** 2).view(m, n // 16, 16).sum(-1), rtol=2.0 ** -21, atol=0)


def normed(ops, m, k, dtype, device, seed=0):
    """`NormedRows` of float32 rows, and the rows behind the norm as the product meets them, in float64."""
    x = rand((m, k), torch.float32, device, 2.0, seed)
    rows = (x * (1 + rand((k,), torch.float32, device, 0.1, seed + 1))).to(dtype)
    sums = (x.double() ** 2).view(m, k // 16, 16).sum(-1).float().contiguous()
    return ops.NormedRows(rows, sums, 1e-5), rows.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-5)


# products of whole K and of K ranges, of two waves (more than a round of workgroups) and four, gated ones of either kernel
TAKES = [(1, 64, 64), (16, 1152, 896), (3, 9472, 3584), (8, 8192, 2048), (16, 4608, 3584), (2, 20000, 896), (5, 37888, 3584)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", TAKES)
@pytest.mark.parametrize("form", ["plain", "float32", "sums", "gated", "activation"])
def test_rows_taken(ops, device, dtype, m, n, k, form):
    if form == "gated":
        n = n // 32 * 32
    x, rows = normed(ops, m, k, dtype, device)
    w, bias = rand((n, k), dtype, device, k ** -0.5, 2), rand((n,), torch.float32, device, 0.1, 3)
    want, size = rows @ w.double().T, rows.abs() @ w.double().abs().T
    weight = ops.shuffle_weight(w)
    if form == "sums":
        splits = ops.linear_partial_splits_rows(weight, m)
        got = ops.linear_normed(x, weight, partial=torch.full((splits, m, n), float("nan"), device=device))
        return close(got.double().sum(0), want, size, torch.float32)
    want, size = want + bias.double(), size + bias.abs().double()
    if form == "gated":
        got = ops.linear_normed(x, weight, torch.empty(m, n // 2, dtype=dtype, device=device), bias=bias, activation="silu")
        gate, up = (v.view(m, n // 32, 2, 16)[:, :, i].reshape(m, -1) for v in (want,) for i in (0, 1))
        gs, us = (v.view(m, n // 32, 2, 16)[:, :, i].reshape(m, -1) for v in (size,) for i in (0, 1))
        # (silu's slope is below 1.1)
        return close(got, gate * torch.sigmoid(gate) * up, 1.1 * gs * up.abs() + us * gate.abs() + 2.0 ** -4 * (gate * up).abs(), dtype)
    if form == "activation":
        got = ops.linear_normed(x, weight, torch.empty(m, n, dtype=dtype, device=device), bias=bias, activation="relu_squared")
        return close(got, want.clamp(min=0) ** 2, 2 * size * want.abs() + 2.0 ** -18 * size ** 2, dtype)
    workspace = torch.empty(ops.linear_workspace_bytes(dtype, m, n, k) // 4 + 4, device=device)
    out = torch.empty(m, n, dtype=torch.float32 if form == "float32" else dtype, device=device)
    close(ops.linear_normed(x, weight, out, bias=bias, workspace=workspace), want, size, out.dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("with_norms", [False, True])
@pytest.mark.parametrize("m,q_heads,kv_heads,dim,rot,adjacent,k", [(1, 14, 2, 64, 64, False, 896), (16, 2, 1, 128, 64, False, 256), (7, 4, 4, 48, 32, True, 320),
                                                                 (9, 3, 1, 16, 16, False, 2048), (2, 1, 1, 80, 0, False, 128), (16, 16, 4, 256, 256, True, 64)])
def test_rotated_product(ops, device, dtype, with_norms, m, q_heads, kv_heads, dim, rot, adjacent, k):
    """Against the product, then `rope_kv_write`: the same values but for the product's float32 order."""
    width, page = (q_heads + 2 * kv_heads) * dim, 16
    x, rows = normed(ops, m, k, dtype, device)
    w, bias = rand((width, k), dtype, device, k ** -0.5, 2), rand((width,), torch.float32, device, 0.1, 3)
    angle = torch.arange(m * max(rot // 2, 1), device=device).view(m, -1)[:, :rot // 2].float() * 0.37
    cos, sin = (angle.cos(), angle.sin()) if rot else (None, None)
    slots = torch.tensor([(5 * i + 3) % (4 * page) if i != 4 else -1 for i in range(m)], dtype=torch.int32, device=device)
    keys, values = (torch.full((4, kv_heads, page, dim), -9.0, dtype=dtype, device=device) for _ in range(2))
    want_keys, want_values = keys.clone(), values.clone()
    if not with_norms:
        x, rows = x.rows, x.rows.double()
    qkv = torch.full((m, width), -9.0, dtype=dtype, device=device)
    ops.linear_rotate(x, ops.shuffle_weight(w), qkv, cos, sin, slots, keys, values, q_heads, kv_heads, dim, page, bias=bias, adjacent=adjacent)
    product = rows @ w.double().T + bias.double()
    size = rows.abs() @ w.double().abs().T + bias.abs().double()
    want = product.to(dtype)
    ops.rope_kv_write(want, cos, sin, slots, want_keys, want_values, q_heads, kv_heads, dim, page, adjacent=adjacent)
    # the product's own error, a rounding of either element of a pair that falls the other way, and the rotated one's: at most a pair's sizes
    slack = 2.0 ** -18 * float(size.max()) + 6 * BITS[dtype] * float(product.abs().max())
    torch.testing.assert_close(qkv[:, :q_heads * dim].float(), want[:, :q_heads * dim].float(), atol=slack, rtol=0)
    torch.testing.assert_close(keys.float(), want_keys.float(), atol=slack, rtol=0)
    torch.testing.assert_close(values.float(), want_values.float(), atol=slack, rtol=0)
    assert (keys == want_keys).float().mean() > (0.9 if dtype == torch.bfloat16 else 0.1) and ((keys == -9) == (want_keys == -9)).all()
    before = keys.clone()
    ops.linear_rotate(x, ops.shuffle_weight(w), qkv, cos, sin, None, None, None, q_heads, kv_heads, dim, page, write_cache=False, bias=bias, adjacent=adjacent)
    assert torch.equal(before, keys)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [64, 2048, 4096])
@pytest.mark.parametrize("eps", [(1e-6, 1e-6), (3.0, 1e-6), (1e-6, 0.5)])
def test_residual_norm_of_rows_behind_a_norm(ops, device, dtype, hidden, eps):
    """Two norms behind one another, each with its own eps."""
    x, y = rand((16, hidden), torch.float32, device, 3.0), rand((3, 16, hidden), torch.float32, device, 1.0, 1)
    w, before, scale = (1 + rand((hidden,), torch.float32, device, 0.1, s) for s in (2, 3, 4))
    out = torch.empty(16, hidden, dtype=dtype, device=device)
    unit = lambda v, eps: v / torch.sqrt((v ** 2).mean(-1, keepdim=True) + eps)       # noqa: E731
    want = unit(0.7 * unit(x.double(), eps[0]) * before.double() + scale.double() * y.double().sum(0), eps[1]) * w.double()
    ops.residual_norm(x, w, eps[1], out=out, add=y, scale=scale, alpha=0.7, before=(before, eps[0]))
    torch.testing.assert_close(x.double(), want, atol=3e-6, rtol=3e-6)             # (as this kernel's other forms)
    torch.testing.assert_close(out, x.to(dtype), atol=0, rtol=0)


def misaligned(t):
    """The same values four bytes behind a multiple of 16."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    assert flat.data_ptr() % 16 == 0
    flat[1:] = t.reshape(-1)
    return flat[1:].view(t.shape)


@pytest.mark.parametrize("which", ["w", "scale", "before", "all"])
def test_residual_norm_of_rows_behind_a_norm_with_any_weights(ops, device, which):
    """As with aligned ones, but for the order of the sums of squares."""
    x, y = rand((5, 896), torch.float32, device, 3.0), rand((3, 5, 896), torch.float32, device, 1.0, 1)
    given = {k: 1 + rand((896,), torch.float32, device, 0.1, i) for i, k in enumerate(("w", "scale", "before"))}
    want, out = x.clone(), torch.empty(5, 896, dtype=torch.bfloat16, device=device)
    ops.residual_norm(want, given["w"], 1e-6, add=y, scale=given["scale"], alpha=0.7, before=(given["before"], 0.5))
    given = {k: misaligned(v) if which in (k, "all") else v for k, v in given.items()}
    ops.residual_norm(x, given["w"], 1e-6, out=out, add=y, scale=given["scale"], alpha=0.7, before=(given["before"], 0.5))
    torch.testing.assert_close(x, want, atol=1e-6, rtol=1e-6)
    assert torch.equal(out, x.to(torch.bfloat16))


DESIGNS = [("qwen2", "A"), ("qwen2", "B"), ("kanavik", "wide"), ("dinutar", "wide"), ("rufusun", "wide"), ("tadalorn", "wide"), ("darolix", "wide"), ("darolix", "odd"),
           ("vulosun", "wide")]


@pytest.mark.parametrize("design,name", DESIGNS)
def test_captured_steps_with_norm_weights_anywhere(device, tmp_path, design, name):
    """Weights that were bound as slices of a larger buffer need not be aligned: captured float32 steps against eager ones with aligned weights,
    to 2e-5 of the logits' spread (sums in other orders). Tadalorn's mLSTM divides by a sum that may nearly cancel, which moves a row in any
    order of operations: one of its rows may lie beyond that, none beyond 1e-3 (as in the design's own tests)."""
    import importlib
    from kanavik_util import Driver, row_error
    from tessweave_engine_amd.parts.base import Norm
    from tessweave_engine_amd.parts.model import walk
    if design == "qwen2":
        from tiny_configs import make_folder
        make_folder(str(tmp_path), name)
        folder = str(tmp_path)
    else:
        util = importlib.import_module(design + "_util")
        config = util.CONFIGS[name]
        folder = util.write_folder(tmp_path, config, util.make_weights(config, seed=3))
    got = []
    for graphs in (False, True):
        d = Driver(folder, "float32", pages=24, page_size=4, graphs=graphs)
        tokens = {rid: [(s * i + 3) % d.model.vocab_size for i in range(12)] for rid, s in (("a", 7), ("b", 5))}
        if graphs:
            for part in walk(d.model):
                for attribute in ("weight", "bias") if isinstance(part, Norm) else ("mixer_scale", "ffn_scale"):
                    if getattr(part, attribute, None) is not None:
                        setattr(part, attribute, misaligned(getattr(part, attribute)))
        got.append(d.run([[("a", 1), ("b", 1)] for _ in range(12)], tokens))
        assert (d.stepper.graph_replays > 0) == (graphs and d.model.graph_safe_model)
        d.close()
    errors = sorted(e for rid in tokens for e in row_error(got[1][rid], got[0][rid]).tolist())
    assert errors[-2 if design == "tadalorn" else -1] < 2e-5 and errors[-1] < 1e-3


def remade(part, **members):
    """PART with a class of its own that overrides MEMBERS."""
    part.__class__ = type("Own" + type(part).__name__, (type(part),), members)


@pytest.mark.parametrize("which", ["attention", "feed-forward", "norm", "last norm", "embedding", "head", "block", "experts", "branch", "post norm", "wrapped", "encoding"])
def test_parts_with_a_forward_of_their_own(device, tmp_path, which):
    """A program's part that overrides `forward` of one of these is run as it is, whatever the part it comes from allows: captured float32 steps
    against eager ones, to 2e-5 of the logits' spread."""
    import importlib
    from kanavik_util import Driver, row_error
    design = {"experts": "darolix", "branch": "kanavik", "post norm": "dinutar"}.get(which, "qwen2")
    if design == "qwen2":
        from tiny_configs import make_folder
        make_folder(str(tmp_path), "B320")
        folder = str(tmp_path)
    else:
        util = importlib.import_module(design + "_util")
        folder = util.write_folder(tmp_path, util.CONFIGS["wide"], util.make_weights(util.CONFIGS["wide"], seed=3))
    got = []
    for graphs in (False, True):
        d = Driver(folder, "float32", pages=24, page_size=4, graphs=graphs)
        blocks, head, embedding = d.model.blocks, d.model.head, d.model.embedding

        def adds(base):
            def forward(self, ctx, *args, **options):          # (the stream is the last of a sublayer's arguments)
                left = base.forward(self, ctx, *args, **options)
                args[-1].add_(0.25)
                return left
            return forward

        def half(ctx, h):
            return torch.mul(h, 0.5, out=ctx.workspace.get("half", tuple(h.shape), h.dtype))

        def halves(base):
            return lambda self, ctx, *args, **options: base.forward(self, ctx, *args, **options).mul_(0.5)
        for block in blocks:
            if which == "attention":
                remade(block.mixer, forward=adds(type(block.mixer)))
            elif which == "feed-forward":
                remade(block.ffn, forward=adds(type(block.ffn)))
            elif which == "norm":
                remade(block.ffn_norm, forward=halves(type(block.ffn_norm)))
            elif which == "post norm":
                remade(block.mixer, forward=lambda self, ctx, run, h, x, accumulate=True, base=type(block.mixer):
                       base.forward(self, ctx, run, half(ctx, h), x, accumulate=accumulate))
            elif which == "experts" and getattr(block, "ffn", None) is not None:
                remade(block.ffn, forward=adds(type(block.ffn)))
            elif which == "branch":
                base = type(block.mixer.branches[0])
                remade(block.mixer.branches[0], forward=lambda self, ctx, run, proj, out, scale, base=base: base.forward(self, ctx, run, proj, out, 0.5 * scale))
            elif which == "wrapped":
                plain = block.mixer.forward
                block.mixer.forward = lambda ctx, run, h, x, plain=plain: plain(ctx, run, half(ctx, h), x)
        if which == "encoding":
            angle = torch.arange(64, device=device)[:, None] * 0.3 ** torch.arange(16, device=device)[None]
            kept = (angle.cos(), angle.sin())

            def tables(self, ctx):
                out = [ctx.workspace.get(name, (ctx.n_tokens, 16), torch.float32) for name in ("own.cos", "own.sin")]
                return tuple(torch.index_select(t, 0, ctx.positions[0], out=o) for t, o in zip(kept, out))
            for position in {id(block.mixer.position): block.mixer.position for block in blocks}.values():
                remade(position, tables=tables)
                position.inv_freq = position.rest = None
        if which == "block":
            base = type(blocks[1])

            def forward(self, ctx, run, x, pending=None):
                for part in pending if pending is not None else ():
                    x.add_(part)
                x.mul_(1.5)
                return base.forward(self, ctx, run, x, None)
            remade(blocks[1], forward=forward)
        elif which == "last norm":
            remade(d.model.final_norm, forward=halves(type(d.model.final_norm)))
        elif which == "embedding":
            remade(embedding, forward=lambda self, ctx, base=type(embedding): base.forward(self, ctx).mul_(3.0))
        elif which == "head":
            remade(head, forward=lambda self, ctx, h, base=type(head): base.forward(self, ctx, half(ctx, h)))
        tokens = {rid: [(s * i + 3) % d.model.vocab_size for i in range(8)] for rid, s in (("a", 7), ("b", 5))}
        got.append(d.run([[("a", 1), ("b", 1)] for _ in range(8)], tokens))
        assert (d.stepper.graph_replays > 0) == graphs
        d.close()
    assert max(row_error(got[1][rid], got[0][rid]).max() for rid in tokens) < 2e-5


@pytest.mark.parametrize("which", ["qkv", "o", "gate_up", "down", "side"])
def test_products_of_their_own(device, tmp_path, which):
    """A product that adds something of its own (and leaves no sums for another kernel to finish) does so for any number of rows: float32, a
    prompt's 24 rows at once against 5 at a time and one by one, captured."""
    from kanavik_util import CONFIGS, Driver, make_weights, row_error, write_folder
    from tiny_configs import make_folder
    if which == "side":
        folder = write_folder(tmp_path, CONFIGS["odd"], make_weights(CONFIGS["odd"], seed=3))
    else:
        make_folder(str(tmp_path), "B320")
        folder = str(tmp_path)
    got, tokens = [], {"a": [(7 * i + 3) % 97 for i in range(24)]}
    for schedule in ([24], [5, 5, 5, 5, 4], [1] * 24):
        d = Driver(folder, "float32", pages=24, page_size=4)
        for block in d.model.blocks:
            part = block.side.gate if which == "side" else getattr(block.ffn if which in ("gate_up", "down") else block.mixer, which)
            name, base = "forward_glu" if which == "gate_up" else "forward", type(part)

            def product(self, ctx, x, out, *args, base=base, name=name, **options):
                getattr(base, name)(self, ctx, x, out, *args, **options)
                return out.add_(0.125)
            remade(part, deferrable=lambda self, n: False, **{name: product})
        got.append(d.run([[("a", n)] for n in schedule], tokens)["a"])
        d.close()
    assert max(row_error(got[1], got[0]).max(), row_error(got[2], got[0]).max()) < 2e-5


@pytest.mark.parametrize("rot", [16, 20, 32])
def test_an_encoding_that_gives_its_tables_alone(device, tmp_path, rot):
    """How much of a head turns is what the tables say: an encoding need not name a size, and one that is no multiple of 16 is turned by the other
    kernel. Against the engine's own encoding."""
    from kanavik_util import Driver
    from tessweave_engine_amd.parts.base import PositionEncoding
    from tessweave_engine_amd.parts.positions import RotaryEmbedding
    from tiny_configs import make_folder

    class Tables(PositionEncoding):
        def __init__(self, inner):
            self.tables = inner.tables
    make_folder(str(tmp_path), "B320")
    got = []
    for wrap in (lambda p: p, Tables):
        d = Driver(str(tmp_path), "float32", pages=24, page_size=4)
        for block in d.model.blocks:
            encoding = RotaryEmbedding(32, 1e4, rotary_dim=rot)
            encoding.bind({}, torch.float32, device)
            block.mixer.position = wrap(encoding)
        tokens = {"a": [(7 * i + 3) % d.model.vocab_size for i in range(12)]}
        got.append(d.run([[("a", 5)]] + [[("a", 1)]] * 7, tokens)["a"])
        d.close()
    assert (got[0] == got[1]).all()


@pytest.mark.parametrize("requests", [1, 16, 17])                       # (17: no norm travels)
@pytest.mark.parametrize("ff,leaves", [(320, True), (8192, False)])      # (the second: a long K, where K ranges and a norm's kernel are faster)
@pytest.mark.parametrize("design", ["qwen2", "dinutar"])
def test_captured_steps_on_either_side_of_the_lines(ops, device, tmp_path, monkeypatch, design, ff, leaves, requests):
    """Layers whose last product leaves its rows, does not, and steps of more rows than may be left, against eager steps: float32, sums in other
    orders. The attention's product leaves its rows in all steps of up to 16."""
    from kanavik_util import Driver, row_error
    if design == "qwen2":
        from tessweave_engine_amd.config import config_from_dict
        from tessweave_engine_amd.weights import write_model_folder
        from tiny_configs import TINY_B
        folder = str(tmp_path)
        write_model_folder(folder, config_from_dict(dict(TINY_B, intermediate_size=ff, rms_norm_eps=1e-3)), 3)
    else:
        from dinutar_util import config, latent, make_weights, retention, write_folder
        c = config([latent(2, 16, 16, 32, 32, 0.25, ff=ff), retention(2, 32, 32, [0.9, 0.99], 32, ff=ff)], width=192, vocab=97, alpha=1.3, scale=0.7, buckets=7,
                   mul_prev=5, mul_cur=3)
        folder = write_folder(tmp_path, c, make_weights(c, seed=4))
    got, widths = [], []
    plain = ops.linear_leave
    monkeypatch.setattr(ops, "linear_leave", lambda x, *a, **k: widths.append(x.shape[1]) or plain(x, *a, **k))
    for graphs in (False, True):
        d = Driver(folder, "float32", pages=64, page_size=4, max_requests=requests, graphs=graphs)
        tokens = {f"r{i}": [(7 * i + 5 * j + 3) % d.model.vocab_size for j in range(6)] for i in range(requests)}
        assert not widths
        got.append(d.run([[(rid, 1) for rid in tokens] for _ in range(6)], tokens))
        assert graphs == (d.stepper.graph_replays > 0)
        d.close()
    assert bool(widths) == (requests <= 16) and (ff in widths) == (leaves and requests <= 16)
    assert max(row_error(got[1][rid], got[0][rid]).max() for rid in tokens) < 2e-5


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,hidden,form", [(1, 64, "norm"), (16, 896, "two norms"), (3, 4096, "norm"), (40, 2064, "rounded"), (5, 16, "rows alone"), (16, 3072, "no tables")])
def test_embed_begin(ops, device, dtype, n, hidden, form):
    """Against the gather, a table at a time and the sums in float64: the same bits where a value is only moved or rounded once."""
    table = rand((50, hidden), dtype, device, 1.5)
    ids = torch.tensor([(7 * i) % 50 for i in range(n - 1)] + [-2], dtype=torch.int32, device=device)
    feed = torch.tensor([3, 17], dtype=torch.int32, device=device)
    positions = torch.tensor([(311 * i) % 5000 for i in range(n)], dtype=torch.int32, device=device)
    weights = [1 + rand((hidden,), torch.float32, device, 0.1, s) for s in (1, 2)]
    rows = [torch.full((n, hidden), float("nan"), dtype=dtype, device=device) for _ in range(2)]
    sums = torch.full((n, hidden // 16), float("nan"), device=device)
    tables, want = [], []
    for half, magnitude, rest in ((32, 1.0, False), (64, 1.25, True), (1, 1.0, True), (5, 0.5, False))[:0 if form == "no tables" else 4]:
        freq = 10000.0 ** (-torch.arange(half, dtype=torch.float32) / half)
        rest = (freq * 1e-8).to(device) if rest else None
        pair = [torch.full((n, half), float("nan"), device=device) for _ in range(4)]
        tables.append((freq.to(device), rest, pair[0], pair[1], magnitude))
        ops.rope_table(positions, freq.to(device), pair[2], pair[3], magnitude, rest=rest)
        want.append(pair)
    options = {"norm": dict(norm=(weights[0], rows[0]), sums=sums), "two norms": dict(norm=(weights[0], rows[0]), second=(weights[1], rows[1]), sums=sums),
               "rounded": dict(rounded=rows[0])}.get(form, {})
    x = torch.full((n, hidden), float("nan"), device=device)
    left = ops.embed_begin(ids, table, x, feed=feed, positions=positions, tables=tables, **options)
    gathered = ops.embed_gather(ids, table, torch.empty_like(x), feed=feed)
    assert torch.equal(x, gathered)
    for cos, sin, want_cos, want_sin in want:
        assert torch.equal(cos, want_cos) and torch.equal(sin, want_sin)
    if form in ("norm", "two norms"):
        assert torch.equal(left.rows, (x * weights[0]).to(dtype)) and (left.second is None) == (form == "norm")
        torch.testing.assert_close(sums.double(), (x.double() ** 2).view(n, hidden // 16, 16).sum(-1), rtol=2.0 ** -21, atol=0)
        if form == "two norms":
            assert torch.equal(left.second.rows, (x * weights[1]).to(dtype))
    elif form == "rounded":
        assert left is None and torch.equal(rows[0], x.to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,c,top,splits", [(1, 64, 1, 0), (4, 2048, 2, 3), (16, 1056, 5, 0), (3, 4096, 8, 1)])
def test_experts_sums_behind_a_norm(ops, device, dtype, n, c, top, splits):
    """The kernel that adds up a token's experts and norms the row, against the same sums and the norm's own kernel."""
    experts, ff = 6, 32
    h, x = rand((n, c), dtype, device), rand((n, c), torch.float32, device, 1.0, 1)
    gate, up = (ops.moe_blocked(rand((experts, ff, c), dtype, device, c ** -0.5, s)) for s in (2, 3))
    down = ops.moe_blocked(rand((experts, c, ff), dtype, device, ff ** -0.5, 4))
    ids = torch.tensor([[(3 * i + 2 * j) % (experts + 2) for j in range(top)] for i in range(n)], dtype=torch.int32, device=device)    # (two return their input)
    weights, norm = rand((n, top), torch.float32, device, 0.3, 5), 1 + rand((c,), torch.float32, device, 0.1, 6)
    more = rand((splits, n, c), torch.float32, device, 1.0, 7) if splits else None
    buffers = {}

    def scratch(tag, shape, dt):
        return buffers.setdefault((tag, dt), torch.empty(shape, dtype=dt, device=device))
    want = x.clone()
    ops.moe_experts(h, ids, weights, gate, up, down, 0.0, want, scratch, kind="silu", more=more)
    wanted = ops.rmsnorm(want, norm, 1e-6, torch.empty_like(h))
    out = h.clone()
    ops.moe_experts(out, ids, weights, gate, up, down, 0.0, x, scratch, kind="silu", more=more, norm=(norm, 1e-6, out))
    assert torch.equal(x, want)
    torch.testing.assert_close(out.float(), wanted.float(), atol=0, rtol=2.0 ** -7 if dtype == torch.bfloat16 else 1e-6)     # (a last place: sums in another order)


# rows, columns, K: one and all rows of a tile, ragged columns, K of four, eight and sixteen waves, and ragged
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k,with_bias", [(1, 128, 2048, False), (16, 64, 256, True), (5, 24, 1032, True), (9, 256, 4096, False), (2, 16, 3072, True)])
def test_product_gated_by_tokens(ops, device, dtype, m, n, k, with_bias):
    """The same bits as the three kernels it stands for; token ids past the table, fed ones and fed ones past the feed."""
    x, weight = rand((m, k + 8), torch.float32, device)[:, :k], ops.shuffle_weight(rand((n, k), dtype, device, k ** -0.5, 1))
    table, bias = rand((37, 3 * n), dtype, device, 1.0, 2), rand((n,), torch.float32, device, 0.1, 3) if with_bias else None
    ids = torch.tensor([5, -1, 36, 99, -3, -7, 0, 12, 12, 1, 2, 3, 4, -2, 6, 7][:m], dtype=torch.int32, device=device)
    feed = torch.tensor([11, 36, 50], dtype=torch.int32, device=device)
    rounded, pre, want = torch.empty(m, k, dtype=dtype, device=device), torch.empty(m, n, device=device), torch.empty(m, n, dtype=dtype, device=device)
    ops.round_rows(x.contiguous(), rounded)
    ops.linear(rounded, weight, pre, bias=bias, force=ops.GEMM_NARROW)
    for offset, fed in ((0, feed), (2 * n, None)):
        ops.token_gate(pre, table, ids, offset, want, feed=fed)
        wide = torch.full((m, n + 8), float("nan"), dtype=dtype, device=device)
        got = ops.linear_token_gate(x, weight, table, ids, offset, wide[:, :n], feed=fed, bias=bias)
        assert torch.equal(got, want) and wide[:, n:].isnan().all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,q_heads,kv_heads,dim,behind,k", [(1, 16, 4, 128, 4096, 2048), (16, 3, 1, 16, 16, 72), (5, 2, 2, 48, 144, 3000)])
def test_product_that_fills_the_cache_with_columns_behind(ops, device, dtype, m, q_heads, kv_heads, dim, behind, k):
    """Against the same product, then `kv_store`: the same bits."""
    width, page = (q_heads + 2 * kv_heads) * dim + behind, 16
    x, w, bias = rand((m, k), dtype, device), ops.shuffle_weight(rand((width, k), dtype, device, k ** -0.5, 1)), rand((width,), torch.float32, device, 0.1, 2)
    slots = torch.tensor([(5 * i + 3) % (4 * page) if i != 4 else -1 for i in range(m)], dtype=torch.int32, device=device)
    keys = torch.full((4, kv_heads, page, dim), -9.0, dtype=dtype, device=device)
    values = torch.full((4, kv_heads, dim, page), -9.0, dtype=dtype, device=device)
    want, want_keys, want_values = torch.empty(m, width, dtype=dtype, device=device), keys.clone(), values.clone()
    ops.linear(x, w, want, bias=bias, force=ops.GEMM_NARROW)
    ops.kv_store(want, q_heads * dim, (q_heads + kv_heads) * dim, slots, want_keys, want_values, kv_heads, dim, dim)
    out = torch.full((m, width + 8), -9.0, dtype=dtype, device=device)
    ops.linear_rotate(x, w, out[:, :width], None, None, slots, keys, values, q_heads, kv_heads, dim, page, bias=bias)
    assert torch.equal(keys, want_keys) and torch.equal(values, want_values)
    q, kv = q_heads * dim, (q_heads + 2 * kv_heads) * dim
    assert torch.equal(out[:, :q], want[:, :q]) and torch.equal(out[:, kv:width], want[:, kv:]) and (out[:, width:] == -9).all()


# one and many rows, either side of the line up to which weights are requested with the row; one, two and four groups a thread
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,hidden,splits", [(1, 64, 3), (8, 2048, 4), (16, 4100, 0), (300, 896, 2), (5, 8196, 1), (3, 16384, 0)])
def test_rows_behind_the_next_norm_as_well(ops, device, dtype, n, hidden, splits):
    x, w, w2 = rand((n, hidden), torch.float32, device, 2.0), 1 + rand((hidden,), torch.float32, device, 0.1, 1), 1 + rand((hidden,), torch.float32, device, 0.1, 2)
    parts = rand((max(splits, 1), n, hidden), torch.float32, device, 1.0, 3)
    source = dict(add=parts) if splits else dict(y=parts[0])
    for step in (ops.residual_norm, ops.add_normed):
        alone, both, rows = x.clone(), x.clone(), torch.full((n, hidden), float("nan"), dtype=dtype, device=device)
        outs = [torch.empty(n, hidden, dtype=dtype, device=device) for _ in range(2)]
        step(alone, w, 1e-6, out=outs[0], **source)
        step(both, w, 1e-6, out=outs[1], next_norm=(w2, 1e-5, rows), **source)
        assert torch.equal(alone, both) and torch.equal(*outs)
        want = both.double() / torch.sqrt((both.double() ** 2).mean(-1, keepdim=True) + 1e-5) * w2.double()
        # the sum of squares, its root and two products: a few 2^-24 of the value, and one rounding to the type
        assert ((rows.double() - want).abs() <= (BITS[dtype] + 2.0 ** -20) * want.abs()).all()
        step(x.clone(), w, 1e-6, next_norm=(w2, 1e-5, rows), **source)                     # (without the rows as they are)
        with pytest.raises(Exception):
            step(x[:, 1:].contiguous(), w[1:].contiguous(), 1e-6, y=parts[0][:, 1:], next_norm=(w2[1:].contiguous(), 1e-5, rows[:, 1:].contiguous()))
