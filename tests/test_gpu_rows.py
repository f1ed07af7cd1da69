"""Products of a few rows (``ckv_linear_rows``) and the decoder's steps that use them."""
from dataclasses import replace

import pytest
import torch
import torch.nn.functional as F

from cascading_kv_cache_amd import row_products as rp

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # of 7 and 10 fraction bits


def operands(rows, n, k, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)   # noqa: E731
    return rand(rows, 1, k), rand(n, k) * 0.1, rand(n), rand(rows, 1, n), 1 + 0.1 * rand(k)


def bound(x, w, dtype):
    """One rounding of the result, float32 sums of k products in any order, and float16's smallest step."""
    size = x.double().abs() @ w.double().abs().T
    return HALF_ULP[dtype] * (x.double() @ w.double().T).abs() + x.size(-1) * 2.0 ** -24 * size + 2.0 ** -24


# one group and part of a workgroup's, fewer stretches than parts or stages, remainders of both; the largest rows that fit
@pytest.mark.parametrize("order", rp.ORDERS)
@pytest.mark.parametrize("rows,n,k", [(1, 16, 64), (2, 48, 128), (16, 80, 192), (3, 16, 576), (1, 4096, 832), (5, 96, 1600), (1, 64, 3584),
                                      (2, 32, 18944),
                                      # several groups a compute unit: one workgroup's, two workgroups', many rounds; rings that just fit
                                      (2, 16 * 1793, 64), (1, 16 * 2305, 128), (1, 16 * 8449, 64), (16, 16 * 2048, 3584), (4, 32, 14336)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_against_float64(order, rows, n, k, dtype):
    x, w, bias, res, norm = operands(rows, n, k, dtype)
    assert rp._fits(rows, n, k, order, False)
    exact = x.double() @ w.double().T
    got = rp.linear_rows(x, w, order)
    lim = bound(x, w, dtype)
    assert got.shape == (rows, 1, n) and ((got.double() - exact).abs() <= lim).all()
    assert ((rp.linear_rows(x, w, order, bias).double() - exact - bias.double()).abs() <= lim + HALF_ULP[dtype] * (exact + bias.double()).abs()).all()
    assert torch.equal(rp.linear_rows(x, w, order, residual=res), res + got)
    if rp._fits(rows, n, k, order, True):
        normed = F.rms_norm(x.double(), (k,), norm.double(), 1e-5)
        err = (rp.linear_rows(x, w, order, norm=norm, eps=1e-5).double() - normed @ w.double().T).abs()
        # each element of the normalised row is rounded once on its way
        assert (err <= bound(normed, w, dtype) + HALF_ULP[dtype] * (normed.abs() @ w.double().abs().T)).all()
    if order[0] == 1:
        up = n // 32 * 16
        if up:
            both = rp.linear_rows(x, w[:2 * up].contiguous(), order)
            gate, other = both.chunk(2, -1)
            assert torch.equal(rp.linear_rows(x, w[:2 * up].contiguous(), order, gated=True), F.silu(gate) * other)


def test_rows_a_stride_apart():
    base = torch.randn(3, 7, 256, device="cuda").bfloat16()
    w = torch.randn(32, 256, device="cuda").bfloat16()
    for x in (base[:, -1:], base[:1, 2:5], base[::2, 3:4]):
        assert rp._rows_apart(x)
        assert torch.equal(rp.linear_rows(x, w, (1, 1)), rp.linear_rows(x.contiguous(), w, (1, 1)))
    for x in (base[:, 1:3], base.transpose(1, 2), base[:, :1, 1:], base[:, :, ::2]):
        assert not rp._rows_apart(x)


@pytest.mark.parametrize("extra", [1, 3, 4, 8])
def test_one_row_of_a_wider_buffer(extra):
    """A single row has no distance to a next one, whatever the buffer's rows have; several such rows are torch's to multiply."""
    w = torch.randn(32, 256, device="cuda").bfloat16()
    wide = torch.randn(1, 2, 256 + extra, device="cuda").bfloat16()
    for x in (wide[:, :1, :256], wide[..., :256]):
        one = x.size(1) == 1
        assert rp._rows_apart(x) == (one or extra % 8 == 0)
        with torch.no_grad():
            got = rp.row_linear(x, w, {1: (1, 1), 2: (1, 1)})
        assert torch.equal(got, rp.linear_rows(x.contiguous(), w, (1, 1)) if one or extra % 8 == 0 else F.linear(x, w))


def agrees_with_torch(orders, n, k, dtype=torch.bfloat16):
    w = torch.randn(n, k, device="cuda").to(dtype)
    return all(torch.equal(rp.linear_rows(x, w, order), F.linear(x, w))
               for rows, order in orders.items() for x in torch.randn(20, rows, 1, k, device="cuda").to(dtype))


@pytest.mark.parametrize("spoil", ["zeros", "nan", "large bias", "autocast"])
def test_orders_do_not_hang_on_the_weight_that_asks_first(spoil, monkeypatch):
    n = k = 4096
    w, b = torch.randn(n, k, device="cuda").bfloat16(), torch.zeros(n, device="cuda").bfloat16()
    want = rp.library_orders(w), rp.library_orders(w, b)
    assert want[0] and agrees_with_torch(want[0], n, k)
    monkeypatch.setattr(rp, "_FOUND", {})
    if spoil == "zeros":
        w = torch.zeros_like(w)
    if spoil == "nan":
        w[5, 7] = float("nan")
    if spoil == "large bias":
        b = b + 1e6
    with torch.autocast("cuda", torch.float16, enabled=spoil == "autocast"):
        assert (rp.library_orders(w), rp.library_orders(w, b)) == want


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k", [(152064, 3584), (152128, 3584), (65568, 4096), (66016, 4096)])
def test_an_order_that_differs_in_a_few_tiles_is_told_from_torchs(n, k, dtype):
    """Products whose tiles do not come out even on a library's workgroups have an output or two a row in another order than the others.
    Whatever is found holds for rows that were not tried."""
    orders = rp.library_orders(torch.empty(n, k, device="cuda", dtype=dtype))
    w = torch.randn(n, k, device="cuda", dtype=dtype)
    for rows, order in orders.items():
        for x in torch.randn(60, rows, 1, k, device="cuda").to(dtype):
            assert torch.equal(rp.linear_rows(x, w, order), F.linear(x, w)), (rows, order)


def test_no_room_to_try_means_no_order(monkeypatch):
    w = torch.empty(4096, 4096, device="cuda", dtype=torch.bfloat16)
    monkeypatch.setattr(rp, "_FOUND", {})
    with monkeypatch.context() as m:
        def full(*args, **kw):
            raise torch.OutOfMemoryError("as on a device that a model fills")
        m.setattr(torch, "randn", full)
        assert rp.library_orders(w) == {}
    assert rp.library_orders(w)


def test_orders_are_asked_again_when_torch_is_told_to_take_another_product():
    n, k = 6144, 4096
    w = torch.randn(n, k, device="cuda").bfloat16()
    assert agrees_with_torch(rp.library_orders(w), n, k)
    blas, flags, seen = torch.backends.cuda.preferred_blas_library, torch.backends.cuda.matmul, {rp.product_settings()}
    was = blas(), flags.allow_bf16_reduced_precision_reduction
    try:
        for library, reduced in (("cublas", True), ("cublas", False), ("cublaslt", False)):
            blas(library)
            flags.allow_bf16_reduced_precision_reduction = reduced
            seen.add(rp.product_settings())
            assert agrees_with_torch(rp.library_orders(w), n, k), (library, reduced)
    finally:
        blas(was[0])
        flags.allow_bf16_reduced_precision_reduction = was[1]
    assert len(seen) == 4 and rp.product_settings() in seen


@pytest.mark.parametrize("n,k,dtype", [(6144, 4096, torch.bfloat16), (4608, 3584, torch.bfloat16), (6144, 4096, torch.float16)])
def test_a_norm_in_front_is_tried_too(n, k, dtype, monkeypatch):
    """Torch's norm with its squares added up in another order: no row count is left."""
    class Norm:
        eps = 1e-5

    w = torch.randn(n, k, device="cuda").to(dtype)
    assert rp.library_orders(w, norm=Norm) == rp.library_orders(w) != {}

    def other(x, shape, weight, eps):
        factor = torch.rsqrt(x.float().pow(2).flip(-1).cumsum(-1)[..., -1:] / x.size(-1) + eps)
        return (weight.float() * (factor * x.float())).to(x.dtype)

    monkeypatch.setattr(rp, "_FOUND", {})
    monkeypatch.setattr(F, "rms_norm", other)
    assert rp.library_orders(w, norm=Norm) == {} != rp.library_orders(w)


def test_other_settings_than_a_layer_was_fused_under_keep_torchs_products():
    from cascading_kv_cache_amd.decoder import PRESETS, CascadeDecoder

    model = CascadeDecoder(replace(PRESETS["llama3.1-8b"], num_layers=1, vocab_size=512), init_on_device=True).fuse_projections()
    layer, cache, x = model.layers[0], model.new_cache(256, 2, num_sink_tokens=4), torch.randn(1, 1, 4096, device="cuda").bfloat16()
    flags = torch.backends.cuda.matmul
    was = flags.allow_bf16_reduced_precision_reduction
    with torch.no_grad():
        assert layer._as_rows(x, cache)
        try:
            flags.allow_bf16_reduced_precision_reduction = not was
            assert not layer._as_rows(x, cache)
        finally:
            flags.allow_bf16_reduced_precision_reduction = was
        assert layer._as_rows(x, cache)


@pytest.mark.parametrize("order", [(1, 1), (4, 1)])
@pytest.mark.parametrize("rows,n,k,runs", [(1, 16 * 16 * 3, 256, 2), (2, 16 * 16 * 5 - 48, 1024, 3), (4, 16 * 77, 1024, 4), (1, 16 * 16 * 7, 4096, 6),
                                           (3, 16 * 700, 768, 37), (1, 16 * 16 * 4, 256, 2), (2, 16 * 40, 256, 1)])
def test_sums_cut_where_a_run_of_tiles_ends(rows, n, k, runs, order):
    """Against the two halves of every cut sum: rows of x that are zero past the cut, or up to it."""
    x, w, bias, res, norm = operands(rows, n, k, torch.bfloat16)
    height, span = (256, k // 64) if order[0] == 1 else (32, k // 256)
    tiles = -(-n // height)
    shared = tiles % runs + runs if tiles % runs else 0
    length = -(-shared * span // runs)
    got = rp.linear_rows(x, w, (*order, runs), residual=res)
    whole = rp.linear_rows(x, w, order, residual=res)
    exact = x.double() @ w.double().T + res.double()
    assert ((got.double() - exact).abs() <= 2 * bound(x, w, torch.bfloat16) + HALF_ULP[torch.bfloat16] * (exact.abs() + res.double().abs())).all()
    cut_tiles = set()
    for tile in range(tiles):
        at = slice(tile * height, min(n, (tile + 1) * height))
        first = (tile - (tiles - shared)) * span
        ends = [e for e in range(length, shared * span, length) if first < e < first + span] if shared else []
        if not ends:
            assert torch.equal(got[..., at], whole[..., at])
            continue
        cut_tiles.add(tile)
        part = (ends[0] - first) * (k // span)
        for keep in (slice(0, part), slice(part, k)):
            y = torch.zeros_like(x)
            y[..., keep] = x[..., keep]
            assert torch.equal(rp.linear_rows(y, w, (*order, runs))[..., at], rp.linear_rows(y, w, order)[..., at])
    assert len(cut_tiles) <= runs and (cut_tiles or not shared or runs == 1)


def test_sums_that_cannot_be_cut_are_refused():
    from cascading_kv_cache_amd import _abi

    x, w, *_ = operands(1, 16 * 32, 256, torch.bfloat16)
    for order in ((1, 1, 3), (4, 1, 17), (2, 2, 2), (4, 2, 2), (1, 2, 2), (1, 1, 1025)):
        with pytest.raises(_abi.CkvError):
            rp.linear_rows(x, w, order)
    with pytest.raises(_abi.CkvError):
        rp.linear_rows(x, w, (1, 1, 2), gated=True)
    with pytest.raises(_abi.CkvError):
        rp.linear_rows(x[..., :192].contiguous(), w[:, :192].contiguous(), (4, 1, 2))


@pytest.mark.parametrize("preset", ["llama3.1-8b", "qwen2-7b"])
def test_every_product_of_a_step_has_torchs_bits(preset, monkeypatch):
    """Logits, caches and greedy tokens of a decoder's steps of one to five streams, and of three tokens at a time, by row products and by torch's operations."""
    from cascading_kv_cache_amd.decoder import PRESETS, CascadeDecoder, generate

    cfg = replace(PRESETS[preset], num_layers=2)
    model = CascadeDecoder(cfg, init_on_device=True).fuse_projections()
    taken = []
    monkeypatch.setattr(rp, "linear_rows", lambda *args, run=rp.linear_rows, **kw: taken.append(args[1].shape) or run(*args, **kw))
    got = []
    for by_rows in (True, False):
        if not by_rows:
            model._head_orders = None
            for layer in model.layers:
                layer._orders = None
        got.append([])
        gen = torch.Generator().manual_seed(4)
        with torch.no_grad():
            for batch in range(1, 6):
                ids = torch.randint(0, cfg.vocab_size, (batch, 40), generator=gen).cuda()
                cache = model.new_cache(256, 2, batch=batch, num_sink_tokens=4)
                logits = [model(cut, cache) for cut in [ids[:, :32], ids[:, 32:35]] + [ids[:, i:i + 1] for i in range(35, 40)]]
                cache_two = model.new_cache(256, 2, batch=batch, num_sink_tokens=4)
                got[-1].append([*logits, *cache.key_cache, *cache.value_cache, generate(model, ids, cache_two, 32, 12)])
        if by_rows:   # the layers' four products and the head
            assert len(set(taken)) == 5, taken
            taken.clear()
    assert not taken
    for batch, (a, b) in enumerate(zip(*got), 1):
        for x, y in zip(a, b):
            assert torch.equal(x, y), batch


@pytest.mark.parametrize("preset", ["llama3.1-8b", "qwen2-7b", "tiny"])
def test_steps_of_a_fused_decoder_have_the_bits_of_torchs_products(preset):
    """One layer's steps by row products where an order is torch's, and by torch's operations: the same bits in the cache, and logits that
    differ by the order of the head's sums alone.  Hooks on a module see their calls."""
    from cascading_kv_cache_amd.decoder import PRESETS, CascadeDecoder

    cfg = replace(PRESETS[preset], num_layers=1, vocab_size=512)
    model = CascadeDecoder(cfg, init_on_device=True).fuse_projections()
    plain = CascadeDecoder(cfg, init_on_device=True).fuse_projections()
    for layer in plain.layers:
        layer._orders = None
    if preset == "tiny":   # too few outputs to tell one order from another by
        assert not any(model.layers[0]._orders.values())
    else:
        assert all(model.layers[0]._orders[name] for name in ("qkv", "o", "gate_up", "down")), model.layers[0]._orders
    for batch in (1, 2, 5):
        ids = torch.randint(0, 512, (batch, 40), device="cuda")
        a, b = (m.new_cache(256, 2, batch=batch, num_sink_tokens=4) for m in (model, plain))
        with torch.no_grad():
            for cut in [ids[:, :32]] + [ids[:, i:i + 1] for i in range(32, 40)]:
                la, lb = model(cut, a), plain(cut, b)
                assert (la - lb).abs().max() <= 2.0 ** -7 * lb.abs().max()
        assert torch.equal(a.key_cache[0], b.key_cache[0]) and torch.equal(a.value_cache[0], b.value_cache[0])
    seen = []
    cache = model.new_cache(256, 2, num_sink_tokens=4)
    one = ids[:1, :1]
    with torch.no_grad():
        for module in (model.layers[0].self_attn.o_proj, model.layers[0].mlp, model.layers[0].input_layernorm, model.norm, model.lm_head):
            handle = module.register_forward_hook(lambda m, i, o: seen.append(m))
            model(one, cache)
            handle.remove()
            assert seen and seen[-1] is module
    model(one, cache).sum().backward() if preset == "tiny" else None   # gradients take torch's operations


def test_gradients_take_torchs_operations():
    """A step of a decoder whose products have orders, with gradients wanted: they are there, and the ones that torch's operations give."""
    from cascading_kv_cache_amd.decoder import PRESETS, CascadeDecoder

    model = CascadeDecoder(replace(PRESETS["llama3.1-8b"], num_layers=1, vocab_size=512), init_on_device=True).fuse_projections()
    layer, grads = model.layers[0], []
    assert all(layer._orders[name] for name in ("qkv", "o", "gate_up", "down"))
    for orders in (layer._orders, None):
        layer._orders = orders
        cache = model.new_cache(256, 2, num_sink_tokens=4)
        model.zero_grad()
        model(torch.tensor([[3]], device="cuda"), cache).float().square().sum().backward()
        grads.append([m.weight.grad for m in (layer.self_attn.o_proj, layer.mlp.down_proj, layer.post_attention_layernorm, model.norm)])
    for a, b in zip(*grads):
        assert a.abs().max() > 0 and torch.equal(a, b)
