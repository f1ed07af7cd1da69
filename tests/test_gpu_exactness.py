"""What the fp32-math paths owe float64 arithmetic on the same inputs.

Head size 64 in the 16-bit formats holds logits, probabilities, dS and every sum in 32 bits: a result is the exact
one rounded once to the tensor dtype, up to the noise of its float32 sums.  There and in float32 a value row of a key
with probability zero is never touched, whatever it holds, and the number of workgroups that share a row's keys changes
nothing but the order of sums.

Cached keys are rotated; with ``inv_freq`` zero the rotation is the identity, so that the staged operands are known to
the bit: queries and keys times sqrt(softmax scale), rounded to the tensor dtype (cascade_attention.py:284-291).
"""
import math

import pytest
import torch

from parity_helpers import backward_in_one_launch, dq_wavefronts

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
HALF_ULP = {BF16: 2.0 ** -8, F16: 2.0 ** -11, F32: 2.0 ** -24}   # relative, at the bottom of a binade


def assert_rounded_once(got, exact, spread, n, what):
    """``got`` is ``exact`` rounded to its dtype behind float32 sums of ``n`` terms, ``spread`` being the root of the sum
    of their squares.  Half a unit in the last place; a float32 chain over n random terms is off by about
    2^-24 sqrt(n) spread and a term itself (a logit of a few units, its exponential) by 2^-22 or so: eight times their
    sum; what a whole row shares (its normaliser, rounded at a magnitude of ten) by 2^-20 of the result; half the
    smallest float16 number."""
    bound = (HALF_ULP[got.dtype] + 2.0 ** -20) * exact.abs() + 2.0 ** -21 * math.sqrt(n) * spread
    bound = bound + (2.0 ** -25 if got.dtype == F16 else 1e-30)
    excess = ((got.double() - exact).abs() / bound).max().item()
    assert excess <= 1.0, f"{what}: {excess:.2f} times the bound"


def visible(n_ctx, n_kv, mask):
    """(n_ctx, n_kv): which key a row sees."""
    causal = torch.ones(n_ctx, n_ctx, dtype=torch.bool, device=mask.device).tril()
    return torch.cat((~mask[None, :].expand(n_ctx, -1), causal), dim=-1)


def exact_attention(q, k, v, see, scale):
    """out, P, row normalisers and the spread of out, in float64 (every head its own kv head)."""
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * scale
    s = s.masked_fill(~see, float("-inf"))
    p = torch.softmax(s, dim=-1)
    vd = v.double()
    return torch.matmul(p, vd), p, torch.logsumexp(s, dim=-1), torch.matmul(p * p, vd * vd).sqrt()


def exact_weights(q, k, v, out, lse, mask, do, scale):
    """P and dS of the backward pass in float64 from what its kernels are given, the forward's output and row normalisers
    among it, and the size that dS's float32 sums of 64 or 128 products are rounded at."""
    see = visible(q.size(2), k.size(2), mask)
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * scale
    p = torch.exp(s - lse.double()[..., None]).masked_fill(~see, 0.0)
    g, vt = do.double(), v.double().transpose(2, 3).contiguous()
    dp, delta = torch.matmul(g, vt), (out.double() * g).sum(-1, keepdim=True)
    size = torch.matmul(g.abs(), vt.abs()) + (out.double() * g).abs().sum(-1, keepdim=True)
    return p, p * (dp - delta) * scale, p * size * abs(scale)


DENSE = [(1, 2, 128, 128), (1, 3, 33, 1 + 33), (2, 4, 200, 1000 + 200), (1, 2, 500, 2048 + 64 + 500), (1, 1, 700, 5000 + 700)]


def dense_case(Z, H, n_ctx, n_kv, D, dtype, std=0.7):
    g = torch.Generator(device="cuda").manual_seed(100 + n_kv)
    q, k, v = ((torch.randn(Z, n, H, D, device="cuda", generator=g) * std).to(dtype).transpose(1, 2) for n in (n_ctx, n_kv, n_kv))
    mask = torch.rand(n_kv - n_ctx, device="cuda", generator=g) > 0.5
    return q, k, v, mask, torch.randn(Z, H, n_ctx, D, device="cuda", generator=g).to(dtype)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("Z,H,n_ctx,n_kv", DENSE)
def test_dense_forward_of_head_size_64_is_rounded_once(Z, H, n_ctx, n_kv, dtype):
    from cascading_kv_cache_amd import flash_attention as fa

    q, k, v, mask, _ = dense_case(Z, H, n_ctx, n_kv, 64, dtype)
    out, scores, lse, _ = fa._forward(q, k, v, True, 0.5, mask, 0.9, True)
    ref, p, ref_lse, spread = exact_attention(q, k, v, visible(n_ctx, n_kv, mask), 0.5)
    assert (lse.double() - ref_lse).abs().max().item() <= 4e-6      # float32 logits and sums, normalisers of up to ten
    assert_rounded_once(out, ref, spread, n_kv, "out")
    w = (0.1 * 0.9 ** torch.arange(n_ctx - 1, -1, -1, device="cuda", dtype=torch.float64))[None, None, :, None]
    assert_rounded_once(scores, (w * p).sum(2), (w * p).square().sum(2).sqrt(), n_ctx, "scores")


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("grad_scale", [1.0, 2.0 ** 12])   # P dP far past float16's largest number is no overflow of dS
@pytest.mark.parametrize("Z,H,n_ctx,n_kv", DENSE)
def test_dense_backward_of_head_size_64_is_rounded_once(Z, H, n_ctx, n_kv, grad_scale, dtype):
    """Against the formula in float64 on what the kernels are given: the forward's output as it was rounded."""
    from cascading_kv_cache_amd import flash_attention as fa

    scale = 0.5
    q, k, v, mask, do = dense_case(Z, H, n_ctx, n_kv, 64, dtype)
    do = (do.float() * grad_scale).to(dtype)
    out, _, lse, m = fa._forward(q, k, v, True, scale, mask, 0.9, True)
    dq, dk, dv = fa._backward(q, k, v, out, lse, m, do, scale)
    _, p, _, _ = exact_attention(q, k, v, visible(n_ctx, n_kv, mask), scale)
    qd, kd, vd, g = q.double(), k.double(), v.double(), do.double()
    dp, delta = torch.matmul(g, vd.transpose(2, 3).contiguous()), (out.double() * g).sum(-1, keepdim=True)
    ds, ds_size = p * (dp - delta) * scale, p * (dp.abs() + delta.abs() + grad_scale) * scale
    pt, dst, ds2t = (t.transpose(2, 3).contiguous() for t in (p, ds, ds_size.square()))
    if grad_scale == 1.0 or dtype == BF16:   # float16 gradients of that size are infinite themselves where they pass 65504
        assert_rounded_once(dv, torch.matmul(pt, g), torch.matmul(pt.square(), g.square()).sqrt(), n_ctx, "dv")
        assert_rounded_once(dk, torch.matmul(dst, qd), torch.matmul(ds2t, qd.square()).sqrt(), n_ctx, "dk")
    want, spread = torch.matmul(ds, kd), torch.matmul(ds_size.square(), kd.square()).sqrt()
    fits = want.abs() < 6e4 if dtype == F16 else torch.ones_like(want, dtype=torch.bool)
    assert_rounded_once(dq[fits], want[fits], spread[fits], n_kv, "dq")


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("octaves", [-24, 24])
def test_dense_backward_of_head_size_64_over_many_octaves(octaves, dtype):
    """dS whose size falls or rises by 2^24 from the first block to the last, along the keys and along the rows."""
    from cascading_kv_cache_amd import flash_attention as fa

    n_ctx, n_kv, scale = 300, 900, 0.5
    q, k, v, mask, do = dense_case(1, 2, n_ctx, n_kv, 64, dtype)
    ramp = lambda n: 2.0 ** (octaves * (torch.arange(n, device="cuda") / (n - 1) - 0.5) / 2)
    v = (v.float() * ramp(n_kv)[:, None]).to(dtype)
    do = (do.float() * ramp(n_ctx)[:, None]).to(dtype)
    out, _, lse, m = fa._forward(q, k, v, True, scale, mask, 0.9, True)
    dq, dk, dv = fa._backward(q, k, v, out, lse, m, do, scale)
    _, p, _, _ = exact_attention(q, k, v, visible(n_ctx, n_kv, mask), scale)
    dp, delta = torch.matmul(do.double(), v.double().transpose(2, 3).contiguous()), (out.double() * do.double()).sum(-1, keepdim=True)
    # delta and dP are float32 sums of 64 products each, rounded at the size of their largest terms
    size = torch.matmul(do.double().abs(), v.double().abs().transpose(2, 3).contiguous()) + (out.double() * do.double()).abs().sum(-1, keepdim=True)
    ds, ds2 = p * (dp - delta) * scale, (p * size * scale).square()
    pt, dst, ds2t = (t.transpose(2, 3).contiguous() for t in (p, ds, ds2))
    assert_rounded_once(dv, torch.matmul(pt, do.double()), torch.matmul(pt.square(), do.double().square()).sqrt(), n_ctx, "dv")
    assert_rounded_once(dk, torch.matmul(dst, q.double()), torch.matmul(ds2t, q.double().square()).sqrt(), n_ctx, "dk")
    assert_rounded_once(dq, torch.matmul(ds, k.double()), torch.matmul(ds2, k.double().square()).sqrt(), n_kv, "dq")


@pytest.mark.parametrize("dtype", [BF16, F16])
def test_small_weights_beside_large_ones_of_head_size_64(dtype):
    """dS is float32 whatever stands beside it: it is 28 octaves smaller in every other row (for dk) and 36 for every other
    key (for dq, as P is), and the large ones meet zeros in one dim of the other operand.  There the sum is the small ones
    alone, to the last bit that the result's format shows."""
    from cascading_kv_cache_amd import flash_attention as fa

    n_ctx, n_kv, scale = 64, 160, 0.5
    q, k, v, mask, do = (t.clone() for t in dense_case(1, 2, n_ctx, n_kv, 64, dtype, std=0.3))
    v = (v.float() * 3).to(dtype)
    do[:, :, ::2] *= 2.0 ** 10
    do[:, :, 1::2] *= 2.0 ** -18
    q[..., 5:8], k[..., 5:8] = 0.0, 0.0
    q[:, :, 1::2, 5] = 2.0 ** 13           # dk, dim 5: the rows of the small gradients alone
    k[:, :, 1::2, 6] = 2.0 ** 14           # dq, dim 6: the keys of the small probabilities alone
    q[..., 7], k[:, :, 1::2, 7] = 8.0, -6.25   # their logits 25 below the others': 2^-36
    out, _, lse, m = fa._forward(q, k, v, True, scale, mask, 0.9, True)
    dq, dk, dv = fa._backward(q, k, v, out, lse, m, do, scale)
    p, ds, size = exact_weights(q, k, v, out, lse, mask, do, scale)
    pt, dst, sizet = (t.transpose(2, 3).contiguous() for t in (p, ds, size))
    large, small = ds[0, :, ::2].abs().amax(), ds[0, :, 1::2].abs().amax()
    assert large > 2.0 ** 24 * small and (dk[0, :, 0, 5] != 0).any() and (dq[0, :, ::2, 6] != 0).any()
    assert_rounded_once(dv, torch.matmul(pt, do.double()), torch.matmul(pt.square(), do.double().square()).sqrt(), n_ctx, "dv")
    assert_rounded_once(dk, torch.matmul(dst, q.double()), torch.matmul(sizet.square(), q.double().square()).sqrt(), n_ctx, "dk")
    assert_rounded_once(dq, torch.matmul(ds, k.double()), torch.matmul(size.square(), k.double().square()).sqrt(), n_kv, "dq")


@pytest.mark.parametrize("dtype", [BF16, F16])
def test_dense_backward_of_head_size_64_with_an_infinite_gradient(dtype):
    """An infinite element of dout is infinite in dv of every key its row sees and of no head but its own, and a key's other
    dims are what they were: its block takes float32 products (zero terms times infinity would be NaN)."""
    from cascading_kv_cache_amd import flash_attention as fa

    n_ctx, n_kv, row, dim = 150, 450, 70, 7
    q, k, v, mask, do = dense_case(1, 2, n_ctx, n_kv, 64, dtype)
    out, _, lse, m = fa._forward(q, k, v, True, 0.5, mask, 0.9, True)
    clean = fa._backward(q, k, v, out, lse, m, do, 0.5)
    do[0, 0, row, dim] = float("inf")
    dq, dk, dv = fa._backward(q, k, v, out, lse, m, do, 0.5)
    for got, want in zip((dq, dk, dv), clean):
        assert torch.equal(got[0, 1], want[0, 1])
    seen = torch.cat((~mask, torch.arange(n_ctx, device="cuda") <= row))
    assert torch.equal(dv[0, 0, seen, dim], torch.full_like(dv[0, 0, seen, dim], float("inf")))
    others = [d for d in range(64) if d != dim]
    err = (dv[0, 0, seen][:, others].double() - clean[2][0, 0, seen][:, others].double()).abs()
    assert (err <= 2 * HALF_ULP[dtype] * clean[2][0, 0, seen][:, others].double().abs() + 2.0 ** -24).all()   # one rounding each
    assert dv[0, 0, :n_kv - n_ctx][mask].abs().max().item() == 0.0
    assert dk[0, 0, seen].isfinite().sum().item() == 0


def rounding_variance(x, dtype):
    """of a number rounded to ``dtype``: uniform over a unit in the last place"""
    bits, least = {BF16: (7, -126), F16: (10, -14)}[dtype]
    ulp = torch.ldexp(torch.ones_like(x), (torch.frexp(x)[1] - 1).clamp(min=least) - bits)
    return ulp.square() / 12


def assert_rounded(got, exact, variance, what):
    """``got`` is ``exact`` but for roundings of which ``variance`` is the sum, its own among them.  One bit less in P or dS shows
    as a root mean square of 1.7 times that, a fault in one place as many deviations there."""
    off = (got.double() - exact).square() / (variance + rounding_variance(exact, got.dtype))
    rms, worst = off.mean().sqrt().item(), off.max().sqrt().item()
    assert rms <= 1.1 and worst <= 8.0, f"{what}: root mean square {rms:.3f}, largest {worst:.2f} of the roundings' deviation"


def check_backward(q, k, v, out, lse, mask, do, scale, dq, dk, dv):
    """Head size 64: float32 but for the result.  Head size 128: P and dS enter the products rounded to the tensor dtype, dS
    with or without the softmax scale, which no rounding of a mantissa tells apart."""
    p, ds, size = exact_weights(q, k, v, out, lse, mask, do, scale)
    n_ctx, n_kv = q.size(2), k.size(2)
    turned = lambda t: t.transpose(2, 3).contiguous()
    for what, got, w, weight_size, rows in (("dv", dv, turned(p), turned(p), do), ("dk", dk, turned(ds), turned(size), q), ("dq", dq, ds, size, k)):
        x = rows.double()
        exact, spread2 = torch.matmul(w, x), torch.matmul(weight_size.square(), x.square())
        if q.size(-1) == 64:
            assert_rounded_once(got, exact, spread2.sqrt(), n_kv if what == "dq" else n_ctx, what)
        else:
            assert_rounded(got, exact, torch.matmul(rounding_variance(w, got.dtype) * (w != 0), x.square()) + 2.0 ** -44 * spread2, what)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("scale", [0.3, -0.125])
@pytest.mark.parametrize("Z,H,n_ctx,n_kv", DENSE)
def test_dense_backward_of_head_size_128_rounds_weights_once(Z, H, n_ctx, n_kv, scale, dtype):
    from cascading_kv_cache_amd import flash_attention as fa

    q, k, v, mask, do = dense_case(Z, H, n_ctx, n_kv, 128, dtype)
    out, _, lse, m = fa._forward(q, k, v, True, scale, mask, 0.9, True)
    check_backward(q, k, v, out, lse, mask, do, scale, *fa._backward(q, k, v, out, lse, m, do, scale))


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("room", ["delta", "delta and order"])
@pytest.mark.parametrize("Z,H,n_ctx,n_kv,masked", [
    (1, 2, 128, 128, None), (1, 3, 33, 1 + 33, None), (1, 1, 31, 64 + 31, slice(0, 64)),   # no cached key, one, none visible
    (2, 4, 200, 1000 + 200, None), (1, 8, 129, 1500 + 129, slice(32, 700)),                 # whole blocks of masked keys
    (1, 1, 300, 95 + 300, slice(0, 33))])
def test_dense_backward_with_less_room_than_it_could_use(Z, H, n_ctx, n_kv, masked, room, D, dtype):
    """A workspace without room for the order of the keys (they are taken as they lie and masked one by one), or without room
    for dq's shares, as ``ckv_dense_bwd_key_order_bytes`` and ``ckv_dense_bwd_split_bytes`` allow."""
    from cascading_kv_cache_amd import _abi
    from cascading_kv_cache_amd import flash_attention as fa

    q, k, v, mask, do = dense_case(Z, H, n_ctx, n_kv, D, dtype)
    if masked is not None:
        mask[masked] = True
    out, _, lse, m = fa._forward(q, k, v, True, 0.3, mask, 0.9, True)
    size = _abi.lib().ckv_dense_bwd_workspace_bytes(Z, H, n_ctx)
    if room == "delta and order":
        size += _abi.lib().ckv_dense_bwd_key_order_bytes(n_kv)
    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(fa, "workspace", lambda device, need, stream: torch.empty(size, dtype=torch.uint8, device=device))
        grads = fa._backward(q, k, v, out, lse, m, do, 0.3)
    check_backward(q, k, v, out, lse, mask, do, 0.3, *grads)
    hidden = torch.cat((mask, torch.zeros(n_ctx, dtype=torch.bool, device="cuda")))
    assert (grads[1][:, :, hidden] == 0).all() and (grads[2][:, :, hidden] == 0).all()


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [0.3, -0.25])
@pytest.mark.parametrize("room", ["delta", "delta and order", "all"])
@pytest.mark.parametrize("Z,H,n_ctx,n_kv,masked", [
    (2, 80, 129, 500 + 129, slice(32, 320)),   # the second workgroup's one row; whole stages and a half of hidden keys
    (1, 90, 400, 75 + 400, slice(0, 75)),      # no cached key visible; two workgroups a head, the second short of rows
    (1, 40, 1000, 250 + 1000, None),           # four, and a diagonal that crosses twelve stages in front of the last's
    (2, 80, 129, 1000 + 129, slice(32, 320)),  # as the first and the second, with keys enough that dk and dv are a launch of their own
    (1, 90, 400, 1500 + 400, slice(0, 1500))])
def test_dense_backward_with_dq_by_eight_wavefronts(Z, H, n_ctx, n_kv, masked, room, scale, D, dtype):
    """dq's wide workgroups with the keys sorted and as they lie (masked one by one, a hidden block of 32 left out), with
    either sign of the scale."""
    from cascading_kv_cache_amd import _abi
    from cascading_kv_cache_amd import flash_attention as fa

    assert dq_wavefronts(Z, H, n_ctx, n_kv, D, dtype, shared=room == "all") == 8
    assert (n_kv in (1000 + 129, 1500 + 400)) == (not backward_in_one_launch(Z, H, n_kv))
    q, k, v, mask, do = dense_case(Z, H, n_ctx, n_kv, D, dtype)
    if masked is not None:
        mask[masked] = True
    out, _, lse, m = fa._forward(q, k, v, True, scale, mask, 0.9, True)
    size = _abi.lib().ckv_dense_bwd_workspace_bytes(Z, H, n_ctx)
    if room == "delta and order":
        size += _abi.lib().ckv_dense_bwd_key_order_bytes(n_kv)
    with pytest.MonkeyPatch.context() as patch:
        if room != "all":
            patch.setattr(fa, "workspace", lambda device, need, stream: torch.empty(size, dtype=torch.uint8, device=device))
        grads = fa._backward(q, k, v, out, lse, m, do, scale)
    check_backward(q, k, v, out, lse, mask, do, scale, *grads)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("row,cached", [(5, 700), (299, 700), (5, 2000), (299, 2000)])   # dk and dv beside dq, and in a launch of their own
def test_infinite_gradient_in_dq_by_eight_wavefronts(row, cached, dtype):
    """The wavefront that holds the row takes float32 products, in both blocks of every stage: its other rows are what they
    were to a rounding, everyone else's to the bit."""
    from cascading_kv_cache_amd import flash_attention as fa

    Z, H, n_ctx, n_kv = 1, 72, 400, cached + 400
    assert dq_wavefronts(Z, H, n_ctx, n_kv, 64, dtype) == 8 and backward_in_one_launch(Z, H, n_kv) == (cached == 700)
    q, k, v, mask, do = dense_case(Z, H, n_ctx, n_kv, 64, dtype)
    out, _, lse, m = fa._forward(q, k, v, True, 0.5, mask, 0.9, True)
    clean = fa._backward(q, k, v, out, lse, m, do, 0.5)[0]
    do[0, 3, row, 7] = float("inf")
    dq = fa._backward(q, k, v, out, lse, m, do, 0.5)[0]
    assert not dq[0, 3, row].isfinite().any()
    mates = [r for r in range(row // 32 * 32, row // 32 * 32 + 32) if r != row]
    same = torch.ones_like(dq, dtype=torch.bool)
    same[0, 3, row // 32 * 32:row // 32 * 32 + 32] = False
    assert torch.equal(dq[same], clean[same])
    p, ds, size = exact_weights(q, k, v, out, lse, mask, torch.where(do.isinf(), 0.0, do), 0.5)   # the mates' rows are finite
    exact, spread2 = torch.matmul(ds[0, 3], k[0, 3].double()), torch.matmul(size[0, 3].square(), k[0, 3].double().square())
    assert_rounded_once(dq[0, 3, mates], exact[mates], spread2[mates].sqrt(), n_kv, "dq")


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("scale", [-0.5, 0.0, 1e-3, 3.0])
def test_any_softmax_scale_of_head_size_64(scale, dtype):
    """The scale joins in float32 behind the logits: negative, zero (every visible key weighs the same), small and large."""
    from cascading_kv_cache_amd import flash_attention as fa

    q, k, v, mask, do = dense_case(1, 3, 150, 700 + 150, 64, dtype)
    out, scores, lse, m = fa._forward(q, k, v, True, scale, mask, 0.9, True)
    ref, p, ref_lse, spread = exact_attention(q, k, v, visible(150, 850, mask), scale)
    assert (lse.double() - ref_lse).abs().max().item() <= 4e-6 * max(1.0, abs(scale) * 8)    # logits of up to thirty
    assert_rounded_once(out, ref, spread * max(1.0, abs(scale) * 4), 850, "out")
    dq, dk, dv = fa._backward(q, k, v, out, lse, m, do, scale)
    dp, delta = torch.matmul(do.double(), v.double().transpose(2, 3).contiguous()), (out.double() * do.double()).sum(-1, keepdim=True)
    ds = p * (dp - delta) * scale
    size = (p * (dp.abs() + delta.abs() + 1.0) * scale).square() * max(1.0, abs(scale) * 4) ** 2
    assert_rounded_once(dq, torch.matmul(ds, k.double()), torch.matmul(size, k.double().square()).sqrt(), 850, "dq")


def one_layer(B, KVH, D, NS, W, C, dtype):
    from cascading_kv_cache_amd.cascading_cache import CascadingKVCache

    return CascadingKVCache(window_length=W, num_sink_tokens=NS, max_batch_size=B, heads=KVH, dim=D, max_seq_len=W * C,
                            device="cuda:0", dtype=dtype, layers=1, verbose=False)


def cascade_case(B, H, KVH, D, NS, W, C, filled, Q, dtype, std=0.7):
    """A cache that holds ``filled`` random tokens, and a chunk; no rotation (inv_freq zero)."""
    g = torch.Generator(device="cuda").manual_seed(7)
    cache = one_layer(B, KVH, D, NS, W, C, dtype)
    rows = lambda h, n: (torch.randn(B, n, h, D, device="cuda", generator=g) * std).to(dtype).transpose(1, 2)
    if filled:
        cache.update(rows(KVH, filled), rows(KVH, filled), 0, torch.rand(B, KVH, filled, device="cuda", generator=g).to(dtype))
    return cache, rows(H, Q), rows(KVH, Q), rows(KVH, Q), torch.zeros(D // 2, device="cuda")


def staged(cache, q, k, v):
    """The operands as the kernels stage them, expanded to the query heads, and the mask of the cached keys."""
    G, rs = q.size(1) // k.size(1), math.sqrt(1 / math.sqrt(q.size(-1)))
    scaled = lambda t: (t.float() * rs).to(t.dtype)
    keys = torch.cat((cache.sink_keys[0], cache.key_cache[0], k), dim=2)
    vals = torch.cat((cache.sink_values[0], cache.value_cache[0], v), dim=2)
    mask = torch.cat((cache.sink_mask[0].reshape(-1, cache.sink_keys[0].size(2))[0], cache.mask[0].reshape(-1, cache.key_cache[0].size(2))[0]))
    return scaled(q), scaled(keys).repeat_interleave(G, 1), vals.repeat_interleave(G, 1), mask.bool()


CASCADE = [
    # B, H, KVH, D, NS, W, C, filled, Q, dtype
    (1, 8, 2, 64, 4, 64, 4, 1000, 96, BF16), (2, 14, 2, 64, 4, 128, 2, 200, 77, F16), (1, 3, 3, 64, 64, 256, 8, 4000, 300, BF16),
    # float32 with fewer row tiles (32 rows each) than compute units and at least 16 key blocks (32 keys each) a share: the
    # keys of a tile are shared out over 4, 2 (the cache half empty) and 8 workgroups
    (1, 8, 2, 128, 4, 512, 4, 4000, 40, F32), (1, 7, 1, 64, 4, 1024, 1, 500, 33, F32), (1, 4, 1, 128, 4, 1024, 4, 3000, 100, F32),
    (1, 32, 8, 128, 4, 128, 4, 1000, 256, F32),   # one share
]


@pytest.mark.parametrize("B,H,KVH,D,NS,W,C,filled,Q,dtype", CASCADE)
def test_cascade_forward_is_rounded_once(B, H, KVH, D, NS, W, C, filled, Q, dtype):
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(B, H, KVH, D, NS, W, C, filled, Q, dtype)
    qs, ks, vs, mask = staged(cache, q, k, v)
    ref, p, _, spread = exact_attention(qs, ks, vs, visible(Q, ks.size(2), mask), 1.0)
    out, _ = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
    assert_rounded_once(out, ref, spread, ks.size(2), "out")


NAN, INF = float("nan"), float("inf")


def poison(v, at):
    """Rows of the chunk that hold what a product with zero does not survive: NaN, both infinities, and one dim with an
    infinity of each sign from two tokens."""
    v[:, :, at, 3], v[:, :, at, 5], v[:, :, at, 7] = NAN, INF, -INF
    v[:, :, at, 9], v[:, :, at + 2, 9] = INF, -INF


def check_classes(out, p, v, what):
    """Finite, infinite and NaN where the sum over the keys with a probability above zero is, and its value where finite."""
    pd, vd = p.float() > 0, v.double()
    finite = torch.where(torch.isfinite(vd), vd, 0.0)
    want = torch.matmul(p, finite)
    hit = lambda sel: torch.matmul(pd.double(), sel.double()) > 0
    up, down, bad = hit(vd == INF), hit(vd == -INF), hit(torch.isnan(vd))
    bad = bad | (up & down)
    assert torch.equal(torch.isnan(out), bad), f"{what}: {(torch.isnan(out) != bad).sum().item()} values NaN or not"
    assert torch.equal(out == INF, up & ~bad) and torch.equal(out == -INF, down & ~bad), f"{what}: infinities"
    fine = ~(up | down | bad)
    err = (out.double() - want)[fine].abs().max().item()
    assert err <= (1e-5 if out.dtype == F32 else 1e-2), f"{what}: {err:.2e}"


@pytest.mark.parametrize("D,dtype", [(64, F32), (128, F32), (64, BF16), (64, F16)])
@pytest.mark.parametrize("n_ctx,n_kv,at", [(96, 96, 37), (300, 1000 + 300, 130), (64, 64, 0), (40, 3000 + 40, 33)])
def test_values_of_later_tokens_reach_no_earlier_row(D, dtype, n_ctx, n_kv, at):
    from cascading_kv_cache_amd.flash_attention import attention

    q, k, v, mask, _ = dense_case(1, 2, n_ctx, n_kv, D, dtype)
    poison(v, n_kv - n_ctx + at)
    out, _ = attention(q, k, v, True, 0.3, mask, 0.9)
    _, p, _, _ = exact_attention(q, k, torch.zeros_like(v), visible(n_ctx, n_kv, mask), 0.3)
    check_classes(out, p, v, "dense")
    assert torch.isfinite(out[:, :, :at].float()).all()


@pytest.mark.parametrize("D,dtype", [(64, F32), (128, F32), (64, BF16), (64, F16)])
def test_values_of_keys_with_probability_zero_are_not_touched(D, dtype):
    """A logit so far below the row's largest that its probability is zero in float32: the value row does not count."""
    from cascading_kv_cache_amd.flash_attention import attention

    q, k, v, mask, _ = dense_case(1, 2, 70, 400 + 70, D, dtype)
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, :, 11, 0], k[:, :, 410, 0] = -256.0, -256.0     # logits 600 below the others
    mask[11] = False
    k[:, :, 224:256, 0] = -256.0                          # and a block of them that nobody else shares
    mask[224:256] = False
    poison(v, 11)
    v[:, :, 410], v[:, :, 224:256] = NAN, INF
    mask[13] = True                                       # poison()'s second row
    out, _ = attention(q, k, v, True, 0.3, mask, 0.9)
    assert torch.isfinite(out.float()).all()


@pytest.mark.parametrize("D,dtype,W,C,filled,Q", [
    (128, F32, 512, 4, 4000, 40), (64, F32, 64, 2, 300, 40), (64, BF16, 512, 4, 4000, 40), (64, F16, 64, 2, 300, 100)])
def test_later_values_of_a_chunk_reach_no_earlier_row(D, dtype, W, C, filled, Q):
    """The same over a cache, with the keys shared out over workgroups (512 x 4) and not."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, 8, 2, D, 4, W, C, filled, Q, dtype)
    poison(v, 21)
    qs, ks, vs, mask = staged(cache, q, k, v)
    _, p, _, _ = exact_attention(qs, ks, torch.zeros_like(vs), visible(Q, ks.size(2), mask), 1.0)
    out, _ = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
    check_classes(out, p, vs, "cascade")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("W,C,filled", [(64, 1, 100), (512, 4, 4000)])   # one share of the keys, and four
def test_a_row_whose_logits_all_overflow_is_nan_however_its_keys_are_shared(D, W, C, filled):
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, 8, 2, D, 4, W, C, filled, 40, F32)
    for t, x in ((q, 1e20), (k, -1e20), (cache.key_cache[0], -1e20), (cache.sink_keys[0], -1e20)):
        t.zero_()
        t[..., 0] = x
    q[:, :, 7] = 0.0          # a row with logits of zero among them
    out, _ = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
    rows = torch.arange(40, device="cuda") != 7
    assert torch.isnan(out[:, :, rows]).all() and torch.isfinite(out[:, :, 7]).all()


@pytest.mark.parametrize("D,dtype", [(64, F32), (128, F32), (64, BF16), (64, F16), (128, BF16), (128, F16)])
@pytest.mark.parametrize("W,C,filled", [(64, 1, 100), (512, 4, 4000)])   # one share of the keys, and several
def test_a_key_that_is_nan_makes_every_row_that_sees_it_nan_however_its_keys_are_shared(D, dtype, W, C, filled):
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, 8, 2, D, 4, W, C, filled, 40, dtype)
    cache.key_cache[0][:, 1, 11] = NAN
    out, _ = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
    assert torch.isnan(out[:, 4:]).all() and torch.isfinite(out[:, :4].float()).all()


@pytest.mark.parametrize("D,dtype", [(64, F32), (128, F32), (64, BF16), (64, F16), (128, BF16), (128, F16)])
@pytest.mark.parametrize("H,KVH,W,C,filled,Q", [(32, 8, 320, 4, 200, 64), (8, 2, 512, 4, 100, 40)])
def test_a_share_of_the_keys_with_nothing_but_nan_reaches_its_rows(H, KVH, W, C, filled, Q, D, dtype):
    """Every cached key is NaN and every key of the chunk finite: they lie in different shares."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, H, KVH, D, 4, W, C, filled, Q, dtype)
    cache.key_cache[0][:, 1] = NAN
    cache.sink_keys[0][:, 1] = NAN
    out, scores = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
    G = H // KVH
    assert torch.isnan(out[:, G:2 * G]).all() and torch.isnan(scores[:, 1]).all()
    assert torch.isfinite(out[:, :G].float()).all() and torch.isfinite(scores[:, 0].float()).all()


def check_nan_keys(H, KVH, D, W, C, filled, Q, dtype, where, **kw):
    """Keys of kv head 1 that are all NaN, the cached ones or the chunk's: its rows are NaN and so are the chunk's scores; no others are."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, H, KVH, D, 4, W, C, filled, Q, dtype)
    for t in (cache.key_cache[0], cache.sink_keys[0]) if where == "cached" else (k,):
        t[:, 1] = NAN
    G = H // KVH
    for update in (False, True, True):   # a step of one token: from the second update on it runs beside the scores
        if where == "cached":            # where the last token's own key has gone in the meantime
            cache.key_cache[0][:, 1] = NAN
        out, scores = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=update, **kw)
        assert torch.isnan(out[:, G:2 * G]).all() and torch.isnan(scores[:, 1]).all()
        assert torch.isfinite(out[:, :G].float()).all() and torch.isfinite(scores[:, 0].float()).all()


@pytest.mark.parametrize("dtype", [BF16, F16, F32])
@pytest.mark.parametrize("where", ["cached", "chunk"])
@pytest.mark.parametrize("do_og_pos", [False, True])
@pytest.mark.parametrize("H,KVH,W,C,filled", [(8, 2, 64, 1, 40), (8, 2, 512, 4, 100), (14, 2, 512, 4, 1500), (32, 8, 4096, 4, 9000)])
def test_nan_keys_in_a_single_token_step(H, KVH, W, C, filled, where, do_og_pos, dtype):
    """Whole tiles of them, also as the only tile with a visible key."""
    check_nan_keys(H, KVH, 128, W, C, filled, 1, dtype, where, do_og_pos=do_og_pos)


@pytest.mark.parametrize("D,Q,dtype", [(64, 1, BF16), (64, 1, F16), (96, 1, F32), (96, 33, F32), (96, 33, BF16), (40, 2, F32), (192, 70, F16),
                                       (64, 33, BF16), (128, 40, F16), (64, 70, F32), (128, 33, F32)])
@pytest.mark.parametrize("where", ["cached", "chunk"])
@pytest.mark.parametrize("W,C,filled", [(64, 1, 40), (64, 1, 60), (512, 4, 100), (512, 4, 1500)])   # 44 and 64 visible keys: part of a
def test_nan_keys_at_any_head_size(W, C, filled, where, D, Q, dtype):                               # chunk of 64 and all of it
    check_nan_keys(8, 2, D, W, C, filled, Q, dtype, where)


@pytest.mark.parametrize("D,dtype", [(128, BF16), (128, F16), (64, F16), (128, F32)])
@pytest.mark.parametrize("H,KVH,W,C,filled,Q", [(8, 2, 1024, 4, 1000, 128), (32, 8, 1024, 4, 4095, 300), (8, 2, 2048, 8, 3000, 33),
                                                (7, 1, 64, 2, 90, 40)])
def test_the_filled_slots_hint_changes_no_bit_of_a_chunk(D, dtype, H, KVH, W, C, filled, Q):
    """Chunks over a cache that is filling, with the hint (from the host's token counter) and without (``replayable``):
    the number of workgroups that share a row's keys is a matter of sizes, not of how many slots hold a token."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, H, KVH, D, 4, W, C, filled, Q, dtype)
    before = cache.score_cache[0].clone()
    results = []
    for replayable in (False, True):
        cache.score_cache[0].copy_(before)
        out, new_scores = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False, replayable=replayable)
        results.append([t.clone().view(torch.uint8) for t in (out, new_scores, cache.score_cache[0])])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def float32_chunk(Q, D, H, KVH, S, seed):
    """A chunk of a first call: an empty cache whose hidden slots hold NaN, no rotation (all frequencies zero)."""
    from cascading_kv_cache_amd.cascading_cache import CascadingKVCache

    cache = CascadingKVCache(window_length=S // 2, num_sink_tokens=3, max_batch_size=1, heads=KVH, dim=D, max_seq_len=S,
                             device="cuda:0", dtype=F32, layers=1, verbose=False)
    for t in (cache.key_cache[0], cache.value_cache[0], cache.sink_keys[0], cache.sink_values[0]):
        t.fill_(float("nan"))
    gen = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(1, h, Q, D, generator=gen).cuda() for h in (H, KVH, KVH))
    return cache, q, k, v, torch.zeros(D // 2, device="cuda")


@pytest.mark.parametrize("D,Q,H,KVH,S", [(128, 70, 4, 2, 64), (64, 33, 7, 1, 10), (128, 31, 2, 2, 700), (64, 300, 8, 2, 98)])
def test_float32_chunk_of_values_that_three_planes_do_not_take(D, Q, H, KVH, S):
    """Infinite, NaN and the largest finite values in queries, keys and values of a float32 chunk, whose operands are the sums of
    three bfloat16 planes: what is not finite reaches the rows that it reaches in float64, and no other."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, freq = float32_chunk(Q, D, H, KVH, S, 3)
    q[0, 0, 7, 3] = float("inf")          # its row is NaN: the rotation multiplies it by zero
    q[0, 1, 9, 0] = float("nan")
    q[0, 0, ::2, 5], q[0, 0, 1::2, 5] = 100., -100.
    k[0, 0, 12, 5] = 3e38                 # logits past the largest number: NaN for every other row, the rest do not see the key
    v[0, 0, 4, 2] = float("inf")
    v[0, 0, 6, 2] = float("-inf")         # from row 6 on both: NaN
    v[0, -1, 20, 1] = 3.4e38              # rounds to no finite bfloat16
    v[0, -1, 21, 0] = float("nan")
    out, scores = cascade_attention(q, k, v, cache, 0, freq, update_cache=False)
    G = H // KVH
    kk, vv = (t.double().cpu().repeat_interleave(G, 1) for t in (k, v))
    logits = ((q.double().cpu()[..., None, :] * kk[:, :, None]).sum(-1) / D ** 0.5).float().double()
    logits[0, 0, 7] = float("nan")
    p = logits.masked_fill(torch.ones(Q, Q, dtype=torch.bool).triu(1), float("-inf")).softmax(-1)
    # a key of probability zero counts for nothing, whatever its value
    terms = torch.where(p[..., None] == 0, 0., p[..., None] * vv[:, :, None])
    want, got = terms.sum(-2), out.double().cpu()
    for test in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(test(got), test(want))
    assert torch.isnan(want).any() and torch.isposinf(want).any() and torch.isfinite(want).sum() > want.numel() // 2
    fine = torch.isfinite(want)
    # a float32 sum of up to Q terms; logits of up to 100 * 4 / 8 = 2^6 are off by a unit or two
    size = terms.abs().sum(-2)[fine]
    assert ((got - want)[fine].abs() <= 2.0 ** -23 * (Q ** 0.5 + 2 * 2 ** 6) * size).all()
    assert torch.isnan(scores[0, 0, :8]).all() and (KVH == 1 or torch.isfinite(scores[0, -1, 10:]).all())   # rows 7 and 9


def ema_scores(p, beta, G):
    """What a chunk adds to the scores of the keys in front of it, in float64: the weighted sums over its rows, averaged over a kv head's."""
    Q = p.size(2)
    w = (1 - beta) * beta ** torch.arange(Q - 1, -1, -1, device=p.device, dtype=torch.float64)
    sums = (p * w[:, None]).sum(2)
    return sums.reshape(p.size(0), -1, G, sums.size(-1)).mean(2)


@pytest.mark.parametrize("octaves", [-112, -122])
@pytest.mark.parametrize("B,H,KVH,D,NS,W,C,filled,Q", [(1, 32, 8, 128, 4, 128, 4, 400, 96), (1, 8, 2, 128, 4, 512, 4, 2000, 40),
                                                       (2, 7, 1, 64, 3, 90, 2, 100, 33), (1, 8, 2, 64, 4, 512, 4, 1500, 70)])
def test_float32_chunk_of_operands_far_below_one(B, H, KVH, D, NS, W, C, filled, Q, octaves):
    """Values, and keys against queries as far above one, of which the lowest of three bfloat16 planes would be no number
    or half of one: no bits are lost."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(B, H, KVH, D, NS, W, C, filled, Q, F32)
    cache.beta = 0.9
    small = 2.0 ** octaves
    qs, ks, vs, mask = staged(cache, q, k, v)
    see = visible(Q, ks.size(2), mask)
    before = cache.score_cache[0].clone()
    # values
    cache.value_cache[0].mul_(small)
    cache.sink_values[0].mul_(small)
    ref, p, _, spread = exact_attention(qs, ks, vs, see, 1.0)
    out, scores = cascade_attention(q, k, v * small, cache, 0, inv_freq, update_cache=False)
    assert_rounded_once(out * 2.0 ** -octaves, ref, spread, ks.size(2), "small values")
    want = cache.beta ** Q * before.double() + ema_scores(p, cache.beta, H // KVH)[..., NS:-Q]
    seen = ~mask[NS:]
    assert ((cache.score_cache[0].double() - want).abs()[..., seen] <= 2.0 ** -17 * want[..., seen]).all()
    # keys, and queries the other way
    cache.value_cache[0].mul_(1 / small)
    cache.sink_values[0].mul_(1 / small)
    cache.score_cache[0].copy_(before)
    for t in (cache.key_cache[0], cache.sink_keys[0]):
        t.mul_(small)
    out2, scores2 = cascade_attention(q / small, k * small, v, cache, 0, inv_freq, update_cache=False)
    assert_rounded_once(out2, ref, spread, ks.size(2), "small keys")
    assert ((cache.score_cache[0].double() - want).abs()[..., seen] <= 2.0 ** -17 * want[..., seen]).all()
    assert ((scores2 - scores).abs() <= 2.0 ** -17 * scores).all()


@pytest.mark.parametrize("octaves", [-104, -130])
@pytest.mark.parametrize("H,KVH,D,NS,W,C,filled,Q", [(32, 8, 128, 4, 128, 4, 400, 96), (8, 2, 128, 4, 512, 4, 2000, 40), (7, 1, 64, 3, 90, 2, 100, 33)])
def test_float32_chunk_of_faint_probabilities(H, KVH, D, NS, W, C, filled, Q, octaves):
    """A sink that takes all but 2^-104 (2^-130: less than the smallest normal number) of every row, and whose value is zero: what is left
    of the row is sums of the others."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    cache, q, k, v, inv_freq = cascade_case(1, H, KVH, D, NS, W, C, filled, Q, F32)
    cache.beta = 0.5
    rs = math.sqrt(1 / math.sqrt(D))
    q[..., 0] = 1.0 / rs
    for t in (k, cache.key_cache[0], cache.sink_keys[0]):
        t[..., 0] = 0.0
    cache.sink_keys[0][:, :, 0] = 0.0
    cache.sink_keys[0][:, :, 0, 0] = -octaves * math.log(2.0) / rs
    cache.sink_values[0][:, :, 0] = 0.0
    cache.score_cache[0].zero_()
    qs, ks, vs, mask = staged(cache, q, k, v)
    see = visible(Q, ks.size(2), mask)
    logits = torch.matmul(qs.double(), ks.double().transpose(2, 3).contiguous()).masked_fill(~see, float("-inf"))
    p = (logits - logits.amax(-1, keepdim=True)).exp()   # torch's softmax on the device has zeros below 2^-126
    p /= p.sum(-1, keepdim=True)
    ref, spread = torch.matmul(p, vs.double()), torch.matmul(p * p, vs.double() ** 2).sqrt()
    assert (ref != 0).all()
    out, _ = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
    # a logit of 90 is off by 2^-18 or so, and a subnormal of 2^-130 holds 19 bits
    bound = 2.0 ** -15 * (ref.abs() + spread) + 2.0 ** -147
    assert ((out.double() - ref).abs() <= bound).all()
    want = ema_scores(p, cache.beta, H // KVH)[..., NS:-Q]
    seen = ~mask[NS:]
    assert ((cache.score_cache[0].double() - want).abs()[..., seen] <= 2.0 ** -15 * want[..., seen] + Q * 2.0 ** -149).all()


@pytest.mark.parametrize("D,Q,H,KVH,S", [(128, 65, 4, 2, 64), (64, 40, 7, 1, 30)])
def test_float32_chunk_of_rows_that_are_not_aligned(D, Q, H, KVH, S):
    """Rows that start at any element are staged element by element: the same result to the bit."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention

    results = []
    for layout in (lambda t: t, lambda t: torch.cat((t[..., :1], t), -1)[..., 1:]):
        cache, q, k, v, freq = float32_chunk(Q, D, H, KVH, S, 5)
        q, k, v = (layout(t) for t in (q, k, v))
        results.append(cascade_attention(q, k, v, cache, 0, freq + 0.01, update_cache=False))
    assert torch.equal(q, float32_chunk(Q, D, H, KVH, S, 5)[1]) and q.data_ptr() % 16 != 0
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Z,H,n_ctx,n_kv", [
    (1, 1, 385, 385), (1, 2, 384, 100 + 384), (1, 3, 1000, 900 + 1000),   # a share of 128 to 256 rows; blocks of chunk keys have fewer
    (1, 8, 257, 257), (3, 5, 513, 31 + 513), (1, 16, 900, 7000 + 900)])   # one share of two tiles, and where blocks fill the chip
def test_dense_score_sums_in_shares_of_the_rows(Z, H, n_ctx, n_kv, D, dtype):
    """Few blocks of keys share their query tiles out over workgroups, whose sums are added in order."""
    from cascading_kv_cache_amd import flash_attention as fa

    q, k, v, mask, _ = dense_case(Z, H, n_ctx, n_kv, D, dtype)
    scale = 0.5 if D == 64 else 0.1
    _, scores, _, _ = fa._forward(q, k, v, True, scale, mask, 0.9, False)
    _, p, _, _ = exact_attention(q, k, v, visible(n_ctx, n_kv, mask), scale)
    w = (0.1 * 0.9 ** torch.arange(n_ctx - 1, -1, -1, device="cuda", dtype=torch.float64))[None, None, :, None]
    want = (w * p).sum(2)
    if D == 64:
        assert_rounded_once(scores, want, (w * p).square().sum(2).sqrt(), n_ctx, "scores")
    else:   # the staged queries are rounded, logits of some 8 are off by 2^-8 (2^-11) of that, and a score by as much
        assert (scores.double() - want).norm() <= 8 * HALF_ULP[dtype] * want.norm()
    hidden = torch.cat((mask, torch.zeros(n_ctx, dtype=torch.bool, device="cuda")))
    assert (scores[:, :, hidden] == 0).all()
