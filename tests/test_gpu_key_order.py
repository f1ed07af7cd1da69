"""The dense operator's masked keys: staging blocks that look for their keys in the mask themselves (up to 16 K cached keys, 4096 at a time)
and a key order from a launch in front of them (more), against the formula."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cached", [0, 1, 63, 64, 65, 4095, 4096, 4097, 8191, 12300, 16383, 16384, 16385])
@pytest.mark.parametrize("masking", ["random", "all", "none", "one", "last stretch", "misaligned"])
def test_masked_keys_are_left_out(n_cached, masking):
    from cascading_kv_cache_amd.flash_attention import attention

    H, n_ctx, D, beta = 2, 70, 128, 0.999
    g = torch.Generator(device="cuda").manual_seed(n_cached)
    q, k, v = (torch.randn(1, H, n, D, generator=g, device="cuda").bfloat16() * 0.7 for n in (n_ctx, n_cached + n_ctx, n_cached + n_ctx))
    mask = torch.rand(n_cached + 1, generator=g, device="cuda") > 0.5
    mask = mask[1:] if masking == "misaligned" else mask[1:].clone()
    if masking in ("all", "one", "last stretch"):
        mask.fill_(True)
    if masking == "none":
        mask.fill_(False)
    if n_cached and masking == "one":
        mask[n_cached // 2] = False
    if n_cached and masking == "last stretch":
        mask[max(0, n_cached - 70):] = False
    out, scores = attention(q, k, v, True, 0.1, mask, beta)
    hidden = torch.cat((mask, torch.zeros(n_ctx, dtype=torch.bool, device="cuda")))[None, :].repeat(n_ctx, 1)
    hidden[:, n_cached:] = torch.ones(n_ctx, n_ctx, device="cuda").triu(1).bool()
    p = (torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * 0.1).masked_fill(hidden, float("-inf")).softmax(-1)
    want = torch.matmul(p, v.double())
    sums = (p * ((1 - beta) * beta ** torch.arange(n_ctx - 1, -1, -1, device="cuda", dtype=torch.float64))[:, None]).sum(2)
    assert (out.double() - want).abs().max() <= 2e-2
    assert (scores.double() - sums).abs().max() <= 2e-2 * sums.max()
    assert not scores[..., :n_cached][..., mask].any()


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (64, torch.bfloat16), (128, torch.float16)])
@pytest.mark.parametrize("n_cached", [1, 65, 4097, 16384, 16385])
@pytest.mark.parametrize("masking", ["random", "last stretch"])
def test_masked_keys_are_left_out_of_gradients_too(masking, n_cached, D, dtype):
    """The other instances of the same staging, and the backward behind them.  A gradient is a sum over rows or keys of products that
    each round P, dP or the result to the format once: four roundings of the largest value, and of the sums that meet in dS."""
    from cascading_kv_cache_amd.flash_attention import attention

    H, n_ctx, beta = 2, 70, 0.999
    g = torch.Generator(device="cuda").manual_seed(n_cached + D)
    q, k, v, do = (torch.randn(1, H, n, D, generator=g, device="cuda").to(dtype) * 0.7 for n in (n_ctx, n_cached + n_ctx, n_cached + n_ctx, n_ctx))
    mask = torch.rand(n_cached, generator=g, device="cuda") > 0.5
    if masking == "last stretch":
        mask.fill_(True)
        mask[max(0, n_cached - 70):] = False
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    out, scores = attention(*leaves, True, 0.1, mask, beta)
    got = torch.autograd.grad(out, leaves, do)
    exact = [t.double().requires_grad_() for t in (q, k, v)]
    hidden = torch.cat((mask, torch.zeros(n_ctx, dtype=torch.bool, device="cuda")))[None, :].repeat(n_ctx, 1)
    hidden[:, n_cached:] = torch.ones(n_ctx, n_ctx, device="cuda").triu(1).bool()
    p = (torch.matmul(exact[0], exact[1].transpose(2, 3).contiguous()) * 0.1).masked_fill(hidden, float("-inf")).softmax(-1)
    o = torch.matmul(p, exact[2])
    want = torch.autograd.grad(o, exact, do.double())
    sums = (p * ((1 - beta) * beta ** torch.arange(n_ctx - 1, -1, -1, device="cuda", dtype=torch.float64))[:, None]).sum(2)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert (out.double() - o).abs().max() <= 4 * unit * o.abs().max()
    assert (scores.double() - sums).abs().max() <= 4 * unit * sums.max() + 2.0 ** -24   # float16's smallest step
    for name, a, b in zip("qkv", got, want):
        assert (a.double() - b).abs().max() <= 4 * unit * b.abs().max(), name
    for grad in got[1:]:
        assert not grad[:, :, :n_cached][:, :, mask].any()
