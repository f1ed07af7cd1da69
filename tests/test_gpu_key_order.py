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
