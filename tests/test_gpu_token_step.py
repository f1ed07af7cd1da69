"""A single-token step whose cache update runs beside its scores (ckv_attn_update) against the same step in two calls
(ckv_attn, then ckv_update): outputs, new scores and every state tensor bit-identical after every token, from an empty
cache through sinks, filling and eviction."""
import ctypes

import pytest
import torch

from parity_helpers import STATE, bits

pytestmark = pytest.mark.gpu


def pair(B, KVH, NS, W, C, dtype, func, eager, reduction):
    from cascading_kv_cache_amd.cascading_cache import CascadingKVCache

    caches = [CascadingKVCache(window_length=W, num_sink_tokens=NS, max_batch_size=B, heads=KVH, dim=128, max_seq_len=W * C,
                               device="cuda:0", dtype=dtype, cascade_func=func, eager_fill=eager, head_reduction=reduction,
                               layers=1, verbose=False) for _ in range(2)]
    for c in caches:
        c.beta = 0.9   # scores that differ from slot to slot and change at every step
    return caches


def run_steps(one, two, B, H, KVH, dtype, tokens, gen, prompt=0):
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq

    inv_freq = default_inv_freq(128, 5e5, "cuda:0")
    draw = lambda h, n: (torch.randn(B, n, h, 128, generator=gen) * 0.7).to(dtype).cuda().transpose(1, 2)   # noqa: E731
    if prompt:
        q, k, v = draw(H, prompt), draw(KVH, prompt), draw(KVH, prompt)
        for c in (one, two):
            cascade_attention(q, k, v, c, 0, inv_freq)
    for t in range(tokens):
        q, k, v = draw(H, 1), draw(KVH, 1), draw(KVH, 1)
        if t % 5 == 3:
            q = torch.zeros_like(q)   # every visible key weighs the same: ties
        out1, new1 = cascade_attention(q, k, v, one, 0, inv_freq)
        out2, new2 = cascade_attention(q, k, v, two, 0, inv_freq, update_cache=False)
        two.update_state(k, v, 0, new2)
        torch.cuda.synchronize()
        assert torch.equal(bits(out1), bits(out2)) and torch.equal(bits(new1), bits(new2)), t
        for name in STATE:
            assert torch.equal(bits(getattr(one, name)[0]), bits(getattr(two, name)[0])), (t, name)
        assert torch.equal(one.seen_tokens_by_layer, two.seen_tokens_by_layer) and one._seen_host == two._seen_host


def step_end(cache, H):
    """How the single-token steps that ``cache`` has seen end on this device: launches apart (0), rows and scores in one (1), the update too
    (2); and whether their argument blocks are such that the update may come along."""
    from cascading_kv_cache_amd import _abi

    lib = ctypes.CDLL(_abi.LIB_PATH)
    B, KVH, S = cache.key_cache[0].shape[:3]
    blocks = [a for a in cache._attn_memo.values() if a.Q == 1 and a._update is not None]
    assert blocks
    belongs = {lib.ckv_decode_update_belongs(ctypes.byref(a), ctypes.byref(a._update)) for a in blocks}
    assert len(belongs) == 1
    sizes = [ctypes.c_int64(n) for n in (B, H, KVH, cache.num_sink_tokens, S, 0)]
    return lib.ckv_decode_step_end(*sizes), bool(belongs.pop())


# windows of one slot, odd ones (position ids one by one), one cascade, as many as a workgroup takes and one more (two calls
# inside), schedules whose periods do not divide each other, more (batch, kv head) pairs than the planning workgroups take
@pytest.mark.parametrize("B,H,KVH,NS,W,C,dtype,func,eager,reduction,tokens", [
    (1, 8, 2, 4, 3, 5, torch.bfloat16, "pow2", True, "mean", 60),
    (2, 4, 4, 1, 4, 4, torch.float16, "pow2", False, "max", 60),
    (1, 14, 2, 0, 2, 6, torch.bfloat16, "iplus1", True, "median", 60),
    (3, 8, 1, 2, 1, 7, torch.float16, "1-then-2", True, "mean", 40),
    (1, 2, 1, 4, 16, 1, torch.bfloat16, "pow2", True, "max", 40),
    (1, 4, 2, 4, 2, 31, torch.bfloat16, "pow2-1", True, "median", 110),
    (1, 4, 2, 4, 2, 32, torch.bfloat16, "pow2-1", False, "mean", 40),
    (33, 8, 8, 3, 4, 3, torch.bfloat16, "pow2-2-4", True, "mean", 24),
])
def test_update_beside_the_scores_equals_two_calls(B, H, KVH, NS, W, C, dtype, func, eager, reduction, tokens):
    one, two = pair(B, KVH, NS, W, C, dtype, func, eager, reduction)
    run_steps(one, two, B, H, KVH, dtype, tokens, torch.Generator().manual_seed(tokens + C), 0)
    assert step_end(one, H) == (2 if B < 33 else 1, C < 32)


# several workgroups of scores and position ids per (batch, kv head); more (batch, kv head) pairs than the planning workgroups take; the
# step in separate launches (its workgroups past four a compute unit); more than four heads per kv head and the update's workgroups past
# the one round
@pytest.mark.parametrize("B,H,KVH,NS,W,C,prompt,end", [(2, 8, 2, 4, 1500, 3, 4800, 2), (1, 28, 4, 64, 4096, 2, 8600, 2),
                                                       (40, 8, 8, 4, 8192, 2, 300, 1), (32, 8, 8, 64, 6144, 2, 300, 0),
                                                       (10, 28, 4, 64, 4096, 4, 700, 1)])
def test_update_beside_the_scores_of_many_slots(B, H, KVH, NS, W, C, prompt, end):
    one, two = pair(B, KVH, NS, W, C, torch.bfloat16, "pow2", True, "mean")
    run_steps(one, two, B, H, KVH, torch.bfloat16, 6, torch.Generator().manual_seed(5), prompt)
    assert step_end(one, H) == (end, True)


def test_a_cache_with_an_update_of_its_own_is_asked_every_time():
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq
    from cascading_kv_cache_amd.cascading_cache import CascadingKVCache

    class Counting(CascadingKVCache):
        calls = 0

        def update_state(self, *args, **kw):
            self.calls += 1
            return super().update_state(*args, **kw)

    args = dict(window_length=8, num_sink_tokens=4, max_batch_size=1, heads=2, dim=128, max_seq_len=32, device="cuda:0",
                dtype=torch.bfloat16, layers=1, verbose=False)
    plain, counting, patched = CascadingKVCache(**args), Counting(**args), CascadingKVCache(**args)
    given = []
    inner = patched.update_state
    patched.update_state = lambda *a, **kw: (given.append(1), inner(*a, **kw))[1]
    inv_freq, gen = default_inv_freq(128, 5e5, "cuda:0"), torch.Generator().manual_seed(3)
    for n in (20, 1, 1, 1, 3, 1):
        q, k, v = ((torch.randn(1, h, n, 128, generator=gen)).bfloat16().cuda() for h in (8, 2, 2))
        outs = [cascade_attention(q, k, v, c, 0, inv_freq)[0] for c in (plain, counting, patched)]
        assert torch.equal(bits(outs[0]), bits(outs[1])) and torch.equal(bits(outs[0]), bits(outs[2]))
    assert counting.calls == 6 and len(given) == 6
    for c in (counting, patched):
        for name in STATE:
            assert torch.equal(bits(getattr(plain, name)[0]), bits(getattr(c, name)[0])), name


def test_a_refused_step_counts_nothing(monkeypatch):
    from cascading_kv_cache_amd import _abi
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq

    cache, _ = pair(1, 2, 4, 8, 2, torch.bfloat16, "pow2", True, "mean")
    inv_freq = default_inv_freq(128, 5e5, "cuda:0")
    q, k = (torch.zeros(1, h, 1, 128, dtype=torch.bfloat16, device="cuda:0") for h in (8, 2))
    for _ in range(2):
        cascade_attention(q, k, k, cache, 0, inv_freq)
    before = cache._seen_tokens, list(cache._seen_host), list(cache._seen_pending)
    assert before == (2, [2], [2])
    for name in ("ckv_attn_update", "ckv_update"):   # what the library says to a call that it refuses
        monkeypatch.setattr(_abi.lib(), name, lambda *args: 3)
    with pytest.raises(_abi.CkvError):
        cascade_attention(q, k, k, cache, 0, inv_freq)
    with pytest.raises(_abi.CkvError):
        cache.update_state(k, k, 0, k[..., 0])
    assert (cache._seen_tokens, cache._seen_host, cache._seen_pending) == before


def lower_median(vals):
    """Of the heads along dim 2: the value that takes place (G - 1) // 2, a NaN behind all others, as counting ranks finds it."""
    G = vals.size(2)
    order = torch.where(vals.isnan(), torch.full_like(vals, float("inf")), vals).sort(dim=2).values
    return order[:, :, (G - 1) // 2]


@pytest.mark.parametrize("B,window", [(1, 96), (40, 64)])   # rows, scores and update in one launch; apart
@pytest.mark.parametrize("G", [1, 2, 4, 7, 8])
@pytest.mark.parametrize("spoilt", [False, True])
def test_median_of_a_groups_heads(spoilt, G, B, window):
    """Scores of a step that starts from zeros, against the median of the same heads' scores as kv heads of their own.  A head of no
    numbers counts as the largest."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq

    KVH, gen = 2, torch.Generator().manual_seed(G)
    inv_freq = default_inv_freq(128, 5e5, "cuda:0")
    draw = lambda h, n: (torch.randn(B, n, h, 128, generator=gen) * 0.7).bfloat16().cuda().transpose(1, 2)   # noqa: E731
    steps = [(draw(KVH * G, n), draw(KVH, n), draw(KVH, n)) for n in (2 * window + 4, 1)]
    if spoilt:
        steps[-1][0][:, 0] = float("nan")
    got = []
    for heads in (KVH, KVH * G):
        cache = pair(B, heads, 4, window, 2, torch.bfloat16, "pow2", True, "median")[0]
        for i, (q, k, v) in enumerate(steps):
            if heads != KVH:
                k, v = (x.repeat_interleave(G, 1) for x in (k, v))
            cache.score_cache[0].zero_()
            new = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=i == 0)[1]
        got.append((cache.score_cache[0].float(), new.float()))
    (scores, new), (each, each_new) = got
    for mine, every in ((scores, each), (new, each_new)):
        want = lower_median(every.view(B, KVH, G, -1))
        if G == 1:
            want = every
        assert torch.equal(mine.isnan(), want.isnan())
        # one rounding to bfloat16 of probabilities that two kernels work out
        assert torch.allclose(mine, want, rtol=2.0 ** -7, atol=1e-9, equal_nan=True)


@pytest.mark.parametrize("B,window", [(1, 96), (40, 64)])   # rows, scores and update in one launch; apart
@pytest.mark.parametrize("G", [1, 2, 4, 7, 8])
@pytest.mark.parametrize("spoilt", [False, True])
def test_median_of_a_groups_heads_is_one_of_their_values(spoilt, G, B, window):
    """To the bit: a head's own values come from the same step with its queries in every head's place, where any reduction gives them."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq

    KVH, gen = 2, torch.Generator().manual_seed(G + 20)
    inv_freq = default_inv_freq(128, 5e5, "cuda:0")
    draw = lambda h, n: (torch.randn(B, n, h, 128, generator=gen) * 0.7).bfloat16().cuda().transpose(1, 2)   # noqa: E731
    (q0, k0, v0), (q, k, v) = ((draw(KVH * G, n), draw(KVH, n), draw(KVH, n)) for n in (2 * window + 4, 1))
    if spoilt:
        q[:, 0] = float("nan")
    cache = pair(B, KVH, 4, window, 2, torch.bfloat16, "pow2", True, "median")[0]
    cascade_attention(q0, k0, v0, cache, 0, inv_freq)

    def scores(queries):
        cache.score_cache[0].zero_()
        new = cascade_attention(queries, k, v, cache, 0, inv_freq, update_cache=False)[1]
        return torch.cat((cache.score_cache[0], new), dim=-1).float()

    got = scores(q)
    heads = q.reshape(B, KVH, G, 1, 128)
    each = torch.stack([scores(heads[:, :, g:g + 1].expand(-1, -1, G, -1, -1).reshape(B, KVH * G, 1, 128)) for g in range(G)], dim=2)
    want = lower_median(each) if G > 1 else each[:, :, 0]
    assert torch.equal(got.isnan(), want.isnan()) and got.isnan().any() == (spoilt and G < 2)
    assert torch.equal(bits(got.nan_to_num()), bits(want.nan_to_num()))
