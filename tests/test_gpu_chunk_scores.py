"""Score sums of a chunk's own keys: weights that are all alike (the default beta) and weights by distance, wavefronts whose 64 keys are
all the chunk's and the one in which the chunk starts, lengths around the 32-row subtiles and the 128-row tiles."""
import ctypes

import pytest
import torch

from oracle.attention import OracleCascadeAttention
from parity_helpers import assert_scores_close, flip_bound, push_state, tol
from test_gpu_attention import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (128, torch.float16), (64, torch.bfloat16)])
@pytest.mark.parametrize("NS", [3, 64])
@pytest.mark.parametrize("beta", [None, 0.9])
def test_scores_of_the_chunks_own_keys(beta, NS, D, dtype):
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq

    B, H, KVH, W, C = 1, 4, 2, 128, 8
    gpu, cpu = make_pair(B, KVH, D, NS, W, C, dtype)
    if beta is not None:
        gpu.beta = cpu.beta = beta
    layer = OracleCascadeAttention(H, KVH, D, rope_theta=5e5, head_reduction="mean")
    inv_freq = default_inv_freq(D, 5e5, "cuda:0")
    gen = torch.Generator().manual_seed(3)
    for q_len in (600, 300, 33, 129, 31, 64, 97):   # the last over a cache that evicts
        q, k, v = ((torch.randn(B, h, q_len, D, generator=gen) * 0.7).to(dtype) for h in (H, KVH, KVH))
        push_state(gpu, cpu)
        out, new = cascade_attention(q.cuda(), k.cuda(), v.cuda(), gpu, 0, inv_freq, update_cache=False)
        scores = gpu.score_cache[0].cpu()
        want = layer.forward(q, k, v, cpu)
        assert (out.float().cpu() - want.float()).abs().max() <= tol(dtype)
        assert_scores_close(new, layer.last_new_scores[:, :KVH], dtype, f"new-token scores, {q_len} rows")
        assert_scores_close(scores, layer.last_score_cache, dtype, f"score cache, {q_len} rows")


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (128, torch.float16), (64, torch.bfloat16)])
@pytest.mark.parametrize("H,KVH", [(8, 2), (7, 1)])
def test_chunks_whose_keys_are_shared_out_two_tiles_each(H, KVH, D, dtype):
    """Few rows over 1 K slots: a workgroup for every two of the 64-key tiles, shares without a visible key while the cache fills, and
    row counts around the 256 (position, head) rows of a workgroup."""
    from test_gpu_attention import run_teacher_forced

    led = run_teacher_forced(1, H, KVH, D, 4, 256, 4, 0, 0, dtype, seed=5, std=0.7, steps=[130, 16, 2, 65, 64, 129, 33, 100, 128, 127, 130, 130])
    assert led.flips <= flip_bound(led), led.summary()


# caches that fill (the walk) and full ones (closed forms), periods that do not divide each other, rings shorter than the chunk, the most
# tokens that share the launch and one more, seven and eight heads per kv head, more workgroups than one round takes
@pytest.mark.parametrize("B,H,KVH,D,NS,W,C,dtype,func,reduction,q_len,calls,rides", [
    (1, 8, 2, 128, 4, 33, 4, torch.bfloat16, "pow2", "mean", 17, 24, True),
    (2, 14, 2, 128, 0, 64, 3, torch.float16, "pow2", "median", 50, 10, True),
    (1, 8, 1, 64, 3, 40, 5, torch.bfloat16, "pow2", "median", 2, 60, True),
    (1, 4, 2, 64, 4, 128, 2, torch.float16, "iplus1", "max", 100, 8, True),
    (1, 8, 2, 128, 4, 128, 4, torch.float32, "pow2", "max", 256, 6, True),
    (3, 6, 2, 64, 1, 96, 1, torch.float32, "pow2", "median", 31, 8, True),
    (1, 4, 1, 128, 64, 512, 8, torch.bfloat16, "pow2", "mean", 1092, 6, True),
    (1, 4, 1, 128, 64, 512, 8, torch.bfloat16, "pow2", "mean", 1093, 6, False),
    (4, 16, 16, 64, 4, 8192, 2, torch.float16, "pow2", "max", 300, 3, False),
])
def test_update_planned_beside_the_finishing_scores_equals_two_calls(B, H, KVH, D, NS, W, C, dtype, func, reduction, q_len, calls, rides):
    from cascading_kv_cache_amd import _abi
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq
    from test_gpu_token_step import STATE, bits

    one, two = (make_pair(B, KVH, D, NS, W, C, dtype, func=func, reduction=reduction)[0] for _ in range(2))
    one.beta = two.beta = 0.99   # scores that change at every call
    inv_freq = default_inv_freq(D, 5e5, "cuda:0")
    gen = torch.Generator().manual_seed(7)
    for call in range(calls):
        q, k, v = ((torch.randn(B, q_len, h, D, generator=gen) * 0.7).to(dtype).cuda().transpose(1, 2) for h in (H, KVH, KVH))
        if call % 4 == 2:
            q = torch.zeros_like(q)   # every visible key weighs the same: ties
        if call == calls - 1:
            q[:, 0, q_len // 2] = float("nan")   # and a head's scores that are no numbers
        out1, new1 = cascade_attention(q, k, v, one, 0, inv_freq)
        out2, new2 = cascade_attention(q, k, v, two, 0, inv_freq, update_cache=False)
        two.update_state(k, v, 0, new2)
        assert torch.equal(bits(out1), bits(out2)) and torch.equal(bits(new1), bits(new2)), call
        for name in STATE:
            assert torch.equal(bits(getattr(one, name)[0]), bits(getattr(two, name)[0])), (call, name)
    lib = ctypes.CDLL(_abi.LIB_PATH)
    blocks = [a for a in one._attn_memo.values() if a.Q == q_len and a._update is not None]
    assert blocks and {bool(lib.ckv_chunk_plan_rides(ctypes.byref(a), ctypes.byref(a._update))) for a in blocks} == {rides}
    # scratch that would lie over what the finishing blocks still read (asked, not run)
    a, u = blocks[-1], type(blocks[-1]._update).from_buffer_copy(blocks[-1]._update)
    u.workspace = a.workspace + _abi.lib().ckv_attn_workspace_bytes(B, H, KVH, q_len, D, NS, W * C, a.dtype) - 512
    assert not lib.ckv_chunk_plan_rides(ctypes.byref(a), ctypes.byref(u))


@pytest.mark.parametrize("D,dtype", [(128, torch.float16), (128, torch.bfloat16), (64, torch.float16)])
def test_scores_do_not_hang_on_which_launch_merges_the_shares(D, dtype):
    """Seven shares of the same 16 K keys, merged in the launch of the score sums (a cache of 16 K slots) and in one of their own (64 K
    slots, three quarters of them empty)."""
    from cascading_kv_cache_amd.cascade_attention import cascade_attention, default_inv_freq

    H = KVH = 8
    tokens, q_len = 16384, 2240
    inv_freq = default_inv_freq(D, 5e5, "cuda:0")
    gen = torch.Generator(device="cuda").manual_seed(2)
    rows = lambda n: torch.randn(1, n, H, D, generator=gen, device="cuda").to(dtype).transpose(1, 2)   # noqa: E731
    k0, v0, k, v = rows(tokens), rows(tokens), rows(q_len), rows(q_len)
    caches = []
    for slots in (tokens, 4 * tokens):
        cache = make_pair(1, KVH, D, 0, slots, 1, dtype)[0]
        cache.beta = 0.5   # scores of the last few rows: a normaliser's last bit shows
        cache.update(k0, v0, 0, torch.zeros(1, KVH, tokens, dtype=dtype, device="cuda"))
        caches.append(cache)
    for _ in range(4):
        q, got = rows(q_len), []
        for cache in caches:
            out, new = cascade_attention(q, k, v, cache, 0, inv_freq, update_cache=False)
            got.append((out, new, cache.score_cache[0][..., :tokens]))
        for a, b in zip(*got):
            assert torch.equal(a, b), (a != b).sum()
