"""Eager steps planned in the binding: over quantised pools, the refusals and host counts of the checked
path; attention calls that must fall back to it; copies of a pool that has stepped."""

import copy
import types

import numpy as np
import pytest
import torch

from attn_ref import decode_attention_reference, within_tolerance
from kvgen import hf_layout, to_bits
from oracle.kv_quant_oracle import QuantLayerOracle

from barqtrain_amd.kv_cache import BarqPagedKVCacheLayer, create_paged_kv_cache
from barqtrain_amd.paged import PagedKVCapacityError, PagedKVPoolExhausted, PagePool, QuantPagePool

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def kv(b, H, t, D, gen):
    return hf_layout(b, H, t, D, BF16, gen), hf_layout(b, H, t, D, BF16, gen)


def test_quantised_steps_match_the_oracle_and_refuse_like_the_checked_path(hip):
    H, D, P, W = 2, 128, 16, 16
    gen = torch.Generator().manual_seed(2)
    pool = QuantPagePool(max_batch=3, max_blocks=6, page_size=P, kv_heads=H, head_dim=D, dtype=BF16, device="cuda",
                         window=W, num_pages=12, num_cold=9)
    oracle = QuantLayerOracle(3, 96, P, W, "bf16")
    for b, t in ((3, 20), (2, 1), (3, 14), (1, 33), (3, 1)):
        k, v = kv(b, H, t, D, gen)
        got = pool.update(k.cuda(), v.cuda())
        for g, w in zip(got, oracle.update(to_bits(k), to_bits(v))):
            assert np.array_equal(to_bits(g), w), (b, t)
        assert pool.lens.tolist() == pool.seq_lens.tolist() and pool.hw.tolist() == pool.high_water.tolist()
        assert pool.free_count == int(pool.ctrl[0]) and pool.cold_free == int(pool.ctrl[2])
    k, v = kv(3, H, 2, D, gen)
    pool.append(k.cuda(), v.cuda())
    oracle.append(to_bits(k), to_bits(v))
    assert np.array_equal(to_bits(pool.gather(3)[0]), oracle.current_tensors()[0])
    state = (pool.lens.tolist(), pool.free_count, pool.cold_free, pool.cold_blocks.tolist())
    one = torch.zeros((1, H, 1, D), dtype=BF16, device="cuda")
    many = torch.zeros((3, H, 20, D), dtype=BF16, device="cuda")
    with pytest.raises(PagedKVCapacityError):
        pool.update(one, one, max_length=int(pool.lens[0]))
    pool.cold_free, cold_free = 0, pool.cold_free
    with pytest.raises(PagedKVPoolExhausted):
        pool.update(many[:1], many[:1])
    pool.cold_free = cold_free
    pool.free_count, free = 0, pool.free_count
    with pytest.raises(PagedKVPoolExhausted):
        pool.append(many[1:], many[1:])
    pool.free_count = free
    with pytest.raises(RuntimeError):
        pool.update(one.float(), one.float())
    with pytest.raises(ValueError):
        pool.append(torch.zeros((4, H, 1, D), dtype=BF16, device="cuda"), torch.zeros((4, H, 1, D), dtype=BF16, device="cuda"))
    assert state == (pool.lens.tolist(), pool.free_count, pool.cold_free, pool.cold_blocks.tolist())
    assert pool.errors() == 0


@pytest.mark.parametrize("quant", [False, True])
def test_a_copied_pool_steps_on_its_own_tensors(hip, quant):
    H, D = 2, 64
    gen = torch.Generator().manual_seed(3)
    geometry = dict(max_batch=2, max_blocks=4, page_size=16, kv_heads=H, head_dim=D, dtype=BF16, device="cuda")
    pool = QuantPagePool(window=16, **geometry) if quant else PagePool(**geometry)
    k, v = (x.cuda() for x in kv(2, H, 30, D, gen))
    first = [x.clone() for x in pool.update(k, v)]
    q = torch.randn((2, 4, 1, D), device="cuda").to(BF16)
    before = pool.attend(q).clone()
    other = copy.deepcopy(pool)
    other.update(*(x.cuda() for x in kv(2, H, 3, D, gen)))
    assert pool.lens.tolist() == [30, 30] and other.lens.tolist() == [33, 33]
    for a, b in zip(first, pool.gather(2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(before, pool.attend(q)) and not torch.equal(before, other.attend(q))


def test_attention_steps_and_their_fallbacks_agree(hip):
    """A strided query (copied first), a workspace too small for the call, explicit arguments."""
    H, D, G = 2, 128, 4
    gen = torch.Generator().manual_seed(4)
    pool = PagePool(max_batch=2, max_blocks=80, page_size=16, kv_heads=H, head_dim=D, dtype=BF16, device="cuda")
    k, v = kv(2, H, 1200, D, gen)
    pool.append(k[:, :, :40].cuda(), v[:, :, :40].cuda())
    for n in (40, 1200):
        if n > 40:
            pool.append(k[:, :, 40:].cuda(), v[:, :, 40:].cuda())  # the workspace grows
        q = torch.randn((2, H * G, 1, 2 * D), generator=gen).to(BF16).cuda()[..., ::2]
        outs = [pool.attend(q), pool.attend(q.contiguous()), pool.attend(q, max_seq=n), pool.attend(q, D ** -0.5)]
        want = decode_attention_reference(q.cpu().float().numpy(), k[:, :, :n].float().numpy(),
                                          v[:, :, :n].float().numpy(), [n, n], D ** -0.5)
        for out in outs:
            assert out.shape == q.shape and torch.equal(out, outs[0])
            # one rounding to bf16 of sums within 2e-5
            assert within_tolerance(out.cpu().double().numpy(), want, 2.0 ** -8 + 2e-5, 2e-5)[0]


def test_overridden_methods_of_layers_and_pools_are_called(hip):
    """A layer's append (fused attention), a pool's update, append, crop and reset."""
    calls = []

    def counting(cls, *names):
        def method(name):
            return lambda self, *a, **kw: calls.append(name) or getattr(cls, name)(self, *a, **kw)
        return type("Counting", (cls,), {name: method(name) for name in names})

    k, v = (x.cuda() for x in kv(1, 2, 3, 64, torch.Generator().manual_seed(4)))
    sub = counting(BarqPagedKVCacheLayer, "append")(max_batch_size=1, max_cache_len=32, fused_attention=True)
    sub.update(k, v)
    sub.update(k, v)
    assert calls == ["append"] * 2 and sub.get_seq_length() == 6
    layer = BarqPagedKVCacheLayer(max_batch_size=1, max_cache_len=32, fused_attention=True)
    layer.update(k, v)
    layer.append = lambda *a: calls.append("replaced") or type(layer).append(layer, *a)
    layer.update(k, v)
    assert calls[2:] == ["replaced"] and layer.get_seq_length() == 6
    for pool_type in (PagePool, QuantPagePool):
        cache = create_paged_kv_cache(types.SimpleNamespace(num_hidden_layers=2), max_batch_size=1, max_cache_len=64)
        for l in range(2):
            cache.update(k, v, l)
            cache.layers[l].pool = counting(pool_type, "append", "update", "crop", "reset")(
                max_batch=1, max_blocks=4, page_size=16, kv_heads=2, head_dim=64, dtype=BF16, device="cuda")
        calls.clear()
        for l, fused in enumerate((False, True)):
            cache.layers[l].fused_attention = fused
            cache.update(k, v, l)
        cache.crop(1)
        cache.reset()
        assert [c for c in calls if c != "reset"] == ["update", "append", "crop", "crop"] and calls[-2:] == ["reset"] * 2
