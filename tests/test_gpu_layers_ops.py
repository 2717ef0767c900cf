"""Crop and reset of a whole cache: one launch for every layer leaves what a crop or reset of each
layer leaves -- lengths, tables, stacks, control words, host shadows -- over more layers than a
launch holds, with and without cold stores, and falls back where pages must be re-opened."""

import types

import pytest
import torch

from kvgen import hf_layout

from barqtrain_amd import kv_cache
from barqtrain_amd.kv_cache import create_paged_kv_cache
from barqtrain_amd.paged import crop_layers

pytestmark = pytest.mark.gpu
H, D, B, BF16 = 2, 64, 3, torch.bfloat16


def filled(layers, quant, tokens=70):
    cache = create_paged_kv_cache(types.SimpleNamespace(num_hidden_layers=layers), max_batch_size=B, max_cache_len=120,
                                  page_size=16, kv_quant="fp8" if quant else None, residual_window=32)
    gen = torch.Generator().manual_seed(layers)
    for l in range(layers):
        k = hf_layout(B, H, tokens, D, BF16, gen).cuda()
        cache.update(k, k * 2, l)
    return cache


def state(pool):
    out = [pool.block_table, pool.seq_lens, pool.high_water, pool.ctrl, pool.page_shares]
    out = [t.tolist() for t in out] + [pool.free_pages[:pool.free_count].tolist(), pool.lens.tolist(), pool.hw.tolist(),
                                       pool.free_count, pool.free_exact, pool.shared]
    if getattr(pool, "quantized", False):
        out += [pool.free_cold[:pool.cold_free].tolist(), pool.cold_shares.tolist(), pool.cold_blocks.tolist(),
                pool.cold_free, pool.cold_exact]
    return out


@pytest.mark.parametrize("layers", [2, 37])
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("length", [0, 5, 33, 64, 70, 500])  # 5: quantised blocks re-open (their own launches)
def test_cache_crop_is_every_layers_crop(hip, layers, quant, length):
    one, each = filled(layers, quant), filled(layers, quant)
    one.crop(length)
    for layer in each.layers:
        layer.crop(length)
    for a, b in zip(one.layers, each.layers):
        if quant and length < 64:  # re-opened blocks take pages in no fixed order
            assert a.pool.lens.tolist() == b.pool.lens.tolist() and a.pool.cold_blocks.tolist() == b.pool.cold_blocks.tolist()
            assert a.pool.seq_lens.tolist() == b.pool.seq_lens.tolist()
        else:
            same = state(a.pool), state(b.pool)
            if quant:  # cold pages are popped in no fixed order either
                same = [[s[i] for i in (1, 2, 3, 6, 7, 8, 13, 14)] for s in same]
            assert same[0] == same[1]
        for x, y in zip(a.current_tensors(), b.current_tensors()):
            assert torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("layers", [2, 37])
@pytest.mark.parametrize("quant", [False, True])
def test_cache_reset_is_every_layers_reset(hip, layers, quant):
    one, each = filled(layers, quant), filled(layers, quant)
    one.reset()
    for layer in each.layers:
        layer.reset()
    for a, b in zip(one.layers, each.layers):
        assert state(a.pool) == state(b.pool)
        assert a.current_batch_size == b.current_batch_size == 0 and a.get_seq_length() == 0
    k = hf_layout(B, H, 3, D, BF16, torch.Generator().manual_seed(1)).cuda()
    got = one.update(k, k, 1)
    assert torch.equal(got[0], k) and got[0].shape == (B, H, 3, D)


def test_cache_crop_after_a_selection_reopens_shared_pages(hip):
    cache = filled(3, False)
    cache.reorder_cache(torch.tensor([0, 0, 1]))
    want = [[x[:, :, :20].clone() for x in layer.current_tensors()] for layer in cache.layers]
    cache.crop(20)
    k = hf_layout(B, H, 4, D, BF16, torch.Generator().manual_seed(2)).cuda()
    for l, (wk, wv) in enumerate(want):
        gk, gv = cache.update(k, k, l)
        assert torch.equal(gk, torch.cat([wk, k], 2)) and torch.equal(gv, torch.cat([wv, k], 2))
        assert cache.layers[l].pool.errors() == 0


@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("uneven", [False, True])
@pytest.mark.parametrize("count", [-1, -3, -69, -500])
def test_cache_crop_by_a_negative_count_is_every_layers_crop(hip, monkeypatch, quant, uneven, count):
    """Tokens to remove: one launch where the layers hold the same length."""
    one, each = filled(5, quant), filled(5, quant)
    if uneven:
        k = hf_layout(B, H, 2, D, BF16, torch.Generator().manual_seed(3)).cuda()
        one.update(k, k, 2), each.update(k, k, 2)
    together = []
    monkeypatch.setattr(kv_cache, "crop_layers", lambda *a: together.append(a) or crop_layers(*a))
    one.crop(count)
    assert len(together) == (not uneven)
    for layer in each.layers:
        layer.crop(count)
    for a, b in zip(one.layers, each.layers):
        assert a.get_seq_length() == b.get_seq_length() == max(70 + 2 * (uneven and a is one.layers[2]) + count, 0)
        assert a.pool.seq_lens.tolist() == b.pool.seq_lens.tolist() == a.pool.lens.tolist()
        assert a.pool.ctrl[[0, 2]].tolist() == b.pool.ctrl[[0, 2]].tolist()
        for x, y in zip(a.current_tensors(), b.current_tensors()):
            assert torch.equal(x.view(torch.int16), y.view(torch.int16))
