"""Pool calls recorded into a graph act on the device's row state of each replay, whatever the host's
shadow said when they were recorded: every replay is compared with a twin pool that makes the same
calls eagerly -- lengths, marks, stack tops and the bits that a gather reads."""

import types

import pytest
import torch

from kvgen import hf_layout

from barqtrain_amd.kv_cache import create_paged_kv_cache
from barqtrain_amd.paged import SEQ_FROM_DEVICE, PagePool, QuantPagePool

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
SHADOW = ("lens", "hw", "cold_blocks", "free_count", "free_exact", "cold_free", "cold_exact")


def take_shadow(dst, src):
    """dst's host shadow becomes src's (a replay does not advance it)."""
    for name in SHADOW:
        if hasattr(src, name):
            value = getattr(src, name)
            if hasattr(value, "copy"):
                getattr(dst, name)[:] = value
            else:
                setattr(dst, name, value)


def record(pools, eager, call):
    """A graph of `call`, of which nothing has run."""
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for pool, twin in zip(pools, eager):
        take_shadow(pool, twin)
    return graph


def same(pool, eager, batch, what):
    for name in ("seq_lens", "high_water"):
        assert torch.equal(getattr(pool, name), getattr(eager, name)), (what, name)
    assert pool.ctrl[[0, 2]].tolist() == eager.ctrl[[0, 2]].tolist(), what
    if int(eager.lens.max()):
        for a, b in zip(pool.gather(batch, int(eager.lens.max())), eager.gather(batch)):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), what
    assert pool.errors() == eager.errors() == 0, what


def quant_pool(B, window=32, **kw):
    geometry = dict(max_batch=B, max_blocks=16, page_size=16, kv_heads=2, head_dim=64, dtype=BF16, device="cuda")
    return QuantPagePool(window=window, **{**geometry, **kw})


def states(gen, B, T, H=2, D=64):
    return tuple(hf_layout(B, H, T, D, BF16, gen).cuda() for _ in range(2))


def test_recorded_fp8_appends_quantise_on_replay(hip):
    """Recorded where no block leaves the window; the replays cross several pages."""
    B, gen = 3, torch.Generator().manual_seed(1)
    pool, eager = quant_pool(B), quant_pool(B)
    k, v = states(gen, B, 1)
    first, some = states(gen, B, 34), states(gen, 1, 9)
    for p in (pool, eager):
        p.append(k, v)
        p.append(*first)
        p.append(*some)  # ragged rows
    assert int(eager._cold_after(B, 1)[1]) == 0
    graph = record([pool], [eager], lambda: pool.append(k, v))
    for it in range(120):
        for x, new in zip((k, v), states(gen, B, 1)):
            x.copy_(new)
        graph.replay()
        eager.append(k, v)
        if it % 7 == 0:
            take_shadow(pool, eager)
            same(pool, eager, B, it)
    assert int(eager.cold_blocks.min()) > 4


@pytest.mark.parametrize("out", [False, True])
def test_recorded_fp8_updates_quantise_on_replay(hip, out):
    """Recorded where no block leaves the window, then replayed over rows cropped below that length."""
    B, gen = 3, torch.Generator().manual_seed(2)
    pool, eager = quant_pool(B), quant_pool(B)
    k, v = states(gen, B, 1)
    first, some = states(gen, B, 100), states(gen, 1, 9)
    for p in (pool, eager):
        p.append(k, v)
        p.append(*first)
    assert int(eager._cold_after(B, 1)[1]) == 0
    buffers = pool._new_out(B, pool.capacity)
    got = []

    def call():
        got[:] = pool.update(k, v, out=buffers, seq_out=pool.capacity, flags=SEQ_FROM_DEVICE) if out else pool.update(k, v)

    graph = record([pool], [eager], call)
    for p in (pool, eager):
        p.crop(B, 34)
        p.append(*some)
    for it in range(50):
        for x, new in zip((k, v), states(gen, B, 1)):
            x.copy_(new)
        graph.replay()
        for a, b in zip(got, eager.update(k, v)):
            assert torch.equal(a[:, :, :b.shape[2]].view(torch.int16), b.view(torch.int16)), it
        if it % 7 == 0:
            take_shadow(pool, eager)
            same(pool, eager, B, it)
    assert int(eager.cold_blocks.min()) > 2


# 16 and 80 vectors a row (the rows kernel), 128: resident at once, and one-page tiles of several rounds
@pytest.mark.parametrize("H,D,B,length", [(2, 64, 3, 60), (5, 128, 3, 60), (8, 128, 3, 60), (8, 128, 64, 200)])
def test_recorded_updates_follow_the_device_state(hip, H, D, B, length):
    gen = torch.Generator().manual_seed(H * B)
    make = lambda: PagePool(max_batch=B, max_blocks=16, page_size=16, kv_heads=H, head_dim=D, dtype=BF16, device="cuda")
    pool, eager = make(), make()
    k, v = states(gen, B, 1, H, D)
    first, some = states(gen, B, length, H, D), states(gen, 2, 5, H, D)
    for p in (pool, eager):
        p.append(*first)
    got = []
    graph = record([pool], [eager], lambda: got.extend(pool.update(k, v)))
    for p in (pool, eager):
        p.free_rows([1])
        p.crop(B, length // 2)
        p.append_rows([0, 2], *some)
    for it in range(6):
        for x, new in zip((k, v), states(gen, B, 1, H, D)):
            x.copy_(new)
        graph.replay()
        for a, b in zip(got, eager.update(k, v)):
            assert torch.equal(a[:, :, :b.shape[2]].view(torch.int16), b.view(torch.int16)), it
        take_shadow(pool, eager)
        same(pool, eager, B, it)
        assert torch.equal(pool.block_table, eager.block_table)


def test_recorded_fp8_crops_reopen_quantised_blocks(hip):
    """A cache's crop recorded where it re-opens nothing, replayed where quantised blocks lie past it."""
    B, layers, gen = 3, 2, torch.Generator().manual_seed(4)
    caches = [create_paged_kv_cache(types.SimpleNamespace(num_hidden_layers=layers), max_batch_size=B, max_cache_len=240,
                                    page_size=16, kv_quant="fp8", residual_window=32) for _ in range(2)]
    pools, eager = ([], [])
    first, more, one = states(gen, B, 70), states(gen, B, 64), states(gen, B, 1)
    for l in range(layers):
        for cache, group in zip(caches, (pools, eager)):
            cache.update(*first, l)
            group.append(cache.layers[l].pool)
    graph = record(pools, eager, lambda: caches[0].crop(40))
    for it in range(3):
        for l in range(layers):
            for cache in caches:
                cache.update(*more, l)
        assert int(eager[0].cold_blocks.min()) * 16 > 40
        graph.replay()
        caches[1].crop(40)
        for l in range(layers):
            take_shadow(pools[l], eager[l])
            same(pools[l], eager[l], B, it)
            for a, b in zip(caches[0].update(*one, l), caches[1].update(*one, l)):
                assert torch.equal(a.view(torch.int16), b.view(torch.int16)), it
            same(pools[l], eager[l], B, it)


@pytest.mark.parametrize("update", [False, True])
def test_recorded_long_fp8_appends_fit_where_chunks_fit(hip, update):
    """A prompt recorded over empty rows, replayed behind 47 tokens in a pool that holds just what chunks
    need (five pages a row: three hot ones before it, three after it, four during it)."""
    B, gen = 3, torch.Generator().manual_seed(5)
    pool, eager = (quant_pool(B, chunk=16, num_pages=5 * B) for _ in range(2))
    prompt, first = states(gen, B, 64), states(gen, B, 47)
    graph = record([pool], [eager], lambda: pool.update(*prompt) if update else pool.append(*prompt))
    for p in (pool, eager):
        p.append(*first)
    graph.replay()
    eager.append(*prompt)
    take_shadow(pool, eager)
    same(pool, eager, B, update)
    assert eager.lens.tolist() == [111] * B
