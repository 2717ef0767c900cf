"""Appends whose row state comes from the host's exact shadow: on twin pools, one of which forgets that
its free count is exact (and so takes the device-read appends, one launch a row for append_rows), the
same block tables, lengths, marks, stack tops and bits."""

import numpy as np
import pytest
import torch

from kvgen import hf_layout

from barqtrain_amd.paged import PagePool

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,D,P,dtype,rows", [(8, 128, 16, torch.bfloat16, 5), (2, 64, 16, torch.float16, 64),
                                              (5, 80, 5, torch.bfloat16, 3), (1, 16, 1, torch.float32, 7),
                                              (16, 128, 32, torch.float32, 2), (3, 20, 4, torch.bfloat16, 3)])
def test_known_appends_match_device_reads(hip, H, D, P, dtype, rows):
    """hv 128, 16, 50, 4, 512 (two positions a tile) and rows 16-byte vectors do not fit (device reads both)."""
    rng = np.random.default_rng(H * D)
    gen = torch.Generator().manual_seed(P)
    blocks = 40
    order = torch.from_numpy(rng.permutation(rows * blocks).astype(np.int32))
    known, plain = (PagePool(max_batch=rows, max_blocks=blocks, page_size=P, kv_heads=H, head_dim=D, dtype=dtype,
                             device="cuda", num_pages=rows * blocks, page_order=order) for _ in range(2))
    for step in range(24):
        t = int(rng.choice([1, 1, 2, P, 9 * P + 1]))
        picked = rng.permutation(rows)[: int(rng.integers(1, rows + 1))].tolist()
        by_rows = step % 3 == 2
        if not by_rows:
            picked = list(range(len(picked)))
        if int(known.lens[picked].max()) + t > known.capacity:
            for pool in (known, plain):
                pool.free_rows(picked[:2])
                pool.crop(rows, known.capacity // 3)  # stale pages below the marks stay mapped
                pool.free_exact = True
            t = 1
        k, v = (hf_layout(len(picked), H, t, D, dtype, gen).cuda() for _ in range(2))
        for pool in (known, plain):
            pool.free_exact = pool is known
            pool.append_rows(picked, k, v) if by_rows else pool.append(k, v)
            assert pool.free_count == int(pool.ctrl[0])
        for name in ("block_table", "seq_lens", "high_water"):
            assert torch.equal(getattr(known, name), getattr(plain, name)), (step, name)
        assert known.seq_lens.tolist() == known.lens.tolist() and known.high_water.tolist() == known.hw.tolist()
        for a, b in zip(known.gather(rows), plain.gather(rows)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), step
    assert known.errors() == plain.errors() == 0


def test_captured_appends_follow_the_device_state(hip):
    """A graph's append (and append_rows) stores at the rows' lengths of each replay."""
    gen = torch.Generator().manual_seed(9)
    make = lambda: PagePool(max_batch=3, max_blocks=8, page_size=4, kv_heads=2, head_dim=64, dtype=torch.bfloat16,
                            device="cuda")
    pool, eager = make(), make()
    k, v = (hf_layout(3, 2, 1, 64, torch.bfloat16, gen).cuda() for _ in range(2))

    def step(p):
        p.append(k, v)
        p.append_rows([2, 0], k[:2], v[:2])

    for p in (pool, eager):
        step(p)
    state = [(a.copy(), a) for a in (pool.lens, pool.hw)], pool.free_count
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(pool)
    for copy, a in state[0]:  # nothing of the recording has run
        a[:] = copy
    pool.free_count = state[1]
    for it in range(5):
        k.copy_(hf_layout(3, 2, 1, 64, torch.bfloat16, gen))
        v.copy_(hf_layout(3, 2, 1, 64, torch.bfloat16, gen))
        graph.replay()
        step(eager)
        torch.cuda.synchronize()
        for name in ("block_table", "seq_lens", "high_water"):
            assert torch.equal(getattr(pool, name), getattr(eager, name)), (it, name)
        for a, b in zip(pool.gather(3, int(eager.lens.max())), eager.gather(3)):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)), it
    assert pool.errors() == eager.errors() == 0
