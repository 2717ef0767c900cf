"""Prompts into empty rows of a pool with fp8 pages, quantised and returned by one launch: beside a pool
whose chunk holds the prompt (append, compress, gather), the same bits, tables' meaning and counts."""

import numpy as np
import pytest
import torch

from kvgen import hf_layout

from barqtrain_amd.paged import QuantPagePool

pytestmark = pytest.mark.gpu

# dtype, kv heads, head_dim, page, window: 1, 2, 4 and 8 vectors a lane, head counts that leave part of a
# workgroup idle, window 0, and a geometry the kernel does not take
CASES = [
    (torch.bfloat16, 8, 64, 8, 40),
    (torch.bfloat16, 2, 64, 16, 0),
    (torch.bfloat16, 8, 128, 16, 32),
    (torch.float16, 5, 128, 16, 24),
    (torch.float16, 4, 128, 32, 48),
    (torch.bfloat16, 3, 256, 16, 16),
    (torch.float32, 4, 64, 16, 24),
    (torch.float32, 17, 16, 16, 20),
    (torch.bfloat16, 2, 128, 5, 8),
]


def states(b, H, t, D, dtype, gen):
    k, v = hf_layout(b, H, t, D, dtype, gen) * 4, hf_layout(b, H, t, D, dtype, gen)
    k[0, 0, t // 2, 3], v[-1, -1, t // 3, 5] = float("inf"), float("nan")
    v[0, 0, 0, 0], k[0, -1, :, 7] = -float("inf"), -0.0
    k[-1, 0, :, 2] *= 2.0 ** -90 if dtype != torch.float16 else 0  # scales the hardware decode does not take
    return k.cuda(), v.cuda()


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-h{c[1]}d{c[2]}p{c[3]}w{c[4]}")
@pytest.mark.parametrize("strided", [False, True])
def test_prompts_into_empty_rows(hip, case, strided):
    dtype, H, D, P, W = case
    B, blocks, chunk = 3, 12, 6
    gen = torch.Generator().manual_seed(D)
    rng = np.random.default_rng(P)
    cap = blocks * P
    num_pages = B * (blocks + 1)
    order = torch.from_numpy(rng.permutation(num_pages).astype(np.int32))
    geometry = dict(max_batch=B, max_blocks=blocks, page_size=P, kv_heads=H, head_dim=D, dtype=dtype, device="cuda",
                    window=W, num_pages=num_pages)
    one = QuantPagePool(chunk=chunk, page_order=order, **geometry)
    whole = QuantPagePool(chunk=cap, **geometry)
    bits = lambda x: x.contiguous().view(torch.uint8)

    def check(what, pair=None):
        for a, b in zip(*(pair or (one.gather(B), whole.gather(B)))):
            assert torch.equal(bits(a), bits(b)), what
        for pool in (one, whole):
            assert pool.errors() == 0
            assert int(pool.ctrl[0]) == pool.free_count and int(pool.ctrl[2]) == pool.cold_free
            assert pool.seq_lens.tolist() == pool.lens.tolist() and pool.high_water.tolist() == pool.hw.tolist()
        assert one.cold_blocks.tolist() == whole.cold_blocks.tolist()

    for t in (chunk + 1, W + 1, W + P, W + P + 1, 8 * P, 11 * P + P // 2 + 1):
        if t <= chunk or t > cap:
            continue
        for batch in (B, 1):
            k, v = states(batch, H, t, D, dtype, gen)
            if strided:  # [B, H, T, D] in memory
                k, v = k.contiguous(), v.contiguous()
            for pool in (one, whole):
                pool.reset()
            check(f"update {t}", (one.update(k, v), whole.update(k, v)))
            check(f"after {t}")
            if t + 1 <= cap:  # the rows go on from what the launch left
                k, v = states(batch, H, 1, D, dtype, gen)
                check(f"step {t}", (one.update(k, v), whole.update(k, v)))
        for pool in (one, whole):  # no output, rows between others
            pool.reset()
        k, v = states(B, H, t, D, dtype, gen)
        for pool in (one, whole):
            pool.append(k, v)
            pool.free_rows([1])
            pool.append_rows([1], k[2:], v[:1])
        check(f"rows {t}")
