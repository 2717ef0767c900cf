"""The dequantising update against the dequantising gather of the same pool (checked against the oracle
elsewhere): what a step returns is what is read afterwards, bit for bit, over batch sizes and lengths
on both sides of the resident tiles, ragged and cropped rows, several new tokens, extreme pages, with
known, device-read and captured row state."""

import numpy as np
import pytest
import torch

from barqtrain_amd.graph import CapturedDecodeStep
from barqtrain_amd.paged import QuantPagePool

pytestmark = pytest.mark.gpu


def states(gen, b, t, H, D, dtype):
    k, v = (torch.randn((b, t, H, D), generator=gen, device="cuda") for _ in range(2))
    k[..., ::8] *= 8
    k[0, t // 2, 0, 1] = float("nan")
    v[0, 0, -1, 3] = float("inf")
    if dtype == torch.bfloat16:
        k[:, :, 0] *= 2.0 ** -100
        v[-1, :, -1] *= 2.0 ** 100
    return (x.to(dtype).transpose(1, 2) for x in (k, v))


def same(a, b, what):
    for x, y in zip(a, b):
        assert torch.equal(x.view(torch.int16), y[:, :, :x.shape[2]].view(torch.int16)), what


# 64, 128 and 256 vectors a row; pages of 16, 32 and 8
@pytest.mark.parametrize("H,D,P,dtype", [(8, 64, 16, torch.bfloat16), (8, 128, 16, torch.bfloat16), (8, 128, 32, torch.float16),
                                         (8, 256, 16, torch.bfloat16), (4, 256, 8, torch.float16)])
@pytest.mark.parametrize("B,prompt", [(1, 5), (1, 700), (7, 333), (16, 645), (64, 130), (40, 1300)])
def test_updates_return_what_the_gather_reads(hip, H, D, P, dtype, B, prompt):
    gen = torch.Generator(device="cuda").manual_seed(B * H)
    pool = QuantPagePool(max_batch=B, max_blocks=-(-(prompt + 90) // P), page_size=P, kv_heads=H, head_dim=D, dtype=dtype,
                         device="cuda", window=48)
    pool.append(*states(gen, B, prompt, H, D, dtype))
    for step, (b, t) in enumerate(((B, 1), (max(B // 2, 1), 3), (B, 1), (B, 17), (1, 40), (B, 1))):
        pool.free_exact = step % 2 == 0  # else the device's row state
        free = pool.free_count
        got = pool.update(*states(gen, b, t, H, D, dtype))
        same(got, pool.gather(b), (step, b, t))
        assert pool.seq_lens.tolist() == pool.lens.tolist() and pool.high_water.tolist() == pool.hw.tolist()
        assert int(pool.ctrl[0]) == pool.free_count and int(pool.ctrl[2]) == pool.cold_free, free
        if step == 3:
            pool.crop(B, int(pool.lens.max()) - 9)  # stale positions past the new lengths stay readable
    assert pool.errors() == 0


def test_captured_steps_return_what_the_gather_reads(hip):
    H, D, P, B, prompt = 8, 128, 16, 16, 600
    gen = torch.Generator(device="cuda").manual_seed(9)
    pools = [QuantPagePool(max_batch=B, max_blocks=48, page_size=P, kv_heads=H, head_dim=D, dtype=torch.bfloat16,
                           device="cuda", window=64) for _ in range(2)]
    for pool in pools:
        pool.append(*states(gen, B, prompt, H, D, torch.bfloat16))
        pool.append(*states(gen, 5, 3, H, D, torch.bfloat16))  # ragged rows
    step = CapturedDecodeStep(pools, B)
    for it in range(40):  # crosses blocks, buckets and quantisations
        for i in range(2):
            k, v = states(gen, B, 1, H, D, torch.bfloat16)
            step.key_in[i].copy_(k)
            step.value_in[i].copy_(v)
        for pool, got in zip(pools, step.replay()):
            same(got, pool.gather(B), it)
    assert all(pool.errors() == 0 for pool in pools)
