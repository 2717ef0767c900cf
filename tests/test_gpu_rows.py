"""Gathers and updates of token rows that are not whole runs of 64 sixteen-byte vectors (2 KV heads x
64, odd head counts): every count of wave loads a page and of slots a wave, known and device-read
row state, ragged rows, stale positions after a crop, long appends; bit for bit against the oracle
or the device mirror."""

import numpy as np
import pytest
import torch

from capi_pool import SEQ_FROM_DEVICE, CPool
from kvgen import hf_layout, to_bits
from mirror import DeviceMirror
from oracle.kv_oracle import DenseLayerOracle
from test_gpu_known import step_both

pytestmark = pytest.mark.gpu

# heads, dim, page, dtype: hv 16 (4 loads a page), 8 (1), 80 (20, not a divisor of 64), 48 (12), 4 (1), 192 (48)
SHAPES = [
    (2, 64, 16, torch.bfloat16),
    (1, 64, 8, torch.float16),
    (5, 128, 16, torch.bfloat16),
    (3, 64, 16, torch.float32),
    (1, 16, 16, torch.float32),
    (6, 256, 16, torch.bfloat16),
]


def same(got, oracle, what):
    ok, ov = oracle.current_tensors()
    for g, w in zip(got, (ok, ov)):
        assert np.array_equal(to_bits(g), w[:, :, :g.shape[2]]), what


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"h{s[0]}d{s[1]}p{s[2]}{str(s[3])[6:]}")
def test_ragged_programs_match_the_oracle(capi, shape):
    H, D, P, dtype = shape
    rng = np.random.default_rng(H * D)
    Bmax, cap = 5, 12 * P
    gen = torch.Generator().manual_seed(H)
    perm = torch.from_numpy(rng.permutation(Bmax * 12 + 1).astype(np.int32))
    pool = CPool(max_batch=Bmax, max_blocks=12, page_size=P, heads=H, dim=D, dtype=dtype, num_pages=Bmax * 12 + 1, order=perm)
    oracle = DenseLayerOracle(Bmax, cap, P)
    for it in range(50):
        b = int(rng.integers(1, Bmax + 1))
        t = int(rng.choice([1, 1, 2, P, 3 * P + 1]))
        if oracle.is_initialized and int(oracle.seq_lens[:b].max()) + t > cap:
            m = int(rng.integers(0, cap // 2))
            pool.crop(Bmax, m)  # stale positions stay readable up to the mark
            oracle.current_batch_size = Bmax
            oracle.crop(m)
            seq = max(oracle.get_seq_length(), 1)
            same(pool.gather(Bmax, seq, SEQ_FROM_DEVICE if it % 2 else 0), oracle, f"crop it{it}")
            continue
        k, v = hf_layout(b, H, t, D, dtype, gen), hf_layout(b, H, t, D, dtype, gen)
        oracle.append(to_bits(k), to_bits(v))
        seq = oracle.get_seq_length()
        got = pool.update(k.cuda(), v.cuda(), seq if it % 3 else min(seq + P, cap), 0 if it % 3 else SEQ_FROM_DEVICE)
        same([x[:, :, :seq] for x in got], oracle, f"update it{it}")
    assert pool.errors() == 0
    pool.check_invariants()


@pytest.mark.parametrize("shape", SHAPES[:4], ids=lambda s: f"h{s[0]}d{s[1]}p{s[2]}{str(s[3])[6:]}")
def test_known_state_matches_device_reads(capi, shape):
    H, D, P, dtype = shape
    gen = torch.Generator().manual_seed(D)
    pools = [CPool(max_batch=3, max_blocks=40, page_size=P, heads=H, dim=D, dtype=dtype) for _ in range(2)]
    seq = 0
    for b, t in ((3, 5), (2, 1), (3, P), (1, 2 * P + 1), (3, 9 * P), (3, 1), (3, 1)):
        k, v = hf_layout(b, H, t, D, dtype, gen).cuda(), hf_layout(b, H, t, D, dtype, gen).cuda()
        seq = int(pools[0].lens[:b].max()) + t
        step_both(capi, *pools, k, v, seq)
    assert seq > 12 * P


@pytest.mark.parametrize("batch,prompt", [(24, 1000), (64, 2001), (1, 30000)])
def test_many_tiles(capi, batch, prompt):
    """3, 8 (several rounds) and 4 slots a wave."""
    H, D, P, dtype = 2, 64, 16, torch.bfloat16
    blocks = prompt // P + 3
    pool = CPool(max_batch=batch, max_blocks=blocks, page_size=P, heads=H, dim=D, dtype=dtype)
    mirror = DeviceMirror(batch, H, blocks * P, D, dtype)
    gen = torch.Generator(device="cuda").manual_seed(batch)
    for b, t in ((batch, prompt), (max(batch // 2, 1), 2), (batch, 1), (batch, 17)):
        k, v = (torch.randn((b, t, H, D), generator=gen, device="cuda").to(dtype).transpose(1, 2) for _ in range(2))
        mirror.append(k, v)
        mirror.check(pool.update(k, v, int(mirror.lens[:b].max())), f"{b} x {t}")
    assert pool.errors() == 0
