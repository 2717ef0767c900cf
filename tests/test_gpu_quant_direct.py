"""Appends that quantise past the residual window straight from the input (BARQ_KV_QUANT_DIRECT, and
QuantPagePool's appends longer than its chunk): bit for bit what the quantisation oracle reads, over
every width of the kernel's per-head units, with rows that start mid-block, were cropped or hold
non-finite values."""

import numpy as np
import pytest
import torch

from kvgen import hf_layout, to_bits
from oracle import kv_quant_oracle as q
from test_gpu_quant import DT, assert_same

from barqtrain_amd import _capi
from capi_pool import CColdPool

pytestmark = pytest.mark.gpu
DIRECT = 8

# dtype, kv heads, head_dim, page, window: 1, 2, 4 and 8 vectors a lane; 2-byte and fp32; odd heads; window 0
CASES = [
    (torch.bfloat16, 8, 64, 8, 40),
    (torch.bfloat16, 2, 64, 16, 0),
    (torch.bfloat16, 8, 128, 16, 32),
    (torch.float16, 5, 128, 16, 24),
    (torch.float16, 4, 128, 32, 48),
    (torch.bfloat16, 3, 256, 16, 16),
    (torch.float32, 4, 64, 16, 24),
    (torch.float32, 17, 16, 16, 20),
]


def states(b, H, t, D, dtype, gen):
    k, v = hf_layout(b, H, t, D, dtype, gen) * 4, hf_layout(b, H, t, D, dtype, gen)
    k[0, 0, t // 2, 3], v[-1, -1, t // 3, 5] = float("inf"), float("nan")
    v[0, 0, 0, 0] = -float("inf")
    return k, v


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{DT[c[0]]}-h{c[1]}d{c[2]}p{c[3]}w{c[4]}")
def test_direct_appends_match_the_oracle(capi, case):
    dtype, H, D, P, W = case
    Bmax, cap = 3, 20 * P
    rng = np.random.default_rng(P * H)
    gen = torch.Generator().manual_seed(H)
    pool = CColdPool(window=W, max_batch=Bmax, max_blocks=20, page_size=P, heads=H, dim=D, dtype=dtype)
    oracle = q.QuantLayerOracle(Bmax, cap, P, W, DT[dtype])
    for it in range(40):
        r = rng.random()
        n = oracle.current_batch_size if oracle.is_initialized else 0
        if r < 0.6 or not n:
            b = int(rng.integers(1, (oracle.max_batch_size if oracle.is_initialized else Bmax) + 1))
            t = int(rng.choice([1, 2, P - 1, P, P + 1, 3 * P, 7 * P + 3]))
            if oracle.is_initialized and int(oracle.seq_lens[:b].max()) + t > cap:
                pool.free_rows(list(range(b)))
                oracle.release_rows(list(range(b)))
            k, v = states(b, H, t, D, dtype, gen)
            oracle.append(to_bits(k), to_bits(v))
            got = pool.update(k.cuda(), v.cuda(), oracle.get_seq_length(), DIRECT)
            ok, ov = oracle.current_tensors()
            assert np.array_equal(to_bits(got[0]), ok) and np.array_equal(to_bits(got[1]), ov), f"update it{it} t{t}"
        elif r < 0.8:
            m = int(rng.integers(0, cap))
            pool.crop(n, m)
            oracle.crop(m)
        else:
            rows = rng.integers(0, n, size=int(rng.integers(1, Bmax + 1))).tolist()
            pool.select_rows(rows)
            oracle.batch_select_indices(rows)
        assert_same(pool, oracle, f"it{it}")
        pool.check_invariants()
    assert pool.errors() == 0


@pytest.mark.parametrize("num_cold,num_pages", [(9, 16), (40, 5)])
def test_direct_append_without_room_changes_nothing(capi, num_cold, num_pages):
    H, D, P, W = 4, 128, 16, 32
    gen = torch.Generator().manual_seed(1)
    pool = CColdPool(window=W, max_batch=2, max_blocks=12, page_size=P, heads=H, dim=D, dtype=torch.bfloat16,
                     num_pages=num_pages, num_cold=num_cold)
    k, v = (x.cuda() for x in states(2, H, 7 * P, D, torch.bfloat16, gen))  # 2 x (5 cold + 2 hot blocks); 9 or 40 cold
    if num_pages == 5:  # 2 hot blocks a row fit 5 pages, 3 do not
        pool.update(k, v, 7 * P, DIRECT)
        assert pool.errors() == 0
        k, v = (x.cuda() for x in states(2, H, 3 * P + 1, D, torch.bfloat16, gen))
    before = [t.clone() for t in (pool.bt, pool.lens, pool.hw, pool.ctrl[:3])]
    seq = int(pool.lens.max()) or P
    kept = [x.clone() for x in pool.gather(2, seq)]
    pool.update(k, v, seq, DIRECT)
    assert pool.errors() & 1
    pool.ctrl[1] = 0
    for a, b in zip(before, (pool.bt, pool.lens, pool.hw, pool.ctrl[:3])):
        assert torch.equal(a, b)
    for a, b in zip(kept, pool.gather(2, seq)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_direct_append_refuses_other_geometry(capi):
    pool = CColdPool(window=8, max_batch=1, max_blocks=8, page_size=5, heads=2, dim=128, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 20, 128, dtype=torch.bfloat16, device="cuda")
    rc = pool.lib.barq_kv_update_cold(pool.ref, pool.cref, k.data_ptr(), k.data_ptr(), 1, 20, k.stride(0), k.stride(1),
                                      k.stride(2), None, None, 0, 0, 0, 0, DIRECT, pool._stream())
    assert rc == 4 and "no kernel" in _capi.load_library().barq_kv_status_string(rc).decode()
    assert int(pool.lens.max()) == 0


@pytest.mark.parametrize("tokens", [65, 64 + 128, 301])
@pytest.mark.parametrize("strided", [False, True])
def test_long_appends_equal_chunked_ones(capi, tokens, strided):
    """QuantPagePool.append / append_rows past the chunk: K and V as the chunked appends (chunk =
    the capacity: append, then compress) leave them, and the host's counts equal the device's."""
    from barqtrain_amd.paged import QuantPagePool

    H, D, P, B, cap = 4, 128, 16, 3, 640
    gen = torch.Generator().manual_seed(tokens)
    geometry = dict(max_batch=B, max_blocks=cap // P, page_size=P, kv_heads=H, head_dim=D, dtype=torch.bfloat16,
                    device="cuda", window=96)
    direct = QuantPagePool(chunk=64, **geometry)
    whole = QuantPagePool(chunk=cap, num_pages=B * (cap // P + 1), **geometry)
    for start, t, crop in ((0, 7, None), (0, tokens, 40), (1, tokens, None)):
        k, v = (x.cuda() for x in states(B, H, t, D, torch.bfloat16, gen))
        if strided:  # [B, H, T, D] in memory
            k, v = k.contiguous(), v.contiguous()
        for pool in (direct, whole):
            pool.append(k, v) if start == 0 else pool.append_rows([2, 0], k[:2], v[:2])
            if crop is not None:
                pool.crop(2, crop)
        for a, b in zip(direct.gather(B), whole.gather(B)):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))
        for pool in (direct, whole):
            assert pool.errors() == 0
            assert int(pool.ctrl[0]) == pool.free_count and int(pool.ctrl[2]) == pool.cold_free
            assert pool.seq_lens.tolist() == pool.lens.tolist() and pool.high_water.tolist() == pool.hw.tolist()
        assert direct.lens.tolist() == whole.lens.tolist() and direct.cold_blocks.tolist() == whole.cold_blocks.tolist()
