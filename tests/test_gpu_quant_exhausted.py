"""A cold store that runs out: the quantised blocks still lead every row, what is read and attended over is
each block's own contents, and an append that quantises from its input is all or nothing."""

import numpy as np
import pytest
import torch

from attn_ref import decode_attention_reference, within_tolerance
from capi_pool import CColdPool, attend_cold
from kvgen import hf_layout, to_bits
from oracle import kv_quant_oracle as q
from test_gpu_attention import F32_TOL

pytestmark = pytest.mark.gpu
NAMES = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32"}
DIRECT = 8


# blocks of a wave's vectors and of less; rows of more blocks than one pass looks at, than two, than 64
@pytest.mark.parametrize("B,H,D,P,blocks,num_cold,dtype",
                         [(3, 8, 128, 16, 6, 7, torch.bfloat16), (3, 2, 64, 16, 6, 1, torch.float16),
                          (4, 3, 256, 16, 5, 10, torch.bfloat16), (3, 4, 64, 16, 6, 11, torch.float32),
                          (2, 2, 64, 16, 300, 400, torch.bfloat16), (1, 2, 64, 16, 300, 270, torch.float16),
                          (2, 2, 64, 16, 900, 1300, torch.bfloat16), (1, 1, 64, 1, 17000, 16950, torch.bfloat16),
                          (2, 1, 8, 4, 6, 5, torch.float32)])
def test_compress_quantises_the_leading_blocks(capi, B, H, D, P, blocks, num_cold, dtype):
    gen = torch.Generator().manual_seed(num_cold)
    pool = CColdPool(window=0, num_cold=num_cold, max_batch=B, max_blocks=blocks, page_size=P, heads=H, dim=D, dtype=dtype)
    oracle = q.QuantLayerOracle(B, blocks * P, P, 0, NAMES[dtype])
    n = (blocks - 1) * P + min(3, P)
    k, v = hf_layout(B, H, n, D, dtype, gen), hf_layout(B, H, n, D, dtype, gen)
    for calls in range(2):  # the second finds the store empty
        if calls == 0:
            pool.update(k.cuda(), v.cuda(), n)
        else:
            pool.compress(B)
        assert pool.errors() == 1  # POOL_EXHAUSTED
        pool.check_invariants()
        cold = pool.bt.cpu().numpy() <= -2
        assert int(cold.sum()) == num_cold
    oracle.append(to_bits(k), to_bits(v))
    exact, read = (to_bits(k), to_bits(v)), oracle.current_tensors()
    got = pool.gather(B, n)
    mine = np.repeat(cold, P, axis=1)[:, None, :n, None]
    for g, e, w in zip(got, exact, read):
        assert np.array_equal(to_bits(g), np.where(mine, w, e))
    if dtype != torch.float32 and D != 256 and P % 16 == 0:
        query = hf_layout(B, 2 * H, 1, D, dtype, gen)
        out = attend_cold(pool, query.cuda())
        want = decode_attention_reference(*(x.double().cpu().numpy() for x in (query, *got)), [n] * B, D ** -0.5)
        assert within_tolerance(out.cpu().numpy(), want, **F32_TOL)[0]
        assert pool.errors() == 1


@pytest.mark.parametrize("short", [0, 1, 6, 13])
def test_direct_appends_count_the_blocks_that_leave_the_window(capi, short):
    """Three rows of four hot blocks each; six more blocks of tokens push those and two new ones out."""
    B, H, D, P, W = 3, 2, 128, 16, 64
    gen = torch.Generator().manual_seed(short)
    pool = CColdPool(window=W, num_cold=18 - short, max_batch=B, max_blocks=12, page_size=P, heads=H, dim=D,
                     dtype=torch.bfloat16)
    oracle = q.QuantLayerOracle(B, 12 * P, P, W, "bf16")
    for t, flags in ((4 * P, 0), (6 * P, DIRECT)):
        k, v = (hf_layout(B, H, t, D, torch.bfloat16, gen) for _ in range(2))
        before = [x.tolist() for x in (pool.bt, pool.lens, pool.hw)], pool.ctrl[[0, 2]].tolist()
        if flags == 0 or not short:
            oracle.append(to_bits(k), to_bits(v))
        pool.update(k.cuda(), v.cuda(), oracle.get_seq_length(), flags)
        pool.check_invariants()
    assert pool.errors() == (1 if short else 0)
    if short:
        assert before == ([x.tolist() for x in (pool.bt, pool.lens, pool.hw)], pool.ctrl[[0, 2]].tolist())
    for got, want in zip(pool.gather(B, oracle.get_seq_length()), oracle.current_tensors()):
        assert np.array_equal(to_bits(got), want)
