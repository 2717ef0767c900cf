"""Blocks quantised by waves at the edges of what a wave takes -- heads whose page is 16, 32 and 64 vectors
a lane (split units), a half, a quarter and less of a wave (packed units, the last of them not full),
and just past both -- against the host pool (which the oracle checks): codes, scales and bits read,
with infinities, NaN, zeros and subnormals among them."""

import pytest
import torch

from kvgen import normal

from barqtrain_amd.paged import QuantPagePool

pytestmark = pytest.mark.gpu


def inputs(B, T, H, D, dtype, gen):
    x = normal((B, T, H, D), dtype, gen)
    x[:, :, :, ::8] *= 8
    x[0, :, 0, :2] = 0
    x[-1, T // 3] *= 2.0 ** (-130 if dtype == torch.bfloat16 else -16)
    x[0, T // 2, -1, 3] = float("nan")
    x[-1, T - 1, 0, -1] = float("-inf")
    return x.transpose(1, 2)


# vectors of one head's page, two-byte (fp32: twice as many): 1024, 1024, 1024, 2048, 2048, 4096, 1024 and 2048 of
# two vectors a row, 32, 16, 8, 16, 1, 64
@pytest.mark.parametrize("H,D,P", [(2, 128, 64), (1, 256, 32), (3, 512, 16), (1, 256, 64), (2, 128, 128), (1, 256, 128),
                                   (1, 16, 512), (1, 16, 1024), (8, 64, 4), (16, 64, 2), (32, 64, 1), (5, 64, 2), (3, 8, 1),
                                   (5, 512, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_blocks_at_the_edges_of_a_wave(hip, H, D, P, dtype):
    B, gen = 3, torch.Generator().manual_seed(H * D + P)
    make = lambda device: QuantPagePool(max_batch=B, max_blocks=9, page_size=P, kv_heads=H, head_dim=D, dtype=dtype,
                                        device=device, window=P + P // 2, chunk=4 * P)
    pool, host = make("cuda"), make("cpu")
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    for b, t in ((B, 4 * P), (1, 1), (B, 3 * P), (2, P)):  # one block of a row, several, ragged rows
        k, v = inputs(b, t, H, D, dtype, gen), inputs(b, t, H, D, dtype, gen)
        pool.append(k.cuda(), v.cuda())
        host.append(k, v)
        table, want = pool.block_table.cpu(), host.block_table
        assert torch.equal(table <= -2, want <= -2) and pool.cold_blocks.tolist() == host.cold_blocks.tolist()
        ours, theirs = (-2 - t[want <= -2].long() for t in (table, want))
        for name in ("key_codes", "value_codes", "key_scales", "value_scales"):
            assert torch.equal(getattr(pool, name).cpu()[ours], getattr(host, name)[theirs]), (name, b, t)
        for x, y in zip(pool.gather(B), host.gather(B)):
            assert torch.equal(x.cpu().view(bits), y.view(bits)), (b, t)
    assert pool.ctrl[[0, 2]].tolist() == [host.free_count, host.cold_free] == [pool.free_count, pool.cold_free]
    assert pool.errors() == 0 and int(pool.cold_blocks.min()) > 0
