"""One-page lean tiles in launches of several rounds: 16, 32 and 64 KiB tiles on both sides of the
bounds that choose them, decode steps, long appends, ragged rows; bit for bit against the device
mirror, with known and device-read row state."""

import numpy as np
import pytest
import torch

from mirror import DeviceMirror

from barqtrain_amd.paged import PagePool

pytestmark = pytest.mark.gpu


# heads, dim, page, rows, prompt: tiles a CU after it (256 CUs)
@pytest.mark.parametrize("H,D,P,B,prompt,dtype", [
    (8, 64, 16, 16, 1500, torch.bfloat16),    # 16 KiB: 11.8
    (2, 64, 32, 40, 1300, torch.float32),     # 16 KiB (2 x 64 fp32: 32 vectors a row): not lean
    (8, 128, 16, 16, 1530, torch.bfloat16),   # 32 KiB: 12, then past the bound
    (8, 128, 32, 4, 6100, torch.float16),     # 64 KiB: 6, then past the bound
    (16, 128, 16, 16, 700, torch.bfloat16),   # 64 KiB, 256 vectors a row: 5.5
])
def test_steps_around_the_round_bounds(hip, H, D, P, B, prompt, dtype):
    gen = torch.Generator(device="cuda").manual_seed(prompt)
    rng = np.random.default_rng(prompt)
    capacity = prompt + 700
    blocks = -(-capacity // P)
    order = torch.from_numpy(rng.permutation(B * blocks).astype(np.int32))
    pool = PagePool(max_batch=B, max_blocks=blocks, page_size=P, kv_heads=H, head_dim=D, dtype=dtype, device="cuda",
                    num_pages=B * blocks, page_order=order)
    mirror = DeviceMirror(B, H, blocks * P, D, dtype)
    for b, t in ((B, prompt), (B, 1), (B // 2, 3), (B, 1), (1, 2 * P), (B, 300), (B, 1)):
        k, v = (torch.randn((b, t, H, D), generator=gen, device="cuda").to(dtype).transpose(1, 2) for _ in range(2))
        mirror.append(k, v)
        pool.free_exact = t != 1 or b == B  # else the device's row state
        mirror.check(pool.update(k, v), f"{b} x {t}")
        seq = int(mirror.lens.max())
        mirror.check(pool.gather(B, seq), f"gather after {b} x {t}")
    assert pool.errors() == 0
