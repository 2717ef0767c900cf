"""Decode attention at head size 256 with up to 4 query rows, on the pair kernel's single-buffered
loop: one, two and several workgroups a pair, rows at the edges of chunks, waves and parts, both
element types and page sizes that hold whole chunks; against the float64 reference."""

import numpy as np
import pytest
import torch

from test_gpu_attention import check, make_rows

pytestmark = pytest.mark.gpu


# rows x 2 kv heads, longest row: several workgroups a pair (8, and 5), two, one (128 pairs and
# more, rows over 44 chunks too), and past the pair kernel's bounds (the flat schedule)
@pytest.mark.parametrize("rows,longest", [(3, 1500), (24, 700), (60, 1000), (64, 1024), (140, 1100), (4, 4000)])
@pytest.mark.parametrize("dtype,page", [(torch.bfloat16, 16), (torch.float16, 32)])
def test_head_dim_256_pairs(rows, longest, dtype, page):
    rng = np.random.default_rng(rows + page)
    edges = [longest, longest - 1, 0, 1, 15, 16, 17, 8 * 16, 8 * 16 + 1, 22 * 16, 22 * 16 + 3, 23 * 16 - 1]
    lens = (edges + rng.integers(0, longest + 1, size=max(rows - len(edges), 0)).tolist())[:rows]
    pool, kd, vd, lens = make_rows(rows, 2, page, lens, dtype, seed=rows, order_seed=rows + 1, D=256)
    ws = None
    for i, (G, T) in enumerate([(4, 1), (2, 2), (1, 1), (1, 3)]):
        ws = check(pool, kd, vd, lens, G, T, dtype, seed=100 + i, ws=ws)
    check(pool, kd, vd, lens, 2, 1, dtype, seed=7, out_f32=False)
    assert pool.errors() == 0
