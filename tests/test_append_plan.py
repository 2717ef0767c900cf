"""Host-side append planning of PagePool (pages an append takes, longest row after it) against a
per-row restatement: row b maps blocks ceil(hw_b / P) .. min(ceil((len_b + T) / P), max_blocks)
- 1 for the first time, on random lengths, high-water marks, page sizes and token counts; and the
capacity error when a row would pass the limit."""

from __future__ import annotations

import pickle

import numpy as np
import pytest
import torch

from barqtrain_amd.paged import PagedKVCapacityError, PagePool


def _reference_need(lens, hw, T, P, mb):
    need = 0
    for l, h in zip(lens.tolist(), hw.tolist()):
        first = -(-h // P)
        end = min(-(-(l + T) // P), mb)
        need += max(end - first, 0)
    return need


def test_plan_matches_per_row_restatement():
    rng = np.random.default_rng(11)
    checked = 0
    for _ in range(1500):
        P = int(rng.choice([1, 3, 16, 32]))
        mb = int(rng.integers(1, 20))
        B = int(rng.integers(1, 9))
        pool = PagePool(max_batch=B, max_blocks=mb, page_size=P, kv_heads=1, head_dim=4, dtype=torch.float32,
                        device="cpu")
        cap = mb * P
        lens = rng.integers(0, cap + 1, size=B)
        hw = np.maximum(lens, rng.integers(0, cap + 1, size=B))
        pool.lens[:] = lens
        pool.hw[:] = hw
        pool.free_count = 10**9
        T = int(rng.integers(1, 2 * P + 2))
        batch = int(rng.integers(1, B + 1))
        if lens[:batch].max() + T > cap:
            with pytest.raises(PagedKVCapacityError):
                pool.check_append(batch, T)
            continue
        need = pool.check_append(batch, T)
        assert need == _reference_need(lens[:batch], hw[:batch], T, P, mb)
        checked += 1
    assert checked > 500


def test_a_pool_saved_without_its_packed_tensors_loads(monkeypatch):
    """Pools pickled before these attributes were set from the start, or with addresses packed in them."""
    pool = PagePool(max_batch=2, max_blocks=2, page_size=4, kv_heads=1, head_dim=4, dtype=torch.float32, device="cpu")
    keys = torch.arange(24, dtype=torch.float32).view(2, 1, 3, 4)
    pool.append(keys, -keys)
    for extra in ({}, {"_handle": (0, torch.zeros(8))}):
        state = {k: v for k, v in pool.__dict__.items() if k not in ("_handle", "_attn_ws")}
        with monkeypatch.context() as m:
            m.setattr(PagePool, "__getstate__", lambda self: {**state, **extra})
            saved = pickle.dumps(pool)
        loaded = pickle.loads(saved)
        assert loaded._handle is None and loaded.attention_workspace(10).numel() >= 10
        assert torch.equal(loaded.gather(2)[0], keys) and loaded.lens.tolist() == [3, 3]
