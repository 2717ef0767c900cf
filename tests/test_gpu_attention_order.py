"""Decode attention gives the same bits whatever other attention kernels the process ran before: the cut
of the work over resident waves is each kernel's own."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import hashlib, sys
import torch
from barqtrain_amd.paged import PagePool

def digest(D, rows):
    # 33000 chunks of 16 positions: more than a range's least, at 2048 waves and at 1024
    gen = torch.Generator(device="cuda").manual_seed(D + rows)
    draw = lambda *shape: torch.randn(shape, generator=gen, device="cuda").bfloat16().transpose(1, 2)
    pool = PagePool(max_batch=66, max_blocks=250, page_size=8, kv_heads=4, head_dim=D, dtype=torch.bfloat16, device="cuda")
    pool.append(draw(66, 1990, 4, D), draw(66, 1990, 4, D))
    out = pool.attend(draw(66, 1, 4 * rows, D))
    return hashlib.sha1(out.contiguous().view(torch.int16).cpu().numpy().tobytes()).hexdigest()

for arg in sys.argv[1:]:
    D, rows = map(int, arg.split("x"))
    print(arg, digest(D, rows), flush=True)
"""


def digests(*calls):
    env = {**os.environ, "PYTHONPATH": os.path.dirname(os.path.dirname(os.path.abspath(__file__)))}
    out = subprocess.run([sys.executable, "-c", CHILD, *calls], env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    return dict(line.split() for line in out.stdout.splitlines() if "x" in line.split()[0])


def test_attention_bits_do_not_depend_on_earlier_calls(hip):
    # (head size x query rows a KV head): two waves a SIMD resident for 128 x 4 and 64 x 8, one for the others
    calls = ["128x4", "64x8", "128x12", "256x4"]
    first = digests(*calls)
    assert set(first) == set(calls)
    assert digests(*reversed(calls)) == first
