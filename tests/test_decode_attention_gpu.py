"""The one-launch decode attention against float64 (needs a GPU).

Sizes at the edges of the kernel's loops: head sizes that divide a workgroup's lanes and ones that do
not, odd cache lengths (single-key loads), lengths below, at and past a wavefront's keys and a pass over
the cache, one key, whole wavefronts masked, the longest cache.  Error bound per element, with eps =
2^-24: the scores carry (d + 6) eps of sum |q k| / sqrt(d) + |mask| absolute error, which the softmax
turns into a relative error of twice that; the exponential, the sums over max_seq keys and the division
add (max_seq + 16) eps; the result is rounded to fp16.
"""

from __future__ import annotations

import pytest
import torch

from kernelforge import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 2.0 ** -24


@pytest.mark.parametrize("heads,kv_heads,d,max_seq,live", [
    (32, 4, 64, 160, 78), (32, 4, 64, 160, 160), (12, 2, 128, 96, 1), (4, 4, 8, 1, 1), (6, 3, 24, 33, 20),
    (2, 1, 256, 97, 97), (8, 2, 64, 191, 190), (8, 2, 64, 192, 192), (8, 8, 64, 193, 150), (4, 1, 80, 683, 683),
    (4, 2, 64, 684, 300), (4, 1, 64, 2047, 2000), (3, 1, 128, 8192, 8192),
    (8, 2, 64, 256, 33), (8, 2, 64, 258, 257), (4, 1, 128, 130, 129),
])
@pytest.mark.parametrize("one_row", [True, False], ids=["row_for_all", "row_per_head"])
def test_against_float64(heads, kv_heads, d, max_seq, live, one_row):
    g = torch.Generator(device=DEV).manual_seed(heads + d + max_seq)
    q = torch.randn(heads, d, generator=g, device=DEV).half()
    k = torch.randn(kv_heads, d, max_seq, generator=g, device=DEV).half()
    v = torch.randn(kv_heads, max_seq, d, generator=g, device=DEV).half()
    mask = torch.randn(1 if one_row else heads, max_seq, generator=g, device=DEV).half()
    mask[:, live:] = float("-inf")
    mask = mask.expand(heads, max_seq)
    out = ops.decode_attention(q, k, v, mask, kv_heads=kv_heads)
    rep = heads // kv_heads
    q64, k64, v64 = q.double(), k.double().repeat_interleave(rep, 0), v.double().repeat_interleave(rep, 0)
    scores = (q64.unsqueeze(2) * k64).sum(1) / d ** 0.5 + mask.double()
    probs = torch.softmax(scores, -1)
    ref = (probs.unsqueeze(2) * v64).sum(1)
    mag = ((q64.abs().unsqueeze(2) * k64.abs()).sum(1) / d ** 0.5 + mask.double().abs())[:, :live].amax(-1)
    rel = 2 * (d + 6) * EPS * mag + (max_seq + 16) * EPS
    bound = rel.unsqueeze(1) * (probs.unsqueeze(2) * v64.abs()).sum(1) + 2.0 ** -11 * ref.abs() + EPS
    err = (out.double() - ref).abs()
    assert bool((err <= bound).all()), f"largest error / bound {float((err / bound).max()):.2f}"


def test_nan_and_fully_masked_rows_give_nan():
    q = torch.ones(2, 8, device=DEV, dtype=torch.float16)
    k, v = torch.ones(1, 8, 4, device=DEV).half(), torch.ones(1, 4, 8, device=DEV).half()
    mask = torch.zeros(2, 4, device=DEV, dtype=torch.float16)
    mask[0] = float("-inf")
    q[1, 3] = float("nan")
    assert bool(ops.decode_attention(q, k, v, mask, kv_heads=1).isnan().all())
