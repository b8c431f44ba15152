"""Sibling GEMMs in shared launches against their own launches, bit for bit (needs a GPU).

int4_linear_grouped above the GEMV's M: siblings of one streaming kind, of the four-k-group DMA tile,
mixtures that share nothing, problems that split K (one workspace), several K in one call, more problems
than one call takes, different inputs, ragged M on both sides of every row-tile height, K = 64 mod 128,
and the smallest K of each group size.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kernelforge import ops
from oracle import int4_oracle as o

pytestmark = pytest.mark.gpu
DEV = "cuda"

SIBLINGS = {
    "qkv": [(2048, 2048), (256, 2048), (256, 2048)],
    "gate_up": [(5632, 2048), (5632, 2048)],
    "wide_narrow": [(64, 1536), (8960, 1536), (192, 1536)],
    "split_and_more": [(1536, 8960), (640, 8960), (320, 4224), (2048, 2048), (64, 4224)],
    "many": [(64 * (1 + i % 3), 448) for i in range(11)],
    "k64": [(256, 64), (256, 64), (64, 64)],
    "k128": [(256, 128), (320, 128)],
}


@pytest.mark.parametrize("m", [5, 8, 9, 16, 17, 27, 33, 64, 65, 129, 200, 333, 517])
@pytest.mark.parametrize("name", SIBLINGS)
def test_bits_of_separate_launches(name, m):
    rng = np.random.Generator(np.random.PCG64(m))
    xs, packed, scales, group = [], [], [], 64 if name in ("many", "k64") else 128
    shared = {}
    for i, (n, k) in enumerate(SIBLINGS[name]):
        p, s = o.quantize_weight((rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)), group)
        x = torch.from_numpy(rng.standard_normal((m, k), dtype=np.float32).astype(np.float16)).to(DEV)
        xs.append(shared.setdefault(k, x) if i % 3 else x)
        packed.append(torch.from_numpy(p).to(DEV))
        scales.append(torch.from_numpy(s).to(DEV))
    ys = ops.int4_linear_grouped(xs, packed, scales, group)
    for i, y in enumerate(ys):
        assert torch.equal(y, ops.int4_linear(xs[i], packed[i], scales[i], group)), f"problem {i}"
