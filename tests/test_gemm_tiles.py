"""Every tile of int4_gemm at its edges against an exact reference (needs a GPU).

Shapes are the smallest that the dispatcher gives to each tile on a 256-CU device, with rows left over in
the last row tile, columns in the last column tile where N allows it, K = 64 mod 128 where the tile takes
it, and one split-K case per tile that splits.  The reference is float64 on the operand the kernels
use, W = fp16(q * s).  Error bound per element: K fp32 additions of exact products, and the fp16
rounding of the result: K 2^-24 sum |x w| + 2^-11 |y| (+ the smallest fp16 step).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kernelforge import ops
from oracle import int4_oracle as o

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (tile, splits, M, N, K)
CASES = [
    ((8, 16), 1, 17, 64, 1856), ((8, 16), 8, 33, 64, 4224), ((16, 16), 1, 129, 256, 1088),
    ((16, 16), 8, 33, 128, 4224), ((16, 32), 1, 385, 320, 1088), ((16, 32), 7, 33, 384, 8960),
    ((16, 64), 1, 161, 1472, 448), ((24, 16), 1, 193, 320, 576), ((24, 16), 8, 81, 128, 7424),
    ((32, 16), 1, 193, 320, 448), ((32, 16), 8, 49, 256, 4224), ((32, 32), 1, 513, 384, 1088),
    ((32, 32), 8, 97, 256, 8960), ((32, 48), 1, 193, 1728, 832), ((32, 48), 4, 63, 1472, 7424),
    ((48, 16), 1, 513, 256, 576), ((48, 16), 8, 161, 128, 8960), ((48, 32), 1, 385, 640, 448),
    ((48, 32), 8, 65, 512, 8960), ((48, 48), 1, 513, 1024, 1088), ((48, 48), 2, 900, 256, 7424),
    ((32, 32), 1, 513, 256, 448), ((32, 32), 7, 25, 2304, 8960), ((48, 48), 1, 513, 1024, 448),
    ((48, 48), 5, 47, 4608, 8960), ((64, 32), 1, 600, 640, 448), ((64, 32), 5, 49, 1472, 4224),
    ((64, 48), 1, 900, 640, 448), ((64, 48), 2, 900, 384, 7424), ((64, 64), 1, 769, 1024, 1856),
    ((64, 64), 2, 900, 512, 4224), ((8, 16), 1, 7, 64, 448), ((16, 16), 1, 257, 128, 448),
    ((32, 128), 1, 769, 1024, 384), ((48, 128), 1, 900, 1280, 384), ((48, 128), 2, 900, 768, 4224),
    ((64, 128), 1, 900, 1728, 384), ((64, 128), 3, 900, 640, 4224), ((80, 128), 1, 769, 2560, 384),
    ((80, 128), 2, 900, 1280, 4224), ((112, 128), 1, 900, 3072, 384), ((112, 128), 2, 900, 1472, 4224),
    ((128, 128), 1, 600, 6400, 640), ((128, 128), 2, 900, 2048, 5632), ((128, 128), 1, 900, 2560, 448),
    ((128, 128), 3, 900, 2304, 6272), ((192, 256), 1, 900, 8960, 384),
]


@pytest.mark.parametrize("tile,splits,m,n,k", CASES)
def test_tile_edges(tile, splits, m, n, k):
    group = 128 if k % 128 == 0 else 64
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        plan = ops.gemm_plan(m, n, k, group)
        assert (plan["tile"], plan["splits"]) == (tile, splits)
    rng = np.random.Generator(np.random.PCG64(m * 7 + n + k))
    w = (rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    packed, scales = o.quantize_weight(w, group)
    x = torch.from_numpy(rng.standard_normal((m, k), dtype=np.float32).astype(np.float16))
    w64 = torch.from_numpy(o.dequantize_fp16(packed, scales, group)).to(DEV, torch.float64)
    x64 = x.to(DEV, torch.float64)
    ref = x64 @ w64.T
    bound = k * 2.0 ** -24 * (x64.abs() @ w64.abs().T) + 2.0 ** -11 * ref.abs() + 2.0 ** -24
    out = ops.int4_gemm(x.to(DEV), torch.from_numpy(packed).to(DEV), torch.from_numpy(scales).to(DEV), group)
    err = (out.to(torch.float64) - ref).abs()
    assert bool((err <= bound).all()), f"largest error / bound {float((err / bound).max()):.2f}"
