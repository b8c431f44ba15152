"""Every configuration of int4_gemm at its edges against an exact reference (needs a GPU).

Shapes are small ones that the dispatcher gives to each configuration (tile, wavefronts, kernel) on a 256-CU
device, with rows left over in the last row tile, columns in the last column tile where N allows it, K = 64
mod 128 where the tile takes it, and one split-K case per configuration that splits.  The reference is float64 on the operand the kernels
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

# (configuration, tile, splits, M, N, K)
CASES = [
    (0, (8, 16), 1, 17, 64, 1088), (0, (8, 16), 8, 17, 64, 9024), (1, (16, 16), 1, 33, 64, 832),
    (1, (16, 16), 8, 17, 192, 9024), (2, (16, 32), 1, 33, 2304, 1088), (2, (16, 32), 7, 33, 384, 10048),
    (3, (16, 64), 1, 33, 4608, 320), (4, (24, 16), 1, 17, 2304, 1856), (4, (24, 16), 6, 33, 320, 10048),
    (5, (32, 16), 1, 1025, 64, 320), (5, (32, 16), 8, 17, 384, 10048), (6, (32, 32), 1, 17, 4608, 1856),
    (6, (32, 32), 6, 97, 320, 9024), (7, (32, 48), 1, 17, 8960, 576), (7, (32, 48), 8, 17, 1472, 10048),
    (8, (48, 16), 1, 65, 1728, 832), (8, (48, 16), 7, 385, 64, 10048), (9, (48, 32), 1, 33, 6144, 320),
    (9, (48, 32), 8, 65, 512, 9024), (10, (48, 48), 1, 33, 8960, 1856), (10, (48, 48), 4, 65, 1472, 9024),
    (11, (32, 32), 1, 17, 6400, 192), (11, (32, 32), 5, 17, 4608, 9024), (12, (48, 48), 1, 33, 8960, 192),
    (12, (48, 48), 7, 33, 1728, 10048), (13, (64, 32), 1, 97, 6400, 192), (13, (64, 32), 6, 49, 2560, 9024),
    (14, (64, 48), 1, 49, 8960, 1088), (14, (64, 48), 5, 49, 2304, 9024), (15, (64, 64), 1, 97, 6400, 2112),
    (15, (64, 64), 2, 2047, 256, 9024), (16, (8, 16), 1, 7, 64, 832), (16, (8, 16), 8, 17, 64, 7424),
    (17, (16, 16), 1, 7, 64, 192), (18, (32, 128), 1, 513, 1472, 128), (18, (32, 128), 7, 17, 4608, 5632),
    (19, (48, 128), 1, 900, 1472, 128), (19, (48, 128), 6, 129, 1728, 8960), (20, (64, 128), 1, 1025, 1472, 384),
    (20, (64, 128), 8, 97, 1728, 11520), (21, (80, 128), 1, 1301, 1728, 128), (21, (80, 128), 8, 145, 1728, 11520),
    (22, (112, 128), 1, 2047, 1472, 384), (22, (112, 128), 7, 97, 4608, 6272), (23, (128, 128), 1, 2047, 1728, 640),
    (23, (128, 128), 5, 2047, 320, 11520), (24, (128, 128), 1, 1301, 1728, 192),
    (24, (128, 128), 6, 769, 1472, 9024), (25, (192, 256), 1, 1301, 8960, 128),
]


@pytest.mark.parametrize("config,tile,splits,m,n,k", CASES)
def test_tile_edges(config, tile, splits, m, n, k):
    group = 128 if k % 128 == 0 else 64
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        plan = ops.gemm_plan(m, n, k, group)
        assert (plan["kernel"], plan["tile"], plan["splits"]) == (config, tile, splits)
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


def test_every_configuration_has_a_case():
    num = ops.gemm_plan(64, 2048, 2048)["num_kernels"]
    assert {c[0] for c in CASES} == set(range(num))
