"""int4_linear's one-pass eager route gives the checked path's shape, or its refusal, for every bias (no GPU).

The kernel launch of both routes is replaced by a fixed product; everything after it is the package's.
"""

from __future__ import annotations

import pytest
import torch

from kernelforge import ops

M, N, K, G = 3, 64, 128, 128
BIASES = {"row": (N,), "row_2d": (1, N), "per_token": (M, N), "scalar": (), "one": (1,), "row_3d": (1, 1, N),
          "full_3d": (1, M, N), "batch": (7, 1, N), "batch_2d": (7, N), "short": (N - 1,)}


def _outcome(bias):
    x, packed, scales = torch.zeros(M, K).half(), torch.zeros(N, K // 8, dtype=torch.int32), torch.ones(N, 1).half()
    try:
        y = ops.int4_linear(x, packed, scales, G, bias)
        return y.shape, y.dtype, y.flatten().tolist()
    except RuntimeError as exc:
        return str(exc)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("bias", BIASES)
def test_bias_shapes(monkeypatch, bias, dtype):
    product = torch.arange(M * N).view(M, N).half()
    values = torch.arange(max(1, torch.Size(BIASES[bias]).numel())).view(BIASES[bias]).to(dtype)
    monkeypatch.setattr(ops, "_check_int4", lambda *a: None)
    monkeypatch.setattr(ops, "_matmul_checked", lambda *a: product.clone())
    monkeypatch.setattr(ops, "_launch", lambda *a: product.clone())
    monkeypatch.setattr(ops, "_eager_shape", lambda *a: None)
    checked = _outcome(values)
    monkeypatch.setattr(ops, "_eager_shape", lambda *a: (M, N, K, 0))
    assert _outcome(values) == checked
