"""MFMA-16 block copy of a weight (kf_int4_reorder_mfma16, kf_int4_gemm_mfma16) and the options that once
attached one to a weight (needs a GPU).

The copy is a pure permutation, checked bit for bit against the oracle's statement of the layout
(oracle/int4_oracle.py:reorder_mfma16, itself pinned element by element in test_oracle.py).  No kernel
reads it: the GEMM entry point that takes one gives kf_int4_gemm's result whatever the copy holds, and the
options change neither memory nor route.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from kernelforge import _lib, ops
from oracle import int4_oracle as o

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _weight(n: int, k: int, g: int, seed: int = 0):
    rng = np.random.default_rng(seed + n * 3 + k)
    packed, scales = o.quantize_weight((rng.standard_normal((n, k)) * 0.02).astype(np.float32), g)
    return packed, scales, torch.from_numpy(packed).to(DEV), torch.from_numpy(scales).to(DEV)


def _gemm_raw(x, dp, ds, g, copy=None):
    """kf_int4_gemm, or kf_int4_gemm_mfma16 with `copy`, straight through the C ABI."""
    lib = _lib.load()
    m, k = x.shape
    n = dp.shape[0]
    y = torch.empty(m, n, dtype=torch.float16, device=DEV)
    wsb = lib.kf_int4_gemm_workspace_bytes(m, n, k, g)
    ws = torch.empty(max(wsb, 16) // 4 + 1, dtype=torch.float32, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    if copy is None:
        st = lib.kf_int4_gemm(x.data_ptr(), dp.data_ptr(), ds.data_ptr(), y.data_ptr(), ws.data_ptr(), wsb, m, n, k,
                              g, stream)
    else:
        st = lib.kf_int4_gemm_mfma16(x.data_ptr(), dp.data_ptr(), ds.data_ptr(), copy[0].data_ptr(),
                                     copy[1].data_ptr(), y.data_ptr(), ws.data_ptr(), wsb, m, n, k, g, stream)
    _lib.check(st, "gemm")
    return y


@pytest.mark.parametrize("n,k,g", [(1, 128, 128), (17, 256, 64), (100, 2048, 128), (5632, 2048, 128),
                                   (1536, 8960, 128), (2048, 5632, 64), (256, 1536, 64)])
def test_reorder_matches_oracle(n, k, g):
    packed, scales, dp, ds = _weight(n, k, g)
    pr, sr = ops.int4_reorder_mfma16(dp, ds, g)
    want_p, want_s = o.reorder_mfma16(packed, scales, g)
    assert np.array_equal(pr.cpu().numpy(), want_p)
    assert np.array_equal(sr.cpu().numpy().view(np.uint16), want_s.view(np.uint16))


@pytest.mark.parametrize("g", [64, 128])
@pytest.mark.parametrize("m", [1, 8, 16, 64])
def test_gemm_with_copy_does_not_read_it(m, g):
    n, k = 320, 1152
    packed, scales, dp, ds = _weight(n, k, g)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).half()
    copy = ops.int4_reorder_mfma16(dp, ds, g)
    ref = _gemm_raw(x.to(DEV), dp, ds, g)
    assert torch.equal(_gemm_raw(x.to(DEV), dp, ds, g, copy), ref)
    copy[0].fill_(-1)
    copy[1].fill_(float("nan"))
    assert torch.equal(_gemm_raw(x.to(DEV), dp, ds, g, copy), ref)
    assert o.max_rel_err(ref.float().cpu().numpy(), o.linear_ref_fp32(x.numpy(), packed, scales, g)) <= 2e-3


@pytest.mark.parametrize("m", [4, 8, 64])
def test_options_change_neither_memory_nor_route(monkeypatch, m):
    g, k = 128, 2048
    weights = [_weight(n, k, g, seed=n)[2:] for n in (2048, 256, 256)]
    x = torch.randn(m, k, device=DEV).half()
    lib, launched = _lib.load(), []

    class Spy:
        def __getattr__(self, name):
            if "workspace" not in name:
                launched.append(name)
            return getattr(lib, name)

    def call():
        launched.clear()
        ys = [ops.int4_linear(x, *weights[0], g),
              *ops.int4_linear_grouped([x] * 3, [p for p, _ in weights], [s for _, s in weights], g)]
        torch.cuda.synchronize()
        return ys, list(launched), torch.cuda.memory_allocated()

    monkeypatch.setattr(ops._lib, "load", Spy)
    call()  # whatever the first call sets up
    ys, route, memory = call()
    expected = ["kf_int4_gemv", "kf_int4_gemv_grouped"] if m <= ops.GEMV_MAX_M else ["kf_int4_gemm", "kf_int4_gemm_grouped"]
    assert route == expected
    monkeypatch.setattr(ops, "MFMA16_CACHE", True)
    for p, s in weights:
        ops.prepare_mfma16(p, s, g)
    again, route2, memory2 = call()
    assert route2 == route and all(torch.equal(a, b) for a, b in zip(again, ys))
    assert memory2 == memory + sum(y.untyped_storage().nbytes() for y in ys)  # the first results are still held
    # An in-place update of a weight is what the next call computes with.
    weights[0][0].copy_(_weight(2048, k, g, seed=9)[2])
    assert not torch.equal(call()[0][0], ys[0])


def test_mfma16_rejections():
    lib = _lib.load()
    pb, sb = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.kf_int4_mfma16_sizes(100, 1152, 128, ctypes.byref(pb), ctypes.byref(sb)) == 0
    assert pb.value == 112 * 1152 // 2 and sb.value == 112 * 9 * 2
    assert lib.kf_int4_mfma16_sizes(100, 192, 64, None, None) != 0  # K % 128
    assert "multiple of 128" in _lib.last_error()
    _, _, dp, ds = _weight(64, 256, 128)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.kf_int4_reorder_mfma16(dp.data_ptr(), ds.data_ptr(), None, None, 64, 256, 128, stream) != 0
    with pytest.raises(TypeError):
        ops.int4_reorder_mfma16(dp.float(), ds, 128)


def test_prepare_refuses_what_has_no_copy():
    _, _, dp, ds = _weight(64, 192, 64)
    with pytest.raises(ValueError, match="multiple of 128"):
        ops.prepare_mfma16(dp, ds, 64)
    with pytest.raises(TypeError):
        ops.prepare_mfma16(dp.float(), ds, 64)
