"""Parity of the gfx950 INT4 kernels with the CPU oracle (needs a GPU).

Mirrors the reference's tests/test_gemm.py: every TinyLlama / Qwen2.5 layer
shape at every GEMV M (1..8) and the GEMM's M grid, both group sizes, ragged
N, the dispatcher, and the rejection messages.  The oracle is the pinned numpy
restatement of ``x.float() @ dequantize(qw, float32).T``; the pass rule is the
reference's ``max|out - ref| <= 2e-3 * max|ref|`` (tests/test_gemm.py:17,36-45),
stricter than the 1e-2 the north star allows.  Inputs are seeded on the CPU
(numpy PCG64), weights ~ 0.02 N(0,1) quantized by the oracle, x ~ N(0,1) fp16.
Dequantization is checked bit for bit.
"""

from __future__ import annotations

import ctypes
import functools
from pathlib import Path

import numpy as np
import pytest
import torch

from kernelforge import _lib, ops
from kernelforge import quantize as kq
from oracle import c_oracle
from oracle import int4_oracle as o

pytestmark = pytest.mark.gpu

REL_TOL = 2e-3
DEV = "cuda"
GOLDEN = Path(__file__).resolve().parent / "golden" / "int4_cases.npz"

LAYER_SHAPES = {
    "tinyllama_qo": (2048, 2048), "tinyllama_kv": (256, 2048), "tinyllama_gate_up": (5632, 2048),
    "tinyllama_down": (2048, 5632), "qwen_qo": (1536, 1536), "qwen_kv": (256, 1536),
    "qwen_gate_up": (8960, 1536), "qwen_down": (1536, 8960),
}


@functools.lru_cache(maxsize=None)
def _weights(n: int, k: int, g: int):
    """Oracle-quantized weight for (N, K, G), seeded by the shape; host arrays and device tensors."""
    rng = np.random.Generator(np.random.PCG64(n * 31 + k))
    w = (rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    packed, scales = o.quantize_weight(w, g)
    return packed, scales, torch.from_numpy(packed).to(DEV), torch.from_numpy(scales).to(DEV)


def _x(m: int, k: int, seed: int) -> np.ndarray:
    rng = np.random.Generator(np.random.PCG64(seed))
    return rng.standard_normal((m, k), dtype=np.float32).astype(np.float16)


def _check(error_log, suite, fn, m, n, k, g, case):
    packed, scales, dp, ds = _weights(n, k, g)
    x = _x(m, k, m * 7 + n + k)
    ref = o.linear_ref_fp32(x, packed, scales, g)
    out = fn(torch.from_numpy(x).to(DEV), dp, ds, g)
    assert out.shape == (m, n) and out.dtype == torch.float16
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all(), f"{case}: non-finite output"
    err = o.max_rel_err(got, ref)
    error_log.add(suite, case=case, shape=[m, n, k], group=g, max_rel_err=err, passed=err <= REL_TOL)
    assert err <= REL_TOL, f"{case} M={m} G={g}: rel err {err:.3e}"
    return out


# ---------------------------------------------------------------------------
# GEMV (reference tests/test_gemm.py:48-79)
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("group", [64, 128])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("layer", list(LAYER_SHAPES))
def test_gemv_layer_shapes(error_log, layer, m, group):
    n, k = LAYER_SHAPES[layer]
    _check(error_log, "int4_gemv", ops.int4_gemv, m, n, k, group, layer)


@pytest.mark.parametrize("n", [1, 7, 9, 129])
def test_gemv_ragged_n(error_log, n):
    _check(error_log, "int4_gemv", ops.int4_gemv, 3, n, 256, 128, f"ragged_n{n}")


@pytest.mark.parametrize("k", [64, 128, 2112, 4160])
def test_gemv_odd_chunk_counts(error_log, k):
    """K whose 32-weight chunk count is not a multiple of 64 lanes (partial last pass)."""
    _check(error_log, "int4_gemv", ops.int4_gemv, 2, 200, k, 64, f"k{k}")


def test_gemv_rejects_k_not_multiple_of_group():
    x = torch.randn(1, 200, device=DEV).half()
    packed = torch.zeros(16, 25, dtype=torch.int32, device=DEV)
    scales = torch.ones(16, 2, dtype=torch.float16, device=DEV)
    with pytest.raises(ValueError, match="not a multiple of group_size"):
        ops.int4_gemv(x, packed, scales, 128)


def test_gemv_rejects_large_m():
    _, _, dp, ds = _weights(64, 256, 128)
    x = torch.randn(9, 256, device=DEV).half()
    with pytest.raises(ValueError, match=r"M in \[1, 8\]"):
        ops.int4_gemv(x, dp, ds, 128)


def test_gemv_rejects_shape_mismatch():
    _, _, dp, ds = _weights(64, 256, 128)
    x = torch.randn(1, 256, device=DEV).half()
    with pytest.raises(ValueError, match="K/8"):
        ops.int4_gemv(x[:, :128].contiguous(), dp, ds, 128)


def test_degenerate_shapes():
    """M = 0 raises what the reference raises: int4_gemv's M check, reached from int4_linear
    (2-D and 3-D x) and int4_matmul, and int4_gemm's "bad M" (csrc/gemm/dequant_gemm_tc.cu:14).
    N = 0 and K = 0, for which the reference's GEMV fails its launch or sums nothing and its
    GEMM's split choice divides by zero, raise the C ABI's size error here."""
    _, _, dp, ds = _weights(64, 256, 128)
    x0 = torch.empty(0, 256, device=DEV, dtype=torch.float16)
    for fn in (ops.int4_gemv, ops.int4_matmul, ops.int4_linear):
        with pytest.raises(ValueError, match=r"M in \[1, 8\], got M=0"):
            fn(x0, dp, ds, 128)
    with pytest.raises(ValueError, match="got M=0"):
        ops.int4_linear(torch.empty(2, 0, 256, device=DEV, dtype=torch.float16), dp, ds, 128)
    with pytest.raises(RuntimeError, match="bad M 0"):
        ops.int4_gemm(x0, dp, ds, 128)
    x = torch.randn(1, 256, device=DEV).half()
    with pytest.raises(ValueError, match="positive, got M=1 N=0 K=256"):
        ops.int4_gemv(x, dp[:0], ds[:0], 128)
    with pytest.raises(ValueError, match="positive, got M=1 N=64 K=0"):
        ops.int4_gemv(x[:, :0], dp[:, :0], ds[:, :0], 128)
    with pytest.raises(ValueError, match="positive, got M=16 N=64 K=0"):
        ops.int4_gemm(torch.empty(16, 0, device=DEV, dtype=torch.float16), dp[:, :0], ds[:, :0], 128)


def test_rejects_cpu_and_wrong_dtype():
    _, _, dp, ds = _weights(64, 256, 128)
    with pytest.raises(TypeError, match="fp16 CUDA"):
        ops.int4_gemv(torch.randn(1, 256).half(), dp, ds, 128)
    with pytest.raises(TypeError, match="int32"):
        ops.int4_gemv(torch.randn(1, 256, device=DEV).half(), dp.float(), ds, 128)


# ---------------------------------------------------------------------------
# Multi-problem GEMV launch
# ---------------------------------------------------------------------------

TL_SEVEN = ["tinyllama_qo", "tinyllama_kv", "tinyllama_kv", "tinyllama_qo", "tinyllama_gate_up",
            "tinyllama_gate_up", "tinyllama_down"]


@pytest.mark.parametrize("m", [1, 2, 5, 8])
@pytest.mark.parametrize("group", [64, 128])
def test_grouped_gemv_bit_identical_to_single(error_log, m, group):
    """All 7 TinyLlama linears (plus Qwen's down, > 8 problems -> two launches) in grouped launches:
    each output equals the single-problem GEMV bit for bit and the oracle within tolerance."""
    names = TL_SEVEN + ["qwen_down", "qwen_kv"]
    xs, ps, ss, refs = [], [], [], []
    for i, name in enumerate(names):
        n, k = LAYER_SHAPES[name]
        packed, scales, dp, ds = _weights(n, k, group)
        x = _x(m, k, 1000 + i)
        xs.append(torch.from_numpy(x).to(DEV))
        ps.append(dp)
        ss.append(ds)
        refs.append(o.linear_ref_fp32(x, packed, scales, group))
    ys = ops.int4_gemv_grouped(xs, ps, ss, group)
    for i, name in enumerate(names):
        single = ops.int4_gemv(xs[i], ps[i], ss[i], group)
        assert torch.equal(ys[i], single), f"{name}: grouped differs from single"
        err = o.max_rel_err(ys[i].float().cpu().numpy(), refs[i])
        error_log.add("int4_gemv_grouped", case=name, shape=[m, *LAYER_SHAPES[name]], group=group,
                      max_rel_err=err, passed=err <= REL_TOL)
        assert err <= REL_TOL, f"{name}: {err:.3e}"


@pytest.mark.parametrize("group", [64, 128])
def test_grouped_tinyllama_m2_x_in_lds(error_log, group):
    """The 7 TinyLlama linears at M = 2 in one launch: x of down (22 KiB) exceeds the default LDS
    budget, yet the plan stages x in LDS, with three rows per wavefront for the largest problems so
    the launch fits the workgroups the LDS holds; every output bit-identical to its single launch
    and within tolerance of the oracle."""
    plan = _lib.gemv_plan(2, [LAYER_SHAPES[n] for n in TL_SEVEN])
    assert plan["x_lds"] and 3 in plan["rows"], plan
    xs, ps, ss, refs = [], [], [], []
    for i, name in enumerate(TL_SEVEN):
        n, k = LAYER_SHAPES[name]
        packed, scales, dp, ds = _weights(n, k, group)
        x = _x(2, k, 2000 + i)
        xs.append(torch.from_numpy(x).to(DEV))
        ps.append(dp)
        ss.append(ds)
        refs.append(o.linear_ref_fp32(x, packed, scales, group))
    ys = ops.int4_gemv_grouped(xs, ps, ss, group)
    for i, name in enumerate(TL_SEVEN):
        assert torch.equal(ys[i], ops.int4_gemv(xs[i], ps[i], ss[i], group)), f"{name}: grouped differs from single"
        err = o.max_rel_err(ys[i].float().cpu().numpy(), refs[i])
        error_log.add("int4_gemv_grouped", case=name, shape=[2, *LAYER_SHAPES[name]], group=group,
                      max_rel_err=err, passed=err <= REL_TOL)
        assert err <= REL_TOL, f"{name}: {err:.3e}"


QWEN_SEVEN = [("q", 1536, 1536), ("k", 256, 1536), ("v", 256, 1536), ("o", 1536, 1536),
              ("gate", 8960, 1536), ("up", 8960, 1536), ("down", 1536, 8960)]


@pytest.mark.parametrize("group", [64, 128])
def test_grouped_qwen_seven_as_benchmarked(error_log, group):
    """BASELINE config 3 exactly as bench.py times it: the 7 Qwen2.5-1.5B linears in one grouped
    launch at M = 1 (flat rows for the six K = 1536 linears, deep rows for down), each output
    bit-identical to its own GEMV launch and within tolerance of the oracle."""
    xs, ps, ss, refs = [], [], [], []
    for i, (_, n, k) in enumerate(QWEN_SEVEN):
        packed, scales, dp, ds = _weights(n, k, group)
        x = _x(1, k, 3000 + i)
        xs.append(torch.from_numpy(x).to(DEV))
        ps.append(dp)
        ss.append(ds)
        refs.append(o.linear_ref_fp32(x, packed, scales, group))
    ys = ops.int4_linear_grouped(xs, ps, ss, group)
    for i, (name, n, k) in enumerate(QWEN_SEVEN):
        assert torch.equal(ys[i], ops.int4_gemv(xs[i], ps[i], ss[i], group)), f"qwen {name}: grouped != single"
        err = o.max_rel_err(ys[i].float().cpu().numpy(), refs[i])
        error_log.add("int4_gemv_grouped", case=f"qwen_seven_{name}", shape=[1, n, k], group=group,
                      max_rel_err=err, passed=err <= REL_TOL)
        assert err <= REL_TOL, f"qwen {name}: {err:.3e}"


@pytest.mark.parametrize("group", [64, 128])
def test_grouped_tinyllama_seven_as_benchmarked(error_log, group):
    """BASELINE config 2 exactly as bench.py times its headline: bench.py's layer table and seeded
    weights (make_layers), and one launch of bench.BoundSteps, which calls kf_int4_gemv_grouped
    through the C ABI with the problem table the timed region uses.  The plan must be the one the
    headline runs (gate at three rows per wavefront, the rest at two, x in LDS); every output must
    equal ops.int4_linear_grouped's and its own GEMV launch bit for bit, and the oracle within the
    reference's tolerance."""
    import bench
    from kernelforge import quantize as kq_

    shapes = [(n, k) for _, n, k in bench.TL_LAYERS]
    assert [nm for nm, _, _ in bench.TL_LAYERS] == ["q", "k", "v", "o", "gate", "up", "down"]
    plan = _lib.gemv_plan(1, shapes)
    assert plan["rows"] == [2, 2, 2, 2, 3, 2, 2] and plan["x_lds"], plan
    layers = bench.make_layers(torch, kq_, bench.TL_LAYERS, group=group)
    xs = [ly["x"].to(DEV) for ly in layers]
    dev = [[(ly["packed"].to(DEV), ly["scales"].to(DEV)) for ly in layers]]
    steps = bench.BoundSteps(torch, _lib, _lib.load(), xs, dev, group)
    print(f"tinyllama seven as benchmarked: G={group} plan {plan}", flush=True)
    steps.launch(0)
    torch.cuda.synchronize()
    via_op = ops.int4_linear_grouped(xs, [p for p, _ in dev[0]], [s for _, s in dev[0]], group)
    for i, ly in enumerate(layers):
        y = steps.ys[i]
        assert torch.equal(y, via_op[i]), f"{ly['name']}: BoundSteps launch != int4_linear_grouped"
        assert torch.equal(y, ops.int4_gemv(xs[i], *dev[0][i], group)), f"{ly['name']}: grouped != single"
        packed, scales = ly["packed"].numpy(), ly["scales"].numpy()
        ref = o.linear_ref_fp32(ly["x"].numpy(), packed, scales, group)
        err = o.max_rel_err(y.float().cpu().numpy(), ref)
        error_log.add("int4_gemv_grouped", case=f"tinyllama_seven_{ly['name']}", shape=[1, ly["N"], ly["K"]],
                      group=group, max_rel_err=err, passed=err <= REL_TOL)
        assert err <= REL_TOL, f"tinyllama {ly['name']}: {err:.3e}"


@pytest.mark.parametrize("shapes,m_leads", [
    ([(9, 256), (129, 512), (64, 4160), (1, 128)], [(1, 1), (2, 3)]),  # ragged N at M <= 8: GEMV fallback
    ([(64, 256), (192, 512), (128, 4160)], [(2, 5), (33,)]),            # M > GEMV_MAX_M: per-problem GEMM
])
def test_grouped_linear_ragged_and_bias(shapes, m_leads):
    """Ragged N, different K per problem, biases, 3-D inputs, and the large-M path."""
    for m_lead in m_leads:
        xs, ps, ss, bs, refs = [], [], [], [], []
        for i, (n, k) in enumerate(shapes):
            packed, scales, dp, ds = _weights(n, k, 64)
            x = _x(int(np.prod(m_lead)), k, 50 + i)
            xs.append(torch.from_numpy(x).to(DEV).reshape(*m_lead, k))
            ps.append(dp)
            ss.append(ds)
            b = torch.randn(n, device=DEV).half() if i % 2 == 0 else None
            bs.append(b)
            ref = o.linear_ref_fp32(x, packed, scales, 64)
            refs.append(ref + (b.float().cpu().numpy() if b is not None else 0))
        ys = ops.int4_linear_grouped(xs, ps, ss, 64, bs)
        for i, y in enumerate(ys):
            assert y.shape == (*m_lead, shapes[i][0])
            assert o.max_rel_err(y.float().cpu().numpy().reshape(refs[i].shape), refs[i]) <= REL_TOL


def test_grouped_rejects_mixed_m():
    _, _, dp, ds = _weights(64, 256, 128)
    with pytest.raises(ValueError, match="share M"):
        ops.int4_gemv_grouped([torch.randn(1, 256, device=DEV).half(), torch.randn(2, 256, device=DEV).half()],
                              [dp, dp], [ds, ds], 128)


# ---------------------------------------------------------------------------
# GEMM (reference tests/test_gemm.py:82-99)
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("group", [64, 128])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 32, 64, 65, 128])
@pytest.mark.parametrize("layer", list(LAYER_SHAPES))
def test_gemm_layer_shapes(error_log, layer, m, group):
    n, k = LAYER_SHAPES[layer]
    _check(error_log, "int4_gemm", ops.int4_gemm, m, n, k, group, layer)


@pytest.mark.parametrize("m", [200, 256, 512, 2048])
@pytest.mark.parametrize("layer", ["tinyllama_gate_up", "tinyllama_down"])
def test_gemm_crossover_sweep_sizes(error_log, layer, m):
    """BASELINE config 4's large-M points at full size, including the M=2048 headline."""
    n, k = LAYER_SHAPES[layer]
    _check(error_log, "int4_gemm", ops.int4_gemm, m, n, k, 128, f"{layer}_large_m")


@pytest.mark.parametrize("n", [64, 192, 320])
def test_gemm_n_multiple_of_64_not_128(error_log, n):
    _check(error_log, "int4_gemm", ops.int4_gemm, 37, n, 512, 64, f"n{n}")


# Ragged shapes over the streaming and the LDS-DMA tiles, with and without split-K: N not a multiple
# of the tile width, M just past a tile boundary, K % 128 != 0.  (Every configuration by itself:
# test_gemm_tiles.py.)
EDGE_CASES = [(513, 2112, 384), (1000, 320, 4224), (1000, 2112, 384), (1500, 640, 8960), (33, 64, 1152),
              (33, 320, 4224), (300, 960, 2048), (33, 192, 2304), (33, 640, 8960), (47, 704, 5120),
              (130, 1600, 640), (65, 192, 4160), (900, 1472, 6272), (600, 1216, 7424), (1300, 6080, 640),
              (33, 1472, 8960), (193, 1472, 14336)]


@pytest.mark.parametrize("m,n,k,group", [(m, n, k, g) for m, n, k in EDGE_CASES for g in (64, 128) if k % g == 0])
def test_gemm_edge_shapes(error_log, m, n, k, group):
    _check(error_log, "int4_gemm", ops.int4_gemm, m, n, k, group, f"edge_{m}x{n}x{k}")


def _kinds(plans):
    """(streaming or LDS-DMA tile, splits K) of each plan: the DMA tiles are 128 or 256 columns wide."""
    return {("dma" if p["tile"][1] >= 128 else "stream", p["splits"] > 1) for p in plans}


def test_edge_shapes_reach_both_kinds_of_tile_and_split_k():
    plans = [ops.gemm_plan(m, n, k, 64) for m, n, k in EDGE_CASES]
    assert _kinds(plans) == {("stream", False), ("stream", True), ("dma", False), ("dma", True)}
    assert len({p["kernel"] for p in plans}) >= 8


@pytest.mark.parametrize("m", [1, 8, 9, 128])
def test_matmul_dispatcher(error_log, m):
    _check(error_log, "int4_matmul", ops.int4_matmul, m, 2048, 2048, 128, "dispatch")


CONFIG4_M = [1, 2, 4, 8, 16, 32, 64, 128, 256, 512, 2048]


@pytest.mark.parametrize("m", CONFIG4_M)
@pytest.mark.parametrize("layer", ["tinyllama_gate_up", "tinyllama_down"])
def test_matmul_config4_grid(error_log, layer, m):
    """BASELINE config 4 in full: int4_matmul (the dispatcher the op calls) on TinyLlama gate and
    down at every M of the crossover sweep, whichever kernel it picks, against the oracle."""
    n, k = LAYER_SHAPES[layer]
    _check(error_log, "int4_matmul", ops.int4_matmul, m, n, k, 128, f"config4_{layer}")


@pytest.mark.parametrize("m", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("layer", ["tinyllama_gate_up", "tinyllama_down"])
def test_gemm_small_m(error_log, layer, m):
    """int4_gemm at the rows around the GEMV / GEMM crossover, against the oracle on config 4's gate and
    down; int4_matmul above it is the same kernel."""
    n, k = LAYER_SHAPES[layer]
    _, _, dp, ds = _weights(n, k, 128)
    out = _check(error_log, "int4_gemm", ops.int4_gemm, m, n, k, 128, f"small_m_{layer}")
    if m > ops.GEMV_MAX_M:
        x = torch.from_numpy(_x(m, k, m * 7 + n + k)).to(DEV)
        assert torch.equal(ops.int4_matmul(x, dp, ds, 128), out)


def test_matmul_ragged_n_follows_the_reference_dispatch():
    """Reference int4_matmul (kernelforge/ops.py:193,212): M <= 7 -> GEMV (any N), M >= 8 -> GEMM,
    which rejects N % 64 != 0."""
    packed, scales, dp, ds = _weights(100, 256, 128)
    x7 = _x(7, 256, 7)
    y = ops.int4_matmul(torch.from_numpy(x7).to(DEV), dp, ds, 128)
    torch.cuda.synchronize()
    assert o.max_rel_err(y.float().cpu().numpy(), o.linear_ref_fp32(x7, packed, scales, 128)) <= REL_TOL
    with pytest.raises(ValueError, match="multiple of 64"):
        ops.int4_matmul(torch.from_numpy(_x(8, 256, 8)).to(DEV), dp, ds, 128)


def test_gemm_rejects_n_not_multiple_of_64():
    _, _, dp, ds = _weights(100, 256, 128)
    x = torch.randn(16, 256, device=DEV).half()
    with pytest.raises(ValueError, match="multiple of 64"):
        ops.int4_gemm(x, dp, ds, 128)


DETERMINISM = [("tinyllama_kv", 128), ("tinyllama_down", 64), ("qwen_down", 33), ("tinyllama_down", 2048),
               ("qwen_down", 517), ("qwen_down", 1536), ("tinyllama_gate_up", 16), ("tinyllama_gate_up", 768)]


@pytest.mark.parametrize("layer,m", DETERMINISM)
def test_gemm_is_deterministic(layer, m):
    """Split-K partials, the DMA kernel's in-block k-group halves and the streaming tiles'
    per-wave K slices are reduced in fixed order: repeated calls are bitwise identical."""
    n, k = LAYER_SHAPES[layer]
    _, _, dp, ds = _weights(n, k, 128)
    x = torch.from_numpy(_x(m, k, 99)).to(DEV)
    outs = [ops.int4_gemm(x, dp, ds, 128) for _ in range(3)]
    assert all(torch.equal(outs[0], o_) for o_ in outs[1:])


def test_determinism_cases_split_k_and_do_not():
    plans = [ops.gemm_plan(m, *LAYER_SHAPES[layer], 128) for layer, m in DETERMINISM]
    assert _kinds(plans) >= {("stream", False), ("dma", False), ("dma", True)}


def test_layer_shapes_reach_both_kinds_of_tile_and_ask_for_a_workspace_where_they_split():
    cases = [(m, *LAYER_SHAPES[layer]) for layer in LAYER_SHAPES for m in (1, 8, 9, 16, 17, 32, 64, 65, 128)]
    cases += [(m, *LAYER_SHAPES[layer]) for layer in ("tinyllama_gate_up", "tinyllama_down")
              for m in (200, 256, 512, 2048)]
    cases += [(33, 128, 4160), (65, 192, 512), (17, 5632, 2048), (300, 2048, 5632), (1536, 1536, 8960),
              (33, 1536, 8960), (517, 1536, 8960)]
    plans = [ops.gemm_plan(m, n, k, 128) for m, n, k in cases]
    assert _kinds(plans) == {("stream", False), ("stream", True), ("dma", False), ("dma", True)}
    for (m, n, k), p in zip(cases, plans):
        ws = _lib.load().kf_int4_gemm_workspace_bytes(m, n, k, 128)
        assert (ws > 0) == (p["splits"] > 1)


# ---------------------------------------------------------------------------
# Bit-exact dequantization and fixed fixtures
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("layer", ["tinyllama_gate_up", "qwen_down"])
@pytest.mark.parametrize("group", [64, 128])
def test_dequant_fp16_bit_exact(layer, group):
    n, k = LAYER_SHAPES[layer]
    packed, scales, dp, ds = _weights(n, k, group)
    got = ops.int4_dequant_fp16(dp, ds, group).cpu().numpy().view(np.uint16)
    want = o.dequantize_fp16(packed, scales, group).view(np.uint16)
    assert np.array_equal(got, want)


def test_golden_fixtures_all_paths(error_log):
    data = np.load(GOLDEN)
    for name in sorted({k.split("__")[0] for k in data.files}):
        g = int(data[f"{name}__g"])
        x = torch.from_numpy(data[f"{name}__x"]).to(DEV)
        dp = torch.from_numpy(data[f"{name}__packed"]).to(DEV)
        ds = torch.from_numpy(data[f"{name}__scales"]).to(DEV)
        ref = data[f"{name}__y_ref32"]
        w16 = ops.int4_dequant_fp16(dp, ds, g).cpu().numpy()
        assert np.array_equal(w16.view(np.uint16), data[f"{name}__w_hat16"].view(np.uint16)), name
        fns = [ops.int4_gemv, ops.int4_matmul] + ([ops.int4_gemm] if dp.shape[0] % 64 == 0 else [])
        for fn in fns:
            got = fn(x, dp, ds, g).float().cpu().numpy()
            err = o.max_rel_err(got, ref)
            error_log.add("golden", case=f"{name}:{fn.__name__}", shape=list(ref.shape), group=g,
                          max_rel_err=err, passed=err <= REL_TOL)
            assert err <= REL_TOL, f"{name} {fn.__name__}: {err:.3e}"


@pytest.mark.parametrize("group", [64, 128])
def test_reference_lcg_workload(error_log, group):
    """The reference's torch-free workload (sanitize_gemm.cu:31-95): N=128, K=1024, 4-way split-K,
    double-precision reference, GEMV at M <= 8 and the GEMM at every M."""
    q, scales, packed, xs = c_oracle.lcg_workload(group)
    dp = torch.from_numpy(packed).to(DEV)
    ds = torch.from_numpy(np.ascontiguousarray(scales)).to(DEV)
    for m, x in xs.items():
        ref = c_oracle.ref_f64(x, packed, scales, group)
        xd = torch.from_numpy(np.ascontiguousarray(x)).to(DEV)
        fns = ([ops.int4_gemv] if m <= 8 else []) + [ops.int4_gemm]
        for fn in fns:
            got = fn(xd, dp, ds, group).float().cpu().numpy()
            err = o.max_rel_err(got, ref)
            error_log.add("lcg", case=fn.__name__, shape=[m, 128, 1024], group=group, max_rel_err=err,
                          passed=err <= REL_TOL)
            assert err <= REL_TOL, f"{fn.__name__} M={m} G={group}: {err:.3e}"


# ---------------------------------------------------------------------------
# Guard bands: no write outside y, every element of y written
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("kind,m,n,k", [("gemv", 3, 129, 256), ("gemv", 8, 2048, 5632), ("gemm", 65, 192, 512),
                                        ("gemm", 17, 5632, 2048), ("gemm", 300, 2048, 5632)])
def test_output_guard_bands(kind, m, n, k):
    g = 128
    packed, scales, dp, ds = _weights(n, k, g)
    x = torch.from_numpy(_x(m, k, 5)).to(DEV)
    guard = 4096
    sentinel = torch.tensor(-12345.0, dtype=torch.float16)  # exactly representable, not a plausible output
    buf = torch.full((guard + m * n + guard,), float(sentinel), dtype=torch.float16, device=DEV)
    y_ptr = buf.data_ptr() + 2 * guard
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "gemv":
        st = lib.kf_int4_gemv(x.data_ptr(), dp.data_ptr(), ds.data_ptr(), y_ptr, m, n, k, g, stream)
    else:
        wsb = lib.kf_int4_gemm_workspace_bytes(m, n, k, g)
        ws = torch.empty(max(wsb, 16) // 4 + 1, dtype=torch.float32, device=DEV)
        st = lib.kf_int4_gemm(x.data_ptr(), dp.data_ptr(), ds.data_ptr(), y_ptr, ws.data_ptr(), wsb, m, n, k, g,
                              stream)
    _lib.check(st, kind)
    host = buf.cpu()
    assert (host[:guard] == sentinel).all() and (host[guard + m * n:] == sentinel).all(), "write outside y"
    y = host[guard:guard + m * n].float().numpy().reshape(m, n)
    assert not (y == float(sentinel)).any(), "unwritten output element"
    assert o.max_rel_err(y, o.linear_ref_fp32(_x(m, k, 5), packed, scales, g)) <= REL_TOL


def _grouped_guarded(m: int, shapes, g: int, seed: int):
    """One kf_int4_gemv_grouped launch with every y inside guard bands; checks that nothing is
    written outside y, every element is written, each y equals its own single GEMV launch bit
    for bit and the oracle within tolerance."""
    guard = 2048
    sentinel = torch.tensor(-12345.0, dtype=torch.float16)
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    cases, bufs = [], []
    probs = (_lib.GemvProblem * len(shapes))()
    for i, (n, k) in enumerate(shapes):
        packed, scales, dp, ds = _weights(n, k, g)
        xh = _x(m, k, seed + i)
        x = torch.from_numpy(xh).to(DEV)
        buf = torch.full((guard + m * n + guard,), float(sentinel), dtype=torch.float16, device=DEV)
        probs[i] = _lib.GemvProblem(x.data_ptr(), dp.data_ptr(), ds.data_ptr(), buf.data_ptr() + 2 * guard, n, k)
        cases.append((n, k, xh, x, packed, scales, dp, ds))
        bufs.append(buf)
    _lib.check(lib.kf_int4_gemv_grouped(probs, len(shapes), m, g, stream), "int4_gemv_grouped")
    for (n, k, xh, x, packed, scales, dp, ds), buf in zip(cases, bufs):
        host = buf.cpu()
        what = f"N={n} K={k}"
        assert (host[:guard] == sentinel).all() and (host[guard + m * n:] == sentinel).all(), f"{what}: write outside y"
        y = host[guard:guard + m * n].reshape(m, n)
        assert not (y == sentinel).any(), f"{what}: unwritten output element"
        assert torch.equal(y.to(DEV), ops.int4_gemv(x, dp, ds, g)), f"{what}: grouped differs from single"
        assert o.max_rel_err(y.float().numpy(), o.linear_ref_fp32(xh, packed, scales, g)) <= REL_TOL, what


@pytest.mark.parametrize("m,k", [(1, 1024), (2, 1024), (1, 2048), (2, 2048)])
def test_grouped_guard_bands_three_row_waves(m, k):
    """A grouped launch too large for one resident round at two rows per wavefront (> 8 per SIMD),
    so its largest problems take three rows: ragged N (not a multiple of 3), every output inside
    its guard bands, bit-identical to its own single launch, within tolerance of the oracle.  At
    M = 1, K = 1024 the small problems keep flat rows (two rows in one full load)."""
    ns = [9001, 8999, 4099, 257, 3, 1]
    shapes = [(n, k) for n in ns]
    plan = _lib.gemv_plan(m, shapes)
    assert 3 in plan["rows"], plan
    if m == 1 and k == 1024:
        assert plan["rows"][3:] == [_lib.KF_GEMV_FLAT + 2] * 3, plan
    _grouped_guarded(m, shapes, 128, 300)


@pytest.mark.parametrize("group", [64, 128])
def test_grouped_flat_and_deep_rows(group):
    """The shaped grouped launch (M = 1): flat rows for K = 1536 (four rows in three full loads) and
    K = 1024 (two rows in one), with N leaving the last wavefront part empty, and deep rows (two
    per wavefront, five (row, block) loads per pass) for K = 8960 (two passes of five), 6144 (a
    pass of five, then one) and 2304 (one pass, one clamped load), odd N leaving a wavefront's
    second row past the end, beside a plain two-row problem: outputs inside their guard bands,
    bit-identical to single launches, within tolerance of the oracle."""
    shapes = [(1534, 1536), (1023, 1024), (3001, 1536), (701, 8960), (515, 2304), (257, 2048), (6, 1536),
              (130, 6144)]
    plan = _lib.gemv_plan(1, shapes)
    flat4, flat2, deep = _lib.KF_GEMV_FLAT + 4, _lib.KF_GEMV_FLAT + 2, _lib.KF_GEMV_DEEP
    assert plan["kernel"] == _lib.KF_GEMV_KERNEL_SHAPED, plan
    assert plan["rows"] == [flat4, flat2, flat4, deep, deep, 2, flat4, deep], plan
    _grouped_guarded(1, shapes, group, 700)


# ---------------------------------------------------------------------------
# int4_linear, modules, graph capture
# ---------------------------------------------------------------------------

def test_int4_linear_leading_dims_and_bias():
    n, k = 256, 2048
    packed, scales, dp, ds = _weights(n, k, 128)
    for lead in [(1, 1), (2, 3), (4, 16)]:
        x = _x(int(np.prod(lead)), k, 17).reshape(*lead, k)
        bias = torch.linspace(-1, 1, n, dtype=torch.float16, device=DEV)
        y = ops.int4_linear(torch.from_numpy(x).to(DEV), dp, ds, 128, bias)
        assert y.shape == (*lead, n) and y.dtype == torch.float16
        ref = o.linear_ref_fp32(x.reshape(-1, k), packed, scales, 128).reshape(*lead, n) + bias.float().cpu().numpy()
        assert o.max_rel_err(y.float().cpu().numpy(), ref) <= REL_TOL


def test_custom_op_registered_and_fake():
    x = torch.from_numpy(_x(4, 256, 3)).to(DEV)
    _, _, dp, ds = _weights(64, 256, 128)
    y = torch.ops.kernelforge.int4_matmul(x, dp, ds, 128)
    assert y.shape == (4, 64)
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode() as mode:
        fx = mode.from_tensor(x)
        fy = torch.ops.kernelforge.int4_matmul(fx, mode.from_tensor(dp), mode.from_tensor(ds), 128)
        assert tuple(fy.shape) == (4, 64) and fy.dtype == torch.float16


@pytest.mark.parametrize("m,n", [(1, 5632), (4, 256), (7, 100), (64, 2048)])
def test_eager_path_equals_the_registered_op(m, n):
    """int4_linear / int4_linear_grouped call the ops' implementations directly in eager mode; the
    results equal the registered kernelforge::int4_matmul(_grouped) ops bit for bit, and errors
    come out the same (GEMV for ragged N at M <= 7, the GEMM's rejection at M = 8)."""
    k = 2048
    _, _, dp, ds = _weights(n, k, 128)
    x = torch.from_numpy(_x(m, k, 5 + m)).to(DEV)
    assert torch.equal(ops.int4_linear(x, dp, ds, 128), torch.ops.kernelforge.int4_matmul(x, dp, ds, 128))
    ys = ops.int4_linear_grouped([x, x], [dp, dp], [ds, ds], 128)
    yo = torch.ops.kernelforge.int4_matmul_grouped([x, x], [dp, dp], [ds, ds], 128)
    assert all(torch.equal(a, b) for a, b in zip(ys, yo))
    if n % 64:
        with pytest.raises(ValueError, match="multiple of 64"):
            ops.int4_linear(torch.from_numpy(_x(8, k, 1)).to(DEV), dp, ds, 128)


def test_int4_linear_compiles_through_the_registered_op():
    """Under torch.compile the op (with its fake impl) is what int4_linear calls."""
    _, _, dp, ds = _weights(256, 2048, 128)
    x = torch.from_numpy(_x(2, 2048, 77)).to(DEV)

    def f(a):
        return ops.int4_linear(a, dp, ds, 128) * 2

    assert torch.equal(torch.compile(f, backend="eager", fullgraph=True)(x), f(x))


def test_quantize_linears_swaps_decoder_linears():
    from kernelforge.modules import KFLinearInt4, quantize_linears_

    class Block(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.q_proj = torch.nn.Linear(256, 256, bias=False)
            self.k_proj = torch.nn.Linear(256, 64, bias=True)
            self.lm_head = torch.nn.Linear(256, 128, bias=False)

    torch.manual_seed(0)
    blk = Block().to(DEV).half()
    w_k = blk.k_proj.weight.detach().float().cpu().numpy()
    b_k = blk.k_proj.bias.detach().cpu()
    assert quantize_linears_(blk, 128) == 2
    assert isinstance(blk.q_proj, KFLinearInt4) and isinstance(blk.lm_head, torch.nn.Linear)
    x = _x(2, 256, 1)
    y = blk.k_proj(torch.from_numpy(x).to(DEV))
    packed, scales = o.quantize_weight(w_k, 128)
    ref = o.linear_ref_fp32(x, packed, scales, 128) + b_k.float().numpy()
    assert o.max_rel_err(y.float().cpu().numpy(), ref) <= REL_TOL
    with pytest.raises(TypeError, match="fp16"):
        blk.q_proj(torch.randn(1, 256, device=DEV))


@pytest.mark.parametrize("layer,m", [("tinyllama_gate_up", 1), ("tinyllama_gate_up", 4), ("tinyllama_gate_up", 16),
                                     ("tinyllama_gate_up", 128), ("tinyllama_down", 64)])
def test_hip_graph_capture_replays_match_eager(layer, m):
    """Capture int4_linear (GEMV, streaming tiles, LDS-DMA tiles, GEMM + split-K) in a graph; every replay
    equals eager bitwise."""
    n, k = LAYER_SHAPES[layer]
    _, _, dp, ds = _weights(n, k, 128)
    static_x = torch.from_numpy(_x(m, k, 23)).to(DEV)
    eager = ops.int4_linear(static_x, dp, ds, 128)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.int4_linear(static_x, dp, ds, 128)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_y = ops.int4_linear(static_x, dp, ds, 128)
    for i in range(4):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(static_y, eager), f"replay {i}"
        ops.int4_linear(static_x, dp, ds, 128)  # eager work between replays
        torch.cuda.synchronize()
    new_x = torch.from_numpy(_x(m, k, 24)).to(DEV)
    static_x.copy_(new_x)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(static_y, ops.int4_linear(new_x, dp, ds, 128))


def test_bandwidth_kernels_roundtrip():
    lib = _lib.load()
    nbytes = 64 << 20
    src = torch.randint(0, 2**31 - 1, (nbytes // 4,), dtype=torch.int32, device=DEV)
    dst = torch.zeros_like(src)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.kf_bw_copy(src.data_ptr(), dst.data_ptr(), nbytes, 0, stream), "copy")
    torch.cuda.synchronize()
    assert torch.equal(src, dst)
    sink = torch.zeros(1 << 16, dtype=torch.int32, device=DEV)
    _lib.check(lib.kf_bw_read(src.data_ptr(), sink.data_ptr(), nbytes, 0, stream), "read")
    _lib.check(lib.kf_bw_write(dst.data_ptr(), nbytes, 0, stream), "write")
    torch.cuda.synchronize()
    assert (dst.view(torch.int16) == 0x3C00).all()
