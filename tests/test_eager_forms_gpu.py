"""int4_linear's one-pass eager route against its checked path over the forms it may be given (needs a GPU).

Every form either gives the same tensor by both or raises the same error.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kernelforge import ops
from oracle import int4_oracle as o

pytestmark = pytest.mark.gpu
DEV = "cuda"
N, K, G = 192, 512, 128


def _operands(m=3, n=N):
    rng = np.random.Generator(np.random.PCG64(m + n))
    p, s = o.quantize_weight(rng.standard_normal((n, K), dtype=np.float32) * np.float32(0.02), G)
    x = torch.from_numpy(rng.standard_normal((m, K), dtype=np.float32).astype(np.float16)).to(DEV)
    return x, torch.from_numpy(p).to(DEV), torch.from_numpy(s).to(DEV)


def _offset(t, elements):
    """A contiguous copy of t that starts `elements` past an aligned address."""
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    return buf[elements:].view(t.shape).copy_(t)


X, P, S = range(3)
FORMS = {
    "plain": lambda a: a,
    "parameter": lambda a: [a[X], torch.nn.Parameter(a[P], requires_grad=False), a[S]],
    "x_3d": lambda a: [a[X].unsqueeze(0), *a[1:]],
    "x_1d": lambda a: [a[X][0], *a[1:]],
    "x_strided": lambda a: [torch.cat([a[X], a[X]], 1)[:, :K], *a[1:]],
    "x_transposed": lambda a: [a[X].t().contiguous().t(), *a[1:]],
    "x_misaligned": lambda a: [_offset(a[X], 1), *a[1:]],
    "x_fp32": lambda a: [a[X].float(), *a[1:]],
    "x_cpu": lambda a: [a[X].cpu(), *a[1:]],
    "x_empty": lambda a: [a[X][:0], *a[1:]],
    "x_short_k": lambda a: [a[X][:, :K - 64].contiguous(), *a[1:]],
    "x_grad": lambda a: [a[X].clone().requires_grad_(), *a[1:]],
    "packed_transposed": lambda a: [a[X], a[P].t().contiguous().t(), a[S]],
    "packed_misaligned": lambda a: [a[X], _offset(a[P], 1), a[S]],
    "packed_int64": lambda a: [a[X], a[P].long(), a[S]],
    "packed_cpu": lambda a: [a[X], a[P].cpu(), a[S]],
    "packed_3d": lambda a: [a[X], a[P].unsqueeze(0), a[S]],
    "scales_misaligned": lambda a: [a[X], a[P], _offset(a[S], 1)],
    "scales_strided": lambda a: [a[X], a[P], torch.cat([a[S], a[S]], 1)[:, :K // G]],
    "scales_short": lambda a: [a[X], a[P], a[S][:-1]],
    "scales_fp32": lambda a: [a[X], a[P], a[S].float()],
    "no_rows": lambda a: [a[X], a[P][:0], a[S][:0]],
}


def _outcome(args, group, bias):
    try:
        return ops.int4_linear(*args, group, bias)
    except Exception as exc:  # noqa: BLE001 - whatever it raises is compared
        return type(exc), str(exc)


@pytest.mark.parametrize("m,n", [(1, N), (4, N - 5), (6, N - 5), (6, N), (8, N - 5), (40, N)])
@pytest.mark.parametrize("form", FORMS)
def test_same_outcome_as_the_checked_path(monkeypatch, form, m, n):
    args = FORMS[form](list(_operands(m, n)))
    one = torch.ones(n, device=DEV).half()
    for group, bias in ((G, None), (G, one), (G, one.float()), (G, one.view(1, 1, n)), (G, one.expand(m, n)),
                        (G, one.expand(7, 1, n)), (G, one[:1]), (64, None), (32, None)):
        got = _outcome(args, group, bias)
        with monkeypatch.context() as patch:
            patch.setattr(ops, "_eager_shape", lambda *a: None)
            ref = _outcome(args, group, bias)
        if isinstance(ref, torch.Tensor):
            assert torch.equal(got, ref) and got.dtype == ref.dtype and got.requires_grad == ref.requires_grad
        else:
            assert got == ref
