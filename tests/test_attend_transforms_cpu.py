"""Decode attention under torch's transforms: attend takes torch's operations there, as they keep tangents,
batch dimensions and traces, never the one-launch kernel (no GPU; the size rule is told to say yes).
"""

from __future__ import annotations

import pytest
import torch
from torch.autograd import forward_ad

from kernelforge import ops, tinyllama

CFG = tinyllama.TinyLlamaConfig(hidden=64, layers=1, heads=4, kv_heads=2, head_dim=16, intermediate=64, vocab=32, max_seq=8)
D, S = CFG.head_dim, CFG.max_seq


class _Launched(Exception):
    pass


@pytest.fixture
def attend(monkeypatch):
    monkeypatch.setattr(tinyllama.Attention, "fused_decode", lambda self, x: True)

    def launch(*a, **kw):
        raise _Launched

    monkeypatch.setattr(ops, "decode_attention", launch)
    attention = tinyllama.Attention(CFG).half()
    g = torch.Generator().manual_seed(0)
    k, v = torch.randn(2, D, S, generator=g).half(), torch.randn(2, S, D, generator=g).half()
    return lambda q, mask: attention.attend(q, k, v, mask)


def _q(batch=()):
    return torch.randn(*batch, 1, CFG.heads, D, generator=torch.Generator().manual_seed(1)).half()


def _mask(batch=()):
    return torch.zeros(*batch, 2, 2, S).half()


def _library(attend, q, mask):
    """attend's library path: gradients are recorded, so the kernel is out of the question."""
    return attend(q.clone().requires_grad_(), mask).detach()


def test_plain_operands_go_to_the_launch(attend):
    with pytest.raises(_Launched):
        attend(_q(), _mask())


def test_forward_mode_keeps_the_tangent(attend):
    q, t = _q(), torch.ones(1, CFG.heads, D).half()
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(attend(forward_ad.make_dual(q, t), _mask()))
    assert torch.equal(out.primal, _library(attend, q, _mask()))
    assert out.tangent is not None and bool((out.tangent != 0).any())


def test_jvp_keeps_the_tangent(attend):
    out, tangent = torch.func.jvp(lambda q: attend(q, _mask()), (_q(),), (torch.ones(1, CFG.heads, D).half(),))
    assert torch.equal(out, _library(attend, _q(), _mask())) and bool((tangent != 0).any())


def test_vmap_over_tokens(attend):
    q, mask = _q((3,)), _mask((3,))
    out = torch.vmap(attend)(q, mask)
    for i in range(3):
        torch.testing.assert_close(out[i], _library(attend, q[i], _mask()), rtol=2e-3, atol=2e-3)


def test_a_jit_trace_records_the_operations(attend):
    traced = torch.jit.trace(lambda q: attend(q, _mask()), (_q(),), check_trace=False)
    other = _q() * 2
    assert torch.equal(traced(other), _library(attend, other, _mask()))
