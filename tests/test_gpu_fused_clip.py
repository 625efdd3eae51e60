"""``dpc_gram_clip_factors``: the Gram norms and the clip factors of one linear
layer in one launch (the split Gram kernel's last work item folds the
records and computes the clip factors).  Against the two-call path
(``dpc_gram_sqnorms`` then ``dpc_clip_factors``), bit for bit, on call after
call on one workspace (each call must leave its tickets zero for the next),
for fixed and AUTO-S scales, several guards, a bias (its column sums in a launch
before, its counters in the workspace), and the shapes that take the separate
launches inside the entry point (an odd number of 128-row blocks, float32)
interleaved with one-launch calls.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from opake_amd import _native as nat
from opake_amd import ops
from opake_amd.clipping import guard_for_linear

pytestmark = pytest.mark.gpu


def _inputs(dev, B, T, din, dout, dtype, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    A = torch.randn(B, T, din, generator=g, device=dev).to(dtype)
    scale = torch.exp(torch.randn(B, 1, 1, generator=g, device=dev))
    G = (torch.randn(B, T, dout, generator=g, device=dev) * 1e-4 * scale).to(dtype)
    return A, G


def _plans(plan, B):
    """The defined words of each guard's plan: nactive, nfast, the fast list
    (front) and the other list (back)."""
    out = []
    for g in range(plan.shape[0]):
        w = plan[g].cpu().view(torch.int32)
        nactive, nfast = int(w[0]), int(w[1])
        active = w[4:4 + B].tolist()
        out.append((nactive, nfast, active[:nfast], active[B - (nactive - nfast):]))
    return out


def _two_calls(A, G, C, guards, bias, kind, gamma):
    sq, err = ops.gram_sqnorms(A, G, with_bias=bias, return_error=True)
    cf = ops.clip_factors(sq, C, guards, err=err, kind=kind, gamma=gamma, count_threshold=C)
    return sq, err, cf


CASES = [
    # B, T, din, dout, dtype, bias
    (32, 512, 512, 384, torch.bfloat16, False),
    (8, 256, 256, 256, torch.bfloat16, False),
    (4, 384, 128, 256, torch.bfloat16, False),   # odd block count: separate launches
    (6, 256, 128, 64, torch.bfloat16, True),     # bias: column sums, then one launch
    (5, 130, 72, 40, torch.float32, False),      # float32: separate launches
    (32, 512, 512, 384, torch.bfloat16, False),  # one launch again on the same workspace
    (16, 1024, 256, 512, torch.bfloat16, False),
]


@pytest.mark.parametrize("kind,gamma", [(nat.SCALE_FIXED, 0.0), (nat.SCALE_AUTO_S, 0.01)])
def test_gram_clip_factors_equals_two_calls(dev, kind, gamma):
    for k, (B, T, din, dout, dtype, bias) in enumerate(CASES):
        A, G = _inputs(dev, B, T, din, dout, dtype, seed=100 * k + kind)
        C = 1.0
        guards = [guard_for_linear(dtype, din, dout, bias)]
        if k % 2 == 0:  # a second guard with a bfloat16 multiply
            guards.append((*guards[0][:2], torch.bfloat16))
        for rep in range(2):  # twice in a row: the tickets were left zero
            sq, err, cf = ops.gram_clip_factors(A, G, C, guards, with_bias=bias, kind=kind,
                                                gamma=gamma, count_threshold=C)
            wsq, werr, wcf = _two_calls(A, G, C, guards, bias, kind, gamma)
            assert torch.equal(sq, wsq), (k, rep)
            assert torch.equal(err, werr), (k, rep)
            assert torch.equal(cf.scale, wcf.scale), (k, rep)
            assert torch.equal(cf.norms, wcf.norms), (k, rep)
            assert torch.equal(cf.nclipped, wcf.nclipped), (k, rep)
            assert _plans(cf.plan, B) == _plans(wcf.plan, B), (k, rep)


def test_gram_clip_factors_leaves_counters_zero(dev):
    # The counter buffer is zero after every call, whatever the shape.
    for B, T, din, dout in [(8, 512, 256, 256), (32, 512, 512, 384), (3, 256, 128, 64)]:
        A, G = _inputs(dev, B, T, din, dout, torch.bfloat16, seed=B)
        guards = [guard_for_linear(torch.bfloat16, din, dout, False)]
        ops.gram_clip_factors(A, G, 1.0, guards, count_threshold=1.0)
        torch.cuda.synchronize()
        counters = ops._GRAM_CLIP_COUNTERS[(str(dev), nat.stream_handle(dev).value or 0)]
        assert counters.numel() * 4 >= nat.load().dpc_gram_clip_counter_bytes(B, T)
        assert torch.count_nonzero(counters).item() == 0, (B, T)


@pytest.mark.parametrize("T", [256, 384])  # the split kernel, and separate launches
def test_a_biased_call_leaves_the_counter_buffer_alone(dev, T):
    """A bias needs no counters and does not touch any it is given (another
    stream's call may be using them): none, and words that are no counters."""
    B, din, dout = 6, 128, 264
    A, G = _inputs(dev, B, T, din, dout, torch.bfloat16, T)
    guard = guard_for_linear(torch.bfloat16, din, dout, True)
    sq, err, cf = _two_calls(A, G, 1.0, [guard], True, nat.SCALE_FIXED, 0.0)
    lib = nat.load()
    ws_bytes = lib.dpc_gram_clip_workspace_bytes(B, T)
    n = lib.dpc_gram_clip_counter_bytes(B, T) // 4
    rel, abs_ = (ctypes.c_double * 1)(guard[0]), (ctypes.c_double * 1)(guard[1])
    for counters in (None, torch.full((n,), 0x5A5A5A5A, dtype=torch.int32, device=dev)):
        ws = torch.full((ws_bytes,), 0xA5, dtype=torch.uint8, device=dev)
        got_sq, got_err = torch.empty_like(sq), torch.empty_like(err)
        scale = torch.empty_like(cf.scale)
        nat.call("dpc_gram_clip_factors", nat.ptr(A), nat.ptr(G), B, T, din, dout,
                 nat.dtype_code(A.dtype), 1, 1.0, nat.SCALE_FIXED, 0.0, rel, abs_, None, 1, 1.0,
                 nat.ptr(got_sq), nat.ptr(got_err), nat.ptr(scale), None, None, None, None, None,
                 nat.ptr(ws), ws_bytes, nat.ptr(counters), 4 * n if counters is not None else 0,
                 nat.stream_handle(dev))
        assert torch.equal(got_sq, sq) and torch.equal(got_err, err)
        assert torch.equal(scale, cf.scale)
        assert counters is None or bool((counters == 0x5A5A5A5A).all())
