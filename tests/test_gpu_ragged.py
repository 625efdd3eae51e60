"""Layers off the usual shapes (GPU tests): token counts that no 64-row step
divides, widths that are not multiples of 8, operands that start at any element,
float32, few tiles over a long K, narrow layers, biases, small batches; clipped
sums, Gram norms and clip factors, one layer and several, and materialised leaves
of any alignment.  Through the package's wrappers and, where they hide the choice,
the C ABI."""

from __future__ import annotations

import ctypes

import pytest
import torch

from opake_amd import _native as nat
from opake_amd import ops
from opake_amd.clipping import _numerics as num
from opake_amd.clipping import guard_for_linear

pytestmark = pytest.mark.gpu


def _operands(B, T, din, dout, seed):
    g = torch.Generator().manual_seed(seed)
    A = torch.randn(B, T, din, generator=g).to(torch.bfloat16)
    G = (torch.randn(B, T, dout, generator=g) * 0.01 *
         torch.exp(torch.randn(B, 1, 1, generator=g))).to(torch.bfloat16)
    return A, G


def _factors(dev, A, G, C=1.0):
    sq, err = ops.gram_sqnorms(A, G, return_error=True)
    guard = guard_for_linear(A.dtype, A.shape[2], G.shape[2], False)
    return ops.clip_factors(sq, num.conservative_bound(C), [guard], err=err,
                            count_threshold=num.float32_of(C))


def _exact(A, G, scale):
    return sum(scale[b] * (G[b].double().t() @ A[b].double()) for b in range(A.shape[0]))


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm())


# Steps of 1, 2, 33, 63 and 65 rows; one and several tiles; split-K; padded
# rows of A, of G and of both, odd (value by value) and even output rows.
@pytest.mark.parametrize("B,T,din,dout", [
    (3, 2, 16, 8), (1, 33, 8, 264), (2, 63, 64, 72), (5, 65, 264, 256), (24, 97, 256, 520),
    (3, 64, 15, 24), (4, 100, 257, 1001), (2, 128, 1030, 9), (16, 130, 259, 250), (1, 7, 1, 3),
    # 1.5 GFLOP and more (below, layers on their own take the fp32 MFMA kernel): ragged steps,
    # padded A, G and both, T % 64 == 0 with padding, many K slices
    (24, 97, 520, 640), (16, 100, 1023, 511), (16, 64, 1000, 801), (100, 130, 248, 257)])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_clipped_sum_ragged(dev, B, T, din, dout, out):
    """fp32 sums of exact bf16 products: K = B T addends of one rounding each
    stay within K 2^-24 of the sum of magnitudes, at random signs far below
    1e-5 of the result; a bf16 output adds 2^-9 per entry."""
    A, G = _operands(B, T, din, dout, B * 1000 + T + din)
    A_d, G_d = A.to(dev), G.to(dev)
    cf = _factors(dev, A_d, G_d)
    w, _ = ops.clipped_sum(A_d, G_d, cf.scale[0], plan=cf.plan[0], out_dtype=out)
    want = _exact(A, G, cf.scale[0].cpu().double())
    tol = 1e-5 if out == torch.float32 else 2.0**-8
    assert _rel(w.cpu(), want) < tol
    if din % 8 == 0 and dout % 8 == 0:  # the bf16 kernel at any size
        m, = ops.clipped_sum_multi([A_d], [G_d], cf.scale[0], plan=cf.plan[0], out_dtype=out)
        assert _rel(m.cpu(), want) < tol


@pytest.mark.parametrize("T,din", [(65, 264), (100, 33)])
def test_clipped_sum_ragged_skips_a_nonfinite_neighbour(dev, T, din):
    """The rows past an example's end belong to the next example: NaN there
    (scale 0) must not reach the sum.  An example of the plan's slow list
    (a scale below 2^-64) sums as the others do."""
    A, G = _operands(4, T, din, 136, 5)
    G[1] = float("nan")
    A[1] = float("inf")
    G[2] = (G[2].float() * 1e19).to(torch.bfloat16)
    A_d, G_d = A.to(dev), G.to(dev)
    cf = _factors(dev, A_d, G_d)
    w, _ = ops.clipped_sum(A_d, G_d, cf.scale[0], plan=cf.plan[0], out_dtype=torch.float32)
    scale = cf.scale[0].cpu().double()
    assert scale[1] == 0 and 0 < scale[2] < 2.0**-64
    keep = [0, 2, 3]
    want = _exact(A[keep], G[keep], scale[keep])
    assert _rel(w.cpu(), want) < 1e-5
    if din % 8 == 0:
        # The bf16 kernel; an entry of the plan between its two lists is not read.
        plan = cf.plan[0].clone()
        words = plan.view(torch.int32)
        assert words[:2].tolist() == [3, 2]
        words[4 + 2] = 1 << 28
        m, = ops.clipped_sum_multi([A_d], [G_d], cf.scale[0], plan=plan, out_dtype=torch.float32)
        assert _rel(m.cpu(), want) < 1e-5


# fp32 MFMA kernel, even and odd rows; the bf16 kernel with and without padding.
@pytest.mark.parametrize("din,dout", [(264, 72), (33, 17), (3000, 1200), (2999, 1201)])
def test_clipped_sum_ragged_noise_matches_add_noise(dev, din, dout):
    A, G = _operands(3, 70, din, dout, 9)
    A_d, G_d = A.to(dev), G.to(dev)
    cf = _factors(dev, A_d, G_d)
    kw = dict(plan=cf.plan[0], normalize_by=2.0)
    spec = ops.NoiseSpec(sigma=0.5, mode=nat.NOISE_PHILOX, seed=77, leaf_id=3)
    plain, _ = ops.clipped_sum(A_d, G_d, cf.scale[0], **kw)
    noised, _ = ops.clipped_sum(A_d, G_d, cf.scale[0], noise=spec, **kw)
    assert torch.equal(noised, ops.add_noise(plain, 0.5, seed=77, leaf_id=3))


def test_clipped_sum_multi_ragged_matches_single_layers(dev):
    dims = [(256, 264), (320, 136), (8, 8)]
    ops_ = [_operands(3, 70, din, dout, 20 + din) for din, dout in dims]
    As, Gs = [a.to(dev) for a, _ in ops_], [g.to(dev) for _, g in ops_]
    cf = _factors(dev, As[0], Gs[0])
    kw = dict(plan=cf.plan[0], out_dtype=torch.float32)
    got = ops.clipped_sum_multi(As, Gs, cf.scale[0], **kw)
    for i, w in enumerate(got):
        assert torch.equal(w, ops.clipped_sum_multi([As[i]], [Gs[i]], cf.scale[0], **kw)[0])
        want = _exact(*ops_[i], cf.scale[0].cpu().double())
        assert _rel(w.cpu(), want) < 1e-5


# One call for several layers and each layer's own call without a workspace:
# small layers and large ones, more tiles than CUs, full and ragged steps; padded
# widths, one token and float32 go layer by layer.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,dims", [
    (3, 128, [(256, 264), (8, 8), (64, 520)]), (3, 70, [(256, 264), (8, 8), (4104, 264)]),
    (2, 64, [(4096, 2304), (520, 2304), (2304, 2304)]), (3, 70, [(256, 264), (33, 8)]),
    (40, 1, [(256, 264), (8, 8)])])
def test_clipped_sum_multi_equals_calls_without_a_workspace(dev, dtype, B, T, dims):
    pairs = [_operands(B, T, din, dout, din + dout) for din, dout in dims]
    As, Gs = [a.to(dev, dtype) for a, _ in pairs], [g.to(dev, dtype) for _, g in pairs]
    sq = (4 * torch.rand(B, dtype=torch.float64, generator=torch.Generator().manual_seed(B))).to(dev)
    cf = ops.clip_factors(sq, 1.0, [guard_for_linear(dtype, *dims[0], False)], count_threshold=1.0)
    n, code, seed = len(dims), nat.dtype_code(dtype), 77
    outs = [torch.empty(dout, din, device=dev) for din, dout in dims]
    vp, ci = ctypes.c_void_p * n, ctypes.c_int * n
    sigmas, leaves = [0.0] + [0.25] * (n - 1), list(range(n))
    nat.call("dpc_clipped_sum_multi", n, vp(*[a.data_ptr() for a in As]),
             vp(*[g.data_ptr() for g in Gs]), ci(*[d[0] for d in dims]), ci(*[d[1] for d in dims]),
             nat.ptr(cf.scale[0]), nat.ptr(cf.plan[0]), B, T, code, 2.0, nat.NOISE_PHILOX, None,
             seed, (ctypes.c_uint32 * n)(*leaves), (ctypes.c_double * n)(*sigmas),
             nat.dtype_code(torch.float32), vp(*[o.data_ptr() for o in outs]),
             nat.stream_handle(dev))
    for a, g, out, sigma, leaf in zip(As, Gs, outs, sigmas, leaves):
        one = torch.empty_like(out)
        nat.call("dpc_clipped_sum", nat.ptr(a), nat.ptr(g), nat.ptr(cf.scale[0]),
                 nat.ptr(cf.plan[0]), B, T, a.shape[2], g.shape[2], code, 2.0, nat.NOISE_PHILOX,
                 None, None, seed, leaf, 0, sigma, nat.dtype_code(torch.float32), nat.ptr(one), 0,
                 None, None, 0, nat.stream_handle(dev))
        assert torch.equal(out, one)


def _in_flat_buffer(t, first):
    """``t`` as a view of a flat buffer from element `first` on."""
    flat = torch.empty(t.numel() + first, dtype=t.dtype, device=t.device)
    view = flat[first:].view(t.shape)
    view.copy_(t)
    return view


# Views that start 2, 4 and 8 bytes past a 16-byte boundary: small and large
# layers, full and ragged steps, padded widths, one token, a bias; each operand.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,din,dout", [(3, 70, 64, 72), (24, 97, 520, 640), (24, 128, 520, 640),
                                          (16, 100, 1023, 511), (40, 1, 64, 72), (8, 256, 64, 136)])
def test_operands_at_any_element(dev, dtype, B, T, din, dout):
    A, G = (x.to(dtype) for x in _operands(B, T, din, dout, B + T))
    A_d, G_d = A.to(dev), G.to(dev)
    guards = [guard_for_linear(dtype, din, dout, True)]

    def outputs(a, g):
        sq, err, cf = ops.gram_clip_factors(a, g, 1.0, guards, with_bias=True, count_threshold=1.0)
        kw = dict(plan=cf.plan[0], out_dtype=torch.float32)
        w, b = ops.clipped_sum(a, g, cf.scale[0], with_bias=True, **kw)
        lay = ops.SegmentLayout([[T] * B], dev)
        flat = [a.view(B * T, din)], [g.view(B * T, dout)], lay
        return [sq, err, cf.scale, w, b, *ops.gram_sqnorms(a, g, with_bias=True, return_error=True),
                *ops.gram_sqnorms_multi([a, a], [g, g], return_error=True),
                *ops.clipped_sum_multi([a, a], [g, g], cf.scale[0], **kw),
                *ops.grouped_gram_sqnorms(*flat, return_error=True),
                ops.grouped_clipped_sum(*flat, cf.scale[:1], out_dtype=torch.float32)]

    want = outputs(A_d, G_d)
    # Copied to the boundary: the same bits.  Else the bias columns are summed in other
    # row groups, T addends in fp32, and the clip factor follows.
    rtol = 0 if dtype == torch.bfloat16 and din % 8 == 0 else T * 2.0**-23
    for fa, fg in ((1, 0), (0, 2), (4, 1)):
        a, g = _in_flat_buffer(A_d, fa), _in_flat_buffer(G_d, fg)
        for x, y in zip(outputs(a, g), want):
            torch.testing.assert_close(x, y, rtol=rtol, atol=rtol * float(y.abs().max()))
    # The C entry points take them as they are.
    cf = ops.clip_factors(want[0], 1.0, guards, err=want[1], count_threshold=1.0)
    lib, code, f32 = nat.load(), nat.dtype_code(dtype), nat.dtype_code(torch.float32)
    a, g = _in_flat_buffer(A_d, 1), _in_flat_buffer(G_d, 1)
    exact = _exact(A, G, cf.scale[0].cpu().double())
    full = lib.dpc_clipped_sum_workspace_bytes(B, T, din, dout, code)
    for ws_bytes in (full, 0):
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev) if ws_bytes else None
        for plan in (cf.plan[0], None):
            w = torch.empty(dout, din, device=dev)
            nat.call("dpc_clipped_sum", nat.ptr(a), nat.ptr(g), nat.ptr(cf.scale[0]), nat.ptr(plan),
                     B, T, din, dout, code, 1.0, nat.NOISE_NONE, None, None, 0, 0, 0, 0.0, f32,
                     nat.ptr(w), 0, None, nat.ptr(ws), ws_bytes, nat.stream_handle(dev))
            assert _rel(w.cpu(), exact) < 1e-5
    outs = [torch.empty(dout, din, device=dev) for _ in range(2)]
    vp, ci = ctypes.c_void_p * 2, ctypes.c_int * 2
    nat.call("dpc_clipped_sum_multi", 2, vp(A_d.data_ptr(), a.data_ptr()),
             vp(G_d.data_ptr(), g.data_ptr()), ci(din, din), ci(dout, dout),
             nat.ptr(cf.scale[0]), nat.ptr(cf.plan[0]), B, T, code, 1.0, nat.NOISE_NONE, None, 0,
             None, (ctypes.c_double * 2)(), f32, vp(*[o.data_ptr() for o in outs]),
             nat.stream_handle(dev))
    for w in outs:
        assert _rel(w.cpu(), exact) < 1e-5


# Row groups of the bias column sums: fewer rows than groups, one more than a
# full turn of them, the unrolled part and its remainder; 16-byte rows and
# rows of any alignment; one and several column blocks and slots, and a
# workspace without the slots.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,dout", [(3, 2, 8), (2, 7, 136), (2, 9, 1001), (40, 33, 264),
                                      (2, 129, 130), (1, 300, 4104)])
def test_bias_norm_and_sum(dev, dtype, B, T, dout):
    g = torch.Generator().manual_seed(B + T + dout)
    A = torch.randn(B, T, 16, generator=g).to(dtype)
    G = (torch.randn(B, T, dout, generator=g) * 0.01 + 0.002).to(dtype)
    cols = G.double().sum(dim=1)
    exact_w = torch.stack([(G[b].double().t() @ A[b].double()).square().sum() for b in range(B)])
    A_d, G_d = A.to(dev), G.to(dev)
    sq, err = ops.gram_sqnorms(A_d, G_d, with_bias=True, return_error=True)
    w_sq, w_err = ops.gram_sqnorms(A_d, G_d, return_error=True)
    want = exact_w + cols.square().sum(dim=1)
    # fp32 column sums of T addends: T 2^-24 of the magnitudes, twice in a
    # square; the weight part is the bias-free call's own.
    tol = 4 * T * 2.0**-24 * G.double().abs().sum(dim=1).square().sum(dim=1)
    bias_sq = (sq - w_sq).cpu()
    assert ((bias_sq - cols.square().sum(dim=1)).abs() <= tol + 1e-9 * want).all()
    assert (err >= w_err).all()
    if (-(-T // 128)) % 2:
        # The smallest workspace: the records of the 64-row tile pairs and two words
        # per example (the workspace query adds finer tiles and shared columns).
        pairs = (-(-T // 64)) * (-(-T // 64) + 1) // 2
        small = -(-(pairs * 12 + 2) * B * 8 // 256) * 256
        ws = torch.empty(small, dtype=torch.uint8, device=dev)
        sq1 = torch.empty(B, dtype=torch.float64, device=dev)
        nat.call("dpc_gram_sqnorms", nat.ptr(A_d), nat.ptr(G_d), B, T, 16, dout,
                 nat.dtype_code(dtype), 1, 0, nat.ptr(sq1), None, nat.ptr(ws), small,
                 nat.stream_handle(dev))
        torch.testing.assert_close(sq1, sq, rtol=1e-12, atol=0)
    scale = torch.rand(B, generator=g).to(dev)
    scale[0] = 0.0 if B > 1 else 0.5
    _, b = ops.clipped_sum(A_d, G_d, scale, with_bias=True, out_dtype=torch.float32)
    want_b = scale.cpu().double() @ cols
    bound = (T + B) * 2.0**-23 * (scale.cpu().double() @ G.double().abs().sum(dim=1))
    assert ((b.cpu().double() - want_b).abs() <= bound).all()


# One workgroup of bias columns and several, an odd last column; the sums behind
# them split over K (fp32 MFMA with din 16; bf16 MFMA with padded rows) and not.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,dout", [(40, 264), (40, 1001), (5, 513)])
def test_bias_finish_with_the_split_sums(dev, dtype, T, dout):
    """The bias finished in the split-K sum's launch and in one of its own: the
    same bits, with noise and normalisation."""
    g = torch.Generator().manual_seed(T + dout)
    B, bias = 40, []
    G = (torch.randn(B, T, dout, generator=g) * 0.01).to(dtype).to(dev)
    sq = (4 * torch.rand(B, dtype=torch.float64, generator=g)).to(dev)
    cf = ops.clip_factors(sq, 1.0, [guard_for_linear(dtype, 16, dout, True)], count_threshold=1.0)
    scale, plan = cf.scale[0], cf.plan[0]
    for din in (16, 1001, 8192):
        A = torch.randn(B, T, din, generator=g).to(dtype).to(dev)
        spec = ops.NoiseSpec(sigma=0.5, seed=77, leaf_id=3, bias_leaf_id=4)
        _, b = ops.clipped_sum(A, G, scale, plan=plan, with_bias=True, noise=spec, normalize_by=2.0)
        _, plain = ops.clipped_sum(A, G, scale, plan=plan, with_bias=True, normalize_by=2.0)
        assert torch.equal(b, ops.add_noise(plain, 0.5, seed=77, leaf_id=4))
        bias.append(b)
    assert torch.equal(bias[0], bias[1]) and torch.equal(bias[0], bias[2])


# The fp64 Gram paths.  FMA kernel: narrow layers, at long sequences one wide
# operand beside a narrow one.  MFMA kernel: one, two and several 32-row tiles with
# ragged last ones, depths around the 32-deep chunks, rows that 16-byte loads do
# not take, din != dout both ways; 64-row tiles (many tile pairs of shallow layers, more
# than 2048 rows); 16.8 million tile pairs, more than one launch holds (2^32 threads).
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,din,dout", [
    (2, 2, 4, 8), (3, 31, 33, 9), (2, 32, 32, 31), (4, 65, 100, 36), (1, 130, 7, 260),
    (2, 257, 64, 65), (1024, 40, 12, 20), (110, 200, 33, 68),
    (2040, 4096, 4, 4),
    (5, 200, 29, 31), (5, 200, 30, 31), (100, 200, 43, 43), (100, 200, 44, 43), (100, 300, 52, 53),
    (2, 1024, 63, 100), (2, 1100, 65, 127), (2, 2048, 31, 300), (2, 2050, 33, 900), (9, 1000, 131, 335),
    (520, 16256, 65, 65)])
def test_gram_f64(dev, dtype, B, T, din, dout):
    """Exact products in fp64: the error is within the kernel's own bound, and
    far below what fp32 sums would leave (2^-24)."""
    g = torch.Generator().manual_seed(B + T + din)
    A = torch.randn(B, T, din, generator=g).to(dtype).to(dev)
    G = torch.randn(B, T, dout, generator=g).to(dtype).to(dev)
    if dtype == torch.bfloat16 and din % 8 == 0 and dout % 8 == 0:
        pytest.skip("takes the bf16 MFMA kernels")
    sq, err = ops.gram_sqnorms(A, G, return_error=True)
    grads = torch.stack([G[b].double().t() @ A[b].double() for b in range(B)])
    want = grads.square().sum(dim=(1, 2))
    # The reference's own fp64 sums: T products per entry, at most 2^-53 each.
    own = (T + 8) * 2.0**-52 * (G.double().abs().transpose(1, 2).contiguous()
                                @ A.double().abs().contiguous()).square().sum(dim=(1, 2))
    assert ((sq - want).abs() <= err + own).all()
    assert ((sq - want).abs() <= 1e-11 * want).all()
    # The bound's own size: by Cauchy-Schwarz over its tiles it is at most
    # (gamma_A + gamma_G + (T^2 + 256) 2^-52) sum |a|^2 sum |g|^2, with gamma of
    # a chain of d products padded to 16.
    gammas = sum(1.125 * (-(-d // 16) * 16) * 2.0**-52 for d in (din, dout))
    rows = A.double().square().sum(dim=(1, 2)) * G.double().square().sum(dim=(1, 2))
    assert (err <= 1.001 * (gammas + (T * T + 256) * 2.0**-52) * rows).all()


# Layers in one call, layer by layer off the bf16 MFMA path: FMA kernel, 32- and
# 64-row tiles, each as in the layer's own call.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T", [(16, 256), (6, 200), (3, 1100)])
def test_gram_multi_matches_consecutive_calls(dev, dtype, B, T):
    g = torch.Generator().manual_seed(B + T)
    dims = [(65, 33), (9, 20), (260, 516), (100, 601)]
    As = [torch.randn(B, T, din, generator=g).to(dtype).to(dev) for din, _ in dims]
    Gs = [torch.randn(B, T, dout, generator=g).to(dtype).to(dev) for _, dout in dims]
    want, want_err = ops.gram_sqnorms(As[0], Gs[0], return_error=True)
    for a, x in zip(As[1:], Gs[1:]):
        ops.gram_sqnorms(a, x, out=want, err=want_err)
    got, err = ops.gram_sqnorms_multi(As, Gs, return_error=True)
    assert torch.equal(got, want) and torch.equal(err, want_err)


def _kernels(fn):
    fn()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    cuda = torch.autograd.DeviceType.CUDA
    return [e.name for e in prof.events() if e.device_type == cuda]


# Narrow layers, where the fp64 MFMA kernel takes up to five times as long, keep the
# FMA kernel; deep ones and single tiles do not.
@pytest.mark.parametrize("B,T,din,dout,kernel", [
    (32, 1024, 12, 12, "gram_generic_kernel"), (4, 4096, 12, 300, "gram_generic_kernel"),
    (66, 312, 27, 59, "gram_generic_kernel"), (16, 256, 516, 516, "gram_f64_kernel"),
    (156, 30, 39, 10, "gram_f64_kernel")])
def test_gram_f64_kernel_of_narrow_layers(dev, B, T, din, dout, kernel):
    A = torch.randn(B, T, din, device=dev)
    G = torch.randn(B, T, dout, device=dev)
    assert any(kernel in n for n in _kernels(lambda: ops.gram_sqnorms(A, G)))


# The fp32 MFMA path: chunks of 16 rows and their remainders, one token per
# example (16 examples a chunk), 64-column tiles and their edges at any
# alignment, one and several splits; a zero-scale example that holds NaN.
@pytest.mark.parametrize("B,T,din,dout", [
    (2, 2, 1, 1), (3, 5, 33, 17), (7, 19, 100, 67), (16, 130, 64, 64), (2, 300, 257, 66),
    (40, 33, 512, 130), (2, 1, 7, 5), (40, 1, 65, 10), (300, 1, 64, 130), (1030, 1, 20, 64)])
def test_clipped_sum_fp32(dev, B, T, din, dout):
    g = torch.Generator().manual_seed(B + T + din)
    A = torch.randn(B, T, din, generator=g)
    G = torch.randn(B, T, dout, generator=g)
    scale = torch.rand(B, generator=g) * torch.exp(3 * torch.randn(B, generator=g))
    G[B // 2] = float("nan")
    scale[B // 2] = 0.0
    A_d, G_d, s_d = A.to(dev), G.to(dev), scale.to(dev)
    got, _ = ops.clipped_sum(A_d, G_d, s_d)
    keep = torch.arange(B) != B // 2
    s64, A64, G64 = scale[keep].double(), A[keep].double(), G[keep].double()
    want = _exact(A64, G64, s64)
    # Sums of K = B T products in fp32, each partial sum rounded once (2^-24),
    # the scaled operand or accumulator twice more.
    mag = _exact(A64.abs(), G64.abs(), s64)
    assert ((got.cpu().double() - want).abs() <= (B * T + 3) * 2.0**-24 * mag).all()
    assert _rel(got.cpu(), want) < 2e-6
    spec = ops.NoiseSpec(sigma=0.5, mode=nat.NOISE_PHILOX, seed=7, leaf_id=2)
    half, _ = ops.clipped_sum(A_d, G_d, s_d, normalize_by=3.0, out_dtype=torch.bfloat16)
    noised, _ = ops.clipped_sum(A_d, G_d, s_d, normalize_by=3.0, out_dtype=torch.bfloat16,
                                noise=spec)
    assert torch.equal(noised, ops.add_noise(half, 0.5, seed=7, leaf_id=2))


# Materialised leaves whose rows start at any element boundary, leaves shorter
# than 8 elements, tiles and waves that a leaf ends in, batches that 8 does not
# divide; fp16 beside bf16 and fp32; diagnostics and the second moment.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B", [1, 7, 17])
@pytest.mark.parametrize("out", [None, torch.float32])
def test_leaves_unaligned_match_oracle(dev, dtype, B, out):
    from opake_amd.clipping import leaves_clip_sum
    from oracle import clip_oracle

    g = torch.Generator().manual_seed(B)
    shapes = [(1,), (7,), (9,), (511,), (513,), (2047,), (2049,), (3, 683), (4096,), (5, 1031)]
    leaves = [(torch.randn(B, *s, generator=g) * 0.05).to(dtype) for s in shapes]
    leaves[3][0, 5] = float("nan")
    leaves[6][B - 1, 2048] = float("inf")
    res = leaves_clip_sum([x.to(dev) for x in leaves], 1.0, with_postsq=True, second_moment=True,
                          sum_dtypes=None if out is None else {dtype: (torch.float32, out)})
    want = clip_oracle.stream_clip_and_sum(leaves, clip_oracle.conservative_bound(1.0),
                                           second_moment=True,
                                           reduce_dtype=None if out is None else {dtype: out})
    torch.testing.assert_close(res.norms.cpu().double(), want.norms.double(), rtol=1e-6, atol=0)
    scale = res.scales[dtype][0].cpu()
    for got, sq, x in zip(res.reduced, res.squared, leaves):
        # The reference's arithmetic on the device's scales: one rounding per
        # product, fp32 sums in example order -- the same bits.
        clean = torch.nan_to_num(x.float(), nan=0.0, posinf=0.0, neginf=0.0)
        prod = clean * scale.view(B, *[1] * (x.dim() - 1))
        stored = prod.to(dtype)
        tiny = torch.finfo(dtype).smallest_normal
        up = (stored.float().abs() <= tiny) & (stored.float().abs() > prod.abs())
        if dtype != torch.float32:
            stored = torch.where(up, torch.zeros_like(stored), stored)
        acc, acc2 = torch.zeros(x.shape[1:]), torch.zeros(x.shape[1:])
        for b in range(B):
            acc = acc + stored[b].float()
            acc2 = acc2 + (stored[b].float() ** 2).to(dtype).float()
        assert torch.equal(got.cpu(), acc.to(out or dtype))
        assert torch.equal(sq.cpu(), acc2.to(out or dtype))
    post = torch.zeros(B, dtype=torch.float64)
    for x in leaves:
        clean = torch.nan_to_num(x.float(), nan=0.0, posinf=0.0, neginf=0.0)
        s = (clean * scale.view(B, *[1] * (x.dim() - 1))).to(dtype).double()
        post += (s.reshape(B, -1) ** 2).sum(dim=1)
    # fp32 sums of 512 squares per wave (fp64 for fp16), then fp64.
    torch.testing.assert_close(res.post_sq.cpu().double(), post, rtol=1e-4 * 2**-4, atol=0)


# Norms and clip factors: finished together for up to 32 examples (one and two
# a wave) of few records, by two launches past that; a bias inside the one-launch path (an even
# number of 128-row blocks) and beside it; call after call on one counter buffer.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T", [(1, 24), (16, 40), (17, 70), (32, 33), (33, 20), (9, 200), (40, 256),
                                 (16, 1152), (32, 1152), (32, 1408)])
@pytest.mark.parametrize("bias", [False, True])
def test_clip_factors_with_the_norms(dev, dtype, B, T, bias):
    A, G = (x.to(dev, dtype) for x in _operands(B, T, 64, 264, B + T))
    G[B // 2, 0, 0] = float("nan")
    guards = [guard_for_linear(dtype, 64, 264, bias)]
    kw = dict(with_bias=bias)
    for _ in range(2):
        sq, err, cf = ops.gram_clip_factors(A, G, 1.0, guards, count_threshold=1.0, **kw)
        wsq, werr = ops.gram_sqnorms(A, G, return_error=True, **kw)
        want = ops.clip_factors(wsq, 1.0, guards, err=werr, count_threshold=1.0)
        for x, y in ((sq, wsq), (err, werr), (cf.scale, want.scale), (cf.norms, want.norms),
                     (cf.nclipped, want.nclipped)):
            assert torch.equal(torch.nan_to_num(x, nan=-1.0), torch.nan_to_num(y, nan=-1.0))
        n = int(cf.plan[0].view(torch.int32)[0])
        assert n == B - 1
        assert torch.equal(cf.plan[0].view(torch.int32)[:4 + n][:2],
                           want.plan[0].view(torch.int32)[:2])
        assert torch.equal(cf.plan[0].view(torch.int32)[4:4 + n],
                           want.plan[0].view(torch.int32)[4:4 + n])


def test_clipped_sum_multi_few_tiles_long_k(dev):
    """Few output tiles and a long K: the layers' own split-K calls, with noise
    tensors of any strides, noise specs without noise, and none at all."""
    dims = [(64, 264), (520, 256), (64, 72)]
    pairs = [_operands(40, 130, din, dout, din + dout) for din, dout in dims]
    As, Gs = [a.to(dev) for a, _ in pairs], [g.to(dev) for _, g in pairs]
    cf = _factors(dev, As[0], Gs[0])
    z = torch.randn(64, 264, device=dev).t()
    noises = [ops.NoiseSpec(0.5, ops.nat.NOISE_INJECTED, noise=z),
              ops.NoiseSpec(0.0, ops.nat.NOISE_INJECTED), None]
    kw = dict(plan=cf.plan[0], out_dtype=torch.float32)
    got = ops.clipped_sum_multi(As, Gs, cf.scale[0], noises=noises, **kw)
    for w, a, g, pair, noise in zip(got, As, Gs, pairs, (0.5 * z, 0, 0)):
        assert torch.equal(w, ops.clipped_sum(a, g, cf.scale[0], **kw)[0] + noise)
        assert _rel((w - noise).cpu(), _exact(*pair, cf.scale[0].cpu().double())) < 1e-5


# Many short examples: a shared launch would walk a nearly empty 64-row step for each.
@pytest.mark.parametrize("B,T,own", [(230, 6, True), (150, 6, False)])
def test_short_examples_of_small_layers_take_their_own_calls(dev, B, T, own):
    pairs = [_operands(B, T, 24, 48, i) for i in range(14)]
    As, Gs = [a.to(dev) for a, _ in pairs], [g.to(dev) for _, g in pairs]
    cf = _factors(dev, As[0], Gs[0])
    kw = dict(plan=cf.plan[0], out_dtype=torch.float32)
    names = _kernels(lambda: ops.clipped_sum_multi(As, Gs, cf.scale[0], **kw))
    assert any("clipped_sum_bf16_kernel" in n for n in names) != own
    for w, pair in zip(ops.clipped_sum_multi(As, Gs, cf.scale[0], **kw), pairs):
        assert _rel(w.cpu(), _exact(*pair, cf.scale[0].cpu().double())) < 1e-5


# bf16 tile pairs of 128 rows: 45 and 66 records an example.
@pytest.mark.parametrize("B,T,one", [(32, 1152, True), (16, 1408, True), (32, 1408, False)])
def test_one_workgroup_finishes_few_records_only(dev, B, T, one):
    A, G = (x.to(dev) for x in _operands(B, T, 16, 8, 1))
    guards = [guard_for_linear(torch.bfloat16, 16, 8, False)]
    names = _kernels(lambda: ops.gram_clip_factors(A, G, 1.0, guards, count_threshold=1.0))
    assert any("gram_finish_clip_kernel" in n for n in names) == one
