"""GPU: the PyTorch modules (reference python/forge/nn/linear.py:115-254) against the oracle.

QuantizedLinear / SparseLinear: weight quantization formula, forward bit-exact to the oracle's
composition (per-token quantize -> INT32 GEMM on the (pruned) weights -> dequant epilogue),
state_dict round trip, QuantizedLinear's backward (input and bias gradients through the
dequantized FP16 weight), and the w_meta conversion to and from the reference's row-major words
(oracle pack_metadata_ref, pack_metadata.cu:23-29)."""
import numpy as np
import pytest

from helpers import fp16_normal, int8_uniform, say, to_dev, to_host

pytestmark = pytest.mark.gpu


def _np_weight_quant(w32):
    """The oracle's restatement of linear.py:168-173 (pinned to the reference's torch
    expression in test_oracle.py)."""
    from oracle import oracle
    q, s16, _ = oracle.quantize_weight_rows(w32)
    return q, s16


@pytest.mark.parametrize("M,K,N,bias", [(7, 256, 96, True), (64, 1024, 320, False), (300, 512, 200, True)])
def test_quantized_linear(dev, orc, M, K, N, bias):
    import torch
    from forge_amd.nn import QuantizedLinear
    rng = np.random.default_rng(M + K + N)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    x = fp16_normal(rng, (M, K))
    say(f"QuantizedLinear M={M} K={K} N={N}")
    m = QuantizedLinear(K, N, bias=bias).to(dev)
    m.quantize_weight(torch.from_numpy(w).to(dev))
    q, s = _np_weight_quant(w)
    assert np.array_equal(to_host(m.w_int8), q)
    assert np.array_equal(to_host(m.w_scale).view(np.uint16), s.view(np.uint16))
    b = None
    if bias:
        b = (rng.standard_normal(N) * 0.1).astype(np.float16)
        m.bias.data.copy_(torch.from_numpy(b).to(dev))
    y = to_host(m(to_dev(x, dev)))
    ref, _, _ = orc.linear(x, q, s, b)
    assert np.array_equal(y.view(np.uint16), ref.view(np.uint16))
    # state_dict round trip into a fresh module
    m2 = QuantizedLinear(K, N, bias=bias).to(dev)
    m2.load_state_dict(m.state_dict())
    assert np.array_equal(to_host(m2(to_dev(x, dev))).view(np.uint16), ref.view(np.uint16))


def test_quantized_linear_backward(dev):
    import torch
    from forge_amd.nn import QuantizedLinear
    rng = np.random.default_rng(5)
    M, K, N = 32, 256, 64
    m = QuantizedLinear(K, N).to(dev)
    m.quantize_weight(torch.from_numpy((rng.standard_normal((N, K)) * 0.05).astype(np.float32)).to(dev))
    x = to_dev(fp16_normal(rng, (M, K)), dev).requires_grad_(True)
    say("QuantizedLinear backward")
    y = m(x)
    g = torch.from_numpy(fp16_normal(rng, (M, N))).to(dev)
    y.backward(g)
    w16 = (m.w_int8.float() * m.w_scale.float().unsqueeze(1)).cpu()
    gx_ref = g.float().cpu() @ w16
    assert x.grad.shape == (M, K) and x.grad.dtype == torch.float16
    assert torch.allclose(x.grad.float().cpu(), gx_ref, rtol=2e-2, atol=2e-2)
    assert torch.allclose(m.bias.grad.float().cpu(), g.float().sum(0).cpu(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("M,K,N", [(1, 16, 8), (17, 100, 70), (513, 588, 1001), (2048, 256, 512), (70, 64, 65), (40, 20, 3)])
def test_linear_backward_passes(dev, M, K, N):
    """The backward's own kernels at ragged sizes. The FP16 weight has the bits of the torch
    expression; the column sums, in FP32 over M terms, are within M 2^-24 sum|g| of the FP64 ones
    before the rounding to FP16 (half an ulp, 2^-11); the gradients equal those through the torch
    operators (taken with create_graph) to the FP16 rounding of a sum in another order."""
    import torch
    from forge_amd import ops
    from forge_amd.nn import QuantizedLinear
    rng = np.random.default_rng(M + K + N)
    w = to_dev(int8_uniform(rng, (N, K)), dev)
    ws = to_dev(rng.uniform(1e-3, 1e-2, N).astype(np.float16), dev)
    g = to_dev(fp16_normal(rng, (M, N)), dev)
    say(f"linear backward passes M={M} K={K} N={N}")
    want = (w.to(torch.float16) * ws.unsqueeze(1)).t().contiguous()
    w16, gb = ops.int8_linear_backward_prep(w, ws, g, N >= 8)
    assert np.array_equal(to_host(w16.t()).view(np.uint16), to_host(want).view(np.uint16))
    if N >= 8:
        ref, bound = g.double().sum(0), g.double().abs().sum(0) * (M * 2.0 ** -24)
        err = (gb.double() - ref).abs()
        assert bool((err <= bound + (ref.abs() + bound) * 2.0 ** -11 + 2.0 ** -25).all())
    m = QuantizedLinear(K, N).to(dev)
    m.w_int8.copy_(w)
    m.w_scale.data.copy_(ws)
    x = to_dev(fp16_normal(rng, (M, K)), dev).requires_grad_(True)
    gx, gb = torch.autograd.grad(m(x), (x, m.bias), g)
    gx2, gb2 = torch.autograd.grad(m(x), (x, m.bias), g, create_graph=True)
    scale = float((g.float().abs() @ want.float().abs().t()).max())
    assert float((gx.float() - gx2.float()).abs().max()) <= scale * (N * 2.0 ** -24 + 2.0 ** -10)
    assert float((gb.float() - gb2.float()).abs().max()) <= float(g.float().abs().sum(0).max()) * (M * 2.0 ** -24 + 2.0 ** -10)


@pytest.mark.parametrize("N,K", [(65535 * 64 + 70, 3), (65536 * 64 + 64, 16), (9, 65536 * 64 + 17)])
def test_linear_backward_many_tiles(dev, N, K):
    """More than 65535 rows or columns of 64 x 64 weight tiles, and more tiles than one grid dimension."""
    import torch
    from forge_amd import ops
    gen = torch.Generator(device=dev).manual_seed(N)
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=dev, generator=gen)
    ws = (torch.rand(N, device=dev, generator=gen) * 0.01 + 0.001).half()
    g = torch.ones((1, N), dtype=torch.float16, device=dev)
    say(f"linear backward many tiles N={N} K={K}")
    w16, gb = ops.int8_linear_backward_prep(w, ws, g, True)
    assert torch.equal(w16, w.half() * ws[:, None]) and torch.equal(gb, g[0])


def test_linear_backward_empty(dev):
    """No columns of the weight: the bias gradient is still the column sum. No tokens: it is zero. Buffers
    of both sizes are filled and freed first, so that fresh memory is not zero by chance."""
    import torch
    from forge_amd import ops
    from forge_amd.nn import QuantizedLinear
    N = 24
    g = torch.arange(5 * N, device=dev).reshape(5, N).half()
    ws = torch.ones(N, dtype=torch.float16, device=dev)
    say("linear backward empty")

    def stale():
        del_me = [torch.full((n,), 7.0, dtype=torch.float16, device=dev) for n in (N, 64 * N)]
        del del_me

    stale()
    w16, gb = ops.int8_linear_backward_prep(torch.empty((N, 0), dtype=torch.int8, device=dev), ws, g, True)
    assert w16.shape == (N, 0) and torch.equal(gb, g.sum(0))
    stale()
    w = torch.ones((N, 32), dtype=torch.int8, device=dev)
    w16, gb = ops.int8_linear_backward_prep(w, ws, g[:0], True)
    assert torch.equal(w16, w.half()) and torch.equal(gb, torch.zeros_like(gb))
    stale()
    m = QuantizedLinear(0, N).to(dev)
    x = torch.empty((5, 0), dtype=torch.float16, device=dev, requires_grad=True)
    gx, gb = torch.autograd.grad(m(x), (x, m.bias), g)
    assert gx.shape == (5, 0) and torch.equal(gb, g.sum(0))


def test_linear_backward_transformed(dev):
    """Gradients that are batched, traced, dual or behind saved-tensor hooks equal those through the
    torch operators: the passes on raw addresses stand aside. Gradients of one token and small
    integers, so every sum is exact and the values are compared exactly."""
    import torch
    import torch.autograd.forward_ad as fwAD
    from torch.fx.experimental.proxy_tensor import make_fx
    from forge_amd.nn import QuantizedLinear
    K, N = 32, 16
    rng = np.random.default_rng(5)
    m = QuantizedLinear(K, N).to(dev)
    m.w_int8.copy_(to_dev(rng.integers(-8, 9, (N, K)).astype(np.int8), dev))
    m.w_scale.data.copy_(to_dev(rng.choice([0.5, 0.25, 1.0], N).astype(np.float16), dev))
    x = to_dev(fp16_normal(rng, (1, K)), dev).requires_grad_(True)
    w = (m.w_int8.half() * m.w_scale.detach()[:, None])
    g = torch.from_numpy(rng.integers(-3, 4, (3, 1, N)).astype(np.float16)).to(dev)
    say("linear backward transformed")
    y = m(x)
    gx, gb = torch.autograd.grad(y, (x, m.bias), g, is_grads_batched=True, retain_graph=True)
    assert torch.equal(gx, (g.float() @ w.float()).half()) and torch.equal(gb, g[:, 0])
    jac = torch.autograd.functional.jacobian(m, x.detach(), vectorize=True)
    assert torch.equal(jac[0, :, 0], w)
    with fwAD.dual_level():
        r = torch.autograd.grad(y, (x, m.bias), fwAD.make_dual(g[0], g[1]), retain_graph=True)
        tx, tb = (fwAD.unpack_dual(t).tangent for t in r)
    assert torch.equal(tx, (g[1].float() @ w.float()).half()) and torch.equal(tb, g[1, 0])
    traced = make_fx(lambda t: torch.autograd.grad(y, (x, m.bias), t, retain_graph=True))(g[0])
    for t in (g[0], g[1]):
        gx, gb = traced(t)
        assert torch.equal(gx, (t.float() @ w.float()).half()) and torch.equal(gb, t[0])
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.t().contiguous().t() if t.dim() == 2 else
                                                  torch.stack([t, t], 1)[:, 0]):
        y = m(x)
    gx, gb = torch.autograd.grad(y, (x, m.bias), g[2])
    assert torch.equal(gx, (g[2].float() @ w.float()).half()) and torch.equal(gb, g[2, 0])


@pytest.mark.parametrize("M,K,N,bias", [(5, 256, 64, True), (200, 1280, 320, True), (129, 512, 96, False)])
def test_sparse_linear(dev, orc, M, K, N, bias):
    import torch
    from forge_amd.nn import SparseLinear
    rng = np.random.default_rng(M * 3 + K + N)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    x = fp16_normal(rng, (M, K))
    say(f"SparseLinear M={M} K={K} N={N}")
    m = SparseLinear(K, N, bias=bias).to(dev)
    m.from_dense_weight(torch.from_numpy(w).to(dev))
    q, s = _np_weight_quant(w)
    comp, raw = orc.prune_compress_24(q)
    assert np.array_equal(to_host(m.W_comp), comp)
    assert np.array_equal(to_host(m.w_meta).reshape(-1).view(np.uint32),
                          orc.pack_metadata_gfx950(raw, N, K).reshape(-1))
    b = None
    if bias:
        b = (rng.standard_normal(N) * 0.1).astype(np.float16)
        m.bias.data.copy_(torch.from_numpy(b).to(dev))
    y = to_host(m(to_dev(x, dev)))
    qx, sx = orc.quantize_rows(x)
    ref = orc.dequant_epilogue(orc.sparse_gemm_s32(comp, qx, raw, N, K), sx, s, b)
    assert np.array_equal(y.view(np.uint16), ref.view(np.uint16))
    m2 = SparseLinear(K, N, bias=bias).to(dev)
    m2.load_state_dict(m.state_dict())
    assert np.array_equal(to_host(m2(to_dev(x, dev))).view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("N,K", [(16, 64), (48, 1024), (320, 1280)])
def test_w_meta_conversion(dev, orc, N, K):
    import torch
    from forge_amd.nn import w_meta_from_reference, w_meta_to_reference
    rng = np.random.default_rng(N + K)
    q = rng.integers(-127, 128, (N, K)).astype(np.int8)
    _, raw = orc.prune_compress_24(q)
    ref_words = orc.pack_metadata_ref(raw, N, K)                 # reference layout (uint32)
    gfx_words = orc.pack_metadata_gfx950(raw, N, K).reshape(N, K // 32)
    say(f"w_meta conversion N={N} K={K}")
    got = w_meta_from_reference(to_dev(ref_words.view(np.int32), dev))
    assert np.array_equal(to_host(got).view(np.uint32), gfx_words)
    back = w_meta_to_reference(to_dev(gfx_words.view(np.int32), dev))
    assert np.array_equal(to_host(back).view(np.uint32), ref_words)


@pytest.mark.parametrize("M,K,N", [(9, 512, 64), (300, 1280, 320)])
def test_sparse_linear_loads_reference_state_dict(dev, orc, M, K, N):
    """A state_dict laid out as the reference's SparseLinear saves it (w_meta in its row-major
    word order, module version 1) loads into a module on the device and computes the oracle's
    outputs for those weights."""
    import collections
    import torch
    from forge_amd.nn import SparseLinear
    rng = np.random.default_rng(M + 2 * K + N)
    q = rng.integers(-127, 128, (N, K)).astype(np.int8)
    comp, raw = orc.prune_compress_24(q)
    ws = rng.uniform(1e-3, 1e-2, N).astype(np.float16)
    b = (rng.standard_normal(N) * 0.1).astype(np.float16)
    sd = collections.OrderedDict()
    sd["W_comp"] = torch.from_numpy(comp)
    sd["w_meta"] = torch.from_numpy(orc.pack_metadata_ref(raw, N, K).view(np.int32).copy())
    sd["w_scale"] = torch.from_numpy(ws)
    sd["bias"] = torch.from_numpy(b)
    sd._metadata = collections.OrderedDict({"": {"version": 1}})
    x = fp16_normal(rng, (M, K))
    say(f"SparseLinear reference state_dict M={M} K={K} N={N}")
    m = SparseLinear(K, N).to(dev)
    m.load_state_dict(sd)
    y = to_host(m(to_dev(x, dev)))
    qx, sx = orc.quantize_rows(x)
    ref = orc.dequant_epilogue(orc.sparse_gemm_s32(comp, qx, raw, N, K), sx, ws, b)
    assert np.array_equal(y.view(np.uint16), ref.view(np.uint16))
