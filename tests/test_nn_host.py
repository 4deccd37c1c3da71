"""CPU checks of forge_amd.nn's host logic: the w_meta word-order conversion against the
oracle's two packings, and SparseLinear's state_dict layout versioning (a reference
state_dict is converted on load; the module's own state_dict round-trips unchanged)."""
import collections

import numpy as np
import pytest
import torch

from forge_amd.nn import SparseLinear, w_meta_from_reference, w_meta_to_reference


@pytest.mark.parametrize("N,K", [(48, 256), (37, 128), (16, 64)])
def test_w_meta_conversion_matches_oracle(orc, N, K):
    rng = np.random.default_rng(N + K)
    raw = rng.integers(0, 16, N * K // 4).astype(np.uint8)
    ref_words = orc.pack_metadata_ref(raw, N, K).view(np.int32)
    gfx_words = orc.pack_metadata_gfx950(raw, N, K).view(np.int32).reshape(N, K // 32)
    got = w_meta_from_reference(torch.from_numpy(ref_words.copy()))
    assert np.array_equal(got.numpy(), gfx_words)
    back = w_meta_to_reference(torch.from_numpy(gfx_words.copy()))
    assert np.array_equal(back.numpy(), ref_words)


def _reference_state_dict(orc, N, K, rng, version):
    """A state_dict shaped as the reference's SparseLinear saves it: w_meta in the reference's
    row-major word order, module metadata version `version` (None: no metadata at all)."""
    W = rng.integers(-127, 128, (N, K)).astype(np.int8)
    comp, raw = orc.prune_compress_24(W)
    sd = collections.OrderedDict()
    sd["W_comp"] = torch.from_numpy(comp)
    sd["w_meta"] = torch.from_numpy(orc.pack_metadata_ref(raw, N, K).view(np.int32).copy())
    sd["w_scale"] = torch.from_numpy(rng.uniform(1e-3, 1e-2, N).astype(np.float16))
    sd["bias"] = torch.from_numpy(rng.standard_normal(N).astype(np.float16))
    if version is not None:
        sd._metadata = collections.OrderedDict({"": {"version": version}})
    gfx = orc.pack_metadata_gfx950(raw, N, K).view(np.int32).reshape(N, K // 32)
    return sd, gfx


@pytest.mark.parametrize("version", [1, None])
def test_reference_state_dict_is_converted(orc, version):
    rng = np.random.default_rng(3)
    N, K = 32, 128
    sd, gfx = _reference_state_dict(orc, N, K, rng, version)
    m = SparseLinear(K, N)
    m.load_state_dict(sd)
    assert np.array_equal(m.w_meta.numpy(), gfx)
    assert torch.equal(m.W_comp, sd["W_comp"])
    # the module's own state_dict says version 2 and loads unchanged
    own = m.state_dict()
    assert own._metadata[""]["version"] == 2
    m2 = SparseLinear(K, N)
    m2.load_state_dict(own)
    assert torch.equal(m2.w_meta, m.w_meta)


def test_nested_reference_state_dict(orc):
    """A SparseLinear inside a model: the prefix and the submodule's own metadata entry."""
    rng = np.random.default_rng(4)
    N, K = 16, 64
    sd, gfx = _reference_state_dict(orc, N, K, rng, None)
    model = torch.nn.Sequential(SparseLinear(K, N))
    nested = collections.OrderedDict((f"0.{k}", v) for k, v in sd.items())
    nested._metadata = collections.OrderedDict({"": {"version": 1}, "0": {"version": 1}})
    model.load_state_dict(nested)
    assert np.array_equal(model[0].w_meta.numpy(), gfx)


def test_reference_state_dict_bad_w_meta_shape(orc):
    rng = np.random.default_rng(5)
    sd, _ = _reference_state_dict(orc, 32, 128, rng, 1)
    sd["w_meta"] = sd["w_meta"][:, :2]
    with pytest.raises(RuntimeError, match="w_meta"):
        SparseLinear(128, 32).load_state_dict(sd)


def test_plain_tensors():
    """What may go to the library by address in a backward: plain tensors with memory of their own, and
    nothing while a transform has to see the operators."""
    import torch.autograd.forward_ad as fwAD
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils.flop_counter import FlopCounterMode
    from forge_amd.nn import _plain
    t = torch.ones(3, 4)
    assert _plain(t, torch.nn.Parameter(t), t.t())
    assert not _plain(t, torch._efficientzerotensor(3))
    seen = []
    torch.vmap(lambda a: (seen.append(_plain(t, a)), a)[1])(t)
    x = torch.ones(4, requires_grad=True)

    class Probe(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a):
            return a * 1

        @staticmethod
        def backward(ctx, g):
            seen.append(_plain(g))
            return g

    torch.autograd.grad(Probe.apply(x), x, t, is_grads_batched=True)
    assert seen == [False, False]
    torch.autograd.grad(Probe.apply(x), x, t[0])
    assert seen.pop()
    with FakeTensorMode():
        fake = torch.ones(3)
    assert not _plain(fake)
    with fwAD.dual_level():
        assert not _plain(t)
    with FlopCounterMode(display=False):
        assert not _plain(t)
    assert _plain(t)


@pytest.mark.parametrize("shape", [(5, 15), (5, 17), (80,), (5, 16, 1), (16, 5)])
def test_backward_prep_refuses_other_shapes(shape):
    """A gradient that is not (M, N) is refused before anything is launched on it."""
    from forge_amd import ops
    w, ws = torch.zeros((16, 32), dtype=torch.int8), torch.ones(16, dtype=torch.float16)
    with pytest.raises(ValueError, match="grad must be"):
        ops.int8_linear_backward_prep(w, ws, torch.zeros(shape, dtype=torch.float16), True)
