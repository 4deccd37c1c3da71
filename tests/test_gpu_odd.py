"""GPU parity at row lengths that are no multiple of a vector and at element alignment: the
quantizer's moved-back last vector (both row kernels) and the GEMM's shifted last chunk, bit for
bit against the oracle, bytes around the outputs untouched."""
import numpy as np
import pytest

from helpers import int8_uniform, say, special_fp16_rows, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(5, 8), (6, 9), (7, 15), (33, 588), (9, 2049), (3, 4101), (2, 16383),
                                 (2049, 27), (2050, 588), (2048, 2047), (2055, 4095)])
@pytest.mark.parametrize("offset", [0, 1])
def test_quantize_any_row(dev, orc, M, K, offset):
    import torch
    from forge_amd import ops
    rng = np.random.default_rng(M + K)
    x = rng.uniform(-3.0, 3.0, (M, K)).astype(np.float16)
    if M >= 20 and K >= 400:
        x = special_fp16_rows(rng, M, K)
    qr, sr = orc.quantize_rows(x)
    say(f"quantize any row M={M} K={K} offset={offset}")
    buf = torch.empty(M * K + offset, dtype=torch.float16, device=dev)
    buf[offset:] = to_dev(np.ascontiguousarray(x).view(np.float16).ravel(), dev)
    qb = torch.full((M * K + 16 + offset,), 0x5A, dtype=torch.int8, device=dev)
    q, s = ops.fused_quantize_activation(buf[offset:], M, K, out=qb[8 + offset:8 + offset + M * K])
    assert np.array_equal(to_host(s).view(np.uint32), sr.view(np.uint32))
    got = to_host(qb)
    assert np.array_equal(got[8 + offset:8 + offset + M * K].reshape(M, K), qr)
    assert (got[:8 + offset] == 0x5A).all() and (got[8 + offset + M * K:] == 0x5A).all()


@pytest.mark.parametrize("M,K,N", [(20, 15, 9), (20, 17, 33), (70, 27, 130), (65, 31, 64), (129, 143, 65), (3, 588, 70),
                                   (1369, 588, 1024), (300, 1001, 517), (2100, 129, 2050), (40, 128, 48)])
def test_gemm_any_row(dev, orc, M, K, N):
    """Both operands one byte past an aligned start."""
    import torch
    from forge_amd import ops
    rng = np.random.default_rng(M + K + N)
    A, B = int8_uniform(rng, (M, K)), int8_uniform(rng, (N, K))
    act = rng.uniform(0.001, 0.05, M).astype(np.float32)
    ws = rng.uniform(0.001, 0.05, N).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, N).astype(np.float16)
    ref = orc.gemm_s32(A, B, threads=orc.cpu_threads())
    say(f"gemm any row M={M} K={K} N={N}")

    def shifted(a):
        buf = torch.empty((a.size + 1,), dtype=torch.int8, device=dev)
        buf[1:] = to_dev(a, dev).view(-1)
        return buf[1:].view(a.shape)

    Ad, Bd = shifted(A), shifted(B)
    assert np.array_equal(to_host(ops.int8_gemm_s32(Ad, Bd)), ref)
    y = to_host(ops.int8_gemm_dequant(Ad, Bd, to_dev(act, dev), to_dev(ws, dev), to_dev(b, dev)))
    assert np.array_equal(y.view(np.uint16), orc.dequant_epilogue(ref, act, ws, b).view(np.uint16))
