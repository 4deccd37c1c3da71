"""GPU parity of the ring-fed tiles: every tile shape of the dense choice (checked by route) at
ragged rows and columns and K not a multiple of 128, each at one or two stages and at 5 or 9, which
refill every slot and start the K loop of seven XCDs in mid-K; both NHWC gathers likewise; and the
transposed conv's scatter. Integer sums are exact, and the FP16 epilogue is the oracle's, so every
output is compared bit for bit."""
import numpy as np
import pytest

from helpers import int8_uniform, poison, say, to_dev, to_host

pytestmark = pytest.mark.gpu

SHAPES = [
    (62, 208, 40, "dma64x64"), (700, 1040, 999, "dma64x64"), (131, 544, 5538, "dma64x128"),
    (322, 656, 5565, "dma64x192"), (67, 48, 3, "dma64x64"),
    (327, 16, 5708, "dma128x128"), (2694, 912, 1001, "dma128x128 4-slot"),
    (642, 16, 5390, "dma192x128"), (1159, 16, 4652, "dma128x192"), (1033, 144, 5418, "dma128x256"),
    (2315, 144, 3339, "dma192x192"), (2092, 16, 5763, "dma192x256"), (2813, 16, 4392, "dma256x192"),
    (2438, 16, 4888, "dma256x256"), (1030, 400, 13001, "dma256x256"),
    # at least 2 slots + 1 stages: the loop's partial waits, slot advance and refills
    (61, 1040, 41, "dma64x64"), (8205, 1040, 65, "dma64x128"), (129, 1040, 10893, "dma64x192"),
    (8203, 528, 193, "dma128x128"), (8267, 1040, 194, "dma128x128 4-slot"), (10921, 1040, 258, "dma192x128"),
    (385, 1040, 10916, "dma128x192"), (8209, 1040, 643, "dma128x256"), (11002, 1040, 516, "dma192x192"),
    (9893, 1040, 769, "dma192x256"), (9796, 1040, 1031, "dma256x192"), (1539, 1040, 7204, "dma256x256"),
    (1000, 1040, 17900, "dma256x256+tail192"),
]


@pytest.mark.parametrize("M,K,N,route", SHAPES)
def test_ring_shapes(dev, orc, M, K, N, route):
    import torch
    from forge_amd import ops
    rng = np.random.default_rng(M + K + N)
    A, B = int8_uniform(rng, (M, K)), int8_uniform(rng, (N, K))
    act = rng.uniform(0.001, 0.05, M).astype(np.float32)
    ws = rng.uniform(0.001, 0.05, N).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, N).astype(np.float16)
    ref = orc.gemm_s32(A, B, threads=orc.cpu_threads())
    say(f"ring M={M} K={K} N={N} {route}")
    Ad, Bd = to_dev(A, dev), to_dev(B, dev)
    C = torch.empty((M, N), dtype=torch.int32, device=dev)
    poison(C, 0x7B)
    assert np.array_equal(to_host(ops.int8_gemm_s32(Ad, Bd, out=C)), ref)
    assert ops.last_route() == route
    for bias in (b, None):
        # one element past an aligned start: rows at every 2-byte alignment
        buf = torch.empty((M * N + 1,), dtype=torch.float16, device=dev)
        poison(buf, 0x5A)
        Y = buf[1:].view(M, N)
        ops.int8_gemm_dequant(Ad, Bd, to_dev(act, dev), to_dev(ws, dev), None if bias is None else to_dev(bias, dev), out=Y)
        assert np.array_equal(to_host(Y).view(np.uint16), orc.dequant_epilogue(ref, act, ws, bias).view(np.uint16))
        assert to_host(buf).view(np.uint8)[:2].tolist() == [0x5A, 0x5A]


@pytest.mark.parametrize("N,H,W,C,Co,k,pad,stride,dil", [
    (2, 20, 23, 16, 24, 7, 3, 2, 1),       # 49 taps, 8 per stage, K % 128 != 0
    (3, 17, 14, 48, 65, 3, 1, 1, 2),       # chunks of a stage straddle taps, ragged columns
    (1, 31, 9, 80, 130, 3, 0, 2, 1),
    (2, 64, 64, 64, 128, 3, 1, 2, 1),
    (2, 24, 24, 320, 192, 1, 0, 1, 1),     # pointwise
])
def test_ring_conv(dev, orc, N, H, W, C, Co, k, pad, stride, dil):
    _conv(dev, orc, N, H, W, C, Co, k, pad, stride, dil)


def _conv(dev, orc, N, H, W, C, Co, k, pad, stride, dil, route=None):
    import torch
    from forge_amd import ops
    rng = np.random.default_rng(H * W + C + Co)
    x, w = int8_uniform(rng, (N, H, W, C)), int8_uniform(rng, (Co, k, k, C))
    ref = orc.conv2d_nhwc_s32(x, w, (pad, pad), (stride, stride), (dil, dil), threads=orc.cpu_threads())
    say(f"ring conv N={N} H={H} W={W} C={C} Co={Co} k={k} p={pad} s={stride} d={dil}")
    xd, wd = to_dev(x, dev), to_dev(w, dev)
    args = ((pad, pad), (stride, stride), (dil, dil))
    assert np.array_equal(to_host(ops.int8_conv2d_nhwc_s32(xd, wd, *args)), ref)
    assert ops.last_route().startswith("dma") if route is None else ops.last_route() == route
    acc = ref.reshape(-1, Co)
    act = rng.uniform(0.001, 0.05, acc.shape[0]).astype(np.float32)
    ws = rng.uniform(0.001, 0.05, Co).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, Co).astype(np.float16)
    Y = torch.empty(ref.shape, dtype=torch.float16, device=dev)
    poison(Y, 0x5A)
    ops.int8_conv2d_nhwc_dequant(xd, wd, to_dev(act, dev), to_dev(ws, dev), to_dev(b, dev), *args, out=Y)
    assert np.array_equal(to_host(Y).reshape(-1, Co).view(np.uint16),
                          orc.dequant_epilogue(acc, act, ws, b).view(np.uint16))


# Every tile shape of both gathers at 9 and 10 stages, which starts the K loop of seven XCDs in mid-K and
# refills every slot: C % 128 == 0 (a stage is one tap), then chunks of 48 channels (a stage straddles
# taps). Ragged rows and columns, padding, strides and dilations.
@pytest.mark.parametrize("N,H,W,C,Co,k,pad,stride,dil,route", [
    (1, 22, 16, 128, 28, 3, 0, 2, 2, "dma64x64"), (8, 40, 29, 128, 65, 3, 0, 1, 1, "dma64x128"),
    (10, 82, 53, 128, 130, 3, 1, 2, 1, "dma64x192"), (11, 81, 59, 128, 65, 3, 1, 1, 2, "dma128x128"),
    (7, 25, 86, 128, 65, 3, 2, 1, 1, "dma128x128 4-slot"), (4, 83, 50, 128, 129, 3, 1, 1, 1, "dma192x128"),
    (8, 78, 43, 128, 129, 3, 0, 1, 1, "dma128x192"), (7, 84, 87, 128, 391, 3, 0, 2, 1, "dma128x256"),
    (7, 71, 66, 128, 129, 3, 1, 1, 1, "dma192x192"), (11, 83, 36, 128, 193, 3, 1, 1, 1, "dma192x256"),
    (10, 72, 73, 128, 129, 3, 0, 1, 1, "dma256x192"), (5, 82, 57, 128, 385, 3, 2, 1, 1, "dma256x256"),
    (6, 50, 55, 1024, 577, 1, 0, 1, 1, "dma256x256"), (6, 50, 55, 896, 577, 1, 0, 1, 1, "dma192x128"),
    (2, 9, 7, 256, 40, 16, 9, 1, 1, "dma64x64"),
    (1, 1, 1, 128, 24, 3, 1, 1, 1, "dma64x64"),         # one pixel in a window of nine: offsets past the image's end
    (1, 15, 15, 48, 33, 5, 0, 2, 2, "dma64x64"), (4, 49, 46, 48, 65, 5, 1, 1, 1, "dma64x128"),
    (9, 86, 59, 48, 131, 5, 1, 2, 1, "dma64x192"), (9, 62, 89, 48, 65, 5, 2, 1, 1, "dma128x128"),
    (10, 76, 27, 48, 65, 5, 0, 1, 1, "dma128x128 4-slot"), (5, 63, 60, 48, 129, 5, 2, 1, 2, "dma192x128"),
    (10, 90, 38, 48, 131, 5, 0, 1, 2, "dma128x192"), (4, 46, 89, 48, 390, 5, 0, 1, 2, "dma128x256"),
    (5, 68, 52, 48, 258, 5, 1, 1, 1, "dma192x192"), (7, 84, 63, 48, 196, 5, 2, 1, 2, "dma192x256"),
    (11, 35, 70, 48, 262, 5, 1, 1, 1, "dma256x192"), (1, 20, 20, 128, 24, 17, 8, 1, 1, "dma64x64"),
])
def test_ring_conv_shapes(dev, orc, N, H, W, C, Co, k, pad, stride, dil, route):
    _conv(dev, orc, N, H, W, C, Co, k, pad, stride, dil, route)


def test_conv_very_wide_kernel(dev, orc):
    """A kernel of 65537 columns: past the range in which the gather's division of the tap by kW is
    exact, so the register-staged gather, which divides truly, runs."""
    from forge_amd import ops
    rng = np.random.default_rng(9)
    x, w = int8_uniform(rng, (1, 3, 65541, 16)), int8_uniform(rng, (24, 1, 65537, 16))
    say("conv of 65537 columns")
    got = to_host(ops.int8_conv2d_nhwc_s32(to_dev(x, dev), to_dev(w, dev)))
    assert ops.last_route().startswith("regstaged")
    for j in range(5):
        want = x[0, :, j:j + 65537].reshape(3, -1).astype(np.int64) @ w.reshape(24, -1).T.astype(np.int64)
        assert np.array_equal(got[0, :, j], want)


@pytest.mark.parametrize("N,C_in,H,W,C_out,bias,route", [
    (1, 48, 7, 12, 5, True, "dma64x64 scatter"), (2, 80, 9, 13, 17, False, "dma64x64 scatter"),   # W % 4 = 0 and not
    (3, 16, 120, 132, 160, True, "dma128x128 scatter"), (2, 272, 100, 120, 96, True, "dma256x256 scatter"),
])
def test_ring_scatter(dev, orc, N, C_in, H, W, C_out, bias, route):
    from forge_amd import ops
    rng = np.random.default_rng(C_in + H + W)
    x = rng.uniform(-1, 1, (N, C_in, H, W)).astype(np.float16)
    w = int8_uniform(rng, (4 * C_out, C_in))
    ws = rng.uniform(0.001, 0.02, C_out).astype(np.float16)
    b = rng.uniform(-0.5, 0.5, C_out).astype(np.float16) if bias else None
    say(f"ring scatter C_in={C_in} H={H} W={W} C_out={C_out}")
    y = to_host(ops.int8_conv_transpose2d_k2s2_forward(to_dev(x, dev), to_dev(w, dev), to_dev(ws, dev),
                                                       None if b is None else to_dev(b, dev)))
    assert ops.last_route() == route
    want = orc.conv_transpose2d_k2s2(x, w, ws, b)
    assert np.array_equal(y.view(np.uint16), np.ascontiguousarray(want).view(np.uint16))
