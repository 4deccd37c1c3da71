"""The calls whose speed is measured, each through a public entry point of forge_amd.

Three families, as the library is used: linear layers of a transformer (decode, prefill, a
training step; dense and 2:4 sparse), convolutions on NCHW FP16 feature maps of an image
network (upscaler resolutions) and on NHWC INT8 maps, and the decoder block of such a network
(depthwise 3x3, then the 2x transposed convolution).

A case is a dict of plain values: "kind" and the sizes. listed() holds the fixed ones, draw()
gives further sizes of the same ranges.
"""
import torch
import torch.nn.functional as F

from forge_amd import nn as fnn
from forge_amd import ops

DEV = "cuda"


def listed():
    return [
        # One token through a square projection: the smallest call, bound by latency.
        {"name": "decode 1x4096x4096", "kind": "linear", "M": 1, "K": 4096, "N": 4096},
        # A batch of 16 tokens against 64 MB of weights: decode of a large layer.
        {"name": "decode 16x8192x8192", "kind": "linear", "M": 16, "K": 8192, "N": 8192},
        # A short prompt through the narrow projection of an MLP: few output tiles, deep K.
        {"name": "linear 1024x6144x1536", "kind": "linear", "M": 1024, "K": 6144, "N": 1536},
        # A width that is no multiple of 128, as networks scaled in steps of 64 have.
        {"name": "linear 1500x2880x2880", "kind": "linear", "M": 1500, "K": 2880, "N": 2880},
        # The first layer of an image transformer: 14x14x3 patches of a 518-pixel image, odd M
        # and a K that is no multiple of 16.
        {"name": "patches 1369x588x1024", "kind": "linear", "M": 1369, "K": 588, "N": 1024},
        # A full prefill through the widest layer: the largest call.
        {"name": "prefill 8192x4096x11008", "kind": "linear", "M": 8192, "K": 4096, "N": 11008},
        # Forward and backward of a QuantizedLinear layer (input and bias gradients).
        {"name": "train 2048x4096x4096", "kind": "train", "M": 2048, "K": 4096, "N": 4096},
        # 2:4 sparse linear layers: a short prompt, and a narrow layer over a large feature map.
        {"name": "sparse 1024x5120x1280", "kind": "sparse", "M": 1024, "K": 5120, "N": 1280},
        {"name": "sparse 147456x1280x320", "kind": "sparse", "M": 147456, "K": 1280, "N": 320},
        # The middle of an image network: 3x3 over 128 channels of a quarter-resolution frame pair.
        {"name": "conv nchw 128ch 135x240", "kind": "conv_nchw", "B": 2, "C": 128, "H": 135, "W": 240, "Co": 128,
         "k": 3, "stride": 1},
        # A downsampling layer on quantized NHWC maps.
        {"name": "conv nhwc 64ch /2", "kind": "conv_nhwc", "B": 32, "C": 64, "H": 112, "W": 112, "Co": 128, "k": 3,
         "stride": 2},
        # The decoder block: depthwise 3x3, then the transposed convolution to twice the size.
        {"name": "decoder 96ch 180x320", "kind": "decoder", "B": 2, "C": 96, "H": 180, "W": 320, "Co": 48},
    ]


def _logint(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], uniform over the logarithm."""
    v = int(round(lo * (hi / lo) ** rng.random() / step)) * step
    return min(max(v, -(-lo // step) * step), hi // step * step)


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 128 or 64, sometimes of 16."""
    return _logint(rng, lo, hi, rng.choice([128, 128, 64, 64, 16]))


def draw(rng):
    kind = rng.choice(["decode", "linear", "linear", "train", "sparse", "sparse", "conv_nchw", "conv_nhwc", "decoder"])
    if kind == "decode":
        return {"kind": "linear", "M": rng.randint(1, 16), "K": _logint(rng, 1024, 8192, 128),
                "N": _logint(rng, 512, 11008, 64)}
    if kind in ("linear", "train"):
        K, N = _width(rng, 256, 6144), _width(rng, 256, 8192)
        if rng.random() < 0.2:
            # a network's first or last layer: any number of inputs, any number of classes
            K, N = (_logint(rng, 27, 1024), N) if rng.random() < 0.5 else (K, _logint(rng, 10, 8192))
        hi = 8192 if kind == "linear" else 4096
        return {"kind": kind, "M": _logint(rng, 17, min(hi, 300_000_000_000 // (K * N))), "K": K, "N": N}
    if kind == "sparse":
        K, N = _logint(rng, 320, 6144, 64), _logint(rng, 320, 6144, 64)
        return {"kind": "sparse", "K": K, "N": N,
                "M": _logint(rng, 1, min(147456, 150_000_000_000 // (K * N), 230_000_000 // (K + N)))}
    if kind == "conv_nchw":
        C, Co = _logint(rng, 16, 256, 16), _logint(rng, 16, 256, 16)
        px = min(2 * 540 * 960, 12_000_000_000 // (C * Co * 9))    # output pixels of the whole batch
        W = _logint(rng, 40, 480, rng.choice([8, 8, 1]))
        H = max(8, min(540, int(px ** 0.5 * rng.uniform(0.4, 0.8))))
        return {"kind": "conv_nchw", "B": rng.randint(1, 2), "C": C, "H": H, "W": W, "Co": Co,
                "k": rng.choice([1, 3, 3]), "stride": rng.choice([1, 1, 2])}
    if kind == "conv_nhwc":
        return {"kind": "conv_nhwc", "B": rng.randint(4, 32), "C": _logint(rng, 32, 256, 32), "H": rng.randint(14, 112),
                "W": rng.randint(14, 112), "Co": _logint(rng, 64, 256, 64), "k": rng.choice([1, 3, 3]),
                "stride": rng.choice([1, 2])}
    return {"kind": "decoder", "B": rng.randint(1, 2), "C": _logint(rng, 32, 256, 32), "H": rng.randint(60, 270),
            "W": _logint(rng, 80, 480, rng.choice([8, 8, 1])), "Co": _logint(rng, 16, 128, 16)}


# ---- inputs ---------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _activations(g, M, K):
    """FP16 activations as a transformer has them: normal, with a few channels far larger."""
    x = torch.randn((M, K), generator=g, device=DEV)
    x[:, torch.randint(0, K, (8,), generator=g, device=DEV)] *= 20.0
    return x.half()


def _weight(g, N, K):
    return torch.randn((N, K), generator=g, device=DEV) * 0.02


def _quant_rows(w):
    """Symmetric per-row INT8 weights and their FP16 scales."""
    s = w.abs().amax(1).clamp_min(1e-8) / 127.0
    return torch.round(w / s[:, None]).clamp(-127, 127).to(torch.int8), s.half()


def _bias(g, N):
    return (torch.randn((N,), generator=g, device=DEV) * 0.1).half()


def _image(g, B, C, H, W):
    return torch.randn((B, C, H, W), generator=g, device=DEV).half()


def _make(c, seed):
    """The tensors of a case: what prepare() hands over and exact() starts from."""
    g = _gen(seed)
    t = {}
    if c["kind"] in ("linear", "train", "sparse"):
        t["x"] = _activations(g, c["M"], c["K"])
        t["w"] = _weight(g, c["N"], c["K"])
        t["bias"] = _bias(g, c["N"])
        if c["kind"] == "train":
            t["grad"] = (torch.randn((c["M"], c["N"]), generator=g, device=DEV) * 0.01).half()
    elif c["kind"] == "conv_nchw":
        t["x"] = _image(g, c["B"], c["C"], c["H"], c["W"])
        t["w"], t["ws"] = _quant_rows(_weight(g, c["Co"], c["C"] * c["k"] ** 2))
        t["bias"] = _bias(g, c["Co"])
    elif c["kind"] == "conv_nhwc":
        Ho, Wo = _out_hw(c)
        q = torch.randn((c["B"], c["H"], c["W"], c["C"]), generator=g, device=DEV) * 30.0
        t["x"] = torch.round(q).clamp(-127, 127).to(torch.int8)
        w, t["ws"] = _quant_rows(_weight(g, c["Co"], c["k"] ** 2 * c["C"]))
        t["w"] = w.view(c["Co"], c["k"], c["k"], c["C"])
        t["as"] = torch.rand((c["B"] * Ho * Wo,), generator=g, device=DEV) * 0.02 + 0.01
        t["bias"] = _bias(g, c["Co"])
    else:
        t["x"] = _image(g, c["B"], c["C"], c["H"], c["W"])
        t["dw"], t["dws"] = _quant_rows(torch.randn((c["C"], 9), generator=g, device=DEV) * 0.3)
        t["db"] = _bias(g, c["C"])
        t["w"], _ = _quant_rows(_weight(g, 4 * c["Co"], c["C"]))
        t["ws"] = (torch.rand((c["Co"],), generator=g, device=DEV) * 1e-3 + 5e-4).half()
        t["bias"] = _bias(g, c["Co"])
    return t


def _out_hw(c):
    p = c["k"] // 2
    return (c["H"] + 2 * p - c["k"]) // c["stride"] + 1, (c["W"] + 2 * p - c["k"]) // c["stride"] + 1


def prepare(case, seed):
    c, t = case, _make(case, seed)
    s = {"case": c}
    if c["kind"] == "linear":
        s["w"], s["ws"] = _quant_rows(t["w"])
        s["x"], s["bias"] = t["x"], t["bias"]
        s["q"] = torch.empty((c["M"], c["K"]), dtype=torch.int8, device=DEV)
        s["qs"] = torch.empty((c["M"],), dtype=torch.float32, device=DEV)
        s["out"] = torch.empty((c["M"], c["N"]), dtype=torch.float16, device=DEV)
    elif c["kind"] == "train":
        layer = fnn.QuantizedLinear(c["K"], c["N"]).to(DEV)
        layer.quantize_weight(t["w"])
        with torch.no_grad():
            layer.bias.copy_(t["bias"])
        s["layer"], s["x"], s["grad"] = layer, t["x"].requires_grad_(True), t["grad"]
    elif c["kind"] == "sparse":
        s["comp"], s["meta"], s["ws"] = ops.prepare_sparse_weight(t["w"])
        s["x"], s["bias"] = t["x"], t["bias"]
        s["q"] = torch.empty((c["M"], c["K"]), dtype=torch.int8, device=DEV)
        s["qs"] = torch.empty((c["M"],), dtype=torch.float32, device=DEV)
        s["split"] = torch.empty((c["M"], c["N"]), dtype=torch.float32, device=DEV)
        s["out"] = torch.empty((c["M"], c["N"]), dtype=torch.float16, device=DEV)
    else:
        s.update(t)
        if c["kind"] == "conv_nchw":
            p, st = c["k"] // 2, c["stride"]
            Ho, Wo = _out_hw(c)
            n = ops.int8_conv2d_workspace_size(c["C"], c["H"], c["W"], c["Co"], c["k"], c["k"], p, p, st, st)
            s["workspace"] = torch.empty((n,), dtype=torch.uint8, device=DEV)
            s["out"] = torch.empty((c["B"], c["Co"], Ho, Wo), dtype=torch.float16, device=DEV)
        elif c["kind"] == "conv_nhwc":
            s["out"] = torch.empty((c["B"], *_out_hw(c), c["Co"]), dtype=torch.float16, device=DEV)
        else:
            n = ops.int8_conv_transpose2d_k2s2_workspace_size(c["C"], c["H"], c["W"], c["Co"])
            s["workspace"] = torch.empty((max(n, 1),), dtype=torch.uint8, device=DEV)
            s["mid"] = torch.empty_like(t["x"])
            s["out"] = torch.empty((c["B"], c["Co"], 2 * c["H"], 2 * c["W"]), dtype=torch.float16, device=DEV)
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "linear":
        return ops.int8_linear(s["x"], s["w"], s["ws"], s["bias"], s["q"], s["qs"], out=s["out"])
    if c["kind"] == "train":
        y = s["layer"](s["x"])
        gx, gb = torch.autograd.grad(y, (s["x"], s["layer"].bias), s["grad"])
        return {"y": y, "grad_x": gx, "grad_bias": gb}
    if c["kind"] == "sparse":
        return ops.sparse_int8_linear(s["x"], s["comp"], s["meta"], s["ws"], s["bias"], s["q"], s["qs"], s["split"],
                                      split_k=0, out=s["out"])
    if c["kind"] == "conv_nchw":
        p = c["k"] // 2
        return ops.int8_conv2d_forward(s["x"], s["w"], s["ws"], s["bias"], c["k"], c["k"], (p, p),
                                       (c["stride"], c["stride"]), workspace=s["workspace"], out=s["out"])
    if c["kind"] == "conv_nhwc":
        p = c["k"] // 2
        return ops.int8_conv2d_nhwc_dequant(s["x"], s["w"], s["as"], s["ws"], s["bias"], (p, p),
                                            (c["stride"], c["stride"]), out=s["out"])
    mid = ops.int8_depthwise_conv2d_forward(s["x"], s["dw"], s["dws"], s["db"], 3, 3, (1, 1), out=s["mid"])
    return ops.int8_conv_transpose2d_k2s2_forward(mid, s["w"], s["ws"], s["bias"], s["workspace"], s["out"])


# ---- what a pass cannot do without --------------------------------------------------------------

def work(case):
    """Each input read once, each output written once; one multiply-add of a stored weight is two
    operations (a 2:4 weight's pruned half is not stored)."""
    c = case
    if c["kind"] in ("linear", "train", "sparse"):
        M, K, N = c["M"], c["K"], c["N"]
        if c["kind"] == "linear":
            return {"bytes": 2 * M * K + N * K + 2 * M * N + 4 * N, "flops": 2 * M * N * K}
        if c["kind"] == "train":
            return {"bytes": 4 * M * K + N * K + 4 * M * N + 6 * N, "flops": 4 * M * N * K}
        return {"bytes": 2 * M * K + N * K * 5 // 8 + 2 * M * N + 4 * N, "flops": M * N * K}
    px_in = c["B"] * c["H"] * c["W"]
    if c["kind"] == "decoder":
        # the map between the two calls is an output of the first and an input of the second
        return {"bytes": px_in * (3 * 2 * c["C"] + 4 * 2 * c["Co"]) + 9 * c["C"] + 4 * c["Co"] * c["C"],
                "flops": 2 * px_in * c["C"] * (9 + 4 * c["Co"])}
    Ho, Wo = _out_hw(c)
    px, K = c["B"] * Ho * Wo, c["C"] * c["k"] ** 2
    in_bytes = px_in * c["C"] * (2 if c["kind"] == "conv_nchw" else 1) + (0 if c["kind"] == "conv_nchw" else 4 * px)
    return {"bytes": in_bytes + c["Co"] * K + 2 * px * c["Co"] + 4 * c["Co"], "flops": 2 * px * c["Co"] * K}


def tolerance(case):
    """FP16 results: rounding to 11 bits is 2.1e-4 in the 2-norm; four times that. The largest
    single difference is an ulp or, behind a quantized intermediate, one INT8 step of an input."""
    if case["kind"] == "decoder":
        return {"rel": 1e-3, "max": 0.06}
    return {"rel": 1e-3, "max": 0.01}


# ---- the same results in 64 bits -----------------------------------------------------------------

def _quant_tokens(x):
    """The per-row activation quantization that defines the operators' INT8 operand (FP32
    arithmetic, as specified), and the scales in FP64."""
    x = x.float()
    s = x.abs().amax(1).clamp_min(1e-8) / 127.0
    q = torch.round(x * (1.0 / s)[:, None]).clamp(-128, 127)
    return q.double(), s.double()


def _dequant(acc, s, ws, bias):
    return acc * (s[:, None] * ws.double()[None, :]) + bias.double()[None, :]


def _prune24(q):
    """The two smaller magnitudes of each group of four are zero (the lower index first among
    equal ones)."""
    N, K = q.shape
    grp = q.view(N, K // 4, 4)
    order = torch.sort(grp.abs().int(), dim=2, stable=True).indices
    return grp.scatter(2, order[..., :2], 0).view(N, K)


def exact(case, seed):
    c, t = case, _make(case, seed)
    if c["kind"] in ("linear", "train", "sparse"):
        w, ws = _quant_rows(t["w"])
        if c["kind"] == "sparse":
            w = _prune24(w)
        q, s = _quant_tokens(t["x"])
        y = torch.empty((c["M"], c["N"]), dtype=torch.float64, device=DEV)
        for i in range(0, c["M"], 16384):
            y[i:i + 16384] = _dequant(q[i:i + 16384] @ w.double().T, s[i:i + 16384], ws, t["bias"])
        if c["kind"] != "train":
            return y
        gd = t["grad"].double()
        return {"y": y, "grad_x": gd @ (w.double() * ws.double()[:, None]), "grad_bias": gd.sum(0)}
    if c["kind"] == "conv_nchw":
        Ho, Wo = _out_hw(c)
        outs = []
        for img in t["x"]:
            cols = F.unfold(img[None].float(), c["k"], padding=c["k"] // 2, stride=c["stride"])[0].T
            parts = []
            for i in range(0, cols.shape[0], 65536):
                q, s = _quant_tokens(cols[i:i + 65536])
                parts.append(_dequant(q @ t["w"].double().T, s, t["ws"], t["bias"]))
            outs.append(torch.cat(parts).T.reshape(c["Co"], Ho, Wo))
        return torch.stack(outs)
    if c["kind"] == "conv_nhwc":
        Ho, Wo = _out_hw(c)
        p, k, st = c["k"] // 2, c["k"], c["stride"]
        x = F.pad(t["x"], (0, 0, p, p, p, p))
        acc = torch.zeros((c["B"] * Ho * Wo, c["Co"]), dtype=torch.float64, device=DEV)
        for i in range(k):
            for j in range(k):
                tap = x[:, i:i + st * (Ho - 1) + 1:st, j:j + st * (Wo - 1) + 1:st, :].reshape(-1, c["C"])
                acc += tap.double() @ t["w"][:, i, j, :].double().T
        return _dequant(acc, t["as"].double(), t["ws"], t["bias"]).view(c["B"], Ho, Wo, c["Co"])
    # decoder: the map between the two calls is FP16 by definition of the first one's output
    B, C, H, W = t["x"].shape
    x = F.pad(t["x"].double(), (1, 1, 1, 1))
    dw = t["dw"].double() * t["dws"].double()[:, None]
    mid = t["db"].double().view(1, C, 1, 1).expand(B, C, H, W).clone()
    for i in range(3):
        for j in range(3):
            mid += x[:, :, i:i + H, j:j + W] * dw[:, 3 * i + j].view(1, C, 1, 1)
    q, s = _quant_tokens(mid.half().permute(0, 2, 3, 1).reshape(-1, C))
    acc = (q @ t["w"].double().T) * s[:, None]                     # columns co*4 + kh*2 + kw
    y = acc.view(B, H, W, c["Co"], 2, 2) * t["ws"].double().view(1, 1, 1, -1, 1, 1) \
        + t["bias"].double().view(1, 1, 1, -1, 1, 1)
    return y.permute(0, 3, 1, 4, 2, 5).reshape(B, c["Co"], 2 * H, 2 * W)
