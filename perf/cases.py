"""The work that a program built on this library has it do, as cases that can be timed and
checked: whole networks through their device entry points, and single layers through the
op-level entry points.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a
program has in hand before the call (the context and its weights, the input tensors), run()
is one pass, work() the bytes and operations it cannot do without, tolerance() how far two
correct implementations may differ and exact() the same result in 64-bit torch.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "sd-vulkan-pixel10-tensor-g5_amd"))

import sdu  # noqa: E402

DEV = "cuda"
WEIGHT_SEED = 1234
AFFINE = sdu.SDU_INIT_RANDOM_AFFINE


def listed():
    return [
        # one denoise step of a 512x512 image: the conditional and the unconditional half
        {"name": "unet_pair", "op": "unet", "B": 2, "H": 64, "W": 64, "L": 77},
        # serving: eight prompts with guidance in one batch, the largest call
        {"name": "unet_batch", "op": "unet", "B": 16, "H": 64, "W": 64, "L": 77},
        # the prompt and the empty prompt of one image
        {"name": "text_pair", "op": "clip", "B": 2},
        # the small decoder, one 512x512 image
        {"name": "image_small_decoder", "op": "taesd", "B": 1, "H": 64, "W": 64},
        # the full decoder, one 512x512 image
        {"name": "image_full_decoder", "op": "vae", "B": 1, "H": 64, "W": 64},
        # first conv of a resnet at the widest level: bias and time projection
        {"name": "conv_64", "op": "conv", "B": 2, "H": 64, "W": 64, "Ci": 320, "Co": 320, "k": 3, "stride": 1, "up": 0,
         "temb": True, "res": False, "relu": False},
        # second conv of a resnet at a deep level: few pixels, many weights, residual
        {"name": "conv_16", "op": "conv", "B": 2, "H": 16, "W": 16, "Ci": 1280, "Co": 1280, "k": 3, "stride": 1, "up": 0,
         "temb": False, "res": True, "relu": False},
        # self-attention of the widest level
        {"name": "attn_self", "op": "attn", "B": 2, "heads": 8, "Sq": 4096, "Sk": 4096, "d": 40, "causal": False},
        # cross-attention over the prompt one level down
        {"name": "attn_cross", "op": "attn", "B": 2, "heads": 8, "Sq": 1024, "Sk": 77, "d": 80, "causal": False},
        # gated feed-forward projection of the widest level
        {"name": "matmul_geglu", "op": "matmul", "M": 8192, "N": 2560, "K": 320, "geglu": True, "gelu": False, "res": False,
         "f32": False},
        # an output projection of the text encoder: the smallest call, a ragged row count
        {"name": "matmul_text", "op": "matmul", "M": 154, "N": 768, "K": 768, "geglu": False, "gelu": False, "res": True,
         "f32": False},
        # GroupNorm + SiLU of an up-path resnet, over two concatenated sources
        {"name": "norm_concat", "op": "gnorm", "B": 2, "HW": 4096, "C1": 640, "C2": 320, "silu": True},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def mult(m, lo, hi):
        return m * max(1, int(round(log(lo, hi) / m)))

    op = rng.choice(["unet", "clip", "taesd", "vae", "conv", "conv", "conv", "attn", "attn", "matmul", "matmul", "gnorm",
                     "lnorm"])
    if op == "unet":
        H, W = mult(8, 24, 96), mult(8, 24, 96)
        return {"op": op, "B": rng.randint(1, max(1, min(12, 49152 // (H * W)))), "H": H, "W": W, "L": rng.choice([77, 77, 154])}
    if op == "clip":
        return {"op": op, "B": log(1, 32)}
    if op == "taesd":
        return {"op": op, "B": rng.randint(1, 4), "H": log(16, 96), "W": log(16, 96)}
    if op == "vae":
        return {"op": op, "B": rng.randint(1, 2), "H": mult(8, 16, 80), "W": mult(8, 16, 80)}  # a UNet latent
    if op == "conv":
        k = rng.choice([3, 3, 3, 3, 1])
        form = rng.choice(["plain", "plain", "plain", "down", "up"]) if k == 3 else "plain"
        side = log(8, 96)
        cmax = 1280 if side <= 32 else 640
        return {"op": op, "B": rng.randint(1, 4), "H": side, "W": max(8, side + rng.randint(-8, 8)),
                "Ci": mult(rng.choice([64, 64, 32, 8]), 64, cmax), "Co": mult(rng.choice([64, 32, 8]), 64, cmax), "k": k,
                "stride": 2 if form == "down" else 1, "up": 1 if form == "up" else 0, "temb": rng.random() < 0.5,
                "res": form == "plain" and rng.random() < 0.5, "relu": rng.random() < 0.25}
    if op == "attn":
        kind = rng.choice(["self", "cross", "causal"])
        d = 64 if kind == "causal" else rng.choice([40, 40, 80, 160, 64])
        S = log(16, 256) if kind == "causal" else log(64, 8192 if d <= 64 else 2304)
        return {"op": op, "B": rng.randint(1, 4), "heads": 12 if kind == "causal" else 8, "Sq": S,
                "Sk": rng.choice([77, 77, 154]) if kind == "cross" else S, "d": d, "causal": kind == "causal"}
    if op == "matmul":
        geglu = rng.random() < 0.25
        K = mult(rng.choice([64, 64, 8]), 128, 5120)
        N = mult(64 if geglu else rng.choice([64, 64, 8]), 128, 5120)
        return {"op": op, "M": min(log(64, 16384), 2 ** 32 // (N * K) * 8), "N": N, "K": K, "geglu": geglu,
                "gelu": not geglu and rng.random() < 0.2, "res": not geglu and rng.random() < 0.5,
                "f32": not geglu and rng.random() < 0.15}
    if op == "gnorm":
        C1, C2 = mult(32, 128, 1280), rng.choice([0, 0, mult(32, 128, 1280)])
        return {"op": op, "B": rng.randint(1, 8), "HW": log(64, 9216), "C1": C1, "C2": C2, "silu": rng.random() < 0.7}
    return {"op": op, "T": log(64, 32768), "C": mult(8, 128, 1280)}


# ------------------------------------------------------------------ inputs

_engines = {}


def _engine(op):
    """One context for the process, as a program keeps it; each network's weights on first use."""
    key = "unet" if op == "unet" else "ops"
    if key not in _engines:
        _engines[key] = sdu.Engine(seed=WEIGHT_SEED, flags=AFFINE if op == "unet" else sdu.SDU_INIT_NO_WEIGHTS)
    eng = _engines[key]
    if op in ("clip", "taesd", "vae") and op not in _engines:
        getattr(eng, op + "_init")(seed=WEIGHT_SEED, flags=AFFINE)
        _engines[op] = eng
    return eng


def _inputs(case, seed):
    """The pass's inputs as torch tensors: activations near N(0, 1), weights scaled to keep it so."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def n(*shape, std=1.0, mean=0.0, dtype=torch.float16):
        return (torch.randn(*shape, device=DEV, generator=g) * std + mean).to(dtype)

    f32 = torch.float32
    op, c = case["op"], case
    if op == "unet":
        t = int(torch.randint(0, 1000, (1,), generator=torch.Generator().manual_seed(seed)))
        return {"lat": n(c["B"], 4, c["H"], c["W"], dtype=f32), "ctx": n(c["B"], c["L"], 768, dtype=f32),
                "temb": torch.from_numpy(sdu.time_proj(t)).to(DEV)}
    if op == "clip":
        return {"ids": torch.randint(0, 49408, (c["B"], 77), device=DEV, generator=g, dtype=torch.int32)}
    if op in ("taesd", "vae"):
        return {"lat": n(c["B"], 4, c["H"], c["W"], dtype=f32)}
    if op == "conv":
        Ho, Wo = _conv_out(c)
        x = {"x": n(c["B"], c["H"], c["W"], c["Ci"]),
             "w": n(c["Co"], c["k"], c["k"], c["Ci"], std=1.0 / math.sqrt(c["k"] * c["k"] * c["Ci"])), "bias": n(c["Co"], std=0.5)}
        if c["temb"]:
            x["temb"] = n(c["Co"], std=0.5, dtype=f32)
        if c["res"]:
            x["res"] = n(c["B"], Ho, Wo, c["Co"])
        return x
    if op == "attn":
        C = c["heads"] * c["d"]
        return {"q": n(c["B"], c["Sq"], C), "k": n(c["B"], c["Sk"], C), "v": n(c["B"], c["Sk"], C)}
    if op == "matmul":
        x = {"a": n(c["M"], c["K"]), "w": n(c["N"], c["K"], std=1.0 / math.sqrt(c["K"])), "bias": n(c["N"], std=0.5)}
        if c["res"]:
            x["res"] = n(c["M"], c["N"])
        return x
    if op == "gnorm":
        C = c["C1"] + c["C2"]
        x = {"x": n(c["B"], c["HW"], c["C1"], std=2.0, mean=0.5), "gamma": n(C, std=0.3, mean=1.0), "beta": n(C, std=0.3)}
        if c["C2"]:
            x["x2"] = n(c["B"], c["HW"], c["C2"], std=1.5, mean=-0.5)
        return x
    return {"x": n(c["T"], c["C"], std=2.0, mean=0.5), "gamma": n(c["C"], std=0.3, mean=1.0), "beta": n(c["C"], std=0.3)}


def _conv_out(c):
    if c["up"]:
        return 2 * c["H"], 2 * c["W"]
    return (c["H"] - 1) // c["stride"] + 1, (c["W"] - 1) // c["stride"] + 1


class _Memory:
    """A library tensor's device memory, for torch to see in place."""

    def __init__(self, t):
        self.owner = t  # kept while torch sees its memory
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": "<f2" if t.dtype == sdu.SDU_F16 else "<f4",
                                         "data": (t.ptr, False), "strides": None, "version": 2}


def _view(t):
    return torch.as_tensor(_Memory(t), device=DEV)


def _out_shape(c):
    if c["op"] == "conv":
        return (c["B"],) + _conv_out(c) + (c["Co"],)
    if c["op"] == "attn":
        return (c["B"], c["Sq"], c["heads"] * c["d"])
    if c["op"] == "matmul":
        return (c["M"], c["N"] // 2 if c["geglu"] else c["N"])
    if c["op"] == "gnorm":
        return (c["B"], c["HW"], c["C1"] + c["C2"])
    return (c["T"], c["C"])


def prepare(case, seed):
    op, c = case["op"], case
    eng, x = _engine(op), _inputs(case, seed)
    s = {"case": dict(case), "eng": eng, "in": x}
    if op == "unet":
        s["out"] = torch.empty_like(x["lat"])
    elif op == "clip":
        s["out"] = torch.empty(c["B"], 77, 768, device=DEV)
    elif op in ("taesd", "vae"):
        s["out"] = torch.empty(c["B"], 3, 8 * c["H"], 8 * c["W"], device=DEV)
    else:
        t = {}
        for k, v in x.items():
            t[k] = eng.tensor(tuple(v.shape), sdu.SDU_F32 if v.dtype == torch.float32 else sdu.SDU_F16)
            _view(t[k]).copy_(v)
        t["y"] = eng.tensor(_out_shape(c), sdu.SDU_F32 if c.get("f32") else sdu.SDU_F16)
        s["t"], s["out"], s["in"] = t, _view(t["y"]), None
        torch.cuda.synchronize()
    return s


def run(s):
    c, eng, x, y = s["case"], s["eng"], s["in"], s["out"]
    op = c["op"]
    if op == "unet":
        eng.forward_device(x["lat"].data_ptr(), x["temb"].data_ptr(), x["ctx"].data_ptr(), c["B"], c["H"], c["W"], c["L"],
                           y.data_ptr())
    elif op == "clip":
        eng.clip_encode_device(x["ids"].data_ptr(), c["B"], y.data_ptr())
    elif op == "taesd":
        eng.taesd_decode_device(x["lat"].data_ptr(), c["B"], c["H"], c["W"], y.data_ptr())
    elif op == "vae":
        eng.vae_decode_device(x["lat"].data_ptr(), c["B"], c["H"], c["W"], y.data_ptr())
    else:
        t = s["t"]
        if op == "conv":
            eng.conv2d(t["x"], t["w"], t["y"], c["B"], c["H"], c["W"], c["Ci"], c["Co"], ksize=c["k"], stride=c["stride"],
                       upsample=bool(c["up"]), bias=t["bias"], temb=t.get("temb"), residual=t.get("res"),
                       flags=sdu.SDU_EPI_RELU if c["relu"] else 0)
        elif op == "attn":
            C = c["heads"] * c["d"]
            eng.attention_ex(t["q"], t["k"], t["v"], t["y"], c["B"], c["heads"], c["Sq"], c["Sk"], c["d"], C, C, C, C,
                             1.0 / math.sqrt(c["d"]), flags=sdu.SDU_ATTN_CAUSAL if c["causal"] else 0)
        elif op == "matmul":
            flags = (sdu.SDU_EPI_GEGLU if c["geglu"] else 0) | (sdu.SDU_EPI_QUICK_GELU if c["gelu"] else 0)
            eng.matmul(t["a"], t["w"], t["y"], c["M"], c["N"], c["K"], bias=t["bias"], residual=t.get("res"),
                       flags=flags | (sdu.SDU_EPI_OUT_F32 if c["f32"] else 0))
        elif op == "gnorm":
            eng.groupnorm(t["x"], t["gamma"], t["beta"], t["y"], c["B"], c["HW"], c["C1"], c["C2"], x2=t.get("x2"),
                          silu=c["silu"])
        else:
            eng.layernorm(t["x"], t["gamma"], t["beta"], t["y"], c["T"], c["C"])
    return y


# ------------------------------------------------------------------ work and tolerance


class _Count:
    """Multiply-adds of a network's matrix products, two operations each, as its 64-bit form walks it."""

    def __init__(self):
        self.flops = 0.0

    def __call__(self, m, n, k):
        self.flops += 2.0 * m * n * k


def _unet_flops(B, H, W, L):
    n = _Count()
    chans = (320, 640, 1280, 1280)
    skips = [320, 320, 320, 320, 640, 640, 640, 1280, 1280, 1280, 1280, 1280]

    def resnet(p, ci, co):
        n(p, co, 9 * ci)
        n(p, co, 9 * co)
        if ci != co:
            n(p, co, ci)

    def transformer(p, c):
        n(p, c, 20 * c)  # proj_in, q k v, out; q, out; gated feed-forward (8 + 4), proj_out
        n(B * L, 2 * c, 768)
        n(p, 2 * (p // B), c)
        n(p, 2 * L, c)

    p = B * H * W
    n(p, 320, 36)
    ci = 320
    for i, c in enumerate(chans):
        for r in range(2):
            resnet(p, ci, c)
            ci = c
            if i < 3:
                transformer(p, c)
        if i < 3:
            p //= 4
            n(p, c, 9 * c)
    resnet(p, 1280, 1280)
    transformer(p, 1280)
    resnet(p, 1280, 1280)
    for i, c in enumerate(chans[::-1]):
        for r in range(3):
            resnet(p, ci + skips.pop(), c)
            ci = c
            if i > 0:
                transformer(p, c)
        if i < 3:
            p *= 4
            n(p, c, 9 * c)
    n(p, 4, 9 * 320)
    return n.flops


def _vae_flops(B, H, W):
    n = _Count()
    p = B * H * W
    n(p, 512, 36)
    for _ in range(4):
        n(p, 512, 9 * 512)
    n(p, 512, 4 * 512)
    n(p, 2 * H * W, 512)
    ci = 512
    for i, c in enumerate((512, 512, 256, 128)):
        for j in range(3):
            n(p, c, 9 * ci)
            n(p, c, 9 * c)
            if ci != c:
                n(p, c, ci)
            ci = c
        if i < 3:
            p *= 4
            n(p, c, 9 * c)
    n(p, 3, 9 * 128)
    return n.flops


def _taesd_flops(B, H, W):
    n = _Count()
    p = B * H * W
    n(p, 64, 36)
    for i, blocks in enumerate((3, 3, 3, 1)):
        n(p, 64, 9 * 64 * 3 * blocks)
        if i < 3:
            p *= 4
            n(p, 64, 9 * 64)
    n(p, 3, 9 * 64)
    return n.flops


def work(case):
    c, op = case, case["op"]
    if op == "unet":
        px = c["B"] * c["H"] * c["W"]
        return {"bytes": 2.0 * 859520964 + 4.0 * (8 * px + c["B"] * c["L"] * 768 + 320), "flops": _unet_flops(c["B"], c["H"], c["W"], c["L"])}
    if op == "clip":
        T = c["B"] * 77
        return {"bytes": 2.0 * (12 * (12 * 768 * 768 + 13 * 768) + 77 * 768 + T * 768) + 4.0 * (T + T * 768),
                "flops": 12 * (2.0 * T * 768 * 12 * 768 + 4.0 * T * 77 * 768)}
    if op in ("taesd", "vae"):
        px = c["B"] * c["H"] * c["W"]
        params = 1222531 if op == "taesd" else 49490199
        return {"bytes": 2.0 * params + 4.0 * (4 * px + 3 * 64 * px),
                "flops": (_taesd_flops if op == "taesd" else _vae_flops)(c["B"], c["H"], c["W"])}
    if op == "conv":
        Ho, Wo = _conv_out(c)
        out, kk = c["B"] * Ho * Wo * c["Co"], c["k"] * c["k"] * c["Ci"]
        return {"bytes": 2.0 * (c["B"] * c["H"] * c["W"] * c["Ci"] + c["Co"] * kk + c["Co"] + out * (2 if c["res"] else 1))
                + (4.0 * c["Co"] if c["temb"] else 0.0), "flops": 2.0 * out * kk}
    if op == "attn":
        C = c["heads"] * c["d"]
        pairs = c["Sq"] * (c["Sq"] + 1) / 2 if c["causal"] else c["Sq"] * c["Sk"]
        return {"bytes": 4.0 * c["B"] * C * (c["Sq"] + c["Sk"]), "flops": 4.0 * c["B"] * C * pairs}
    if op == "matmul":
        out = c["M"] * c["N"] // (2 if c["geglu"] else 1)
        return {"bytes": 2.0 * (c["M"] * c["K"] + c["N"] * c["K"] + c["N"] + (out if c["res"] else 0)) + (4.0 if c["f32"] else 2.0) * out,
                "flops": 2.0 * c["M"] * c["N"] * c["K"]}
    n = c["B"] * c["HW"] * (c["C1"] + c["C2"]) if op == "gnorm" else c["T"] * c["C"]
    return {"bytes": 4.0 * n, "flops": 10.0 * n}


def tolerance(case):
    # four times the error against exact() of fp16 storage with fp32 sums: 1.3e-3 (UNet), 1.1e-3
    # (text encoder), 1.7e-4 (small decoder), 2.8e-3 (full decoder), 2.5e-4 to 2.9e-4
    # (attention, whose probabilities are fp16), 2.1e-4 (the other layers: one fp16 rounding)
    rel = {"unet": 5.2e-3, "clip": 4.4e-3, "taesd": 8e-4, "vae": 1.1e-2, "attn": 1.2e-3}
    return {"rel": rel.get(case["op"], 8.5e-4)}


# ------------------------------------------------------------------ 64-bit reference

_M64 = (1 << 64) - 1


def _splitmix(x):
    """splitmix64 of an int64 tensor (wrapping arithmetic, logical shifts)."""
    def shr(v, k):
        return (v >> k) & ((1 << (64 - k)) - 1)

    def signed(v):
        return v - (1 << 64) if v >> 63 else v

    x = x + signed(0x9E3779B97F4A7C15)
    x = (x ^ shr(x, 30)) * signed(0xBF58476D1CE4E5B9)
    x = (x ^ shr(x, 27)) * signed(0x94D049BB133111EB)
    return x ^ shr(x, 31)


class _Weights:
    """The seeded weights of a network by name: element i of tensor `name` is the fp16 value of
    mean + std sqrt(-2 ln u1) cos(2 pi u2), u1 and u2 from splitmix64(key + 2i), (key + 2i + 1),
    key = fnv1a64(name) ^ splitmix64(seed).  Norm gammas N(1, .02), betas and biases N(0, .02)."""

    def __init__(self, std, linear_std=None):
        self.std, self.linear_std = std, linear_std or std

    def __call__(self, name, *shape, norm=False):
        h = 0xCBF29CE484222325
        for ch in name.encode():
            h = ((h ^ ch) * 0x100000001B3) & _M64
        key = int(_splitmix(torch.tensor([WEIGHT_SEED], dtype=torch.int64))[0])
        key ^= h - (1 << 64) if h >> 63 else h
        n = math.prod(shape)
        i = torch.arange(n, device=DEV, dtype=torch.int64) * 2 + key
        u1 = (((_splitmix(i) >> 11) & ((1 << 53) - 1)) + 1).double() * 2.0 ** -53
        u2 = ((_splitmix(i + 1) >> 11) & ((1 << 53) - 1)).double() * 2.0 ** -53
        z = torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(6.283185307179586 * u2)
        std = 0.02 if len(shape) == 1 else self.linear_std if len(shape) == 2 else self.std
        return ((1.0 if norm else 0.0) + std * z).float().half().double().reshape(shape)


def _conv3(x, w, b=None, stride=1):
    """x [B,H,W,Ci], w [Co,Ci,3,3], pad 1 -> [B,Ho,Wo,Co], one product per tap."""
    B, H, W, Ci = x.shape
    xp = F.pad(x, (0, 0, 1, 1, 1, 1))
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    y = torch.zeros(B * Ho * Wo, w.shape[0], device=DEV, dtype=torch.float64)
    for ky in range(3):
        for kx in range(3):
            a = xp[:, ky:ky + stride * (Ho - 1) + 1:stride, kx:kx + stride * (Wo - 1) + 1:stride].reshape(-1, Ci)
            y += a.contiguous() @ w[:, :, ky, kx].t().contiguous()
    return (y if b is None else y + b).reshape(B, Ho, Wo, -1)


def _lin(x, w, b=None):
    y = x.reshape(-1, x.shape[-1]) @ w.t().contiguous()
    return (y if b is None else y + b).reshape(*x.shape[:-1], w.shape[0])


def _up(x):
    return x.repeat_interleave(2, 1).repeat_interleave(2, 2)


def _gn(x, gamma, beta, eps, groups=32):
    """x [B, ..., C]: statistics over each image's group of channels."""
    B, C = x.shape[0], x.shape[-1]
    g = x.reshape(B, -1, groups, C // groups)
    mean = g.mean((1, 3), keepdim=True)
    var = ((g - mean) ** 2).mean((1, 3), keepdim=True)
    return ((g - mean) / torch.sqrt(var + eps)).reshape(x.shape) * gamma + beta


def _attend(q, k, v, heads, causal=False):
    """[B,S,C] each, one (image, head) at a time."""
    B, Sq, C = q.shape
    d, out = C // heads, torch.empty_like(q)
    for b in range(B):
        for h in range(heads):
            j = slice(h * d, (h + 1) * d)
            s = q[b, :, j].contiguous() @ k[b, :, j].t().contiguous() / math.sqrt(d)
            if causal:
                s = s.masked_fill(torch.ones(Sq, Sq, dtype=torch.bool, device=DEV).triu(1), -math.inf)
            out[b, :, j] = torch.softmax(s, -1) @ v[b, :, j].contiguous()
    return out


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _unet(x):
    P = _Weights(0.02)
    lat, ctx, temb = x["lat"].double().permute(0, 2, 3, 1).contiguous(), x["ctx"].double(), x["temb"].double()
    t = F.silu(_lin(temb, P("time_embedding.linear_1.weight", 1280, 320), P("time_embedding.linear_1.bias", 1280)))
    t = _lin(t, P("time_embedding.linear_2.weight", 1280, 1280), P("time_embedding.linear_2.bias", 1280))

    def norm(pf, v, act, eps=1e-5):
        C = v.shape[-1]
        y = _gn(v, P(pf + ".weight", C, norm=True), P(pf + ".bias", C), eps)
        return F.silu(y) if act else y

    def conv(pf, v, co, stride=1):
        return _conv3(v, P(pf + ".weight", co, v.shape[-1], 3, 3), P(pf + ".bias", co), stride)

    def lin(pf, v, co, bias=True, conv1=False):
        w = P(pf + ".weight", *((co, v.shape[-1], 1, 1) if conv1 else (co, v.shape[-1]))).reshape(co, -1)
        return _lin(v, w, P(pf + ".bias", co) if bias else None)

    def ln(pf, v):
        C = v.shape[-1]
        return F.layer_norm(v, (C,), P(pf + ".weight", C, norm=True), P(pf + ".bias", C), 1e-5)

    def resnet(pf, v, co):
        h = conv(pf + ".conv1", norm(pf + ".norm1", v, True), co)
        h = h + lin(pf + ".time_emb_proj", F.silu(t), co)
        h = conv(pf + ".conv2", norm(pf + ".norm2", h, True), co)
        return h + (lin(pf + ".conv_shortcut", v, co, conv1=True) if v.shape[-1] != co else v)

    def transformer(pf, v):
        B, H, W, C = v.shape
        b = pf + ".transformer_blocks.0"
        u = lin(pf + ".proj_in", norm(pf + ".norm", v, False), C, conv1=True).reshape(B, H * W, C)
        for i, kv in ((1, None), (2, ctx)):
            h = ln(f"{b}.norm{i}", u)
            kv = h if kv is None else kv
            a = _attend(lin(f"{b}.attn{i}.to_q", h, C, False), lin(f"{b}.attn{i}.to_k", kv, C, False),
                        lin(f"{b}.attn{i}.to_v", kv, C, False), 8)
            u = u + lin(f"{b}.attn{i}.to_out.0", a, C)
        f = lin(b + ".ff.net.0.proj", ln(b + ".norm3", u), 8 * C)
        u = u + lin(b + ".ff.net.2", f[..., :4 * C] * _gelu(f[..., 4 * C:]), C)
        return v + lin(pf + ".proj_out", u, C, conv1=True).reshape(B, H, W, C)

    chans = (320, 640, 1280, 1280)
    h = conv("conv_in", lat, 320)
    skips = [h]
    for i, co in enumerate(chans):
        for r in range(2):
            h = resnet(f"down_blocks.{i}.resnets.{r}", h, co)
            h = transformer(f"down_blocks.{i}.attentions.{r}", h) if i < 3 else h
            skips.append(h)
        if i < 3:
            h = conv(f"down_blocks.{i}.downsamplers.0.conv", h, co, 2)
            skips.append(h)
    h = resnet("mid_block.resnets.0", h, 1280)
    h = transformer("mid_block.attentions.0", h)
    h = resnet("mid_block.resnets.1", h, 1280)
    for i, co in enumerate(chans[::-1]):
        for r in range(3):
            h = resnet(f"up_blocks.{i}.resnets.{r}", torch.cat([h, skips.pop()], -1), co)
            h = transformer(f"up_blocks.{i}.attentions.{r}", h) if i > 0 else h
        h = conv(f"up_blocks.{i}.upsamplers.0.conv", _up(h), co) if i < 3 else h
    return conv("conv_out", norm("conv_norm_out", h, True), 4).permute(0, 3, 1, 2).contiguous()


def _clip(x):
    P = _Weights(0.02)
    ids = x["ids"].long()
    B, C = ids.shape[0], 768
    h = P("text_model.embeddings.token_embedding.weight", 49408, C)[ids] + P("text_model.embeddings.position_embedding.weight", 77, C)

    def lin(pf, v, co):
        return _lin(v, P(pf + ".weight", co, v.shape[-1]), P(pf + ".bias", co))

    def ln(pf, v):
        return F.layer_norm(v, (C,), P(pf + ".weight", C, norm=True), P(pf + ".bias", C), 1e-5)

    for i in range(12):
        pf = f"text_model.encoder.layers.{i}"
        n = ln(pf + ".layer_norm1", h)
        a = _attend(*(lin(f"{pf}.self_attn.{p}_proj", n, C) for p in "qkv"), 12, causal=True)
        h = h + lin(pf + ".self_attn.out_proj", a, C)
        f = lin(pf + ".mlp.fc1", ln(pf + ".layer_norm2", h), 3072)
        h = h + lin(pf + ".mlp.fc2", f * torch.sigmoid(1.702 * f), C)
    return ln("text_model.final_layer_norm", h)


def _taesd(x):
    P = _Weights(0.04)

    def conv(i, v, co=64, bias=True):
        return _conv3(v, P(f"decoder.layers.{i}.weight", co, v.shape[-1], 3, 3), P(f"decoder.layers.{i}.bias", co) if bias else None)

    h = (torch.tanh(x["lat"].double() / 3.0) * 3.0).permute(0, 2, 3, 1).contiguous()
    h = F.relu(conv(0, h))
    i = 2
    for blocks in (3, 3, 3, 1):
        for _ in range(blocks):
            y = F.relu(conv(f"{i}.conv.0", h))
            y = F.relu(conv(f"{i}.conv.2", y))
            h = F.relu(conv(f"{i}.conv.4", y) + h)
            i += 1
        if blocks == 3:
            h = conv(i + 1, _up(h), bias=False)
            i += 2
    return (2.0 * conv(i, h, 3) - 1.0).permute(0, 3, 1, 2).contiguous()


def _vae(x):
    P = _Weights(0.02, 0.1)

    def norm(pf, v, act):
        C = v.shape[-1]
        y = _gn(v, P(pf + ".weight", C, norm=True), P(pf + ".bias", C), 1e-6)
        return F.silu(y) if act else y

    def conv(pf, v, co):
        return _conv3(v, P(pf + ".weight", co, v.shape[-1], 3, 3), P(pf + ".bias", co))

    def one(pf, v, co):
        return _lin(v, P(pf + ".weight", co, v.shape[-1], 1, 1).reshape(co, -1), P(pf + ".bias", co))

    def resnet(pf, v, co):
        h = conv(pf + ".conv1", norm(pf + ".norm1", v, True), co)
        h = conv(pf + ".conv2", norm(pf + ".norm2", h, True), co)
        return h + (one(pf + ".conv_shortcut", v, co) if v.shape[-1] != co else v)

    h = one("post_quant_conv", (x["lat"].double() / 0.18215).permute(0, 2, 3, 1).contiguous(), 4)
    h = resnet("decoder.mid_block.resnets.0", conv("decoder.conv_in", h, 512), 512)
    a = "decoder.mid_block.attentions.0"
    n = norm(a + ".group_norm", h, False).reshape(h.shape[0], -1, 512)
    q, k, v = (_lin(n, P(f"{a}.to_{p}.weight", 512, 512), P(f"{a}.to_{p}.bias", 512)) for p in "qkv")
    h = h + _lin(_attend(q, k, v, 1), P(a + ".to_out.0.weight", 512, 512), P(a + ".to_out.0.bias", 512)).reshape(h.shape)
    h = resnet("decoder.mid_block.resnets.1", h, 512)
    for i, co in enumerate((512, 512, 256, 128)):
        for j in range(3):
            h = resnet(f"decoder.up_blocks.{i}.resnets.{j}", h, co)
        h = conv(f"decoder.up_blocks.{i}.upsamplers.0.conv", _up(h), co) if i < 3 else h
    return conv("decoder.conv_out", norm("decoder.conv_norm_out", h, True), 3).permute(0, 3, 1, 2).contiguous()


def exact(case, seed):
    c, op = case, case["op"]
    if op == "unet" and c["B"] * c["H"] * c["W"] > 4 * 64 * 64:
        return None  # minutes, at the largest batch
    with torch.no_grad():
        x = _inputs(case, seed)
        if op in ("unet", "clip", "taesd", "vae"):
            return {"unet": _unet, "clip": _clip, "taesd": _taesd, "vae": _vae}[op](x)
        x = {k: v.double() for k, v in x.items()}
        if op == "conv":
            v = _up(x["x"]) if c["up"] else x["x"]
            if c["k"] == 3:
                y = _conv3(v, x["w"].permute(0, 3, 1, 2), x["bias"], c["stride"])
            else:
                y = _lin(v, x["w"].reshape(c["Co"], -1), x["bias"])
            y = y + x["temb"] if c["temb"] else y
            y = y + x["res"] if c["res"] else y
            return F.relu(y) if c["relu"] else y
        if op == "attn":
            return _attend(x["q"], x["k"], x["v"], c["heads"], c["causal"])
        if op == "matmul":
            y = _lin(x["a"], x["w"], x["bias"])
            if c["geglu"]:  # rows of w go in blocks of 32 values and their 32 gates
                y = y.reshape(c["M"], -1, 2, 32)
                y = (y[:, :, 0] * _gelu(y[:, :, 1])).reshape(c["M"], -1)
            y = y + x["res"] if c["res"] else y
            return y * torch.sigmoid(1.702 * y) if c["gelu"] else y
        if op == "gnorm":
            y = _gn(torch.cat([x["x"], x["x2"]], -1) if c["C2"] else x["x"], x["gamma"], x["beta"], 1e-5)
            return F.silu(y) if c["silu"] else y
        return F.layer_norm(x["x"], (c["C"],), x["gamma"], x["beta"], 1e-5)
