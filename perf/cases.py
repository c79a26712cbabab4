"""The work that programs have this library do, as timed and checked cases.

Every case is one pass through a public entry point (`HipBackend`, `run_tiled`)
of the package: a whole image through one of the model families the library
serves, or one residual Swin stage on a feature plane. `via` names the entry:

  device    forward_device: an image in HBM to an image in HBM
  noalloc   forward_device_noalloc: the same on the library's static workspace
  batch     forward_device_batch: several images of one size in HBM, two lanes
  host      forward: host arrays in and out (and the aux image where the head
            makes one), upload and download included
  tiled     run_tiled(batch=True): a host image cut into tiles with context,
            the crops in one batched call, the tiles pasted together
  rstb      rstb_device: one stage (6 Swin blocks and the closing conv) on an
            unpadded channel-last plane

Images are u8-quantised sinusoid textures with noise, as a decoded photograph
or video frame arrives, mean-adjusted as the crate hands them over. The weights
are synthetic checkpoints in the crate's layout with every bias, norm and logit
scale off its trivial value, loaded once per model, as a program that serves
many images does. torch is imported before the library, so that both share one
HIP runtime and torch tensors are its device buffers.
"""
import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
M = pkg.model

DEV = "cuda"

# the model families at their released widths and heads
FAMILIES = {
    "classical": lambda scale: M.classical(scale),
    "lightweight": lambda scale: M.lightweight(scale),
    "realworld": lambda scale: M.realworld(),
    "compressed": lambda scale: M.compressed(),
}
SCALES = {"classical": (2, 4, 8), "lightweight": (2, 3, 4), "realworld": (4,), "compressed": (4,)}
SEEDS = {"classical": 3, "lightweight": 0, "realworld": 4, "compressed": 5}


def listed():
    def image(name, family, scale, via, h, w, n=1, **more):
        return dict(name=name, family=family, scale=scale, via=via, h=h, w=w, n=n, **more)

    return [
        # the lightweight model's benchmark size: a chat avatar or thumbnail,
        # where the number of launches is what counts
        image("light_x2_64", "lightweight", 2, "device", 64, 64),
        # a ragged thumbnail under a caller that may not allocate
        image("light_x3_45x71", "lightweight", 3, "noalloc", 45, 71),
        # a quarter-HD video frame through the lightweight model
        image("light_x2_540x960", "lightweight", 2, "device", 540, 960),
        # the smallest request of the classical model, from and to host memory
        image("classical_x4_24x40", "classical", 4, "host", 24, 40),
        # the headline: 256^2 -> 1024^2
        image("classical_x4_256", "classical", 4, "device", 256, 256),
        # four odd-sized pictures of one size at once: a serving queue
        image("classical_x4_91x127_n4", "classical", 4, "batch", 91, 127, 4),
        # a whole 720p frame, the largest plane this path meets untiled
        image("classical_x4_720x1280", "classical", 4, "device", 720, 1280),
        # the classical x2 benchmark size (another head)
        image("classical_x2_256", "classical", 2, "device", 256, 256),
        # the real-world model on a VGA camera frame (nearest+conv head)
        image("realworld_x4_480x640", "realworld", 4, "device", 480, 640),
        # the compressed model's tile loop, 256-pixel tiles with 64 of context
        image("compressed_x4_tiled", "compressed", 4, "tiled", 512, 600, tile=256, pad=64),
        # one stage on the micro-benchmark's plane, and on a small one
        dict(name="rstb_256", family="classical", scale=4, via="rstb", h=256, w=256, n=1),
        dict(name="rstb_40x72", family="classical", scale=4, via="rstb", h=40, w=72, n=1),
    ]


# the largest listed case's padded pixels, which no drawn one passes
MOST = 728 * 1288


def draw(rng):
    family = rng.choice(("classical", "classical", "classical", "lightweight", "lightweight",
                         "realworld", "compressed"))
    scale = rng.choice(SCALES[family])
    via = rng.choice(("device", "device", "device", "host", "batch", "noalloc", "tiled", "rstb"))
    # heads that work on the upscaled plane (8x, nearest+conv, the bicubic
    # branch) cost more per pixel; host entries, tile loops (whose crops
    # overlap) and batches are met at moderate sizes
    most = {"classical": MOST, "lightweight": MOST, "realworld": MOST // 4, "compressed": MOST // 2}[family]
    if scale == 8:
        most = MOST // 4
    n = 1
    if via == "batch":
        n = rng.randint(2, 5)
        most = min(most // n, 256 * 256)
    elif via in ("host", "tiled"):
        most = min(most, 384 * 512)
    elif via == "noalloc":
        # what fits the 256 MiB workspace in every family
        most = {"classical": 104 * 104, "compressed": 104 * 104, "realworld": 80 * 80,
                "lightweight": 192 * 192}[family]
    least = 16 if via == "tiled" else 8
    px = math.exp(rng.uniform(math.log(least * least * 2), math.log(most)))
    aspect = math.exp(rng.uniform(math.log(0.4), math.log(2.5)))
    h = max(least, int(math.sqrt(px * aspect)))
    w = max(least, int(px / h))
    if via == "rstb":
        h, w = max(8, h // 8 * 8), max(8, w // 8 * 8)
    while (h // 8 + 1) * (w // 8 + 1) * 64 > most + 64 * 16 and max(h, w) > 16:
        h, w = (h - 1, w) if h > w else (h, w - 1)
    c = dict(family=family, scale=scale, via=via, h=h, w=w, n=n)
    if via == "tiled":
        c["tile"], c["pad"] = rng.choice((128, 200, 256)), rng.choice((16, 32, 64))
    return c


def arch_of(case):
    return FAMILIES[case["family"]](case["scale"])


_weights, _models = {}, {}


def weights_of(case):
    key = (case["family"], case["scale"])
    if key not in _weights:
        _weights[key] = M.make_weights(arch_of(case), seed=SEEDS[case["family"]], perturb=True)
    return _weights[key]


def model_of(case):
    """The loaded model: one context per checkpoint for the program's life."""
    key = (case["family"], case["scale"])
    if key not in _models:
        _models[key] = pkg.HipBackend(arch_of(case), weights_of(case))
    return _models[key]


def pictures(case, seed):
    """[n][3][h][w] in [0, 1], on the GPU: eight random sinusoids per picture
    and gaussian noise of four levels, quantised to u8."""
    g = torch.Generator(device="cpu").manual_seed(seed)
    n, h, w = case["n"], case["h"], case["w"]
    y = torch.arange(h, device=DEV, dtype=torch.float64)[:, None]
    x = torch.arange(w, device=DEV, dtype=torch.float64)[None, :]
    img = torch.full((n, 3, h, w), 128.0, device=DEV, dtype=torch.float64)
    u = torch.rand((n, 8, 6), generator=g, dtype=torch.float64).tolist()
    for i in range(n):
        for fy, fx, amp, *phase in u[i]:
            for c in range(3):
                img[i, c] += (6 + 14 * amp) * torch.sin(
                    2 * math.pi * (0.15 * fy * y + 0.15 * fx * x + phase[c]))
    noise = torch.Generator(device=DEV).manual_seed(seed + 1)
    img += 4 * torch.randn(img.shape, generator=noise, device=DEV, dtype=torch.float64)
    return (img.round().clamp(0, 255).float() / 255.0)


def adjusted(arch, img):
    mean = torch.tensor(arch.mean, dtype=torch.float32, device=img.device)[:, None, None]
    return ((img - mean) * arch.img_range).contiguous()


def plane(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn((case["h"] * case["w"], arch_of(case).embed), generator=g, device=DEV)


def prepare(case, seed):
    arch, via = arch_of(case), case["via"]
    st = {"case": case, "arch": arch, "model": model_of(case)}
    h, w, s = case["h"], case["w"], arch.scale
    if via == "rstb":
        st["in"] = plane(case, seed)
        st["out"] = torch.empty_like(st["in"])
    elif via == "tiled":
        st["in"] = pictures(case, seed)[0].cpu().numpy()
    elif via == "host":
        st["in"] = adjusted(arch, pictures(case, seed)[0]).cpu().numpy()
    else:
        st["in"] = adjusted(arch, pictures(case, seed))
        st["out"] = torch.empty((case["n"], 3, h * s, w * s), device=DEV)
    # the inputs are ready before the library's own stream reads them
    torch.cuda.synchronize()
    return st


def run(st):
    case, be = st["case"], st["model"]
    h, w, via = case["h"], case["w"], case["via"]
    if via == "device":
        be.forward_device(h, w, st["in"].data_ptr(), st["out"].data_ptr())
    elif via == "noalloc":
        be.forward_device_noalloc(h, w, st["in"].data_ptr(), st["out"].data_ptr())
    elif via == "batch":
        be.forward_device_batch(h, w, [t.data_ptr() for t in st["in"]],
                                [t.data_ptr() for t in st["out"]])
    elif via == "rstb":
        be.rstb_device(0, h, w, st["in"].data_ptr(), st["out"].data_ptr())
    elif via == "tiled":
        return pkg.tiling.run_tiled(st["arch"], be, st["in"], case["tile"], case["pad"], batch=True)
    else:
        out = be.forward(h, w, st["in"])
        aux = be.aux()
        return out if aux is None else [out, aux]
    return st["out"]


def crops(case):
    """The (y0, y1, x0, x1) of every forward of one pass."""
    h, w = case["h"], case["w"]
    if case["via"] != "tiled":
        return [(0, h, 0, w)] * case["n"]
    t = max(case["tile"] // 8, 1) * 8
    p = max(-(-case["pad"] // 8), 1) * 8
    return [(max(y - p, 0), min(y + t + p, h), max(x - p, 0), min(x + t + p, w))
            for y in range(0, h, t) for x in range(0, w, t)]


def work(case):
    """The network's own multiply-adds (the 1x1 convs folded into the 3x3 ones
    before them), each image and each weight once."""
    a = arch_of(case)
    C, F, s = a.embed, a.feat, a.scale
    block = 2 * (3 + 1 + 2 * a.mlp_ratio) * C * C + 4 * 64 * C
    conv = lambda i, o: 18 * i * o
    flops = 0.0
    for y0, y1, x0, x1 in crops(case):
        if case["via"] == "rstb":
            flops += case["h"] * case["w"] * (a.depths[0] * block + conv(C, C))
            continue
        P = ((y1 - y0) // 8 + 1) * ((x1 - x0) // 8 + 1) * 64
        per = 2 * conv(3, C) + sum(a.depths) * block + (len(a.depths) + 1) * conv(C, C)
        if a.upsampler == "pixelshuffledirect":
            per += conv(C, 3 * s * s)
        else:
            per += conv(C, F) + s * s * conv(F, 3)
            if a.upsampler == "nearest+conv":
                per += (4 + 16 + 16) * conv(F, F)
            else:
                per += sum(4 ** o * conv(F, 4 * F) for o in range(a.octaves))
                if a.upsampler == "pixelshuffle_aux":
                    per += conv(F, 3) + conv(3, F) + s * s * conv(3, F)
        flops += P * per
    if case["via"] == "rstb":
        per_image = 2 * case["h"] * case["w"] * C
        weights = a.depths[0] * 8 * C * C + 9 * C * C
    else:
        per_image = case["n"] * case["h"] * case["w"] * 3 * (1 + s * s)
        weights = sum(a.depths) * 8 * C * C + (len(a.depths) + 1) * 9 * C * C
    return {"bytes": 4.0 * (per_image + weights), "flops": float(flops)}


def tolerance(case):
    # fp32 sums of up to 3,240 terms through 25 to 43 layers. Against 64 bits an
    # image is 0.4 to 3.4e-7 off, a drawn one at most 7.1e-7 (its values sit
    # around the RGB mean of 0.4), a stage's plane 2.7e-6.
    return {"rel": 1.2e-5} if case["via"] == "rstb" else {"rel": 2e-6}


# ---------------------------------------------------------------------------
# The same network in 64 bits, in plain torch, as published: torch.roll and
# window partition, post-norm blocks, direct convolutions, every octave's plane.
# Planes are [h][w][c].
# ---------------------------------------------------------------------------

def _conv(x, w, b):
    h, wd, ci = x.shape
    k = w.shape[-1]
    y = b.expand(h * wd, -1).clone()
    r = k // 2
    xp = torch.zeros((h + 2 * r, wd + 2 * r, ci), dtype=x.dtype, device=x.device)
    xp[r:r + h, r:r + wd] = x
    for i in range(k):
        for j in range(k):
            y += xp[i:i + h, j:j + wd].reshape(-1, ci) @ w[:, :, i, j].t().contiguous()
    return y.reshape(h, wd, -1)


def _norm(x, w, b):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w, b, 1e-5)


def _shuffle(x, r):
    h, w, c = x.shape
    return (x.reshape(h, w, c // (r * r), r, r).permute(0, 3, 1, 4, 2)
            .reshape(h * r, w * r, c // (r * r)))


def _lrelu(x, slope):
    return torch.nn.functional.leaky_relu(x, slope)


def _bias_table(g):
    r = torch.arange(-7, 8, dtype=torch.float64, device=DEV) / 7 * 8
    t = torch.stack(torch.meshgrid(r, r, indexing="ij"), -1).reshape(-1, 2)
    t = torch.sign(t) * torch.log2(t.abs() + 1) / 3
    m = torch.relu(t @ g("attn.cpb_mlp.0.weight").t() + g("attn.cpb_mlp.0.bias"))
    m = m @ g("attn.cpb_mlp.2.weight").t()
    i = torch.arange(64, device=DEV)
    dy = i[:, None] // 8 - i[None, :] // 8 + 7
    dx = i[:, None] % 8 - i[None, :] % 8 + 7
    return (16 * torch.sigmoid(m))[dy * 15 + dx].permute(2, 0, 1)


def _windows(x):
    h, w, c = x.shape
    return x.reshape(h // 8, 8, w // 8, 8, c).transpose(1, 2).reshape(-1, 64, c)


def _block(x, g, heads, shift):
    h, w, c = x.shape
    xs = torch.roll(x, (-shift, -shift), (0, 1)) if shift else x
    t = _windows(xs)
    n = t.shape[0]

    def split(v):
        return v.reshape(n, 64, heads, c // heads).transpose(1, 2).contiguous()

    q = split(t @ g("attn.qkv.wq").t().contiguous() + g("attn.qkv.q_bias"))
    k = split(t @ g("attn.qkv.wk").t().contiguous())
    v = split(t @ g("attn.qkv.wv").t().contiguous() + g("attn.qkv.v_bias"))
    q = torch.nn.functional.normalize(q, dim=-1)
    k = torch.nn.functional.normalize(k, dim=-1)
    s = q @ k.transpose(-1, -2).contiguous()
    s = s * g("attn.logit_scale").reshape(1, heads, 1, 1).clamp(max=math.log(100.0)).exp()
    s += _bias_table(g)
    if shift:
        band = lambda m: ((torch.arange(m, device=DEV) >= m - 8).long()
                          + (torch.arange(m, device=DEV) >= m - shift).long())
        reg = _windows((band(h)[:, None] * 3 + band(w)[None, :])[..., None])[..., 0]
        s -= 100.0 * (reg[:, :, None] != reg[:, None, :]).double()[:, None]
    o = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(n, 64, c)
    o = o @ g("attn.proj.weight").t().contiguous() + g("attn.proj.bias")
    o = o.reshape(h // 8, w // 8, 8, 8, c).transpose(1, 2).reshape(h, w, c)
    if shift:
        o = torch.roll(o, (shift, shift), (0, 1))
    x = x + _norm(o, g("norm1.weight"), g("norm1.bias"))
    m = torch.nn.functional.gelu(x @ g("mlp.fc1.weight").t().contiguous() + g("mlp.fc1.bias"))
    m = m @ g("mlp.fc2.weight").t().contiguous() + g("mlp.fc2.bias")
    return x + _norm(m, g("norm2.weight"), g("norm2.bias"))


def _stage(x, g, a, i):
    y = x
    for b in range(a.depths[i]):
        p = "layers.%d.residual_group.blocks.%d." % (i, b)
        y = _block(y, lambda k: g(p + k), a.heads, 0 if b % 2 == 0 else 4)
    y = _conv(y, g("layers.%d.conv.weight" % i), g("layers.%d.conv.bias" % i))
    p = "layers.%d.patch_embed.proj." % i
    return _conv(y, g(p + "weight"), g(p + "bias")) + x


def _bicubic(x, s):
    y = torch.nn.functional.interpolate(x.permute(2, 0, 1)[None], scale_factor=s, mode="bicubic",
                                        align_corners=False)
    return y[0].permute(1, 2, 0).contiguous()


def _network(a, g, x, h, w):
    """(the [3][h s][w s] image, the padded aux image or None) of a
    mean-adjusted [3][h][w] image."""
    hp, wp, s = (h // 8 + 1) * 8, (w // 8 + 1) * 8, a.scale
    x = torch.cat([x, x.flip(1)], 1)[:, :hp]
    x = torch.cat([x, x.flip(2)], 2)[:, :, :wp].permute(1, 2, 0).contiguous()
    conv = lambda v, name: _conv(v, g(name + ".weight"), g(name + ".bias"))
    first = conv(x, "conv_first")
    f = _norm(conv(first, "patch_embed.proj"), g("patch_embed.norm.weight"), g("patch_embed.norm.bias"))
    for i in range(len(a.depths)):
        f = _stage(f, g, a, i)
    f = conv(_norm(f, g("norm.weight"), g("norm.bias")), "conv_after_body") + first
    mean = torch.tensor(a.mean, dtype=torch.float32).double().to(DEV)
    finish = lambda v: (v / a.img_range + mean).permute(2, 0, 1).contiguous()
    aux = None
    if a.upsampler == "pixelshuffledirect":
        y = _shuffle(conv(f, "upsample.0"), s)
    else:
        y = _lrelu(conv(f, "conv_before_upsample.0"), 0.01)
        if a.upsampler == "nearest+conv":
            for name in ("conv_up1", "conv_up2"):
                y = y.repeat_interleave(2, 0).repeat_interleave(2, 1)
                y = _lrelu(conv(y, name), 0.2)
            y = conv(_lrelu(conv(y, "conv_hr"), 0.2), "conv_last")
        else:
            if a.upsampler == "pixelshuffle_aux":
                aux = conv(y, "conv_aux")
                y = _lrelu(conv(aux, "conv_after_aux.0"), 0.01)
            for o in range(a.octaves):
                y = _shuffle(conv(y, "upsample.%d" % (2 * o)), 2)
            if aux is not None:
                y = y + conv(_bicubic(x, s), "conv_bicubic")
                aux = finish(aux)
            y = conv(y, "conv_last")
    return finish(y[:h * s, :w * s]), aux


def exact(case, seed):
    a, via = arch_of(case), case["via"]
    wts = weights_of(case)
    held = {}

    def g(name):
        if name not in held:
            held[name] = torch.from_numpy(np.ascontiguousarray(wts[name])).to(DEV).double()
        return held[name]

    h, w, s = case["h"], case["w"], a.scale
    if via == "rstb":
        x = plane(case, seed).double().reshape(h, w, -1)
        return _stage(x, g, a, 0).reshape(h * w, -1)
    img = pictures(case, seed)
    if via == "tiled":
        out = torch.zeros((3, h * s, w * s), dtype=torch.float64, device=DEV)
        t = max(case["tile"] // 8, 1) * 8
        at = [(y, x) for y in range(0, h, t) for x in range(0, w, t)]
        for (y, x), (y0, y1, x0, x1) in zip(at, crops(case)):
            r, _ = _network(a, g, adjusted(a, img[0, :, y0:y1, x0:x1]).double(), y1 - y0, x1 - x0)
            r = r[:, (y - y0) * s:(min(y + t, h) - y0) * s, (x - x0) * s:(min(x + t, w) - x0) * s]
            out[:, y * s:y * s + r.shape[1], x * s:x * s + r.shape[2]] = r
        return out.cpu().numpy()
    got = [_network(a, g, x.double(), h, w) for x in adjusted(a, img)]
    if via == "host":
        out, aux = got[0]
        return out.cpu().numpy() if aux is None else [out.cpu().numpy(), aux.cpu().numpy().reshape(-1)]
    return torch.stack([o for o, _ in got])
