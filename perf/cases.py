"""Timed cases of the codec: the calls a program makes, at the sizes it makes
them.

listed() names fixed cases, draw(rng) makes more of the same ranges;
prepare(case, seed) makes what a program holds before the call (pictures,
blocks, buffers, a batch handle), run(state) is one call and returns its whole
output, work(case) the bytes and operations the call cannot do without.

Case keys: "op" (which entry point), "fmt", "alg", "w", "h", and where the
entry point takes them "weights" (perceptual / uniform), "by_alpha" (weigh
colour by alpha), "alpha" (opaque / field / cutout: the picture's alpha
channel), "stream" (library: the library's own stream, caller: one of the
program's), "count" / "side" (textures of a batch and their longest side).

The outputs are block bytes and pixels: whole values, bit-exact.
"""
import math
import random

import numpy as np
import torch
import torch.nn.functional as F

import texpresso_amd as tx

FORMATS = ("Bc1", "Bc2", "Bc3", "Bc4", "Bc5")
ALGORITHMS = ("RangeFit", "ClusterFit", "IterativeClusterFit")
WEIGHTS = {"perceptual": tx.COLOUR_WEIGHTS_PERCEPTUAL, "uniform": tx.COLOUR_WEIGHTS_UNIFORM}


def listed():
    return [
        # the smallest call: one icon from host memory to host memory, as an
        # editor's thumbnail cache or a user interface packer makes it
        {"name": "icon-host-bc1-64", "op": "compress", "fmt": "Bc1", "alg": "ClusterFit", "w": 64, "h": 64,
         "weights": "perceptual", "by_alpha": False, "alpha": "opaque"},
        # an ordinary opaque texture with the default parameters
        {"name": "albedo-bc1-512", "op": "compress_device", "fmt": "Bc1", "alg": "ClusterFit", "w": 512, "h": 512,
         "weights": "perceptual", "by_alpha": False, "alpha": "opaque", "stream": "library"},
        # the largest: a final-quality bake of a texture with an alpha channel
        {"name": "bake-bc3-iterative-2048", "op": "compress_device", "fmt": "Bc3", "alg": "IterativeClusterFit",
         "w": 2048, "h": 2048, "weights": "perceptual", "by_alpha": False, "alpha": "field", "stream": "library"},
        # a tangent-space normal map
        {"name": "normals-bc5-2048", "op": "compress_device", "fmt": "Bc5", "alg": "ClusterFit", "w": 2048, "h": 2048,
         "weights": "perceptual", "by_alpha": False, "alpha": "opaque", "stream": "library"},
        # a fast preview of a screen-sized picture, neither side a multiple of 4
        {"name": "preview-bc1-range-1366x767", "op": "compress_device", "fmt": "Bc1", "alg": "RangeFit", "w": 1366,
         "h": 767, "weights": "perceptual", "by_alpha": False, "alpha": "cutout", "stream": "library"},
        # foliage with a cutout alpha, colours weighed by it, on the caller's stream
        {"name": "foliage-bc2-1021x1531", "op": "compress_device", "fmt": "Bc2", "alg": "ClusterFit", "w": 1021,
         "h": 1531, "weights": "uniform", "by_alpha": True, "alpha": "cutout", "stream": "caller"},
        # an asset with all its levels, pixels already on the device
        {"name": "chain-bc3-1024", "op": "compress_mips_device", "fmt": "Bc3", "alg": "ClusterFit", "w": 1024,
         "h": 1024, "weights": "perceptual", "by_alpha": False, "alpha": "field", "stream": "caller"},
        # importing a ragged picture with all its levels from host memory
        {"name": "import-bc1-iterative-500x375", "op": "compress_mips", "fmt": "Bc1", "alg": "IterativeClusterFit",
         "w": 500, "h": 375, "weights": "perceptual", "by_alpha": False, "alpha": "cutout"},
        # reading a large texture back
        {"name": "decode-bc3-4096", "op": "decompress_device", "fmt": "Bc3", "w": 4096, "h": 4096,
         "stream": "library"},
        # and a small ragged one of two channels, between host buffers
        {"name": "decode-host-bc5-333x250", "op": "decompress", "fmt": "Bc5", "w": 333, "h": 250},
        # the levels of a wide picture alone
        {"name": "levels-4096x2048", "op": "generate_mips_device", "w": 4096, "h": 2048, "stream": "library"},
        # a scene's textures of mixed sizes and formats with their levels, as
        # one batch that is run again whenever the pictures change
        {"name": "scene-batch-24", "op": "batch", "alg": "ClusterFit", "count": 24, "side": 768},
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(("compress_device",) * 5 + ("compress", "compress_mips_device", "compress_mips",
                                                "decompress_device", "decompress", "generate_mips_device", "batch"))
    if op == "batch":
        return {"op": op, "alg": rng.choice(ALGORITHMS), "count": side(8, 32), "side": side(64, 768)}
    stream = rng.choice(("library", "caller"))
    if op == "generate_mips_device":
        return {"op": op, "w": side(64, 4096), "h": side(64, 4096), "stream": stream}
    fmt = rng.choice(FORMATS)
    if op in ("decompress", "decompress_device"):
        low, top = (384, 4096) if op == "decompress_device" else (16, 1024)
        case = {"op": op, "fmt": fmt, "w": side(low, top), "h": side(low, top)}
    else:
        alg = rng.choice(ALGORITHMS)
        quick = alg == "RangeFit" or fmt in ("Bc4", "Bc5")
        low = 256 if op == "compress_device" and quick else 16
        top = {"compress_device": 4096 if quick else 1800, "compress_mips_device": 1500}.get(op, 1024)
        case = {"op": op, "fmt": fmt, "alg": alg, "w": side(low, top), "h": side(low, top),
                "weights": rng.choice(("perceptual", "perceptual", "uniform")), "by_alpha": rng.random() < 0.25,
                "alpha": rng.choice(("opaque", "field", "cutout"))}
    if op.endswith("_device"):
        case["stream"] = stream
    return case


# ---------------------------------------------------------------- pictures


def picture(w, h, seed, alpha="opaque"):
    """An RGBA8 picture on the GPU, (h, w, 4): four octaves of noise, a
    gradient, hard-edged shapes (a quarter of them filled with one colour),
    and the alpha channel asked for."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = random.Random(seed)

    def noise(channels, period, amp):
        gw, gh = w // period + 2, h // period + 2
        lattice = (torch.rand((1, channels, gh, gw), generator=gen, device="cuda") * 2 - 1) * amp
        return F.interpolate(lattice, size=(gh * period, gw * period), mode="bilinear")[0, :, :h, :w]

    img = torch.full((3, h, w), 128.0, device="cuda")
    for period, amp in ((64, 96.0), (32, 48.0), (16, 24.0), (8, 12.0)):
        img += noise(3, period, amp)
    turn = rng.uniform(0.0, 2 * math.pi)
    img += 200.0 * math.cos(turn) * (torch.arange(w, device="cuda") / w - 0.5)
    img += 200.0 * math.sin(turn) * (torch.arange(h, device="cuda") / h - 0.5)[:, None]
    for k in range(24):
        x, y = rng.randrange(w), rng.randrange(h)
        part = img[:, y:y + rng.randint(8, 256), x:x + rng.randint(8, 256)]
        colour = torch.tensor([rng.uniform(-80, 80) for _ in range(3)], device="cuda")[:, None, None]
        if k % 4 == 0:
            part[:] = 128.0 + colour
        else:
            part += colour
    if alpha == "opaque":
        a = torch.full((1, h, w), 255.0, device="cuda")
    else:
        a = 128.0 + noise(1, 128, 100.0) + noise(1, 64, 50.0)
        hard = torch.where(a >= 128.0, 255.0, 0.0)
        if alpha == "field":  # smooth, with a tenth of the blocks binary
            pick = torch.rand((1, (h + 3) // 4, (w + 3) // 4), generator=gen, device="cuda") < 0.1
            pick = pick.repeat_interleave(4, 1).repeat_interleave(4, 2)[:, :h, :w]
            hard = torch.where(pick, hard, a)
        a = hard
    return torch.cat([img, a]).round().clamp(0, 255).to(torch.uint8).permute(1, 2, 0).contiguous()


def normals(w, h, seed):
    """A tangent-space normal map of a fractal height field, (h, w, 4)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    height = torch.zeros((h, w), device="cuda")
    amp = 64.0
    for period in (256, 128, 64, 32, 16):
        gw, gh = w // period + 2, h // period + 2
        lattice = torch.rand((1, 1, gh, gw), generator=gen, device="cuda") * 2 - 1
        height += amp * F.interpolate(lattice, size=(gh * period, gw * period), mode="bicubic")[0, 0, :h, :w]
        amp *= 0.5
    nx = (height.roll(1, 1) - height.roll(-1, 1)) * 0.5
    ny = (height.roll(1, 0) - height.roll(-1, 0)) * 0.5
    n = torch.stack([nx, ny, torch.ones_like(nx)])
    n = n / n.square().sum(0).sqrt()
    n = ((n * 0.5 + 0.5) * 255.0).round().clamp(0, 255)
    return torch.cat([n, torch.full((1, h, w), 255.0, device="cuda")]).to(torch.uint8).permute(1, 2, 0).contiguous()


# ------------------------------------------------------------------- cases


def _params(case):
    return tx.Params(tx.Algorithm[case.get("alg", "ClusterFit")], WEIGHTS[case.get("weights", "perceptual")],
                     case.get("by_alpha", False))


def _stream(case):
    return torch.cuda.Stream() if case.get("stream") == "caller" else None


def _handle(state):
    return state["stream"].cuda_stream if state["stream"] is not None else None


def _bytes(n):
    return torch.zeros(max(1, n), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        return _prepare_batch(case, seed)
    w, h = case["w"], case["h"]
    s = {"op": op, "w": w, "h": h, "stream": _stream(case)}
    if op == "generate_mips_device":
        s["levels"] = tx.mip_levels(w, h)
        s["rgba"] = picture(w, h, seed)
        s["chain"] = _bytes(tx.mip_chain_rgba_bytes(w, h, s["levels"]))
        return s
    fmt = s["fmt"] = tx.Format[case["fmt"]]
    s["params"] = _params(case)
    img = normals(w, h, seed) if fmt == tx.Format.Bc5 else picture(w, h, seed, case.get("alpha", "field"))
    size = fmt.compressed_size(w, h)
    if op in ("decompress", "decompress_device"):
        blocks = _bytes(size)
        torch.cuda.synchronize()
        fmt.compress_device(img.data_ptr(), w, h, tx.Params(tx.Algorithm.RangeFit), blocks.data_ptr(), size)
        torch.cuda.synchronize()
        if op == "decompress":
            s["blocks"], s["out"] = blocks.cpu().numpy(), np.zeros((h, w, 4), np.uint8)
        else:
            s["blocks"], s["out"] = blocks, _bytes(4 * w * h)
        return s
    if op in ("compress", "compress_mips"):
        s["rgba"] = img.cpu().numpy()
        s["out"] = np.zeros(size, np.uint8)
        return s
    s["rgba"] = img
    if op == "compress_mips_device":
        s["levels"] = tx.mip_levels(w, h)
        s["chain"] = _bytes(tx.mip_chain_rgba_bytes(w, h, s["levels"]))
        size = fmt.mip_chain_size(w, h, s["levels"])
    s["out"] = _bytes(size)
    return s


def _batch_items(case, seed):
    """(format, width, height) of every level of the batch's textures, the
    same sizes for every seed."""
    rng = random.Random(case["count"] * 4099 + case["side"])
    items = []
    for _ in range(case["count"]):
        w, h = (int(round(math.exp(rng.uniform(math.log(3), math.log(case["side"]))))) for _ in range(2))
        items.append((tx.Format[rng.choice(("Bc1", "Bc3", "Bc4", "Bc5"))], w, h))
    return items


def _prepare_batch(case, seed):
    s = {"op": "batch", "keep": [], "out": []}
    textures = []
    for k, (fmt, w, h) in enumerate(_batch_items(case, seed)):
        levels = tx.mip_levels(w, h)
        img = normals(w, h, seed + k) if fmt == tx.Format.Bc5 else picture(w, h, seed + k, "field")
        chain = _bytes(tx.mip_chain_rgba_bytes(w, h, levels))
        out = _bytes(fmt.mip_chain_size(w, h, levels))
        torch.cuda.synchronize()
        tx.generate_mips_device(img.data_ptr(), w, h, levels, chain.data_ptr(), chain.numel())
        at, to = 0, 0
        for level in range(levels):
            lw, lh = tx.mip_dims(w, h, level)
            src = img.data_ptr() if level == 0 else chain.data_ptr() + at
            textures.append((fmt, _params(case), src, out.data_ptr() + to, lw, lh))
            at += 0 if level == 0 else 4 * lw * lh
            to += fmt.compressed_size(lw, lh)
        s["keep"].append((img, chain))
        s["out"].append(out)
    torch.cuda.synchronize()
    s["batch"] = tx.Batch(textures, tx.tuned("batch-1000")[0])
    return s


def run(s):
    op = s["op"]
    if op == "batch":
        s["batch"].run()
        return s["out"]
    w, h = s["w"], s["h"]
    if op == "generate_mips_device":
        tx.generate_mips_device(s["rgba"].data_ptr(), w, h, s["levels"], s["chain"].data_ptr(), s["chain"].numel(),
                                _handle(s))
        return s["chain"]
    fmt = s["fmt"]
    if op == "compress":
        fmt.compress(s["rgba"], w, h, s["params"], s["out"])
    elif op == "compress_mips":
        return fmt.compress_mips(s["rgba"], w, h, s["params"])
    elif op == "compress_device":
        fmt.compress_device(s["rgba"].data_ptr(), w, h, s["params"], s["out"].data_ptr(), s["out"].numel(),
                            _handle(s))
    elif op == "compress_mips_device":
        fmt.compress_mips_device(s["rgba"].data_ptr(), w, h, s["params"], s["levels"], s["chain"].data_ptr(),
                                 s["chain"].numel(), s["out"].data_ptr(), s["out"].numel(), _handle(s))
        return {"chain": s["chain"], "out": s["out"]}
    elif op == "decompress":
        fmt.decompress(s["blocks"], w, h, s["out"])
    else:
        fmt.decompress_device(s["blocks"].data_ptr(), w, h, s["out"].data_ptr(), _handle(s))
    return s["out"]


# -------------------------------------------------------------------- work

# Operations per 4x4 block.  One ordering of 16 colours has 967 four-colour
# splits of 159 operations and 151 three-colour ones of 138; the front of a
# block (colour set, axis) and a range fit take about 1500; an alpha or
# single-channel block 16 distances to 14 codes.
SPLITS4, SPLITS3, FRONT, CHANNEL = 967 * 159, 151 * 138, 1500, 16 * 14 * 3


def _encode_work(fmt, alg, w, h):
    blocks = tx.num_blocks(w) * tx.num_blocks(h)
    ops = {"Bc1": 0, "Bc2": 16 * 3, "Bc3": CHANNEL, "Bc4": CHANNEL, "Bc5": 2 * CHANNEL}[fmt.name]
    if fmt in (tx.Format.Bc1, tx.Format.Bc2, tx.Format.Bc3):
        ops += FRONT
        if alg != "RangeFit":
            ops += SPLITS4 + (SPLITS3 if fmt == tx.Format.Bc1 else 0)
    return 4 * w * h + fmt.compressed_size(w, h), ops * blocks


def _levels(w, h):
    return [tx.mip_dims(w, h, k) for k in range(tx.mip_levels(w, h))]


def work(case):
    op = case["op"]
    total_bytes, total_ops = 0, 0
    if op == "batch":
        for fmt, w, h in _batch_items(case, 0):
            for lw, lh in _levels(w, h):
                b, o = _encode_work(fmt, case["alg"], lw, lh)
                total_bytes, total_ops = total_bytes + b, total_ops + o
        return {"bytes": total_bytes, "flops": total_ops}
    w, h = case["w"], case["h"]
    chain = sum(lw * lh for lw, lh in _levels(w, h)[1:])  # pixels of levels 1 and up
    if op == "generate_mips_device":
        return {"bytes": 4 * (w * h + chain), "flops": 20 * chain}
    fmt = tx.Format[case["fmt"]]
    if op in ("decompress", "decompress_device"):
        return {"bytes": fmt.compressed_size(w, h) + 4 * w * h, "flops": 10 * w * h}
    if op in ("compress_mips", "compress_mips_device"):
        for lw, lh in _levels(w, h):
            total_ops += _encode_work(fmt, case["alg"], lw, lh)[1]
        out = fmt.mip_chain_size(w, h) + (4 * chain if op == "compress_mips_device" else 0)
        return {"bytes": 4 * w * h + out, "flops": total_ops}
    total_bytes, total_ops = _encode_work(fmt, case["alg"], w, h)
    return {"bytes": total_bytes, "flops": total_ops}
