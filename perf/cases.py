"""What a program does with this library, as a set of measurable cases.

A material's life with neural texture sets: its images are written into a set and reduced to mips (`write`), the
decoded set is compared with what went in (`compare`), the game decodes whole sets, one or a batch at a time
(`decode`) or samples them at scattered points (`queries`), takes single textures out of a decoded set (`read`) and
turns them into block-compressed ones (`blocks`).  Every pass goes through the public entry points on buffers and
descriptors that such a program keeps.
"""
import ctypes as C
import importlib
import math

import numpy as np
import torch

ntc = importlib.import_module("rtxntc-library_amd")
A, P = ntc.abi, ntc.presets

SRGB, HLG, LINEAR = 1, 2, 0
_FORMATS = {"planar": A.OUT_FP16_PLANAR_PAIRS, "fp16": A.OUT_FP16_PIXELS, "unorm8": A.OUT_UNORM8_PIXELS}
# A user's image formats: ChannelFormat, bytes per channel.
_PIXELS = {"u8": (A.FORMAT_UNORM8, 1), "u16": (A.FORMAT_UNORM16, 2), "f16": (A.FORMAT_FLOAT16, 2), "f32": (A.FORMAT_FLOAT32, 4)}
_SPACES = {"s": SRGB, "h": HLG, "l": LINEAR}

# Textures of a set as "first channel:channels:channels of a pixel:format:colour space", separated by blanks: colour
# textures are stored and exchanged in sRGB, emissive ones are stored in HLG and exchanged as linear halves.
_PBR = "0:3:4:u8:s 3:2:2:u8:l 5:1:1:u8:l 6:1:1:u8:l 7:1:1:u8:l 8:3:4:f16:h"      # colour, normal, three masks, emissive
_TWO_RGBA = "0:4:4:u8:s 4:4:4:u8:l"
_PBR16 = "0:4:4:u16:s 4:2:2:u16:l 6:3:4:u8:l"
_FLOAT = "0:3:3:f32:l 3:1:1:f32:l"
_MATERIALS = {_PBR: 12, _TWO_RGBA: 8, _PBR16: 10, _FLOAT: 4}

_device = None


def device():
    global _device
    if _device is None:
        _device = ntc.Device(0)
    return _device


# ---- the cases ---------------------------------------------------------------------------------------------------

def _decode(name, net, width, height, mips, channels, fmt, sets=1, grid_scale=2, sigma=0.35):
    return {"name": name, "op": "decode", "net": net, "width": width, "height": height, "mips": mips, "channels": channels,
            "format": fmt, "sets": sets, "grid_scale": grid_scale, "sigma": sigma}


def listed():
    return [
        # a thumbnail or a streamed-in small mip: launch and table cost
        _decode("decode_small_128", "cfg01", 128, 128, 1, 8, "planar"),
        # the headline set of the benchmark: a hero material with its whole mip chain
        _decode("decode_4096", "cfg01", 4096, 4096, 13, 16, "planar"),
        # loading a level: several sets in one call, straight to 8-bit pixels
        _decode("decode_batch_8x2048", "cfg2", 2048, 2048, 12, 12, "unorm8", sets=8),
        # a set whose size is no power of two (a decal, a screen-sized background, a scan) and 9 channels of it
        _decode("decode_1920x1080", "ref16", 1920, 1080, 11, 9, "unorm8"),
        # the network that LibNTC decodes by default (FP8), whole mip chain
        _decode("decode_fp8_2048", "fp8_16", 2048, 2048, 12, 16, "planar"),
        # the wide decoder with e4m3 weights, one mip
        _decode("decode_e4m3_4096", "cfg3", 4096, 4096, 1, 16, "planar"),
        # inference on sample: scattered points of a large set, all its mips
        {"name": "queries_8192_16M", "op": "queries", "net": "cfg01", "size": 8192, "queries": 1 << 24, "ordered": True, "grid_scale": 2, "sigma": 0.35},
        # every texture of a decoded mip into its own image, 8-bit ones dithered
        {"name": "read_pbr_2048", "op": "read", "textures": _PBR, "width": 2048, "height": 2048, "dither": True},
        # a material's images into a set, then its mips
        {"name": "write_pbr_2048", "op": "write", "textures": _PBR, "width": 2048, "height": 2048},
        # how good the decoded set is: error of each mip, and an exported texture against its original
        {"name": "compare_4096", "op": "compare", "channels": 16, "width": 4096, "height": 4096, "mips": 13, "image": "u8", "msle": False},
        # transcoding on load: colour to BC7 with the modes that the file brings, normal map to BC5, a mask to BC4, emissive to BC6H
        {"name": "blocks_material_2048", "op": "blocks", "formats": "7m 5 4 6", "width": 2048, "height": 2048},
        # authoring: the full BC7 search
        {"name": "blocks_bc7_1024", "op": "blocks", "formats": "7", "width": 1024, "height": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, lo, hi):
    """A power-of-two square, a power-of-two rectangle or any size."""
    kind = rng.random()
    if kind < 0.4:
        n = 1 << rng.randint(int(math.log2(lo)), int(math.log2(hi)))
        return n, n
    if kind < 0.55:
        n = 1 << rng.randint(int(math.log2(lo)) + 1, int(math.log2(hi)))
        return (n, n // 2) if rng.random() < 0.5 else (n // 2, n)
    w = _log(rng, lo, hi)
    return w, min(hi, max(lo, int(w * rng.uniform(0.4, 2.0))))


def draw(rng):
    op = rng.choice(["decode", "decode", "decode", "queries", "read", "write", "compare", "blocks"])
    if op == "decode":
        net = rng.choice(["cfg01", "cfg01", "cfg2", "cfg3", "ref16", "ref12", "ref8", "ref4", "fp8_16", "fp8_16", "fp8_12", "fp8_8", "fp8_4"])
        w, h = _shape(rng, 64, 3072 if net.startswith("fp8") or net == "cfg3" else 4096)
        mips = rng.choice([1, P.full_mip_count(w, h)])
        sets = rng.choice([1, 1, rng.randint(2, 8)]) if w * h <= 1 << 20 else 1
        c = _decode("", net, w, h, mips, rng.randint(3, 16), rng.choice(["planar", "planar", "fp16", "unorm8", "unorm8"]), sets,
                    rng.choice([2, 2, 3, 4]), rng.choice([0.35, 0.35, 1.5]))
        del c["name"]
        return c
    if op == "queries":
        return {"op": op, "net": rng.choice(["cfg01", "cfg01", "cfg2", "ref16", "fp8_16"]), "size": 1 << rng.randint(8, 13), "queries": _log(rng, 1 << 12, 1 << 23),
                "ordered": rng.random() < 0.75, "grid_scale": 2, "sigma": 0.35}
    if op in ("read", "write"):
        w, h = _shape(rng, 64, 4096)
        c = {"op": op, "textures": rng.choice([_PBR, _PBR, _TWO_RGBA, _PBR16, _FLOAT]), "width": w, "height": h}
        if op == "read":
            c["dither"] = rng.random() < 0.6
        return c
    if op == "compare":
        w, h = _shape(rng, 64, 4096)
        return {"op": op, "channels": 2 * rng.randint(2, 8), "width": w, "height": h, "mips": rng.choice([1, P.full_mip_count(w, h)]),
                "image": rng.choice(["u8", "u8", "f16"]), "msle": rng.random() < 0.25}
    formats = rng.choice(["7m 5 4 6", "7m 5 4", "1 5 4", "3 5", "1", "2", "4", "5", "6", "7m", "7"])
    w, h = _shape(rng, 64, 1024 if formats == "7" else 2048)
    return {"op": op, "formats": formats, "width": w, "height": h}


# ---- geometry, sizes, work -----------------------------------------------------------------------------------------

def _spec(net):
    if net.startswith("ref"):
        return P.spec_ref092(int(net[3:]))
    if net.startswith("fp8_"):
        return P.spec_ref092_fp8(int(net[4:]))
    return {"cfg01": P.spec_cfg01, "cfg2": P.spec_cfg2, "cfg3": P.spec_cfg3}[net]()


def _mips(case, width, height, count):
    spec = _spec(case["net"])
    if case["net"].startswith(("ref", "fp8")):
        mips, latent_bytes = P.mips_ref092(spec, width, height, count, case["grid_scale"])
    else:
        mips, latent_bytes = P.mips_private_grids(spec, width, height, count)
    return spec, mips, latent_bytes


def _macs(spec):
    return sum(spec.layer_inputs(layer) * spec.layer_outputs(layer) for layer in range(A.MLP_LAYERS))


def _mip_sizes(width, height, count):
    return [(max(width >> m, 1), max(height >> m, 1)) for m in range(count)]


def _textures(text):
    out = []
    for word in text.split():
        first, count, pixel, fmt, space = word.split(":")
        out.append((int(first), int(count), int(pixel), fmt, _SPACES[space]))
    return out


def _block_source(fmt):
    """Channels and format of the image that a block format is made from."""
    return {"4": (1, "u8"), "5": (2, "u8"), "6": (4, "f16")}.get(fmt, (4, "u8"))


def _block_bytes(fmt):
    return 8 if fmt in ("1", "4") else 16


def work(case):
    op = case["op"]
    if op == "decode":
        spec, mips, latent_bytes = _mips(case, case["width"], case["height"], case["mips"])
        texels = sum(d.width * d.height for d in mips)
        out = texels * case["channels"] * (1 if case["format"] == "unorm8" else 2)
        weights = ntc.synth.weight_layout(spec).bufferSize
        return {"bytes": case["sets"] * (latent_bytes + weights + out), "flops": 2.0 * _macs(spec) * texels * case["sets"]}
    if op == "queries":
        spec, mips, latent_bytes = _mips(case, case["size"], case["size"], P.full_mip_count(case["size"], case["size"]))
        cells = 4 * (spec.hrFeatures * spec.hrBits + spec.lrFeatures * spec.lrBits) // 8        # the 2 x 2 cells of both grids
        n = case["queries"]
        return {"bytes": n * (12 + 32) + min(latent_bytes, n * cells), "flops": 2.0 * _macs(spec) * n}
    w, h = case["width"], case["height"]
    if op in ("read", "write"):
        image = sum(pixel * _PIXELS[fmt][1] for _, _, pixel, fmt, _ in _textures(case["textures"])) * w * h
        planar = 2 * sum(count for _, count, _, _, _ in _textures(case["textures"])) * w * h
        total = image + planar
        if op == "write":
            sizes = [2 * _MATERIALS[case["textures"]] * a * b for a, b in _mip_sizes(w, h, P.full_mip_count(w, h))]
            total += sum(sizes[:-1]) + sum(sizes[1:])                                            # each mip is made from the one above
        return {"bytes": total, "flops": 0}
    if op == "compare":
        planar = sum(2 * case["channels"] * a * b for a, b in _mip_sizes(w, h, case["mips"]))
        return {"bytes": 2 * planar + 2 * 4 * _PIXELS[case["image"]][1] * w * h, "flops": 0}
    total = 0
    for fmt in case["formats"].split():
        channels, source = _block_source(fmt)
        total += channels * _PIXELS[source][1] * w * h + _block_bytes(fmt[0]) * ((w + 3) // 4) * ((h + 3) // 4)
    return {"bytes": total, "flops": 0}


def tolerance(case):
    if case["op"] in ("read", "write"):
        # transfer functions through a math library: a unit in the last place of a half, one 8- or 16-bit code at a tie
        return {"rel": 2e-4, "max": 2e-3, "differ": 1e-3}
    if case["op"] == "compare":
        return {"rel": 1e-5}            # sums of squares; the image difference adds integers
    return "exact"                      # the decoder and the block compressors are defined to the bit


# ---- inputs --------------------------------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _bytes(count, g):
    return torch.randint(0, 256, (int(count),), dtype=torch.uint8, device="cuda", generator=g)


def _planes(channels, width, height, g):
    """Smooth surfaces with detail and a little noise, in [0, 1]: channels x height x width."""
    coarse = torch.rand((1, channels, max(2, height // 64 + 2), max(2, width // 64 + 2)), device="cuda", generator=g)
    fine = torch.rand((1, channels, max(2, height // 8 + 2), max(2, width // 8 + 2)), device="cuda", generator=g)
    up = lambda t: torch.nn.functional.interpolate(t, size=(height, width), mode="bilinear", align_corners=True)[0]  # noqa: E731
    v = 0.75 * up(coarse) + 0.25 * up(fine)
    v += torch.randn((channels, height, width), device="cuda", generator=g) * 0.015
    return v.clamp_(0.0, 1.0)


def _planar(planes):
    """LibNTC's internal layout (rows of channel pairs, halves) of an image given as channels x height x width."""
    c, h, w = planes.shape
    return planes.to(torch.float16).reshape(c // 2, 2, h, w).permute(2, 0, 3, 1).contiguous().reshape(-1)


def _pixels(planes, fmt):
    """Pitch-linear pixels of `fmt`."""
    p = planes.permute(1, 2, 0)
    if fmt == "u8":
        p = (p * 255.0).round().to(torch.uint8)
    elif fmt == "u16":
        p = (p * 65535.0).round().to(torch.int32).to(torch.uint16)
    else:
        p = p.to(torch.float16 if fmt == "f16" else torch.float32)
    return p.contiguous().reshape(-1)


def _nbytes(t):
    return t.numel() * t.element_size()


def _weights(spec, seed, sigma):
    if spec.weightType == A.WEIGHTS_FP8:
        blob = ntc.synth.make_fp8_weights(spec, seed, weight_sigma=sigma)
    else:
        # scales that keep the activations of uniform weights and inputs inside HGELU's range, as training does
        blob = ntc.synth.make_weights(spec, seed, (-17.0, -12.0))
    return torch.from_numpy(blob).cuda()


def _prepare_decode(case, seed):
    dev, g = device(), _generator(seed)
    spec, mips, latent_bytes = _mips(case, case["width"], case["height"], case["mips"])
    fmt = _FORMATS[case["format"]]
    stride, out_bytes = P.assign_output_offsets(mips, case["channels"], fmt)
    keep, sets, outs = [], [], []
    for s in range(case["sets"]):
        latents, weights = _bytes(latent_bytes, g), _weights(spec, 8 * seed + s, case["sigma"])
        out = torch.zeros((out_bytes + 15) // 16 * 16, dtype=torch.uint8, device="cuda")
        sets.append(ntc.make_texture_set(spec, mips, case["channels"], fmt, latents.data_ptr(), _nbytes(latents),
                                         weights.data_ptr(), _nbytes(weights), out.data_ptr(), _nbytes(out), stride))
        keep.append((latents, weights))
        outs.append(out if case["format"] == "unorm8" else out.view(torch.float16))
    return {"run": _run_decode, "device": dev, "sets": dev.pack_sets(sets), "outs": outs, "keep": keep}


def _run_decode(s):
    s["device"].decode(s["sets"])
    return s["outs"]


def _prepare_queries(case, seed):
    dev, g = device(), _generator(seed)
    size, n = case["size"], case["queries"]
    spec, mips, latent_bytes = _mips(case, size, size, P.full_mip_count(size, size))
    P.assign_output_offsets(mips, 16, A.OUT_FP16_PLANAR_PAIRS)
    latents, weights = _bytes(latent_bytes, g), _weights(spec, seed, case["sigma"])
    sets = dev.pack_sets([ntc.make_texture_set(spec, mips, 16, A.OUT_FP16_PLANAR_PAIRS, latents.data_ptr(), _nbytes(latents),
                                               weights.data_ptr(), _nbytes(weights), None, 0)])
    points = torch.empty((n, 3), dtype=torch.float32, device="cuda")                             # NtcHipQuery: u, v, mip
    points[:, :2] = torch.rand((n, 2), device="cuda", generator=g)
    points.view(torch.int32)[:, 2] = torch.randint(0, len(mips), (n,), dtype=torch.int32, device="cuda", generator=g)
    out = torch.zeros((n, 16), dtype=torch.float16, device="cuda")
    bricks = None
    if case["ordered"]:
        bricks = torch.zeros(dev.lib.ntc_hip_query_latents_bytes(sets), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        dev.call("build_query_latents", sets, bricks.data_ptr(), _nbytes(bricks))
        sets[0].queryLatents, sets[0].queryLatentsBytes = bricks.data_ptr(), _nbytes(bricks)
    return {"run": _run_queries, "device": dev, "sets": sets, "points": points, "n": n, "out": out, "out_bytes": _nbytes(out),
            "keep": (latents, weights, bricks)}


def _run_queries(s):
    s["device"].call("decode_queries", s["sets"], s["points"].data_ptr(), s["n"], s["out"].data_ptr(), s["out_bytes"])
    return s["out"]


def _storage(textures):
    """Storage colour space of each channel of a set."""
    spaces = [LINEAR] * 16
    for first, count, _, _, space in textures:
        for k in range(min(count, 3)):                  # alpha is linear
            spaces[first + k] = space
    return spaces


def _fill_spaces(call, storage, first, count, to_image):
    for k in range(count):
        stored = storage[first + k]
        image = LINEAR if stored == HLG else stored
        call.srcColorSpaces[k], call.dstColorSpaces[k] = (stored, image) if to_image else (image, stored)


def _prepare_read(case, seed):
    dev, g = device(), _generator(seed)
    w, h, textures = case["width"], case["height"], _textures(case["textures"])
    channels = _MATERIALS[case["textures"]]
    planar = _planar(_planes(channels, w, h, g))
    storage, calls, outs = _storage(textures), [], []
    for first, count, pixel, fmt, _ in textures:
        code, size = _PIXELS[fmt]
        # (16-bit codes as int16, which torch can index)
        out = torch.zeros(w * h * pixel, dtype={"u8": torch.uint8, "u16": torch.int16, "f16": torch.float16, "f32": torch.float32}[fmt], device="cuda")
        rc = A.ReadChannels()
        rc.planarPairs, rc.planarBytes = planar.data_ptr(), _nbytes(planar)
        rc.width, rc.height, rc.setChannels, rc.firstChannel, rc.numChannels = w, h, channels, first, count
        rc.dst, rc.dstBytes, rc.format, rc.pixelStride, rc.rowPitch = out.data_ptr(), _nbytes(out), code, pixel * size, w * pixel * size
        rc.useDithering = int(case["dither"] and fmt == "u8")
        _fill_spaces(rc, storage, first, count, True)
        calls.append(rc)
        outs.append(out)
    return {"run": _run_read, "device": dev, "calls": calls, "outs": outs, "keep": planar}


def _run_read(s):
    for rc in s["calls"]:
        s["device"].call("read_channels", rc)
    return s["outs"]


def _prepare_write(case, seed):
    dev, g = device(), _generator(seed)
    w, h, textures = case["width"], case["height"], _textures(case["textures"])
    channels = _MATERIALS[case["textures"]]
    sizes = _mip_sizes(w, h, P.full_mip_count(w, h))
    page = torch.zeros(sum(a * b for a, b in sizes) * channels, dtype=torch.float16, device="cuda")
    storage, calls, keep, resizes = _storage(textures), [], [], []
    for first, count, pixel, fmt, _ in textures:
        code, size = _PIXELS[fmt]
        image = _pixels(_planes(pixel, w, h, g), fmt)
        wc = A.WriteChannels()
        wc.src, wc.srcBytes, wc.format, wc.pixelStride, wc.rowPitch = image.data_ptr(), _nbytes(image), code, pixel * size, w * pixel * size
        wc.planarPairs, wc.planarBytes = page.data_ptr(), _nbytes(page)
        wc.width, wc.height, wc.setChannels, wc.firstChannel, wc.numChannels = w, h, channels, first, count
        _fill_spaces(wc, storage, first, count, False)
        calls.append(wc)
        keep.append(image)
    spaces = (C.c_uint8 * 16)(*storage)
    at = page.data_ptr()
    for (sw, sh), (dw, dh) in zip(sizes[:-1], sizes[1:]):
        below = at + 2 * channels * sw * sh
        resizes.append((at, 2 * channels * sw * sh, sw, sh, below, 2 * channels * dw * dh, dw, dh, channels, spaces))
        at = below
    return {"run": _run_write, "device": dev, "calls": calls, "resizes": resizes, "page": page, "keep": keep}


def _run_write(s):
    dev = s["device"]
    for wc in s["calls"]:
        dev.call("write_channels", wc)
    for r in s["resizes"]:
        dev.call("resize_planar", *r)
    return s["page"]


def _prepare_compare(case, seed):
    dev, g = device(), _generator(seed)
    w, h, channels = case["width"], case["height"], case["channels"]
    losses, keep = [], []
    for a, b in _mip_sizes(w, h, case["mips"]):
        reference = _planar(_planes(channels, a, b, g))
        decoded = (reference + 0.02 * torch.randn(reference.shape, dtype=torch.float16, device="cuda", generator=g))
        losses.append((decoded.data_ptr(), reference.data_ptr(), _nbytes(decoded), a, b, channels, (1 << channels) - 1, -1, 0))
        keep += [reference, decoded]
    fmt, size = _PIXELS[case["image"]]
    first = _planes(4, w, h, g)
    second = (first + 0.02 * torch.randn(first.shape, device="cuda", generator=g)).clamp_(0.0, 1.0)
    sums = torch.zeros(4, dtype=torch.int64, device="cuda")
    d = A.ImageDifference()
    for image, planes in ((d.a, first), (d.b, second)):
        t = _pixels(planes, case["image"])
        image.data, image.bytes, image.pixelStride, image.rowPitch = t.data_ptr(), _nbytes(t), 4 * size, 4 * size * w
        image.width, image.height, image.format, image.numChannels = w, h, fmt, 4
        keep.append(t)
    d.width, d.height, d.useMSLE, d.output, d.outputBytes = w, h, int(case["msle"]), sums.data_ptr(), _nbytes(sums)
    return {"run": _run_compare, "device": dev, "losses": losses, "difference": d, "sums": sums, "mse": np.zeros((case["mips"], 16), dtype=np.float32), "keep": keep}


def _run_compare(s):
    dev = s["device"]
    row = (C.c_float * 16)()
    for m, loss in enumerate(s["losses"]):
        dev.call("image_loss", *loss, row)
        s["mse"][m] = row
    dev.call("memset", s["difference"].output, 0, 32)      # the pass adds to what is there
    dev.call("image_difference", s["difference"])
    return {"mse": s["mse"], "difference": s["sums"]}


def _mode_buffer(blocks):
    """The 9-bit modes and partitions of an encoded image, packed as MakeBC7ModeBuffer packs them."""
    first = blocks.view(torch.int32).reshape(-1, 4)[:, 0].to(torch.int64) & 0xFFFFFFFF
    mode = torch.log2((first & -first).to(torch.float32)).to(torch.int64).clamp_(0, 7)
    partition = (first >> (mode + 1)) & torch.tensor([15, 63, 63, 63, 7, 3, 0, 63], device="cuda")[mode]
    entry = (mode << 6) | partition
    entry = torch.where(entry == 0, torch.full_like(entry, 0x1BF), entry)
    bits = ((entry[:, None] >> torch.arange(9, device="cuda")) & 1).reshape(-1)
    bits = torch.nn.functional.pad(bits, (0, -bits.numel() % 32 + 32)).reshape(-1, 8)
    return (bits << torch.arange(8, device="cuda")).sum(1).to(torch.uint8)


def _prepare_blocks(case, seed):
    dev, g = device(), _generator(seed)
    w, h = case["width"], case["height"]
    bw, bh = (w + 3) // 4, (h + 3) // 4
    calls, outs, keep = [], [], []
    for fmt in case["formats"].split():
        channels, source = _block_source(fmt)
        planes = _planes(channels, w, h, g)
        if source == "f16":
            planes = planes * planes * 8.0                               # emissive: mostly below 1, up to 8
        elif channels == 4:
            cut = torch.rand((h, w), device="cuda", generator=g) < 0.1   # a tenth of the right half is cut out, the left is opaque
            planes[3] = torch.where(cut, 0.0, 1.0)
            planes[3, :, : w // 2] = 1.0
        image = _pixels(planes, source)
        code, size = _PIXELS[source]
        bc = A.BlockCompress()
        bc.src.data, bc.src.bytes, bc.src.pixelStride, bc.src.rowPitch = image.data_ptr(), _nbytes(image), channels * size, w * channels * size
        bc.src.width, bc.src.height, bc.src.format, bc.src.numChannels = w, h, code, channels
        out = torch.zeros(bw * bh * _block_bytes(fmt[0]), dtype=torch.uint8, device="cuda")
        bc.widthInBlocks, bc.heightInBlocks, bc.dstFormat, bc.alphaThreshold = bw, bh, int(fmt[0]), 1.0 / 255.0
        bc.dst, bc.dstBytes, bc.dstRowPitch = out.data_ptr(), _nbytes(out), bw * _block_bytes(fmt[0])
        if fmt == "7m":                                                  # the file's mode map comes from a full search when it was made
            torch.cuda.synchronize()
            dev.call("block_compress", bc)
            dev.synchronize()
            modes = _mode_buffer(out)
            bc.modeBuffer, bc.modeBufferBytes, bc.modeMapWidthInBlocks, bc.modeMapHeightInBlocks = modes.data_ptr(), _nbytes(modes), bw, bh
            keep.append(modes)
        calls.append(bc)
        outs.append(out)
        keep.append(image)
    return {"run": _run_blocks, "device": dev, "calls": calls, "outs": outs, "keep": keep}


def _run_blocks(s):
    for bc in s["calls"]:
        s["device"].call("block_compress", bc)
    return s["outs"]


_PREPARE = {"decode": _prepare_decode, "queries": _prepare_queries, "read": _prepare_read, "write": _prepare_write,
            "compare": _prepare_compare, "blocks": _prepare_blocks}


def prepare(case, seed):
    return _PREPARE[case["op"]](case, seed)


def run(state):
    return state["run"](state)
