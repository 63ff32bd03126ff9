"""The work whose speed is measured: what programs built with this framework
have it do, each case through the public Python entry points.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  a program's own state: linked and lowered executable,
                       input images on the GPU, output images
  run(state)           one pass: a launch (or a pool execution) and its outputs
  work(case)           bytes and flops one pass cannot do without
  exact(case, seed)    float outputs in 64 bits with plain torch

Images are smooth with some grain, as photographs and rendered layers are;
layers carry soft alpha masks with fully transparent and fully opaque areas.
Executables are lowered and launched as they come, without the autotuner.
"""
import math

import numpy as np
import torch

import zosimos_amd as z
from zosimos_amd import workloads as W

SB, SP, T, P = z.SampleBits, z.SampleParts, z.Transfer, z.Primaries
RGBA8, RGBA16F = W.RGBA8, W.RGBA16F
RGBA32F = z.Texel(SB.Float32x4, SP.RgbA)
LINEAR_709, P3_LINEAR = W.LINEAR_709, W.P3_LINEAR
ROW_ALIGN = 256  # row pitch of images read from buffers

# Formats with a staged codec, as video, print and compact images use them:
# name -> (texel, transfer, primaries)
STAGED = {
    "10bit_bt2020": (z.Texel(SB.UInt2101010, SP.RgbA), T.Bt2020_10bit, P.Bt2020),
    "16bit_srgb": (z.Texel(SB.UInt16x4, SP.RgbA), T.Srgb, P.Bt709),
    "8bit_bt709": (z.Texel(SB.UInt8x4, SP.RgbA), T.Bt709, P.Bt709),
    "rgb8_srgb": (z.Texel(SB.UInt8x3, SP.Rgb), T.Srgb, P.Bt709),
    "rgb565_srgb": (z.Texel(SB.UInt565, SP.Rgb), T.Srgb, P.Bt709),
    "luma8_srgb": (z.Texel(SB.UInt8, SP.Luma), T.Srgb, P.Bt709),
}


def listed():
    return [
        # The reference's own loop: one inscribe program relaunched from a
        # pool, host images in, host image out (512x512, tests/loop.rs).
        dict(name="relaunch_512", kind="relaunch", w=512, h=512, fw=157, fh=151),
        # Two 8-bit layers blended and placed by an affine map: an editor's
        # interactive preview, the smallest device-resident launch.
        dict(name="blend_affine_1024x768", kind="blend_affine", w=1024, h=768, scale=0.75, degrees=15.0),
        # Grading a full 8K frame in Oklab under a half-float overlay.
        dict(name="grade_over_7680x4320", kind="grade_over", w=7680, h=4320),
        # A library of 256 images of uneven sizes, 8-bit and half float,
        # converted and resampled by one program.
        dict(name="resample_batch_256", kind="batch", n=256, lo=64, hi=4096, shapes=0),
        # The Oklab colour chain over a burst of 4K frames.
        dict(name="chain_16x3840x2160", kind="chain", n=16, w=3840, h=2160, space="oklab"),
        # Eight rotated and scaled half-float layers composited into a frame.
        dict(name="composite_8x3840x2160", kind="composite", layers=8, w=3840, h=2160, maps=0),
        # 10-bit Bt.2020 video frames into linear Display P3 for compositing.
        dict(name="decode_10bit_3840x2160", kind="decode", fmt="10bit_bt2020", out="f16", w=3840, h=2160),
        # Writing a linear half-float result as a 16-bit sRGB image.
        dict(name="encode_16bit_3840x2160", kind="encode", fmt="16bit_srgb", w=3840, h=2160),
        # Two 8-bit layers with 256-byte rows (images read from buffers) at an
        # odd size, blended in linear light into half float.
        dict(name="padded_over_1919x1079", kind="padded_over", w=1919, h=1079),
        # Pasting an HD picture into a 4K frame (nearest, texels moved as is).
        dict(name="paste_3840x2160", kind="paste", op="inscribe", w=3840, h=2160, fw=1920, fh=1080),
        # An edge filter (3x3 derivative) over an 8-bit 4K picture.
        dict(name="sobel_3840x2160", kind="filter", method="sobel", axis="width", texel="u8", w=3840, h=2160),
        # A procedural texture: four octaves of fractal noise.
        dict(name="noise_2048", kind="generate", op="noise", octaves=4, texel="u8", w=2048, h=2048),
    ]


def _size(rng, lo, hi):
    """A side length spread over the logarithm of [lo, hi], often odd."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _frame(rng, lo, hi):
    """Width and height of aspect 1:1 to 2:1."""
    w = _size(rng, lo, hi)
    return w, max(1, int(round(w * rng.uniform(0.5, 1.0))))


def draw(rng):
    kind = rng.choice(["relaunch", "blend_affine", "grade_over", "batch", "chain", "composite", "decode", "encode",
                       "padded_over", "paste", "filter", "generate"])
    if kind == "relaunch":
        w, h = _frame(rng, 64, 1024)
        return dict(kind=kind, w=w, h=h, fw=rng.randint(1, w), fh=rng.randint(1, h))
    if kind == "blend_affine":
        w, h = _frame(rng, 128, 2048)
        return dict(kind=kind, w=w, h=h, scale=round(rng.uniform(0.4, 1.6), 3), degrees=round(rng.uniform(-90, 90), 1))
    if kind == "grade_over":
        w, h = _frame(rng, 320, 7680)
        return dict(kind=kind, w=w, h=min(h, 4320))
    if kind == "batch":
        return dict(kind=kind, n=_size(rng, 4, 96), lo=rng.choice([16, 64]), hi=_size(rng, 256, 2048),
                    shapes=rng.randint(1, 1 << 20))
    if kind == "chain":
        w, h = _frame(rng, 256, 3840)
        return dict(kind=kind, n=_size(rng, 1, 16), w=w, h=min(h, 2160),
                    space=rng.choice(["oklab", "oklab", "srlab2"]))
    if kind == "composite":
        w, h = _frame(rng, 256, 3840)
        return dict(kind=kind, layers=rng.randint(2, 8), w=w, h=min(h, 2160), maps=rng.randint(1, 1 << 20))
    if kind == "decode":
        w, h = _frame(rng, 256, 4096)
        return dict(kind=kind, fmt=rng.choice(sorted(STAGED)), out=rng.choice(["f16", "f32"]), w=w, h=h)
    if kind == "encode":
        w, h = _frame(rng, 256, 4096)
        return dict(kind=kind, fmt=rng.choice(sorted(STAGED)), w=w, h=h)
    if kind == "padded_over":
        w, h = _frame(rng, 101, 3839)
        return dict(kind=kind, w=w | 1, h=h | 1)
    if kind == "paste":
        w, h = _frame(rng, 128, 4096)
        return dict(kind=kind, op=rng.choice(["inscribe", "crop", "rotate", "resize"]), w=w, h=h,
                    fw=rng.randint(1, w), fh=rng.randint(1, h))
    if kind == "filter":
        w, h = _frame(rng, 128, 4096)
        return dict(kind=kind, method=rng.choice(["sobel", "scharr3"]), axis=rng.choice(["width", "height"]),
                    texel=rng.choice(["u8", "f16"]), w=w, h=h)
    w, h = _frame(rng, 128, 2048)
    return dict(kind=kind, op=rng.choice(["noise", "normal", "ramp"]), octaves=rng.randint(1, 6),
                texel=rng.choice(["u8", "f16"]), w=w, h=h)


# ---- synthetic images ----------------------------------------------------------------
def _generator(seed, k):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + 7919 * k + 1) & 0x7FFFFFFFFFFFFFFF)
    return g


def _smooth(g, w, h, channels):
    """(h, w, channels) in [0, 1]: features of about 1/12 of the image and a
    little grain."""
    low = torch.rand((1, channels, 13, 13), device="cuda", generator=g)
    v = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=False)[0]
    v = v.permute(1, 2, 0).contiguous()
    v.add_(torch.rand(v.shape, device="cuda", generator=g), alpha=0.06).sub_(0.03)
    return v.clamp_(0.0, 1.0)


def _picture(g, w, h, alpha):
    """RGBA floats; alpha "soft" is a mask with transparent and opaque areas."""
    v = _smooth(g, w, h, 4)
    if alpha == "soft":
        v[..., 3] = ((v[..., 3] - 0.5) * 2.5 + 0.5).clamp_(0.0, 1.0)
    elif alpha == "opaque":
        v[..., 3] = 1.0
    return v


def _u8(g, w, h, alpha="opaque"):
    return (_picture(g, w, h, alpha) * 255.0).round_().to(torch.uint8)


def _f16(g, w, h, alpha="soft"):
    """Linear light with highlights above 1."""
    v = _picture(g, w, h, alpha)
    v[..., :3] *= v[..., :3] * 1.25
    return v.to(torch.float16)


def _bytes(t):
    """The tensor's own memory as bytes, rows in order."""
    return t.contiguous().view(-1).view(torch.uint8)


_CONTEXT = []


def _context():
    """A program's one device and stream."""
    if not _CONTEXT:
        _CONTEXT.append(z.Context(0))
    return _CONTEXT[0]


_VIEW = {SB.UInt8x4: (torch.uint8, 4), SB.Float16x4: (torch.float16, 4), SB.Float32x4: (torch.float32, 4),
         SB.UInt16x4: (torch.int16, 4), SB.UInt2101010: (torch.int32, 1), SB.UInt8x3: (torch.uint8, 3),
         SB.UInt565: (torch.int16, 1), SB.UInt8: (torch.uint8, 1), SB.UInt16x2: (torch.int16, 2)}


def _view(desc, memory):
    dtype, n = _VIEW[desc.texel.bits]
    return memory.view(dtype).view(desc.height, desc.width, n)


def _state(commands, inputs, outputs, out_memory=None):
    """Lower the program and wrap its device images.  inputs: register ->
    (descriptor, tensor); outputs: register -> descriptor."""
    ctx = _context()
    exe = z.Linker.from_included().compile(commands).lower_to(ctx)
    ins, outs, keep, result = {}, {}, [], {}
    for reg, (d, t) in inputs.items():
        b = _bytes(t)
        ins[reg] = ctx.wrap(d, b.data_ptr(), b.numel())
        keep.append(b)
    for k, (reg, d) in enumerate(outputs.items()):
        m = out_memory[reg] if out_memory else torch.empty(d.nbytes, device="cuda", dtype=torch.uint8)
        outs[reg] = ctx.wrap(d, m.data_ptr(), m.numel())
        keep.append(m)
        if not out_memory:
            result["out%d" % k] = _view(d, m)
    torch.cuda.synchronize()
    return dict(exe=exe, ins=ins, outs=outs, keep=keep, result=result)


def _padded(desc):
    return desc.with_(row_stride=(desc.width * desc.texel.bytes + ROW_ALIGN - 1) // ROW_ALIGN * ROW_ALIGN)


def _pad_rows(t, desc):
    rows = t.contiguous().view(desc.height, -1).view(torch.uint8)
    out = torch.zeros((desc.height, desc.row_stride), device="cuda", dtype=torch.uint8)
    out[:, :rows.shape[1]] = rows
    return out


def _staged_codes(g, fmt, w, h):
    """Texels of a staged format as a video or image file holds them."""
    v = _smooth(g, w, h, 4)
    if fmt == "10bit_bt2020":
        c = (64 + v * (940 - 64)).to(torch.int64)
        return (c[..., 0] | (c[..., 1] << 10) | (c[..., 2] << 20) | (3 << 30)).to(torch.int32)
    if fmt == "16bit_srgb":
        v[..., 3] = 1.0
        return (v * 65535.0).to(torch.int32).to(torch.int16)
    if fmt == "8bit_bt709":
        v[..., 3] = 1.0
        return (v * 255.0).to(torch.uint8)
    if fmt == "rgb8_srgb":
        return (v[..., :3] * 255.0).to(torch.uint8)
    if fmt == "rgb565_srgb":
        r, gr, b = (v[..., 0] * 31).to(torch.int32), (v[..., 1] * 63).to(torch.int32), (v[..., 2] * 31).to(torch.int32)
        return (r | (gr << 5) | (b << 11)).to(torch.int16)
    return (v[..., 0] * 255.0).to(torch.uint8)


# ---- programs ------------------------------------------------------------------------
def _batch_shapes(case):
    return W.c3_shapes(case["n"], case["shapes"], lo=case["lo"], hi=case["hi"])


def _batch_layout(case):
    """Byte offset of every output image in its format's buffer."""
    offsets, total = [], [0, 0]
    for w, h, fmt, s in _batch_shapes(case):
        ow, oh = max(1, int(round(w * s))), max(1, int(round(h * s)))
        offsets.append(total[fmt])
        total[fmt] += (ow * oh * (4, 8)[fmt] + 255) // 256 * 256
    return offsets, total


def _composite_affines(case):
    rng = np.random.default_rng([case["maps"], 5])
    rots = rng.uniform(-math.pi / 4, math.pi / 4, case["layers"])
    scales = rng.uniform(0.5, 1.5, case["layers"])
    return [W.about_centre(case["w"], case["h"], float(s), float(r)) for s, r in zip(scales, rots)]


def prepare(case, seed):
    kind = case["kind"]
    g = _generator(seed, 0)
    cmd = z.CommandBuffer()
    if kind == "relaunch":
        w, h, fw, fh = case["w"], case["h"], case["fw"], case["fh"]
        bg_d, fg_d = z.Descriptor.rgba8_srgb(w, h), z.Descriptor.rgba8_srgb(fw, fh)
        bg, fg = cmd.input(bg_d), cmd.input(fg_d)
        o, _ = cmd.output(cmd.inscribe(bg, z.Rectangle(0, 0, fw, fh), fg))
        exe = z.Linker.from_included().compile(cmd).lower_to(_context())
        pool = z.Pool()
        return dict(exe=exe, pool=pool, out=o,
                    keys={bg: pool.insert(bg_d, _u8(g, w, h).cpu().numpy()),
                          fg: pool.insert(fg_d, _u8(g, fw, fh, "soft").cpu().numpy())})
    if kind == "batch":
        shapes, (offsets, total) = _batch_shapes(case), _batch_layout(case)
        memory = [torch.zeros(max(n, 256), device="cuda", dtype=torch.uint8) for n in total]
        inputs, outputs, out_memory = {}, {}, {}
        for k, (w, h, fmt, s) in enumerate(shapes):
            ow, oh = max(1, int(round(w * s))), max(1, int(round(h * s)))
            if fmt == 0:
                din, conv, tex = z.Descriptor.rgba8_srgb(w, h), z.Color(primaries=P.DisplayP3), RGBA8
            else:
                din, conv, tex = z.Descriptor(w, h, RGBA16F, LINEAR_709), P3_LINEAR, RGBA16F
            r = cmd.input(din)
            c = cmd.color_convert(r, conv, tex)
            canvas = cmd.solid_rgba(z.Descriptor(ow, oh, tex, conv), (0.0, 0.0, 0.0, 0.0))
            o, od = cmd.output(cmd.affine(canvas, z.Affine.new(z.AffineSample.BiLinear).scale(ow / w, oh / h), c))
            gk = _generator(seed, 300 + k)
            inputs[r] = (din, _u8(gk, w, h, "soft") if fmt == 0 else _f16(gk, w, h))
            outputs[o] = od
            out_memory[o] = memory[fmt][offsets[k]:offsets[k] + od.nbytes]
        st = _state(cmd, inputs, outputs, out_memory)
        st["result"] = {"u8": memory[0], "f16": memory[1].view(torch.float16)}
        return st
    if kind == "chain":
        w, h = case["w"], case["h"]
        d = z.Descriptor.rgba8_srgb(w, h)
        inputs, outputs = {}, {}
        for k in range(case["n"]):
            r = cmd.input(d)
            if case["space"] == "oklab":
                v = W.color_chain(cmd, r)
            else:
                lab = cmd.color_convert(r, z.Color.SRLAB2_D65, W.LABA16F)
                v = cmd.color_convert(lab, z.Color.SRGB, RGBA8)
            o, od = cmd.output(v)
            inputs[r], outputs[o] = (d, _u8(_generator(seed, k), w, h)), od
        return _state(cmd, inputs, outputs)
    if kind == "composite":
        w, h = case["w"], case["h"]
        d = z.Descriptor(w, h, RGBA16F, LINEAR_709)
        acc = cmd.solid_rgba(d, (0.0, 0.0, 0.0, 0.0))
        inputs = {}
        for k, aff in enumerate(_composite_affines(case)):
            r = cmd.input(d)
            acc = cmd.affine(acc, aff, r)
            inputs[r] = (d, _f16(_generator(seed, k), w, h))
        o, od = cmd.output(W.color_chain(cmd, acc))
        return _state(cmd, inputs, {o: od})
    w, h = case["w"], case["h"]
    if kind == "blend_affine":
        d = z.Descriptor.rgba8_srgb(w, h)
        a, b = cmd.input(d), cmd.input(d)
        ab = cmd.blend(a, z.Rectangle(0, 0, w, h), b)
        canvas = cmd.solid_rgba(d, (0.0, 0.0, 0.0, 0.0))
        aff = W.about_centre(w, h, case["scale"], math.radians(case["degrees"]))
        o, od = cmd.output(cmd.affine(canvas, aff, ab))
        return _state(cmd, {a: (d, _u8(g, w, h)), b: (d, _u8(g, w, h, "soft"))}, {o: od})
    if kind == "grade_over":
        wl = W.c2(w, h)
        src, layer = list(wl.inputs)
        return _state(wl.commands, {src: (wl.inputs[src], _u8(g, w, h)), layer: (wl.inputs[layer], _f16(g, w, h))},
                      wl.outputs)
    if kind == "decode":
        texel, transfer, prim = STAGED[case["fmt"]]
        d = z.Descriptor(w, h, texel, z.Color(primaries=prim, transfer=transfer))
        a = cmd.input(d)
        o, od = cmd.output(cmd.color_convert(a, P3_LINEAR, RGBA16F if case["out"] == "f16" else RGBA32F))
        return _state(cmd, {a: (d, _staged_codes(g, case["fmt"], w, h))}, {o: od})
    if kind == "encode":
        texel, transfer, prim = STAGED[case["fmt"]]
        d = z.Descriptor(w, h, RGBA16F, P3_LINEAR)
        a = cmd.input(d)
        o, od = cmd.output(cmd.color_convert(a, z.Color(primaries=prim, transfer=transfer), texel))
        return _state(cmd, {a: (d, _f16(g, w, h, "opaque"))}, {o: od})
    if kind == "padded_over":
        d = _padded(z.Descriptor.rgba8_srgb(w, h))
        a, b = cmd.input(d), cmd.input(d)
        ab = cmd.blend(a, z.Rectangle(0, 0, w, h), b)
        o, od = cmd.output(cmd.color_convert(ab, P3_LINEAR, RGBA16F))
        return _state(cmd, {a: (d, _pad_rows(_u8(g, w, h), d)), b: (d, _pad_rows(_u8(g, w, h, "soft"), d))}, {o: od})
    if kind == "paste":
        fw, fh = case["fw"], case["fh"]
        d, fd = z.Descriptor.rgba8_srgb(w, h), z.Descriptor.rgba8_srgb(fw, fh)
        a = cmd.input(d)
        inputs = {a: (d, _u8(g, w, h))}
        if case["op"] == "crop":
            v = cmd.crop(a, z.Rectangle(0, 0, fw, fh))
        elif case["op"] == "resize":
            v = cmd.resize(a, fw, fh)
        else:
            b = cmd.input(fd)
            inputs[b] = (fd, _u8(g, fw, fh, "soft"))
            if case["op"] == "inscribe":
                v = cmd.inscribe(a, z.Rectangle(0, 0, fw, fh), b)
            else:
                aff = W.about_centre(fw, fh, 0.9, math.radians(30.0), z.AffineSample.Nearest, out_wh=(w, h))
                v = cmd.affine(a, aff, b)
        o, od = cmd.output(v)
        return _state(cmd, inputs, {o: od})
    if kind == "filter":
        d = z.Descriptor.rgba8_srgb(w, h) if case["texel"] == "u8" else z.Descriptor(w, h, RGBA16F, LINEAR_709)
        a = cmd.input(d)
        method = z.DerivativeMethod.Sobel if case["method"] == "sobel" else z.DerivativeMethod.Scharr3
        axis = z.Direction.Width if case["axis"] == "width" else z.Direction.Height
        o, od = cmd.output(cmd.derivative(a, method, axis))
        return _state(cmd, {a: (d, _u8(g, w, h) if case["texel"] == "u8" else _f16(g, w, h, "opaque"))}, {o: od})
    # generate: the seed moves the parameters
    d = z.Descriptor.rgba8_srgb(w, h) if case["texel"] == "u8" else z.Descriptor(w, h, RGBA16F, LINEAR_709)
    rng = np.random.default_rng(int(seed))
    if case["op"] == "noise":
        n = z.FractalNoise.with_octaves(case["octaves"])
        n.grid_scale = (float(rng.uniform(20, 200)), float(rng.uniform(20, 200)))
        v = cmd.distribution_fractal_noise(d, n)
    elif case["op"] == "normal":
        d = d.with_(texel=z.Texel(SB.UInt8, SP.Luma)) if case["texel"] == "u8" else d.with_(
            texel=z.Texel(SB.UInt16x2, SP.LumaA))
        v = cmd.distribution_normal2d(d, z.DistributionNormal2d.with_diagonal(float(rng.uniform(0.3, 1.0)),
                                                                              float(rng.uniform(0.3, 1.0))))
    else:
        c = [tuple(float(x) for x in rng.uniform(0, 0.5, 3)) + (0.5,) for _ in range(4)]
        v = cmd.bilinear(d, z.Bilinear(u_min=c[0], u_max=c[1], v_min=c[2], v_max=c[3]))
    o, od = cmd.output(v)
    return _state(cmd, {}, {o: od})


def run(state):
    if "pool" in state:
        pool = state["pool"]
        e = state["exe"].launch_pool(pool, state["keys"], {state["out"]: 0})
        key = e.retire_output(state["out"])
        e.finish()
        image = pool.as_bytes(key)
        pool.remove(key)
        return image
    state["exe"].launch(state["ins"], state["outs"])
    return state["result"]


# ---- what a pass cannot do without -----------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "batch":
        bytes_, px = 0, 0
        for w, h, fmt, s in _batch_shapes(case):
            ow, oh = max(1, int(round(w * s))), max(1, int(round(h * s)))
            bytes_ += (4, 8)[fmt] * (w * h + ow * oh)
            px += ow * oh
        return dict(bytes=bytes_, flops=60 * px)
    px = case["w"] * case["h"]
    if kind == "relaunch":
        return dict(bytes=8 * px, flops=0)  # the frame in and out; the foreground replaces what it covers
    if kind == "blend_affine":
        s2 = case["scale"] ** 2
        return dict(bytes=int(8 * px * min(1.0, 1.0 / s2)) + 4 * px, flops=90 * px)
    if kind == "grade_over":
        return dict(bytes=16 * px, flops=80 * px)
    if kind == "chain":
        return dict(bytes=8 * px * case["n"], flops=60 * px * case["n"])
    if kind == "composite":
        seen = 0.0
        for aff in _composite_affines(case):
            m = aff.transformation
            seen += min(1.0, 1.0 / max(1e-9, abs(m[0] * m[4] - m[1] * m[3])))
        return dict(bytes=int(8 * px * seen) + 4 * px, flops=(45 * case["layers"] + 60) * px)
    if kind in ("decode", "encode"):
        texel = STAGED[case["fmt"]][0]
        wide = 16 if case.get("out") == "f32" else 8
        return dict(bytes=(texel.bytes + wide) * px, flops=45 * px)
    if kind == "padded_over":
        return dict(bytes=16 * px, flops=50 * px)
    if kind == "paste":
        out = case["fw"] * case["fh"] if case["op"] == "resize" else px
        return dict(bytes=8 * out, flops=0)
    if kind == "filter":
        return dict(bytes=2 * (4 if case["texel"] == "u8" else 8) * px, flops=54 * px)
    bpp = {("normal", "u8"): 1, ("normal", "f16"): 4}.get((case["op"], case["texel"]), 4 if case["texel"] == "u8" else 8)
    # a noise octave: four hashed corners of 30 integer operations, blended in four channels
    return dict(bytes=bpp * px, flops=(160 * case["octaves"] if case["op"] == "noise" else 30) * px)


# ---- 64-bit values of the floating outputs ------------------------------------------------
_CHROMATICITIES = {P.Bt709: ((0.640, 0.330), (0.300, 0.600), (0.150, 0.060)),
                   P.Bt2020: ((0.708, 0.292), (0.170, 0.797), (0.131, 0.046)),
                   P.DisplayP3: ((0.680, 0.320), (0.265, 0.690), (0.150, 0.060))}


def _to_xyz(primaries):
    m = np.array([[x / y, 1.0, (1 - x - y) / y] for x, y in _CHROMATICITIES[primaries]]).T
    x, y = 0.3127, 0.3290
    return m * np.linalg.solve(m, np.array([x / y, 1.0, (1 - x - y) / y]))


def _convert(v, src, dst):
    """Linear RGB of (h, w, 4) from primaries to primaries."""
    m = torch.tensor(np.linalg.solve(_to_xyz(dst), _to_xyz(src)), device=v.device)
    return torch.cat([v[..., :3] @ m.T, v[..., 3:]], dim=-1)


def _eotf(v, transfer):
    if transfer == T.Srgb:
        return torch.where(v <= 0.04045, v / 12.92, ((v + 0.055) / 1.055).clamp(min=0) ** 2.4)
    t = 1.099 * 0.018 ** 0.45 - 0.099
    return torch.where(v >= t, ((v + 0.099) / 1.099).clamp(min=0) ** (1 / 0.45), v / 4.5)


def _decode_u8(t):
    v = t.to(torch.float64) / 255.0
    return torch.cat([_eotf(v[..., :3], T.Srgb), v[..., 3:]], dim=-1)


def _exact_decode(case, seed):
    fmt = case["fmt"]
    _, transfer, prim = STAGED[fmt]
    codes = _staged_codes(_generator(seed, 0), fmt, case["w"], case["h"])
    if fmt == "10bit_bt2020":
        c = codes.to(torch.int64) & 0xFFFFFFFF
        v = torch.stack([c & 1023, (c >> 10) & 1023, (c >> 20) & 1023], dim=-1).double() / 1023.0
        alpha = (c >> 30).double() / 3.0
    elif fmt == "16bit_srgb":
        v = (codes.to(torch.int64) & 0xFFFF).double() / 65535.0
        alpha, v = v[..., 3], v[..., :3]
    elif fmt == "rgb565_srgb":
        c = codes.to(torch.int64) & 0xFFFF
        v = torch.stack([(c & 31).double() / 31.0, ((c >> 5) & 63).double() / 63.0, (c >> 11).double() / 31.0], dim=-1)
        alpha = torch.ones_like(v[..., 0])
    else:
        v = codes.double() / 255.0
        if fmt == "luma8_srgb":
            v = torch.stack([v, v, v], dim=-1)
        alpha = v[..., 3] if fmt == "8bit_bt709" else torch.ones_like(v[..., 0])
        v = v[..., :3]
    return {"out0": _convert(torch.cat([_eotf(v, transfer), alpha[..., None]], dim=-1), prim, P.DisplayP3)}


def _exact_padded_over(case, seed):
    g = _generator(seed, 0)
    below, above = _decode_u8(_u8(g, case["w"], case["h"])), _decode_u8(_u8(g, case["w"], case["h"], "soft"))
    ta, ba = above[..., 3:], below[..., 3:] * (1 - above[..., 3:])
    alpha = ta + ba
    rgb = torch.where(alpha > 0, (above[..., :3] * ta + below[..., :3] * ba) / alpha.clamp(min=1e-300),
                      torch.zeros_like(alpha))
    return {"out0": _convert(torch.cat([rgb, alpha], dim=-1), P.Bt709, P.DisplayP3)}


def _axis_taps(n_out, n_in, scale32):
    """Left tap, its weight and the right tap's, zero outside the source."""
    u = (torch.arange(n_out, device="cuda", dtype=torch.float64) + 0.5) / scale32 - 0.5
    i = torch.floor(u)
    f = u - i
    i = i.long()
    left = torch.where((i >= 0) & (i < n_in), 1 - f, torch.zeros_like(f))
    right = torch.where((i + 1 >= 0) & (i + 1 < n_in), f, torch.zeros_like(f))
    return i.clamp(0, n_in - 1), (i + 1).clamp(0, n_in - 1), left, right


def _exact_batch(case, seed):
    offsets, total = _batch_layout(case)
    out = torch.zeros(max(total[1], 256) // 2, device="cuda", dtype=torch.float64)
    for k, (w, h, fmt, s) in enumerate(_batch_shapes(case)):
        if fmt == 0:
            continue
        ow, oh = max(1, int(round(w * s))), max(1, int(round(h * s)))
        v = _convert(_f16(_generator(seed, 300 + k), w, h).double(), P.Bt709, P.DisplayP3)
        v[..., :3] *= v[..., 3:]
        i0, i1, a, b = _axis_taps(oh, h, float(np.float32(oh / h)))
        v = v[i0] * a[:, None, None] + v[i1] * b[:, None, None]
        i0, i1, a, b = _axis_taps(ow, w, float(np.float32(ow / w)))
        v = v[:, i0] * a[None, :, None] + v[:, i1] * b[None, :, None]
        rgb = torch.where(v[..., 3:] > 0, v[..., :3] / v[..., 3:].clamp(min=1e-300), torch.zeros_like(v[..., :3]))
        v = torch.cat([rgb, v[..., 3:]], dim=-1).reshape(-1)
        out[offsets[k] // 2:offsets[k] // 2 + v.numel()] = v
    return {"u8": None, "f16": out}


def _exact_filter(case, seed):
    w, h = case["w"], case["h"]
    v = _f16(_generator(seed, 0), w, h, "opaque").double()
    side = {"sobel": (0.25, 0.5), "scharr3": (46.84 / 256.0, 162.32 / 256.0)}[case["method"]]
    smooth, diff = (side[0], side[1], side[0]), (0.5, 0.0, -0.5)
    out = torch.zeros_like(v)
    ys, xs = torch.arange(h, device="cuda"), torch.arange(w, device="cuda")
    for dy in range(3):
        for dx in range(3):
            k = smooth[dy] * diff[dx] if case["axis"] == "width" else smooth[dx] * diff[dy]
            out += k * v[(ys + dy - 1).clamp(0, h - 1)][:, (xs + dx - 1).clamp(0, w - 1)]
    out[..., 3] = 1.0
    return {"out0": out}


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _exact_decode(case, seed)
    if kind == "padded_over":
        return _exact_padded_over(case, seed)
    if kind == "batch":
        return _exact_batch(case, seed)
    if kind == "filter" and case["texel"] == "f16":
        return _exact_filter(case, seed)
    if kind == "generate" and case["op"] == "ramp" and case["texel"] == "f16":
        rng = np.random.default_rng(int(seed))
        c = [torch.tensor([float(x) for x in rng.uniform(0, 0.5, 3)] + [0.5], device="cuda", dtype=torch.float32).double()
             for _ in range(4)]
        u = ((torch.arange(case["w"], device="cuda", dtype=torch.float64) + 0.5) / case["w"])[None, :, None]
        v = ((torch.arange(case["h"], device="cuda", dtype=torch.float64) + 0.5) / case["h"])[:, None, None]
        return {"out0": c[0] + (c[1] - c[0]) * u + c[2] + (c[3] - c[2]) * v}
    return None
